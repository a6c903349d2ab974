"""Plans whose tables went up on one stream, launched on others that have to wait for them."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")


# views and records go up by a kernel, groups are laid out by one, long tables go up by the copy engine
@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["views", "records", "groups", "long"])
def test_streams_find_the_tables_of_another_stream(pkg, gpu, kind):
    """Fresh plans over and over in recycled table blocks, so that tables read too early or out of a
    cache would be those of the plan before; the same plan is then bound anew."""
    lib, capi = pkg._capi.load(), pkg._capi
    streams = []
    for _ in range(3):
        s = C.c_void_p()
        capi.check(lib.axr_stream_create(C.byref(s)))
        streams.append(s.value)
    parent = torch.randint(0, 256, (700, 9, 2048), dtype=torch.uint8, device=gpu)
    flat = parent.view(-1)

    def tensors(k):
        if kind == "views":
            return [parent[i, 1:, :1400 + (i + k) % 7] for i in range(200)]
        if kind == "records":
            return [parent[i, 0, :2000 + (i + k) % 48] for i in range(700)]
        if kind == "groups":
            return [parent[i, 0, :100 + (i + k) % 48] for i in range(700)]
        return [flat[40 * i:40 * i + 21 + (i + k) % 17] for i in range(20000)] + [parent[:3, ::2, :1500 + k]]

    def want(ts, plan):
        out = torch.zeros(plan.payload_bytes, dtype=torch.uint8, device=gpu)
        for t, at, n in zip(ts, *plan.layout()):
            out[at:at + n] = t.reshape(-1)
        return out

    for k in range(6 if kind != "long" else 2):
        ts = tensors(k)
        with pkg.BundlePlan.create(ts, align=16) as plan:
            expect = want(ts, plan)
            outs = [torch.zeros_like(expect) for _ in range(4)]
            torch.cuda.synchronize()
            for out, s in zip(outs, [None] + streams):
                plan.pack(out.data_ptr(), out.numel(), s, order=False)
            torch.cuda.synchronize()
            assert all(torch.equal(out, expect) for out in outs)
            if kind == "long":
                continue
            plan.bind([t.clone() for t in ts])    # tables anew, uploaded on another stream
            for out in outs:
                out.zero_()
            torch.cuda.synchronize()
            for out, s in zip(outs, streams + [None]):
                plan.pack(out.data_ptr(), out.numel(), s, order=False)
            torch.cuda.synchronize()
            assert all(torch.equal(out, expect) for out in outs)
    for s in streams:
        capi.check(lib.axr_stream_destroy(s))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["views", "records", "groups"])
def test_prepared_plans_on_streams_that_wait_for_nothing(pkg, gpu, kind):
    """axr_plan_prepare on one stream, launches on three others with no event between them, over and over in
    recycled table blocks; then with the tables rebuilt for other tensors, prepared on a stream that had not
    launched the plan before."""
    lib, capi = pkg._capi.load(), pkg._capi
    streams = []
    for _ in range(3):
        s = C.c_void_p()
        capi.check(lib.axr_stream_create(C.byref(s)))
        streams.append(s.value)
    parent = torch.randint(0, 256, (700, 9, 2048), dtype=torch.uint8, device=gpu)

    def tensors(k):
        if kind == "views":
            return [parent[i, 1:, :1400 + (i + k) % 7] for i in range(200)]
        return [parent[i, 0, :(2000 if kind == "records" else 100) + (i + k) % 48] for i in range(700)]

    for k in range(8):
        ts = tensors(k)
        with pkg.BundlePlan.create(ts, align=16) as plan:
            expect = torch.zeros(plan.payload_bytes, dtype=torch.uint8, device=gpu)
            for t, at, n in zip(ts, *plan.layout()):
                expect[at:at + n] = t.reshape(-1)
            outs = [torch.zeros_like(expect) for _ in range(3)]
            for first in (0, 1):
                torch.cuda.synchronize()
                plan.prepare(streams[(k + first) % 3])
                for j, out in enumerate(outs):
                    plan.pack(out.data_ptr(), out.numel(), streams[(k + first + 1 + j) % 3], order=False)
                torch.cuda.synchronize()
                assert all(torch.equal(out, expect) for out in outs)
                plan.bind([t.clone() for t in ts])
                for out in outs:
                    out.zero_()
            # uploaded by a launch, prepared on another stream, launched on the third one
            torch.cuda.synchronize()
            for j in range(2):
                plan.pack(outs[j].data_ptr(), outs[j].numel(), streams[0], order=False)
            plan.prepare(streams[1])
            plan.pack(outs[2].data_ptr(), outs[2].numel(), streams[2], order=False)
            torch.cuda.synchronize()
            assert all(torch.equal(out, expect) for out in outs)
    for s in streams:
        capi.check(lib.axr_stream_destroy(s))


@pytest.mark.gpu
@pytest.mark.parametrize("tensors", [200, 700])    # tables of pitched views, by a kernel, and records laid out by one
def test_tables_are_there_before_the_first_launch_is_done(pkg, gpu, tensors):
    """What waits for a plan's tables (another stream, axr_plan_prepare on the host) does not wait for the launch
    behind them: of the time that a pack of 6 GiB, some 2 ms, needs to end, a prepare takes the first few per cent."""
    import time
    parent = torch.zeros(tensors, (6 << 30) // tensors // 4096, 4096, dtype=torch.uint8, device=gpu)
    ts = [t[1:, :4000] if tensors == 200 else t[1:] for t in parent]
    payload = None
    for _ in range(3):      # the first one loads kernels and allocates
        with pkg.BundlePlan.create(ts, align=16) as plan:
            payload = torch.empty(plan.payload_bytes, dtype=torch.uint8, device=gpu) if payload is None else payload
            torch.cuda.synchronize()
            plan.pack(payload.data_ptr(), payload.numel(), order=False)
            start = time.perf_counter()
            plan.prepare()
            prepared = time.perf_counter()
            torch.cuda.synchronize()
            done = time.perf_counter()
            assert plan.launch_info()["last_launch"] & 15 == (3 if tensors == 200 else 4)    # uploaded, device-built
    assert prepared - start < (done - start) / 2
