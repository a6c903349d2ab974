"""Which way bundles are launched: where the tables of a first and of a later launch are, which kernel moves them
and how much of a streaming payload stays in the cache, on both sides of the rules' borders.  (The bytes that
each way moves are compared elsewhere; here a way that is silently never taken shows.)"""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

KIB, MIB = 1 << 10, 1 << 20
ARGUMENTS, PINNED, UPLOADED, DEVICE_BUILT = 1, 2, 3, 4
RUNS, ELEMENTS, ROWS, BLOCKS, WALKED, PLANES, ANY = range(7)


def route(plan):
    """(tables, kernel, MiB of cached tail) of the plan's latest launch."""
    last = plan.launch_info()["last_launch"]
    return last & 15, last >> 4 & 15, last >> 8


def carve(gpu, sizes):
    store = torch.zeros(sum(sizes), dtype=torch.uint8, device=gpu)
    return list(store.split(list(sizes)))


def launches(pkg, tensors, count=2, align=256):
    """The routes of that many packs of one plan.  (Asking for a route builds host tables where a kernel had
    laid them out, so a plan that is asked after its first launch is not launched again.)"""
    out = []
    for n in range(1, count + 1):
        with pkg.BundlePlan.create(tensors, align=align) as plan:
            payload = torch.empty(plan.payload_bytes, dtype=torch.uint8, device=tensors[0].device)
            for _ in range(n):
                plan.pack(payload.data_ptr(), payload.numel())
            out.append(route(plan))
            torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("sizes,first,later", [
    ([64 * KIB] * 98, ARGUMENTS, UPLOADED),            # 3.5 KiB hold 99 records of 32 bytes, an index of as many blocks
    ([64 * KIB] * 99, PINNED, UPLOADED),               # and a mark, no more
    ([64 * KIB] * 383, PINNED, UPLOADED),
    ([64 * KIB] * 384, DEVICE_BUILT, DEVICE_BUILT),
    ([300] * 300, PINNED, UPLOADED),                   # blocks of groups: up to 32 KiB of them,
    ([300] * 511, UPLOADED, UPLOADED),                 # from a third more tensors on laid out by a kernel
    ([300] * 512, DEVICE_BUILT, DEVICE_BUILT),
    ([16384 * 2 * KIB], ARGUMENTS, UPLOADED),          # small bundles end at 16,384 tiles,
    ([16385 * 2 * KIB], ARGUMENTS, UPLOADED),          # a long tensor's index fits in wide blocks,
    ([20 * MIB] + [600] * 100 + [16 * MIB], UPLOADED, UPLOADED),     # but not with many short ones in a block
    ([320 * KIB] * 112, UPLOADED, UPLOADED),           # beyond 16,384 tiles nothing is read in pinned memory
], ids=lambda v: f"{len(v)}x{v[0]}" if isinstance(v, list) else str(v))
def test_where_the_tables_are(pkg, gpu, sizes, first, later):
    group = 512 if sizes[0] < KIB else 0
    pkg.tune(group_bytes=group)
    try:
        assert [r[:2] for r in launches(pkg, carve(gpu, sizes))] == [(first, RUNS), (later, RUNS)]
    finally:
        pkg.tune(group_bytes=512)


def test_views_with_their_own_records_are_uploaded(pkg, gpu):
    store = torch.zeros(8, 400, 4 * KIB, dtype=torch.uint8, device=gpu)
    alike = [store[:, i, :2 * KIB] for i in range(400)]
    differ = [store[:1 + i % 8, i, :1300 + i] for i in range(120)]
    assert [r[0] for r in launches(pkg, alike)] == [PINNED, UPLOADED]
    assert [r[0] for r in launches(pkg, differ)] == [UPLOADED, UPLOADED]


def test_switched_off(pkg, gpu):
    pkg.tune(inline_tables=0, device_tables=0)
    try:
        for n in (3, 200, 600):
            assert [r[0] for r in launches(pkg, carve(gpu, [64 * KIB] * n))] == [UPLOADED, UPLOADED]
    finally:
        pkg.tune(inline_tables=16384, device_tables=384)


VIEWS = {
    RUNS: lambda s: [s[:70000]],
    ELEMENTS: lambda s: [s[:32768].view(4096, 8)[:, :6]],
    ROWS: lambda s: [s[:40 * 131].view(40, 131)[:, :100], s[:90 * 512].view(90, 512)[:, 256:448]],
    BLOCKS: lambda s: [s[:300 * 196].view(300, 196).t()],
    WALKED: lambda s: [s[:2051 * 17001 * 2].view(torch.int16).view(2051, 17001).t()],
    PLANES: lambda s: [s[:3 * 70 * 33 * 4].view(4, 70, 33, 3).permute(0, 3, 1, 2)],
}


@pytest.mark.parametrize("kind", VIEWS)
def test_every_kind_has_its_kernel(pkg, gpu, kind):
    store = torch.zeros(2051 * 17001 * 2 + 70000, dtype=torch.uint8, device=gpu)
    views = VIEWS[kind](store)
    # in the arguments: kernels for runs, for rows and for any
    assert [r[1] for r in launches(pkg, views)] == [ANY if kind in (ELEMENTS, BLOCKS, PLANES) else kind, kind]
    if kind != RUNS:
        assert [r[1] for r in launches(pkg, views + [store[-70000:]])] == [ANY, ANY]
        pkg.tune(tile_rows=4)
        try:
            assert launches(pkg, views)[1][1] == ANY
        finally:
            pkg.tune(tile_rows=0)


@pytest.mark.parametrize("kinds,want", [((ROWS, ROWS), (ROWS, ROWS)), ((ROWS, RUNS), (ANY, ANY)), ((BLOCKS, BLOCKS), (ANY, ANY)),
                                        ((PLANES, PLANES), (PLANES, PLANES)), ((PLANES, ROWS), (ANY, ANY)),
                                        ((RUNS, RUNS), (RUNS, RUNS)), (("many", RUNS), (ROWS, RUNS)), (("many", ROWS), (ROWS, ROWS)),
                                        ((BLOCKS, "many"), (BLOCKS, ROWS)), ((ROWS, "many", RUNS), (ROWS, ROWS, RUNS)),
                                        ((ROWS, RUNS, "many"), (ANY, ANY, ROWS)), (("some", "some", RUNS), (ROWS, ROWS, RUNS)),
                                        (("some", RUNS), (ANY, ANY))], ids=str)
def test_kinds_in_one_submission(pkg, gpu, kinds, want):
    capi = pkg._capi
    store = torch.zeros(40000 * 131, dtype=torch.uint8, device=gpu)
    rows = {"many": 40000, "some": 20000}      # tiles of 16: 2500 and 1250 of them
    plans = [pkg.BundlePlan.create([store.view(40000, 131)[:rows[k], :100]] if k in rows else VIEWS[k](store), align=64).prepare() for k in kinds]
    payloads = [torch.empty(p.payload_bytes, dtype=torch.uint8, device=gpu) for p in plans]
    jobs = (capi.Job * len(plans))()
    for j, p, y in zip(jobs, plans, payloads):
        j.plan, j.payload, j.payload_bytes = p._h, y.data_ptr(), y.numel()
    capi.check(capi.load().axr_submit(jobs, len(plans), C.c_void_p()))
    assert tuple(route(p)[1] for p in plans) == want
    torch.cuda.synchronize()
    for p in plans:
        p.close()


def test_cached_tail(pkg, gpu):
    """Seven eighths of the cache, of payloads that stream in 1 KiB tiles, when they are packed and nothing else is asked for."""
    tensors = carve(gpu, [5 * MIB, 4 * MIB])
    strided = [torch.zeros(9 * MIB // 256, 300, dtype=torch.uint8, device=gpu)[:, :256]]
    pkg.tune(payload_cache_bytes=8 * MIB)
    try:
        assert [r[2] for r in launches(pkg, tensors)] == [7, 7]
        assert [r[2] for r in launches(pkg, tensors[:1] + [tensors[1][:3 * MIB]])] == [0, 0]      # 8 MiB do not stream
        assert [r[2] for r in launches(pkg, strided)] == [0, 0]
        with pkg.BundlePlan.create(tensors, align=256) as send, \
                pkg.BundlePlan.from_header(send.header).bind([t.clone() for t in tensors]) as recv:
            payload = torch.empty(send.payload_bytes, dtype=torch.uint8, device=gpu)
            job = pkg._capi.Job()
            job.plan, job.payload, job.payload_bytes, job.flags = send._h, payload.data_ptr(), payload.numel(), pkg._capi.JOB_PAYLOAD_STREAMING
            pkg._capi.check(pkg._capi.load().axr_submit(job, 1, None))
            assert route(send)[2] == 0
            recv.unpack(payload.data_ptr(), payload.numel())
            assert route(recv)[2] == 0
            torch.cuda.synchronize()
        pkg.tune(nontemporal=3)
        assert [r[2] for r in launches(pkg, tensors)] == [0, 0]
    finally:
        pkg.tune(payload_cache_bytes=256 * MIB, nontemporal=-1)
