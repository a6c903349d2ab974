"""Skewed blocks moved by a workgroup together: whole and ragged groups in either direction, bundles whose kernel
moves them one by one instead, empty tiles behind the last group."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

BITS = {2: torch.int16, 4: torch.int32, 8: torch.int64}


def bundle(gpu, item, a, b, batch, lead):
    """(a, b): extents along the payload's rows and along the tensor's; beyond 28 MiB together with the filler."""
    n = batch * a * b * item
    store = torch.randint(0, 256, (n + 64,), dtype=torch.uint8, device=gpu)
    return store[lead * item:lead * item + n].view(BITS[item]).view(batch, a, b).permute(0, 2, 1), store


def move(pkg, gpu, views, align, joint=False):
    plan = pkg.BundlePlan.create(views, align=align)
    n = plan.payload_bytes
    payload = torch.full((n + 32,), 0x5a, dtype=torch.uint8, device=gpu)
    outs = [torch.zeros_like(v.contiguous().permute(0, 2, 1).contiguous()).permute(0, 2, 1) if v.dim() == 3 else torch.zeros_like(v)
            for v in views]
    recv = pkg.BundlePlan.from_header(plan.header).bind(outs)
    plan.pack(payload.data_ptr(), n)
    for v, at, size in zip(views, *plan.layout()):
        assert torch.equal(payload[at:at + size], v.contiguous().view(-1).view(torch.uint8))
    assert bool((payload[n:] == 0x5a).all())
    if joint:      # both directions in one launch, in the kernel for any mode
        from execution_ucx_amd import _capi
        second = torch.zeros_like(payload)
        jobs = (_capi.Job * 2)()
        jobs[0].plan, jobs[0].payload, jobs[0].payload_bytes, jobs[0].unpack = plan._h, second.data_ptr(), n, 0
        jobs[1].plan, jobs[1].payload, jobs[1].payload_bytes, jobs[1].unpack = recv._h, payload.data_ptr(), n, 1
        _capi.check(_capi.load().axr_submit(jobs, 2, None))
        assert torch.equal(second[:n], payload[:n])
    else:
        recv.unpack(payload.data_ptr(), n)
    assert all(torch.equal(v, o) for v, o in zip(views, outs))
    info = plan.launch_info()
    plan.close()
    recv.close()
    return info


# extents of 9 to 12 blocks and one element more or less, against a long other side, both ways round
@pytest.mark.gpu
@pytest.mark.parametrize("item,edges", [(2, (513, 576, 577, 639, 640, 641, 704, 705, 768, 769)), (4, (1025, 1055, 1056, 1057, 1120, 1153)),
                                        (8, (129, 159, 160, 161, 191, 192, 193, 225, 256, 257))])
@pytest.mark.parametrize("turned", [False, True])
def test_groups(pkg, gpu, item, edges, turned):
    for edge in edges:
        other = (30 << 20) // (edge * item) + 41
        a, b = (other, edge) if turned else (edge, other)
        for align, lead, batch in ((1, 0, 1), (256, 3, 3 if edge < 600 else 1)):
            view, _ = bundle(gpu, item, a, b if batch == 1 else b // 2 + 3, batch, lead)
            move(pkg, gpu, [view], align)


@pytest.mark.gpu
def test_other_kernels_move_the_same_tiles(pkg, gpu):
    lib = pkg._capi.load()
    view, _ = bundle(gpu, 2, 705, 30011, 1, 1)
    wide, _ = bundle(gpu, 4, 1031, 8009, 1, 1)
    for joint in (False, True):
        move(pkg, gpu, [view], 1, joint)
        move(pkg, gpu, [view, wide, view[:, :, 3:]], 1, joint)
        move(pkg, gpu, [view, torch.randint(0, 256, (100001,), dtype=torch.uint8, device=gpu), wide], 1, joint)
    for name, value, usual in (("threads", 128, 0), ("threads", 256, 0), ("max_waves", 1000, 1 << 20), ("xcd_remap", 0, -1), ("xcd_remap", 1, -1)):
        pkg._capi.check(lib.axr_tune_set(name.encode(), value))
        try:
            move(pkg, gpu, [view, wide], 1)
        finally:
            pkg._capi.check(lib.axr_tune_set(name.encode(), usual))
