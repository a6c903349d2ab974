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


WALKED, ANY = 4, 6      # kernels that a launch is said to have taken


def move(pkg, gpu, views, align, joint=False, witness=None, prepared=False):
    """The kernels that moved the bundle, packing and unpacking."""
    plan = pkg.BundlePlan.create(views, align=align)
    n = plan.payload_bytes
    payload = torch.full((n + 32,), 0x5a, dtype=torch.uint8, device=gpu)
    outs = [torch.zeros_like(v.contiguous().permute(0, 2, 1).contiguous()).permute(0, 2, 1) if v.dim() == 3 else torch.zeros_like(v)
            for v in views]
    recv = pkg.BundlePlan.from_header(plan.header).bind(outs)
    if prepared:
        plan.prepare()
        recv.prepare()
    plan.pack(payload.data_ptr(), n)
    for v, at, size in zip(views, *plan.layout()):
        assert torch.equal(payload[at:at + size], v.contiguous().view(-1).view(torch.uint8))
    assert bool((payload[n:] == 0x5a).all())
    if joint:      # both directions in one launch, in the kernel for any mode
        second = torch.zeros_like(payload)
        jobs = [(plan, second, 0), (recv, payload, 1)]
        if witness is not None:      # walked blocks alone, whose kernel tells whether a launch was shared
            third = pkg.BundlePlan.create(witness, align=align)
            jobs.insert(1, (third, torch.zeros(third.payload_bytes, dtype=torch.uint8, device=gpu), 0))
        table = (pkg._capi.Job * len(jobs))()
        for j, (p, y, unpack) in zip(table, jobs):
            j.plan, j.payload, j.payload_bytes, j.unpack = p._h, y.data_ptr(), p.payload_bytes, unpack
        pkg._capi.check(pkg._capi.load().axr_submit(table, len(jobs), None))
        assert torch.equal(second[:n], payload[:n])
        if witness is not None:
            for v, at, size in zip(witness, *third.layout()):
                assert torch.equal(jobs[1][1][at:at + size], v.contiguous().view(-1).view(torch.uint8))
            assert third.launch_info()["last_launch"] >> 4 & 15 == ANY
            third.close()
    else:
        recv.unpack(payload.data_ptr(), n)
    assert all(torch.equal(v, o) for v, o in zip(views, outs))
    kernels = [p.launch_info()["last_launch"] >> 4 & 15 for p in (plan, recv)]
    plan.close()
    recv.close()
    return kernels


# extents of 9 to 12 blocks and one element more or less, against a long other side, both ways round
@pytest.mark.gpu
@pytest.mark.parametrize("item,edges", [(2, (513, 576, 577, 639, 640, 641, 704, 705, 768, 769)), (4, (1025, 1055, 1056, 1057, 1120, 1153)),
                                        (8, (129, 159, 160, 161, 191, 192, 193, 225, 256, 257))])
@pytest.mark.parametrize("turned", [False, True])
def test_groups(pkg, gpu, item, edges, turned):
    for edge in edges:
        for align, lead, batch in ((1, 0, 1), (256, 3, 3 if edge < 600 else 1)):
            other = (30 << 20) // (edge * item) + 41
            other = (other if batch == 1 else other // 2 + 3) | 1     # odd: with both sides' rows on lines blocks stay plain
            a, b = (other, edge) if turned else (edge, other)
            view, _ = bundle(gpu, item, a, b, batch, lead)
            assert move(pkg, gpu, [view], align) == [WALKED, WALKED], (a, b, batch)


@pytest.mark.gpu
def test_other_kernels_move_the_same_tiles(pkg, gpu):
    lib = pkg._capi.load()
    view, _ = bundle(gpu, 2, 705, 30011, 1, 1)
    wide, _ = bundle(gpu, 4, 1031, 8009, 1, 1)
    compact = torch.randint(0, 256, (100001,), dtype=torch.uint8, device=gpu)
    for joint in (False, True):
        # (bundles whose workgroups are handed to the dies in turn have launches to themselves)
        pkg.tune(xcd_remap=0 if joint else -1)
        try:
            alone = [ANY if joint else WALKED] * 2
            assert move(pkg, gpu, [view], 1, joint) == alone
            assert move(pkg, gpu, [view, wide, view[:, :, 3:]], 1, joint) == alone
            assert move(pkg, gpu, [view, compact, wide], 1, joint, [view]) == [ANY, ANY]
        finally:
            pkg.tune(xcd_remap=-1)
    for name, value, usual, kernel in (("threads", 128, 0, ANY), ("threads", 256, 0, WALKED), ("max_waves", 1000, 1 << 20, ANY),
                                       ("xcd_remap", 1, -1, WALKED), ("xcd_remap", 0, -1, WALKED)):
        pkg._capi.check(lib.axr_tune_set(name.encode(), value))
        try:
            # (workgroups in the order of the dies: the first launch has its tables in the arguments, and a kernel for any mode)
            first = ANY if (name, value) == ("xcd_remap", 0) else kernel
            assert move(pkg, gpu, [view, wide], 1) == [first, first], name
            assert move(pkg, gpu, [view, wide], 1, prepared=True) == [kernel, kernel], name
        finally:
            pkg._capi.check(lib.axr_tune_set(name.encode(), usual))
