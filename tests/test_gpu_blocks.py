"""Transposed views at the edges of their blocks: skewed blocks (bundles beyond 28 MiB whose written
rows do not start on 64-byte boundaries) and few planes against interleaved elements.  Packed bytes
against torch's compact copies, views scattered back into zeroed twins, nothing written beside them."""
import pytest

pytestmark = pytest.mark.gpu

DTYPES = {1: "uint8", 2: "int16", 4: "int32", 8: "int64", 16: "complex128"}


def storage(torch, gpu, n, item, lead, seed):
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    # (bytes below 120: no NaN among the complex numbers)
    raw = torch.randint(0, 256 if item < 16 else 120, ((n + lead) * item,), dtype=torch.uint8, device=gpu, generator=g)
    return raw.view(getattr(torch, DTYPES[item]))


def round_trip(pkg, gpu, stores, views_of, align, shift=0):
    import torch
    views = views_of(stores)
    plan = pkg.BundlePlan.create(views, align=align)
    n = plan.payload_bytes
    buf = torch.full((n + shift + 64,), 0xCD, dtype=torch.uint8, device=gpu)
    plan.pack(buf.data_ptr() + shift, n)
    twins = [torch.zeros_like(s) for s in stores]
    outs = views_of(twins)
    recv = pkg.BundlePlan.from_header_bound(plan.header, outs)
    recv.unpack(buf.data_ptr() + shift, n)
    torch.cuda.synchronize()
    for v, o, off, size in zip(views, outs, *plan.layout()):
        assert torch.equal(buf[shift + off:shift + off + size], v.contiguous().reshape(-1).view(torch.uint8))
        assert torch.equal(o, v)
    assert (buf[:shift] == 0xCD).all() and (buf[shift + n:] == 0xCD).all()
    for t, o in zip(twins, outs):
        o.zero_()
        assert not t.any()
    recv.close()
    plan.close()


# shapes around the block edge (128, 64, 32, 32 elements; bytes are not skewed) and the staged window, next to a large matrix
# that takes the bundle beyond the limit; odd rows, odd starts, one side aligned, a gap behind rows
@pytest.mark.parametrize("item", [1, 2, 4, 8])
@pytest.mark.parametrize("align,lead,shift", [(1, 0, 0), (256, 1, 0), (2, 3, 6)])
def test_skewed_blocks(pkg, gpu, item, align, lead, shift):
    import torch
    edge = {1: 128, 2: 64}.get(item, 32)
    shapes = [(2051, (34 << 20) // 2051 // item | 1), (edge, edge), (edge, edge + 1), (edge + 1, edge),
              (2 * edge - 1, edge + 31), (3 * edge + 5, 2 * edge), (4 * edge, edge + 17), (edge - 1, 300), (777, 130)]
    stores = [storage(torch, gpu, r * c, item, lead, i) for i, (r, c) in enumerate(shapes)]

    def views(ss):
        full = [s[lead:].view(r, c).t() for s, (r, c) in zip(ss, shapes)]
        return full[:-1] + [full[-1][:123]]        # the last one leaves a gap behind every row

    round_trip(pkg, gpu, stores, views, align, shift)


# Shapes at the edges of the rule that takes blocks to the skewed routine and to strips (rows of
# `least` elements; B four times as long as A; one dimension just above a block), with batch
# dimensions, next to a matrix that takes the bundle beyond 32 or 96 MiB; several tiles per wavefront,
# streaming on both sides, either die mapping
@pytest.mark.parametrize("item", [2, 4, 8, 16])
@pytest.mark.parametrize("mib", [33, 97])
@pytest.mark.parametrize("tunables", [{}, {"nontemporal": 3, "max_waves": 3001}, {"nontemporal": 0, "threads": 64},
                                      {"xcd_remap": 1}, {"xcd_remap": 0, "max_waves": 500}], ids=str)
@pytest.mark.parametrize("align,lead", [(1, 1), (256, 0)])
def test_blocks_at_the_edges_of_their_rule(pkg, gpu, item, mib, tunables, align, lead):
    import torch
    edge, least = {2: (64, 512), 4: (32, 1024), 8: (32, 128), 16: (16, 512)}[item]
    shapes = [(least, least), (least + 1, least + edge - 1), (least + edge + 31, least + 1), (least - 1, 4 * least),
              (edge, max(4 * edge, least)), (edge + 3, max(4 * edge + 12, least) + 1), (edge + 3, 4 * edge + 11),
              (4 * least + 3, least), (2, 3, least + 5, least + edge // 2 + 1), (5, edge + 9, max(4 * edge + 36, least) + 3)]
    if align == 256:     # rows on lines on one side or the other
        lines = 128 // min(item, 128)
        shapes += [(least + 1, (least // lines + 2) * lines), ((least // lines + 2) * lines, least + 1)]
    have = sum(torch.Size(s).numel() for s in shapes) * item
    rows = 2051
    shapes.append((rows, max(((mib << 20) - have) // rows // item, 1) | 1))
    stores = [storage(torch, gpu, torch.Size(s).numel(), item, lead, i) for i, s in enumerate(shapes)]

    def views(ss):
        return [s[lead:lead + torch.Size(shape).numel()].view(shape).transpose(-1, -2) for s, shape in zip(ss, shapes)]

    try:
        pkg.tune(**tunables)
        round_trip(pkg, gpu, stores, views, align, 0 if align > 1 else 3)
    finally:
        pkg.tune(nontemporal=-1, max_waves=1 << 20, threads=0, xcd_remap=-1)


@pytest.mark.parametrize("item", [2, 4, 8])
@pytest.mark.parametrize("remap", [-1, 0])
def test_skewed_blocks_in_submitted_jobs_at_another_address(pkg, gpu, item, remap):
    """Joint and single launches of plans moved by a tensor delta that changes how rows lie to
    64-byte boundaries."""
    import torch
    lib, capi = pkg._capi.load(), pkg._capi
    r, c = 2051, (34 << 20) // 2051 // item | 1
    there, back = 5, 9          # elements from where the plans were made
    src, dst = (torch.randint(0, 120, (r * c + 16,), dtype=torch.uint8, device=gpu).to(getattr(torch, DTYPES[item])) for _ in "ab")
    want_dst = dst.clone()
    flat = [torch.randint(0, 256, (100001,), dtype=torch.uint8, device=gpu) for _ in range(2)]

    def view(s, at):
        return s[at:at + r * c].view(r, c).t()

    try:
        pkg.tune(xcd_remap=remap)
        send, other = pkg.BundlePlan.create([view(src, 0)], align=1), pkg.BundlePlan.create([flat[0]], align=1)
        recv = pkg.BundlePlan.from_header_bound(send.header, [view(dst, 0)])
        n = send.payload_bytes
        payload, small = torch.zeros(n + 3, dtype=torch.uint8, device=gpu), torch.zeros(100001, dtype=torch.uint8, device=gpu)
        jobs = (capi.Job * 2)()
        jobs[0] = capi.Job(send._h, 0, payload.data_ptr() + 3, n, there * item)
        jobs[1] = capi.Job(other._h, 0, small.data_ptr(), small.numel(), 0)
        capi.check(lib.axr_submit(jobs, 2, None))
        torch.cuda.synchronize()
        assert torch.equal(payload[3:], view(src, there).contiguous().reshape(-1).view(torch.uint8))
        assert torch.equal(small, flat[0])
        jobs[0] = capi.Job(other._h, 0, small.data_ptr(), small.numel(), 0)
        jobs[1] = capi.Job(recv._h, 1, payload.data_ptr() + 3, n, back * item)
        capi.check(lib.axr_submit(jobs, 2, None))
        torch.cuda.synchronize()
        view(want_dst, back).copy_(view(src, there))
        assert torch.equal(dst, want_dst)
    finally:
        pkg.tune(xcd_remap=-1)
    for p in (send, other, recv):
        p.close()


# the long dimension below one vector, one vector, ragged, a whole block, one element more, several
@pytest.mark.parametrize("item", [1, 2, 4])
@pytest.mark.parametrize("planes", [2, 3, 4])
@pytest.mark.parametrize("long", [15, 16, 343, 1024, 2048, 2049, 5001])
def test_planes_and_interleaved(pkg, gpu, item, planes, long):
    import torch
    stores = [storage(torch, gpu, 3 * long * planes, item, lead, lead) for lead in (0, 1)]

    def views(ss):
        inter = [s[k:].view(3, long, planes).permute(0, 2, 1) for k, s in enumerate(ss)]    # tensor interleaved
        return inter

    def planar(ss):
        return [s[k:].view(3, planes, long).permute(0, 2, 1) for k, s in enumerate(ss)]     # payload interleaved

    for make in (views, planar):
        for align, shift in ((1, 0), (256, 3)):
            round_trip(pkg, gpu, stores, make, align, shift)


# ends that are no whole vector: one vector and a bit, just below and above a block (2048, 1024 and
# 1024 / 680 / 512 elements), less than a vector behind the last whole block; several tiles per
# wavefront and streaming on both sides
@pytest.mark.parametrize("item", [1, 2, 4])
@pytest.mark.parametrize("planes", [2, 3, 4])
@pytest.mark.parametrize("long", [17, 90, 345, 511, 513, 679, 681, 1023, 1025, 1361, 2047, 2051, 3000, 4097])
@pytest.mark.parametrize("tunables", [{}, {"nontemporal": 3, "max_waves": 37}], ids=["plain", "streams"])
def test_ragged_planes(pkg, gpu, item, planes, long, tunables):
    import torch
    stores = [storage(torch, gpu, 40 * long * planes, item, lead, lead) for lead in (0, 1)]

    def inter(ss):
        return [s[k:].view(40, long, planes).permute(0, 2, 1) for k, s in enumerate(ss)]

    def planar(ss):
        return [s[k:].view(40, planes, long).permute(0, 2, 1) for k, s in enumerate(ss)]

    def apart(ss):       # a gap behind every plane
        return [s[k:].view(20, planes, 2 * long)[:, :, :long].permute(0, 2, 1) for k, s in enumerate(ss)]

    try:
        pkg.tune(**tunables)
        for make in (inter, planar, apart):
            round_trip(pkg, gpu, stores, make, 1, 3)
            round_trip(pkg, gpu, stores, make, 256, 0)
    finally:
        pkg.tune(nontemporal=-1, max_waves=1 << 20)
