"""Transposed views at the edges of their blocks: skewed blocks (bundles beyond 24 MiB whose written
rows do not start on 64-byte boundaries) and few planes against interleaved elements.  Packed bytes
against torch's compact copies, views scattered back into zeroed twins, nothing written beside them."""
import pytest

pytestmark = pytest.mark.gpu

DTYPES = {1: "uint8", 2: "int16", 4: "int32", 8: "int64"}


def storage(torch, gpu, n, item, lead, seed):
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    raw = torch.randint(0, 256, ((n + lead) * item,), dtype=torch.uint8, device=gpu, generator=g)
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
    shapes = [(2051, (26 << 20) // 2051 // item | 1), (edge, edge), (edge, edge + 1), (edge + 1, edge),
              (2 * edge - 1, edge + 31), (3 * edge + 5, 2 * edge), (4 * edge, edge + 17), (edge - 1, 300), (777, 130)]
    stores = [storage(torch, gpu, r * c, item, lead, i) for i, (r, c) in enumerate(shapes)]

    def views(ss):
        full = [s[lead:].view(r, c).t() for s, (r, c) in zip(ss, shapes)]
        return full[:-1] + [full[-1][:123]]        # the last one leaves a gap behind every row

    round_trip(pkg, gpu, stores, views, align, shift)


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
