"""How a plan's tables reach the device, and what views of one geometry share in them."""
import pytest

pytestmark = pytest.mark.gpu


def _round_trip(pkg, gpu, views, align, torch):
    """Packed bytes against torch's own compact copies, and back into views of zeroed twins."""
    plan = pkg.BundlePlan.create(views, align=align)
    n = plan.payload_bytes
    payload = torch.full((n,), 0xCD, dtype=torch.uint8, device=gpu)
    plan.pack(payload.data_ptr(), n)
    offs, sizes = plan.layout()
    twins = [torch.zeros_like(v._base if v._base is not None else v) for v in views]
    outs = [t.as_strided(v.shape, v.stride(), v.storage_offset()) for t, v in zip(twins, views)]
    recv = pkg.BundlePlan.from_header_bound(plan.header, outs)
    recv.unpack(payload.data_ptr(), n)
    torch.cuda.synchronize()
    for v, o, off, size in zip(views, outs, offs, sizes):
        want = v.contiguous().reshape(-1).view(torch.uint8)
        assert torch.equal(payload[off:off + size], want)
        assert torch.equal(o.contiguous().reshape(-1).view(torch.uint8), want)
    for t, o in zip(twins, outs):   # nothing beside the views is written
        o.zero_()
        assert not t.any()
    recv.close()
    plan.close()


# one tensor, the last table vector partly used, more than one workgroup of the upload, and a table
# of several hundred kilobytes
@pytest.mark.parametrize("views,distinct", [(1, 1), (20, 20), (129, 129), (1500, 1500), (600, 2)])
def test_tables_of_strided_views(pkg, gpu, views, distinct):
    """`distinct` geometries in turn: runs of equal neighbours share a record, others do not."""
    import torch
    parent = torch.randint(0, 256, (views, 6, 4, 2048), dtype=torch.uint8, device=gpu)
    picked = []
    for i in range(views):
        j = i % distinct if distinct > 2 else (i // 7) % 2      # in turn, or in runs of seven
        picked.append(parent[i, :, j % 3, :1 + (j * 37) % 2048] if distinct > 2 else parent[i, :, j, :1400 + 300 * j])
    _round_trip(pkg, gpu, picked, 16, torch)
