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
    bases = [v._base if v._base is not None else v for v in views]
    twins = {b.data_ptr(): torch.zeros_like(b) for b in {id(b): b for b in bases}.values()}
    outs = [twins[b.data_ptr()].as_strided(v.shape, v.stride(), v.storage_offset()) for b, v in zip(bases, views)]
    recv = pkg.BundlePlan.from_header_bound(plan.header, outs)
    recv.unpack(payload.data_ptr(), n)
    torch.cuda.synchronize()
    for v, o, off, size in zip(views, outs, offs, sizes):
        want = v.contiguous().reshape(-1).view(torch.uint8)
        assert torch.equal(payload[off:off + size], want)
        assert torch.equal(o.contiguous().reshape(-1).view(torch.uint8), want)
    for o in outs:   # nothing beside the views is written
        o.zero_()
    assert not any(t.any() for t in twins.values())
    recv.close()
    plan.close()


# one tensor, the last table vector partly used, more than one workgroup of the upload, a table of
# several hundred kilobytes, and one of more than a megabyte, which the copy engine brings up
@pytest.mark.parametrize("views,distinct", [(1, 1), (20, 20), (129, 129), (1500, 1500), (600, 2), (6000, 6000)])
def test_tables_of_strided_views(pkg, gpu, views, distinct):
    """`distinct` geometries in turn: runs of equal neighbours share a record, others do not."""
    import torch
    parent = torch.randint(0, 256, (views, 6, 4, 2048), dtype=torch.uint8, device=gpu)
    picked = []
    for i in range(views):
        j = i % distinct if distinct > 2 else (i // 7) % 2      # in turn, or in runs of seven
        picked.append(parent[i, :, j % 3, :1 + (j * 37) % 2048] if distinct > 2 else parent[i, :, j, :1400 + 300 * j])
    _round_trip(pkg, gpu, picked, 16, torch)


# one group, groups full by members (1 byte each), by slots (512 bytes; alignment gaps as zero slots),
# both kinds in turn, gaps too long for a group on the way (1024), the last tensor too long for one,
# an empty tensor among them, and enough for several workgroups of the kernel that lays groups out
@pytest.mark.parametrize("align", [1, 16, 256, 1024])
@pytest.mark.parametrize("slots", [128, 64])
@pytest.mark.parametrize("sizes", [
    [5], [1] * 16, [1] * 17, [512] * 40, [1, 512] * 50, list(range(1, 513)), [16 + k % 3 for k in range(700)],
    [8, 500, 33] * 30 + [513], [8, 0, 33] * 30, [1 + 7 * k % 512 for k in range(9001)]], ids=lambda s: f"{len(s)}x{s[-1]}")
def test_group_blocks_laid_out_by_the_device(pkg, gpu, sizes, slots, align):
    """Short contiguous tensors, blocks from the device ("device_tables") and from the host: the
    packed bytes and gaps, the scattered tensors, and the plan after its tables were asked for."""
    import torch
    gaps = [(3 * k) % 31 for k in range(len(sizes))]
    total = sum(sizes) + sum(gaps)
    arena = torch.randint(0, 256, (total,), dtype=torch.uint8, device=gpu)

    def carve(store):
        out, at = [], 0
        for n, gap in zip(sizes, gaps):
            out.append(store[at + gap:at + gap + n])
            at += gap + n
        return out

    views = carve(arena)
    want_twin = torch.full_like(arena, 0xEE)
    for o, v in zip(carve(want_twin), views):
        o.copy_(v)
    try:
        pkg.tune(group_slots=slots)
        for device_tables in (1, 0):
            pkg.tune(device_tables=device_tables)
            plan = pkg.BundlePlan.create(views, align=align)
            n = plan.payload_bytes
            want = torch.zeros(n, dtype=torch.uint8, device=gpu)
            for v, off, size in zip(views, *plan.layout()):
                want[off:off + size] = v
            for shift in (0, 3):
                payload = torch.full((n + shift + 64,), 0xCD, dtype=torch.uint8, device=gpu)
                plan.pack(payload.data_ptr() + shift, n)
                twin = torch.full_like(arena, 0xEE)
                recv = pkg.BundlePlan.from_header_bound(plan.header, carve(twin))
                recv.unpack(payload.data_ptr() + shift, n)
                assert torch.equal(payload[shift:shift + n], want), (device_tables, shift)
                assert (payload[:shift] == 0xCD).all() and (payload[shift + n:] == 0xCD).all()
                assert torch.equal(twin, want_twin), (device_tables, shift)
                recv.close()
                assert plan.launch_info()["tiles"] > 0     # host tables from here on
            plan.close()
    finally:
        pkg.tune(group_slots=128, device_tables=512)


# tables from the host (strided views), from compact records, and group blocks: all three go up on
# the default stream with the plan's first launch
@pytest.mark.parametrize("kind", ["views", "records", "groups"])
def test_a_launch_elsewhere_waits_for_the_upload_only(pkg, gpu, kind):
    """A plan whose tables went up on the default stream, launched on a stream of its own while the
    default stream is busy with something else: it is done long before that."""
    import ctypes as C

    import torch
    lib, capi = pkg._capi.load(), pkg._capi
    parent = torch.randint(0, 256, (700, 9, 2048), dtype=torch.uint8, device=gpu)
    if kind == "views":
        tensors = [parent[i, 1:, :1400 + i % 7] for i in range(200)]
    else:
        tensors = [parent[i, 0, :(2000 if kind == "records" else 100) + i % 48] for i in range(700)]
    plan = pkg.BundlePlan.create(tensors, align=16)
    n = plan.payload_bytes
    payload = torch.zeros(n, dtype=torch.uint8, device=gpu)
    stream = C.c_void_p()
    capi.check(lib.axr_stream_create(C.byref(stream)))
    plan.pack(payload.data_ptr(), n)
    plan.pack(payload.data_ptr(), n)      # (tables that rode in kernel arguments go up now)
    want = payload.clone()
    payload.zero_()
    torch.cuda.synchronize()
    torch.cuda._sleep(800_000_000)        # 0.4 s or so that the plan has nothing to do with
    busy = torch.cuda.Event()
    busy.record()
    plan.pack(payload.data_ptr(), n, stream.value, order=False)
    capi.check(lib.axr_stream_synchronize(stream.value))
    still_busy = not busy.query()
    torch.cuda.synchronize()
    assert torch.equal(payload, want)
    assert still_busy
    plan.close()
    capi.check(lib.axr_stream_destroy(stream.value))


def test_gaps_too_long_for_groups_take_no_room_for_them(pkg, gpu):
    """Short tensors whose alignment gaps fit no group: the table block stays at what the general path
    needs (a record of 32 bytes and an index entry each), it is not sized for groups of gaps."""
    import torch
    n = 60000
    arena = torch.randint(0, 256, (16 * n,), dtype=torch.uint8, device=gpu)
    views = [arena[16 * i:16 * i + 8] for i in range(n)]
    plan = pkg.BundlePlan.create(views, align=4096)
    payload = torch.full((plan.payload_bytes,), 0xCD, dtype=torch.uint8, device=gpu)
    first = pkg.BundlePlan.create(views[:1], align=4096)    # whatever a first launch takes
    first.pack(payload.data_ptr(), first.payload_bytes)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    plan.pack(payload.data_ptr(), plan.payload_bytes)
    torch.cuda.synchronize()
    taken = before - torch.cuda.mem_get_info()[0]
    # 40 bytes per tensor, in a block of a power of two, in pages of 2 MiB
    assert taken <= 2 * 40 * n + (4 << 20), taken
    want = torch.zeros_like(payload)
    want.as_strided((n, 8), (4096, 1)).copy_(arena.view(n, 16)[:, :8])
    assert torch.equal(payload, want)
    plan.close()
