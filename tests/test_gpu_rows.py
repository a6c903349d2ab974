"""Views with short rows of 16 bytes and more: row lengths around 16-byte pieces, 64-byte units and what a
wavefront holds, from every kind of start, with row counts around a tile, in one to three strided dimensions.
Packed bytes against torch's compact copies, rows scattered back into poisoned twins of their storages."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu

LENGTHS = [16, 17, 31, 47, 63, 64, 65, 79, 96, 127, 128, 129, 250, 256, 500, 511, 512, 513, 767, 1000, 1023, 1024, 1025, 1279]


def bytes_of(gpu, n, seed):
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    return torch.randint(0, 256, (n,), dtype=torch.uint8, device=gpu, generator=g)


def round_trip(pkg, gpu, n, views_of, align, shift, move=0):
    """`move`: the plans are made for the views and moved by that many bytes before they run."""
    store = bytes_of(gpu, n + move, n)
    twin, want = torch.full_like(store, 0xA5), torch.full_like(store, 0xA5)
    made, views, wants = views_of(store[:n]), views_of(store[move:]), views_of(want[move:])
    for w, v in zip(wants, views):
        w.copy_(v)
    send = pkg.BundlePlan.create(made, align=align)
    recv = pkg.BundlePlan.from_header_bound(send.header, views_of(twin[:n]))
    assert {s["mode"] for s in send.segments()} == {2}
    size = send.payload_bytes
    payload = torch.full((shift + size + 64,), 0xCD, dtype=torch.uint8, device=gpu)
    for plan, unpack in ((send, 0), (recv, 1)):
        job = (pkg._capi.Job * 1)()
        job[0].plan, job[0].payload, job[0].payload_bytes = plan._h, payload.data_ptr() + shift, size
        job[0].unpack, job[0].tensor_delta = unpack, move
        pkg._capi.check(pkg._capi.load().axr_submit(job, 1, C.c_void_p()))
    torch.cuda.synchronize()
    for v, off, nbytes in zip(views, *send.layout()):
        assert torch.equal(payload[shift + off:shift + off + nbytes], v.contiguous().reshape(-1))
    assert (payload[:shift] == 0xCD).all() and (payload[shift + size:] == 0xCD).all()
    assert torch.equal(twin, want)
    send.close()
    recv.close()


@pytest.mark.parametrize("length", LENGTHS)
@pytest.mark.parametrize("gap,lead", [(1, 0), (3, 1), (64, 0), (64, 7), (16, 16), (33, 2)])
@pytest.mark.parametrize("align,shift", [(1, 0), (256, 0), (1, 5)])
def test_short_rows(pkg, gpu, length, gap, lead, align, shift):
    pitch = length + gap if gap < 64 else -(-length // 64) * 64 + (64 if length % 64 == 0 else 0)
    counts = [1, 2, 5, 31, 32, 33, 257]      # tiles hold 2 to 64 rows

    def views(s):
        out, at = [], lead
        for c in counts:
            out.append(s[at:at + (c + 1) * pitch].view(c + 1, pitch)[1:, :length] if c > 1 else
                       s[at:at + 3 * pitch].view(3, pitch)[::2, :length])
            at += (c + 2) * pitch
        return out

    round_trip(pkg, gpu, lead + sum((c + 2) * pitch for c in counts), views, align, shift)


@pytest.mark.parametrize("length", [16, 50, 64, 130, 999])
@pytest.mark.parametrize("tunables", [{}, {"max_waves": 3}, {"nontemporal": 3, "threads": 64}, {"nontemporal": 0, "tile_rows": 16},
                                      {"gather_run_bytes": 4096}], ids=str)
def test_rows_in_several_dimensions(pkg, gpu, length, tunables):
    defaults = {"max_waves": 1 << 20, "nontemporal": -1, "threads": 0, "tile_rows": 0, "gather_run_bytes": 1280}
    pitch = length + 5

    def views(s):
        a = s[:7 * 9 * 11 * pitch].view(7, 9, 11, pitch)
        return [a[:, :, :, 2:2 + length], a[1::2, 2:8, ::3, :length], a[:, 4, 1:9, 1:1 + length], a[::6, 1:, :, 5:]]

    pkg.tune(**tunables)
    try:
        round_trip(pkg, gpu, 7 * 9 * 11 * pitch, views, 1, 0)
        round_trip(pkg, gpu, 7 * 9 * 11 * pitch, views, 64, 1)
    finally:
        pkg.tune(**{k: defaults[k] for k in tunables})


@pytest.mark.parametrize("move", [1, 16, 63, 64])
@pytest.mark.parametrize("length", [48, 64, 100, 512, 1278])
def test_moved_plans(pkg, gpu, length, move):
    """Plans for rows that start on units, run where they do not: the slots they have no longer fit every start."""
    pitch = -(-length // 64) * 64 + 64
    round_trip(pkg, gpu, 100 * pitch, lambda s: [s.view(-1)[:100 * pitch].view(100, pitch)[:, :length]], 256, 0, move)


def test_long_rows_up_to_the_limit(pkg, gpu):
    """With the limit for short rows raised, rows are moved whole up to 1984 bytes."""
    pkg.tune(gather_run_bytes=4096)
    try:
        for length in (1280, 1536, 1983, 1984):
            round_trip(pkg, gpu, 100 * 2100 + 1, lambda s: [s[1:100 * 2100 + 1].view(100, 2100)[:, :length]], 1, 0)
    finally:
        pkg.tune(gather_run_bytes=1280)


@pytest.mark.parametrize("length,pitch,mib", [(130, 131, 25), (200, 232, 25), (256, 292, 25), (72, 73, 2), (72, 73, 130), (24, 64, 66),
                                              (40, 41, 66), (384, 385, 257)])
def test_rows_of_larger_bundles(pkg, gpu, length, pitch, mib):
    """Payloads around the sizes from which rows are given other slots, on one side or on both."""
    rows = mib * (1 << 20) // length + 1
    round_trip(pkg, gpu, rows * pitch, lambda s: [s[:rows * pitch].view(rows, pitch)[:, :length]], 256, 0)
