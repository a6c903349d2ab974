"""First launches that read their tables in pinned memory: the same bytes as later ones, from blocks new and used."""
import ctypes as C
import random

import pytest

torch = pytest.importorskip("torch")

KIB = 1 << 10


def tensors(kind, count, gpu, seed):
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    rng = random.Random(seed)

    def raw(n):
        return torch.randint(0, 256, (n,), dtype=torch.uint8, device=gpu, generator=g)

    if kind == "mixed":
        return [raw(rng.choice([1, 40, 300, 700, 2049, 5000, 40 * KIB, 65537])) for _ in range(count)]
    if kind == "short":               # groups of short tensors next to others
        return [raw(rng.randint(1, 512) if i % 9 else 3000) for i in range(count)]
    store = raw(8 * count * 4 * KIB).view(8, count, 4 * KIB)
    if kind == "blocks":              # views of one geometry
        return [store[:, i, :2 * KIB] for i in range(count)]
    return [store[:1 + i % 8, i, :1300 + i] for i in range(count)]      # views that all differ


def expected(src, plan, gpu):
    want = torch.zeros(plan.payload_bytes, dtype=torch.uint8, device=gpu)
    for t, at in zip(src, plan.layout()[0]):
        want[at:at + t.numel()] = t.reshape(-1)
    return want


@pytest.mark.gpu
@pytest.mark.parametrize("align", [1, 256])
@pytest.mark.parametrize("kind, count", [("mixed", 112), ("mixed", 319), ("mixed", 320), ("mixed", 383), ("mixed", 384), ("short", 300), ("blocks", 110),
                                         ("blocks", 400), ("views", 120)])
def test_first_second_and_rebound_launches(pkg, gpu, kind, count, align):
    src = tensors(kind, count, gpu, 3)
    dst, other = [torch.zeros_like(t) for t in src], [torch.zeros_like(t) for t in src]
    send = pkg.BundlePlan.create(src, align=align)
    recv = pkg.BundlePlan.from_header(send.header).bind(dst)
    want = expected(src, send, gpu)
    n = send.payload_bytes
    lib, side = pkg._capi.load(), C.c_void_p()
    pkg._capi.check(lib.axr_stream_create(C.byref(side)))
    torch.cuda.synchronize()
    for stream in (None, None, side.value):
        payload = torch.full_like(want, 0x5a)
        for t in dst:
            t.zero_()
        torch.cuda.synchronize()
        send.pack(payload.data_ptr(), n, stream)
        recv.unpack(payload.data_ptr(), n, stream)
        torch.cuda.synchronize()
        assert torch.equal(payload, want)
        assert all(torch.equal(a, b) for a, b in zip(dst, src))
    recv.bind(other)                  # new tables, in the block that earlier launches have read
    recv.unpack(want.data_ptr(), n)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(other, src))
    send.close()
    recv.close()
    pkg._capi.check(lib.axr_stream_destroy(side))


@pytest.mark.gpu
def test_used_blocks_hold_no_tables_of_earlier_plans(pkg, gpu):
    """Fresh plans one after the other take over each other's blocks: every launch sees its own tables."""
    pool = tensors("mixed", 500, gpu, 4)
    rng = random.Random(4)
    for _ in range(100):
        src = rng.sample(pool, rng.randint(105, 319))
        send = pkg.BundlePlan.create(src, align=64)
        payload = torch.full((send.payload_bytes,), 0x5a, dtype=torch.uint8, device=gpu)
        send.pack(payload.data_ptr(), payload.numel())
        want = expected(src, send, gpu)
        send.close()
        assert torch.equal(payload, want)
