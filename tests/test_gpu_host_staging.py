"""Host (kDLCPU) tensors on their way through the staging blocks: in pieces with flags behind them, or whole."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KIB, MIB = 1 << 10, 1 << 20


def sizes_of(total, parts, rng):
    cuts = np.sort(rng.choice(np.arange(1, total), size=parts - 1, replace=False)) if parts > 1 else []
    return np.diff(np.concatenate([[0], cuts, [total]]).astype(np.int64))


# edges of a flag's piece (16 KiB), a thread's unit (64 KiB), the first transfer (256 KiB), helpers (2 MiB), the
# copy engine (2 MiB) and a block (8 MiB: two, then three of them)
@pytest.mark.parametrize("total,parts", [
    (1, 1), (15, 2), (16 * KIB - 1, 1), (16 * KIB + 1, 7), (64 * KIB, 3), (64 * KIB + 5, 1), (256 * KIB - 3, 9),
    (256 * KIB + 17, 1), (2 * MIB - 4096, 40), (2 * MIB + 3, 5), (5 * MIB + 1, 300), (8 * MIB, 1), (8 * MIB + 1, 2),
    (15 * MIB + 11, 6), (17 * MIB + 3, 3)])
@pytest.mark.parametrize("align", [1, 256])
def test_staged_bytes(pkg, orc, gpu, total, parts, align):
    import torch
    rng = np.random.default_rng(total * 7 + parts)
    src = [rng.integers(0, 256, size=n, dtype=np.uint8) for n in sizes_of(total, parts, rng)]
    stream = torch.cuda.Stream()
    plan = pkg.BundlePlan.create(src, align=align)
    n = plan.payload_bytes
    out = [np.zeros_like(a) for a in src]
    recv = pkg.BundlePlan.from_header(plan.header).bind(out)
    expect = orc.pack(src, align)
    for shift in (0, 5):       # a payload that starts anywhere
        buf = torch.full((n + 64,), 0x5a, dtype=torch.uint8, device=gpu)
        torch.cuda.synchronize()
        plan.pack(buf.data_ptr() + shift, n, stream.cuda_stream)
        for o in out:
            o[...] = 0
        recv.unpack(buf.data_ptr() + shift, n, stream.cuda_stream)    # returns with the bytes in place
        assert all(np.array_equal(a, b) for a, b in zip(src, out)), shift
        stream.synchronize()
        host = buf.cpu().numpy()
        assert np.array_equal(host[shift:shift + n], expect), shift
        assert (host[:shift] == 0x5a).all() and (host[shift + n:] == 0x5a).all(), shift
    plan.close()
    recv.close()


@pytest.mark.parametrize("total", [1000, 300 * KIB, 3 * MIB])
def test_payload_in_pinned_host_memory(pkg, orc, gpu, total):
    """A payload that is no device memory moves whole."""
    import torch
    rng = np.random.default_rng(total)
    src = [rng.integers(0, 256, size=n, dtype=np.uint8) for n in sizes_of(total, 3, rng)]
    plan = pkg.BundlePlan.create(src, align=64)
    n = plan.payload_bytes
    payload = torch.zeros(n, dtype=torch.uint8, pin_memory=True)
    plan.pack(payload.data_ptr(), n)
    torch.cuda.synchronize()
    assert np.array_equal(payload.numpy(), orc.pack(src, 64))
    out = [np.zeros_like(a) for a in src]
    recv = pkg.BundlePlan.from_header(plan.header).bind(out)
    recv.unpack(payload.data_ptr(), n)
    assert all(np.array_equal(a, b) for a, b in zip(src, out))
    plan.close()
    recv.close()


def test_behind_work_longer_than_the_flags_are_polled(pkg, gpu):
    import torch
    rng = np.random.default_rng(3)
    src = [rng.integers(0, 256, size=3 * MIB, dtype=np.uint8)]
    out = [np.zeros_like(src[0])]
    plan = pkg.BundlePlan.create(src)
    n = plan.payload_bytes
    recv = pkg.BundlePlan.from_header(plan.header).bind(out)
    buf = torch.zeros(n, dtype=torch.uint8, device=gpu)
    work = torch.zeros(1 << 28, dtype=torch.float32, device=gpu)
    plan.pack(buf.data_ptr(), n)
    for _ in range(20):
        work += 1.0     # some milliseconds on the same stream
    recv.unpack(buf.data_ptr(), n)
    assert np.array_equal(src[0], out[0])
    plan.close()
    recv.close()


def test_later_work_on_the_stream_is_not_waited_for(pkg, gpu):
    """An unpack that waits behind other work returns with its bytes while what another thread has put on the same
    stream in the meantime is still running.  (Put there in the time in which flags are polled, which a thread may miss:
    one of a few attempts has to show it.)"""
    import threading
    import time
    import torch
    rng = np.random.default_rng(4)
    src = [rng.integers(0, 256, size=900000, dtype=np.uint8)]
    out = [np.zeros_like(src[0])]
    plan = pkg.BundlePlan.create(src)
    n = plan.payload_bytes
    recv = pkg.BundlePlan.from_header(plan.header).bind(out)
    buf = torch.zeros(n, dtype=torch.uint8, device=gpu)
    plan.pack(buf.data_ptr(), n)
    recv.unpack(buf.data_ptr(), n)      # (its buffers are there from now on)
    work = torch.zeros(1 << 28, dtype=torch.float32, device=gpu)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        torch.cuda._sleep(1)
    for _ in range(4):
        out[0][...] = 0
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            for _ in range(30):
                work += 1.0      # some 10 ms
        started = threading.Event()

        def unpack():
            started.set()
            recv.unpack(buf.data_ptr(), n, stream.cuda_stream, False)
        moved = threading.Thread(target=unpack)
        moved.start()
        started.wait()
        now = time.perf_counter()
        while time.perf_counter() < now + 5e-5:
            time.sleep(0)
        with torch.cuda.stream(stream):
            torch.cuda._sleep(1 << 27)      # some 50 ms
        moved.join()
        back = time.perf_counter()
        assert np.array_equal(src[0], out[0])
        torch.cuda.synchronize()
        not_waited_for = time.perf_counter() - back > back - now
        if not_waited_for:
            break
    assert not_waited_for
    plan.close()
    recv.close()
