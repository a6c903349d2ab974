"""Streaming payloads whose end is written with ordinary stores: the same bytes on both sides of the border."""
import pytest

torch = pytest.importorskip("torch")

KIB, MIB = 1 << 10, 1 << 20


def tensors(name, gpu, seed):
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)

    def raw(n):
        return torch.randint(0, 256, (n,), dtype=torch.uint8, device=gpu, generator=g)

    if name == "border_inside":       # 7 MiB from the end lie inside the first tensor
        return [raw(9 * MIB + 5), raw(MIB), raw(1), raw(2 * KIB - 1)]
    if name == "border_between":
        return [raw(5 * MIB), raw(7 * MIB)]
    if name == "barely":              # one tile beyond what the cache is taken to hold
        return [raw(8 * MIB + 1)]
    if name == "runs":                # views with long runs, the last tile of each in part
        return [raw(1200 * 5000).view(1200, 5000)[:, :4111], raw(5 * MIB).view(1024, 5120)[:, 7:4103], raw(333)]
    return [raw(4 * MIB), raw(40 * 200 * 1500).view(40, 200, 1500)[:, ::2, :1301].permute(1, 0, 2), raw(77 * KIB)]


@pytest.mark.gpu
@pytest.mark.parametrize("align", [1, 256])
@pytest.mark.parametrize("name", ["border_inside", "border_between", "barely", "runs", "permuted"])
def test_payload_with_a_cached_tail(pkg, gpu, name, align):
    src = tensors(name, gpu, 11)
    dst = [torch.zeros_like(t) for t in src]
    pkg.tune(payload_cache_bytes=8 * MIB, group_bytes=0)      # 7 MiB of the payload stay
    try:
        send = pkg.BundlePlan.create(src, align=align)
        recv = pkg.BundlePlan.from_header(send.header).bind(dst)
        want = torch.zeros(send.payload_bytes, dtype=torch.uint8, device=gpu)
        for t, at in zip(src, send.layout()[0]):
            want[at:at + t.numel()] = t.reshape(-1)
        assert send.payload_bytes > 8 * MIB
        n = send.payload_bytes
        payload = torch.empty_like(want)
        send.prepare()
        recv.prepare()
        for attempt in range(3):
            payload.fill_(0x5a)
            if attempt == 1:          # all of it streams where that is asked for
                job = pkg._capi.Job()
                job.plan, job.payload, job.payload_bytes, job.flags = send._h, payload.data_ptr(), n, pkg._capi.JOB_PAYLOAD_STREAMING
                pkg._capi.check(pkg._capi.load().axr_submit(job, 1, None))
            else:
                send.pack(payload.data_ptr(), n)
            assert torch.equal(payload, want)
        for t in dst:
            t.zero_()
        recv.unpack(payload.data_ptr(), n)
        assert all(torch.equal(a, b) for a, b in zip(dst, src))
        send.close()
        recv.close()
    finally:
        pkg.tune(payload_cache_bytes=256 * MIB, group_bytes=512)
