"""Streamed transfers whose chunks run in line on one lane's stream and slot, next to chunks that
take their lanes in turn."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes,streams", [(1, 1), (2, 1), (2, 2), (3, 2)])
@pytest.mark.parametrize("cache", ["fits", "one byte short", "holds one", "beyond"])
def test_chunks_in_line(pkg, gpu, lanes, streams, cache):
    """Two geometries in turn; `streams` payloads of the larger one just fit the cache, or do not, or
    one and no more does (in line), or not even one does."""
    import torch
    big, small = (4, 257, 300), (3, 5, 300)          # views, rows, columns
    tune = pkg._capi.load().axr_tune_set
    src = torch.randint(0, 256, (12, 4, 257, 400), dtype=torch.uint8, device=gpu)
    dst = torch.zeros_like(src)

    def plans(views, rows, cols):
        send = pkg.BundlePlan.create([v[:rows, :cols] for v in src[0, :views]], align=1)
        return send, pkg.BundlePlan.from_header(send.header).bind([v[:rows, :cols] for v in dst[0, :views]])

    pairs = [plans(*big), plans(*small)]
    largest = pairs[0][0].payload_bytes
    transfer = pkg.StreamedTransfer(largest, streams=streams, lanes=lanes)
    want = torch.zeros_like(src)
    torch.cuda.synchronize()
    try:
        limit = {"fits": streams * largest, "one byte short": streams * largest - 1, "holds one": largest,
                 "beyond": largest - 1}[cache]
        assert tune(b"payload_cache_bytes", limit) == 0
        for k in range(12):
            views, rows, cols = (big, small)[k % 5 == 3]
            send, recv = pairs[k % 5 == 3]
            transfer.submit_plans(send, k * src[0].numel(), recv, k * src[0].numel())
            want[k, :views, :rows, :cols] = src[k, :views, :rows, :cols]
        transfer.finish()
    finally:
        tune(b"payload_cache_bytes", 256 << 20)
    assert torch.equal(dst, want)
    transfer.close()
    for send, recv in pairs:
        send.close()
        recv.close()
