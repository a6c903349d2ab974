"""First launches of bundles whose tables travel in the kernel arguments beyond the small ones."""
import pytest

torch = pytest.importorskip("torch")

KIB, MIB = 1 << 10, 1 << 20


def sizes(name):
    return {
        "one": [40 * MIB],
        "layer": [9 * MIB + 6, 9 * MIB, 25 * MIB - 2, 25 * MIB, 8192, 8192],
        "tails": [3 * MIB + 1, 1, 2047, 2 * MIB + 2049, 1023, 5 * MIB - 15],
        # a long tensor among more short ones than a wavefront should walk: wide blocks are out of the question
        "crowd": [20 * MIB] + [600] * 100 + [4 * MIB],
        "crowd_short_index": [6 * MIB] + [600] * 60,
        # an index that only fits in wide blocks (1 KiB tiles): two segments, and one tensor more than fits
        "long": [150 * MIB, 130 * MIB + 77],
        "many": [5 * MIB + 16 * i for i in range(105)],
        "too_many": [3 * MIB] * 120,
    }[name]


@pytest.mark.gpu
@pytest.mark.parametrize("streaming", [False, True])
@pytest.mark.parametrize("align", [1, 256])
@pytest.mark.parametrize("name", ["one", "layer", "tails", "crowd", "crowd_short_index", "long", "many", "too_many"])
def test_first_and_later_launches_move_the_same_bytes(pkg, gpu, name, align, streaming):
    g = torch.Generator(device=gpu)
    g.manual_seed(5)
    src = [torch.randint(0, 256, (n,), dtype=torch.uint8, device=gpu, generator=g) for n in sizes(name)]
    dst = [torch.zeros_like(t) for t in src]
    pkg.tune(inline_tables=64, group_bytes=0, payload_cache_bytes=MIB if streaming else 256 * MIB)
    try:
        send = pkg.BundlePlan.create(src, align=align)
        recv = pkg.BundlePlan.from_header(send.header).bind(dst)
        want = torch.zeros(send.payload_bytes, dtype=torch.uint8, device=gpu)
        for t, at in zip(src, send.layout()[0]):
            want[at:at + t.numel()] = t
        for launch in range(2):      # from the kernel arguments where they fit, then uploaded
            payload = torch.full_like(want, 0x5a)
            send.pack(payload.data_ptr(), payload.numel())
            in_arguments = launch == 0 and name not in ("crowd", "too_many")
            assert send.launch_info()["last_launch"] & 15 == (1 if in_arguments else 3)
            assert torch.equal(payload, want)
            for t in dst:
                t.zero_()
            recv.unpack(payload.data_ptr(), payload.numel())
            assert all(torch.equal(a, b) for a, b in zip(dst, src))
        send.close()
        recv.close()
    finally:
        pkg.tune(inline_tables=16384, group_bytes=512, payload_cache_bytes=256 * MIB)


@pytest.mark.gpu
def test_large_bundles_are_captured_after_prepare_only(pkg, gpu):
    src = [torch.randint(0, 256, (40 * MIB,), dtype=torch.uint8, device=gpu)]
    with pkg.BundlePlan.create(src, align=256) as plan:
        payload = torch.zeros(plan.payload_bytes, dtype=torch.uint8, device=gpu)
        torch.cuda.synchronize()
        stream = torch.cuda.Stream()
        with pytest.raises(Exception, match="prepare"):
            with torch.cuda.graph(torch.cuda.CUDAGraph(), stream=stream):
                plan.pack(payload.data_ptr(), payload.numel(), stream)
        torch.cuda.synchronize()
        plan.pack(payload.data_ptr(), payload.numel())
        assert torch.equal(payload, src[0])
