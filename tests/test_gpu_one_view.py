"""Bundles of a single view, which consult no tile-block index: every mode, through every way a plan is launched."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")

VIEWS = {
    "elements": lambda s: s[:300 * 7 * 9].view(300, 7, 9)[::2, :, 1:4],
    "rows": lambda s: s[:5000 * 131].view(5000, 131)[:, :100],
    "one_row": lambda s: s[:2 * 131].view(2, 131)[:1, 3:90],
    "blocks": lambda s: s[:700 * 901].view(700, 901).t(),
    "planes": lambda s: s[:3 * 300 * 301].view(300, 301, 3).permute(2, 0, 1),
    "runs": lambda s: s[:40 * 5000].view(40, 5000)[:, :4096],
    "walked": lambda s: s.view(torch.int16)[:1031 * 16001].view(1031, 16001).t(),
    "one_block": lambda s: s[:20 * 33].view(20, 33).t(),
}
JOINT = {"elements": 6, "blocks": 6, "walked": 6, "one_block": 6, "planes": 5, "rows": 2}    # kernels of joint launches: any mode, planes, rows


@pytest.mark.gpu
@pytest.mark.parametrize("kind", VIEWS)
@pytest.mark.parametrize("align", [1, 256])
def test_every_way(pkg, gpu, kind, align):
    lib, capi = pkg._capi.load(), pkg._capi
    store = torch.randint(0, 256, (34 << 20,), dtype=torch.uint8, device=gpu)
    view = VIEWS[kind](store)
    want = view.contiguous().view(-1).view(torch.uint8)
    send = pkg.BundlePlan.create([view], align=align)
    n = send.payload_bytes
    payload = torch.zeros(n + 16, dtype=torch.uint8, device=gpu)

    def packed():
        assert torch.equal(payload[:want.numel()], want) and bool((payload[n:] == 0).all())
        payload.zero_()
    for _ in range(3):             # tables in the arguments or in pinned memory, then uploaded
        send.pack(payload.data_ptr(), n)
        packed()
    fresh = pkg.BundlePlan.create([view], align=align)
    capi.check(lib.axr_pack_noalloc(fresh._h, payload.data_ptr(), n, None))
    torch.cuda.synchronize()
    packed()
    fresh.prepare()
    fresh.pack(payload.data_ptr(), n)
    packed()
    back = torch.zeros_like(store)
    out = VIEWS[kind](back)
    if kind == "walked":           # (workgroups that are handed to the dies in turn share no launch)
        send.close()
        pkg.tune(xcd_remap=0)
    try:
        if kind == "walked":
            send = pkg.BundlePlan.create([view], align=align).prepare()
        recv = pkg.BundlePlan.from_header(send.header).bind([out]).prepare()
    finally:
        pkg.tune(xcd_remap=-1)
    jobs = (capi.Job * 2)()
    second = torch.zeros_like(payload)
    second[:want.numel()] = want
    jobs[0].plan, jobs[0].payload, jobs[0].payload_bytes, jobs[0].unpack = send._h, payload.data_ptr(), n, 0
    jobs[1].plan, jobs[1].payload, jobs[1].payload_bytes, jobs[1].unpack = recv._h, second.data_ptr(), n, 1
    for _ in range(2):
        capi.check(lib.axr_submit(jobs, 2, None))
        packed()
        assert torch.equal(out, view)
        if kind in JOINT:     # in one launch: alone each of them has a kernel of its own
            assert [p.launch_info()["last_launch"] >> 4 & 15 for p in (send, recv)] == [JOINT[kind]] * 2
        back.zero_()
    recv.unpack(second.data_ptr(), n)
    assert torch.equal(out, view)
    assert int((back != 0).sum()) == int((out.contiguous().view(-1).view(torch.uint8) != 0).sum())    # and nothing else written
    for p in (send, fresh, recv):
        p.close()
