"""Bundles of one kind of segments (views of a single mode, each moved by a kernel of its own) and of several,
launched alone and several to a launch.  Packed bytes against torch's compact copies, views scattered back
into poisoned twins of their storages, nothing written beside them."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


def storage(gpu, nbytes, seed):
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    return torch.randint(0, 256, (nbytes,), dtype=torch.uint8, device=gpu, generator=g)


# name -> bytes of storage, views of it
FAMILIES = {
    "whole_rows": (90 * 512, lambda s: [s.view(90, 512)[:, :128], s.view(90, 512)[:, 256:448]]),
    "odd_rows": (91 * 259, lambda s: [s.view(91, 259)[:, 1:101], s.view(91, 259)[5:, 102:259]]),
    "many_rows": (40000 * 131, lambda s: [s.view(40000, 131)[:, :100]]),
    "narrow_rows": (1 << 15, lambda s: [s.view(4096, 8)[:, :6]]),
    "blocks": (300 * 196, lambda s: [s.view(300, 196).t(), s.view(300, 196)[1:, 3:190].t()]),
    "odd_blocks": (2051 * 17001 * 2, lambda s: [s.view(torch.int16).view(2051, 17001).t()]),
    "planes": (3 * 70 * 33 * 4, lambda s: [s.view(4, 70, 33, 3).permute(0, 3, 1, 2)]),
    "runs": (70000, lambda s: [s[3:65000], s[65000:65001]]),
    "long_rows": (40 * 5000, lambda s: [s.view(40, 5000)[:, :3001]]),
    "short": (64 * 1000, lambda s: [s[i * 1000 + 7:i * 1000 + 7 + 9 * i + 1] for i in range(50)]),
}
BUNDLES = [[name] for name in FAMILIES if name not in ("short", "many_rows")] + [
    ["short"], ["odd_rows", "runs"], ["planes", "short"], ["blocks", "whole_rows"], ["narrow_rows", "odd_rows", "long_rows"],
    [name for name in FAMILIES if name not in ("odd_blocks", "many_rows")]]


def tunables_now(pkg, names):
    v = C.c_int64()
    out = {}
    for k in names:
        pkg._capi.check(pkg._capi.load().axr_tune_get(k.encode(), C.byref(v)))
        out[k] = v.value
    return out


class Moved:
    """A bundle of some families, its plans in both directions and what they should produce."""

    def __init__(self, pkg, gpu, names, align, seed):
        self.names = names
        self.stores = [storage(gpu, FAMILIES[n][0], seed + i) for i, n in enumerate(names)]
        self.twins = [torch.full_like(s, 0xA5) for s in self.stores]
        self.want = [torch.full_like(s, 0xA5) for s in self.stores]
        views, outs, wants = (self.views(x) for x in (self.stores, self.twins, self.want))
        for w, v in zip(wants, views):
            w.copy_(v)
        self.send = pkg.BundlePlan.create(views, align=align)
        self.recv = pkg.BundlePlan.from_header_bound(self.send.header, outs)
        self.n = self.send.payload_bytes
        self.pieces = [(off, v) for off, v in zip(self.send.layout()[0], views)]
        self.payload = torch.full((self.n + 64,), 0xCD, dtype=torch.uint8, device=gpu)

    def views(self, stores):
        return [v for s, n in zip(stores, self.names) for v in FAMILIES[n][1](s)]

    def check(self):
        torch.cuda.synchronize()
        at = 0
        for off, v in self.pieces:
            assert not self.payload[at:off].any()          # gaps are zero
            flat = v.contiguous().reshape(-1).view(torch.uint8)
            at = off + flat.numel()
            assert torch.equal(self.payload[off:at], flat)
        assert (self.payload[self.n:] == 0xCD).all()
        for t, w, n in zip(self.twins, self.want, self.names):
            assert torch.equal(t, w), n

    def close(self):
        self.send.close()
        self.recv.close()


@pytest.mark.parametrize("names", BUNDLES, ids="+".join)
@pytest.mark.parametrize("tunables", [{}, {"max_waves": 7}, {"tile_rows": 4, "nontemporal": 3}, {"nontemporal": 0}], ids=str)
@pytest.mark.parametrize("align", [1, 256])
def test_kinds(pkg, gpu, names, tunables, align):
    old = tunables_now(pkg, tunables)
    pkg.tune(**tunables)
    try:
        m = Moved(pkg, gpu, names, align, 1)
        for _ in range(2):       # tables in the kernel arguments where they fit, then uploaded ones
            m.payload.fill_(0xCD)
            m.send.pack(m.payload.data_ptr(), m.n)
            for t in m.twins:
                t.fill_(0xA5)
            m.recv.unpack(m.payload.data_ptr(), m.n)
            m.check()
        m.close()
    finally:
        pkg.tune(**old)


@pytest.mark.parametrize("left,right", [("odd_rows", "odd_rows"), ("odd_rows", "short"), ("blocks", "planes"), ("short", "blocks"),
                                        ("runs", "whole_rows"), ("odd_rows", "runs")])
@pytest.mark.parametrize("threads", [64, 128])
@pytest.mark.parametrize("nontemporal", [1, 3])
def test_kinds_in_one_launch(pkg, gpu, left, right, threads, nontemporal):
    capi = pkg._capi
    old = tunables_now(pkg, ("threads", "nontemporal", "submit_interleave"))
    pkg.tune(threads=threads, nontemporal=nontemporal, submit_interleave=2)
    try:
        a, b = Moved(pkg, gpu, [left], 256, 5), Moved(pkg, gpu, [right], 1, 50)
        for unpack in (0, 1):
            jobs = (capi.Job * 2)()
            for j, m in zip(jobs, (a, b)):
                j.plan, j.unpack = (m.recv if unpack else m.send)._h, unpack
                j.payload, j.payload_bytes = m.payload.data_ptr(), m.n
            capi.check(capi.load().axr_submit(jobs, 2, C.c_void_p()))
        a.check()
        b.check()
        a.close()
        b.close()
    finally:
        pkg.tune(**old)


@pytest.mark.parametrize("others", [["runs"], ["blocks"], ["short", "odd_rows"]], ids="+".join)
def test_many_rows_submitted_with_others(pkg, gpu, others):
    """More tiles of short rows than share a launch with another kind: every job's bytes, whichever launch it is in."""
    capi = pkg._capi
    bundles = [Moved(pkg, gpu, [n], 64, 9 + i) for i, n in enumerate(["many_rows"] + others + ["many_rows"])]
    assert sum(s["tiles"] for s in bundles[0].send.segments()) > 2048
    for unpack in (0, 1):
        jobs = (capi.Job * len(bundles))()
        for j, m in zip(jobs, bundles):
            j.plan, j.unpack = (m.recv if unpack else m.send)._h, unpack
            j.payload, j.payload_bytes = m.payload.data_ptr(), m.n
        capi.check(capi.load().axr_submit(jobs, len(bundles), C.c_void_p()))
    for m in bundles:
        m.check()
        m.close()
