"""Few planes against the same elements interleaved, in blocks of one round or of two, in bundles of their own and wherever
else such a plan is launched: every byte against the tensors, and the kernel that moved it."""
import pytest

torch = pytest.importorskip("torch")

PLANES, ANY = 5, 6      # kernels that a launch is said to have taken


def views(gpu, item, planes, pixels, images, interleaved, lead):
    dtype = {1: torch.uint8, 2: torch.int16, 4: torch.int32}[item]
    n = images * planes * pixels
    store = torch.randint(-100, 100, (n + lead,), device=gpu).to(dtype)
    if interleaved:
        return store[lead:].view(images, pixels, planes).permute(0, 2, 1)
    return store[lead:].view(images, planes, pixels).permute(0, 2, 1)


class Mover:
    """Plans both ways, with a payload whose end is watched."""

    def __init__(self, pkg, ts, align):
        self.pkg, self.ts = pkg, ts
        self.outs = [torch.zeros_like(t) for t in ts]      # (strides and all)
        assert all(o.stride() == t.stride() for o, t in zip(self.outs, ts))
        self.send = pkg.BundlePlan.create(ts, align=align)
        self.n = self.send.payload_bytes
        self.recv = pkg.BundlePlan.from_header(self.send.header).bind(self.outs)
        self.payload = torch.full((self.n + 64,), 0x5a, dtype=torch.uint8, device=ts[0].device)

    def check(self, kernel):
        for t, at, size in zip(self.ts, *self.send.layout()):
            assert torch.equal(self.payload[at:at + size], t.contiguous().view(-1).view(torch.uint8))
        assert bool((self.payload[self.n:] == 0x5a).all())
        assert all(torch.equal(t, o) for t, o in zip(self.ts, self.outs))
        assert [p.launch_info()["last_launch"] >> 4 & 15 for p in (self.send, self.recv)] == [kernel, kernel]
        self.payload[:self.n] = 0
        for o in self.outs:
            o.zero_()

    def alone(self, kernel, prepared=True):
        if prepared:
            self.send.prepare()
            self.recv.prepare()
        self.send.pack(self.payload.data_ptr(), self.n)
        self.recv.unpack(self.payload.data_ptr(), self.n)
        self.check(kernel)

    def close(self):
        self.send.close()
        self.recv.close()


def together(pkg, movers, kernel):
    """All packs in one launch, and then all unpacks with a pack."""
    for unpack in (0, 1):
        jobs = [(m.recv if unpack else m.send, m.payload, unpack) for m in movers]
        if unpack:
            second = torch.zeros_like(movers[0].payload)
            jobs.append((movers[0].send, second, 0))
        table = (pkg._capi.Job * len(jobs))()
        for j, (p, y, u) in zip(table, jobs):
            j.plan, j.payload, j.payload_bytes, j.unpack = p._h, y.data_ptr(), p.payload_bytes, u
        pkg._capi.check(pkg._capi.load().axr_submit(table, len(jobs), None))
    n = movers[0].n
    assert torch.equal(second[:n], movers[0].payload[:n])
    for m in movers:
        m.check(kernel)


# a round is 1024 bytes of every plane, a block one or two: less than one, one and a bit, just below and above two, more
# of them, ends that are no whole vector
@pytest.mark.gpu
@pytest.mark.parametrize("item,planes", [(1, 3), (1, 4), (2, 3), (1, 2), (2, 4), (4, 3)])
@pytest.mark.parametrize("interleaved", [True, False])
def test_ends_of_blocks(pkg, gpu, item, planes, interleaved):
    r = 1024 // item
    for images, pixels in ((40, r - 1), (40, r), (40, r + 1), (40, r + 17), (40, 2 * r - 1), (40, 2 * r), (40, 2 * r + 3), (40, 3 * r),
                           (40, 3 * r + 1), (40, 4 * r - 7), (1, r + 2), (1, 7 * r + 5), (3, 50176)):
        if item == 4 and pixels == r:      # (whole vectors of 4-byte elements in one round are moved as plain blocks)
            continue
        for align, lead in ((1, 0), (256, 1)):
            m = Mover(pkg, [views(gpu, item, planes, pixels, images, interleaved, lead)], align)
            m.alone(ANY, prepared=False)          # tables in the arguments
            m.alone(PLANES)
            together(pkg, [m], PLANES)
            m.close()


@pytest.mark.gpu
def test_neighbours(pkg, gpu):
    """Planes in blocks of one round and of two, next to each other and to runs, in one bundle and in one launch."""
    three = views(gpu, 1, 3, 5003, 9, True, 1)
    four = views(gpu, 1, 4, 3001, 7, False, 0)
    wide = views(gpu, 4, 3, 2005, 5, True, 0)
    compact = torch.randint(0, 256, (70001,), dtype=torch.uint8, device=gpu)
    large = views(gpu, 1, 3, 50177, 100, True, 0)      # two rounds next to others
    for ts, kernel in (([three, four], PLANES), ([three, wide], PLANES), ([three, compact], ANY), ([compact, four, wide], ANY),
                       ([large, compact], ANY), ([large, three, wide], PLANES)):
        m = Mover(pkg, ts, 256)
        m.alone(kernel)
        m.alone(kernel)
        m.close()
    for lists, kernel in (([[three], [four]], PLANES), ([[wide], [three]], PLANES), ([[three], [wide], [four]], PLANES),
                          ([[three], [compact]], ANY), ([[large], [three, compact]], ANY), ([[large], [three]], PLANES), ([[compact], [four], [three]], ANY), ([[three, compact], [four]], ANY)):
        movers = [Mover(pkg, ts, 256) for ts in lists]
        for _ in range(2):
            together(pkg, movers, kernel)
        for m in movers:
            m.close()


@pytest.mark.gpu
@pytest.mark.parametrize("tunables", [{"threads": 192}, {"threads": 64}, {"max_waves": 37}, {"max_waves": 3}, {"xcd_remap": 1}, {"nontemporal": 3}], ids=str)
def test_launch_shapes(pkg, gpu, tunables):
    usual = {"threads": 0, "max_waves": 1 << 20, "xcd_remap": -1, "nontemporal": -1}
    view = views(gpu, 1, 3, 9001, 30, True, 0)
    try:
        pkg.tune(**tunables)
        m = Mover(pkg, [view], 1)
        m.alone(PLANES)
        m.alone(PLANES)
        m.close()
    finally:
        pkg.tune(**{name: usual[name] for name in tunables})


@pytest.mark.gpu
def test_captured(pkg, gpu):
    m = Mover(pkg, [views(gpu, 2, 3, 4001, 12, True, 1)], 256)
    m.alone(PLANES)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        s = torch.cuda.current_stream().cuda_stream
        m.send.pack(m.payload.data_ptr(), m.n, s, False)
        m.recv.unpack(m.payload.data_ptr(), m.n, s, False)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        m.check(PLANES)
    m.close()
