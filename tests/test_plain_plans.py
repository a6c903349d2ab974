"""Plans made straight from lists of torch tensors against plans made of their DLPack capsules."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

DTYPES = [torch.uint8, torch.int8, torch.int16, torch.int32, torch.int64, torch.float16, torch.bfloat16, torch.float32,
          torch.float64, torch.bool, torch.complex64, torch.complex128, torch.uint16, torch.uint32, torch.uint64,
          torch.float8_e4m3fn, torch.float8_e5m2]


def views(device):
    """Twice every type (the second one is read without the converter), in one storage and in several, with
    size-1, size-0, stepped and permuted dimensions, 130 and more tensors (lots of 64) among them."""
    out = []
    for dt in DTYPES:
        try:
            torch.utils.dlpack.to_dlpack(torch.zeros(4, dtype=dt, device=device))
        except (BufferError, RuntimeError, TypeError):
            continue
        for _ in range(2):
            base = torch.zeros(4 * 6 * 8, dtype=dt, device=device)
            cube = base.view(4, 6, 8)
            out += [base, cube, cube[:, ::2, 1:], cube.permute(2, 0, 1), cube[1], base.view(4, 1, 48)[:, :, ::3],
                    base[:0], cube[:, :0], base[3:4].reshape(()), base.view(192, 1).t(), base[5:77]]
    return out


def records(plan):
    return plan.header, plan.segments()


def check(pkg, tensors):
    from execution_ucx_amd import bundle, dlpack
    made = dlpack.plain_plan(pkg._capi.load(), tensors, 64)
    assert made is not None and all(a is b for a, b in zip(made[1], tensors))
    pkg._capi.check(pkg._capi.load().axr_plan_free(made[0]))
    with pkg.BundlePlan.create(tensors, align=64) as plan, \
            pkg.BundlePlan.create(dlpack.TensorArray(dlpack.extract_many(tensors)), align=64) as want:
        assert records(plan) == records(want)
        header = plan.header
    with bundle._bind_header(header, tensors, None) as plan, \
            pkg.BundlePlan.from_header(header).bind(dlpack.TensorArray(dlpack.extract_many(tensors))) as want:
        assert plan._header is not None and records(plan) == records(want)
        plan.bind(list(tensors))
        assert plan.header == header


@pytest.mark.parametrize("count", [0, 1, 63, 64, 65, None])
def test_host_tensors(pkg, count):
    check(pkg, views("cpu")[:count])


@pytest.mark.gpu
@pytest.mark.parametrize("count", [0, 1, 63, 64, 65, None])
def test_device_tensors(pkg, gpu, count):
    check(pkg, views(gpu)[:count])


@pytest.mark.gpu
def test_device_and_host_tensors_alternate(pkg, gpu):
    check(pkg, [t for pair in zip(views(gpu), views("cpu")) for t in pair])


def test_what_is_refused_is_refused_as_before(pkg):
    from execution_ucx_amd import bundle, dlpack
    lib = pkg._capi.load()
    good = torch.zeros(3, 5)
    for other in (torch.zeros(3, requires_grad=True), np.zeros(3), object(), torch.zeros(3, device="meta"),
                  torch.zeros(3, dtype=torch.complex64).conj(), torch.zeros(3, 3).to_sparse()):
        assert dlpack.plain_plan(lib, [good, other], 1) is None
    assert dlpack.plain_plan(lib, iter([good]), 1) is None
    with pytest.raises(BufferError, match="gradient"):
        pkg.BundlePlan.create([good, torch.zeros(3, requires_grad=True)])
    with pytest.raises(Exception, match="power of two"):
        pkg.BundlePlan.create([good], align=3)
    with pkg.BundlePlan.create([good, np.zeros(7, np.float32)], align=1) as plan:
        header = plan.header
    for out, why in (([good], "count"), ([good, torch.zeros(8)], "tensor 1"), ([good, torch.zeros(7, dtype=torch.float16)], "tensor 1")):
        with pytest.raises(Exception, match=why):
            bundle._bind_header(header, out, None)
    with pytest.raises(Exception, match="magic"):      # reported ahead of the destinations
        bundle._bind_header(b"x" * len(header), [good], None)
    with pytest.raises(Exception, match="truncated|trailing|bad tensor record"):
        bundle._bind_header(header[:-8], [good, torch.zeros(7)], None)


def test_null_sources_are_refused(pkg):
    """What the siblings that take an array refuse: no result, no source, a source that cannot describe."""
    import ctypes as C
    lib = pkg._capi.load()

    class Source(C.Structure):
        _fields_ = [("count", C.c_size_t), ("describe", C.c_void_p)]

    create, bind = lib.axr_plan_create_from, lib.axr_plan_bind_from
    create.argtypes, create.restype = [C.c_void_p, C.c_uint32, C.c_void_p], C.c_int
    bind.argtypes, bind.restype = [C.c_void_p, C.c_size_t, C.c_void_p, C.c_void_p], C.c_int
    with pkg.BundlePlan.create([torch.zeros(3)], align=1) as plan:
        header = plan.header
    h, mute, none = C.c_void_p(), Source(1, None), Source(0, None)
    invalid = -1
    assert create(C.byref(none), 1, None) == invalid and bind(header, len(header), C.byref(none), None) == invalid
    for source in (None, C.byref(mute)):
        assert create(source, 1, C.byref(h)) == invalid and not h.value
        assert bind(header, len(header), source, C.byref(h)) == invalid and not h.value
    assert bind(None, 0, C.byref(none), C.byref(h)) == invalid
    assert create(C.byref(none), 1, C.byref(h)) == 0 and h.value      # no tensors: nothing to describe
    pkg._capi.check(lib.axr_plan_free(h))


def test_lists_with_other_arrays_are_not_tried(pkg, monkeypatch):
    """An array in front, in the middle or at the end of many tensors, or in front of a few: no attempt that reads the
    tensors for nothing."""
    from execution_ucx_amd import dlpack

    class Native:
        def __getattr__(self, name):
            raise AssertionError(f"{name} was asked")

    good, other = torch.zeros(3), np.zeros(3, np.float32)
    monkeypatch.setattr(dlpack, "_native_torch", lambda: Native())
    for count, at in ((512, 0), (512, 256), (512, 511), (9, 0)):
        objs = [good] * count
        objs[at] = other
        assert dlpack.plain_plan(pkg._capi.load(), objs, 1) is None
        assert dlpack.plain_plan(pkg._capi.load(), tuple(objs), header=b"") is None
    with pytest.raises(AssertionError, match="plan_create"):
        dlpack.plain_plan(pkg._capi.load(), [good] * 9, 1)
