"""Keys of a chunk's geometry: the C helper tells apart exactly what the Python loop tells apart."""
import itertools

import pytest

torch = pytest.importorskip("torch")


def arrays(pkg):
    from execution_ucx_amd.dlpack import TensorArray, TensorView
    big = torch.zeros(4, 64, 48, dtype=torch.float32)
    lists = [[big[0], big[1]], [big[1], big[2]], [big[0], big[2]], [big[0, :, :40], big[1, :, :40]], [big[2, :, :40], big[3, :, :40]],
             [big[0].t(), big[1]], [big[0].view(torch.int32), big[1]], [big[0], big[1], big[2]], [big[0].view(-1), big[1]],
             [big[0].reshape(64, 1, 48), big[1]], [big[0, 0, 0], big[0, 0, 1]], [big[1, 0, 0], big[1, 0, 1]]]
    out = [TensorArray.from_objects(x) for x in lists] + [TensorArray([])]
    for device, strides, offset, lanes in itertools.product((1, 10), (None, (8, 1)), (0, 16), (1, 2)):
        for at in (1 << 20, 1 << 21):
            out.append(TensorArray([TensorView(at, device, 0, (2, 32, lanes), (4, 8), strides, offset),
                                    TensorView(at + 4096, device, 0, (2, 32, 1), (), None)]))
    return out


def test_native_keys_agree_with_python(pkg, monkeypatch):
    from execution_ucx_amd import pipeline
    if pipeline._native() is None:
        pytest.skip("the C helper has not been built")
    made = arrays(pkg)
    native = [pipeline._geometry(a) for a in made]
    monkeypatch.setattr(pipeline, "_native", lambda: None)
    plain = [pipeline._geometry(a) for a in made]
    assert [base for base, _ in native] == [base for base, _ in plain]
    for (_, k), (_, p) in zip(native, plain):
        assert [k == other for _, other in native] == [p == other for _, other in plain]
