"""The group encoder on the matrix cores against the general kernel (which an x
off a 16-byte boundary takes): every field's bytes, over head dims, groups,
widths, input and parameter types, ragged counts, residuals, and special
values."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from polarquant_kv import _lib
from polarquant_kv_cuda.compress_kernel import compress_gpu

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CODE = {torch.float32: _lib.F32, torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}


def _compress(x, R, bits, gs, pdt, resid, rt):
    n, d = x.shape
    pt = torch.float16 if pdt == _lib.F16 else torch.float32
    row = d * {4: 4, 2: 2}.get(bits, 8) // 8
    f = {"radius": torch.full((n,), 7.0, dtype=pt, device=DEV), "codes": torch.full((n, row), 99, dtype=torch.uint8, device=DEV),
         "mins": torch.full((n, d // gs), 7.0, dtype=pt, device=DEV), "scales": torch.full((n, d // gs), 7.0, dtype=pt, device=DEV),
         "resid": torch.full((n, d), 7.0, device=DEV) if resid else None}
    Rt = R.t().contiguous() if rt else None
    _lib.check(_lib.lib().pqkv_group_gpu_compress(x.data_ptr(), CODE[x.dtype], R.data_ptr(), _lib.ptr(Rt), n, d, bits, gs,
                                                  f["radius"].data_ptr(), f["codes"].data_ptr(), f["mins"].data_ptr(),
                                                  f["scales"].data_ptr(), pdt, _lib.ptr(f["resid"]), _lib.stream_of(x)))
    return f


def _same(a, b):
    for k in a:
        if a[k] is None:
            continue
        x, y = a[k], b[k]
        if x.dtype.is_floating_point:
            nan = torch.isnan(y)
            assert torch.equal(torch.isnan(x), nan), k
            it = torch.int16 if x.dtype == torch.float16 else torch.int32
            assert torch.equal(x.view(it)[~nan], y.view(it)[~nan]), k
        else:
            assert torch.equal(x, y), k


def _both(x, R, bits, gs, pdt, resid, rt=True):
    """x through the matrix-core kernel and, one element off, the general one."""
    n, d = x.shape
    flat = torch.empty(n * d + 8, dtype=x.dtype, device=DEV)
    got = _compress(x.contiguous(), R, bits, gs, pdt, resid, rt)
    off = flat[1:1 + n * d].view(n, d)
    off.copy_(x)
    _same(got, _compress(off, R, bits, gs, pdt, resid, rt))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("gs", [8, 16, 32, 64, 128])
@pytest.mark.parametrize("bits", [2, 3, 4, 8])
def test_every_group_and_width(d, gs, bits):
    if gs > d:
        pytest.skip("a group is at most the vector")
    print(f"group compress d={d} gs={gs} bits={bits}", flush=True)
    g = torch.Generator().manual_seed(d + gs + bits)
    R = torch.from_numpy(O.rotation_matrix(d, 42).astype(np.float32)).to(DEV)
    x = torch.randn(531, d, generator=g) * torch.randn(531, 1, generator=g).exp()
    _both(x.to(DEV), R, bits, gs, _lib.F16, False)
    _both(x.half().to(DEV), R, bits, gs, _lib.F32, True, rt=False)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 65, 30001])
def test_counts_and_types(d, dtype, n):
    print(f"group compress d={d} {dtype} n={n}", flush=True)
    g = torch.Generator().manual_seed(d + n)
    R = torch.from_numpy(O.rotation_matrix(d, 43).astype(np.float32)).to(DEV)
    _both(torch.randn(n, d, generator=g).to(dtype).to(DEV), R, 4, 32, _lib.F16, n != 33)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("identity", [False, True])
def test_special_values(d, identity):
    """Zero, tiny, flat, signed-zero, huge, infinite and NaN vectors."""
    g = torch.Generator().manual_seed(d)
    x = torch.randn(64, d, generator=g)
    x[0] = 0.0
    x[1] = x[1] * 1e-36
    x[2] = 1.0
    x[3] = x[3].abs() * (torch.arange(d) % 3 > 0)      # zeros among positives ...
    x[4] = x[3]
    x[4, ::3] = -0.0                                   # ... of either sign
    x[5] = x[4]
    x[5, ::6] = 0.0
    x[6] *= 1e6                                        # clamped to 65000
    x[7, 2], x[8, 3], x[9, 4] = float("inf"), float("-inf"), float("nan")
    x[10] *= 1e-20
    R = torch.eye(d) if identity else torch.from_numpy(O.rotation_matrix(d, 42).astype(np.float32))
    for gs in (8, 16, d):
        _both(x.to(DEV), R.to(DEV), 4, gs, _lib.F32, True)


@pytest.mark.parametrize("d,gs,off,transposed", [(128, 32, 0, False), (64, 64, 0, False), (128, 32, 1, True),
                                                 (128, 12, 0, True), (96, 32, 0, True)])
def test_general_kernel_gets_the_transposed_rotation(d, gs, off, transposed, monkeypatch):
    """compress_gpu transposes R exactly where the general kernel runs: without
    R^T its lanes read a row of R each."""
    R = torch.from_numpy(np.linalg.qr(np.random.default_rng(3).standard_normal((d, d)))[0].astype(np.float32)).to(DEV)
    flat = torch.empty(d * d + 8, device=DEV)
    Ro = flat[off:off + d * d].view(d, d)
    Ro.copy_(R)
    x = torch.randn(1, 2, 33, d, generator=torch.Generator().manual_seed(d)).to(DEV)
    lib, seen = _lib.lib(), []

    class Spy:
        def __getattr__(self, name):
            f = getattr(lib, name)
            if name != "pqkv_group_gpu_compress":
                return f
            return lambda *a: seen.append(a[3] is not None) or f(*a)

    monkeypatch.setattr(_lib, "_lib", Spy())
    got, want = compress_gpu(x, Ro, 4, gs), compress_gpu(x, R, 4, gs)
    assert seen[0] == transposed
    for f in ("radius", "quantized_direction", "group_mins", "group_scales"):
        assert torch.equal(getattr(got, f), getattr(want, f)), f
