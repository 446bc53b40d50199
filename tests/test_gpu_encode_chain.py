"""The exact encoder on the matrix cores against the general exact encoder
(which an x off a 16-byte boundary takes): blocks and signs byte for byte at
step remainders and past one resident round, over head dims, widths, input
types, strided rows, and the SoA output."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from polarquant_kv import _lib
from polarquant_kv.lloyd_max import padded_codebook_torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CODE = {torch.float32: _lib.F32, torch.bfloat16: _lib.BF16}


def _mats(d):
    R = torch.from_numpy(O.rotation_matrix(d, 42).astype(np.float32)).to(DEV)
    P = torch.from_numpy((O.jl_matrix(d, d, 43) @ O.rotation_matrix(d, 42).T).astype(np.float32)).to(DEV)
    return R, P


def _states(n, d, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(n, d, generator=g) * torch.randn(n, 1, generator=g).exp()
    x[:: 97] = 0.0
    x[1:: 97] *= 1e-30                   # radii the Markstein form does not take
    return x.to(dtype).to(DEV)


def _encode(x, rows, d, bits, R, P, cb, pad):
    """x viewed as `rows` rows; blocks and signs rows `pad` vectors apart more."""
    n = x.shape[0] // rows
    vb = d // 32 * (18 if bits == 4 else 10)
    b = torch.zeros(rows, n + pad, vb, dtype=torch.uint8, device=DEV)
    q = torch.zeros(rows, n + pad, d // 8, dtype=torch.uint8, device=DEV) if P is not None else None
    _lib.check(_lib.lib().pqkv_encode(x.data_ptr(), CODE[x.dtype], n * d, R.data_ptr(), cb.data_ptr(), bits,
                                      b.data_ptr(), (n + pad) * vb, rows, n, d, _lib.ptr(P), d if P is not None else 0,
                                      _lib.ptr(q), (n + pad) * (d // 8), _lib.stream_of(x)))
    return b, q


@pytest.mark.parametrize("d,bits", [(64, 4), (64, 2), (128, 4), (128, 2)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,n,pad", [(1, 1, 0), (1, 31, 0), (1, 33, 0), (3, 65, 5), (2, 128, 1), (1, 25001, 0),
                                        (5, 11003, 3)])
def test_blocks_and_signs(d, bits, dtype, rows, n, pad):
    print(f"encode chain d={d} bits={bits} {dtype} {rows} x {n}", flush=True)
    R, P = _mats(d)
    cb = padded_codebook_torch(d, bits, DEV)
    x = _states(rows * n, d, dtype, d + bits + n)
    flat = torch.empty(x.numel() + 8, dtype=dtype, device=DEV)
    off = flat[1:1 + x.numel()].view_as(x)
    off.copy_(x)
    for p in (None, P):
        got, want = _encode(x, rows, d, bits, R, p, cb, pad), _encode(off, rows, d, bits, R, p, cb, pad)
        assert torch.equal(got[0], want[0])
        if p is not None:   # the same chains of one fused multiply-add per residual
            assert torch.equal(got[1], want[1])


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n", [1, 33, 65, 25001])
def test_soa(d, n):
    R, _ = _mats(d)
    cb = padded_codebook_torch(d, 4, DEV)
    x = _states(n, d, torch.float32, d + n)
    flat = torch.empty(x.numel() + 8, device=DEV)
    off = flat[1:1 + x.numel()].view_as(x)
    off.copy_(x)
    got = []
    for t in (x, off):
        r, p = torch.zeros(n, device=DEV), torch.zeros(n, d // 2, dtype=torch.uint8, device=DEV)
        _lib.lib().polarquant_compress_cuda_c(t.data_ptr(), R.data_ptr(), cb.data_ptr(), r.data_ptr(), p.data_ptr(), n, d,
                                              16, _lib.stream_of(x))
        got.append((r, p))
    assert torch.equal(got[0][0].view(torch.int32), got[1][0].view(torch.int32)) and torch.equal(got[0][1], got[1][1])
