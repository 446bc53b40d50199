"""Rotations and decodes of many vectors on the fp32 matrix cores: every output
bit equals the one-FMA-chain form (the C oracle, and the small-launch kernel on
special values), at the sizes around the dispatch line, step remainders, row
strides and odd alignments."""

import numpy as np
import pytest
import torch

import oracle as OC
from oracle import oracle as O
from polarquant_kv import _lib, quantizer

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rotate(x, R, inverse, out):
    _lib.check(_lib.lib().pqkv_rotate(x.data_ptr(), _lib.dtype_code(x.dtype), R.data_ptr(), out.data_ptr(),
                                      _lib.dtype_code(out.dtype), x.shape[0], x.shape[1], inverse, _lib.stream_of(x)))
    return out


def _bits(t):
    return t.contiguous().view(torch.int32 if t.dtype == torch.float32 else torch.int16)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("inverse", [0, 1])
@pytest.mark.parametrize("extra", [-1, 0, 1, 31, 33, 4095])
def test_rotate_bits_around_the_line(d, inverse, extra):
    n = (2048 if d == 128 else 4096) + extra
    print(f"rotate d={d} inverse={inverse} n={n}", flush=True)
    g = torch.Generator().manual_seed(n + d)
    x = torch.randn(n, d, generator=g)
    x[0], x[1], x[2] = 0.0, x[1] * 2.0 ** -140, x[2] * 2.0 ** 100
    R = torch.from_numpy(O.rotation_matrix(d, 42).astype(np.float32))
    want = OC.c_rotate_fma(x.numpy(), R.numpy(), inverse=bool(inverse))
    Rd = R.to(DEV)
    got = _rotate(x.to(DEV), Rd, inverse, torch.empty(n, d, device=DEV))
    assert np.array_equal(got.cpu().numpy().view(np.uint32), want.view(np.uint32))
    xh = x.half()
    want16 = OC.c_rotate_fma(xh.float().numpy(), R.numpy(), inverse=bool(inverse))
    got16 = _rotate(xh.to(DEV), Rd, inverse, torch.empty(n, d, device=DEV, dtype=torch.float16))
    with np.errstate(over="ignore"):
        assert np.array_equal(got16.cpu().numpy().view(np.uint16), want16.astype(np.float16).view(np.uint16))


@pytest.mark.parametrize("d", [64, 128])
def test_rotate_special_values_and_odd_alignment(d):
    """Infinities and NaN as in the small launches; an x off a 16-byte boundary
    still takes the general kernel."""
    n = 5000
    x = torch.randn(n + 1, d)
    x[7, 3], x[8, 5], x[9, d - 1], x[10, 0] = float("inf"), float("-inf"), float("nan"), 3e38
    R = torch.from_numpy(O.rotation_matrix(d, 42).astype(np.float32)).to(DEV)
    flat = torch.empty((n + 1) * d + 1, device=DEV)
    for off in (0, 1):
        xd = flat[off:off + n * d].view(n, d)
        xd.copy_(x[:n])
        many = _rotate(xd, R, 0, torch.empty(n, d, device=DEV))
        few = torch.cat([_rotate(xd[i:i + 500], R, 0, torch.empty(500, d, device=DEV)) for i in range(0, n, 500)])
        nan = torch.isnan(few)
        assert torch.equal(torch.isnan(many), nan)
        assert torch.equal(_bits(many)[~nan], _bits(few)[~nan])


@pytest.mark.parametrize("d,bits", [(64, 2), (64, 4), (128, 2), (128, 4)])
@pytest.mark.parametrize("B,H,S,cap", [(1, 1, 1, 1), (2, 3, 33, 64), (3, 2, 700, 701), (1, 4, 2049, 2049)])
def test_dequantize_rows_bits(d, bits, B, H, S, cap):
    """Every head of a cache longer than its valid positions in one launch,
    and a batch stride of its own; a mixed cache's heads as the uniform ones'."""
    print(f"dequantize d={d} bits={bits} B={B} H={H} S={S}", flush=True)
    rng = np.random.default_rng(d + bits + S)
    idx = rng.integers(0, 1 << bits, (B * H * cap, d)).astype(np.uint8)
    r = rng.lognormal(0, 2, B * H * cap).astype(np.float32)
    blocks = O.pack_blocks(r, idx, bits)
    cb = O.lloyd_max_codebook(d, bits)[0]
    R = O.rotation_matrix(d, 42).astype(np.float32)
    r16, idx2 = O.unpack_blocks(blocks, d, bits)
    xr = (r16.astype(np.float32)[:, None] * cb[idx2]).astype(np.float32)
    want = OC.c_rotate_fma(xr, R, inverse=True).reshape(B, H, cap, d)[:, :, :S]
    cache = quantizer.allocate_cache(B, H, cap, d, bits, DEV)
    cache.blocks.copy_(torch.from_numpy(blocks).view(B, H, cap, -1))
    cache.seq_len = S
    Rt = torch.from_numpy(R).to(DEV)
    got = quantizer.dequantize(cache, Rt, torch.float32)
    assert np.array_equal(got.cpu().numpy().view(np.uint32), want.view(np.uint32))
    wide = torch.zeros(B, H + 1, cap, cache.blocks.shape[-1], dtype=torch.uint8, device=DEV)
    wide[:, :H] = cache.blocks
    cache.blocks = wide[:, :H]
    assert torch.equal(_bits(quantizer.dequantize(cache, Rt, torch.float32)), _bits(got))
    mixed = quantizer.allocate_cache(B, H, cap, d, (bits,) * H, DEV)
    mixed.blocks.copy_(wide[:, :H].reshape(B, -1))
    mixed.seq_len = S
    assert torch.equal(_bits(quantizer.dequantize(mixed, Rt, torch.float32)), _bits(got))


def _block_cache(B, H, S, cap, d, bits):
    """A cache whose first S positions hold random codes and radii, and the
    same vectors one after the other."""
    g = torch.Generator().manual_seed(d + bits + S)
    cache = quantizer.allocate_cache(B, H, cap, d, bits, DEV)
    cache.blocks.copy_(torch.randint(0, 256, cache.blocks.shape, generator=g, dtype=torch.uint8))
    r = (torch.randn(B, H, cap, 1, 1, generator=g) * 2).exp().half().view(torch.uint8).to(DEV)
    cache.blocks.unflatten(-1, (d // 32, -1))[..., :2] = r.reshape(B, H, cap, 1, 2)
    cache.seq_len = S
    return cache, cache.blocks[:, :, :S].reshape(B * H * S, -1)


def _in_chunks(rows, R, codebook, bits, d, dtype, step):
    out = torch.empty(rows.shape[0], d, dtype=dtype, device=DEV)
    for i in range(0, rows.shape[0], step):
        n = min(step, rows.shape[0] - i)
        _lib.check(_lib.lib().pqkv_dequantize(rows[i:].data_ptr(), codebook.data_ptr(), bits, R.data_ptr(),
                                              out[i:].data_ptr(), _lib.dtype_code(dtype), n, d, _lib.stream_of(out)))
    return out


@pytest.mark.parametrize("d,bits", [(64, 2), (64, 4), (128, 2), (128, 4)])
@pytest.mark.parametrize("B,H,S,cap", [(1, 1, 1024, 1024), (5, 1, 205, 300), (2, 2, 256, 257), (1, 8, 512, 520),
                                       (1, 17, 241, 250)])
def test_dequantize_bits_on_both_sides_of_the_line(d, bits, B, H, S, cap):
    """1024 / 1025 vectors at d = 128, 4096 / 4097 at d = 64, rows apart: every
    bit is what one vector at a time gives (few vectors: the vector ALU kernel)."""
    print(f"dequantize line d={d} bits={bits} B={B} H={H} S={S}", flush=True)
    cache, rows = _block_cache(B, H, S, cap, d, bits)
    R = torch.from_numpy(O.rotation_matrix(d, 42).astype(np.float32)).to(DEV)
    for dtype in (torch.float16, torch.float32):
        got = quantizer.dequantize(cache, R, dtype).reshape(-1, d)
        assert torch.equal(_bits(got), _bits(_in_chunks(rows, R, cache.codebooks, bits, d, dtype, 333)))


@pytest.mark.parametrize("bits", [4, (4, 2, 4)])
def test_dequantize_of_empty_and_expanded_caches(bits):
    """No batch rows give an empty result; a cache whose batch rows (or heads)
    are one set of bytes expanded gives that set's values in each."""
    d, S, cap = 128, 33, 40
    R = torch.from_numpy(O.rotation_matrix(d, 42).astype(np.float32)).to(DEV)
    one = quantizer.allocate_cache(1, 3, cap, d, bits, DEV)
    x = torch.randn(1, 3, S, d, generator=torch.Generator().manual_seed(1)).to(DEV)
    quantizer.compress_pq(x, R, cache=one, start=0)
    want = quantizer.dequantize(one, R, torch.float32)
    empty = quantizer.allocate_cache(0, 3, cap, d, bits, DEV)
    assert quantizer.dequantize(empty, R, positions=S).shape == (0, 3, S, d)
    beams = quantizer.allocate_cache(4, 3, cap, d, bits, DEV, codebooks=one.codebooks)
    beams.blocks, beams.seq_len = one.blocks.expand(4, *one.blocks.shape[1:]), S
    assert torch.equal(quantizer.dequantize(beams, R, torch.float32), want.expand(4, -1, -1, -1))
    with pytest.raises(ValueError):
        quantizer.dequantize(one, R, positions=cap + 1)
    if bits == 4:
        heads = quantizer.allocate_cache(2, 3, cap, d, bits, DEV)
        heads.blocks, heads.seq_len = one.blocks[:, :1].expand(2, 3, -1, -1), S
        assert torch.equal(quantizer.dequantize(heads, R, torch.float32), want[:, :1].expand(2, 3, -1, -1))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("inverse", [0, 1])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_rotate_bits_past_one_resident_round(d, inverse, dtype):
    """About 2.5 steps per workgroup (four of them per compute unit, 32 vectors a
    step, 64 at d = 64) and a remainder, against small launches."""
    n = (82000 if d == 128 else 164000) + 7
    print(f"rotate steady state d={d} inverse={inverse} {dtype}", flush=True)
    assert n > 2 * 4 * torch.cuda.get_device_properties(0).multi_processor_count * (32 if d == 128 else 64)
    R = torch.from_numpy(O.rotation_matrix(d, 42).astype(np.float32)).to(DEV)
    x = torch.randn(n, d, generator=torch.Generator(DEV).manual_seed(d), device=DEV).to(dtype)
    many = _rotate(x, R, inverse, torch.empty(n, d, device=DEV))
    few = torch.empty(n, d, device=DEV)
    for i in range(0, n, 2000):
        _rotate(x[i:i + 2000], R, inverse, few[i:i + 2000])
    assert torch.equal(_bits(many), _bits(few))


@pytest.mark.parametrize("d,bits", [(64, 2), (64, 4), (128, 2), (128, 4)])
def test_dequantize_bits_past_one_resident_round(d, bits):
    """The same for rows of a cache longer than its valid positions."""
    B, H, S, cap = 3, 4, 6841 if d == 128 else 13677, 13700
    print(f"dequantize steady state d={d} bits={bits}", flush=True)
    cache, rows = _block_cache(B, H, S, cap, d, bits)
    R = torch.from_numpy(O.rotation_matrix(d, 42).astype(np.float32)).to(DEV)
    for dtype in (torch.float16, torch.float32):
        got = quantizer.dequantize(cache, R, dtype).reshape(-1, d)
        assert torch.equal(_bits(got), _bits(_in_chunks(rows, R, cache.codebooks, bits, d, dtype, 1000)))
