"""Chunked prefill with the preferred workspace (tokens split over workgroups;
from 12 row blocks, 6 at d = 64, tiles decoded once per call) against the same
call with the smallest one (a workgroup per row block that decodes them): odd
lengths, chunks whose early rows see none of a split's tokens, sign corrections,
per-head widths, paged caches."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from polarquant_kv import _lib, attention, quantizer

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# (B, Hq, Hkv, Sq, q_start, d, causal)
SHAPES = [(1, 8, 2, 9, 1000, 128, 1), (2, 14, 2, 33, 2111, 64, 1), (1, 4, 1, 300, 515, 128, 1),
          (1, 32, 8, 130, 4000, 128, 0), (3, 6, 2, 65, 767, 64, 0), (1, 1, 1, 513, 0, 128, 1),
          (1, 8, 2, 801, 100, 128, 1), (2, 14, 2, 300, 1003, 64, 1), (1, 4, 4, 3073, 0, 128, 1), (1, 14, 2, 217, 333, 64, 0)]


def _run(q, kc, vc, R, jl, q_start, causal, preferred):
    """One call with the workspace of the asked size, fp32 out."""
    lib = _lib.lib()
    B, Hq, Sq, d = q.shape
    Hkv, S = kc.num_heads, kc.seq_len
    base = lib.pqkv_prefill_workspace_bytes(B, Hq, Hkv, Sq, S, d)
    need = lib.pqkv_prefill_workspace_preferred_bytes(B, Hq, Hkv, Sq, S, d, int(jl is not None))
    assert need > base, "the shape takes no other plan"
    real = lib.pqkv_prefill_workspace_preferred_bytes
    if preferred:
        return attention.prefill_attention(q, kc, vc, R, q_start, causal=bool(causal), out_dtype=torch.float32, jl_rot=jl)

    class Small:
        def __getattr__(self, name):
            return (lambda *a: base) if name == real.__name__ else getattr(lib, name)

    old, _lib._lib = _lib._lib, Small()
    try:
        return attention.prefill_attention(q, kc, vc, R, q_start, causal=bool(causal), out_dtype=torch.float32, jl_rot=jl)
    finally:
        _lib._lib = old


def _check(got, want, vc, R):
    """Both evaluate the same fp32-grade products (each within 2^-21 of its
    term): with logits up to 8 in magnitude a weight moves by at most
    2 (8 + 1) 2^-21 of itself, a weighted sum by that and 2 2^-21 of max |v|."""
    vmax = float(quantizer.dequantize(vc, None, torch.float32).abs().max())
    assert float((got - want).abs().max()) <= 20 * 2.0 ** -21 * vmax * np.sqrt(R.shape[0])
    assert torch.isfinite(got).all()


def _states(B, H, S, d, seed):
    return torch.from_numpy(O.synth_kv(B, H, S, d, seed, "normal")).to(DEV)


@pytest.mark.parametrize("B,Hq,Hkv,Sq,q_start,d,causal", SHAPES)
@pytest.mark.parametrize("kind", ["4", "2", "qjl", "mixed", "paged"])
def test_split_equals_whole(B, Hq, Hkv, Sq, q_start, d, causal, kind):
    print(f"prefill {B} {Hq} {Hkv} Sq={Sq} q_start={q_start} d={d} causal={causal} {kind}", flush=True)
    S = q_start + Sq
    R = torch.from_numpy(O.rotation_matrix(d, 42).astype(np.float32)).to(DEV)
    jl = None
    if kind == "qjl":
        jl = torch.from_numpy((O.jl_matrix(d, d, 43) @ O.rotation_matrix(d, 42).T).astype(np.float32)).to(DEV)
    caches = []
    for i in range(2):
        if kind == "paged":
            c = quantizer.allocate_paged_cache(B, Hkv, d, 4, DEV, page_tokens=64)
        else:
            bits = tuple(4 if h % 2 else 2 for h in range(Hkv)) if kind == "mixed" else 2 if kind == "2" else 4
            c = quantizer.allocate_cache(B, Hkv, S + 7, d, bits, DEV, jl_dim=d if jl is not None and i == 0 else 0)
        caches.append(quantizer.compress_pq(_states(B, Hkv, S, d, 5 + i), R, cache=c, start=0, jl_rot=jl if i == 0 else None))
    kc, vc = caches
    q = (0.5 * torch.randn(B, Hq, Sq, d, generator=torch.Generator().manual_seed(S))).half().to(DEV)
    whole = _run(q, kc, vc, R, jl, q_start, causal, False)
    split = _run(q, kc, vc, R, jl, q_start, causal, True)
    _check(split, whole, vc if kind != "paged" else vc.to_contiguous(), R)


# (B, Hq, Hkv, Sq, q_start, d, kind, streams of a pass): the records of all
# streams exceed their 2 GiB
PASSES = [(2, 32, 8, 1531, 138469, 128, "4", 10),
          (2, 32, 8, 1531, 138469, 128, "paged", 10),
          (2, 32, 8, 1531, 138469, 128, "mixed", 10),  # 14 streams of one pair of widths, 2 of the other
          (4, 32, 8, 955, 138000, 64, "2", 17),
          (1, 3, 3, 3071, 1500000, 64, "4", 1)]        # each split over 21 workgroups


@pytest.mark.parametrize("B,Hq,Hkv,Sq,q_start,d,kind,streams", PASSES)
def test_passes_over_streams(B, Hq, Hkv, Sq, q_start, d, kind, streams):
    """The records are written, read and joined again for each pass of streams."""
    print(f"prefill passes {B} {Hq} {Hkv} Sq={Sq} q_start={q_start} d={d} {kind}", flush=True)
    S = q_start + Sq
    L = _lib.lib()
    extra = (L.pqkv_prefill_workspace_preferred_bytes(B, Hq, Hkv, Sq, S, d, 0)
             - L.pqkv_prefill_workspace_bytes(B, Hq, Hkv, Sq, S, d))
    assert extra // (-(-S // 64) * (512 * d + 512)) == streams
    R = torch.from_numpy(O.rotation_matrix(d, 42).astype(np.float32)).to(DEV)
    caches = []
    for i in range(2):
        if kind == "paged":
            c = quantizer.allocate_paged_cache(B, Hkv, d, 4, DEV, page_tokens=1024)
        else:
            bits = (4,) * (Hkv - 1) + (2,) if kind == "mixed" else int(kind)
            c = quantizer.allocate_cache(B, Hkv, S, d, bits, DEV)
        x = torch.randn(B, Hkv, S, d, generator=torch.Generator(DEV).manual_seed(i), device=DEV, dtype=torch.float16)
        caches.append(quantizer.compress_pq(x, R, cache=c, start=0))
        del x
    kc, vc = caches
    # queries that look at few keys, so that a stream's values show
    q = (4 * torch.randn(B, Hq, Sq, d, generator=torch.Generator().manual_seed(S))).half().to(DEV)
    got, want = _run(q, kc, vc, R, None, q_start, 1, True), _run(q, kc, vc, R, None, q_start, 1, False)
    # logits reach 50: 2 (50 + 1) 2^-21 of a weight, and 2 2^-21 of max |v|, a norm of 20
    assert float((got - want).abs().max()) <= 104 * 2.0 ** -21 * 20 and torch.isfinite(got).all()
    assert float(want.abs().mean()) > 0.01


def _call(q, kc, vc, R, jl, q_start, causal, ws):
    """pqkv_prefill_attn on a workspace of the caller's (a uint8 tensor), fp32 out."""
    B, Hq, Sq, d = q.shape
    mixed = kc.mixed
    kcb, vcb = attention._codebook_tables(kc, vc, mixed, kc.num_heads)
    out = torch.empty(B, Hq, Sq, d, device=DEV)
    _lib.check(_lib.lib().pqkv_prefill_attn(
        q.data_ptr(), _lib.dtype_code(q.dtype), R.data_ptr(), kc.blocks.data_ptr(), vc.blocks.data_ptr(), kcb.data_ptr(),
        vcb.data_ptr(), kc.head_bits()[0], vc.head_bits()[0], _lib.int_array(kc.head_bits()) if mixed else None,
        _lib.int_array(vc.head_bits()) if mixed else None, _lib.ptr(kc.qjl_signs if jl is not None else None), _lib.ptr(jl),
        d if jl is not None else 0, B, Hq, kc.num_heads, Sq, q_start, kc.seq_len, kc.max_seq_len, d, d ** -0.5, causal,
        out.data_ptr(), _lib.F32, ws.data_ptr(), ws.numel(), _lib.stream_of(q)))
    return out


@pytest.mark.parametrize("B,Hq,Hkv,Sq,q_start,d,qjl", [(1, 8, 2, 9, 1000, 128, False), (1, 8, 2, 801, 100, 128, False),
                                                       (2, 32, 8, 40, 1000, 128, True), (2, 14, 2, 300, 1003, 64, False)])
def test_workspace_off_a_16_byte_boundary(B, Hq, Hkv, Sq, q_start, d, qjl):
    """A workspace on a dword boundary only, of any size, gives what the
    smallest aligned one gives, bit for bit."""
    print(f"prefill workspace + 4 bytes {B} {Hq} {Hkv} Sq={Sq} d={d} qjl={qjl}", flush=True)
    S = q_start + Sq
    R = torch.from_numpy(O.rotation_matrix(d, 42).astype(np.float32)).to(DEV)
    jl = torch.from_numpy((O.jl_matrix(d, d, 43) @ O.rotation_matrix(d, 42).T).astype(np.float32)).to(DEV) if qjl else None
    kc, vc = (quantizer.compress_pq(_states(B, Hkv, S, d, 5 + i), R, jl_rot=jl if i == 0 else None) for i in range(2))
    q = torch.randn(B, Hq, Sq, d, generator=torch.Generator().manual_seed(S)).half().to(DEV)
    L = _lib.lib()
    base = L.pqkv_prefill_workspace_bytes(B, Hq, Hkv, Sq, S, d)
    most = L.pqkv_prefill_workspace_preferred_bytes(B, Hq, Hkv, Sq, S, d, int(qjl))
    assert most > base
    want = _call(q, kc, vc, R, jl, q_start, 1, torch.empty(base, dtype=torch.uint8, device=DEV))
    ws = torch.empty(most + 4, dtype=torch.uint8, device=DEV)
    for n in (base, most):
        assert torch.equal(_call(q, kc, vc, R, jl, q_start, 1, ws[4:4 + n]), want)


def test_decode_workspace_off_a_16_byte_boundary():
    """The same for the query rotations of a decode of many rows with sign corrections."""
    B, Hq, Hkv, S, d = 66, 32, 8, 70, 128
    R = torch.from_numpy(O.rotation_matrix(d, 42).astype(np.float32)).to(DEV)
    jl = torch.from_numpy((O.jl_matrix(d, d, 43) @ O.rotation_matrix(d, 42).T).astype(np.float32)).to(DEV)
    kc, vc = (quantizer.compress_pq(_states(B, Hkv, S, d, 5 + i), R, jl_rot=jl if i == 0 else None) for i in range(2))
    q = torch.randn(B, Hq, d, generator=torch.Generator().manual_seed(S)).half().to(DEV)
    ws = torch.empty(_lib.lib().pqkv_decode_workspace_bytes(B, Hq, Hkv, S, d) + 4, dtype=torch.uint8, device=DEV)
    got = [attention.decode_attention(q, kc, vc, R, jl_rot=jl, out_dtype=torch.float32, workspace=w) for w in (ws[:-4], ws[4:])]
    assert torch.equal(*got)


@pytest.mark.parametrize("B,Hq,Hkv,Sq,q_start,d", [(1, 8, 2, 65, 1000, 128), (1, 8, 2, 801, 100, 128),
                                                   (2, 14, 2, 300, 1003, 64)])
@pytest.mark.parametrize("where", ["query", "key", "value"])
@pytest.mark.parametrize("what", [float("inf"), float("nan"), 65504.0, 0.0])
def test_values_at_the_ends_of_the_range(B, Hq, Hkv, Sq, q_start, d, where, what):
    """Infinite, NaN, largest and zero queries and radii: NaN exactly where the
    kernel that decodes per row block has it, the other rows as close as ever."""
    print(f"prefill {where} {what} {B} {Hq} {Hkv} Sq={Sq} d={d}", flush=True)
    S = q_start + Sq
    R = torch.from_numpy(O.rotation_matrix(d, 42).astype(np.float32)).to(DEV)
    kc, vc = (quantizer.compress_pq(_states(B, Hkv, S, d, 5 + i), R) for i in range(2))
    q = (0.5 * torch.randn(B, Hq, Sq, d, generator=torch.Generator().manual_seed(S))).to(DEV)
    if where == "query":
        q[0, 0, 3], q[0, 1, 5, 2], q[-1, -1, Sq - 1, d - 1] = what, what, -what
    else:
        r = (kc if where == "key" else vc).blocks.view(B, Hkv, S, d // 32, 18)
        for b, h, t in ((0, 0, S // 2), (B - 1, Hkv - 1, S - 1)):
            r[b, h, t, :, :2] = torch.tensor([what], dtype=torch.float16).view(torch.uint8).to(DEV)
    got, want = _run(q, kc, vc, R, None, q_start, 1, True), _run(q, kc, vc, R, None, q_start, 1, False)
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan) and not torch.isinf(got).any()
    assert nan.any() or np.isfinite(what)
    # (a largest query or key radius makes logits whose 2^-21 moves a weight freely)
    if not nan.all() and not (what == 65504.0 and where != "value"):
        size = 65504.0 if what == 65504.0 else float(quantizer.dequantize(vc, None, torch.float32).nan_to_num(0, 0, 0).abs().max())
        assert float((got - want)[~nan].abs().max()) <= 20 * 2.0 ** -21 * size * np.sqrt(d)


@pytest.mark.parametrize("paged", [False, True])
def test_no_room_for_the_preferred_workspace(paged, monkeypatch):
    """A device too full for the preferred workspace runs the base plan."""
    B, Hq, Hkv, Sq, q_start, d = 1, 8, 2, 801, 100, 128
    S = q_start + Sq
    R = torch.from_numpy(O.rotation_matrix(d, 42).astype(np.float32)).to(DEV)
    caches = [quantizer.allocate_paged_cache(B, Hkv, d, 4, DEV, page_tokens=64) if paged else
              quantizer.allocate_cache(B, Hkv, S, d, 4, DEV) for _ in range(2)]
    kc, vc = (quantizer.compress_pq(_states(B, Hkv, S, d, 5 + i), R, cache=c, start=0) for i, c in enumerate(caches))
    q = (0.5 * torch.randn(B, Hq, Sq, d, generator=torch.Generator().manual_seed(S))).half().to(DEV)
    want = _run(q, kc, vc, R, None, q_start, 1, False)
    base, real, refused = _lib.lib().pqkv_prefill_workspace_bytes(B, Hq, Hkv, Sq, S, d), torch.empty, []

    def empty(*size, **kw):
        if len(size) == 1 and size[0] > base:
            refused.append(size[0])
            raise torch.cuda.OutOfMemoryError("out of memory")
        return real(*size, **kw)

    monkeypatch.setattr(torch, "empty", empty)
    got = attention.prefill_attention(q, kc, vc, R, q_start, out_dtype=torch.float32)
    assert refused and torch.equal(got, want)
