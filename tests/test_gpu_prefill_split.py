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
