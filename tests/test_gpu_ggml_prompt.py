"""flash_attn_ext with several query rows per sequence: the prefill kernel over
tiles decoded once per call (masks and key counts it reads in fours) and the
split decode kernel (every other mask), both against the oracle's float64
attention, at the edges of tiles (64 tokens), row blocks (256 rows) and splits."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from polarquant_kv import ggml
from test_gpu_ggml import _case

pytestmark = pytest.mark.gpu


def _aligned(mask, n_kv):
    """The same mask with rows of a multiple of four elements."""
    if mask is None:
        return None
    wide = torch.full((*mask.shape[:-1], n_kv + 8), float("-inf"), dtype=mask.dtype, device=mask.device)
    wide[..., :n_kv] = mask[..., :n_kv]
    return wide


@pytest.mark.parametrize("d,Hq,Hkv,n_q,ns,ns_kv,n_kv,kind", [
    (128, 32, 8, 64, 1, 1, 4096, "causal"),  # the smallest work, one whole row block, whole tiles
    (128, 32, 8, 65, 1, 1, 4164, "causal"),  # one row more, a part of a last tile
    (64, 14, 2, 1030, 1, 1, 2040, "causal"),  # G = 7: rows of a block left over
    (128, 8, 8, 257, 2, 2, 516, "rowmasked"),
    (128, 4, 4, 700, 1, 1, 772, "random"),
    (128, 8, 8, 300, 3, 1, 300, None),       # a shared cache, no splits
])
@pytest.mark.parametrize("q_mag,v_mag", [(1.0, 1.0), (300.0, 1.0), (1.0, 2.0 ** -10)])
def test_many_query_rows_match_the_oracle(d, Hq, Hkv, n_q, ns, ns_kv, n_kv, kind, q_mag, v_mag):
    print(f"ggml prompt d={d} Hq={Hq} Hkv={Hkv} n_q={n_q} ns={ns} ns_kv={ns_kv} n_kv={n_kv} {kind} "
          f"q x {q_mag} v x {v_mag}", flush=True)
    st, q, (kv, vv), mask, q_np, (k_val, v_val), m_np = _case(d, Hq, Hkv, n_q, ns, ns_kv, n_kv, kind, n_kv + n_q)
    scale = 1.0 / np.sqrt(d) / q_mag               # large queries, the same logits
    q, q_np = q * q_mag, q_np * np.float32(q_mag)
    if v_mag != 1.0:                               # values of small radius: 2^-10 of an fp16 above 2^-4 is exact
        r = vv.unflatten(-1, (d // 32, 18))[..., :2]
        r.copy_((r.contiguous().view(torch.float16) * v_mag).view(torch.uint8))
        v_val = v_val * v_mag
    want = O.ggml_flash_attn_ext(q_np, k_val, v_val, m_np, scale)
    routes = []
    for m in (_aligned(mask, n_kv), mask):
        got = ggml.flash_attn_ext(st, q, kv, vv, m, scale).cpu().numpy()
        assert np.isfinite(got).all()
        routes.append(got)
        if kind == "rowmasked":
            assert not got[0, n_q - 1].any()
    rel = [np.linalg.norm(a - b) / np.linalg.norm(b) for a, b in ((routes[0], want), (routes[1], want), routes)]
    print("against the oracle {:.2e}, split decode {:.2e}, between them {:.2e}".format(*rel), flush=True)
    # Each operand carries 2^-22 of itself and logits reach a few tens, so the
    # routes differ by a few 1e-6 at most. The oracle attends to the values
    # in the original space: R is orthogonal to a few 1e-7 per entry, which
    # the logits see once more.
    assert rel[2] <= 4e-6 and rel[0] <= 2e-5, rel
    st.close()
