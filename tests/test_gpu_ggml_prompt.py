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


def _both_routes(st, q, k, v, mask, n_kv, scale):
    return [ggml.flash_attn_ext(st, q, k, v, m, scale) for m in (_aligned(mask, n_kv), mask)]


def test_passes_over_streams():
    """Records of more than their 2 GiB: 7 streams in passes of 4 and 3, each
    split over many workgroups, against the split decode kernel."""
    d, H, n_q, n_kv = 128, 7, 64, 300000
    print(f"ggml passes H={H} n_q={n_q} n_kv={n_kv}", flush=True)
    gen = torch.Generator("cuda").manual_seed(3)
    with ggml.State(d, H, H) as st:
        caches = []
        for _ in range(2):
            c = torch.zeros(1, n_kv, H * ggml.row_size(d), dtype=torch.uint8, device="cuda")
            ggml.cpy(st, torch.randn(1, 1, n_kv, H * d, generator=gen, device="cuda", dtype=torch.float32), c[None])
            caches.append(c.view(1, n_kv, H, -1).transpose(1, 2))
        q = 4 * torch.randn(1, n_q, H, d, generator=gen, device="cuda").transpose(1, 2)
        mask = torch.zeros(1, 1, n_q, n_kv + 1, dtype=torch.float16, device="cuda")
        mask[..., n_kv - 100:].masked_fill_(torch.rand(n_q, 101, generator=gen, device="cuda") < 0.5, float("-inf"))
        a, b = _both_routes(st, q, *caches, mask, n_kv, d ** -0.5)
    rel = float((a - b).norm() / b.norm())
    print(f"between the routes {rel:.2e}", flush=True)
    assert rel <= 4e-6 and float(b.abs().mean()) > 0.01


@pytest.mark.parametrize("d,Hq,Hkv,n_q,n_kv", [(128, 32, 8, 64, 4096), (64, 14, 2, 1030, 2040)])
@pytest.mark.parametrize("where", ["query", "key", "value", "mask"])
@pytest.mark.parametrize("what", [float("inf"), float("nan"), 65504.0])
def test_values_at_the_ends_of_the_range(d, Hq, Hkv, n_q, n_kv, where, what):
    """Infinities, NaN and the largest values in queries, radii and masks (those
    negative, over a whole row): NaN exactly where the split decode kernel has
    it, the other rows as close as ever."""
    print(f"ggml {where} {what} d={d} n_q={n_q}", flush=True)
    st, q, (kv, vv), mask, _, _, _ = _case(d, Hq, Hkv, n_q, 1, 1, n_kv, "causal", 7)
    if where == "query":
        q[0, 0, 3], q[0, 1, 5, 2] = what, what
    elif where == "mask":
        mask[0, 0, 1, :n_kv], mask[0, 0, 2, 7] = -what, what
    else:
        c = (kv if where == "key" else vv).unflatten(-1, (d // 32, 18))
        for h, t in ((0, n_kv // 2), (Hkv - 1, n_kv - 1)):
            c[0, h, t, :, :2] = torch.tensor([what], dtype=torch.float16).view(torch.uint8).to(c.device)
    a, b = _both_routes(st, q, kv, vv, mask, n_kv, d ** -0.5)
    st.close()
    nan = torch.isnan(b)
    assert torch.equal(torch.isnan(a), nan) and not torch.isinf(a).any()
    if where == "mask" and what == float("inf"):
        assert not b[0, 1].any()                   # a row that sees nothing
    ok = ~nan
    if where == "mask":                            # logits of -65504 round to 2^-7
        ok[0, 1] = False
    if ok.any() and not (where in ("key", "query") and what == 65504.0):   # (logits of 1e5 move a weight freely)
        assert float((a - b)[ok].norm() / b[ok].norm()) <= 4e-6
