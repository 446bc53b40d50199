"""The work whose speed is measured: what programs built on this package have
it do, called through its public entry points.

A case is a dict of plain values; "op" names the entry point:

  encode      quantizer.compress_pq: new keys and values into a preallocated cache
  decode      attention.decode_attention: one query token per sequence
  prefill     attention.prefill_attention: a chunk of query tokens, causal
  decompress  quantizer.dequantize: a cache back to dense states
  ggml        ggml.flash_attn_ext: llama.cpp's layout, with ggml's mask
  group       polarquant_kv_cuda: compress_gpu of keys and values, then
              compressed_attention_gpu on them (the min / scale format)

Caches that attention reads are built here in plain torch (rotate, polar
split, nearest centroid, pack), so that the inputs do not depend on the
package's encoders.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "polarquant-kv_amd"))

from polarquant_kv import attention, ggml, quantizer  # noqa: E402
from polarquant_kv.qjl import generate_jl_matrix, rotated_jl_matrix  # noqa: E402
from polarquant_kv.rotation import generate_rotation_matrix  # noqa: E402
from polarquant_kv_cuda.attention_kernel import compressed_attention_gpu  # noqa: E402
from polarquant_kv_cuda.compress_kernel import compress_gpu  # noqa: E402

DEV = "cuda"
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
BLOCK_BYTES = {4: 18, 2: 10}            # fp16 radius + 32 codes


# ------------------------------------------------------------------- the cases

def listed():
    return [
        # One decode step's new keys and values of a serving batch of 8.
        dict(name="append_step", op="encode", B=8, Hkv=8, T=1, d=128, bits=4, dtype="f16", qjl=False, start=777,
             law="outlier"),
        # A bf16 model's prompt, encoded as it enters the cache of one layer.
        dict(name="encode_prompt_bf16", op="encode", B=1, Hkv=8, T=8191, d=128, bits=4, dtype="bf16", qjl=False,
             start=0, law="outlier"),
        # 2-bit keys with the sign sketch that corrects them, 16K tokens, batch 4.
        dict(name="encode_qjl_16k", op="encode", B=4, Hkv=8, T=16384, d=128, bits=2, dtype="f16", qjl=True, start=0,
             law="outlier"),
        # The whole 32K context of a batch of 8: the largest encode.
        dict(name="encode_32k", op="encode", B=8, Hkv=8, T=32768, d=128, bits=4, dtype="f16", qjl=False, start=0,
             law="outlier"),
        # One token of a small model at a short context: launches and host time.
        dict(name="decode_small", op="decode", B=1, Hq=14, Hkv=2, S=512, d=64, bits="4", qjl=False, paged=False,
             law="normal"),
        # One token per sequence at 32K context, batch 8: the headline decode.
        dict(name="decode_32k", op="decode", B=8, Hq=32, Hkv=8, S=32768, d=128, bits="4", qjl=False, paged=False,
             law="outlier"),
        # Mixed 2 / 4-bit heads with the sign correction, 16K tokens, batch 4.
        dict(name="decode_mixed_qjl", op="decode", B=4, Hq=32, Hkv=8, S=16384, d=128, bits="mixed", qjl=True,
             paged=False, law="outlier"),
        # A prompt of odd length, attending to itself through a paged cache.
        dict(name="prefill_prompt", op="prefill", B=2, Hq=32, Hkv=8, Sq=1531, q_start=0, d=128, bits="4", qjl=False,
             paged=True, law="normal"),
        # A 2048-token chunk against 131072 cached tokens: the largest call.
        dict(name="prefill_long", op="prefill", B=1, Hq=64, Hkv=8, Sq=2048, q_start=131072, d=128, bits="4",
             qjl=False, paged=False, law="normal"),
        # A cache handed to an attention that reads dense states.
        dict(name="decompress_8k", op="decompress", B=2, Hkv=8, S=8001, d=128, bits=4, dtype="f16", law="outlier"),
        # llama.cpp's prompt batch of 512 tokens on top of 3584 cached ones.
        dict(name="ggml_prompt", op="ggml", n_seq=1, Hq=32, Hkv=8, n_q=512, n_kv=4096, used=4096, d=128),
        # The reference's own benchmark: compress a 4096-token cache in its
        # min / scale format, then one query token per head.
        dict(name="group_flow", op="group", B=1, Hq=32, Hkv=32, S=4096, Sq=1, d=128, bits=4, group=32, qjl=False,
             dtype="f16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# (query heads, kv heads, head dim) of the shapes the cases above use, and
# one kv head per query head
SHAPES = [(14, 2, 64), (32, 8, 128), (64, 8, 128), (32, 32, 128)]


def draw(rng):
    op = rng.choice(["encode", "encode", "decode", "decode", "prefill", "prefill", "decompress", "ggml", "group"])
    Hq, Hkv, d = rng.choice(SHAPES)
    law = rng.choice(["normal", "outlier"])
    if op == "encode":
        B = _log(rng, 1, 16)
        T = 1 if rng.random() < 0.25 else _log(rng, 2, min(32768, 2097152 // (B * Hkv)))
        return dict(op=op, B=B, Hkv=Hkv, T=T, d=d, bits=rng.choice([4, 4, 2]), dtype=rng.choice(["f16", "bf16", "f32"]),
                    qjl=rng.random() < 0.3, start=rng.randrange(0, 300), law=law)
    if op == "decode":
        B = _log(rng, 1, 16)
        S = _log(rng, 33, 2097152 // (B * Hkv) if B * Hkv > 64 else 32768)
        paged = rng.random() < 0.4
        bits = rng.choice(["4", "4", "2"] if paged else ["4", "4", "2", "mixed"])
        return dict(op=op, B=B, Hq=Hq, Hkv=Hkv, S=S, d=d, bits=bits, qjl=rng.random() < 0.3, paged=paged, law=law)
    if op == "prefill":
        B, Sq = rng.choice([1, 1, 2, 4]), _log(rng, 9, 2048)
        q_start = 0 if rng.random() < 0.4 else _log(rng, 64, 65536)
        # no costlier than the longest listed prefill
        while B * Hq * Sq * (q_start + Sq) > 64 * 2048 * 65536:
            q_start //= 2
        paged = rng.random() < 0.4
        bits = rng.choice(["4", "4", "2"] if paged else ["4", "4", "2", "mixed"])
        return dict(op=op, B=B, Hq=Hq, Hkv=Hkv, Sq=Sq, q_start=q_start, d=d, bits=bits, qjl=rng.random() < 0.25,
                    paged=paged, law=law)
    if op == "decompress":
        return dict(op=op, B=_log(rng, 1, 8), Hkv=Hkv, S=_log(rng, 16, 8192), d=d, bits=rng.choice([4, 2]),
                    dtype=rng.choice(["f16", "f32"]), law=law)
    if op == "ggml":
        n_seq, n_q = rng.choice([1, 1, 2]), 1 if rng.random() < 0.3 else _log(rng, 2, 512)
        used = n_q + _log(rng, 1, 3584)
        return dict(op=op, n_seq=n_seq, Hq=Hq, Hkv=Hkv, n_q=n_q, n_kv=-(-used // 256) * 256, used=used, d=d)
    Sq = 1 if rng.random() < 0.5 else _log(rng, 2, 64)
    return dict(op=op, B=rng.choice([1, 1, 2]), Hq=Hq, Hkv=Hkv, S=_log(rng, 65, 4096), Sq=Sq, d=d,
                bits=rng.choice([4, 4, 2, 3]), group=rng.choice([32, 32, 16]), qjl=rng.random() < 0.3,
                dtype=rng.choice(["f16", "bf16"]))


# ------------------------------------------------------------------- inputs

def _states(gen, B, H, T, d, law, dtype):
    """[B, H, T, d] keys or values: N(0, 1) with a per-token norm factor
    LogNormal(0, 0.5), or per-channel std LogNormal(0, 1) with 1 % of the
    channels 20 times larger."""
    x = torch.randn(B, H, T, d, generator=gen, device=DEV)
    if law == "normal":
        x *= torch.randn(B, H, T, 1, generator=gen, device=DEV).mul_(0.5).exp_()
    else:
        std = torch.randn(1, H, 1, d, generator=gen, device=DEV).exp_()
        std *= 1 + 19 * (torch.rand(1, H, 1, d, generator=gen, device=DEV) < 0.01)
        x *= std
    return x.to(dtype)


def _pack(codes, radius, bits):
    """codes [..., d] uint8, radius [...] fp32 -> block bytes [..., vector bytes]."""
    per = 8 // bits
    parts = codes.unflatten(-1, (codes.shape[-1] // 32, 32 // per, per))
    qs = parts[..., 0].clone()
    for i in range(1, per):
        qs |= parts[..., i] << (bits * i)
    r = radius.clamp(max=65504).half().unsqueeze(-1).view(torch.uint8).unsqueeze(-2).expand(*qs.shape[:-1], 2)
    return torch.cat([r, qs], -1).flatten(-2)


def _blocks(x, R, cb, bits, p_rot=None):
    """Block bytes of states x [..., d] (and, with p_rot, their sign sketches)."""
    y = x.float() @ R.T
    r = y.norm(dim=-1)
    u = y / r.clamp(min=1e-30).unsqueeze(-1)
    c = cb[: 1 << bits]
    codes = torch.bucketize(u, (c[1:] + c[:-1]) / 2)
    signs = None
    if p_rot is not None:
        s = ((y - r.unsqueeze(-1) * c[codes]) @ p_rot.T >= 0).unflatten(-1, (p_rot.shape[0] // 8, 8))
        signs = (s * (1 << torch.arange(8, device=DEV))).sum(-1).to(torch.uint8)
    return _pack(codes.to(torch.uint8), r, bits), signs


def _unpack(blocks, d, bits, cb):
    """Block bytes [..., vector bytes] -> rotated-space vectors r c[code], float64 [..., d]."""
    nb, bb, per = d // 32, BLOCK_BYTES[bits], 8 // bits
    b = blocks.unflatten(-1, (nb, bb))
    r = b[..., 0, :2].contiguous().view(torch.float16).double()
    qs = b[..., 2:].unsqueeze(-1) >> (bits * torch.arange(per, device=DEV, dtype=torch.uint8))
    codes = (qs & ((1 << bits) - 1)).flatten(-3).long()
    return cb.double()[codes] * r


def _cache(gen, c, S, jl=False, P=None, R=None):
    """A key or value cache holding S positions, filled as above."""
    B, H, d = c["B"], c["Hkv"], c["d"]
    bits = c["bits"]
    n_bits = tuple(4 if h % 2 else 2 for h in range(H)) if bits == "mixed" else int(bits)
    if c.get("paged"):
        cache = quantizer.allocate_paged_cache(B, H, d, n_bits, DEV, jl_dim=d if jl else 0)
        cache.ensure(S)
    else:
        cache = quantizer.allocate_cache(B, H, -(-S // 256) * 256, d, n_bits, DEV, jl_dim=d if jl else 0)
    cache.seq_len = S
    heads = list(n_bits) if bits == "mixed" else [n_bits] * H
    for h in range(H):
        x = _states(gen, B, 1, S, d, c["law"], torch.float16)[:, 0]
        cb = cache.codebooks if cache.codebooks.dim() == 1 else cache.codebooks[h]
        blocks, signs = _blocks(x, R, cb, heads[h], P if jl else None)
        if c.get("paged"):
            for p, g in enumerate(cache.groups):
                part = slice(p * cache.page_tokens, min(S, (p + 1) * cache.page_tokens))
                g[:, h, :part.stop - part.start] = blocks[:, part]
                if jl:
                    cache.sign_groups[p][:, h, :part.stop - part.start] = signs[:, part]
            continue
        if bits == "mixed":
            off = cache.head_offset(h)
            cache.blocks[:, off:off + S * blocks.shape[-1]] = blocks.flatten(1)
        else:
            cache.blocks[:, h, :S] = blocks
        if jl:
            cache.qjl_signs[:, h, :S] = signs
    return cache


def _matrices(d, jl):
    R = generate_rotation_matrix(d, seed=42, device=DEV).float()
    if not jl:
        return R, None, None
    P = generate_jl_matrix(d, d, seed=43)
    return R, P, rotated_jl_matrix(P, R.cpu().numpy(), DEV)


_ggml_states = {}


def _ggml_state(case):
    """The type's device state: a program makes one per model."""
    key = (case["d"], case["Hkv"], case["Hq"])
    if key not in _ggml_states:
        _ggml_states[key] = ggml.State(case["d"], case["Hkv"], case["Hq"])
    return _ggml_states[key]


def prepare(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed))
    op, d = case["op"], case["d"]
    st = {"case": case}
    if op == "encode":
        B, H, T = case["B"], case["Hkv"], case["T"]
        st["R"], _, st["P"] = _matrices(d, case["qjl"])
        st["k"], st["v"] = (_states(gen, B, H, T, d, case["law"], DTYPES[case["dtype"]]) for _ in range(2))
        cap = -(-(case["start"] + T) // 256) * 256
        st["kc"] = quantizer.allocate_cache(B, H, cap, d, case["bits"], DEV, jl_dim=d if case["qjl"] else 0)
        st["vc"] = quantizer.allocate_cache(B, H, cap, d, case["bits"], DEV)
    elif op in ("decode", "prefill"):
        S = case["S"] if op == "decode" else case["q_start"] + case["Sq"]
        st["R"], _, st["P"] = _matrices(d, case["qjl"])
        st["kc"] = _cache(gen, case, S, jl=case["qjl"], P=st["P"], R=st["R"])
        st["vc"] = _cache(gen, case, S, R=st["R"])
        shape = (case["B"], case["Hq"], d) if op == "decode" else (case["B"], case["Hq"], case["Sq"], d)
        st["q"] = torch.randn(shape, generator=gen, device=DEV).half()
    elif op == "decompress":
        st["R"] = _matrices(d, False)[0]
        st["kc"] = _cache(gen, case, case["S"], R=st["R"])
    elif op == "ggml":
        st["state"] = _ggml_state(case)
        R = torch.from_numpy(ggml.rotation(d)).to(DEV)
        cb = torch.from_numpy(ggml.default_codebook()).to(DEV)
        ns, n_q, n_kv, used = case["n_seq"], case["n_q"], case["n_kv"], case["used"]
        # the cache as llama.cpp lays it out: a token's heads side by side
        for name in ("k", "v"):
            x = _states(gen, ns, case["Hkv"], n_kv, d, "normal", torch.float32)
            rows = torch.empty(ns, n_kv, case["Hkv"], ggml.row_size(d), dtype=torch.uint8, device=DEV)
            rows.copy_(_blocks(x, R, cb, 4)[0].transpose(1, 2))
            st[name] = rows.transpose(1, 2)
        st["q"] = torch.randn(ns, n_q, case["Hq"], d, generator=gen, device=DEV).transpose(1, 2)
        pos = torch.arange(used - n_q, used, device=DEV)
        mask = torch.full((1, 1, -(-n_q // 32) * 32, n_kv), float("-inf"), device=DEV)
        mask[0, 0, :n_q].masked_fill_(torch.arange(n_kv, device=DEV)[None] <= pos[:, None], 0.0)
        st["mask"], st["R"], st["cb"] = mask.half(), R, cb
    else:
        B, H, S = case["B"], case["Hkv"], case["S"]
        st["R"], P, _ = _matrices(d, case["qjl"])
        st["P"] = None if P is None else torch.as_tensor(P, dtype=torch.float32).to(DEV)
        st["k"], st["v"] = (_states(gen, B, H, S, d, "normal", DTYPES[case["dtype"]]) for _ in range(2))
        st["q"] = torch.randn(B, case["Hq"], case["Sq"], d, generator=gen, device=DEV).half()
    return st


# ------------------------------------------------------------------- one pass

def run(st):
    case = st["case"]
    op = case["op"]
    if op == "encode":
        quantizer.compress_pq(st["k"], st["R"], cache=st["kc"], start=case["start"], jl_rot=st["P"])
        quantizer.compress_pq(st["v"], st["R"], cache=st["vc"], start=case["start"])
        return {"k": st["kc"].blocks, "v": st["vc"].blocks, "signs": st["kc"].qjl_signs}
    if op == "decode":
        return attention.decode_attention(st["q"], st["kc"], st["vc"], st["R"], jl_rot=st["P"])
    if op == "prefill":
        return attention.prefill_attention(st["q"], st["kc"], st["vc"], st["R"], case["q_start"], jl_rot=st["P"])
    if op == "decompress":
        return quantizer.dequantize(st["kc"], st["R"], DTYPES[case["dtype"]])
    if op == "ggml":
        return ggml.flash_attn_ext(st["state"], st["q"], st["k"], st["v"], st["mask"], scale=case["d"] ** -0.5)
    kc = compress_gpu(st["k"], st["R"], case["bits"], case["group"], jl_matrix=st["P"])
    vc = compress_gpu(st["v"], st["R"], case["bits"], case["group"])
    out = compressed_attention_gpu(st["q"], kc, vc, st["R"], jl_matrix=st["P"])
    found = {"out": out}
    for name, c in (("k", kc), ("v", vc)):
        found[name] = {"codes": c.quantized_direction, "radius": c.radius, "mins": c.group_mins,
                       "scales": c.group_scales, "signs": c.qjl_signs, "norms": c.residual_norms}
    return found


# ------------------------------------------------------------------- what a pass cannot do without

def _vector_bytes(d, bits):
    return d // 32 * BLOCK_BYTES[bits]


def _pair_bytes(case):
    """Mean cache bytes of one position of one kv head, key and value."""
    d, bits = case["d"], case["bits"]
    one = (_vector_bytes(d, 2) + _vector_bytes(d, 4)) / 2 if bits == "mixed" else _vector_bytes(d, int(bits))
    return 2 * one + (d / 8 if case["qjl"] else 0)


def work(case):
    op, d = case["op"], case["d"]
    if op == "encode":
        n, es = 2 * case["B"] * case["Hkv"] * case["T"], DTYPES[case["dtype"]].itemsize
        q = n / 2 if case["qjl"] else 0
        return {"bytes": n * (d * es + _vector_bytes(d, case["bits"])) + q * d / 8 + 4 * d * d,
                "flops": 2.0 * (n + q) * d * d}
    if op == "decode":
        B, Hq, S = case["B"], case["Hq"], case["S"]
        return {"bytes": B * case["Hkv"] * S * _pair_bytes(case) + 4 * B * Hq * d + 4 * d * d,
                "flops": B * Hq * (4.0 * S * d * (1.5 if case["qjl"] else 1) + 4 * d * d)}
    if op == "prefill":
        B, Hq, Sq, q0 = case["B"], case["Hq"], case["Sq"], case["q_start"]
        pairs = Sq * q0 + Sq * (Sq + 1) // 2
        return {"bytes": B * case["Hkv"] * (q0 + Sq) * _pair_bytes(case) + 4 * B * Hq * Sq * d + 4 * d * d,
                "flops": B * Hq * (4.0 * pairs * d * (1.5 if case["qjl"] else 1) + 4.0 * Sq * d * d)}
    if op == "decompress":
        n = case["B"] * case["Hkv"] * case["S"]
        return {"bytes": n * (_vector_bytes(d, case["bits"]) + d * DTYPES[case["dtype"]].itemsize) + 4 * d * d,
                "flops": 2.0 * n * d * d}
    if op == "ggml":
        ns, Hq, n_q, used = case["n_seq"], case["Hq"], case["n_q"], case["used"]
        pairs = n_q * (used - n_q) + n_q * (n_q + 1) // 2
        return {"bytes": 2 * ns * case["Hkv"] * used * _vector_bytes(d, 4) + 8 * ns * Hq * n_q * d
                + 2 * n_q * case["n_kv"], "flops": ns * Hq * (4.0 * pairs * d + 4.0 * n_q * d * d)}
    B, S, ng = case["B"], case["S"], -(-d // case["group"])
    n = B * case["Hkv"] * S
    row = 2 + 4 * ng + d * {4: 1 / 2, 2: 1 / 4}.get(case["bits"], 1)
    sk = d / 8 + 2 if case["qjl"] else 0
    rows = B * case["Hq"] * case["Sq"]
    return {"bytes": 2 * n * (2 * d + row) + n * sk + 4 * rows * d + 4 * d * d,
            "flops": 2.0 * n * d * d * (3 if case["qjl"] else 2) + rows * (4.0 * S * d + 4 * d * d)}


def tolerance(case):
    # encoded bytes are whole values
    if case["op"] == "encode":
        return "exact"
    # fp32 results of fp32-grade products
    if case["op"] == "ggml":
        return {"rel": 4e-6, "max": 1e-4}
    if case["op"] == "decompress" and case["dtype"] == "f32":
        return {"rel": 1e-6, "max": 1e-5}
    # results rounded once to fp16: a value on the edge may round to its neighbour
    return {"rel": 4e-4, "max": 4e-3}


# ------------------------------------------------------------------- the same in 64 bits

def _attend(q, k, v, scale, bias=None, corr=None):
    """softmax(scale q k^T (+ corr) + bias) v in float64; q [n, d], k, v [S, d];
    bias(i0, i1) / corr(i0, i1): score terms of query rows i0 .. i1."""
    out = torch.empty_like(q)
    step = max(1, (1 << 28) // k.shape[0])
    for i in range(0, q.shape[0], step):
        j = min(q.shape[0], i + step)
        s = (q[i:j] @ k.T).mul_(scale)
        if corr is not None:
            s += corr(i, j)
        if bias is not None:
            s += bias(i, j)
        s -= s.amax(-1, keepdim=True)
        s.exp_()
        out[i:j] = (s @ v) / s.sum(-1, keepdim=True)
    return out


def _bits01(signs, m):
    return ((signs.unsqueeze(-1) >> torch.arange(8, device=DEV, dtype=torch.uint8)) & 1).flatten(-2)[..., :m].double()


def _stream(cache, b, h, S, what="blocks"):
    """The bytes of the first S positions of stream (b, h), and its width."""
    if hasattr(cache, "groups"):
        groups = cache.groups if what == "blocks" else cache.sign_groups
        return torch.cat([g[b, h] for g in groups])[:S], cache.n_bits
    if what != "blocks":
        return cache.qjl_signs[b, h, :S], 1
    bits = cache.head_bits()[h]
    if not cache.mixed:
        return cache.blocks[b, h, :S], bits
    vb, off = _vector_bytes(cache.head_dim, bits), cache.head_offset(h)
    return cache.blocks[b, off:off + S * vb].view(S, vb), bits


def _table(cache, h):
    return cache.codebooks if cache.codebooks.dim() == 1 else cache.codebooks[h]


def exact(case, seed):
    op, d = case["op"], case["d"]
    if op == "encode":
        return None                      # bytes: compared bit for bit instead
    st = prepare(case, seed)
    if op == "decompress":
        R, c = st["R"].double(), st["kc"]
        n = case["B"] * case["Hkv"]
        rows = [_unpack(_stream(c, i // case["Hkv"], i % case["Hkv"], case["S"])[0], d, case["bits"], c.codebooks) @ R
                for i in range(n)]
        out = torch.stack(rows).view(case["B"], case["Hkv"], case["S"], d)
        return out.clamp(-65504, 65504) if case["dtype"] == "f16" else out
    if op in ("decode", "prefill"):
        R, B, Hq, Hkv = st["R"].double(), case["B"], case["Hq"], case["Hkv"]
        S = case["S"] if op == "decode" else case["q_start"] + case["Sq"]
        q = st["q"].double()
        q = q.unsqueeze(2) if op == "decode" else q
        Sq, G, out = q.shape[2], Hq // Hkv, torch.empty_like(q)
        for b in range(B):
            for h in range(Hkv):
                qr = (q[b, h * G:(h + 1) * G].reshape(G * Sq, d)) @ R.T
                kb, kbits = _stream(st["kc"], b, h, S)
                vb, vbits = _stream(st["vc"], b, h, S)
                k, v = _unpack(kb, d, kbits, _table(st["kc"], h)), _unpack(vb, d, vbits, _table(st["vc"], h))
                corr = bias = None
                if case["qjl"]:
                    sg = _bits01(_stream(st["kc"], b, h, S, "signs")[0], d)
                    sg = (2 * sg - 1) * (~sg.bool().all(-1, keepdim=True))
                    pq = qr @ st["P"].double().T / d
                    corr = lambda i, j: (pq[i:j] @ sg.T) * d ** -0.5  # noqa: E731
                if op == "prefill":
                    t = torch.arange(S, device=DEV)
                    bias = lambda i, j: torch.where(  # noqa: E731
                        t[None] > case["q_start"] + torch.arange(i, j, device=DEV)[:, None] % Sq,
                        -math.inf, 0.0).double()
                o = _attend(qr, k, v, d ** -0.5, bias, corr) @ R
                out[b, h * G:(h + 1) * G] = o.view(G, Sq, d)
        return out[:, :, 0] if op == "decode" else out
    if op == "ggml":
        R, n_q, Hq, Hkv = st["R"].double(), case["n_q"], case["Hq"], case["Hkv"]
        G = Hq // Hkv
        out = torch.empty(case["n_seq"], n_q, Hq, d, dtype=torch.float64, device=DEV)
        m = st["mask"][0, 0, :n_q].double()
        for b in range(case["n_seq"]):
            for h in range(Hkv):
                qr = st["q"][b, h * G:(h + 1) * G].double().reshape(G * n_q, d) @ R.T
                k, v = (_unpack(st[n][b, h], d, 4, st["cb"]) for n in ("k", "v"))
                o = _attend(qr, k, v, d ** -0.5, lambda i, j: m[torch.arange(i, j, device=DEV) % n_q]) @ R
                out[b, :, h * G:(h + 1) * G] = o.view(G, n_q, d).transpose(0, 1)
        return out
    # group: codes are whole values, None in their place
    R, g, L = st["R"].double(), case["group"], (1 << case["bits"]) - 1
    ng = -(-d // g)
    found, dense = {}, {}
    for name in ("k", "v"):
        y = st[name].double() @ R.T
        r = y.norm(dim=-1)
        u = torch.nn.functional.pad(y / r.unsqueeze(-1).clamp(min=1e-30), (0, ng * g - d)).unflatten(-1, (ng, g))
        lo = u.amin(-1)
        s = (u.amax(-1) - lo) / L
        s = torch.where(s == 0, torch.ones_like(s), s)
        code = ((u - lo.unsqueeze(-1)) / s.unsqueeze(-1)).clamp(0, L).round()
        found[name] = {"codes": None, "radius": r, "mins": lo, "scales": s, "signs": None, "norms": None}
        dense[name] = ((code * s.half().double().unsqueeze(-1) + lo.half().double().unsqueeze(-1)).flatten(-2)[..., :d]
                       * r.half().double().unsqueeze(-1))
        if name == "k" and case["qjl"]:
            e = (y - (code * s.unsqueeze(-1) + lo.unsqueeze(-1)).flatten(-2)[..., :d] * r.unsqueeze(-1)) @ R
            found[name]["norms"] = e.norm(dim=-1)
            sketch = 2 * (e @ st["P"].double().T >= 0).double() - 1
    B, Hq, Hkv, Sq = case["B"], case["Hq"], case["Hkv"], case["Sq"]
    G, out = Hq // Hkv, torch.empty(B, Hq, Sq, d, dtype=torch.float64, device=DEV)
    for b in range(B):
        for h in range(Hkv):
            q = st["q"][b, h * G:(h + 1) * G].double().reshape(G * Sq, d)
            corr = None
            if case["qjl"]:
                pq = q @ st["P"].double().T / st["P"].shape[0]
                corr = lambda i, j: (pq[i:j] @ sketch[b, h].T) * d ** -0.5  # noqa: E731
            o = _attend(q @ R.T, dense["k"][b, h], dense["v"][b, h], d ** -0.5, None, corr) @ R
            out[b, h * G:(h + 1) * G] = o.view(G, Sq, d)
    found["out"] = out
    return found
