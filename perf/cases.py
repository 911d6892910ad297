"""The work a user of this framework has it do, as cases that can be timed and compared.

Kinds, each through its public entry point:
  hsdb      Y = W X with a block-coded (HSDB) W on the device (hsdr.HsdbSegment.matmul), or two
            matrices of one MLP in one call (hsdr.matmul_group): token generation (M = 1), a
            batch of sequences (M <= 16), prompts (M up to 256)
  hsdr      the same call on a stream of the compressor's own 1-row geometry (one tile per row)
  quant     Q4_K / GGUF dequant-matmul (q4k.linear, gguf.linear)
  attn      decode attention over an fp16 K/V cache (csdr_attn_decode)
  decode    a decoder's token loop from a filled context (Decoder.decode), logits at the end
  prefill   a decoder's prompt pass (Decoder.prefill), logits of the last position
  compress  an fp32 matrix in host memory to its HSDR stream (encode.compress)

Inputs are made from the seed alone: weights and coefficients normal, atoms unit length, atom
indices distinct within a block, quantised blocks with uniform quants.
"""
import ctypes
import math
import random

import numpy as np
import torch

from cortexsdr_amd import _lib, encode, formats, gguf, q4k
from cortexsdr_amd.decoder import LINEARS, Decoder, DecoderSpec, DecoderWeights
from cortexsdr_amd.hsdr import HsdbSegment, group_workspace, matmul_group

BLOCK = 64  # features per coded block
HEAD = dict(qwen=(14, 2, 64), llama=(32, 32, 128), gqa=(32, 8, 128))
QUANTS = {"q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210), "q8_0": (32, 34),
          "q4_0": (32, 18)}
VOCAB = 151936


def listed():
    return [
        # one attention projection of a 4096-wide model for one token: the smallest call
        dict(name="hsdb_4096_m1", kind="hsdb", R=4096, C=4096, K=512, s=4, M=1, x="f32",
             pair=False),
        # the two MLP matrices of a 4096-wide model for one token, one grouped call: the
        # benchmark's own step
        dict(name="hsdb_mlp_pair_m1", kind="hsdb", R=4096, C=11008, K=1024, s=8, M=1, x="f16",
             pair=True),
        # a batch of eight sequences generating together
        dict(name="hsdb_mlp_m8", kind="hsdb", R=11008, C=4096, K=1024, s=8, M=8, x="f32",
             pair=False),
        # a prompt's rows through one MLP matrix
        dict(name="hsdb_mlp_m256", kind="hsdb", R=4096, C=11008, K=1024, s=8, M=256, x="f16",
             pair=False),
        # an MLP matrix as the compressor writes it (1-row tiles, 3 stages of 8), a batch of 8
        dict(name="hsdr_mlp_m8", kind="hsdr", R=4864, C=896, K=512, S=3, k=8, M=8),
        # GGUF models: one token, and 32 rows of a prompt or batch
        dict(name="q4k_m1", kind="quant", fmt="q4_k", R=4096, C=14336, M=1, x="f16"),
        dict(name="q6k_m1", kind="quant", fmt="q6_k", R=4096, C=4096, M=1, x="f16"),
        dict(name="q4k_m32", kind="quant", fmt="q4_k", R=4096, C=14336, M=32, x="f16"),
        # the attention of a 7B-shaped model's step, eight sequences of context 4096
        dict(name="attn_4096_b8", kind="attn", heads="llama", B=8, T=4096),
        # Qwen2-0.5B-shaped blocks (4 of its 24): eight tokens after a 512-token context, and
        # the 512-token prompt itself
        dict(name="decode_qwen", kind="decode", layers=4, T=512, steps=8, batch=1),
        dict(name="prefill_qwen", kind="prefill", layers=4, T=512, batch=1),
        # an MLP matrix of that model compressed with the default refinement passes
        dict(name="compress_mlp", kind="compress", R=4864, C=896, K=512, S=3, k=8, iters=12),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["hsdb", "hsdb", "hsdr", "quant", "quant", "attn", "decode", "prefill",
                       "compress"])
    if kind == "hsdb":
        while True:
            R, C = _log(rng, 256, 14336), _log(rng, 256, 14336)
            if R * C <= 4096 * 11008:
                break
        M = rng.choice([1, _log(rng, 2, 16), _log(rng, 1, 256)])
        return dict(kind=kind, R=R, C=C, K=rng.choice([256, 512, 1024]),
                    s=rng.choice([4, 8, 16]), M=M, x=rng.choice(["f16", "f32"]),
                    pair=M == 1 and rng.random() < 0.3)
    if kind == "hsdr":
        return dict(kind=kind, R=_log(rng, 256, 8192), C=_log(rng, 256, 2048),
                    K=rng.choice([256, 512]), S=3, k=rng.choice([5, 8]), M=_log(rng, 1, 16))
    if kind == "quant":
        M = rng.choice([1, _log(rng, 2, 64)])
        return dict(kind=kind, fmt=rng.choice(list(QUANTS)), R=_log(rng, 256, 14336),
                    C=256 * _log(rng, 2, 16 if M > 1 else 56), M=M,
                    x=rng.choice(["f16", "f32"]) if M == 1 else "f16")
    if kind == "attn":
        return dict(kind=kind, heads=rng.choice(list(HEAD)), B=_log(rng, 1, 8),
                    T=_log(rng, 100, 4096))
    if kind == "decode":
        return dict(kind=kind, layers=rng.randint(1, 4), T=_log(rng, 20, 600),
                    steps=rng.randint(2, 8), batch=rng.choice([1, 1, 2, 4]))
    if kind == "prefill":
        return dict(kind=kind, layers=rng.randint(1, 4), T=_log(rng, 20, 700),
                    batch=rng.choice([1, 1, 2]))
    R = _log(rng, 600, 4864)
    return dict(kind=kind, R=R, C=_log(rng, 64, 1024), K=rng.choice([256, 512]), S=3,
                k=rng.choice([5, 8]), iters=rng.randint(0, 8))


# ---------------------------------------------------------------------------------- inputs


def _gen(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1009 + salt)
    return g


def _normal(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def _dict_atoms(g, K, width):
    d = _normal(g, K, width)
    return d / d.norm(dim=1, keepdim=True)


def _distinct(g, n, k, K):
    """n rows of k distinct values below K (the k-th draw counts only the values left)."""
    sel = torch.empty((n, k), dtype=torch.int64, device="cuda")
    for j in range(k):
        c = torch.randint(K - j, (n,), generator=g, device="cuda")
        prev = sel[:, :j].sort(dim=1).values
        for i in range(j):
            c = c + (prev[:, i] <= c)
        sel[:, j] = c
    return sel


def _hsdb_parts(g, R, C, D, s, sigma):
    """Codes, fp16 coefficients and edge strip of an R x C matrix against D."""
    nb = C // BLOCK
    idx = _distinct(g, R * nb, s, D.shape[0])
    coef = (_normal(g, R * nb, s) * sigma).half()
    ce = C - nb * BLOCK
    edge = _normal(g, R, ce) * (sigma / 8) if ce else None
    return idx, coef, edge


def _hsdb_stream(R, C, D, parts):
    idx, coef, edge = parts
    return formats.pack_hsdb(R, C, D.cpu().numpy(), idx.to(torch.int16).cpu().numpy(),
                             coef.cpu().numpy(), edge=edge.cpu().numpy() if edge is not None else None)


def _hsdb_dense64(R, C, D, parts):
    idx, coef, edge = parts
    w = torch.zeros(R * (C // BLOCK), BLOCK, dtype=torch.float64, device="cuda")
    for j in range(idx.shape[1]):
        w += coef[:, j:j + 1].double() * D[idx[:, j]].double()
    w = w.reshape(R, C // BLOCK * BLOCK)
    return w if edge is None else torch.cat([w, edge.double()], dim=1)


def _hsdb_inputs(case, seed):
    g = _gen(seed)
    D = _dict_atoms(g, case["K"], BLOCK)
    shapes = [(case["R"], case["C"])] + ([(case["C"], case["R"])] if case["pair"] else [])
    mats = [(R, C, _hsdb_parts(g, R, C, D, case["s"], 0.5)) for R, C in shapes]
    dt = torch.float16 if case["x"] == "f16" else torch.float32
    xs = [_normal(g, C, case["M"], dtype=dt) for _, C in shapes]
    return D, mats, xs


def _hsdr_inputs(case, seed):
    g = _gen(seed)
    R, C, K, S, k = (case[n] for n in ("R", "C", "K", "S", "k"))
    D = _dict_atoms(g, K, C) * (0.02 * math.sqrt(C) / math.sqrt(S * k))
    idx = torch.cat([_distinct(g, R, k, K) for _ in range(S)], dim=1)  # distinct per stage
    sign = torch.randint(2, (R, S * k), generator=g, device="cuda")
    gamma = 0.5 ** np.arange(S, dtype=np.float32)
    return D, idx, sign, gamma, _normal(g, C, case["M"])


def _hsdr_stream(case, D, idx, sign, gamma):
    R, C = case["R"], case["C"]
    head = formats.HEADER.pack(b"HSDR", 2, R, C, R, 1, C, case["K"], case["S"], case["k"], 0.5, 0)
    codes = (idx | (sign << 15)).cpu().numpy().astype("<u2")
    return b"".join([head, gamma.tobytes(), D.cpu().numpy().tobytes(), codes.tobytes()])


def _quant_inputs(case, seed):
    g = _gen(seed)
    be, bb = QUANTS[case["fmt"]]
    n = case["R"] * (case["C"] // be)
    w = torch.randint(256, (n, bb), generator=g, device="cuda", dtype=torch.uint8)
    d = 0.001 + 0.049 * torch.rand(n, 2, generator=g, device="cuda")
    d16 = d.half().view(torch.uint8).reshape(n, 4)
    if case["fmt"] == "q4_k":
        w[:, 0:4] = d16
    elif case["fmt"] == "q6_k":
        w[:, 208:210] = d16[:, :2]
    else:
        w[:, 0:2] = d16[:, :2]
    dt = torch.float16 if case["x"] == "f16" else torch.float32
    return w, _normal(g, case["M"], case["C"], dtype=dt)


def _attn_inputs(case, seed):
    g = _gen(seed)
    hq, hkv, hd = HEAD[case["heads"]]
    B, T = case["B"], case["T"]
    q = _normal(g, B, hq, hd)
    k = _normal(g, B, T, hkv, hd, dtype=torch.float16)
    v = _normal(g, B, T, hkv, hd, dtype=torch.float16)
    lens = torch.full((B,), T, dtype=torch.int32, device="cuda")
    return q, k, v, lens


def _model(case, seed):
    """Blocks of the Qwen2-0.5B shape: parts of every matrix, a prompt and a next token."""
    steps = case.get("steps", 0)
    spec = DecoderSpec(case["layers"], 896, 14, 2, 64, 4864, VOCAB, case["T"] + steps + 8)
    g = _gen(seed)
    D = _dict_atoms(g, 1024, BLOCK)
    shapes = spec.shapes()
    layers = [{n: _hsdb_parts(g, *shapes[n], D, 8, 0.1) for n in LINEARS}
              for _ in range(spec.n_layers)]
    head = _hsdb_parts(g, spec.vocab, spec.hidden, D, 8, 0.1)
    prompt = torch.randint(spec.vocab, (case["batch"], case["T"]), generator=g, device="cuda")
    token = torch.randint(spec.vocab, (case["batch"],), generator=g, device="cuda")
    return spec, D, layers, head, prompt, token


def _decoder(spec, D, layers, head, batch):
    shapes = spec.shapes()
    ones = np.ones(spec.hidden, np.float32)
    packed = []
    for L in layers:
        P = {n: _hsdb_stream(*shapes[n], D, L[n]) for n in LINEARS}
        P["attn_norm"] = P["ffn_norm"] = ones
        packed.append(P)
    lm = _hsdb_stream(spec.vocab, spec.hidden, D, head)
    return Decoder(DecoderWeights(spec, packed, lm, ones), batch=batch)


def _matrix(case, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal((case["R"], case["C"]), dtype=np.float32) * np.float32(0.02)


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind == "hsdb":
        D, mats, xs = _hsdb_inputs(case, seed)
        st["segs"] = [HsdbSegment(_hsdb_stream(R, C, D, p)) for R, C, p in mats]
        st["xs"] = xs
        st["ys"] = [torch.empty(R, case["M"], device="cuda") for R, _, _ in mats]
        st["ws"] = (group_workspace(st["segs"], case["M"]) if case["pair"]
                    else st["segs"][0].workspace(case["M"]))
    elif kind == "hsdr":
        D, idx, sign, gamma, x = _hsdr_inputs(case, seed)
        seg = HsdbSegment(_hsdr_stream(case, D, idx, sign, gamma))
        st.update(segs=[seg], xs=[x], ys=[torch.empty(case["R"], case["M"], device="cuda")],
                  ws=seg.workspace(case["M"]))
    elif kind == "quant":
        w, x = _quant_inputs(case, seed)
        st.update(w=w.reshape(-1), x=x, y=torch.empty(case["M"], case["R"], device="cuda"))
        if case["fmt"] != "q4_k":
            st["fmt"] = gguf.format_id(case["fmt"])
    elif kind == "attn":
        q, k, v, lens = _attn_inputs(case, seed)
        hq, _, hd = HEAD[case["heads"]]
        n = _lib.load().csdr_attn_decode_workspace_bytes(case["B"], hq, hd, case["T"])
        st.update(q=q, k=k, v=v, lens=lens, out=torch.empty_like(q),
                  ws=torch.zeros(n, dtype=torch.uint8, device="cuda"))
    elif kind in ("decode", "prefill"):
        spec, D, layers, head, prompt, token = _model(case, seed)
        st["dec"] = _decoder(spec, D, layers, head, case["batch"])
        st["prompt"] = prompt.cpu().numpy().astype(np.int32)
        st["token"] = token.cpu().numpy().astype(np.int32)
        if kind == "decode":
            st["dec"].prefill(st["prompt"], penalty=0.0)
    else:
        st["w"] = _matrix(case, seed)
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind in ("hsdb", "hsdr"):
        if case.get("pair"):
            return matmul_group(st["segs"], st["xs"], st["ys"], workspace=st["ws"])
        return st["segs"][0].matmul(st["xs"][0], out=st["ys"][0], workspace=st["ws"])
    if kind == "quant":
        if case["fmt"] == "q4_k":
            return q4k.linear(st["w"], case["R"], case["C"], st["x"], out=st["y"])
        return gguf.linear(st["w"], st["fmt"], case["R"], case["C"], st["x"], out=st["y"])
    if kind == "attn":
        hq, hkv, hd = HEAD[case["heads"]]
        _lib.check(_lib.load().csdr_attn_decode(
            st["q"].data_ptr(), st["k"].data_ptr(), st["v"].data_ptr(), st["lens"].data_ptr(), 0,
            case["B"], case["T"], hq, hkv, hd, ctypes.c_float(0.0), st["out"].data_ptr(),
            st["ws"].data_ptr(), st["ws"].numel(), torch.cuda.current_stream().cuda_stream))
        return st["out"]
    if kind == "decode":
        st["dec"].set_position(case["T"], st["token"])
        st["dec"].decode(case["steps"], penalty=0.0)
        return st["dec"].logits()
    if kind == "prefill":
        st["dec"].prefill(st["prompt"], penalty=0.0)
        return st["dec"].logits()
    out = encode.compress(st["w"], 1, case["C"], case["K"], case["S"], case["k"],
                          ksvd_iters=case["iters"])
    return np.frombuffer(out, np.uint8)


# ------------------------------------------------------------------------------------ work


def work(case):
    kind = case["kind"]
    if kind == "hsdb":
        n = 2 if case["pair"] else 1
        R, C, M, s = case["R"], case["C"], case["M"], case["s"]
        nb = (C // BLOCK) * R + ((R // BLOCK) * C if case["pair"] else 0)
        xb = 2 if case["x"] == "f16" else 4
        io = (C + (R if case["pair"] else 0)) * M * xb + (R + (C if case["pair"] else 0)) * M * 4
        return {"bytes": nb * s * 4 + case["K"] * BLOCK * 4 + io,
                "flops": 2 * M * min(n * R * C, nb * s + case["K"] * n * C)}
    if kind == "hsdr":
        R, C, K, M, s = case["R"], case["C"], case["K"], case["M"], case["S"] * case["k"]
        return {"bytes": R * s * 2 + K * C * 4 + C * M * 4 + R * M * 4,
                "flops": 2 * M * (K * C + R * s)}
    if kind == "quant":
        be, bb = QUANTS[case["fmt"]]
        R, C, M = case["R"], case["C"], case["M"]
        return {"bytes": R * (C // be) * bb + C * M * (2 if case["x"] == "f16" else 4) + R * M * 4,
                "flops": 2 * M * R * C}
    if kind == "attn":
        hq, hkv, hd = HEAD[case["heads"]]
        B, T = case["B"], case["T"]
        return {"bytes": 2 * B * T * hkv * hd * 2 + 2 * B * hq * hd * 4,
                "flops": 4 * B * T * hq * hd}
    if kind in ("decode", "prefill"):
        spec = DecoderSpec(case["layers"], 896, 14, 2, 64, 4864, VOCAB, 8)
        B, T = case["batch"], case["T"]
        lin = sum(r * c for r, c in spec.shapes().values())
        codes = case["layers"] * lin // BLOCK * 8 * 4
        head = VOCAB * 896 // BLOCK * 8 * 4
        kv = case["layers"] * B * T * 2 * 128 * 4
        if kind == "decode":
            return {"bytes": case["steps"] * (codes + head + kv) + B * VOCAB * 4, "flops": 0}
        return {"bytes": codes + head + kv + B * VOCAB * 4,
                "flops": case["layers"] * B * T * (2 * lin + 2 * T * 2 * 896 // 2)}
    n, C, K, s = case["R"], case["C"], case["K"], case["S"] * case["k"]
    passes = case["iters"] + 1
    # per pass: every tile's product with every atom once, then per pick the scores and the
    # residual updated; per refinement the residuals and the atoms' corrections
    return {"bytes": n * C * 4 + K * C * 4 + n * s * 2,
            "flops": passes * (2 * n * K * C + n * s * (2 * K + 2 * C)) +
            case["iters"] * 4 * n * s * C}


def tolerance(case):
    """About four times the error against 64 bits that the paths show: fp32 sums of a few
    thousand terms 2e-7 (5e-6 leaves room for another order over the whole range), fp16 x with
    fp32 sums of scaled quants 4e-6, logits after several blocks 8e-6 (more for sharper
    attention), and where weights are rounded to fp16 (the block-coded product from M = 9, the
    GGUF products from M = 2) 2e-4 to 5e-4."""
    kind = case["kind"]
    if kind == "compress":
        return "exact"
    if kind == "hsdb":
        return {"rel": 2e-3, "max": 0.02} if case["M"] > 8 else {"rel": 5e-6, "max": 1e-4}
    if kind == "attn":
        return {"rel": 1e-5, "max": 2e-4}
    if kind in ("decode", "prefill"):
        return {"rel": 1e-4, "max": 1e-3}
    if kind == "quant" and case["M"] > 1 and case["fmt"] != "q4_k":
        return {"rel": 2e-3, "max": 0.02}
    if kind == "quant":
        return {"rel": 2e-5, "max": 4e-4}
    return {"rel": 5e-6, "max": 1e-4}


# ----------------------------------------------------------------------------------- exact


def _unpack64(case, w):
    """The quantised matrix in 64 bits, in the element orders the engine decodes."""
    fmt = case["fmt"]
    if fmt == "q4_k":
        d, dmin = (w[:, o:o + 2].contiguous().view(torch.float16).double() for o in (0, 2))
        q = w[:, 4:16].int()
        sc = torch.cat([q[:, 0:4] & 63, (q[:, 8:12] & 15) | ((q[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([q[:, 4:8] & 63, (q[:, 8:12] >> 4) | ((q[:, 4:8] >> 6) << 4)], 1)
        qs = w[:, 16:144].reshape(-1, 4, 32)
        v = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
        out = d[:, :, None] * sc[:, :, None] * v - dmin[:, :, None] * mn[:, :, None]
    elif fmt == "q6_k":
        d = w[:, 208:210].contiguous().view(torch.float16).double()
        ql = w[:, 0:128].reshape(-1, 2, 2, 32).int()
        qh = w[:, 128:192].reshape(-1, 2, 32).int()
        sc = w[:, 192:208].contiguous().view(torch.int8).reshape(-1, 2, 8).double()
        quarters = [(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | ((qh >> 2 & 3) << 4),
                    (ql[:, :, 0] >> 4) | ((qh >> 4 & 3) << 4),
                    (ql[:, :, 1] >> 4) | ((qh >> 6 & 3) << 4)]
        out = torch.stack([sc[:, :, 2 * i:2 * i + 1] * (quarters[i] - 32).double()
                           for i in range(4)], 2) * d[:, :, None, None]
    else:
        d = w[:, 0:2].contiguous().view(torch.float16).double()
        if fmt == "q8_0":
            out = w[:, 2:].contiguous().view(torch.int8).double() * d
        elif fmt == "q4_0":
            out = (torch.stack([w[:, 2:] & 15, w[:, 2:] >> 4], 2).reshape(-1, 32).double() - 8) * d
        else:  # q5_k by the packed rule: 5 bits an element, lowest bits first, from byte 16
            bits = (w[:, 16:, None].int() >> torch.arange(8, device="cuda")) & 1
            v = (bits.reshape(-1, 256, 5) << torch.arange(5, device="cuda")).sum(2)
            out = (v - 16).double() * d
    return out.reshape(case["R"], case["C"])


def _rms64(x):
    return x / (x.square().mean(-1, keepdim=True) + 1e-5).sqrt()


def _forward64(spec, W, head, tokens):
    """Logits after `tokens` (B x T): the whole context through every block in 64 bits."""
    B, T = tokens.shape
    hq, hkv, hd = spec.n_heads, spec.n_kv_heads, spec.head_dim
    inv = spec.rope_theta ** (-torch.arange(0, hd, 2, device="cuda").double() / hd)
    ang = torch.arange(T, device="cuda").double()[:, None] * inv
    cos, sin = ang.cos()[:, None, :], ang.sin()[:, None, :]

    def rope(t):
        a, b = t[..., 0::2], t[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)

    mask = torch.full((T, T), -math.inf, device="cuda", dtype=torch.float64).triu(1)
    x = head[tokens]
    for L in W:
        h = _rms64(x)
        q = rope((h @ L["q"].T).reshape(B, T, hq, hd))
        k = rope((h @ L["k"].T).reshape(B, T, hkv, hd)).repeat_interleave(hq // hkv, 2)
        v = (h @ L["v"].T).reshape(B, T, hkv, hd).repeat_interleave(hq // hkv, 2)
        q, k, v = (t.transpose(1, 2).contiguous() for t in (q, k, v))
        p = torch.softmax(q @ k.transpose(2, 3).contiguous() / math.sqrt(hd) + mask, -1)
        a = (p @ v).transpose(1, 2).reshape(B, T, hq * hd)
        x = x + a @ L["o"].T
        h = _rms64(x)
        f = torch.nn.functional.silu(h @ L["gate"].T) * (h @ L["up"].T)
        x = x + f @ L["down"].T
    return _rms64(x[:, -1]) @ head.T


def exact(case, seed):
    kind = case["kind"]
    if kind == "hsdb":
        D, mats, xs = _hsdb_inputs(case, seed)
        ys = [_hsdb_dense64(R, C, D, p) @ x.double() for (R, C, p), x in zip(mats, xs)]
        return ys if case["pair"] else ys[0]
    if kind == "hsdr":
        D, idx, sign, gamma, x = _hsdr_inputs(case, seed)
        w = torch.zeros(case["R"], case["C"], dtype=torch.float64, device="cuda")
        for j in range(idx.shape[1]):
            w += (float(gamma[j // case["k"]]) * (1 - 2 * sign[:, j:j + 1])).double() * \
                D[idx[:, j]].double()
        return w @ x.double()
    if kind == "quant":
        w, x = _quant_inputs(case, seed)
        return x.double() @ _unpack64(case, w).T
    if kind == "attn":
        q, k, v, _ = _attn_inputs(case, seed)
        hq, hkv, hd = HEAD[case["heads"]]
        out = []
        for b in range(case["B"]):
            kb, vb = (t[b].double().repeat_interleave(hq // hkv, 1) for t in (k, v))
            p = torch.softmax((kb * q[b].double()).sum(-1) / math.sqrt(hd), 0)
            out.append((p[:, :, None] * vb).sum(0))
        return torch.stack(out)
    if kind in ("decode", "prefill"):
        spec, D, layers, head, prompt, token = _model(case, seed)
        shapes = spec.shapes()
        W = [{n: _hsdb_dense64(*shapes[n], D, L[n]) for n in LINEARS} for L in layers]
        H = _hsdb_dense64(spec.vocab, spec.hidden, D, head)
        ctx = prompt
        if kind == "prefill":
            lg = _forward64(spec, W, H, ctx)
        else:
            ctx = torch.cat([ctx, token[:, None]], 1)
            for i in range(case["steps"]):
                lg = _forward64(spec, W, H, ctx)
                ctx = torch.cat([ctx, lg.argmax(-1)[:, None]], 1)
        return (lg[0] if case["batch"] == 1 else lg).cpu().numpy()
    return None  # a byte stream
