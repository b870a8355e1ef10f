"""Performance cases: the calls a program that serves a Llama-shaped model over
the compressed KV cache makes, at the sizes it makes them.

Five kinds of case:

  step      one decode token through the attention of every layer of a model,
            captured once in a HIP graph and replayed per token: per layer RoPE
            of q and k with the stream append (ops.rope_stream_append_at), then
            the fused attention (ops.decode_attn), with the stream row, the
            stream length and the position in device memory.
  attend    one decode token of one layer, called eagerly as the patched
            attention forward calls it: layer.fused_rope_append and
            fused_attention_compressed (streaming), or the attention alone over
            fp16 decode tokens with a padding mask (not streaming).
  rebuild   layer.keys / layer.values of a compressed cache's layers: the fp16
            K and V that unfused consumers read.
  encode    one layer's prefill compression onto a fixed basis and codebook
            (the fp16 projection with undo-RoPE fused in, the int4 chain, the
            channel scales and the table assignment of V).
  compress  Cache.compress() of one layer after its prefill, with its own PCA
            basis, bit allocation and k-means codebook, then its rebuilt K/V.

Inputs are seeded and made on the GPU.  Compressed layers of the decode and
rebuild cases are drawn directly in the stored format (codes of Gaussian
coefficients under an exponential spectrum, unit-variance keys).
"""
import functools
import itertools
import math

import torch

DEV = "cuda"
THETA = 500000.0
SINK, WIN = 4, 64      # fp16 tokens kept on either side of the compressed span
MEAN_STD = 0.1
STREAM_BITS = 8


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    llama8b = dict(n_q=32, n_kv=8, hd=128, rank=192)
    llama1b = dict(n_q=32, n_kv=8, hd=64, rank=192)
    llama3b = dict(n_q=24, n_kv=8, hd=128, rank=192)
    return [
        # interactive decoding after a short prompt, a 32-layer model
        dict(name="step_2k", kind="step", layers=32, batch=1, tokens=2048, stream=64, **llama8b),
        # the headline context, batch 1
        dict(name="step_8k", kind="step", layers=32, batch=1, tokens=8192, stream=64, **llama8b),
        # long context with a 512-token decode stream
        dict(name="step_32k_stream512", kind="step", layers=32, batch=1, tokens=32768, stream=512, **llama8b),
        # a small batch on the head_dim-64 model (16 layers), a ragged prompt
        dict(name="step_pairs_b4_5k", kind="step", layers=16, batch=4, tokens=5003, stream=33, **llama1b),
        # batch serving: one layer of the batch-16 end-to-end run
        dict(name="attend_b16_16k", kind="attend", batch=16, tokens=16384, stream=64, masked=False, **llama8b),
        # a left-padded pair of prompts, 3 query heads per kv head, no stream
        dict(name="attend_masked_gqa3", kind="attend", batch=2, tokens=3001, stream=17, masked=True, **llama3b),
        # fp16 K/V of two layers for a consumer without the fused path
        dict(name="rebuild_8k", kind="rebuild", layers=2, batch=1, tokens=8192, stream=16, **llama8b),
        # the same on a batch of the head_dim-64 model
        dict(name="rebuild_pairs_b4_3k", kind="rebuild", layers=2, batch=4, tokens=3001, stream=0, **llama1b),
        # prefill compression of a short ragged prompt's layer, and of the
        # benchmark's layer (batch 4 x 8192)
        dict(name="encode_1k", kind="encode", batch=1, tokens=1003, n_kv=8, hd=128, rank=192),
        dict(name="encode_b4_8k", kind="encode", batch=4, tokens=8192, n_kv=8, hd=128, rank=192),
        # Cache.compress() at the first decode step: an ordinary prompt, and
        # one layer of the batch-16 end-to-end run
        dict(name="compress_2k", kind="compress", batch=1, tokens=2048, n_kv=8, hd=128, rank=192),
        dict(name="compress_b16_16k", kind="compress", batch=16, tokens=16384, n_kv=8, hd=128, rank=192),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "attend", "attend", "rebuild", "encode", "compress"])
    n_q, n_kv, hd = rng.choice([(32, 8, 128), (32, 8, 128), (32, 8, 64), (24, 8, 128), (8, 2, 128), (32, 4, 64)])
    rank = rng.choice([192, 192, 192, 128, 64])
    c = dict(kind=kind, n_q=n_q, n_kv=n_kv, hd=hd, rank=rank)
    if kind == "step":
        c["batch"] = rng.choice([1, 1, 1, 2, 3, 4, 8])
        c["tokens"] = _log(rng, 512, 32768 // c["batch"])
        c.update(layers=rng.choice([8, 16]), stream=_log(rng, 1, 600))
    elif kind == "attend":
        c["batch"] = _log(rng, 1, 16)
        c.update(tokens=_log(rng, 512, 16384), stream=_log(rng, 1, 300), masked=rng.random() < 0.3)
    elif kind == "rebuild":
        c["batch"] = rng.choice([1, 1, 2, 4])
        c["tokens"] = _log(rng, 512, 32768 // c["batch"])
        c.update(layers=2, stream=rng.choice([0, 1, 40]))
    else:
        c.pop("n_q")
        if kind == "encode":
            c.update(n_kv=rng.choice([8, 4]), hd=128, batch=rng.choice([1, 2, 4]))
            c["tokens"] = _log(rng, 512, 8192)
        else:
            c.update(n_kv=rng.choice([8, 8, 4]), hd=128, rank=192, batch=rng.choice([1, 2, 4]))
            c["tokens"] = _log(rng, 1024, 16384)
    return c


# ---------------------------------------------------------------------------
# inputs: tensors made from the seed alone
# ---------------------------------------------------------------------------
def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1009 + salt)


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device=DEV, dtype=dtype)


@functools.lru_cache(maxsize=None)
def _inv_freq(hd):
    return 1.0 / (THETA ** (torch.arange(0, hd, 2, dtype=torch.float32) / hd))


@functools.lru_cache(maxsize=None)
def _stream_codebook(hd):
    """Lloyd-Max levels of N(0, 1/hd) for the 8-bit stream (fp32)."""
    n = 1 << STREAM_BITS
    c = torch.special.ndtri((torch.arange(n, dtype=torch.float64) + 0.5) / n)
    pdf = lambda x: torch.exp(-0.5 * x * x) / math.sqrt(2 * math.pi)
    for _ in range(200):
        edge = torch.cat([c.new_tensor([-math.inf]), (c[1:] + c[:-1]) / 2, c.new_tensor([math.inf])])
        mass = torch.special.ndtr(edge[1:]) - torch.special.ndtr(edge[:-1])
        c = (pdf(edge[:-1]) - pdf(edge[1:])) / mass
    return (c / math.sqrt(hd)).float()


def _stored_layer(case, g):
    """One compressed layer in the stored format (B, G, n compressed tokens)."""
    B, G, hd, rank = case["batch"], case["n_kv"], case["hd"], case["rank"]
    n, p = case["tokens"] - SINK - WIN, G * hd
    sigma = torch.exp(-torch.arange(rank, device=DEV, dtype=torch.float32) * (math.log(100.0) / 384))
    sigma *= math.sqrt(p / float(sigma.pow(2).sum()))           # unit variance per key dim
    basis = _randn(g, p, rank) / math.sqrt(p)
    scale = basis.abs().amax(0) / 127
    basis_q = (basis / scale).round().clamp(-127, 127)
    codes = (_randn(g, B * n, rank) * (7 / 4)).round().clamp(-7, 7)  # column maximum near 4 sigma
    shifted = (codes + 8).to(torch.uint8).view(-1)
    mean = (_randn(g, p) * MEAN_STD).half()
    fp16 = lambda t: _randn(g, B, G, t, hd).half()
    fmt = {
        "k_coeffs": shifted[0::2] | (shifted[1::2] << 4), "k_coeffs_shape": (B * n, rank),
        "k_coeff_scale": (sigma * (4 / 7)).half(),
        "k_basis_f16": (basis_q.half() * scale.half()).contiguous(), "k_mean_f16": mean,
        "v_indices": torch.randint(0, 256, (B, G, n, hd // 4), generator=g, device=DEV).to(torch.uint8),
        "v_centroids_f16": (_randn(g, 256, 4) * 0.3).clamp(-1, 1).half(),
        "v_ch_f16": (torch.rand(B, G, hd, generator=g, device=DEV) + 3.5).half(),
        "sink_k": fp16(SINK), "sink_v": fp16(SINK), "win_k": fp16(WIN), "win_v": fp16(WIN),
        "n_compress": n, "batch": B, "compress_start": SINK, "n_kv": G, "head_dim": hd, "rank": rank,
    }
    return fmt


def _raw_layer(case, seed, li):
    """The inputs of layer li: stored layer, decode tokens so far, the new token."""
    g = _gen(seed, li)
    B, G, hd, s = case["batch"], case["n_kv"], case["hd"], case["stream"]
    raw = {"fmt": _stored_layer(case, g)}
    raw["signs"] = (torch.randint(0, 2, (hd,), generator=g, device=DEV) * 2 - 1).float()
    raw["stream_k"] = _randn(g, s, B, G, hd).half()
    raw["stream_v"] = _randn(g, s, B, G, hd).half()
    if "n_q" in case:
        raw["q"] = _randn(g, B, case["n_q"], 1, hd).half()
        raw["k"] = _randn(g, B, G, 1, hd).half()
        raw["v"] = _randn(g, B, G, 1, hd).half()
    return raw


def _position(case):
    return case["tokens"] + case["stream"]      # of the new decode token


def _cos_sin(case):
    ph = _position(case) * _inv_freq(case["hd"]).double()
    ph = torch.cat([ph, ph]).to(DEV)[None]
    return ph.cos().half(), ph.sin().half()     # (1, hd), as a Llama model hands them over


def _pad_mask(case, seed):
    """(B, 1, 1, keys) boolean, True = attend: rows padded on the left by up to
    a quarter of the prompt."""
    B, n = case["batch"], case["tokens"] + case["stream"]
    pad = torch.randint(0, case["tokens"] // 4, (B,), generator=_gen(seed, 7777), device=DEV)
    pad[0] = 0
    return (torch.arange(n, device=DEV)[None] >= pad[:, None])[:, None, None]


def _prefill_kv(case, seed):
    """Post-RoPE keys with an exponential spectrum and unit variance, values
    with two outlier channels: fp16 (B, G, T, hd)."""
    g = _gen(seed, 1)
    B, G, T, hd = case["batch"], case["n_kv"], case["tokens"], case["hd"]
    p = G * hd
    w, _ = torch.linalg.qr(_randn(g, p, p))
    sigma = torch.exp(-torch.arange(p, device=DEV) * (math.log(100.0) / 384))
    mix = sigma[:, None] * w.T
    mix = mix / mix.pow(2).sum(0).sqrt()
    k = torch.empty(B, G, T, hd, dtype=torch.float16, device=DEV)
    v = torch.empty_like(k)
    ph = torch.arange(T, device=DEV).float()[:, None] * _inv_freq(hd).to(DEV)[None]
    cos, sin = ph.cos(), ph.sin()
    shift = _randn(g, p) * MEAN_STD
    outliers = torch.randperm(p, generator=g, device=DEV)[:2]
    for b in range(B):
        x = (_randn(g, T, p) @ mix + shift).view(T, G, hd).transpose(0, 1)
        lo, hi = x[..., : hd // 2], x[..., hd // 2:]
        k[b] = torch.cat([lo * cos - hi * sin, hi * cos + lo * sin], -1).half()
        y = _randn(g, T, p)
        y[:, outliers] *= 8.0
        v[b] = y.view(T, G, hd).transpose(0, 1).half()
    return k, v


def _fixed_basis(case, seed):
    g = _gen(seed, 2)
    p = case["n_kv"] * case["hd"]
    w, _ = torch.linalg.qr(_randn(g, p, case["rank"]))
    return w.t().contiguous().half()            # (rank, p)


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def _stream_buffers(case, raw, room):
    """The stream so far in the cache's buffers, with `room` rows to spare."""
    from shard_amd import ops
    s, cb = case["stream"], _stream_codebook(case["hd"]).to(DEV)
    bufs = {"signs": raw["signs"], "stream_codebook": cb, "stream_bits": STREAM_BITS}
    for name in "kv":
        x = raw["stream_" + name]
        rows = {"idx": torch.zeros(s + room, *x.shape[1:], dtype=torch.uint8, device=DEV),
                "norm": torch.zeros(s + room, *x.shape[1:-1], dtype=torch.float16, device=DEV),
                "deq": torch.zeros(s + room, *x.shape[1:], dtype=torch.float16, device=DEV)}
        if s:
            idx, norm, deq = ops.stream_quant(x, raw["signs"], cb, with_deq=True)
            rows["idx"][:s], rows["norm"][:s], rows["deq"][:s] = idx, norm, deq
        bufs.update({f"{name}_{part}_buf": t for part, t in rows.items()})
    bufs["_stream_cap"] = s + room
    bufs["stream_n"] = s * case["batch"]
    return bufs


def _device_layer(case, raw, stream=True):
    from shard_amd.cache import finalize_format
    fmt = raw["fmt"]
    finalize_format(fmt, _inv_freq(case["hd"]), torch.device(DEV))
    if stream:
        fmt.update(_stream_buffers(case, raw, 1))
    return fmt


def _cache_of(case, layers):
    from shard_amd import Cache
    cache = Cache(head_dim=case["hd"], num_layers=len(layers), n_kv_heads=case["n_kv"], device=DEV,
                  rope_inv_freq=_inv_freq(case["hd"]))
    for layer, fmt in zip(cache.layers, layers):
        layer._gpu_compressed = fmt
        layer._needs_decompress = True
        layer._seq_len = case["tokens"] + case["stream"]
    cache._compressed = True
    return cache


def _prepare_step(case, seed):
    from shard_amd import ops
    B, H, G, hd, s, L = (case[k] for k in ("batch", "n_q", "n_kv", "hd", "stream", "layers"))
    rows = torch.tensor([s, s + 1], dtype=torch.int32, device=DEV)
    pos = torch.tensor([_position(case)], dtype=torch.int64, device=DEV)
    cos, sin = _cos_sin(case)
    out = torch.zeros(L, B, H, hd, dtype=torch.float16, device=DEV)
    q_rope = torch.zeros_like(out)
    layers = []
    for li in range(L):
        raw = _raw_layer(case, seed, li)
        fmt = _device_layer(case, raw)
        call = ops.make_decode_args(q_rope[li], fmt, pos, None, out=out[li], stream_n=s + 1,
                                    stream_n_dev=rows[1:2])
        layers.append((fmt, call, raw["q"].view(B, H, hd), raw["k"].view(B, G, hd), raw["v"].view(B, G, hd)))
    ws = torch.zeros(max(ops.decode_workspace_bytes(c[1]) for c in layers), dtype=torch.uint8, device=DEV)

    def token():
        for li, (fmt, call, q, k, v) in enumerate(layers):
            base = [fmt[n].data_ptr() for n in ("k_idx_buf", "k_norm_buf", "k_deq_buf",
                                                "v_idx_buf", "v_norm_buf", "v_deq_buf")]
            ops.rope_stream_append_at(q, k, v, cos, sin, fmt["signs"], fmt["stream_codebook"], q_rope[li],
                                      *base, row_dev=rows[0:1], row_cap=s + 1)
            ops.decode_attn(call, ws, allocate=False)

    token()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        token()
    results = {"out": out, "q": q_rope}
    for part in ("k_idx", "k_norm", "k_deq", "v_idx", "v_norm", "v_deq"):
        results[part] = [fmt[part + "_buf"][s] for fmt, *_ in layers[:4]]
    return {"graph": graph, "results": results, "keep": (layers, ws, rows, pos, cos, sin)}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _prepare_step(case, seed)
    if kind == "attend":
        raw = _raw_layer(case, seed, 0)
        fmt = _device_layer(case, raw, stream=not case["masked"])
        if case["masked"]:
            fmt["decode_k"] = raw["stream_k"].permute(1, 2, 0, 3).contiguous()
            fmt["decode_v"] = raw["stream_v"].permute(1, 2, 0, 3).contiguous()
        cache = _cache_of(case, [fmt])
        cache._streaming = not case["masked"]
        cos, sin = _cos_sin(case)
        return {"case": case, "cache": cache, "fmt": fmt, "q": raw["q"], "k": raw["k"], "v": raw["v"],
                "cos": cos[None], "sin": sin[None],
                "pos": torch.tensor([_position(case)], dtype=torch.int64, device=DEV),
                "mask": _pad_mask(case, seed) if case["masked"] else None}
    if kind == "rebuild":
        layers = [_device_layer(case, _raw_layer(case, seed, li), stream=case["stream"] > 0)
                  for li in range(case["layers"])]
        return {"case": case, "cache": _cache_of(case, layers)}
    k, v = _prefill_kv(case, seed)
    if kind == "compress":
        return {"case": case, "k": k, "v": v}
    from shard_amd import ops
    B, G, T, hd = k.shape
    x, _, _ = ops.vq_prepare(v.view(B * G, T, hd))
    codebook = x[torch.randperm(x.shape[0], generator=_gen(seed, 3), device=DEV)[:256]].contiguous()
    return {"case": case, "k": k, "v": v, "basis": ops.rope_basis(_fixed_basis(case, seed)),
            "bits": torch.full((case["rank"],), 4, dtype=torch.int32, device=DEV),
            "phases": ops.rope_phases(0, T, _inv_freq(hd).to(DEV)), "table": ops.VqTable(codebook)}


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["results"]
    from shard_amd import fused_attention_compressed, ops
    case = state["case"]
    if case["kind"] == "attend":
        layer, fmt = state["cache"].layers[0], state["fmt"]
        inv = state["cache"]._rope_inv_freq
        if case["masked"]:
            return {"out": fused_attention_compressed(state["q"], layer, state["pos"], inv, state["mask"])}
        fmt["stream_n"] = case["stream"] * case["batch"]     # the same token again
        q = layer.fused_rope_append(state["q"], state["k"], state["v"], state["cos"], state["sin"]).unsqueeze(2)
        out = {"out": fused_attention_compressed(q, layer, state["pos"], inv), "q": q}
        for part in ("k_idx", "k_norm", "k_deq", "v_idx", "v_norm", "v_deq"):
            out[part] = fmt[part + "_buf"][case["stream"]]
        return out
    if case["kind"] == "rebuild":      # each access evicts the layer read before it
        return [(layer.keys, layer.values) for layer in state["cache"].layers]
    if case["kind"] == "encode":
        k, v = state["k"], state["v"]
        B, G, T, hd = v.shape
        coded = ops.int4_quant_pack(ops.pca_project_rope(k, 0, T, state["phases"], state["basis"]), state["bits"])
        vr = v.view(B * G, T, hd)
        ch, ch16, rcp = ops.vq_scales(vr)
        return {**coded, "ch": ch, "ch16": ch16, "v_idx": ops.vq_encode_table(vr, ch, rcp, state["table"])}
    from shard_amd import Cache
    cache = Cache(head_dim=case["hd"], num_layers=1, n_kv_heads=case["n_kv"], device=DEV,
                  max_rank_k=case["rank"], rope_inv_freq=_inv_freq(case["hd"]))
    cache.layers[0].update(state["k"], state["v"])
    cache.compress()
    layer = cache.layers[0]
    return {"keys": layer.keys, "values": layer.values, "v_idx": layer._gpu_compressed["v_indices"],
            "v_ch": layer._gpu_compressed["v_ch_f16"], "k_mean": layer._gpu_compressed["k_mean_f16"]}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    B, G, hd, rank, T = case["batch"], case["n_kv"], case["hd"], case["rank"], case["tokens"]
    p, n = G * hd, B * (T - SINK - WIN)
    stored = rank / 2 + p / 4                    # bytes per compressed token
    tables = p * rank + 4 * rank + 2 * p + 2048 + 2 * p * B
    if case["kind"] in ("step", "attend"):
        extra = B * (SINK + WIN) * p * 4 + B * case["stream"] * (2 * p + 4 * G)
        if case.get("masked"):
            extra = B * (SINK + WIN + case["stream"]) * p * 4 + B * (T + case["stream"])
        io = 2 * 2 * B * case["n_q"] * hd + (8 * B * p if not case.get("masked") else 0)
        flops = n * (2 * p * rank + 5 * case["n_q"] * hd) + (B * (SINK + WIN + case["stream"])) * 4 * case["n_q"] * hd
        layers = case.get("layers", 1)
        return {"bytes": layers * (n * stored + tables + extra + io), "flops": layers * flops}
    if case["kind"] == "rebuild":
        rest = B * (SINK + WIN + case["stream"]) * p * 4
        return {"bytes": case["layers"] * (n * (stored + 4 * p) + tables + 2 * rest),
                "flops": case["layers"] * 2 * n * p * rank}
    if case["kind"] == "encode":
        n = B * T
        return {"bytes": n * (4 * p + rank / 2 + p) + p * rank * 2, "flops": 2 * n * p * rank}
    # compress: K and V once, V once more per k-means iteration; covariance,
    # projection and rebuild, a few operations per value and iteration
    return {"bytes": n * (4 * p + 30 * 2 * p + stored + 4 * p),
            "flops": n * (2 * p * p + 4 * p * rank + 30 * 12 * p)}


# ---------------------------------------------------------------------------
# tolerances and the 64-bit results
# ---------------------------------------------------------------------------
def tolerance(case):
    if case["kind"] in ("step", "attend"):
        # fp16 operands of the score and value products, fp16 output
        return {"rel": 2e-3, "max": 2e-2}
    if case["kind"] == "rebuild":
        # sums of fp16 products, rounded to fp16 before the mean and the rotation
        return {"rel": 2e-3, "max": 1e-2}
    if case["kind"] == "encode":
        # fp16 operands; sums in another order flip codes at ties only
        return {"rel": 3e-4, "max": 1e-2, "differ": 2e-3}
    # eigenvectors follow the rounding of the covariance, and codes flip with
    # them: summing the covariance in another order moves the keys by 8e-3
    return {"rel": 3e-2, "max": 0.9}


def _rope64(x, start, inv):
    """(.., T, hd) double rotated to positions start + t."""
    ph = (start + torch.arange(x.shape[-2], device=x.device)).double()[:, None] * inv.to(x.device).double()[None]
    c, s = ph.cos(), ph.sin()
    lo, hi = x.chunk(2, -1)
    return torch.cat([lo * c - hi * s, hi * c + lo * s], -1)


def _hadamard64(x):
    x = x.double()
    d = x.shape[-1]
    h = 1
    while h < d:
        y = x.view(*x.shape[:-1], d // (2 * h), 2, h)
        x = torch.stack([y[..., 0, :] + y[..., 1, :], y[..., 0, :] - y[..., 1, :]], -2).reshape(x.shape)
        h *= 2
    return x / math.sqrt(d)


def _coefficients64(fmt):
    b = fmt["k_coeffs"]
    nib = torch.stack([b & 15, b >> 4], -1).view(fmt["k_coeffs_shape"]).double() - 8
    return nib * fmt["k_coeff_scale"].double()


def _span64(fmt, hd):
    """K (RoPE applied) and V of the compressed span, (B, G, n, hd) double."""
    B, n, G = fmt["batch"], fmt["n_compress"], fmt["n_kv"]
    k = _coefficients64(fmt) @ fmt["k_basis_f16"].double().T + fmt["k_mean_f16"].double()
    k = _rope64(k.view(B, n, G, hd).transpose(1, 2), fmt["compress_start"], _inv_freq(hd))
    v = fmt["v_centroids_f16"].double()[fmt["v_indices"].long()].view(B, G, n, hd)
    return k, _hadamard64(v * fmt["v_ch_f16"].double()[:, :, None])


def _quantized64(x, signs, hd):
    """Stream tokens (.., hd) as stored: (norm, dequantized)."""
    x = x.double()
    norm = x.norm(dim=-1).clamp(min=1e-8)
    r = _hadamard64(x / norm[..., None] * signs.double())
    cb = _stream_codebook(hd).to(DEV).double()
    edges = (cb[1:] + cb[:-1]) / 2
    code = torch.bucketize(r, edges)
    return norm, _hadamard64(cb[code]) * signs.double() * norm.half().double()[..., None]


def _attention64(case, raw, mask=None):
    fmt, hd, B = raw["fmt"], case["hd"], case["batch"]
    cos, sin = (t.double() for t in _cos_sin(case))
    turn = lambda x: x * cos + torch.cat([-x[..., hd // 2:], x[..., : hd // 2]], -1) * sin
    q = raw["q"].double()
    ks, vs = [fmt["sink_k"].double()], [fmt["sink_v"].double()]
    k, v = _span64(fmt, hd)
    ks += [k, fmt["win_k"].double()]
    vs += [v, fmt["win_v"].double()]
    norms = rows = None
    if mask is None:
        q = turn(q)
        new = {"k": turn(raw["k"].double()), "v": raw["v"].double()}
        norms, rows = {}, {}
        for name, seg in (("k", ks), ("v", vs)):
            x = torch.cat([raw["stream_" + name].double(), new[name].permute(2, 0, 1, 3)], 0)
            norm, deq = _quantized64(x, raw["signs"], hd)
            norms[name], rows[name] = norm[-1], deq[-1]
            seg.append(deq.permute(1, 2, 0, 3))
    else:
        ks.append(raw["stream_k"].double().permute(1, 2, 0, 3))
        vs.append(raw["stream_v"].double().permute(1, 2, 0, 3))
    k, v = torch.cat(ks, 2), torch.cat(vs, 2)
    out = torch.empty_like(q)
    per = case["n_q"] // case["n_kv"]
    for g in range(case["n_kv"]):
        sc = q[:, g * per:(g + 1) * per, 0] @ k[:, g].transpose(1, 2).contiguous() / math.sqrt(hd)
        if mask is not None:
            sc = sc.masked_fill(~mask[:, 0], -math.inf)
        out[:, g * per:(g + 1) * per, 0] = sc.softmax(-1) @ v[:, g].contiguous()
    return out, q, norms, rows


def _allocation(var, budget):
    """Bits per component: groups of 64 get 0/2/4/6/8 bits, 64 b / 16 units
    each, at most budget // 16 + 1 units, least total error."""
    groups = [float(v.sum()) for v in var.split(64)]
    sizes = [len(v) for v in var.split(64)]
    best = None
    for bits in itertools.product((0, 2, 4, 6, 8), repeat=len(groups)):
        if sum(-(-s * b // 16) for s, b in zip(sizes, bits)) > budget // 16 + 1:
            continue
        err = sum(v * 4 if b == 0 else v / (3 * 4 ** b) for v, b in zip(groups, bits))
        if best is None or err < best[0]:
            best = (err, bits)
    return [b for s, b in zip(sizes, best[1]) for _ in range(s)]


def _compress64(case, k, v):
    B, G, T, hd = k.shape
    p, n = G * hd, T - SINK - WIN
    inv = _inv_freq(hd)
    x = _rope64(k[:, :, SINK:SINK + n].double(), SINK, -inv).transpose(1, 2).reshape(B * n, p)
    mean = x.mean(0)
    x -= mean
    val, vec = torch.linalg.eigh((x.T @ x / (B * n)).cpu())
    rank = min(case["rank"], p, B * n - 1)
    basis, var = vec.flip(1)[:, :rank].to(DEV), val.flip(0)[:rank].clamp(min=0)
    bits = _allocation(var, max(64, p * 16 // 20))
    bits = [b for b in bits if b]
    keep = len(bits)
    basis = basis[:, :keep]
    scale = basis.abs().amax(0).clamp(min=1e-6) / 127
    basis_q = (basis / scale).round().clamp(-127, 127)
    proj = x @ (basis_q * scale)
    lo, hi = proj.amin(0), proj.amax(0)
    rng = (hi - lo).clamp(min=1e-6)
    levels = torch.tensor([2.0 ** b - 1 for b in bits], device=DEV, dtype=torch.float64)
    y = ((proj - lo) / rng * levels).round() / levels * rng + lo
    cs = y.abs().amax(0).clamp(min=1e-6) / 7
    coef = (y / cs).round().clamp(-7, 7) * cs.half().double()
    rebuilt = coef @ (basis_q * scale.half().double()).T + mean.half().double()
    mid = _rope64(rebuilt.view(B, n, G, hd).transpose(1, 2), SINK, inv)
    keys = torch.cat([k[:, :, :SINK].double(), mid, k[:, :, SINK + n:].double()], 2)
    ch = _hadamard64(v[:, :, SINK:SINK + n]).abs().amax(2)
    return {"keys": keys, "values": None, "v_idx": None, "v_ch": ch, "k_mean": mean}


def exact(case, seed):
    kind = case["kind"]
    hd, G, B = case["hd"], case["n_kv"], case["batch"]
    if kind == "step":
        outs, qs, norms, rows = zip(*(_attention64(case, _raw_layer(case, seed, li)) for li in range(case["layers"])))
        res = {"out": torch.stack(outs)[:, :, :, 0], "q": torch.stack(qs)[:, :, :, 0], "k_idx": None, "v_idx": None}
        for name in "kv":
            res[name + "_norm"] = [x[name] for x in norms[:4]]
            res[name + "_deq"] = [x[name] for x in rows[:4]]
        return res
    if kind == "attend":
        raw = _raw_layer(case, seed, 0)
        if case["masked"]:
            return {"out": _attention64(case, raw, _pad_mask(case, seed))[0]}
        out, q, norms, rows = _attention64(case, raw)
        return {"out": out, "q": q, "k_idx": None, "v_idx": None, "k_norm": norms["k"], "v_norm": norms["v"],
                "k_deq": rows["k"], "v_deq": rows["v"]}
    if kind == "rebuild":
        res = []
        for li in range(case["layers"]):
            raw = _raw_layer(case, seed, li)
            fmt = raw["fmt"]
            k, v = _span64(fmt, hd)
            parts = {"k": [fmt["sink_k"].double(), k, fmt["win_k"].double()],
                     "v": [fmt["sink_v"].double(), v, fmt["win_v"].double()]}
            for name in "kv":
                if case["stream"]:
                    parts[name].append(_quantized64(raw["stream_" + name], raw["signs"], hd)[1].permute(1, 2, 0, 3))
            res.append((torch.cat(parts["k"], 2), torch.cat(parts["v"], 2)))
        return res
    k, v = _prefill_kv(case, seed)
    if kind == "compress":
        return _compress64(case, k, v)
    T = case["tokens"]
    x = _rope64(k.double(), 0, -_inv_freq(hd)).transpose(1, 2).reshape(B * T, G * hd)
    proj = x @ _fixed_basis(case, seed).double().T
    lo, hi = proj.amin(0), proj.amax(0)
    ch = _hadamard64(v.view(B * G, T, hd)).abs().amax(1)
    # a column's largest quantized magnitude is that of one of its two ends
    return {"packed": None, "coeff_scale": torch.maximum(lo.abs(), hi.abs()) / 7, "lo": lo, "rng": hi - lo,
            "ch": ch, "ch16": ch, "v_idx": None}
