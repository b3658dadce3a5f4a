"""Performance cases of the KV-cache path: what a decoding or serving program asks of it.

Every case runs the public entry points of ``atomflow_amd.kv`` on the Llama-3.2-3B-shaped layer of
the benchmark (24 query heads, 8 KV heads, head_dim 128, MLP width 8192) or on the same layer with
16 or 32 query heads. Kinds:

* ``decode``  a batch-1 token step, captured in a graph over all layers: QKV projection + RoPE +
              append, then attention over the contiguous cache;
* ``serve``   a paged decode batch of one layer: batched QKV projection + RoPE + append, then
              attention through the block tables, fp16 or FP8 pool; with ``prefix`` the sequences
              are forks of one prompt and take the shared-prefix form;
* ``prompt``  the attention block of a prompt chunk on the contiguous cache: QKV projection,
              RoPE + append, causal attention, output projection;
* ``attend``  causal attention alone, of a chunk whose rows are in the cache already;
* ``chunks``  a serving step's prefill chunks of several sequences through the paged pool: fused
              QKV projection + append, then one batched causal attention launch;
* ``mlp``     the gate, up and down projections of m tokens (m = 1: the graph of every layer).
"""
import math

import numpy as np
import torch

import atomflow_amd
from atomflow_amd import device, kv

HD = 128
NKV = 8
KV_DIM = NKV * HD
THETA = 500000.0
GROUP_SIZE = 128
FP8_MAX = 448.0


def listed():
    return [
        # One chat user, short context: 56 small launches a token, latency and gaps count.
        {"name": "decode_ctx1k", "kind": "decode", "ctx": 1024, "layers": 28, "nq": 24},
        # The benchmark's headline step: one user at 8k context, 28 layers.
        {"name": "decode_ctx8k", "kind": "decode", "ctx": 8192, "layers": 28, "nq": 24},
        # A long document: the cache read dominates (8 of the layers, the state stays small).
        {"name": "decode_ctx32k", "kind": "decode", "ctx": 32768, "layers": 8, "nq": 24},
        # Continuous batching, mixed lengths, 16-token blocks.
        {"name": "serve_b32", "kind": "serve", "batch": 32, "lo": 128, "hi": 8192, "fp8": False,
         "block": 16, "prefix": 0, "nq": 24},
        # The large long-context batch over an FP8 pool.
        {"name": "serve_b128_fp8", "kind": "serve", "batch": 128, "lo": 8192, "hi": 16384,
         "fp8": True, "block": 32, "prefix": 0, "nq": 24},
        # 64 samples of one 2048-token prompt, each with its own continuation.
        {"name": "forks_b64", "kind": "serve", "batch": 64, "lo": 1, "hi": 1024, "fp8": False,
         "block": 16, "prefix": 2048, "nq": 24},
        # A whole 2k prompt in one chunk (time to first token).
        {"name": "prompt_2k", "kind": "prompt", "p0": 0, "n": 2048, "nq": 24},
        # The attention of a 16k prompt: the largest causal launch.
        {"name": "attend_16k", "kind": "attend", "p0": 0, "n": 16384, "nq": 24},
        # A serving step's chunked prefill: five sequences, ragged chunks at ragged positions.
        {"name": "chunks_5", "kind": "chunks", "count": 5, "n": 512, "hi": 6144, "fp8": False,
         "block": 16, "nq": 24},
        # The MLP of one decoded token, every layer's weights streamed from HBM.
        {"name": "mlp_token", "kind": "mlp", "m": 1, "dim": 3072, "hidden": 8192, "layers": 28},
        # The MLP of a decode batch that is not a multiple of any tile.
        {"name": "mlp_b45", "kind": "mlp", "m": 45, "dim": 3072, "hidden": 8192, "layers": 1},
        # The MLP of a prefill step's tokens (decode rows and chunks together, ragged).
        {"name": "mlp_2011", "kind": "mlp", "m": 2011, "dim": 3072, "hidden": 8192, "layers": 1},
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "serve", "serve", "prompt", "attend", "chunks", "mlp", "mlp"])
    nq = rng.choice([16, 24, 24, 32])
    if kind == "decode":
        return {"kind": kind, "ctx": _log(rng, 64, 32768), "layers": 8, "nq": nq}
    if kind == "serve":
        fp8 = rng.random() < 0.5
        prefix = rng.choice([0, 0, 32 * _log(rng, 8, 128)])
        hi = _log(rng, 64, 1024 if prefix else 12288)
        return {"kind": kind, "batch": _log(rng, 2, 96), "lo": max(1, hi // 16), "hi": hi, "fp8": fp8,
                "block": rng.choice([16, 32]), "prefix": prefix, "nq": nq}
    if kind == "prompt":
        return {"kind": kind, "p0": rng.choice([0, _log(rng, 16, 6144)]), "n": _log(rng, 17, 4096),
                "nq": nq}
    if kind == "attend":
        return {"kind": kind, "p0": rng.choice([0, _log(rng, 16, 8192)]), "n": _log(rng, 64, 12288),
                "nq": rng.choice([16, 24])}
    if kind == "chunks":
        return {"kind": kind, "count": rng.randint(2, 8), "n": _log(rng, 64, 512),
                "hi": _log(rng, 64, 8192), "fp8": rng.random() < 0.5, "block": rng.choice([16, 32]),
                "nq": nq}
    dim, hidden = rng.choice([(3072, 8192), (2048, 8192), (4096, 14336)])
    return {"kind": kind, "m": _log(rng, 2, 2048), "dim": dim, "hidden": hidden, "layers": 1}


# ---- inputs -----------------------------------------------------------------------------------


def _generator(seed, salt=0):
    return torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + salt)


def _weight(n, k, gen):
    """[n, k] E4M3 codes and [n, k / 128] fp16 scales of N(0, 1/k) weights, absmax scaled."""
    w = torch.randn(n, k // GROUP_SIZE, GROUP_SIZE, device="cuda", generator=gen) / math.sqrt(k)
    scale = w.abs().amax(dim=2, keepdim=True) / FP8_MAX
    codes = (w / scale).clamp(-FP8_MAX, FP8_MAX).to(torch.float8_e4m3fn).view(torch.uint8)
    return codes.reshape(n, k), scale.reshape(n, -1).half()


def _rope_tables(rows):
    inv = THETA ** (-torch.arange(0, HD, 2, dtype=torch.float64, device="cuda") / HD)
    angle = torch.arange(rows, dtype=torch.float64, device="cuda")[:, None] * inv
    return angle.cos().float(), angle.sin().float()


def _fill_rows(t, gen, scales=None):
    """N(0,1) cache rows [..., KV_DIM], in place; FP8 pools hold codes under per-head scales
    [K, V][kv_head] of the two outer slabs of t."""
    if scales is None:
        for part in t.reshape(-1).split(1 << 27):
            part.copy_(torch.randn(part.numel(), device="cuda", generator=gen))
        return
    for slab in (0, 1):
        for part in t[slab].reshape(-1, NKV, HD).split(1 << 16):
            x = torch.randn(part.shape, device="cuda", generator=gen) / scales[slab][:, None]
            part.copy_(x.clamp(-FP8_MAX, FP8_MAX).to(torch.float8_e4m3fn).view(torch.uint8))


def _lengths(case, gen):
    """Rows of each sequence (past the shared prefix): evenly spread over [lo, hi], in any order."""
    b, lo, hi = case["batch"], case["lo"], case["hi"]
    i = torch.randperm(b, device="cuda", generator=gen)
    return lo + ((hi - lo) * (2 * i + 1)) // (2 * b)


def _chunk_list(case, seed):
    """(p0, n, kv_len, first row) of each chunk: start positions evenly spread over [0, hi], in any
    order; the last chunk is a prompt's ragged end, the others n tokens."""
    count, n, hi = case["count"], case["n"], case["hi"]
    out, row = [], 0
    for i, j in enumerate(np.random.default_rng([int(seed), 7]).permutation(count)):
        p0, rows = hi * (2 * int(j) + 1) // (2 * count), n if i + 1 < count else n - n // 3
        out.append((p0, rows, p0 + rows, row))
        row += rows
    return out


class State:
    """Buffers, weights, plans and (for graph cases) the captured step of one case."""

    graph = stream = None

    def __del__(self):
        try:
            if self.graph is not None:
                device.synchronize()
                self.graph.destroy()
                self.stream.destroy()
        except Exception:
            pass


def _empty(*shape, dtype=torch.float16):
    return torch.zeros(*shape, device="cuda", dtype=dtype)


def _stream():
    return torch.cuda.current_stream().cuda_stream


def prepare(case, seed):
    s = State()
    s.case = case
    {"decode": _prepare_decode, "serve": _prepare_serve, "prompt": _prepare_prompt,
     "attend": _prepare_attend, "chunks": _prepare_chunks, "mlp": _prepare_mlp}[case["kind"]](
         s, case, seed)
    return s


def _prepare_layer(s, case, seed, layers, m):
    """QKV weights of `layers` layers and m input rows each."""
    s.nq, s.dim = case["nq"], case["nq"] * HD
    s.qkv_dim = s.dim + 2 * KV_DIM
    gen = _generator(seed, 1)
    s.x = torch.randn(layers, m, s.dim, device="cuda", generator=gen).half()
    s.w = [_weight(s.qkv_dim, s.dim, gen) for _ in range(layers)]
    s.qkv = _empty(layers, m, s.qkv_dim)
    s.out = _empty(layers, m, s.dim)


def _capture(s, body):
    torch.cuda.synchronize()
    s.stream = device.Stream()
    s.graph = device.Graph.capture(s.stream, lambda: body(s.stream))


def _prepare_decode(s, case, seed):
    layers, pos = case["layers"], case["ctx"]
    _prepare_layer(s, case, seed, layers, 1)
    s.rows = (pos + 64) // 64 * 64
    s.cache = _empty(layers, 2, s.rows, KV_DIM)
    _fill_rows(s.cache, _generator(seed, 2))
    s.cos, s.sin = _rope_tables(s.rows)
    s.pos = torch.tensor([pos], device="cuda", dtype=torch.int32)
    s.len = s.pos + 1
    s.ws = kv.AttentionWorkspace(1, s.nq, NKV, HD)

    def body(stream):
        for l in range(layers):
            k, v = s.cache[l, 0].data_ptr(), s.cache[l, 1].data_ptr()
            kv.launch_qkv_rope_append(
                s.x[l].data_ptr(), s.w[l][0].data_ptr(), s.w[l][1].data_ptr(), s.dim,
                s.qkv[l].data_ptr(), k, v, s.cos.data_ptr(), s.sin.data_ptr(), 0, s.rows, s.nq, NKV,
                HD, GROUP_SIZE, d_pos=s.pos.data_ptr(), stream=stream)
            kv.launch_cached_attention_ex(s.qkv[l].data_ptr(), k, v, s.out[l].data_ptr(), 0, s.rows,
                                          HD, s.nq, NKV, s.ws, d_seq_len=s.len.data_ptr(),
                                          stream=stream)

    _capture(s, body)


def _paged_pool(s, case, seed, blocks):
    """One layer's pool of `blocks` blocks, values N(0, 1)."""
    gen, bs = _generator(seed, 2), case["block"]
    s.scales = None
    if case["fp8"]:  # absmax / 448 of N(0,1) rows, one scale per (K or V, KV head)
        s.scales = (4.5 + torch.rand(2, NKV, device="cuda", generator=gen)) / FP8_MAX
    s.pool_mem = _empty(2, blocks * bs, KV_DIM,
                        dtype=torch.uint8 if case["fp8"] else torch.float16)
    _fill_rows(s.pool_mem, gen, s.scales)
    s.pool = kv.make_pool(
        s.pool_mem.data_ptr(),
        atomflow_amd.AF_KV_FP8_E4M3 if case["fp8"] else atomflow_amd.AF_KV_FP16, bs, 1, NKV, HD,
        blocks, None if s.scales is None else s.scales.data_ptr(),
        flags=atomflow_amd.AF_KV_POOL_SHARED_BLOCKS if case.get("prefix") else 0)


def _prepare_serve(s, case, seed):
    b, bs, prefix = case["batch"], case["block"], case["prefix"]
    _prepare_layer(s, case, seed, 1, b)
    gen = _generator(seed, 3)
    own = _lengths(case, gen)
    s.lens = (prefix + own).int()
    s.max_len = prefix + case["hi"]
    shared = prefix // bs  # prefixes are whole blocks: no sequence holds a copied tail
    s.max_blocks = -(-s.max_len // bs)
    need = -(-s.lens.long() // bs) - shared
    blocks = shared + int(need.sum())
    perm = torch.randperm(blocks, device="cuda", generator=gen).int()
    s.tables = _empty(b, s.max_blocks, dtype=torch.int32)
    s.tables[:, :shared] = perm[:shared]
    first = shared + torch.cumsum(need, 0) - need
    col = torch.arange(s.max_blocks - shared, device="cuda")
    mine = col[None, :] < need[:, None]
    s.tables[:, shared:][mine] = perm[(first[:, None] + col[None, :])[mine]]
    s.positions = s.lens - 1
    p = s.positions.long()
    tail = s.tables.gather(1, (p // bs)[:, None])[:, 0].long()
    s.slots = tail * bs + p % bs
    _paged_pool(s, case, seed, blocks)
    s.cos, s.sin = _rope_tables(s.max_len)
    s.ws = kv.AttentionWorkspace(b, s.nq, NKV, HD)


def _prepare_prompt(s, case, seed):
    p0, n = case["p0"], case["n"]
    _prepare_layer(s, case, seed, 1, n)
    s.wo = _weight(s.dim, s.dim, _generator(seed, 4))
    s.y = _empty(n, s.dim)
    s.rows = p0 + n
    s.cache = _empty(2, s.rows, KV_DIM)
    _fill_rows(s.cache, _generator(seed, 2))
    s.cos, s.sin = _rope_tables(s.rows)
    s.ws = kv.PrefillWorkspace(p0, n, p0 + n, s.nq)


def _prepare_attend(s, case, seed):
    p0, n = case["p0"], case["n"]
    s.nq, s.dim = case["nq"], case["nq"] * HD
    s.rows = p0 + n
    s.q = torch.randn(n, s.dim, device="cuda", generator=_generator(seed, 1)).half()
    s.cache = _empty(2, s.rows, KV_DIM)
    _fill_rows(s.cache, _generator(seed, 2))
    s.out = _empty(n, s.dim)
    s.ws = kv.PrefillWorkspace(p0, n, p0 + n, s.nq)


def _prepare_chunks(s, case, seed):
    chunks, bs = _chunk_list(case, seed), case["block"]
    s.m = chunks[-1][3] + chunks[-1][1]
    _prepare_layer(s, case, seed, 1, s.m)
    need = [-(-(c[0] + case["n"]) // bs) for c in chunks]  # room for whole chunks
    s.max_blocks = max(need)
    blocks = sum(need)
    perm = torch.randperm(blocks, device="cuda", generator=_generator(seed, 3)).int()
    s.tables = _empty(len(chunks), s.max_blocks, dtype=torch.int32)
    slots, positions, at = [], [], 0
    for i, (p0, n, kv_len, _) in enumerate(chunks):
        s.tables[i, :need[i]] = perm[at:at + need[i]]
        at += need[i]
        pos = torch.arange(p0, kv_len, device="cuda")
        slots.append(s.tables[i].long()[pos // bs] * bs + pos % bs)
        positions.append(pos)
    s.slots, s.positions = torch.cat(slots), torch.cat(positions).int()
    _paged_pool(s, case, seed, blocks)
    s.max_pos = max(c[2] for c in chunks)
    s.cos, s.sin = _rope_tables(s.max_pos)
    s.chunks = torch.tensor(chunks, device="cuda", dtype=torch.int32)
    entries, s.groups, s.most, nbytes = kv.prefill_piece_map(chunks, s.nq)
    s.entries = torch.from_numpy(entries).cuda()
    s.ws = kv.RecordWorkspace(nbytes)


def _prepare_mlp(s, case, seed):
    m, dim, hidden, layers = case["m"], case["dim"], case["hidden"], case["layers"]
    gen = _generator(seed, 1)
    s.x = torch.randn(layers, m, dim, device="cuda", generator=gen).half()
    s.h = torch.randn(layers, m, hidden, device="cuda", generator=gen).half()  # down's input
    s.w = [(_weight(hidden, dim, gen), _weight(hidden, dim, gen), _weight(dim, hidden, gen))
           for _ in range(layers)]
    s.gate, s.up, s.down = _empty(layers, m, hidden), _empty(layers, m, hidden), _empty(layers, m, dim)
    if m > 1:
        return

    def body(stream):
        for l, ((wg, sg), (wu, su), (wd, sd)) in enumerate(s.w):
            kv.launch_w8a16_gemv_pair(s.x[l].data_ptr(), wg.data_ptr(), sg.data_ptr(),
                                      s.gate[l].data_ptr(), hidden, wu.data_ptr(), su.data_ptr(),
                                      s.up[l].data_ptr(), hidden, dim, GROUP_SIZE, stream=stream)
            kv.launch_w8a16_gemv(s.h[l].data_ptr(), wd.data_ptr(), sd.data_ptr(),
                                 s.down[l].data_ptr(), dim, hidden, GROUP_SIZE, stream=stream)

    _capture(s, body)


# ---- one pass ---------------------------------------------------------------------------------


def run(s):
    return {"decode": _run_decode, "serve": _run_serve, "prompt": _run_prompt,
            "attend": _run_attend, "chunks": _run_chunks, "mlp": _run_mlp}[s.case["kind"]](s)


def _run_decode(s):
    s.graph.launch(_stream())
    pos = s.case["ctx"]
    return {"attn": s.out, "qkv": s.qkv, "rows": s.cache[:, :, pos], "cache": s.cache}


def _project(x, weight, y, m, n, k, stream):
    kv.launch_w8a16_gemm_batched(x.data_ptr(), k, m, weight[0].data_ptr(), weight[1].data_ptr(),
                                 y.data_ptr(), n, n, k, GROUP_SIZE, stream=stream)


def _project_append(s, m, max_pos, stream):
    kv.launch_paged_qkv_rope_append(
        s.x.data_ptr(), s.dim, m, s.w[0][0].data_ptr(), s.w[0][1].data_ptr(), s.dim,
        s.qkv.data_ptr(), s.pool, 0, s.slots.data_ptr(), s.positions.data_ptr(), s.cos.data_ptr(),
        s.sin.data_ptr(), max_pos, s.nq, GROUP_SIZE, stream=stream)


def _run_serve(s):
    stream, b, prefix = _stream(), s.case["batch"], s.case["prefix"]
    _project_append(s, b, s.max_len, stream)
    if prefix:
        kv.launch_paged_attention_shared_prefix(
            s.qkv.data_ptr(), s.qkv_dim, s.pool, 0, s.tables.data_ptr(), prefix,
            s.tables.data_ptr(), s.max_blocks, s.lens.data_ptr(), b, s.max_len, s.out.data_ptr(),
            s.dim, s.nq, s.ws, stream=stream)
    else:
        kv.launch_paged_attention(s.qkv.data_ptr(), s.qkv_dim, s.pool, 0, s.tables.data_ptr(),
                                  s.max_blocks, s.lens.data_ptr(), b, s.max_len, s.out.data_ptr(),
                                  s.dim, s.nq, s.ws, stream=stream)
    return {"attn": s.out, "qkv": s.qkv, "pool": s.pool_mem}


def _run_prompt(s):
    stream, p0, n = _stream(), s.case["p0"], s.case["n"]
    k, v = s.cache[0].data_ptr(), s.cache[1].data_ptr()
    _project(s.x, s.w[0], s.qkv, n, s.qkv_dim, s.dim, stream)
    kv.launch_prefill_rope_append(s.qkv.data_ptr(), n, k, v, s.cos.data_ptr(), s.sin.data_ptr(), p0,
                                  s.rows, s.nq, NKV, HD, stream=stream)
    kv.launch_prefill_attention_ws(s.qkv.data_ptr(), s.qkv_dim, k, v, s.out.data_ptr(), s.dim, p0, n,
                                   p0 + n, s.rows, s.nq, NKV, HD, s.ws, stream=stream)
    _project(s.out, s.wo, s.y, n, s.dim, s.dim, stream)
    return {"y": s.y, "attn": s.out, "qkv": s.qkv, "cache": s.cache}


def _run_attend(s):
    p0, n = s.case["p0"], s.case["n"]
    kv.launch_prefill_attention_ws(s.q.data_ptr(), s.dim, s.cache[0].data_ptr(),
                                   s.cache[1].data_ptr(), s.out.data_ptr(), s.dim, p0, n, p0 + n,
                                   s.rows, s.nq, NKV, HD, s.ws, stream=_stream())
    return {"attn": s.out}


def _run_chunks(s):
    stream = _stream()
    _project_append(s, s.m, s.max_pos, stream)
    kv.launch_paged_prefill_attention_batched_ws(
        s.qkv.data_ptr(), s.qkv_dim, s.pool, 0, s.tables.data_ptr(), s.max_blocks,
        s.chunks.data_ptr(), s.entries.data_ptr(), s.entries.shape[0], s.groups, s.most,
        s.out.data_ptr(), s.dim, s.nq, s.ws, stream=stream)
    return {"attn": s.out, "qkv": s.qkv, "pool": s.pool_mem}


def _run_mlp(s):
    m, dim, hidden = s.case["m"], s.case["dim"], s.case["hidden"]
    stream = _stream()
    if m == 1:
        s.graph.launch(stream)
    else:
        gate, up, down = s.w[0]
        _project(s.x, gate, s.gate, m, hidden, dim, stream)
        _project(s.x, up, s.up, m, hidden, dim, stream)
        _project(s.h, down, s.down, m, dim, hidden, stream)
    return {"gate": s.gate, "up": s.up, "down": s.down}


# ---- what a pass cannot do without ------------------------------------------------------------


def _weight_bytes(n, k):
    return n * k + 2 * n * (k // GROUP_SIZE)


def _causal(p0, n):
    """Attended (query, key) pairs of a chunk."""
    return n * p0 + n * (n + 1) // 2


def work(case):
    """Bytes: weights, attended rows, inputs and outputs once. Flops: 2 per product and sum."""
    kind = case["kind"]
    if kind == "mlp":
        m, dim, hidden = case["m"], case["dim"], case["hidden"]
        w = 2 * _weight_bytes(hidden, dim) + _weight_bytes(dim, hidden)
        return {"bytes": case["layers"] * (w + 2 * m * (2 * dim + 3 * hidden)),
                "flops": case["layers"] * 6.0 * m * dim * hidden}
    dim = case["nq"] * HD
    qkv = dim + 2 * KV_DIM
    if kind == "decode":
        l, rows = case["layers"], case["ctx"] + 1
        return {"bytes": l * (_weight_bytes(qkv, dim) + 4 * KV_DIM * rows + 2 * (2 * dim + qkv)),
                "flops": l * (2.0 * qkv * dim + 4.0 * dim * rows)}
    elem = 1 if case.get("fp8") else 2
    if kind == "serve":
        b, mean = case["batch"], (case["lo"] + case["hi"]) / 2
        rows = case["prefix"] + b * mean
        return {"bytes": _weight_bytes(qkv, dim) + 2 * KV_DIM * elem * rows + 2 * b * (2 * dim + qkv),
                "flops": b * (2.0 * qkv * dim + 4.0 * dim * (case["prefix"] + mean))}
    if kind == "chunks":
        count, n, p0 = case["count"], case["n"], case["hi"] / 2
        m = count * n - n // 3
        return {"bytes": _weight_bytes(qkv, dim) + 2 * KV_DIM * elem * (count * p0 + m) +
                2 * m * (2 * dim + qkv),
                "flops": 2.0 * m * qkv * dim + 4.0 * dim * (m * p0 + count * n * n / 2)}
    p0, n = case["p0"], case["n"]
    attend = {"bytes": 4 * KV_DIM * (p0 + n) + 4 * n * dim, "flops": 4.0 * dim * _causal(p0, n)}
    if kind == "attend":
        return attend
    return {"bytes": _weight_bytes(qkv, dim) + _weight_bytes(dim, dim) + attend["bytes"] +
            2 * n * (2 * dim + qkv),
            "flops": attend["flops"] + 2.0 * n * dim * (qkv + dim)}


def tolerance(case):
    """fp16 results of fp32 sums: about four times what a pass differs from 64-bit arithmetic by.
    The projections round once; attention also rounds its probabilities to fp16, and a block
    rounds between its stages. FP8 pools quantise the appended rows, where a value on a rounding
    boundary may take the neighbouring code."""
    if case["kind"] == "mlp":
        return {"rel": 1e-3, "max": 4e-3}
    if case.get("fp8"):
        return {"rel": 4e-3, "max": 4e-2, "differ": 1e-3}
    return {"rel": 3e-3, "max": 3e-2}


# ---- the same in 64 bits ----------------------------------------------------------------------


def _dequant(weight):
    codes, scales = weight
    n, k = codes.shape
    w = codes.view(torch.float8_e4m3fn).to(torch.float32).double().reshape(n, -1, GROUP_SIZE)
    return (w * scales.double()[:, :, None]).reshape(n, k)


def _rotate(x, cos, sin):
    """RoPE of [m, heads, HD] at the given table rows, pairs (d, d + HD / 2)."""
    c, s = cos.double()[:, None], sin.double()[:, None]
    a, b = x[..., :HD // 2], x[..., HD // 2:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _project_rope(s, l, pos):
    """(qkv with Q and K rotated, q, k, v) of layer l's input rows at positions pos."""
    qkv = s.x[l].double() @ _dequant(s.w[l]).T
    m = qkv.shape[0]
    heads = qkv.reshape(m, -1, HD)
    turned = _rotate(heads[:, :s.nq + NKV], s.cos[pos], s.sin[pos])
    v = heads[:, s.nq + NKV:]
    return (torch.cat([turned, v], 1).reshape(m, -1), turned[:, :s.nq], turned[:, s.nq:], v)


def _attend(q, k, v, lim=None):
    """[m, nq, HD] queries over [rows, NKV, HD] keys; query i sees keys below lim[i] (None: all)."""
    m, nq, _ = q.shape
    out = torch.empty_like(q)
    for h in range(nq):
        kh = h * NKV // nq
        for i in range(0, m, 4096):
            sc = q[i:i + 4096, h] @ k[:, kh].T / math.sqrt(HD)
            if lim is not None:
                sc.masked_fill_(torch.arange(k.shape[0], device="cuda") >= lim[i:i + 4096, None],
                                -math.inf)
            out[i:i + 4096, h] = torch.softmax(sc, -1) @ v[:, kh]
    return out.reshape(m, -1)


def _pool_rows(s, table, rows):
    """K and V rows [0, rows) of one block table, dequantised."""
    bs = s.case["block"]
    t = torch.arange(rows, device="cuda")
    slot = table.long()[t // bs] * bs + t % bs
    got = []
    for side in (0, 1):
        x = s.pool_mem[side][slot]
        if s.scales is not None:
            x = x.view(torch.float8_e4m3fn).float()
        x = x.double().reshape(rows, NKV, HD)
        got.append(x if s.scales is None else x * s.scales[side].double()[None, :, None])
    return got


def _stored(s, side, rows):
    """Appended rows as an FP8 pool holds them."""
    if s.scales is None:
        return rows
    sc = s.scales[side].double()[None, :, None]
    x = (rows / sc).clamp(-FP8_MAX, FP8_MAX).float().to(torch.float8_e4m3fn)
    return x.float().double() * sc


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "mlp":
        outs = [[], [], []]
        for l in range(case["layers"]):
            for o, x, w in zip(outs, (s.x[l], s.x[l], s.h[l]), s.w[l]):
                o.append(x.double() @ _dequant(w).T)
        return {k: torch.stack(o) for k, o in zip(("gate", "up", "down"), outs)}
    if kind == "attend":
        k, v = (c.double().reshape(-1, NKV, HD) for c in s.cache)
        lim = torch.arange(case["p0"] + 1, s.rows + 1, device="cuda")
        return {"attn": _attend(s.q.double().reshape(case["n"], s.nq, HD), k, v, lim)}
    if kind == "decode":
        pos = case["ctx"]
        attn, qkvs, rows = [], [], []
        for l in range(case["layers"]):
            qkv, q, kn, vn = _project_rope(s, l, s.pos.long())
            k, v = (torch.cat([s.cache[l, i, :pos].double().reshape(pos, NKV, HD), new])
                    for i, new in ((0, kn), (1, vn)))
            attn.append(_attend(q, k, v))
            qkvs.append(qkv)
            rows.append(torch.stack([kn.reshape(-1), vn.reshape(-1)]))
        return {"attn": torch.stack(attn), "qkv": torch.stack(qkvs), "rows": torch.stack(rows),
                "cache": None}
    if kind == "prompt":
        p0, n = case["p0"], case["n"]
        pos = torch.arange(p0, s.rows, device="cuda")
        qkv, q, kn, vn = _project_rope(s, 0, pos)
        k, v = (torch.cat([s.cache[i, :p0].double().reshape(p0, NKV, HD), new])
                for i, new in ((0, kn), (1, vn)))
        attn = _attend(q, k, v, pos + 1)
        return {"y": attn @ _dequant(s.wo).T, "attn": attn[None], "qkv": qkv[None],
                "cache": torch.stack([k.reshape(-1, KV_DIM), v.reshape(-1, KV_DIM)])}
    pos = s.positions.long()
    qkv, q, kn, vn = _project_rope(s, 0, pos)
    new = [_stored(s, i, x) for i, x in ((0, kn), (1, vn))]
    attn = torch.empty(q.shape[0], s.dim, dtype=torch.float64, device="cuda")
    if kind == "serve":
        for b, length in enumerate(s.lens.tolist()):
            k, v = _pool_rows(s, s.tables[b], length)
            k[-1], v[-1] = new[0][b], new[1][b]
            attn[b] = _attend(q[b:b + 1], k, v)[0]
    else:
        for i, (p0, n, kv_len, row) in enumerate(_chunk_list(case, seed)):
            k, v = _pool_rows(s, s.tables[i], kv_len)
            mine = slice(row, row + n)
            k[p0:], v[p0:] = new[0][mine], new[1][mine]
            attn[mine] = _attend(q[mine], k, v, pos[mine] + 1)
    return {"attn": attn[None], "qkv": qkv[None], "pool": None}
