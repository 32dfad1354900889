"""The workloads this library is timed on: one pass of each is what a serving loop enqueues for one token,
one chunk of a prompt or one batch of page moves, through the Python host layer (breccia_amd.kv.Pool).

A case is a dict of plain values.  `kind` says which part of the loop it is:

  decode   one token for every sequence of a batch, through all layers of the pool.  form "step" is the fused
           step (bkv_decode_step: append + attention in one call), form "kprep" the model's own order of calls
           (RMSNorm + rotary + append of the new K row, then dense attention with the output gate), form
           "select" the long-context order (pooled indexer key, block selection, append, attention over the list)
  prefill  one chunk of every sequence of a batch behind what its cache holds: append, then causal attention
  append   a prompt's rows into the pool, without attention
  copy     the page copies that forks of shared pages cost (all layers of a page)

Pools are shuffled (random free order), contents and queries are N(0, 1) as in the benchmark; q, K and V of a
pass stay in the state, positions too: a pass writes the same cells every time, so it can be repeated.
"""
import random

import numpy as np
import torch

from breccia_amd import lib as L
from breccia_amd.kv import Pool, rope_table

HD, PAGE, BLOCK = 256, 16, 4            # head dim, cells of a page, cells of a selection block
EPS, N_ROT, FREQ = 1e-6, 64, 1e7        # the K preparation of the model
IDX_HEADS, IDX_DIM, TOPK = 4, 128, 512  # its indexer
LAYOUTS = {"f16": L.LAYOUT_F16, "q8v": L.LAYOUT_Q8V, "i8h": L.LAYOUT_I8H}
# bytes of one (cell, kv head): K row + V row
ROW = {"f16": 2 * 512, "q8v": 512 + 288, "i8h": 2 * 272}


def _text(values):
    return ",".join(str(int(v)) for v in values)


def _ints(text):
    return [int(v) for v in text.split(",")]


def _uniform(seed, n, lo, hi):
    r = random.Random(seed)
    return [r.randint(lo, hi) for _ in range(n)]


def _decode(ctx, layout="f16", form="step", layers=1, n_q=16, n_kv=2, gate=False):
    """ctx: cells every sequence holds before this token."""
    return dict(kind="decode", form=form, layout=layout, layers=layers, n_q=n_q, n_kv=n_kv, gate=gate, ctx=_text(ctx))


def _prefill(prefix, tokens, layout="f16", source="f32", layers=1, n_q=16, n_kv=2, gate=False):
    """source: "f32" or "f16" rows are appended as they are, "kprep" rows go through the K preparation."""
    return dict(kind="prefill", source=source, layout=layout, layers=layers, n_q=n_q, n_kv=n_kv, gate=gate,
                prefix=_text(prefix), tokens=_text(tokens))


def _append(prefix, tokens, layout="f16", source="f32", layers=1, n_kv=2):
    return dict(kind="append", source=source, layout=layout, layers=layers, n_kv=n_kv, prefix=_text(prefix),
                tokens=_text(tokens))


def _copy(pages, layout="f16", layers=12, n_kv=2):
    return dict(kind="copy", layout=layout, layers=layers, n_kv=n_kv, pages=pages)


def listed():
    named = [
        # four short conversations, the sizes of the CPU reference configuration: launches and latency
        ("decode_short_b4", _decode([37, 512, 1000, 2048], layers=12)),
        # a single stream at 4k context through the model's 12 attention layers
        ("decode_4k_b1", _decode([4096], layers=12)),
        # the headline batch: eight sequences of 1k to 32k
        ("decode_mixed_b8", _decode(_uniform(3, 8, 1024, 32768), layers=4)),
        # the same range with the model's own calls and heads: K preparation, 24 q heads, output gate, q8_0 V
        ("decode_q8v_kprep_b8", _decode(_uniform(4, 8, 1024, 32768), "q8v", "kprep", layers=4, n_q=24, gate=True)),
        # compressed cache at long context: 16 sequences of 8k to 128k, int8 K and V
        ("decode_i8h_b16", _decode(_uniform(5, 16, 8192, 131072), "i8h", layers=2)),
        # long context through the block selection: 512 blocks of four cells a query
        ("decode_select_b8", _decode(_uniform(6, 8, 8192, 32768), form="select", layers=4, n_q=24, gate=True)),
        # chunked prefill: 1024-token chunks behind a shared-length prefix of 2048
        ("prefill_4x1024", _prefill([2048] * 4, [1024] * 4, source="f16")),
        # a whole prompt in one call, the model's heads and K preparation, q8_0 V
        ("prefill_prompt_4k", _prefill([0], [4096], "q8v", "kprep", n_q=24, gate=True)),
        # chunks of odd sizes at odd places, int8 cache
        ("prefill_ragged", _prefill([1501, 37, 900], [333, 700, 1021], "i8h")),
        # a short follow-up question in a conversation, all 12 layers
        ("prefill_short", _prefill([517], [41], layers=12)),
        # prompts on their way into the cache: 4 x 16384 tokens with K preparation
        ("append_bulk", _append([0] * 4, [16384] * 4, "f16", "kprep")),
        # 256 shared pages of a 12-layer cache made private
        ("copy_pages", _copy(256)),
    ]
    return [dict(case, name=name) for name, case in named]


def _log(rng, lo, hi):
    """An integer of lo..hi, uniform in its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "kprep", "select", "prefill", "prefill", "prefill", "append", "copy"])
    layout = rng.choice(["f16", "q8v", "i8h"])
    n_kv = rng.choice([2, 2, 2, 1, 4])
    n_q = n_kv * rng.choice([8, 8, 12, 4, 16] if n_kv < 4 else [8, 8, 4])
    gate = rng.random() < 0.5
    if kind in ("step", "kprep", "select"):
        lo = 2048 if kind == "select" else 16
        hi = _log(rng, lo * 2, 131072)
        n = _log(rng, 1, 64 if kind != "select" else 16)
        ctx = [_log(rng, max(lo, hi // 32), hi) for _ in range(n)]
        most = 900_000_000 // (ROW[layout] * n_kv)  # cells a pass may walk
        while sum(ctx) > most and len(ctx) > 1:
            ctx.pop()
        layers = max(1, min(12, most // sum(ctx)))
        if kind == "select":
            layers = max(1, min(layers, 32 // len(ctx)))
        return _decode(ctx, layout, kind, layers, n_q, n_kv, gate)
    if kind == "prefill":
        tokens = [_log(rng, 16, 4096) for _ in range(_log(rng, 1, 16))]
        prefix = [rng.choice([0, _log(rng, 16, 8192)]) for _ in tokens]
        pairs = [t * p + t * (t + 1) // 2 for t, p in zip(tokens, prefix)]
        while sum(pairs) * n_q > 180_000_000 and len(pairs) > 1:
            tokens.pop(), prefix.pop(), pairs.pop()
        if sum(pairs) * n_q > 180_000_000:
            tokens, prefix = [rng.randint(300, 1400)], [rng.randint(0, 3000)]
            pairs = [tokens[0] * prefix[0] + tokens[0] * (tokens[0] + 1) // 2]
        layers = max(1, min(12, 60_000_000 // (sum(pairs) * n_q)))
        return _prefill(prefix, tokens, layout, rng.choice(["f32", "f16", "kprep"]), layers, n_q, n_kv, gate)
    if kind == "append":
        n, total = _log(rng, 1, 16), _log(rng, 16, 65536 * 2 // n_kv)
        tokens = [max(1, total // n + rng.randint(-min(total // n // 2, 100), min(total // n // 2, 100))) for _ in range(n)]
        return _append([rng.choice([0, rng.randint(1, 2000)]) for _ in tokens], tokens, layout,
                       rng.choice(["f32", "f16", "kprep"]), max(1, min(12, 4096 // total)), n_kv)
    layers = rng.choice([1, 4, 12])
    return _copy(_log(rng, 1, 12288 // layers // n_kv), layout, layers, n_kv)


class _Slab:
    """A pool that lives as long as anything that looks at its memory (the tensor over its bytes does)."""

    def __init__(self, pool):
        self.pool = pool
        base, _ = pool.layer_ptr(0, 0)
        last, n = pool.layer_ptr(pool.desc.n_layers - 1, 1)
        self.__cuda_array_interface__ = {"shape": ((last.value + n - base.value) // 8,), "typestr": "<i8",
                                         "data": (base.value, False), "version": 2}

    def __del__(self):
        self.pool.destroy()


class _State:
    pass


def _pool(case, held, grow):
    """A shuffled pool with one sequence per entry of `held`, room for `grow` more cells in each."""
    pages = sum((h + g + PAGE - 1) // PAGE for h, g in zip(held, grow))
    n_pages = max(int(pages / 0.6) + 1, case.get("pages", 0) * 2)
    pool = Pool(n_layers=case["layers"], n_pages=n_pages, n_kv_head=case["n_kv"], head_dim=HD, layout=LAYOUTS[case["layout"]],
                max_seqs=len(held), max_pages_per_seq=max((h + g) // PAGE + 2 for h, g in zip(held, grow)))
    return pool, n_pages


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    order = np.random.RandomState(seed)

    def randn(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    kind, layers, n_kv = case["kind"], case["layers"], case["n_kv"]
    s = _State()
    s.case = case
    if kind == "decode":
        held = _ints(case["ctx"])
        tokens = [1] * len(held)
    elif kind == "copy":
        held, tokens = [case["pages"] * PAGE], [0]
    else:
        held, tokens = _ints(case["prefix"]), _ints(case["tokens"])
    pool, n_pages = _pool(case, held, tokens)
    s.pool, s.slab = pool, torch.as_tensor(_Slab(pool), device="cuda")
    pool.set_free_order(order.permutation(n_pages).astype(np.int32))
    s.seqs = np.array([pool.seq_create() for _ in held], dtype=np.int32)
    for i, (h, t) in enumerate(zip(held, tokens)):
        pool.seq_reserve(int(s.seqs[i]), h + t)
    # what the cache holds
    step = 16384
    for layer in range(layers):
        for i, h in enumerate(held):
            for at in range(0, h, step):
                n = min(step, h - at)
                k, v = randn(n, n_kv, HD), randn(n, n_kv, HD)
                pool.append(layer, [int(s.seqs[i])], [at], [n], k.data_ptr(), v.data_ptr())
                del k, v
    if kind == "copy":
        used = pool.block_table(int(s.seqs[0]))
        free = np.setdiff1d(np.arange(n_pages, dtype=np.int32), used)
        s.pairs = np.stack([order.permutation(used), order.permutation(free)[:used.size]], axis=1).astype(np.int32)
        torch.cuda.synchronize()
        return s

    s.pos = np.array(held, dtype=np.int64)      # first cell of this pass
    s.n_tok = np.array(tokens, dtype=np.int32)
    total = int(s.n_tok.sum())
    # K and V of the pass, one tensor per layer, and what their preparation needs
    dt = torch.float16 if case.get("source") == "f16" else torch.float32
    s.k = [randn(total, n_kv, HD).to(dt) for _ in range(layers)]
    s.v = [randn(total, n_kv, HD).to(dt) for _ in range(layers)]
    form = case.get("form", case.get("source"))
    if form in ("kprep", "select"):
        s.max_pos = max(h + t for h, t in zip(held, tokens))
        s.table = torch.from_numpy(rope_table(FREQ, N_ROT, s.max_pos)).cuda()
        s.gamma = 1.0 + 0.1 * randn(HD)
    if kind != "append":
        n_q = case["n_q"]
        s.q = [randn(total, n_q, HD) for _ in range(layers)]
        s.gate = [randn(total, n_q, HD) for _ in range(layers)] if case["gate"] else None
        s.out = torch.zeros(layers, total, n_q, HD, device="cuda")
    if form == "select":
        # per layer: the pooled indexer keys of every complete block, the rolling tail of the incomplete one,
        # this token's indexer key and queries, and the list the selection fills
        n = len(held)
        s.blocks = [h // BLOCK + 1 for h in held]
        s.n_blocks = np.array([(h + 1) // BLOCK for h in held], dtype=np.int32)
        s.pooled = [[randn(b, IDX_DIM) for b in s.blocks] for _ in range(layers)]
        s.tail = [randn(n, BLOCK - 1, IDX_DIM) for _ in range(layers)]
        s.idx_k = [randn(n, IDX_DIM) for _ in range(layers)]
        s.idx_q = [randn(n, IDX_HEADS, IDX_DIM) for _ in range(layers)]
        s.idx_gamma = 1.0 + 0.1 * randn(IDX_DIM)
        s.max_ids = TOPK + 1
        s.ids = torch.zeros(layers, n, s.max_ids, dtype=torch.int32, device="cuda")
        s.counts = torch.zeros(layers, n, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    return s


def _append_rows(s, layer):
    source = s.case.get("form", s.case.get("source"))
    k, v = s.k[layer].data_ptr(), s.v[layer].data_ptr()
    if source == "kprep":
        s.pool.append_kprep(layer, s.seqs, s.pos, s.n_tok, k, v, s.gamma.data_ptr(), EPS, s.table.data_ptr(), N_ROT,
                            s.max_pos)
    else:
        s.pool.append(layer, s.seqs, s.pos, s.n_tok, k, v, f16_rows=source == "f16")


def run(s):
    case, pool = s.case, s.pool
    if case["kind"] == "copy":
        pool.page_copy(s.pairs)
        return s.slab
    if case["kind"] == "append":
        for layer in range(case["layers"]):
            _append_rows(s, layer)
        return s.slab
    n_q, scale = case["n_q"], 1.0 / 16.0
    gate = {}
    if case["kind"] == "prefill":
        for layer in range(case["layers"]):
            if s.gate:
                gate = dict(gate_dev=s.gate[layer].data_ptr(), gate_tok_stride=n_q * HD, gate_head_stride=HD)
            _append_rows(s, layer)
            pool.prefill_attn(layer, s.seqs, s.pos, s.n_tok, n_q, s.q[layer].data_ptr(), s.out[layer].data_ptr(), scale, **gate)
        return s.out, s.slab
    # decode: a token begins with room for it in every sequence
    for seq, p in zip(s.seqs.tolist(), s.pos.tolist()):
        pool.seq_reserve(seq, p + 1)
    for layer in range(case["layers"]):
        q, out = s.q[layer].data_ptr(), s.out[layer].data_ptr()
        if s.gate:
            gate = dict(gate_dev=s.gate[layer].data_ptr(), gate_seq_stride=n_q * HD, gate_head_stride=HD)
        if case["form"] == "step":
            pool.decode_step(layer, s.seqs, s.pos, s.k[layer].data_ptr(), s.v[layer].data_ptr(), n_q, q, out, scale, **gate)
        elif case["form"] == "kprep":
            _append_rows(s, layer)
            pool.decode_attn(layer, s.seqs, s.pos, n_q, q, out, scale, **gate)
        else:
            for i, p in enumerate(s.pos.tolist()):
                pool.idx_pool(s.pooled[layer][i].data_ptr(), s.blocks[i], s.tail[layer][i].data_ptr(),
                              s.idx_k[layer][i].data_ptr(), p, 1, s.idx_gamma.data_ptr(), EPS, s.table.data_ptr(), N_ROT,
                              s.max_pos, IDX_DIM)
            ids, counts = s.ids[layer].data_ptr(), s.counts[layer].data_ptr()
            pool.select_blocks(s.pos, s.idx_q[layer].data_ptr(), [t.data_ptr() for t in s.pooled[layer]], s.n_blocks, IDX_HEADS,
                               IDX_DIM, TOPK, ids, s.max_ids, counts, s.max_ids)
            _append_rows(s, layer)
            pool.decode_attn_select(layer, s.seqs, s.pos, n_q, q, out, scale, ids, s.max_ids, counts, s.max_ids, **gate)
    if case["form"] == "select":
        return s.out, s.slab, s.ids, s.counts, torch.cat([t for layer in s.tail for t in layer])
    return s.out, s.slab


def work(case):
    kind, layers, n_kv, row = case["kind"], case["layers"], case["n_kv"], ROW[case["layout"]]
    if kind == "copy":
        return {"bytes": 2 * case["pages"] * layers * PAGE * n_kv * row, "flops": 0}
    source = 2 if case.get("source") == "f16" else 4
    new = n_kv * (2 * HD * source + row)        # bytes of appending one token
    if kind == "append":
        return {"bytes": layers * sum(_ints(case["tokens"])) * new, "flops": 0}
    n_q = case["n_q"]
    token = (3 if case["gate"] else 2) * n_q * HD * 4   # q, out, gate
    if kind == "prefill":
        prefix, tokens = _ints(case["prefix"]), _ints(case["tokens"])
        pairs = sum(t * p + t * (t + 1) // 2 for t, p in zip(tokens, prefix))
        read = sum(p + t for t, p in zip(tokens, prefix)) * n_kv * row
        return {"bytes": layers * (sum(tokens) * (new + token) + read), "flops": layers * pairs * n_q * HD * 4}
    ctx = [c + 1 for c in _ints(case["ctx"])]
    cells = ctx
    extra = 0
    if case["form"] == "select":
        cells = [min(c, (TOPK + 1) * BLOCK) for c in ctx]
        extra = sum(c // BLOCK * IDX_DIM * 4 + IDX_HEADS * IDX_DIM * 4 for c in ctx)
    table = sum((c + PAGE - 1) // PAGE * 4 for c in ctx)
    return {"bytes": layers * (sum(cells) * n_kv * row + table + len(ctx) * (token + new) + extra),
            "flops": layers * sum(cells) * n_q * HD * 4}


def tolerance(case):
    # pool bytes, lists and tails are whole numbers or bit-exact; attention outputs are f32 sums over f16 values
    # with q and the weights carried at 22 bits: against the same attention in 64 bits they are off by up to
    # 5e-7 in the 2-norm and 8e-6 of the root mean square in single values
    if case["kind"] in ("append", "copy"):
        return "exact"
    return {"rel": 3e-6, "max": 4e-5}


def _blocks(x, half_scale):
    """x (f32, rows of 256) as int8 codes times a scale of every 32 values, back in 64 bits."""
    b = x.reshape(*x.shape[:-1], HD // 32, 32)
    amax = b.abs().amax(-1, keepdim=True)
    # quotients through 64 bits: rounded once, as IEEE division does
    scale = torch.where(amax > 0, (amax.double() / 127.0).float(), torch.ones_like(amax))
    if half_scale:
        scale = torch.where(amax > 0, scale.half().float().clamp_min(2.0 ** -14), scale)
    t = (b.double() / scale.double()).float().clamp(-127.0, 127.0)
    code = torch.trunc(t + torch.copysign(torch.full_like(t, 0.5), t))
    return (code.double() * scale.double()).reshape(x.shape)


def _kept(x, layout, is_k):
    """What the cache holds of f32 rows."""
    if layout == "i8h" or (layout == "q8v" and not is_k):
        return _blocks(x, layout == "i8h")
    h = x.half().double()
    return torch.where(h.abs() < 2.0 ** -14, torch.zeros_like(h), h)


def _norm_rotate(x, gamma, at):
    """RMSNorm and the rotary of the first N_ROT values; x [n, ..., d], at [n] positions; f32 between the steps."""
    x = x.double()
    y = (x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * gamma.double()).float().double()
    half = N_ROT // 2
    inv = torch.tensor([FREQ ** (-2.0 * i / N_ROT) for i in range(half)], dtype=torch.float64, device=x.device)
    angle = (at.double()[:, None] * inv).reshape(at.numel(), *([1] * (x.dim() - 2)), half)
    cos, sin = torch.cos(angle).float().double(), torch.sin(angle).float().double()
    a, b = y[..., :half], y[..., half:N_ROT]
    return torch.cat([a * cos - b * sin, a * sin + b * cos, y[..., N_ROT:]], -1).float()


def _attend(q, k, v, seen, n_kv, gate):
    """q [T, n_q, HD], k and v [C, n_kv, HD] in 64 bits, seen [T, C] or None (all)."""
    tokens, n_q = q.shape[:2]
    group = n_q // n_kv
    out = torch.empty_like(q)
    for h in range(n_kv):
        keys, values = k[:, h].t().contiguous(), v[:, h].contiguous()
        step = max(1, (1 << 27) // (keys.shape[1] * group))
        for t in range(0, tokens, step):
            rows = q[t:t + step, h * group:(h + 1) * group]
            s = (rows.reshape(-1, HD) @ keys / 16.0).reshape(rows.shape[0], group, -1)
            if seen is not None:
                s = s.masked_fill(~seen[t:t + step, None, :], float("-inf"))
            p = torch.softmax(s, -1).reshape(-1, keys.shape[1])
            out[t:t + step, h * group:(h + 1) * group] = (p @ values).reshape(rows.shape)
    return out if gate is None else out * torch.sigmoid(gate.double())


def exact(case, seed):
    """The attention outputs in 64 bits over what the cache holds; everything else that a pass returns is bytes or
    whole numbers.  The draws repeat those of prepare(), in its order."""
    kind, layers, n_kv, layout = case["kind"], case["layers"], case["n_kv"], case["layout"]
    if kind in ("append", "copy"):
        return None
    g = torch.Generator(device="cuda").manual_seed(seed)

    def randn(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    held = _ints(case["ctx"] if kind == "decode" else case["prefix"])
    tokens = [1] * len(held) if kind == "decode" else _ints(case["tokens"])
    cache = []
    for _ in range(layers):
        rows = []
        for h in held:
            k, v = [randn(0, n_kv, HD)], [randn(0, n_kv, HD)]
            for at in range(0, h, 16384):
                n = min(16384, h - at)
                k.append(randn(n, n_kv, HD))
                v.append(randn(n, n_kv, HD))
            rows.append((torch.cat(k), torch.cat(v)))
        cache.append(rows)
    total, n_q = sum(tokens), case["n_q"]
    dt = torch.float16 if case.get("source") == "f16" else torch.float32
    new_k = [randn(total, n_kv, HD).to(dt).float() for _ in range(layers)]
    new_v = [randn(total, n_kv, HD).to(dt).float() for _ in range(layers)]
    form = case.get("form", case.get("source"))
    gamma = 1.0 + 0.1 * randn(HD) if form in ("kprep", "select") else None
    q = [randn(total, n_q, HD) for _ in range(layers)]
    gate = [randn(total, n_q, HD) for _ in range(layers)] if case["gate"] else None
    if form == "select":
        pooled = [[randn(h // BLOCK + 1, IDX_DIM) for h in held] for _ in range(layers)]
        tail = [randn(len(held), BLOCK - 1, IDX_DIM) for _ in range(layers)]
        idx_k = [randn(len(held), IDX_DIM) for _ in range(layers)]
        idx_q = [randn(len(held), IDX_HEADS, IDX_DIM) for _ in range(layers)]
        idx_gamma = 1.0 + 0.1 * randn(IDX_DIM)
    out = torch.empty(layers, total, n_q, HD, dtype=torch.float64, device="cuda")
    for layer in range(layers):
        first = 0
        for i, (h, t) in enumerate(zip(held, tokens)):
            mine = slice(first, first + t)
            first += t
            k, v = new_k[layer][mine], new_v[layer][mine]
            if form == "kprep":
                k = _norm_rotate(k, gamma, torch.arange(h, h + t, device="cuda"))
            k = _kept(torch.cat([cache[layer][i][0], k]), layout, True)
            v = _kept(torch.cat([cache[layer][i][1], v]), layout, False)
            seen = None
            if kind == "prefill":
                seen = torch.arange(h + t, device="cuda")[None, :] <= torch.arange(h, h + t, device="cuda")[:, None]
            if form == "select":
                keys = pooled[layer][i]
                if (h + 1) % BLOCK == 0:
                    raw = torch.cat([tail[layer][i], idx_k[layer][i][None]])
                    mean = ((raw[0] / BLOCK + raw[1] / BLOCK) + raw[2] / BLOCK) + raw[3] / BLOCK
                    keys[h // BLOCK] = _norm_rotate(mean[None], idx_gamma, torch.tensor([h // BLOCK * BLOCK], device="cuda"))[0]
                n = (h + 1) // BLOCK
                score = (idx_q[layer][i].double() @ keys[:n].double().t().contiguous()).clamp_min(0.0).sum(0)
                chosen = torch.sort(score, descending=True, stable=True).indices[:TOPK]
                chosen = torch.unique(torch.cat([chosen, torch.tensor([h // BLOCK], device="cuda")]))
                cells = (chosen[:, None] * BLOCK + torch.arange(BLOCK, device="cuda")).reshape(-1)
                cells = cells[cells <= h]
                k, v = k[cells], v[cells]
            out[layer, mine] = _attend(q[layer][mine].double(), k, v, seen, n_kv, gate[layer][mine] if gate else None)
    return (out, None, None, None, None) if form == "select" else (out, None)
