"""The work that programs hand to this library, as cases to be timed: decoding tokens and prompt passes through the
attention blocks of gpt-oss-20b (64 query heads over 8 kv heads of width 64, hidden width 2,880, Q8_0 projections,
layers that see 128 positions and layers that see all of them in turn), and the attention operator alone, at these
heads and at the wide ones (128-512) it also serves.

Kinds of case:
  token    one decoding step of `seqs` sequences through `layers` attention blocks, recorded as one batch: hidden rows,
           RMS norm + q, k, v projections, biases + rotation + cache append, attention, output projection + residual
  prompt   `t` rows of one sequence, after `start` earlier ones, through `layers` blocks, recorded as one batch
  table    the attention of `seqs` decoding sequences of unequal length, a full and a 128-position layer each
  rows     one call of the attention operator on `t` rows (the prompt-pass form, or the plain one where t < 32)
  static   one call of the entry point that allocates nothing, on the caller's stream and memory
"""
import math
import random

import torch

from loadngo_amd import compute as C

HIDDEN, HEADS, KV, DIM, WINDOW = 2880, 64, 8, 64, 128
QW, KW = HEADS * DIM, KV * DIM
EPS, SCALE = 1e-5, 0.125
RING = WINDOW + 512  # rows of a sliding layer's cache: its window and the largest chunk of a prompt
SIZE = {"f32": 4, "bf16": 2}
TYPE = {"f32": C.F32, "bf16": C.BF16}
TORCH = {"f32": torch.float32, "bf16": torch.bfloat16}


def listed():
    return [
        # the first tokens of a chat, with the caches in f32 as the reference program keeps them
        {"name": "token f32 ctx 300", "kind": "token", "seqs": 1, "ctx": 300, "layers": 24, "dtype": "f32", "seed": 1},
        # a token of one long conversation
        {"name": "token bf16 ctx 4096", "kind": "token", "seqs": 1, "ctx": 4096, "layers": 24, "dtype": "bf16", "seed": 1},
        # a server's step: sixteen conversations of very different lengths
        {"name": "token x16 ragged", "kind": "token", "seqs": 16, "ctx": 8192, "layers": 24, "dtype": "bf16", "seed": 2},
        # one chunk of a prompt, the 512 rows that the reference program feeds at a time
        {"name": "prompt 512 after 1536", "kind": "prompt", "t": 512, "start": 1536, "layers": 2, "dtype": "bf16"},
        # what is left of a prompt after its last whole chunk: a ragged number of rows late in the context
        {"name": "prompt 77 after 4096", "kind": "prompt", "t": 77, "start": 4096, "layers": 2, "dtype": "bf16"},
        # a long prompt in one call
        {"name": "prompt 8192", "kind": "prompt", "t": 8192, "start": 0, "layers": 2, "dtype": "bf16"},
        # the first chunk of a prompt over f32 caches
        {"name": "prompt f32 512", "kind": "prompt", "t": 512, "start": 0, "layers": 2, "dtype": "f32"},
        # the cache-bound end of decoding: sixteen sequences of 131,072 positions
        {"name": "table x16 131072", "kind": "table", "seqs": 16, "low": 131072, "high": 131072, "dtype": "bf16", "seed": 3},
        # continuous batching: thirty-two sequences of unequal length
        {"name": "table x32 ragged", "kind": "table", "seqs": 32, "low": 128, "high": 8192, "dtype": "bf16", "seed": 4},
        # wide heads, a chunk of a prompt in a ring that wraps (the reference's own timing shape)
        {"name": "rows f32 w256 512", "kind": "rows", "t": 512, "start": 3000, "heads": 32, "kv_heads": 16, "dim": 256,
         "window": 1024, "slots": 1536, "dtype": "f32"},
        # wide heads, one token over a sliding cache
        {"name": "rows bf16 w256 token", "kind": "rows", "t": 1, "start": 3000, "heads": 32, "kv_heads": 16, "dim": 256,
         "window": 1024, "slots": 1536, "dtype": "bf16"},
        # one layer's attention called from a loop that allocates nothing
        {"name": "static token ctx 1000", "kind": "static", "t": 1, "ctx": 1000, "window": 0, "dtype": "bf16"},
    ]


def _log(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["token", "token", "prompt", "prompt", "prompt", "table", "rows", "rows", "static"])
    dtype = rng.choice(["bf16", "bf16", "f32"])
    if kind == "token":  # the positions of all sequences together stay under 16 x 8,192
        seqs = _log(rng, 1, 31)
        return {"kind": kind, "seqs": seqs, "ctx": _log(rng, 16, min(32768, 131072 // seqs)),
                "layers": rng.choice([4, 8, 12, 24]), "dtype": dtype, "seed": rng.randrange(1 << 20)}
    if kind == "prompt":  # f32 attention is sixteen times the matrix work
        t = _log(rng, 33, 8192 if dtype == "bf16" else 2048)
        return {"kind": kind, "t": t, "start": rng.choice([0, _log(rng, 1, max(1, 8192 - t))]), "layers": 2, "dtype": dtype}
    if kind == "table":
        seqs = _log(rng, 2, 256)
        high = _log(rng, 256, (2097152 if dtype == "bf16" else 1048576) // seqs)
        return {"kind": kind, "seqs": seqs, "low": max(1, high // rng.choice([1, 4, 64])), "high": high, "dtype": dtype,
                "seed": rng.randrange(1 << 20)}
    if kind == "rows":
        kv_heads, dim = rng.choice([(16, 256), (4, 512), (8, 128)])
        most = 1024 if dtype == "bf16" else 512
        t = rng.choice([1, _log(rng, 2, 31), _log(rng, 33, most), _log(rng, 33, most)])
        window, start = rng.choice([0, 1024]), _log(rng, 64, 4096)
        slots = 1024 + 32 * ((t + 31) // 32) if window else 0  # a ring that holds the window and the new rows
        return {"kind": kind, "t": t, "start": start, "heads": 32, "kv_heads": kv_heads, "dim": dim, "window": window,
                "slots": slots, "dtype": dtype}
    return {"kind": kind, "t": rng.choice([1, 1, _log(rng, 2, 16)]), "ctx": _log(rng, 32, 65536), "window": rng.choice([0, WINDOW]),
            "dtype": dtype}


# ---- shared pieces --------------------------------------------------------------------------------------------------

_gpu = None


def gpu():
    global _gpu
    if _gpu is None:
        _gpu = C.Gpu(0)
    return _gpu


class _Memory:
    """Tells torch about a library buffer, and keeps it alive."""

    def __init__(self, buffer, size):
        self.buffer = buffer
        self.__cuda_array_interface__ = {"shape": (buffer.len // size,), "typestr": {2: "<i2", 4: "<f4"}[size],
                                         "data": (buffer.device_ptr(), False), "version": 2}


def tensor_of(buffer, dtype):
    """A library buffer as a torch tensor over the same memory."""
    t = torch.as_tensor(_Memory(buffer, SIZE[dtype]), device="cuda")
    return t.view(torch.bfloat16) if dtype == "bf16" else t


def up32(n):
    return (n + 31) // 32 * 32


def full(window):
    return C.FULL if not window else window


def lengths(case):
    """The sequences' lengths (positions that the step's query may see, itself included), longest possible first."""
    rng = random.Random(case["seed"])
    low, high = (max(1, case["ctx"] // 64), case["ctx"]) if case["kind"] == "token" else (case["low"], case["high"])
    return [high] + [rng.randint(low, high) for _ in range(case["seqs"] - 1)]


def seen(t, start, window):
    """Unmasked (query, key) pairs of t rows after `start`."""
    if not window or window >= start + t:
        return t * start + t * (t + 1) // 2
    return sum(min(start + i + 1, window) for i in range(t))


class Fill:
    """Inputs from a seed, made on the device."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, shape, std=1.0, dtype=torch.float32):
        return torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32).mul_(std).to(dtype)

    def into(self, buffer, dtype, std=1.0):
        flat, step = tensor_of(buffer, dtype), 1 << 28
        for at in range(0, flat.numel(), step):
            part = flat[at:at + step]
            part.copy_(self.normal(part.shape, std))

    def q8_0(self, rows, cols):
        """Codes and binary16 scales of a random weight matrix quantised as Q8_0 is: 127 steps to a block's largest value."""
        w = self.normal((rows * cols // 32, 32), 0.02)
        scales = (w.abs().amax(1, keepdim=True) / 127).half()
        codes = (w / scales.float()).round().clamp_(-127, 127).to(torch.int8)
        return codes.reshape(-1), scales.reshape(-1)


class State:
    pass


def _weights(s, fill, layers):
    """Every layer's matrices and vectors, in three residents: codes, scales, f32 vectors. Slices name them by the numbers
    they have in a batch that attaches the three in this order after its `n` buffers."""
    codes, scales, vectors, s.plan = [], [], [], []
    for _ in range(layers):
        entry = {}
        for name, rows, cols in (("q", QW, HIDDEN), ("k", KW, HIDDEN), ("v", KW, HIDDEN), ("o", HIDDEN, QW)):
            c, d = fill.q8_0(rows, cols)
            entry[name] = (sum(x.numel() for x in codes), c.numel(), 2 * sum(x.numel() for x in scales), 2 * d.numel(), rows, cols)
            codes.append(c)
            scales.append(d)
        for name, n, std, mean in (("norm", HIDDEN, 0.1, 1.0), ("qb", QW, 0.1, 0.0), ("kb", KW, 0.1, 0.0), ("vb", KW, 0.1, 0.0),
                                   ("ob", HIDDEN, 0.1, 0.0), ("sinks", HEADS, 1.0, 0.0)):
            entry[name] = (4 * sum(x.numel() for x in vectors), 4 * n)
            vectors.append(fill.normal(n, std) + mean)
        s.plan.append(entry)
    s.residents = [gpu().resident(torch.cat(x).cpu().numpy()) for x in (codes, scales, vectors)]


def _named(s, n):
    """The plan's entries as slices, for batches of n buffers."""
    for entry in s.plan:
        for name, at in list(entry.items()):
            if len(at) == 6:
                entry[name] = ((C.Slice(n, at[0], at[1]), C.Slice(n + 1, at[2], at[3])), at[4], at[5])
            else:
                entry[name] = C.Slice(n + 2, *at)


def _begin(s):
    batch = gpu().batch(s.buffers)
    for r in s.residents:
        batch.attach(r)
    return batch


def _finish(batch):
    done = batch.run()
    batch.drop()
    if isinstance(done.gpu_time, C.Error):
        raise done.gpu_time


def _rope(positions):
    inv = 150000.0 ** (-torch.arange(0, DIM, 2, dtype=torch.float64) / DIM)
    return C.rope_table(inv.numpy(), 1.0, positions[0], 1) if len(positions) == 1 else \
        torch.cat([torch.from_numpy(C.rope_table(inv.numpy(), 1.0, p, 1)) for p in positions]).numpy()


# ---- token: one decoding step through the blocks --------------------------------------------------------------------

def _prepare_token(case, seed):
    s, fill, dtype = State(), Fill(seed), case["dtype"]
    es, lens, n, layers = SIZE[case["dtype"]], lengths(case), case["seqs"], case["layers"]
    _weights(s, fill, layers)
    rows_full = [sum(lens[:i]) for i in range(n + 1)]
    g = gpu()
    # even layers see 128 positions through a ring, odd ones see every position
    b = {"embed": g.buffer(n * HIDDEN * 4), "h": g.buffer(n * HIDDEN * 4), "q": g.buffer(n * QW * 4), "k": g.buffer(n * KW * 4),
         "v": g.buffer(n * KW * 4), "table": g.upload(_rope([x - 1 for x in lens])), "qr": g.buffer(n * QW * es),
         "att": g.buffer(n * QW * es)}
    for name in ("ks", "vs"):
        b[name] = g.buffer((layers + 1) // 2 * n * RING * KW * es)
    for name in ("kf", "vf"):
        b[name] = g.buffer(layers // 2 * rows_full[n] * KW * es)
    names = list(b)
    s.buffers = [b[x] for x in names]
    at = {x: i for i, x in enumerate(names)}
    fill.into(b["embed"], "f32")
    for name in ("ks", "vs", "kf", "vf"):
        fill.into(b[name], dtype)
    _named(s, len(names))
    s.steps = []
    for i, entry in enumerate(s.plan):
        kb, vb, slides = (at["ks"], at["vs"], True) if i % 2 == 0 else (at["kf"], at["vf"], False)
        where = [((i // 2) * n * RING + j * RING if slides else (i // 2) * rows_full[n] + rows_full[j]) * KW * es for j in range(n)]
        slots = [RING if slides else x for x in lens]
        prepare = C.prepare_items([C.PrepareItem(
            q_offset=j * QW * 4, k_offset=j * KW * 4, v_offset=j * KW * 4, table_offset=j * DIM * 4, q_out_offset=j * QW * es,
            k_cache_offset=where[j], v_cache_offset=where[j], n=1, start=lens[j] - 1, slots=slots[j]) for j in range(n)])
        step = {"prepare": prepare, "buffers": dict(q=at["q"], k=at["k"], v=at["v"], table=at["table"], q_out=at["qr"], k_cache=kb, v_cache=vb),
                "matrices": [(entry[m][0], C.Slice(at[m], 0, n * entry[m][1] * 4), entry[m][1]) for m in ("q", "k", "v")]}
        if n == 1:
            rows = min(slots[0], lens[0])
            step["qkv"] = (C.Slice(at["qr"], 0, QW * es), C.Slice(kb, where[0], rows * KW * es), C.Slice(vb, where[0], rows * KW * es))
            step["shape"] = C.GroupedShape(1, lens[0] - 1, HEADS, KV, DIM, WINDOW if slides else C.FULL, slots[0], SCALE)
        else:
            step["items"] = C.decode_items([C.DecodeItem(
                j * QW * es, j * QW * es, where[j], where[j], entry["sinks"].offset, lens[j] - 1,
                WINDOW if slides else C.FULL, slots[j]) for j in range(n)])
            step["caches"] = (kb, vb)
        s.steps.append((entry, step))
    s.n, s.dtype, s.sinks_buffer = n, TYPE[dtype], len(names) + 2
    s.embed, s.h = C.Slice(at["embed"], 0, n * HIDDEN * 4), C.Slice(at["h"], 0, n * HIDDEN * 4)
    s.att, s.at = C.Slice(at["att"], 0, n * QW * es), at
    s.outputs = {"h": tensor_of(b["h"], "f32"), "att": tensor_of(b["att"], dtype)}
    s.outputs.update({x: tensor_of(b[x], dtype) for x in ("ks", "vs", "kf", "vf")})
    return s


def _run_token(s):
    batch, n = _begin(s), s.n
    batch.copy_rows((s.embed, HIDDEN), (s.h, HIDDEN), n, HIDDEN)
    for entry, step in s.steps:
        batch.gemm_q8_0_many_normed(step["matrices"], s.h, (entry["norm"], EPS), HIDDEN, n, HIDDEN)
        batch.prepare_attention(step["buffers"], step["prepare"], HEADS, KV, DIM, DIM, s.dtype, entry["qb"], entry["kb"], entry["vb"])
        if n == 1:
            batch.attention_grouped_with_sinks(step["qkv"], entry["sinks"], s.att, step["shape"], s.dtype)
        else:
            batch.attention_decode_batched(s.at["qr"], *step["caches"], s.at["att"], s.sinks_buffer, step["items"], HEADS, KV, DIM,
                                           SCALE, s.dtype)
        batch.gemm_q8_0_residual(entry["o"][0], s.att, entry["ob"], s.h, HIDDEN, QW, n, (QW, HIDDEN), s.dtype)
    _finish(batch)
    return s.outputs


# ---- prompt: rows of one sequence through the blocks ----------------------------------------------------------------

def _prepare_prompt(case, seed):
    s, fill, dtype = State(), Fill(seed), case["dtype"]
    es, t, start, layers = SIZE[dtype], case["t"], case["start"], case["layers"]
    tp, last = up32(t), case["start"] + case["t"]
    slots_full = up32(last)
    slots_ring = WINDOW + max(512, tp)
    _weights(s, fill, layers)
    g = gpu()
    inv = (150000.0 ** (-torch.arange(0, DIM, 2, dtype=torch.float64) / DIM)).numpy()
    b = {"embed": g.buffer(tp * HIDDEN * 4), "h": g.buffer(tp * HIDDEN * 4), "x": g.buffer(tp * HIDDEN * 4), "q": g.buffer(tp * QW * 4),
         "k": g.buffer(tp * KW * 4), "v": g.buffer(tp * KW * 4), "table": g.upload(C.rope_table(inv, 1.0, start, t)),
         "qr": g.buffer(tp * QW * es), "att": g.buffer(tp * QW * es), "tmp": g.buffer(tp * HIDDEN * 4)}
    for name in ("ks", "vs"):
        b[name] = g.buffer((layers + 1) // 2 * slots_ring * KW * es)
    for name in ("kf", "vf"):
        b[name] = g.buffer(layers // 2 * slots_full * KW * es)
    names = list(b)
    s.buffers = [b[x] for x in names]
    at = {x: i for i, x in enumerate(names)}
    for name in ("embed", "qr", "att"):  # the rows that pad t to a multiple of 32 hold values too
        fill.into(b[name], "f32" if name == "embed" else dtype)
    for name in ("ks", "vs", "kf", "vf"):
        fill.into(b[name], dtype)
    _named(s, len(names))
    s.steps = []
    for i, entry in enumerate(s.plan):
        slides = i % 2 == 0
        kb, vb, slots = (at["ks"], at["vs"], slots_ring) if slides else (at["kf"], at["vf"], slots_full)
        where = (i // 2) * slots * KW * es
        held = slots if slots < last else up32(last)
        s.steps.append((entry, {
            "prepare": C.prepare_items([C.PrepareItem(k_cache_offset=where, v_cache_offset=where, n=t, start=start, slots=slots)]),
            "buffers": dict(q=at["q"], k=at["k"], v=at["v"], table=at["table"], q_out=at["qr"], k_cache=kb, v_cache=vb),
            "matrices": [(entry[m][0], C.Slice(at[m], 0, tp * entry[m][1] * 4), entry[m][1]) for m in ("q", "k", "v")],
            "qkv": (C.Slice(at["qr"], 0, tp * QW * es), C.Slice(kb, where, held * KW * es), C.Slice(vb, where, held * KW * es)),
            "shape": C.GroupedShape(t, start, HEADS, KV, DIM, WINDOW if slides else C.FULL, slots, SCALE)}))
    s.t, s.tp, s.dtype = t, tp, TYPE[dtype]
    for name in ("embed", "h", "x", "tmp"):
        setattr(s, name, C.Slice(at[name], 0, tp * HIDDEN * 4))
    s.att = C.Slice(at["att"], 0, tp * QW * es)
    s.outputs = {"h": tensor_of(b["h"], "f32")[:t * HIDDEN], "att": tensor_of(b["att"], dtype)[:t * QW]}
    s.outputs.update({x: tensor_of(b[x], dtype) for x in ("ks", "vs", "kf", "vf")})
    return s


def _run_prompt(s):
    batch, tp = _begin(s), s.tp
    batch.copy_rows((s.embed, HIDDEN), (s.h, HIDDEN), tp, HIDDEN)
    for entry, step in s.steps:
        batch.copy_rows((s.h, HIDDEN), (s.x, HIDDEN), tp, HIDDEN)
        batch.rmsnorm_rows((s.x, entry["norm"]), tp, (HIDDEN, HIDDEN), EPS)
        batch.gemm_q8_0_many(step["matrices"], s.x, HIDDEN, tp, HIDDEN)
        batch.prepare_attention(step["buffers"], step["prepare"], HEADS, KV, DIM, DIM, s.dtype, entry["qb"], entry["kb"], entry["vb"])
        batch.attention_grouped_tiled_with_sinks(step["qkv"], entry["sinks"], s.att, step["shape"], s.dtype)
        if s.dtype == C.BF16:
            batch.gemm_q8_0_bf16(entry["o"][0], s.att, s.tmp, HIDDEN, QW, tp, (QW, HIDDEN))
        else:
            batch.gemm_q8_0_tiled(entry["o"][0], s.att, s.tmp, HIDDEN, QW, tp, (QW, HIDDEN))
        batch.add_rows(s.tmp, (entry["ob"], 0), tp, HIDDEN)
        batch.add_rows(s.h, (s.tmp, HIDDEN), tp, HIDDEN)
    _finish(batch)
    return s.outputs


# ---- table, rows, static: the attention operator alone --------------------------------------------------------------

def _prepare_table(case, seed):
    s, fill, dtype = State(), Fill(seed), case["dtype"]
    es, lens, n = SIZE[dtype], lengths(case), case["seqs"]
    g = gpu()
    total = sum(lens)
    s.buffers = [g.buffer(2 * n * QW * es), g.buffer(total * KW * es), g.buffer(total * KW * es), g.buffer(2 * n * QW * es), g.buffer(2 * HEADS * 4)]
    for b, d in zip(s.buffers, (dtype, dtype, dtype, dtype, "f32")):
        fill.into(b, d)
    at, items = 0, [[], []]
    for j, x in enumerate(lens):
        for layer, window in enumerate((C.FULL, WINDOW)):  # the same cache serves as both layers' here
            row = layer * n + j
            items[layer].append(C.DecodeItem(row * QW * es, row * QW * es, at * KW * es, at * KW * es, layer * HEADS * 4, x - 1, window, x))
        at += x
    s.items, s.dtype = C.decode_items(items[0] + items[1]), TYPE[dtype]
    s.outputs = {"out": tensor_of(s.buffers[3], dtype)}
    s.residents = []
    return s


def _run_table(s):
    batch = _begin(s)
    batch.attention_decode_batched(0, 1, 2, 3, 4, s.items, HEADS, KV, DIM, SCALE, s.dtype)
    _finish(batch)
    return s.outputs


def _prepare_rows(case, seed):
    s, fill, dtype = State(), Fill(seed), case["dtype"]
    es, t, width, kw = SIZE[dtype], case["t"], case["heads"] * case["dim"], case["kv_heads"] * case["dim"]
    s.tiled = t >= 32
    last = case["start"] + t
    slots = case["slots"] or up32(last)
    held = min(slots, last) if not s.tiled else slots if slots < last else up32(last)
    tp = up32(t) if s.tiled else t
    g = gpu()
    rows = max(slots, held)
    s.buffers = [g.buffer(tp * width * es), g.buffer(rows * kw * es), g.buffer(rows * kw * es), g.buffer(tp * width * es)]
    for b in s.buffers:
        fill.into(b, dtype)
    s.qkvo = (C.Slice(0, 0, tp * width * es), C.Slice(1, 0, held * kw * es), C.Slice(2, 0, held * kw * es), C.Slice(3, 0, tp * width * es))
    s.shape = C.GroupedShape(t, case["start"], case["heads"], case["kv_heads"], case["dim"], full(case["window"]), slots, 1.0 / math.sqrt(case["dim"]))
    s.dtype, s.residents = TYPE[dtype], []
    s.outputs = {"out": tensor_of(s.buffers[3], dtype)[:t * width]}
    return s


def _run_rows(s):
    batch = _begin(s)
    (batch.attention_grouped_tiled if s.tiled else batch.attention_grouped)(*s.qkvo, s.shape, s.dtype)
    _finish(batch)
    return s.outputs


def _prepare_static(case, seed):
    s, fill, kind = State(), Fill(seed), TORCH[case["dtype"]]
    t, ctx = case["t"], case["ctx"]
    s.q, s.k, s.v = fill.normal((t, QW), 1.0, kind), fill.normal((ctx, KW), 1.0, kind), fill.normal((ctx, KW), 1.0, kind)
    s.sinks, s.out = fill.normal(HEADS), torch.zeros((t, QW), device="cuda", dtype=kind)
    s.shape = C.GroupedShape(t, ctx - t, HEADS, KV, DIM, full(case["window"]), ctx, SCALE)
    s.dtype = TYPE[case["dtype"]]
    return s


def _run_static(s):
    gpu().attention_grouped_static(s.q.data_ptr(), s.k.data_ptr(), s.v.data_ptr(), s.out.data_ptr(), s.sinks.data_ptr(), s.shape,
                                   s.dtype, torch.cuda.current_stream().cuda_stream)
    return s.out


_PREPARE = {"token": _prepare_token, "prompt": _prepare_prompt, "table": _prepare_table, "rows": _prepare_rows, "static": _prepare_static}
_RUN = {"token": _run_token, "prompt": _run_prompt, "table": _run_table, "rows": _run_rows, "static": _run_static}


def prepare(case, seed):
    s = _PREPARE[case["kind"]](case, seed)
    s.kind = case["kind"]
    torch.cuda.synchronize()  # torch's stream is not the library's
    return s


def run(state):
    return _RUN[state.kind](state)


def work(case):
    es = SIZE[case["dtype"]]
    kind = case["kind"]
    if kind in ("token", "prompt"):
        n, layers = case["seqs"] if kind == "token" else case["t"], case["layers"]
        slide, all_ = (layers + 1) // 2, layers // 2
        weights = (QW + 2 * KW) * HIDDEN + HIDDEN * QW
        if kind == "token":
            pairs = [sum(min(x, w) for x in lengths(case)) for w in (WINDOW, case["ctx"])]
            held = pairs
        else:
            pairs = [seen(case["t"], case["start"], w) for w in (WINDOW, 0)]
            held = [min(case["start"] + n, WINDOW - 1 + n), case["start"] + n]
        cache = (slide * held[0] + all_ * held[1]) * 2 * KW * es
        return {"bytes": layers * (weights * 34 // 32 + (HIDDEN * 2 + QW + 2 * KW + HEADS) * 4) + cache + layers * n * 2 * KW * es
                + n * (2 * HIDDEN * 4 + DIM * 4 + QW * es),
                "flops": layers * 2 * n * weights + 4 * DIM * HEADS * (slide * pairs[0] + all_ * pairs[1])}
    if kind == "table":
        lens = lengths(case)
        positions = sum(lens)  # the 128-position layer's rows are among the other layer's
        return {"bytes": positions * 2 * KW * es + 4 * len(lens) * QW * es + 2 * HEADS * 4,
                "flops": 4 * DIM * HEADS * sum(x + min(x, WINDOW) for x in lens)}
    if kind == "rows":
        t, start, window = case["t"], case["start"], case["window"]
        held = min(start + t, window - 1 + t if window else start + t)
        return {"bytes": (2 * t * case["heads"] + 2 * held * case["kv_heads"]) * case["dim"] * es,
                "flops": 4 * case["dim"] * case["heads"] * seen(t, start, window)}
    t, ctx, window = case["t"], case["ctx"], case["window"]
    held = min(ctx, window - 1 + t) if window else ctx
    return {"bytes": (2 * t * QW + 2 * held * KW) * es + HEADS * 4, "flops": 4 * DIM * HEADS * seen(t, ctx - t, window)}


def tolerance(case):
    """The largest relative difference between two correct ways to compute a case: the library's own alternative kernels and
    other numbers of chunks and splits (sums in another order), over the listed cases and drawn ones. Attention alone: f32
    6e-7, bf16 1.5e-3 (outputs and weights rounded to bf16). Through blocks: f32 4e-6 - the products take f32 positions as
    two bf16 values, 2^-17 of each, which another split of the same 16 bits rounds differently and 24 layers carry on -
    and bf16 4e-3 (a rounding of every layer's attention, carried to the next)."""
    blocks = case["kind"] in ("token", "prompt")
    if case["dtype"] == "f32":
        return {"rel": 3e-5 if blocks else 1e-5}
    return {"rel": 1e-2 if blocks else 6e-3}
