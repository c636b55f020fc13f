"""What a program that serves a model through this backend has it do, as cases that can be timed.

A case is a dict of plain values; `prepare` makes what the program holds before the call (tensors
of the backend, page tables, the attached workspace), `run` is one pass through the public entry
points of clori_amd.backend, `work` what the pass cannot do without, `tolerance` how far two
correct implementations may be apart.  Kinds of cases:

  decode         one new token of a session over its token-major [K | V] history, bf16: the history
                 writer (rotation of Q and K and both rows), then gated attention
  decoder_block  the same step as an unchanged caller of the reference's operator table makes it:
                 thirteen calls on F32 activations, each complete before the next
  prefill        new tokens of a prompt, bf16, at the end of a history or with none
  prefill_exact  the same under the EXACT_F32 contract
  paged          one token each of a batch of sessions over paged KV, bf16 or Q8_0 pages
  mla            absorbed-latent decode of a batch: 128 heads over 512 + 64 latent lanes
  reduce         the shared-KV reduce: 64 heads over 512-lane rows, sliding window, compressed rows
                 (dense or selected), sink logits, inverse rotation of the output
  append         the KV page writer: rotation of the keys, bf16 or Q8_0 pages

Everything but decoder_block runs with deferred completion, as a program does that enqueues a
whole step and waits once."""
import math
import weakref

import numpy as np
import torch

from clori_amd import binding as B
from clori_amd.backend import Backend, Tensor

PAGE_LATENT = 64
GEOMETRIES = ((32, 8, 128), (40, 8, 128), (24, 4, 256), (16, 4, 64))


def listed():
    return [
        # one token of an interactive session: the smallest call, all launches and latency
        dict(name="decode-token", kind="decode", heads=32, kv_heads=8, dim=128, context=4096),
        # the same through the reference's own slots, completed call by call
        dict(name="decode-token-exact", kind="decoder_block", heads=32, kv_heads=8, dim=128, context=4096),
        # a prompt without a history, sizes of the quoted prefill configuration
        dict(name="prefill-prompt", kind="prefill", heads=40, kv_heads=8, dim=128, tokens=2048, start=0,
             gate=False, interleaved=False),
        # one chunk of a long document: many tokens behind a long history, ragged, with the gate
        dict(name="prefill-chunk", kind="prefill", heads=24, kv_heads=4, dim=256, tokens=2000, start=13333,
             gate=True, interleaved=True),
        # a few drafted tokens checked at once (or a short user turn) over a long history
        dict(name="prefill-drafts", kind="prefill", heads=40, kv_heads=8, dim=128, tokens=9, start=12001,
             gate=False, interleaved=True),
        # the reference engine's own prefill request, a prompt of odd length
        dict(name="prefill-exact", kind="prefill_exact", heads=40, kv_heads=8, dim=128, tokens=1777, start=0,
             interleaved=True),
        # a full batch of sessions of mixed length, bf16 pages: the quoted paged configuration
        dict(name="paged-bf16", kind="paged", storage="bf16", heads=32, kv_heads=8, dim=128, sessions=32,
             page=16, shortest=512, longest=16384, lengths=3, gate=False),
        # long quantised contexts: the quoted Q8_0 configuration, the largest by bytes
        dict(name="paged-q8", kind="paged", storage="q8_0", heads=32, kv_heads=8, dim=128, sessions=32,
             page=16, shortest=4096, longest=32768, lengths=4, gate=False),
        # a handful of short sessions with the gate in the epilogue, wide heads
        dict(name="paged-few", kind="paged", storage="bf16", heads=24, kv_heads=4, dim=256, sessions=5,
             page=64, shortest=100, longest=3000, lengths=5, gate=True),
        # latent attention over a batch whose contexts differ, as they do in serving
        dict(name="mla-mixed", kind="mla", batch=16, shortest=2048, longest=14336, lengths=6),
        # the reference's reduce at its model's geometry: window of 128, 512 selected rows
        dict(name="reduce-selected", kind="reduce", batch=32, window=128, shortest=1000, longest=20000,
             lengths=7, selected=512),
        # the keys and values of a batch of prompts going into Q8_0 pages
        dict(name="append-q8", kind="append", storage="q8_0", kv_heads=8, dim=128, sessions=16, page=16,
             shortest=300, longest=3700, lengths=8),
    ]


def _log(rng, low, high):
    """A whole number in [low, high], even over the logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(("decode", "decoder_block", "prefill", "prefill", "prefill_exact", "paged", "paged",
                       "mla", "reduce", "append"))
    heads, kv_heads, dim = rng.choice(GEOMETRIES)
    case = dict(kind=kind, heads=heads, kv_heads=kv_heads, dim=dim)
    lengths = rng.randrange(1000)
    if kind == "decode":
        case.update(context=_log(rng, 64, 65536))
    elif kind == "decoder_block":
        case.update(context=_log(rng, 64, 16384))
    elif kind in ("prefill", "prefill_exact"):
        start = rng.choice((0, _log(rng, 16, 32768)))
        case.update(tokens=_log(rng, 2 if start else 16, 8192 if kind == "prefill" else 4096), start=start,
                    interleaved=rng.random() < 0.5)
        if kind == "prefill":
            case.update(gate=rng.random() < 0.5)
        most = 6e11 if kind == "prefill" else 5e10
        while work(case)["flops"] > most:  # no more than the largest listed case costs
            case["start"] //= 2
            case["tokens"] = max(2, case["tokens"] * 7 // 8)
    elif kind == "paged":
        storage = rng.choice(("bf16", "q8_0"))
        if storage == "q8_0":
            heads, kv_heads, dim = rng.choice(GEOMETRIES[:2])
            case.update(heads=heads, kv_heads=kv_heads, dim=dim)
        longest = _log(rng, 256, 32768)
        case.update(storage=storage, sessions=_log(rng, 1, 64), page=rng.choice((16, 64)), longest=longest,
                    shortest=max(1, longest // rng.choice((2, 8, 32))), lengths=lengths, gate=rng.random() < 0.5)
        while work(case)["bytes"] > 1.4e9:
            case["sessions"] -= 1 + case["sessions"] // 8
    elif kind in ("mla", "reduce"):
        longest = _log(rng, 256, 32768)
        case = dict(kind=kind, batch=_log(rng, 1, 64), longest=longest,
                    shortest=max(1, longest // rng.choice((1, 2, 8, 32))), lengths=lengths)
        if kind == "reduce":
            case.update(window=128, selected=rng.choice((0, 512)))
        while case["batch"] > 1 and work(case)["flops"] > 1e11:
            case["batch"] -= 1 + case["batch"] // 8
    else:
        storage = rng.choice(("bf16", "q8_0"))
        if storage == "q8_0":
            dim = 128
        longest = _log(rng, 1, 4096)
        case = dict(kind=kind, storage=storage, kv_heads=kv_heads, dim=dim, sessions=_log(rng, 1, 64),
                    page=rng.choice((16, 64)), longest=longest, shortest=max(1, longest // 8), lengths=lengths)
    return case


# ------------------------------------------------------------------------ what a case holds --

def _contexts(case):
    """The lengths of a batch's sessions (part of the case, whatever the seed of its values)."""
    count = case.get("sessions") or case["batch"]
    return np.random.default_rng(case["lengths"]).integers(case["shortest"], case["longest"] + 1,
                                                           count).astype(np.int32)


def _compressed(case, contexts):
    """Stored compressed rows of every batch element, and how many of them it attends to: one row
    per four tokens and up to `selected` of them by a list, or one per 128 tokens and all."""
    if case["selected"]:
        stored = np.maximum(contexts // 4, 1)
        return stored, np.minimum(stored, case["selected"]).astype(np.int32)
    stored = contexts // 128
    return np.maximum(stored, 1), stored.astype(np.int32)


def work(case):
    kind = case["kind"]
    if kind in ("decode", "decoder_block"):
        size = 2 if kind == "decode" else 4
        h, kv, d, n = case["heads"], case["kv_heads"], case["dim"], case["context"]
        return dict(bytes=2 * n * kv * d * size + 3 * h * d * size, flops=4 * h * d * n)
    if kind in ("prefill", "prefill_exact"):
        size = 2 if kind == "prefill" else 4
        h, kv, d, t, s = case["heads"], case["kv_heads"], case["dim"], case["tokens"], case["start"]
        gate = t * h * d * size if case.get("gate") else 0
        return dict(bytes=2 * t * h * d * size + 2 * (s + t) * kv * d * size + gate,
                    flops=4 * d * h * (t * s + t * (t + 1) // 2))
    contexts = _contexts(case).astype(np.int64)
    tokens = int(contexts.sum())
    if kind == "paged":
        h, kv, d = case["heads"], case["kv_heads"], case["dim"]
        row = d // 32 * 34 if case["storage"] == "q8_0" else 2 * d
        return dict(bytes=2 * tokens * kv * row + int((-(-contexts // case["page"])).sum()) * 4 +
                    len(contexts) * h * d * (6 if case["gate"] else 4), flops=4 * h * d * tokens)
    if kind == "mla":
        b = len(contexts)
        return dict(bytes=tokens * 1152 + b * 128 * (576 + 512) * 2 + b * 128 * 4, flops=2 * 128 * (576 + 512) * tokens)
    if kind == "reduce":
        b = len(contexts)
        rows = int(np.minimum(contexts, case["window"]).sum() + _compressed(case, contexts)[1].sum())
        return dict(bytes=rows * 1024 + b * 64 * 1024 * 2 + b * 64 * 4, flops=2 * 64 * 1024 * rows)
    kv, d = case["kv_heads"], case["dim"]
    row = d // 32 * 34 if case["storage"] == "q8_0" else 2 * d
    return dict(bytes=tokens * (2 * kv * d * 2 + 2 * kv * row + d * 4), flops=3 * tokens * kv * d)


def tolerance(case):
    if case["kind"] == "append":
        return "exact"
    if case["kind"] == "prefill_exact":
        return dict(rel=3e-6, max=1e-4)
    if case["kind"] == "decoder_block":
        # F32 arithmetic, but the attention rows are rounded to bf16: a last bit of F32 can be a
        # bf16 step of one value
        return dict(rel=1e-3, max=8e-3)
    # seen against 64 bits: 0.3 % in the 2-norm, two bf16 steps of single values
    return dict(rel=1e-2, max=6e-2)


# ---------------------------------------------------------------------------------- program --

class _Memory:
    """A tensor of the backend as torch sees it (torch keeps this object, and so the memory)."""

    def __init__(self, tensor, typestr, count):
        self.tensor = tensor
        self.__cuda_array_interface__ = dict(shape=(count,), typestr=typestr, version=3,
                                             data=(int(tensor.handle.contents.data), False))


_TORCH = {B.DTYPE_BF16: ("<i2", torch.bfloat16), B.DTYPE_F32: ("<f4", torch.float32),
          B.DTYPE_I8: ("|i1", torch.int8), B.DTYPE_I32: ("<i4", torch.int32),
          B.DTYPE_I64: ("<i8", torch.int64)}


def _seen(tensor):
    typestr, dtype = _TORCH[tensor.dtype]
    count = tensor.nbytes // B.DTYPE_BYTES[tensor.dtype]
    return torch.as_tensor(_Memory(tensor, typestr, count), device="cuda").view(dtype).reshape(tensor.shape)


_PROGRAMS = {}


class Program:
    """What a process keeps from call to call: one backend with its completion mode and the
    attached workspace, as large as the largest request so far."""

    def __init__(self, mode):
        self.backend = Backend()
        # looking for a kernel in several code objects leaves the runtime's "not found" behind,
        # which torch would report at its next launch
        try:
            torch.zeros(1, device="cuda")
        except RuntimeError:
            pass
        self.backend.set_completion_mode(mode)
        self.workspace = None

    def room(self, nbytes):
        if nbytes and (self.workspace is None or self.workspace.nbytes < nbytes):
            self.backend.sync()
            if self.workspace is not None:
                self.backend.workspace_detach()
                self.workspace.release()
            self.workspace = self.backend.tensor("workspace", B.DTYPE_I8, (nbytes,))
            self.backend.workspace_attach(self.workspace)


def _program(mode):
    if mode not in _PROGRAMS:
        _PROGRAMS[mode] = Program(mode)
    return _PROGRAMS[mode]


def _give_back(backend, handle):
    Tensor(backend, handle, None, ()).release()


class State:
    """What one prepared case holds.  A tensor goes back to the backend when nothing refers to it
    any more: neither the state, nor a view of it, nor a torch tensor over its memory (the outputs
    of a pass, which may outlive the state)."""

    def __init__(self, case, seed, mode=B.COMPLETION_DEFERRED):
        self.case = case
        self.program = _program(mode)
        self.backend = self.program.backend
        self.generator = torch.Generator(device="cuda").manual_seed(seed)
        self.host = np.random.default_rng(seed)

    def tensor(self, name, dtype, shape, values=None):
        t = self.backend.tensor(name, dtype, shape)
        self.backend.tensors.remove(t)
        weakref.finalize(t, _give_back, self.backend, t.handle).atexit = False
        if values is None:
            t.zero()
        else:
            t.write(values)
        return t

    def normal(self, name, dtype, shape, head_scale=None):
        """N(0, 1) values, by head times `head_scale` (a [heads] tensor) when it is given."""
        t = self.tensor(name, dtype, shape)
        seen = _seen(t)
        seen.normal_(generator=self.generator)
        if head_scale is not None:
            seen.mul_(head_scale.to(seen.dtype)[:, None])
        return t

    def angles(self, tokens, rotary):
        angles = self.host.uniform(-3.0, 3.0, (tokens, rotary))
        return (self.tensor("cos", B.DTYPE_F32, (tokens, rotary), np.cos(angles).astype(np.float32)),
                self.tensor("sin", B.DTYPE_F32, (tokens, rotary), np.sin(angles).astype(np.float32)))


def _paged_table(state, contexts, page, longest):
    """Page tables of a batch: the pages of the pool in a random order."""
    need = (contexts + page - 1) // page
    stride = (longest + page - 1) // page
    order = state.host.permutation(int(need.sum())).astype(np.int32)
    table = np.zeros((len(contexts), stride), dtype=np.int32)
    at = 0
    for row, n in enumerate(need):
        table[row, :n] = order[at:at + n]
        at += int(n)
    return table, int(need.sum())


def _rows(state, dtype, tokens, width):
    """The session layer's history, one [K | V] row per token: the rows, the view of the keys, the
    view of the values, elements from token to token."""
    rows = state.normal("history", dtype, (tokens, 2 * width))
    span = (tokens - 1) * 2 * width + width
    return (rows, rows.view(0, dtype, (span,)), rows.view(width * B.DTYPE_BYTES[dtype], dtype, (span,)),
            2 * width)


def _history(state, dtype, tokens, kv_heads, dim, interleaved):
    """Key view, value view and their token strides (0: packed)."""
    if interleaved:
        _, k, v, stride = _rows(state, dtype, tokens, kv_heads * dim)
        return k, v, stride, stride
    return (state.normal("k", dtype, (tokens, kv_heads, dim)),
            state.normal("v", dtype, (tokens, kv_heads, dim)), 0, 0)


def _prepare_decode(case, seed):
    s = State(case, seed)
    h, kv, d, n = case["heads"], case["kv_heads"], case["dim"], case["context"]
    s.query = s.normal("q", B.DTYPE_BF16, (1, h, d))
    s.gate = s.normal("gate", B.DTYPE_BF16, (1, h, d))
    s.key, s.value = s.normal("k-new", B.DTYPE_BF16, (1, kv, d)), s.normal("v-new", B.DTYPE_BF16, (1, kv, d))
    s.cosine, s.sine = s.angles(1, 64)
    s.history, s.k, s.v, s.k_stride = _rows(s, B.DTYPE_BF16, n, kv * d)
    s.v_stride = s.k_stride
    s.out = s.tensor("out", B.DTYPE_BF16, (1, h, d))
    s.requirement = s.backend.attention_requirement(
        1, n, h, kv, d, causal=True, query_start=n - 1, dtype=B.DTYPE_BF16,
        contract=B.NUMERIC_BF16_F32_ACCUMULATE, k_stride=s.k_stride, v_stride=s.v_stride)
    s.program.room(s.backend.attention_workspace_required(s.requirement))
    s.result = dict(out=_seen(s.out), query=_seen(s.query), history=_seen(s.history))
    return s


def _run_decode(s):
    c = s.case
    s.backend.history_append_execute(
        s.key, s.value, s.k, s.v, c["context"] - 1, c["kv_heads"], head_dimension=c["dim"], cosine=s.cosine,
        sine=s.sine, rotary_dimension=64, key_token_stride=s.k_stride, value_token_stride=s.v_stride,
        rotary_mode=B.ROTARY_F32_ROUNDED, query=s.query, query_heads=c["heads"])
    s.backend.attention_execute(s.requirement, s.query, s.k, s.v, s.out, gate=s.gate)
    return s.result


def _prepare_decoder_block(case, seed):
    s = State(case, seed, B.COMPLETION_IMMEDIATE)
    h, kv, d, n = case["heads"], case["kv_heads"], case["dim"], case["context"]
    width = kv * d
    s.projection = s.normal("qg", B.DTYPE_F32, (1, h, 2, d))
    s.key, s.value = s.normal("k-new", B.DTYPE_F32, (1, kv, d)), s.normal("v-new", B.DTYPE_F32, (1, kv, d))
    s.cosine, s.sine = s.angles(1, 64)
    history, s.k, s.v, stride = _rows(s, B.DTYPE_F32, n, width)
    row = (n - 1) * stride * 4
    s.k_slot = history.view(row, B.DTYPE_F32, (width,))
    s.v_slot = history.view(row + width * 4, B.DTYPE_F32, (width,))
    s.k_row, s.v_row = s.key.view(0, B.DTYPE_F32, (width,)), s.value.view(0, B.DTYPE_F32, (width,))
    s.query, s.gate, s.mixer, s.gated = (s.tensor(name, B.DTYPE_F32, (1, h * d))
                                         for name in ("q", "gate", "mixer", "gated"))
    positions = s.tensor("positions", B.DTYPE_I64, (n,))
    s.position_slot = positions.view((n - 1) * 8, B.DTYPE_I64, (1,))
    s.position = np.array([n - 1], dtype=np.int64)
    s.requirement = s.backend.attention_requirement(1, n, h, kv, d, causal=True, query_start=n - 1,
                                                    k_stride=stride, v_stride=stride)
    s.program.room(s.backend.attention_workspace_required(s.requirement))
    s.result = dict(out=_seen(s.gated), history=_seen(history))
    return s


def _run_decoder_block(s):
    b, c = s.backend, s.case
    h, kv, d = c["heads"], c["kv_heads"], c["dim"]
    b.split_interleaved_two_f32(s.projection, s.query, s.gate, 1, h, d)
    b.rotary_half_f32(s.query, s.cosine, s.sine, 1, h, d, 64)
    b.bf16_round(s.query, h * d)
    b.rotary_half_f32(s.key, s.cosine, s.sine, 1, kv, d, 64)
    b.bf16_round(s.key, kv * d)
    s.k_slot.copy_from_async(s.k_row)
    s.v_slot.copy_from_async(s.v_row)
    s.position_slot.write(s.position)
    key, value = s.key.read(), s.value.read()  # the session layer keeps the new rows on the host too
    b.attention_execute(s.requirement, s.query, s.k, s.v, s.mixer)
    b.bf16_round(s.mixer, h * d)
    b.sigmoid_product_bf16(s.mixer, s.gate, s.gated, h * d)
    return dict(s.result, key=key, value=value)


def _prepare_prefill(case, seed):
    exact = case["kind"] == "prefill_exact"
    dtype = B.DTYPE_F32 if exact else B.DTYPE_BF16
    s = State(case, seed)
    h, kv, d, t, n = case["heads"], case["kv_heads"], case["dim"], case["tokens"], case["start"] + case["tokens"]
    scale = torch.empty(h, device="cuda").uniform_(0.5, 1.5, generator=s.generator)
    s.query = s.normal("q", dtype, (t, h, d), scale)
    s.k, s.v, k_stride, v_stride = _history(s, dtype, n, kv, d, case["interleaved"])
    s.gate = s.normal("gate", dtype, (t, h, d)) if case.get("gate") else None
    s.out = s.tensor("out", dtype, (t, h, d))
    s.requirement = s.backend.attention_requirement(
        t, n, h, kv, d, causal=True, query_start=case["start"], dtype=dtype,
        contract=B.NUMERIC_EXACT_F32 if exact else B.NUMERIC_BF16_F32_ACCUMULATE, k_stride=k_stride,
        v_stride=v_stride)
    s.program.room(s.backend.attention_workspace_required(s.requirement))
    s.result = dict(out=_seen(s.out))
    return s


def _run_prefill(s):
    s.backend.attention_execute(s.requirement, s.query, s.k, s.v, s.out, gate=s.gate)
    return s.result


def _prepare_paged(case, seed):
    s = State(case, seed)
    h, kv, d, page = case["heads"], case["kv_heads"], case["dim"], case["page"]
    contexts = _contexts(case)
    table, pages = _paged_table(s, contexts, page, case["longest"])
    s.table = s.tensor("table", B.DTYPE_I32, table.shape, table)
    s.context = s.tensor("contexts", B.DTYPE_I32, contexts.shape, contexts)
    storage = B.KV_Q8_0 if case["storage"] == "q8_0" else B.KV_BF16
    if storage == B.KV_BF16:
        s.k, s.v = (s.normal(name, B.DTYPE_BF16, (pages * kv * page * d,)) for name in ("k-pages", "v-pages"))
    else:
        # quantised as the program quantises: by the page writer, session by session
        count = pages * kv * page * (d // 32 * 34)
        s.k, s.v = (s.tensor(name, B.DTYPE_I8, (count,)) for name in ("k-pages", "v-pages"))
        most = int(contexts.max())
        key, value = (s.tensor(name, B.DTYPE_BF16, (most, kv, d)) for name in ("k-rows", "v-rows"))
        zero = s.tensor("zero", B.DTYPE_I32, (1,))
        for row, n in enumerate(contexts.tolist()):
            for t in (key, value):
                _seen(t).normal_(generator=s.generator)
            s.backend.kv_append_execute(
                key.view(0, B.DTYPE_BF16, (n, kv, d)), value.view(0, B.DTYPE_BF16, (n, kv, d)), zero, zero,
                s.context.view(row * 4, B.DTYPE_I32, (1,)),
                s.table.view(row * table.shape[1] * 4, B.DTYPE_I32, (1, table.shape[1])), s.k, s.v, kv, pages,
                n, storage=storage, head_dimension=d, page_tokens=page)
    s.query = s.normal("q", B.DTYPE_BF16, (len(contexts), h, d))
    s.gate = s.normal("gate", B.DTYPE_BF16, (len(contexts), h, d)) if case["gate"] else None
    s.out = s.tensor("out", B.DTYPE_BF16, (len(contexts), h, d))
    s.lse = s.tensor("lse", B.DTYPE_F32, (len(contexts), h))
    s.requirement = s.backend.paged_requirement(len(contexts), h, kv, d, page, pages, table.shape[1],
                                                case["longest"], storage=storage)
    s.program.room(s.backend.paged_decode_workspace_required(s.requirement))
    s.result = dict(out=_seen(s.out), lse=_seen(s.lse))
    return s


def _run_paged(s):
    s.backend.paged_decode_execute(s.requirement, s.query, s.k, s.v, s.table, s.context, s.out, s.lse,
                                   gate=s.gate)
    return s.result


def _prepare_mla(case, seed):
    s = State(case, seed)
    reduce = case["kind"] == "reduce"
    heads, key_dim = (64, 512) if reduce else (128, 576)
    contexts = _contexts(case)
    batch = len(contexts)
    table, pages = _paged_table(s, contexts, PAGE_LATENT, case["longest"])
    s.table = s.tensor("table", B.DTYPE_I32, table.shape, table)
    s.context = s.tensor("contexts", B.DTYPE_I32, contexts.shape, contexts)
    s.pool = s.normal("latent-pages", B.DTYPE_BF16, (pages, PAGE_LATENT, key_dim))
    s.query = s.normal("q", B.DTYPE_BF16, (batch, heads, key_dim))
    s.out = s.tensor("out", B.DTYPE_BF16, (batch, heads, 512))
    s.lse = s.tensor("lse", B.DTYPE_F32, (batch, heads))
    s.sinks = s.compressed = None
    more = {}
    if reduce:
        stored, attended = _compressed(case, contexts)
        c_table, c_pages = _paged_table(s, stored, PAGE_LATENT, int(stored.max()))
        s.sinks = s.normal("sinks", B.DTYPE_F32, (heads,))
        s.compressed = [s.normal("compressed-pages", B.DTYPE_BF16, (c_pages, PAGE_LATENT, key_dim)),
                        s.tensor("compressed-table", B.DTYPE_I32, c_table.shape, c_table),
                        s.tensor("compressed-rows", B.DTYPE_I32, (batch,), attended)]
        if case["selected"]:
            lists = np.zeros((batch, case["selected"]), dtype=np.int32)
            for row in range(batch):
                lists[row, :attended[row]] = s.host.permutation(int(stored[row]))[:attended[row]]
            s.compressed.append(s.tensor("selected", B.DTYPE_I32, lists.shape, lists))
        more = dict(sliding_window=case["window"], compressed_pool_pages=c_pages,
                    compressed_table_stride=c_table.shape[1],
                    max_compressed_tokens=int(c_table.shape[1] * PAGE_LATENT),
                    compressed_selected_stride=case["selected"],
                    output_inverse_rope=dict(rope_dimensions=64, theta=10000, scaling_factor=40,
                                             original_context=4096, beta_fast=32, beta_slow=1))
    s.requirement = s.backend.mla_requirement(batch, heads, key_dim, 512, PAGE_LATENT, pages, table.shape[1],
                                              case["longest"], **more)
    s.program.room(s.backend.mla_decode_workspace_required(s.requirement))
    s.result = dict(out=_seen(s.out), lse=_seen(s.lse))
    return s


def _run_mla(s):
    s.backend.mla_decode_execute(s.requirement, s.query, s.pool, s.table, s.context, s.out, s.lse,
                                 sinks=s.sinks, compressed=s.compressed)
    return s.result


def _prepare_append(case, seed):
    s = State(case, seed)
    kv, d, page = case["kv_heads"], case["dim"], case["page"]
    counts = _contexts(case)
    starts = np.random.default_rng(case["lengths"] + 1).integers(0, 4096, len(counts)).astype(np.int32)
    ends = starts + counts
    table, s.pages = _paged_table(s, ends, page, int(ends.max()))
    total = int(counts.sum())
    s.most = int(counts.max())
    s.storage = B.KV_Q8_0 if case["storage"] == "q8_0" else B.KV_BF16
    s.key, s.value = (s.normal(name, B.DTYPE_BF16, (total, kv, d)) for name in ("k-new", "v-new"))
    s.cosine, s.sine = s.angles(total, d)
    rows = np.concatenate(([0], np.cumsum(counts)[:-1])).astype(np.int32)
    s.rows, s.starts, s.counts = (s.tensor(name, B.DTYPE_I32, x.shape, x) for name, x in
                                  (("rows", rows), ("starts", starts), ("counts", counts)))
    s.table = s.tensor("table", B.DTYPE_I32, table.shape, table)
    dtype, count = ((B.DTYPE_I8, s.pages * kv * page * (d // 32 * 34)) if s.storage == B.KV_Q8_0 else
                    (B.DTYPE_BF16, s.pages * kv * page * d))
    s.k, s.v = (s.tensor(name, dtype, (count,)) for name in ("k-pages", "v-pages"))
    # pages are bytes to the writer: compared as whole numbers
    s.result = dict(k=_seen(s.k).view(torch.int8), v=_seen(s.v).view(torch.int8))
    return s


def _run_append(s):
    c = s.case
    s.backend.kv_append_execute(s.key, s.value, s.rows, s.starts, s.counts, s.table, s.k, s.v, c["kv_heads"],
                                s.pages, s.most, storage=s.storage, cosine=s.cosine, sine=s.sine,
                                rotary_dimension=c["dim"], head_dimension=c["dim"], page_tokens=c["page"],
                                rotary_mode=B.ROTARY_F32_ROUNDED)
    return s.result


_KINDS = dict(decode=(_prepare_decode, _run_decode),
              decoder_block=(_prepare_decoder_block, _run_decoder_block),
              prefill=(_prepare_prefill, _run_prefill), prefill_exact=(_prepare_prefill, _run_prefill),
              paged=(_prepare_paged, _run_paged), mla=(_prepare_mla, _run_mla),
              reduce=(_prepare_mla, _run_mla), append=(_prepare_append, _run_append))


def prepare(case, seed):
    s = _KINDS[case["kind"]][0](case, seed)
    s.backend.sync()
    torch.cuda.synchronize()
    return s


def run(state):
    return _KINDS[state.case["kind"]][1](state)
