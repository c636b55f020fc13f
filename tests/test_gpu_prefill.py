"""GPU parity: bf16 MFMA prefill (multi-token GQA, causal and full) against the CPU
operator, through the reference's attention_execute contract."""
import numpy as np
import pytest

from clori_amd import binding as B
from clori_amd.backend import YvexError
from gpu_common import ORACLE, assert_close_bf16, assert_lse, backend, bf16_normal  # noqa: F401

pytestmark = pytest.mark.gpu


def run_prefill(backend, q, k, v, query_start=0, causal=True, want_lse=True):
    tq, hq, d = q.shape
    tk, hkv, _ = k.shape
    req = backend.attention_requirement(tq, tk, hq, hkv, d, causal=causal, query_start=query_start,
                                        dtype=B.DTYPE_BF16,
                                        contract=B.NUMERIC_BF16_F32_ACCUMULATE)
    out = backend.tensor("o", B.DTYPE_BF16, q.shape)
    lse = backend.tensor("lse", B.DTYPE_F32, (tq, hq)) if want_lse else None
    facts = backend.attention_execute(req, backend.tensor("q", B.DTYPE_BF16, q.shape, q),
                                      backend.tensor("k", B.DTYPE_BF16, k.shape, k),
                                      backend.tensor("v", B.DTYPE_BF16, v.shape, v), out, lse=lse)
    return out.read(), (lse.read() if lse else None), facts


@pytest.mark.parametrize("tq,tk,start,hq,hkv,causal", [
    (2, 2, 0, 2, 1, True), (5, 5, 0, 1, 1, True), (64, 64, 0, 4, 2, True),
    (65, 65, 0, 5, 1, True), (257, 257, 0, 2, 2, True), (300, 300, 0, 10, 2, False),
    (3, 131, 128, 8, 2, True), (200, 1000, 800, 5, 1, True), (129, 640, 100, 4, 4, False),
    (512, 512, 0, 40, 8, True),
])
def test_prefill_matches_cpu_operator(backend, tq, tk, start, hq, hkv, causal):
    rng = np.random.default_rng(tq * 1000 + tk)
    q = bf16_normal(rng, (tq, hq, 128))
    k = bf16_normal(rng, (tk, hkv, 128))
    v = bf16_normal(rng, (tk, hkv, 128))
    got, lse, facts = run_prefill(backend, q, k, v, query_start=start, causal=causal)
    rc, ref, _, ref_lse = ORACLE.gqa_bf16(q, k, v, query_start=start, causal=causal)
    assert rc == 0
    label = "tq=%d tk=%d start=%d %s" % (tq, tk, start, "causal" if causal else "full")
    assert_close_bf16(got, ref, label)
    assert_lse(lse, ref_lse, label)
    assert facts.kernel_launches == 1 and facts.device_synchronizations == 1
    if causal and start == 0:
        # the first causal row sees only key 0: the output is exactly V[0] of its kv head
        for h in range(hq):
            assert np.array_equal(got[0, h], v[0, h // (hq // hkv)])


def test_config2_prefill_qwen_shape(backend):
    """Benchmark configuration 2: T=2048, 40/8 heads, d=128, causal, N(0,1) values with a per-head
    scale drawn U[0.5,1.5], seed 2."""
    rng = np.random.default_rng(2)
    t, hq, hkv, d = 2048, 40, 8, 128
    q = bf16_normal(rng, (t, hq, d)) if False else None
    sq = rng.uniform(0.5, 1.5, size=(1, hq, 1)).astype(np.float32)
    skv = rng.uniform(0.5, 1.5, size=(1, hkv, 1)).astype(np.float32)
    q = ORACLE.bf16_encode(rng.standard_normal((t, hq, d)).astype(np.float32) * sq)
    k = ORACLE.bf16_encode(rng.standard_normal((t, hkv, d)).astype(np.float32) * skv)
    v = ORACLE.bf16_encode(rng.standard_normal((t, hkv, d)).astype(np.float32) * skv)
    got, lse, _ = run_prefill(backend, q, k, v)
    rc, ref, _, ref_lse = ORACLE.gqa_bf16(q, k, v, query_start=0, causal=True)
    assert rc == 0
    assert_close_bf16(got, ref, "config2")
    assert_lse(lse, ref_lse, "config2")
    again, lse2, _ = run_prefill(backend, q, k, v)
    assert np.array_equal(got, again) and np.array_equal(lse, lse2)   # deterministic


def test_prefill_strided_views_equal_packed(backend):
    rng = np.random.default_rng(9)
    tq, tk, hq, hkv, d = 70, 200, 8, 2, 128
    q = bf16_normal(rng, (tq, hq, d))
    k = bf16_normal(rng, (tk, hkv, d))
    v = bf16_normal(rng, (tk, hkv, d))
    qw, kw = hq * d, hkv * d
    qi = np.full((tq, 2 * qw), 0x7FC0, dtype=np.uint16)      # [Q | gate], gate = NaN pattern
    qi[:, :qw] = q.reshape(tq, qw)
    kvi = np.zeros((tk, 2 * kw), dtype=np.uint16)           # [K | V]
    kvi[:, :kw] = k.reshape(tk, kw)
    kvi[:, kw:] = v.reshape(tk, kw)
    qs = backend.tensor("q-storage", B.DTYPE_BF16, qi.shape, qi)
    kvs = backend.tensor("kv-storage", B.DTYPE_BF16, kvi.shape, kvi)
    q_view = qs.view(0, B.DTYPE_BF16, ((tq - 1) * 2 * qw + qw,))
    k_view = kvs.view(0, B.DTYPE_BF16, ((tk - 1) * 2 * kw + kw,))
    v_view = kvs.view(kw * 2, B.DTYPE_BF16, ((tk - 1) * 2 * kw + kw,))
    out = backend.tensor("o", B.DTYPE_BF16, (tq, hq, d))
    req = backend.attention_requirement(tq, tk, hq, hkv, d, query_start=tk - tq,
                                        dtype=B.DTYPE_BF16,
                                        contract=B.NUMERIC_BF16_F32_ACCUMULATE,
                                        q_stride=2 * qw, k_stride=2 * kw, v_stride=2 * kw)
    backend.attention_execute(req, q_view, k_view, v_view, out)
    packed, _, _ = run_prefill(backend, q, k, v, query_start=tk - tq, want_lse=False)
    assert np.array_equal(out.read(), packed)


def test_prefill_refusals(backend):
    rng = np.random.default_rng(10)
    q = bf16_normal(rng, (4, 2, 128))
    k = bf16_normal(rng, (4, 1, 128))
    with pytest.raises(YvexError) as e:                      # query range beyond KV history
        run_prefill(backend, q, k, k, query_start=1)
    assert e.value.code == B.YVEX_ERR_INVALID_ARG
    req = backend.attention_requirement(4, 4, 2, 1, 96, dtype=B.DTYPE_BF16,
                                        contract=B.NUMERIC_BF16_F32_ACCUMULATE)
    with pytest.raises(YvexError) as e:                      # head dimension the MFMA path lacks
        backend.attention_workspace_required(req)
    assert e.value.code == B.YVEX_ERR_UNSUPPORTED
    qn = q.copy()
    qn[1, 0, 3] = 0x7FC0                                     # NaN query -> FORMAT, output unwritten
    out = backend.tensor("o", B.DTYPE_BF16, q.shape)
    req = backend.attention_requirement(4, 4, 2, 1, 128, dtype=B.DTYPE_BF16,
                                        contract=B.NUMERIC_BF16_F32_ACCUMULATE)
    with pytest.raises(YvexError) as e:
        backend.attention_execute(req, backend.tensor("q", B.DTYPE_BF16, q.shape, qn),
                                  backend.tensor("k", B.DTYPE_BF16, k.shape, k),
                                  backend.tensor("v", B.DTYPE_BF16, k.shape, k), out)
    assert e.value.code == B.YVEX_ERR_FORMAT and not out.is_written


@pytest.mark.parametrize("tq,tk,start,hq,hkv", [(4100, 4100, 0, 4, 1), (700, 9000, 8300, 4, 2)])
def test_prefill_long_sequences(backend, tq, tk, start, hq, hkv):
    """Twice the benchmark's sequence length, and a prompt chunk behind a long history."""
    rng = np.random.default_rng(tq + tk)
    q = bf16_normal(rng, (tq, hq, 128))
    k = bf16_normal(rng, (tk, hkv, 128))
    v = bf16_normal(rng, (tk, hkv, 128))
    got, lse, _ = run_prefill(backend, q, k, v, query_start=start, causal=True)
    rc, ref, _, ref_lse = ORACLE.gqa_bf16(q, k, v, query_start=start, causal=True)
    assert rc == 0
    assert_close_bf16(got, ref, "long prefill %d/%d" % (tq, tk))
    assert_lse(lse, ref_lse, "long prefill %d/%d" % (tq, tk))


@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("tq,tk,start,hq,hkv,causal", [
    (2, 2, 0, 2, 1, True), (65, 65, 0, 5, 1, True), (257, 257, 0, 4, 2, True),
    (300, 300, 0, 6, 2, False), (3, 131, 128, 8, 2, True), (200, 1000, 800, 4, 1, True),
    (1, 700, 699, 8, 2, True),          # one query token: a one-row tile of the same kernel
])
def test_prefill_other_head_dimensions(backend, d, tq, tk, start, hq, hkv, causal):
    """Head dimensions 64 and 256 are the same kernel with other counts (k-steps, dim blocks,
    loads per tile, LDS swizzle for 128-byte rows)."""
    rng = np.random.default_rng(d * 100000 + tq * 1000 + tk)
    q = bf16_normal(rng, (tq, hq, d))
    k = bf16_normal(rng, (tk, hkv, d))
    v = bf16_normal(rng, (tk, hkv, d))
    got, lse, facts = run_prefill(backend, q, k, v, query_start=start, causal=causal)
    rc, ref, _, ref_lse = ORACLE.gqa_bf16(q, k, v, query_start=start, causal=causal)
    assert rc == 0
    label = "d=%d tq=%d tk=%d start=%d %s" % (d, tq, tk, start, "causal" if causal else "full")
    assert_close_bf16(got, ref, label)
    assert_lse(lse, ref_lse, label)
    assert facts.kernel_launches == 1 and facts.accelerated_matrix_launches == 1
    if causal and start == 0:
        for h in range(hq):
            assert np.array_equal(got[0, h], v[0, h // (hq // hkv)])


@pytest.mark.parametrize("t,hq,hkv,d", [(1024, 24, 4, 256), (1024, 16, 4, 64)])
def test_prefill_reference_qwen_patterns(backend, t, hq, hkv, d):
    """The geometry of the reference's own Qwen attention test (24 query heads, 4 KV heads,
    head dimension 256: tests/unit/cuda/quant_qtype.c:2413-2454) and its narrow sibling, as
    causal prefill under the bf16 contract, with per-head scales as in configuration 2."""
    rng = np.random.default_rng(t + d)
    sq = rng.uniform(0.5, 1.5, size=(1, hq, 1)).astype(np.float32)
    skv = rng.uniform(0.5, 1.5, size=(1, hkv, 1)).astype(np.float32)
    q = ORACLE.bf16_encode(rng.standard_normal((t, hq, d)).astype(np.float32) * sq)
    k = ORACLE.bf16_encode(rng.standard_normal((t, hkv, d)).astype(np.float32) * skv)
    v = ORACLE.bf16_encode(rng.standard_normal((t, hkv, d)).astype(np.float32) * skv)
    got, lse, _ = run_prefill(backend, q, k, v)
    rc, ref, _, ref_lse = ORACLE.gqa_bf16(q, k, v, query_start=0, causal=True)
    assert rc == 0
    assert_close_bf16(got, ref, "qwen pattern d=%d" % d)
    assert_lse(lse, ref_lse, "qwen pattern d=%d" % d)
    again, lse2, _ = run_prefill(backend, q, k, v)
    assert np.array_equal(got, again) and np.array_equal(lse, lse2)


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("tq,tk,start,hq,hkv,causal,gated", [
    (2, 700, 690, 8, 1, True, False),     # 16 packed rows: one wave of the tile has rows
    (9, 4000, 3991, 10, 2, True, True),   # 45 rows, runs that end inside a tile
    (33, 3001, 2960, 16, 4, False, False),
    (26, 1500, 0, 5, 1, True, False),     # nothing to cut: the launch stays whole
    (300, 5000, 4700, 6, 1, True, True),  # 15 items of 128 rows
    (1300, 2600, 1300, 26, 2, True, False),  # 264 items: 256 walked whole, 8 cut
])
def test_prefill_packed_heads_and_cut_walks(backend, d, tq, tk, start, hq, hkv, causal, gated):
    """The query heads of a kv head share the rows of a tile, and with a workspace attached the
    walks that would leave compute units idle are cut into runs merged by a second launch: tails
    of rows and keys, groups from 1 to 13, runs no row of a wave sees, gate, LSE."""
    rng = np.random.default_rng(d + tq)
    q, k, v = (bf16_normal(rng, shape) for shape in ((tq, hq, d), (tk, hkv, d), (tk, hkv, d)))
    gate = bf16_normal(rng, q.shape) if gated else None
    req = backend.attention_requirement(tq, tk, hq, hkv, d, causal=causal, query_start=start, dtype=B.DTYPE_BF16,
                                        contract=B.NUMERIC_BF16_F32_ACCUMULATE)
    need = backend.attention_workspace_required(req)
    out, lse = backend.tensor("o", B.DTYPE_BF16, q.shape), backend.tensor("lse", B.DTYPE_F32, (tq, hq))
    tensors = [backend.tensor(n, B.DTYPE_BF16, x.shape, x) for n, x in (("q", q), ("k", k), ("v", v))]
    tg = backend.tensor("g", B.DTYPE_BF16, gate.shape, gate) if gated else None
    work = backend.tensor("w", B.DTYPE_I8, (max(need, 256),))
    backend.workspace_attach(work)
    try:
        facts = backend.attention_execute(req, *tensors, out, lse=lse, gate=tg)
    finally:
        backend.workspace_detach()
    assert facts.kernel_launches == (2 if need else 1) and facts.temporary_bytes == need
    assert need > 0 or tk <= 1500
    rc, ref, _, ref_lse = ORACLE.gqa_bf16(q, k, v, query_start=start, causal=causal)
    assert rc == 0
    label = "cut d=%d tq=%d tk=%d" % (d, tq, tk)
    if gated:
        ref = ref / (1.0 + np.exp(-ORACLE.bf16_decode(gate).astype(np.float64)))
    assert_close_bf16(out.read(), ref, label)
    assert_lse(lse.read(), ref_lse, label)


@pytest.mark.parametrize("d", [64, 128, 256])
def test_prefill_workspace_is_an_offer(backend, d):
    """A request that would be cut walks whole, with the same bits, when the workspace is absent or one
    byte short of what it asked for; cut and whole agree with the oracle, and either repeats itself."""
    rng = np.random.default_rng(d)
    tq, tk, hq, hkv = 7, 3000, 12, 2
    q, k, v = (bf16_normal(rng, shape) for shape in ((tq, hq, d), (tk, hkv, d), (tk, hkv, d)))
    req = backend.attention_requirement(tq, tk, hq, hkv, d, query_start=tk - tq, dtype=B.DTYPE_BF16,
                                        contract=B.NUMERIC_BF16_F32_ACCUMULATE)
    need = backend.attention_workspace_required(req)
    rc, ref, _, ref_lse = ORACLE.gqa_bf16(q, k, v, query_start=tk - tq, causal=True)
    assert rc == 0 and need > 0
    tensors = [backend.tensor(n, B.DTYPE_BF16, x.shape, x) for n, x in (("q", q), ("k", k), ("v", v))]
    out, lse = backend.tensor("o", B.DTYPE_BF16, q.shape), backend.tensor("lse", B.DTYPE_F32, (tq, hq))
    results = {}
    for size in (0, need - 1, need, need + 4096, 0):
        work = backend.tensor("w", B.DTYPE_I8, (size,)) if size else None
        if work:
            backend.workspace_attach(work)
        try:
            facts = backend.attention_execute(req, *tensors, out, lse=lse)
        finally:
            if work:
                backend.workspace_detach()
                work.release()
        cut = size >= need
        assert facts.kernel_launches == (2 if cut else 1) and facts.temporary_bytes == (need if cut else 0)
        got = out.read(), lse.read()
        assert_close_bf16(got[0], ref, "workspace of %d" % size)
        assert_lse(got[1], ref_lse, "workspace of %d" % size)
        first = results.setdefault(cut, got)
        assert np.array_equal(got[0], first[0]) and np.array_equal(got[1], first[1]), size


@pytest.mark.parametrize("tq,tk,start,hq,hkv,causal", [
    (2, 3, 1, 12, 2, True),         # one step, two rows of one wave
    (130, 130, 0, 6, 1, True),      # a second tile of two tokens
    (63, 256, 193, 24, 4, True),    # four steps below 64 tokens
    (200, 447, 247, 6, 3, False),   # seven, every row up to a ragged end
    (448, 448, 0, 24, 4, True),     # seven
    (449, 449, 0, 4, 4, True),      # eight: pairs of waves
])
def test_prefill_short_walks_at_head_dimension_256(backend, tq, tk, start, hq, hkv, causal):
    rng = np.random.default_rng(tq + tk)
    q, k, v = (bf16_normal(rng, shape) for shape in ((tq, hq, 256), (tk, hkv, 256), (tk, hkv, 256)))
    got, lse, facts = run_prefill(backend, q, k, v, query_start=start, causal=causal)
    rc, ref, _, ref_lse = ORACLE.gqa_bf16(q, k, v, query_start=start, causal=causal)
    assert rc == 0 and facts.kernel_launches == 1
    assert_close_bf16(got, ref, "short tq=%d tk=%d" % (tq, tk))
    assert_lse(lse, ref_lse, "short tq=%d tk=%d" % (tq, tk))


@pytest.mark.parametrize("tq,tk,start,hq,hkv,cut", [(70, 70, 0, 2, 1, False), (5, 1500, 1495, 12, 2, True),
                                                    (200, 1000, 800, 4, 2, False)])
def test_prefill_scores_far_above_the_first_tiles(backend, tq, tk, start, hq, hkv, cut):
    """Scores whose weight exceeds the first 64 keys' by more than a float holds: the walk relative to
    the first tile overflows and is done again with rescaling (head dimension 256).  Values of
    half size: the softmax picks single rows, one bf16 step of which stays below the bar."""
    rng = np.random.default_rng(tq)
    d = 256
    q = bf16_normal(rng, (tq, hq, d))
    k = ORACLE.bf16_encode(rng.standard_normal((tk, hkv, d)).astype(np.float32) *
                           np.where(np.arange(tk) < 64, 0.5, 48.0).astype(np.float32)[:, None, None])
    v = bf16_normal(rng, (tk, hkv, d), 0.5)
    req = backend.attention_requirement(tq, tk, hq, hkv, d, causal=True, query_start=start, dtype=B.DTYPE_BF16,
                                        contract=B.NUMERIC_BF16_F32_ACCUMULATE)
    out, lse = backend.tensor("o", B.DTYPE_BF16, q.shape), backend.tensor("lse", B.DTYPE_F32, (tq, hq))
    tensors = [backend.tensor(n, B.DTYPE_BF16, x.shape, x) for n, x in (("q", q), ("k", k), ("v", v))]
    work = backend.tensor("w", B.DTYPE_I8, (max(backend.attention_workspace_required(req), 256),))
    if cut:
        backend.workspace_attach(work)
    try:
        facts = backend.attention_execute(req, *tensors, out, lse=lse)
    finally:
        backend.workspace_detach()
    assert facts.kernel_launches == (2 if cut else 1)
    rc, ref, _, ref_lse = ORACLE.gqa_bf16(q, k, v, query_start=start, causal=True)
    assert rc == 0 and ref_lse.max() > 100.0  # e^88.8 is the first weight a float does not hold
    assert_close_bf16(out.read(), ref, "far above %d" % tq)
    # an LSE of some hundreds: its float spacing is 3e-5, the scores' own rounding (256 products) more
    assert np.abs(lse.read().astype(np.float64) - ref_lse).max() <= 1e-3
    # what is not finite in the inputs is reported, not walked into silence
    q[tq - 1, 0, 3] = 0x7F80
    tensors[0].write(q)
    with pytest.raises(YvexError) as e:
        backend.attention_execute(req, *tensors, out)
    assert e.value.code == B.YVEX_ERR_FORMAT


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("tq,tk,hq,hkv,groups", [
    (5, 4000, 10, 2, 4),  # many runs, merged by four groups of threads
    (5, 1000, 10, 2, 1),  # few runs, one group
])
def test_prefill_reports_a_run_of_keys_that_are_not_numbers(backend, d, tq, tk, hq, hkv, groups):
    """A cut walk one of whose runs sees nothing but NaN scores fails as the whole walk does, wherever
    the run lies: the first, one in the middle, the last, and as many as a group of the merge takes."""
    rng = np.random.default_rng(d + tk)
    q, k, v = (bf16_normal(rng, shape) for shape in ((tq, hq, d), (tk, hkv, d), (tk, hkv, d)))
    req = backend.attention_requirement(tq, tk, hq, hkv, d, causal=True, query_start=tk - tq, dtype=B.DTYPE_BF16,
                                        contract=B.NUMERIC_BF16_F32_ACCUMULATE)
    need = backend.attention_workspace_required(req)
    items = -(-tq * (hq // hkv) // 128) * hkv
    runs = need // (items * 128 * (d + 2) * 4)
    steps = -(-tk // 64)
    run_keys = -(-steps // runs) * 64
    assert runs >= 3 and (runs > 8) == (groups == 4)
    out, lse = backend.tensor("o", B.DTYPE_BF16, q.shape), backend.tensor("lse", B.DTYPE_F32, (tq, hq))
    tq_, tk_, tv_ = (backend.tensor(n, B.DTYPE_BF16, x.shape, x) for n, x in (("q", q), ("k", k), ("v", v)))
    work = backend.tensor("w", B.DTYPE_I8, (need,))
    group_keys = -(-runs // groups) * run_keys
    last = (steps - 1) // -(-steps // runs) * run_keys  # first key of the last run that has any
    try:
        for first, end in ((0, run_keys), (run_keys, 2 * run_keys), (last, tk), (0, group_keys), (run_keys, tk)):
            poisoned = k.copy()
            poisoned[first:end] = 0x7FC0
            tk_.write(poisoned)
            for attached in (False, True):
                if attached:
                    backend.workspace_attach(work)
                try:
                    with pytest.raises(YvexError) as e:
                        backend.attention_execute(req, tq_, tk_, tv_, out, lse=lse)
                finally:
                    if attached:
                        backend.workspace_detach()
                assert e.value.code == B.YVEX_ERR_FORMAT, (first, end, attached)
    finally:
        for t in (out, lse, tq_, tk_, tv_, work):
            t.release()


def far_above_first_tile(backend, cut, keys_of_the_sum, log2_sum):
    """Rows whose later keys all have the same score, so far above the first 64 (score 0) that the
    weights of `keys_of_the_sum` of them add up to 2^log2_sum relative to the first tile."""
    rng = np.random.default_rng(5)
    tq, tk, hq, hkv, d = 5, 1500, 12, 2, 256
    # score = (64 q0 + q1) / 16: a step of q1 is 0.09 in log2 units; all of it whole bf16 numbers
    units = round((log2_sum - np.log2(keys_of_the_sum)) * 16.0 * np.log(2.0))
    q, k = np.zeros((tq, hq, d), np.float32), np.zeros((tk, hkv, d), np.float32)
    q[:, :, 0], q[:, :, 1] = units // 64, units % 64
    k[64:, :, 0], k[64:, :, 1] = 64.0, 1.0
    # small signed values: the accumulators stay finite where the row sum does not
    v = 0.02 * rng.standard_normal((tk, hkv, d)) + np.where(np.arange(tk) < 192, 0.06, -0.04)[:, None, None]
    q, k, v = (ORACLE.bf16_encode(x.astype(np.float32)) for x in (q, k, v))
    req = backend.attention_requirement(tq, tk, hq, hkv, d, causal=True, query_start=tk - tq, dtype=B.DTYPE_BF16,
                                        contract=B.NUMERIC_BF16_F32_ACCUMULATE)
    need = backend.attention_workspace_required(req)
    out, lse = backend.tensor("o", B.DTYPE_BF16, q.shape), backend.tensor("lse", B.DTYPE_F32, (tq, hq))
    tensors = [backend.tensor(n, B.DTYPE_BF16, x.shape, x) for n, x in (("q", q), ("k", k), ("v", v))]
    work = backend.tensor("w", B.DTYPE_I8, (need,))
    if cut:
        backend.workspace_attach(work)
    try:
        facts = backend.attention_execute(req, *tensors, out, lse=lse)
    finally:
        if cut:
            backend.workspace_detach()
    assert facts.kernel_launches == (2 if cut else 1)
    rc, ref, _, ref_lse = ORACLE.gqa_bf16(q, k, v, query_start=tk - tq, causal=True)
    assert rc == 0
    label = "2^%.1f %s" % (log2_sum, "cut" if cut else "whole")
    assert_close_bf16(out.read(), ref, label)
    assert_lse(lse.read(), ref_lse, label)
    for t in [out, lse, work] + tensors:
        t.release()


@pytest.mark.parametrize("log2_sum", [float(x) for x in np.arange(125.0, 131.5, 0.5)])
def test_prefill_row_sums_about_the_largest_float(backend, log2_sum):
    """Sums that a float just holds and just does not, spread over the lanes and waves that share a
    row (each holds a quarter, which is finite up to 2^130)."""
    far_above_first_tile(backend, False, 1500 - 5 - 64, log2_sum)


@pytest.mark.parametrize("log2_sum", [float(x) for x in np.arange(125.0, 131.5, 0.5)])
def test_prefill_run_sums_about_the_largest_float(backend, log2_sum):
    """The same in one run of a cut walk (the first, which alone starts below the other keys): its
    partial is scaled by a power of two, and its share of the weights is a few per cent."""
    far_above_first_tile(backend, True, 64, log2_sum)
