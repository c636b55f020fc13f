"""GPU parity for the exact F32 contract: the reference's own test vectors and refusal
behaviour (tests/unit/backend_ops.c:444-532, tests/unit/cuda/ops.c:567-623,
tests/unit/cuda/quant_qtype.c:2100-2970), run through the C ABI."""
import math

import numpy as np
import pytest

import reference_vectors as rv
from clori_amd import binding as B
from clori_amd.backend import YvexError
from gpu_common import ORACLE, backend  # noqa: F401

pytestmark = pytest.mark.gpu


def f32(backend, name, array=None, shape=None):
    if array is not None:
        array = np.ascontiguousarray(array, dtype=np.float32)
        return backend.tensor(name, B.DTYPE_F32, array.shape, array)
    return backend.tensor(name, B.DTYPE_F32, shape)


def test_bounded_primitive_reference_literals(backend):
    q = f32(backend, "attention_query", rv.CPU_OP_QUERY)
    k = f32(backend, "attention_keys", rv.CPU_OP_KEYS)
    v = f32(backend, "attention_values", rv.CPU_OP_VALUES)
    s = f32(backend, "attention_scores", shape=(3,))
    p = f32(backend, "attention_probabilities", shape=(3,))
    o = f32(backend, "attention_out", shape=(4,))
    assert not o.is_written
    backend.op_attention(q, k, v, 3, 0, 0.5, True, s, p, o)
    assert np.allclose(o.read(), rv.CPU_OP_VALUES[0], atol=1e-6) and o.is_written
    backend.op_attention(q, k, v, 3, 2, 0.5, True, s, p, o)
    rc, ref, ref_s, ref_p, _ = ORACLE.attention_head(rv.CPU_OP_QUERY, rv.CPU_OP_KEYS,
                                                     rv.CPU_OP_VALUES, 2, 0.5)
    assert np.allclose(o.read(), ref, atol=1e-6)
    assert np.allclose(s.read(), ref_s, atol=1e-7) and np.allclose(p.read(), ref_p, atol=1e-7)
    backend.op_attention(q, k, v, 3, 0, 0.5, False, s, p, o)      # non-causal sees all rows
    assert np.allclose(o.read(), ref, atol=1e-6)
    with pytest.raises(YvexError) as e:
        backend.op_attention(q, k, v, 3, 3, 0.5, True, s, p, o)
    assert e.value.code == B.YVEX_ERR_BOUNDS and "position-out-of-range" in e.value.message
    with pytest.raises(YvexError) as e:
        backend.op_attention(q, k, v, 0, 0, 0.5, True, s, p, o)
    assert e.value.code == B.YVEX_ERR_INVALID_ARG
    for scale in (float("nan"), 0.0, -1.0, float("inf")):
        with pytest.raises(YvexError) as e:
            backend.op_attention(q, k, v, 3, 0, scale, True, s, p, o)
        assert e.value.code == B.YVEX_ERR_INVALID_ARG
    wrong = f32(backend, "wrong", shape=(5,))
    with pytest.raises(YvexError) as e:
        backend.op_attention(q, k, v, 3, 0, 0.5, True, s, p, wrong)
    assert e.value.code == B.YVEX_ERR_FORMAT
    half = backend.tensor("half", B.DTYPE_BF16, (4,))
    with pytest.raises(YvexError) as e:
        backend.op_attention(q, k, v, 3, 0, 0.5, True, s, p, half)
    assert e.value.code == B.YVEX_ERR_UNSUPPORTED


def test_bounded_primitive_long_row_matches_cpu_operator(backend):
    rng = np.random.default_rng(12)
    n, d = 4096, 128
    qv = rng.standard_normal(d).astype(np.float32)
    kv = rng.standard_normal((n, d)).astype(np.float32)
    vv = rng.standard_normal((n, d)).astype(np.float32)
    q, k, v = f32(backend, "q", qv), f32(backend, "k", kv), f32(backend, "v", vv)
    s, p, o = f32(backend, "s", shape=(n,)), f32(backend, "p", shape=(n,)), f32(backend, "o", shape=(d,))
    scale = 1.0 / math.sqrt(d)
    backend.op_attention(q, k, v, n, n - 1, scale, True, s, p, o)
    rc, ref, ref_s, ref_p, _ = ORACLE.attention_head(qv, kv, vv, n - 1, scale)
    assert np.allclose(o.read(), ref, atol=1e-6)
    assert np.allclose(s.read(), ref_s, atol=1e-6) and abs(p.read().sum() - 1.0) < 1e-5


def execute(backend, q, k, v, query_start=0, causal=True, **kw):
    tq, hq, d = q.shape
    tk, hkv, _ = k.shape
    req = backend.attention_requirement(tq, tk, hq, hkv, d, causal=causal, query_start=query_start,
                                        **kw)
    out = f32(backend, "out", shape=(tq, hq, d))
    facts = backend.attention_execute(req, f32(backend, "q", q), f32(backend, "k", k),
                                      f32(backend, "v", v), out)
    return out.read(), facts


def test_gqa_known_answer(backend):
    q, k, v, mixed = rv.gqa_kat()
    out, facts = execute(backend, q, k, v, causal=True)
    assert facts.kernel_launches == 1 and facts.device_synchronizations == 1
    assert np.array_equal(out[0], np.array([[2.0, 4.0], [2.0, 4.0]], np.float32))
    assert np.allclose(out[1], mixed, atol=1e-6)
    out, _ = execute(backend, q, k, v, causal=False)
    assert np.allclose(out, np.broadcast_to(mixed, (2, 2, 2)), atol=1e-6)
    req = backend.attention_requirement(2, 2, 2, 1, 2)
    assert backend.attention_workspace_required(req) == 0


@pytest.mark.parametrize("maker,tol_abs,tol_rel", [
    (rv.small_5x128, 2e-5, 0.0), (rv.qwen_24_4_256, 2e-4, 2e-4), (rv.tiled_257x128, 0.0, 2e-3)])
def test_gqa_reference_patterns(backend, maker, tol_abs, tol_rel):
    q, k, v = maker()
    for causal in (True, False):
        out, _ = execute(backend, q, k, v, causal=causal)
        rc, ref, _ = ORACLE.gqa(q, k, v, causal=causal)
        assert rc == 0
        assert np.all(np.abs(out - ref) <= tol_abs + tol_rel * (1.0 + np.abs(ref)) + 1e-7)
        # and far tighter against the CPU operator: double statistics on the row kernel, float
        # ones (as in the reference's device kernel) on the matrix-core kernel
        assert np.abs(out - ref).max() < (2e-5 if q.shape[0] >= 32 else 2e-6)
        again, _ = execute(backend, q, k, v, causal=causal)
        assert np.array_equal(out, again)               # deterministic: byte-identical repeat


def test_gqa_cached_decode_strided_and_refusals(backend):
    q, k, v = rv.cached_decode_qwen()
    out, _ = execute(backend, q, k, v, query_start=2)
    rc, ref, _ = ORACLE.gqa(q, k, v, query_start=2)
    assert np.abs(out - ref).max() < 2e-6
    with pytest.raises(YvexError) as e:
        execute(backend, q, k, v, query_start=3)                    # query range beyond KV
    assert e.value.code == B.YVEX_ERR_INVALID_ARG
    # strided [Q|gate] and [K|V] views
    q, k, v = rv.strided_qwen()
    tq, hq, d = q.shape
    tk, hkv, _ = k.shape
    qi = np.full((tq, 2 * hq * d), 55.0, np.float32)
    qi[:, :hq * d] = q.reshape(tq, -1)
    kvi = np.zeros((tk, 2 * hkv * d), np.float32)
    kvi[:, :hkv * d] = k.reshape(tk, -1)
    kvi[:, hkv * d:] = v.reshape(tk, -1)
    qs = f32(backend, "q-storage", qi)
    kvs = f32(backend, "kv-storage", kvi)
    q_view = qs.view(0, B.DTYPE_F32, ((tq - 1) * 2 * hq * d + hq * d,))
    k_view = kvs.view(0, B.DTYPE_F32, ((tk - 1) * 2 * hkv * d + hkv * d,))
    v_view = kvs.view(hkv * d * 4, B.DTYPE_F32, ((tk - 1) * 2 * hkv * d + hkv * d,))
    out_t = f32(backend, "out", shape=(tq, hq, d))
    req = backend.attention_requirement(tq, tk, hq, hkv, d, query_start=2, q_stride=2 * hq * d,
                                        k_stride=2 * hkv * d, v_stride=2 * hkv * d)
    backend.attention_execute(req, q_view, k_view, v_view, out_t)
    packed, _ = execute(backend, q, k, v, query_start=2)
    assert np.array_equal(out_t.read(), packed)                     # strided == packed, bit for bit
    req.query_token_stride = hq * d - 1
    with pytest.raises(YvexError) as e:
        backend.attention_execute(req, q_view, k_view, v_view, out_t)
    assert e.value.code == B.YVEX_ERR_INVALID_ARG                   # stride below the row width


def test_gqa_admission_is_fail_closed(backend):
    q, k, v = rv.small_5x128()
    # head dimension beyond the admitted bound
    req = backend.attention_requirement(3, 3, 24, 4, 257)
    with pytest.raises(YvexError) as e:
        backend.attention_workspace_required(req)
    assert e.value.code == B.YVEX_ERR_UNSUPPORTED
    # a bf16 output under the exact contract is a silent precision change: refused
    req = backend.attention_requirement(5, 5, 1, 1, 128)
    req.output_dtype = B.DTYPE_BF16
    with pytest.raises(YvexError) as e:
        backend.attention_workspace_required(req)
    assert e.value.code == B.YVEX_ERR_UNSUPPORTED
    # F32 tensors under the bf16 contract are refused as well
    req = backend.attention_requirement(5, 5, 1, 1, 128, contract=B.NUMERIC_BF16_F32_ACCUMULATE)
    with pytest.raises(YvexError) as e:
        backend.attention_workspace_required(req)
    assert e.value.code == B.YVEX_ERR_UNSUPPORTED
    req = backend.attention_requirement(5, 5, 1, 1, 128, deterministic=0)
    with pytest.raises(YvexError) as e:
        backend.attention_workspace_required(req)
    assert e.value.code == B.YVEX_ERR_UNSUPPORTED
    # NaN input -> YVEX_ERR_FORMAT through the device status word; output stays unwritten
    qn = q.copy()
    qn[2, 0, 5] = np.nan
    req = backend.attention_requirement(5, 5, 1, 1, 128)
    out = f32(backend, "out", shape=(5, 1, 128))
    with pytest.raises(YvexError) as e:
        backend.attention_execute(req, f32(backend, "q", qn), f32(backend, "k", k),
                                  f32(backend, "v", v), out)
    assert e.value.code == B.YVEX_ERR_FORMAT and not out.is_written
    # inputs that were never written are refused
    with pytest.raises(YvexError) as e:
        backend.attention_execute(req, f32(backend, "q", shape=(5, 1, 128)), f32(backend, "k", k),
                                  f32(backend, "v", v), out)
    assert e.value.code == B.YVEX_ERR_FORMAT
    good, _ = execute(backend, q, k, v)                            # backend still healthy
    assert np.all(np.isfinite(good))


def test_gqa_uniform_analytic_large(backend):
    for tokens in (65, 5757):
        q, k, v = rv.uniform_large(tokens, 2)
        out, _ = execute(backend, q, k, v, causal=False)
        assert np.abs(out - v).max() <= 2e-3 and np.abs(out - v).max() < 1e-5


def test_lse_output_exact_contract(backend):
    rng = np.random.default_rng(8)
    q = rng.standard_normal((3, 4, 64)).astype(np.float32)
    k = rng.standard_normal((9, 2, 64)).astype(np.float32)
    v = rng.standard_normal((9, 2, 64)).astype(np.float32)
    req = backend.attention_requirement(3, 9, 4, 2, 64, query_start=6)
    out = f32(backend, "out", shape=(3, 4, 64))
    lse = f32(backend, "lse", shape=(3, 4))
    backend.attention_execute(req, f32(backend, "q", q), f32(backend, "k", k), f32(backend, "v", v),
                              out, lse=lse)
    rc, ref, ref_lse = ORACLE.gqa(q, k, v, query_start=6)
    assert np.abs(out.read() - ref).max() < 2e-6
    assert np.abs(lse.read() - ref_lse).max() < 1e-5


# ------------------------------------------------ the fp32 matrix-core kernel ----

def run_exact(backend, q, k, v, **kw):
    tq, hq, d = q.shape
    tk, hkv, _ = k.shape
    req = backend.attention_requirement(tq, tk, hq, hkv, d, **kw)
    tensors = [f32(backend, "q", q), f32(backend, "k", k), f32(backend, "v", v)]
    out, lse = f32(backend, "out", shape=(tq, hq, d)), f32(backend, "lse", shape=(tq, hq))
    facts = backend.attention_execute(req, *tensors, out, lse=lse)
    result = out.read(), lse.read(), facts
    for t in tensors + [out, lse]:
        t.release()
    return result


@pytest.mark.parametrize("tq,tk,hq,hkv,d,start,causal", [
    (32, 32, 4, 2, 64, 0, True), (33, 33, 4, 1, 128, 0, True), (128, 128, 2, 2, 128, 0, True),
    (129, 129, 5, 1, 64, 0, True), (257, 257, 8, 2, 128, 0, True), (257, 257, 8, 2, 128, 0, False),
    (100, 371, 4, 4, 64, 271, True), (40, 1000, 10, 2, 128, 960, True), (64, 95, 3, 3, 128, 0, False),
    (32, 32, 6, 1, 256, 0, True), (161, 161, 6, 2, 256, 0, True), (70, 333, 24, 4, 256, 263, True),
    (96, 200, 4, 4, 256, 0, False),
])
def test_gqa_matrix_core_kernel_matches_cpu_operator(backend, tq, tk, hq, hkv, d, start, causal):
    """Prefill-shaped EXACT_F32 requests run in tiles on the fp32 matrix cores.  Tolerance is
    the reference's own for its float device kernel against the CPU operator
    (tests/unit/cuda/quant_qtype.c:2293-2333: 2e-5 absolute on N(0,1)-scale rows); ragged
    query and key tails, GQA groups of 1 to 5, cached prefixes and both masks."""
    rng = np.random.default_rng(tq * 131 + tk + d)
    q = rng.standard_normal((tq, hq, d)).astype(np.float32)
    k = rng.standard_normal((tk, hkv, d)).astype(np.float32)
    v = rng.standard_normal((tk, hkv, d)).astype(np.float32)
    out, lse, facts = run_exact(backend, q, k, v, query_start=start, causal=causal)
    assert facts.kernel_launches == 1 and facts.accelerated_matrix_launches == 1
    rc, ref, ref_lse = ORACLE.gqa(q, k, v, query_start=start, causal=causal)
    assert rc == 0
    assert np.abs(out - ref).max() < 2e-5, np.abs(out - ref).max()
    assert np.abs(lse - ref_lse).max() < 2e-5
    again, _, _ = run_exact(backend, q, k, v, query_start=start, causal=causal)
    assert np.array_equal(out, again)                   # deterministic: byte-identical repeat


def test_gqa_kernel_choice_is_a_function_of_geometry(backend):
    """Decode-shaped and odd-sized requests keep the row kernel (double statistics); the two
    kernels agree within the float kernel's tolerance where both could run."""
    rng = np.random.default_rng(77)
    k = rng.standard_normal((300, 2, 128)).astype(np.float32)
    v = rng.standard_normal((300, 2, 128)).astype(np.float32)
    q = rng.standard_normal((32, 4, 128)).astype(np.float32)
    tiled, _, facts = run_exact(backend, q, k, v, query_start=268)
    assert facts.accelerated_matrix_launches == 1
    rows, _, facts = run_exact(backend, q[:31], k[:299], v[:299], query_start=268)   # 31 tokens
    assert facts.accelerated_matrix_launches == 0
    assert np.abs(rows - tiled[:31]).max() < 2e-5
    _, _, facts = run_exact(backend, rng.standard_normal((40, 2, 96)).astype(np.float32),
                            rng.standard_normal((40, 1, 96)).astype(np.float32),
                            rng.standard_normal((40, 1, 96)).astype(np.float32))     # d = 96
    assert facts.accelerated_matrix_launches == 0
    # interleaved [K|V] rows: strided == packed, bit for bit, on the matrix-core kernel too
    tq, hq, d, tk, hkv = 64, 4, 64, 200, 2
    q = rng.standard_normal((tq, hq, d)).astype(np.float32)
    k = rng.standard_normal((tk, hkv, d)).astype(np.float32)
    v = rng.standard_normal((tk, hkv, d)).astype(np.float32)
    kvi = np.zeros((tk, 2 * hkv * d), np.float32)
    kvi[:, :hkv * d] = k.reshape(tk, -1)
    kvi[:, hkv * d:] = v.reshape(tk, -1)
    kvs = f32(backend, "kv-storage", kvi)
    k_view = kvs.view(0, B.DTYPE_F32, ((tk - 1) * 2 * hkv * d + hkv * d,))
    v_view = kvs.view(hkv * d * 4, B.DTYPE_F32, ((tk - 1) * 2 * hkv * d + hkv * d,))
    out_t = f32(backend, "out", shape=(tq, hq, d))
    req = backend.attention_requirement(tq, tk, hq, hkv, d, query_start=tk - tq,
                                        k_stride=2 * hkv * d, v_stride=2 * hkv * d)
    facts = backend.attention_execute(req, f32(backend, "q", q), k_view, v_view, out_t)
    assert facts.accelerated_matrix_launches == 1
    packed, _, _ = run_exact(backend, q, k, v, query_start=tk - tq)
    assert np.array_equal(out_t.read(), packed)


def test_gqa_matrix_core_kernel_flags_non_finite_input(backend):
    rng = np.random.default_rng(78)
    q = rng.standard_normal((64, 2, 64)).astype(np.float32)
    k = rng.standard_normal((64, 1, 64)).astype(np.float32)
    v = rng.standard_normal((64, 1, 64)).astype(np.float32)
    k[17, 0, 3] = np.nan
    with pytest.raises(YvexError) as e:
        run_exact(backend, q, k, v)
    assert e.value.code == B.YVEX_ERR_FORMAT
    good, _, _ = run_exact(backend, q, np.nan_to_num(k), v)       # backend still healthy
    assert np.all(np.isfinite(good))


def test_gqa_matrix_core_kernel_config2_shape(backend):
    """The prefill configuration (2048 tokens, 40/8 heads, d=128) under the exact contract:
    a uniform-key input has the running mean of V as its closed form, and sampled heads are
    held against the CPU operator."""
    rng = np.random.default_rng(79)
    t, hq, hkv, d = 2048, 40, 8, 128
    q = rng.standard_normal((t, hq, d)).astype(np.float32)
    k = rng.standard_normal((t, hkv, d)).astype(np.float32)
    v = rng.standard_normal((t, hkv, d)).astype(np.float32)
    out, lse, facts = run_exact(backend, q, k, v)
    assert facts.accelerated_matrix_launches == 1
    for head in (0, 17, 39):
        group = head // (hq // hkv)
        rc, ref, ref_lse = ORACLE.gqa(q[:, head:head + 1], k[:, group:group + 1], v[:, group:group + 1])
        assert rc == 0
        assert np.abs(out[:, head] - ref[:, 0]).max() < 2e-5
        assert np.abs(lse[:, head] - ref_lse[:, 0]).max() < 2e-5
    # zero queries: every visible key weighs the same, the output is the causal running mean
    out, lse, _ = run_exact(backend, np.zeros_like(q), k, v)
    mean = np.cumsum(v.astype(np.float64), axis=0) / np.arange(1, t + 1)[:, None, None]
    want = np.repeat(mean, hq // hkv, axis=1)
    assert np.abs(out - want).max() < 1e-5
    assert np.abs(lse - np.log(np.arange(1, t + 1))[:, None]).max() < 1e-5


@pytest.mark.parametrize("tq,start,hq,hkv,d", [(1000, 0, 40, 8, 128), (777, 300, 48, 8, 64),
                                               (2048, 0, 24, 4, 256)])
def test_gqa_matrix_core_kernel_scheduled_launch_equals_the_first(backend, tq, start, hq, hkv, d):
    """A causal geometry that repeats is launched from item lists (equal work per compute unit)
    from its second call on: the same items, so every output bit and every LSE bit equals the
    first call's, ragged last tiles and a query offset included; sampled heads against the CPU
    operator."""
    rng = np.random.default_rng(tq + d)
    tk = start + tq
    q = rng.standard_normal((tq, hq, d)).astype(np.float32)
    k = rng.standard_normal((tk, hkv, d)).astype(np.float32)
    v = rng.standard_normal((tk, hkv, d)).astype(np.float32)
    req = backend.attention_requirement(tq, tk, hq, hkv, d, query_start=start)
    tensors = [f32(backend, "q", q), f32(backend, "k", k), f32(backend, "v", v)]
    results = []
    for _ in range(3):
        out, lse = f32(backend, "out", shape=(tq, hq, d)), f32(backend, "lse", shape=(tq, hq))
        facts = backend.attention_execute(req, *tensors, out, lse=lse)
        assert facts.accelerated_matrix_launches == 1
        results.append((out.read(), lse.read()))
        out.release()
        lse.release()
    for out, lse in results[1:]:
        assert np.array_equal(out.view(np.uint32), results[0][0].view(np.uint32))
        assert np.array_equal(lse.view(np.uint32), results[0][1].view(np.uint32))
    for head in (0, hq // 2 + 1, hq - 1):
        group = head // (hq // hkv)
        rc, ref, ref_lse = ORACLE.gqa(q[:, head:head + 1], k[:, group:group + 1], v[:, group:group + 1],
                                      query_start=start)
        assert rc == 0
        assert np.abs(results[2][0][:, head] - ref[:, 0]).max() < 2e-5
        assert np.abs(results[2][1][:, head] - ref_lse[:, 0]).max() < 2e-5
    for t in tensors:
        t.release()


def as_halves_cases():
    """(name, q, k, v): rows of other magnitudes than N(0,1)."""
    def rows(seed, tq, tk, hq, hkv, d):
        rng = np.random.default_rng(seed)
        return (rng.standard_normal((tq, hq, d)).astype(np.float32),
                rng.standard_normal((tk, hkv, d)).astype(np.float32),
                rng.standard_normal((tk, hkv, d)).astype(np.float32))
    for d, hq, hkv in ((64, 2, 1), (128, 2, 2), (256, 2, 1)):
        q, k, v = rows(d, 65, 161, hq, hkv, d)
        yield "powers-%d" % d, q * np.float32(2.0 ** -40), k * np.float32(2.0 ** 40), v * np.float32(2.0 ** -90)
        yield "largest-%d" % d, q * np.float32(2.0 ** 45), k * np.float32(2.0 ** -45), v * np.float32(2.0 ** 45)
        # value rows that grow along the history, and whole groups of keys and values that are zero
        grown = v * np.exp2(np.linspace(-20, 12, v.shape[0])).astype(np.float32)[:, None, None]
        grown[:8] = 0.0
        grown[64:96] = 0.0
        zeroed = k.copy()
        zeroed[8:16] = 0.0
        yield "grown-%d" % d, q, zeroed, grown
        # one value, and one key, far past the others
        past = v.copy()
        past[100, 0, 3] = np.float32(2.0 ** 70)
        yield "past-%d" % d, q, k, past
        low = k.copy()
        low[40] = np.float32(-2.0 ** 60) * np.sign(q[0, 0])
        yield "far-key-%d" % d, np.abs(q) + np.float32(0.5), -np.abs(low), v


@pytest.mark.parametrize("case", list(as_halves_cases()), ids=lambda c: c[0])
@pytest.mark.parametrize("causal", [True, False])
def test_gqa_matrix_core_kernel_follows_magnitudes(backend, case, causal):
    """Scores keep the size that N(0,1) rows give (or saturate to a weight of zero), so every element keeps its bits
    relative to sum w |v| of it, in one launch and with the workspace."""
    _, q, k, v = case
    start = k.shape[0] - q.shape[0] - 7 if causal else 0
    out, lse, facts = run_exact(backend, q, k, v, query_start=start, causal=causal)
    assert facts.accelerated_matrix_launches == 1
    rc, ref, ref_lse = ORACLE.gqa(q, k, v, query_start=start, causal=causal)
    assert rc == 0
    attached, attached_lse, facts, need = run_attached(backend, q, k, v, query_start=start, causal=causal)
    assert need > 0 and facts.temporary_bytes == need
    # (scores of the far key's case are all of one sign, up to 16)
    bound = spread_bound("sink-deep" if "far-key" in case[0] else "", q.shape[2])
    for got, got_lse in ((out, lse), (attached, attached_lse)):
        assert relative_to_weighted_magnitudes(got, q, k, v, start, causal) < bound
        assert np.abs(got_lse - ref_lse).max() < 2e-5 * max(1.0, np.abs(ref_lse).max())


def spread_cases(d, power, tq=64, tk=500, hq=4, hkv=2):
    """(label, q, k, v, query_start): N(0,1) rows, and one row, channel or component that is 2^power of that while
    scores stay moderate (or exclude a key altogether).  Dimension 0 of the queries is positive, so that a key can be
    excluded through it; the last keys are seen by no query."""
    rng = np.random.default_rng(power * 1000 + d + tk)
    q, k, v = (rng.standard_normal(s).astype(np.float32) for s in ((tq, hq, d), (tk, hkv, d), (tk, hkv, d)))
    q[..., 0] = np.abs(q[..., 0]) + np.float32(1.0)
    big = np.float32(2.0 ** power)
    start = tk - tq - 21
    last = start + tq                       # the first key that no query sees

    def changed(array, where, by):
        array = array.copy()
        array[where] = by(array[where])
        return array

    def grow(x):
        return x * big

    for label, key in (("octet", last), ("tile", last + 8), ("later", last - 1), ("later-tile", last - 30)):
        yield "key-" + label, q, changed(k, np.s_[key, :, 1:], grow), v, start
        yield "value-" + label, q, k, changed(v, key, grow), start
    for label, key in (("early", 3), ("late", start - 5)):
        excluded = changed(k, np.s_[key, :, 0], lambda x: -big * np.float32(d))
        yield "excluded-" + label, q, excluded, v, start
        yield "excluded-value-" + label, q, excluded, changed(v, key, grow), start
        yield "excluded-component-" + label, q, excluded, changed(v, np.s_[key, :, 5], grow), start
        yield "component-" + label, q, k, changed(v, np.s_[key, :, 5], grow), start
    yield "value-channel", q, k, changed(v, np.s_[:, :, 7], grow), start
    yield "value-row-small", q, k, changed(v, np.s_[40:48], lambda x: x / big), start
    quiet_k, quiet_q = changed(k, np.s_[..., 9], np.zeros_like), changed(q, np.s_[..., 9], np.zeros_like)
    yield "query-channel", changed(q, np.s_[..., 9], grow), quiet_k, v, start
    yield "query-one", changed(q, np.s_[tq // 2, 1], grow), k, v, start
    yield "key-channel", quiet_q, changed(k, np.s_[..., 9], grow), v, start
    # a first key that takes all but 2^-5 to 2^-17 of the weight, with a value near zero, or zero
    for label, extra, factor in (("", 8.0, 1e-4), ("-deep", 16.0, 1e-6), ("-zero", 16.0, 0.0)):
        sink = changed(k, np.s_[0, :, 0], lambda x: np.float32(extra * math.sqrt(d)))
        yield "sink" + label, changed(q, np.s_[..., 0], lambda x: np.ones_like(x)), sink, \
            changed(v, 0, lambda x: x * np.float32(factor)), start


def relative_to_weighted_magnitudes(out, q, k, v, start, causal=True):
    """The largest error of an output element against 64 bits, relative to sum w |v| of that element."""
    tq, hq, d = q.shape
    worst = 0.0
    for head in range(hq):
        kv = head // (hq // k.shape[1])
        scores = q[:, head].astype(np.float64) @ k[:, kv].astype(np.float64).T / math.sqrt(d)
        if causal:
            scores[np.arange(k.shape[0])[None, :] > (start + np.arange(tq))[:, None]] = -np.inf
        weights = np.exp(scores - scores.max(axis=1, keepdims=True))
        weights /= weights.sum(axis=1, keepdims=True)
        values = v[:, kv].astype(np.float64)
        size = weights @ np.abs(values)
        error = np.abs(out[:, head].astype(np.float64) - weights @ values)
        worst = max(worst, float((error / np.where(size > 0.0, size, 1.0)).max()))
    return worst


# A score is a sum of d products, rounded d / 2 times on the way (two lane halves): a random walk of
# sqrt(d / 2) 2^-25 sum |q k| / sqrt(d), with |q k| of 0.64 on average 0.6e-7 d, 1.5e-6 at 256 where all of it goes
# one way; weights carry it into the sum, which adds a few 2^-24 of its own (seen: 2.6e-6 of 4e-6).  Behind a sink the
# weights are relative to a score of 8 (16 where it is deep), summed first, so that each of the d / 2 roundings
# is one of that size: sqrt(d / 2) 2^-25 of it, 5.4e-6 at 256, twice that for the largest of some 10^5 rows (seen:
# 5.8e-6 and 1.1e-5; both forms alike).
def spread_bound(label, d):
    sink = 0.0 if not label.startswith("sink") else 8.0 if label == "sink" else 16.0
    return 4e-6 + 2.0 * math.sqrt(d / 2.0) * 2.0 ** -25 * sink


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("power", [16, 24, 32, 40, 50])
def test_gqa_matrix_core_kernel_holds_the_spread(backend, d, power):
    """One row, channel or component of 2^16 to 2^50 among N(0,1) ones, seen, unseen or of weight zero, and sinks:
    every output element keeps its bits relative to sum w |v| of that element."""
    for label, q, k, v, start in spread_cases(d, power):
        out, lse, facts = run_exact(backend, q, k, v, query_start=start)
        assert facts.accelerated_matrix_launches == 1 and facts.kernel_launches == 1
        worst = relative_to_weighted_magnitudes(out, q, k, v, start)
        assert worst < spread_bound(label, d), (label, worst)


@pytest.mark.parametrize("d,hq,hkv", [(64, 2, 1), (128, 5, 1), (256, 2, 1)])
def test_gqa_matrix_core_kernel_infinities(backend, d, hq, hkv):
    """An infinite key that no query sees changes nothing; one that a query sees, with a product of one sign
    that excludes the key, or an infinite value, ends as the fp32 walk ends it."""
    rng = np.random.default_rng(d + 1)
    q = (np.abs(rng.standard_normal((64, hq, d))) + 0.1).astype(np.float32)
    k = rng.standard_normal((96, hkv, d)).astype(np.float32)
    v = rng.standard_normal((96, hkv, d)).astype(np.float32)
    good, _, _ = run_exact(backend, q, k, v, query_start=0)
    bad = k.copy()
    bad[64:] = np.inf
    same, _, _ = run_exact(backend, q, bad, v, query_start=0)       # keys 64.. are past every query
    assert np.abs(same - good).max() < 2e-5
    bad = k.copy()
    bad[5, 0, 2] = -np.inf                                         # a score of -inf: a weight of zero
    out, _, _ = run_exact(backend, q, bad, v, query_start=0)
    rc, ref, _ = ORACLE.gqa(q, np.where(np.isinf(bad), np.float32(-1e30), bad), v)
    assert rc == 0 and np.abs(out - ref).max() < 2e-5
    for value in (np.inf, np.nan):
        bad = v.copy()
        bad[9, 0, 1] = value
        with pytest.raises(YvexError) as e:
            run_exact(backend, q, k, bad, query_start=0)
        assert e.value.code == B.YVEX_ERR_FORMAT


def run_attached(backend, q, k, v, short=0, **kw):
    """run_exact with the workspace that the request asks for attached (`short` bytes less of it)."""
    tq, hq, d = q.shape
    tk, hkv, _ = k.shape
    need = backend.attention_workspace_required(backend.attention_requirement(tq, tk, hq, hkv, d, **kw))
    work = backend.tensor("work", B.DTYPE_I8, (max(need - short, 256),))
    backend.workspace_attach(work)
    try:
        return run_exact(backend, q, k, v, **kw) + (need,)
    finally:
        backend.workspace_detach()
        work.release()


@pytest.mark.parametrize("tq,tk,hq,hkv,d,start,causal", [
    (32, 64, 4, 2, 128, 32, True), (64, 64, 3, 1, 64, 0, True), (33, 65, 2, 1, 256, 32, True),
    (95, 96, 5, 1, 64, 0, False),
    (33, 320, 4, 1, 128, 287, True), (129, 385, 10, 2, 128, 256, True), (1000, 1000, 5, 1, 128, 0, True),
    (40, 3001, 10, 2, 128, 2950, True), (64, 799, 3, 3, 128, 0, False), (520, 1040, 40, 8, 128, 520, True),
    (32, 256, 6, 2, 64, 224, True), (1300, 1300, 16, 4, 64, 0, True), (77, 9000, 7, 1, 64, 8923, True),
    (100, 700, 4, 4, 64, 3, False), (32, 448, 6, 1, 256, 416, True), (700, 700, 6, 2, 256, 0, True),
    (50, 4000, 24, 4, 256, 3950, True), (96, 900, 4, 4, 256, 0, False),
])
def test_gqa_split_beforehand_matches_cpu_operator(backend, tq, tk, hq, hkv, d, start, causal):
    """With its workspace attached a prefill-shaped request splits keys and values beforehand, packs the query
    heads of a kv head into the rows of a tile and cuts walks that would leave units idle: the same bound as
    without, at the edges of tiles of 32 keys and 128 rows, from the shortest walk that takes this way."""
    rng = np.random.default_rng(tq * 17 + tk + d)
    q = rng.standard_normal((tq, hq, d)).astype(np.float32)
    k = rng.standard_normal((tk, hkv, d)).astype(np.float32)
    v = rng.standard_normal((tk, hkv, d)).astype(np.float32)
    out, lse, facts, need = run_attached(backend, q, k, v, query_start=start, causal=causal)
    assert need > 0 and facts.temporary_bytes == need
    assert facts.kernel_launches in (2, 3) and facts.accelerated_matrix_launches == 1
    rc, ref, ref_lse = ORACLE.gqa(q, k, v, query_start=start, causal=causal)
    assert rc == 0
    assert np.abs(out - ref).max() < 2e-5, np.abs(out - ref).max()
    assert np.abs(lse - ref_lse).max() < 2e-5
    again, lse_again, _, _ = run_attached(backend, q, k, v, query_start=start, causal=causal)
    assert np.array_equal(out, again) and np.array_equal(lse, lse_again)
    # one byte short of what it asked for: one launch, nothing allocated
    whole, lse_whole, facts, _ = run_attached(backend, q, k, v, short=1, query_start=start, causal=causal)
    assert facts.kernel_launches == 1 and facts.temporary_bytes == 0
    assert np.abs(whole - ref).max() < 2e-5 and np.abs(lse_whole - ref_lse).max() < 2e-5


@pytest.mark.parametrize("d", [64, 128, 256])
def test_gqa_split_beforehand_follows_magnitudes_and_views(backend, d):
    """Rows over many magnitudes, interleaved rows, keys and queries past the range of the parts in a cut walk (their
    rows are walked in fp32), infinities and NaN."""
    rng = np.random.default_rng(d + 5)
    tq, tk, hq, hkv = 45, 1500, 6, 2
    q, k, v = (rng.standard_normal(shape).astype(np.float32)
               for shape in ((tq, hq, d), (tk, hkv, d), (tk, hkv, d)))
    start = tk - tq
    grown = v * np.exp2(np.linspace(-20, 12, tk)).astype(np.float32)[:, None, None]
    grown[:8] = 0.0
    past = v.copy()
    past[777, 0, 3] = np.float32(2.0 ** 70)
    for label, case in (("powers", (q * np.float32(2.0 ** -40), k * np.float32(2.0 ** 40), v * np.float32(2.0 ** -90))),
                        ("grown", (q, k, grown)), ("past", (q, k, past))):
        out, lse, facts, _ = run_attached(backend, *case, query_start=start)
        assert facts.kernel_launches == 3
        rc, ref, ref_lse = ORACLE.gqa(*case, query_start=start)
        assert rc == 0
        assert relative_to_weighted_magnitudes(out, *case, start) < spread_bound(label, d), label
        assert np.abs(lse - ref_lse).max() < 2e-5 * max(1.0, np.abs(ref_lse).max())
    # interleaved [K | V] rows: the same bits
    packed, _, _, need = run_attached(backend, q, k, v, query_start=start)
    rows = f32(backend, "rows", np.concatenate([k.reshape(tk, -1), v.reshape(tk, -1)], axis=1))
    span, stride = (2 * tk - 1) * hkv * d, 2 * hkv * d
    req = backend.attention_requirement(tq, tk, hq, hkv, d, query_start=start, k_stride=stride, v_stride=stride)
    work, out_t = backend.tensor("work", B.DTYPE_I8, (need,)), f32(backend, "out", shape=q.shape)
    assert backend.attention_workspace_required(req) == need
    backend.workspace_attach(work)
    backend.attention_execute(req, f32(backend, "q", q), rows.view(0, B.DTYPE_F32, (span,)),
                              rows.view(hkv * d * 4, B.DTYPE_F32, (span,)), out_t)
    backend.workspace_detach()
    assert np.array_equal(out_t.read(), packed)
    # a key of -inf that every score excludes, infinities that no query sees, and values that are not finite
    positive = np.abs(q) + np.float32(0.1)
    excluded = k.copy()
    excluded[5, 0, 2] = -np.inf
    out, _, _, _ = run_attached(backend, positive, excluded, v, query_start=start)
    rc, ref, _ = ORACLE.gqa(positive, np.where(np.isinf(excluded), np.float32(-1e30), excluded), v, query_start=start)
    assert rc == 0 and np.abs(out - ref).max() < 2e-5
    unseen = k.copy()
    unseen[tk - 30:] = np.inf
    out, _, _, _ = run_attached(backend, q, unseen, v, query_start=start - 30)
    rc, ref, _ = ORACLE.gqa(q, k[:tk - 30], v[:tk - 30], query_start=start - 30)
    assert rc == 0 and np.abs(out - ref).max() < 2e-5
    for bad, at in ((np.inf, v), (np.nan, v), (np.nan, k)):
        tensor = at.copy()
        tensor[700, 1, 7] = bad
        with pytest.raises(YvexError) as e:
            run_attached(backend, q, k if at is v else tensor, tensor if at is v else v, query_start=start)
        assert e.value.code == B.YVEX_ERR_FORMAT


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("power", [8, 16, 24, 32, 40, 50])
@pytest.mark.parametrize("tk", [500, 1500])
def test_gqa_split_beforehand_holds_the_spread(backend, d, power, tk):
    """One row, channel or component of 2^8 to 2^50 among N(0,1) ones, seen, unseen or of weight zero, and sinks: as
    test_gqa_matrix_core_kernel_holds_the_spread, with the workspace, cut walks among them."""
    for label, q, k, v, start in spread_cases(d, power, tk=tk):
        out, lse, facts, need = run_attached(backend, q, k, v, query_start=start)
        assert facts.kernel_launches == 3 and facts.temporary_bytes == need
        worst = relative_to_weighted_magnitudes(out, q, k, v, start)
        # (scores of a key or query of 2^8, up to 1000, are rounded to 2^-25 of that; in one launch it is 9e-6 as well)
        large = power == 8 and label.startswith(("key-later", "query-one"))
        assert worst < (3e-5 if large else spread_bound(label, d)), (label, worst)


@pytest.mark.parametrize("d,hq,hkv", [(64, 16, 4), (128, 16, 4), (256, 40, 8)])
@pytest.mark.parametrize("power", [20, 40])
def test_gqa_split_beforehand_holds_the_spread_in_whole_walks(backend, d, hq, hkv, power):
    """The same where no walk is cut: rows left by the first walk and by the fp32 walk lie in one tile."""
    for label, q, k, v, start in spread_cases(d, power, tq=520, tk=600, hq=hq, hkv=hkv):
        out, lse, facts, _ = run_attached(backend, q, k, v, query_start=start)
        assert facts.kernel_launches == 2
        worst = relative_to_weighted_magnitudes(out, q, k, v, start)
        assert worst < spread_bound(label, d), (label, worst)


@pytest.mark.parametrize("tq,start,hq,hkv,d", [
    (100, 0, 24, 4, 256), (500, 0, 12, 2, 256), (70, 1500, 12, 2, 256), (100, 0, 10, 2, 128), (500, 0, 10, 2, 128),
    (70, 1500, 10, 2, 128), (100, 0, 8, 2, 64), (500, 0, 8, 2, 64), (70, 1500, 8, 2, 64)])
def test_gqa_split_beforehand_is_no_further_from_64_bits(backend, tq, start, hq, hkv, d):
    """The distance from 64 bits, in the 2-norm, of the walk over parts is smaller than that of the fp32 walk: its sums
    take fewer roundings (seen: 0.3 to 0.75 of it)."""
    rng = np.random.default_rng(tq + start + d)
    tk = start + tq
    q, k, v = (rng.standard_normal(s).astype(np.float32) for s in ((tq, hq, d), (tk, hkv, d), (tk, hkv, d)))
    q *= rng.uniform(0.5, 1.5, hq).astype(np.float32)[None, :, None]
    attached = run_attached(backend, q, k, v, query_start=start)[0]
    one = run_exact(backend, q, k, v, query_start=start)[0]
    apart = []
    for head in range(hq):
        scores = q[:, head].astype(np.float64) @ k[:, head // (hq // hkv)].astype(np.float64).T / math.sqrt(d)
        scores[np.arange(tk)[None, :] > (start + np.arange(tq))[:, None]] = -np.inf
        weights = np.exp(scores - scores.max(axis=1, keepdims=True))
        want = weights / weights.sum(axis=1, keepdims=True) @ v[:, head // (hq // hkv)].astype(np.float64)
        apart.append([((got[:, head] - want) ** 2).sum() for got in (attached, one)])
    of_parts, of_fp32 = np.sqrt(np.sum(apart, axis=0))
    assert of_parts <= 0.9 * of_fp32, (of_parts, of_fp32)


@pytest.mark.parametrize("d,hq,hkv", [(64, 5, 1), (128, 6, 2), (256, 4, 2)])
@pytest.mark.parametrize("tq,start", [(600, 0), (70, 2000)])
@pytest.mark.parametrize("form", ["attached", "one launch"])
def test_gqa_prefill_rows_do_not_depend_on_later_rows(backend, d, hq, hkv, tq, start, form):
    """Queries, keys and values of later tokens changed, to ordinary ones and to ones that end in the fp32 walk for the
    rows that see them: every bit of the earlier tokens' results stays, in the same wave, tile and run."""
    rng = np.random.default_rng(d + tq)
    tk = start + tq
    q, k, v = (rng.standard_normal(s).astype(np.float32) for s in ((tq, hq, d), (tk, hkv, d), (tk, hkv, d)))
    run = run_attached if form == "attached" else run_exact
    out, lse = run(backend, q, k, v, query_start=start)[:2]
    keep = tq * 2 // 3 - 7                             # tokens
    for label, q_by, k_by, v_by in (("ordinary", 1.0, 1.0, 1.0), ("grown", 4.0, 2.0 ** 6, 2.0 ** 20),
                                    ("keys past the range", 1.0, 2.0 ** 40, 1.0), ("queries", 2.0 ** 20, 1.0, 1.0),
                                    ("values", 1.0, 1.0, 2.0 ** 100)):
        q2, k2, v2 = q.copy(), k.copy(), v.copy()
        for new, from_, by in ((q2, keep, q_by), (k2, start + keep, k_by), (v2, start + keep, v_by)):
            new[from_:] = rng.standard_normal(new[from_:].shape).astype(np.float32) * np.float32(by)
        out2, lse2 = run(backend, q2, k2, v2, query_start=start)[:2]
        assert np.array_equal(out[:keep].view(np.uint32), out2[:keep].view(np.uint32)), label
        assert np.array_equal(lse[:keep].view(np.uint32), lse2[:keep].view(np.uint32)), label
        assert np.abs(out2[keep:] - out[keep:]).max() > 0.0


def test_gqa_split_beforehand_reaches_the_last_of_its_parts(backend):
    """The most keys whose parts a request may ask for (2 GiB less a tile or two, one kv head of 256): every head's one
    key of weight 1 lies elsewhere, the last in the last tile, and the head's rows are that key's values."""
    tq, tk, hq, d = 32, 838800, 4, 256
    places = [5, 400000, 700001, tk - tq - 3]
    q, k = np.zeros((tq, hq, d), np.float32), np.zeros((tk, 1, d), np.float32)
    v = (np.arange(tk, dtype=np.float32) % 1021.0 + 1.0)[:, None, None] * \
        np.linspace(0.5, 1.5, d, dtype=np.float32)[None, None, :]
    for head, key in enumerate(places):
        q[:, head, head] = 8.0
        k[key, 0, head] = 400.0                     # a score of 200, the others' is 0
    need = backend.attention_workspace_required(backend.attention_requirement(tq, tk, hq, 1, d, query_start=tk - tq))
    assert (1 << 31) - (4 << 20) < need < (1 << 31) + (96 << 20)
    out, lse, facts, _ = run_attached(backend, q, k, v, query_start=tk - tq)
    assert facts.kernel_launches == 3 and facts.temporary_bytes == need
    for head, key in enumerate(places):
        assert np.allclose(out[:, head], v[key, 0], rtol=1e-6, atol=0.0), head
    assert np.abs(lse - 200.0).max() < 1e-4
    assert backend.attention_workspace_required(
        backend.attention_requirement(tq, tk + 96, hq, 1, d, query_start=tk + 96 - tq)) == 0


# ------------------------------------------------ decode-shaped requests over long contexts ----

@pytest.mark.parametrize("tq,tk,hq,hkv,d,causal", [
    (1, 4096, 32, 8, 128, True), (1, 600, 4, 4, 64, True), (4, 5000, 6, 2, 96, True),
    (2, 1024, 3, 1, 256, True), (1, 513, 2, 2, 8, True), (3, 2000, 4, 2, 128, False),
    (31, 700, 2, 1, 40, True), (1, 16384, 8, 8, 128, True), (1, 70000, 1, 1, 64, True),
])
def test_gqa_split_runs_match_cpu_operator(backend, tq, tk, hq, hkv, d, causal):
    """The decode step of the session layer under the exact contract (one or a few query tokens
    over the whole cached history, src/runtime/stateful_attention.c:326-352): the keys are cut
    into runs, one wave per (token, head, run), double statistics, eight runs per workgroup,
    the workgroups of a (token, head) merged in the kernel by the one that arrives last.
    Same tight bound against the CPU operator as the row kernel."""
    rng = np.random.default_rng(tq * 7 + tk + d)
    q = rng.standard_normal((tq, hq, d)).astype(np.float32)
    k = rng.standard_normal((tk, hkv, d)).astype(np.float32)
    v = rng.standard_normal((tk, hkv, d)).astype(np.float32)
    start = tk - tq if causal else 0
    out, lse, facts = run_exact(backend, q, k, v, query_start=start, causal=causal)
    assert facts.kernel_launches == 1 and facts.accelerated_matrix_launches == 0
    assert facts.temporary_bytes > 0
    rc, ref, ref_lse = ORACLE.gqa(q, k, v, query_start=start, causal=causal)
    assert rc == 0
    assert np.abs(out - ref).max() < 2e-6, np.abs(out - ref).max()
    assert np.abs(lse - ref_lse).max() < 1e-5
    again, _, _ = run_exact(backend, q, k, v, query_start=start, causal=causal)
    assert np.array_equal(out, again)
    # with an attached workspace of the advertised size: no temporary, same bits
    req = backend.attention_requirement(tq, tk, hq, hkv, d, query_start=start, causal=causal)
    need = backend.attention_workspace_required(req)
    assert need == facts.temporary_bytes
    work = backend.tensor("work", B.DTYPE_I8, (need,))
    backend.workspace_attach(work)
    before = backend.memory_stats().allocation_events
    attached, _, facts2 = run_exact(backend, q, k, v, query_start=start, causal=causal)
    assert backend.memory_stats().allocation_events == before + 5      # the five tensors of run_exact
    backend.workspace_detach()
    work.release()
    assert np.array_equal(out, attached) and facts2.kernel_launches == 1


def test_gqa_split_threshold_and_failures(backend):
    rng = np.random.default_rng(80)
    q = rng.standard_normal((1, 4, 64)).astype(np.float32)
    k = rng.standard_normal((511, 2, 64)).astype(np.float32)
    v = rng.standard_normal((511, 2, 64)).astype(np.float32)
    out, _, facts = run_exact(backend, q, k, v, query_start=510)
    assert facts.kernel_launches == 1 and facts.temporary_bytes == 0     # short history: the row kernel
    rc, ref, _ = ORACLE.gqa(q, k, v, query_start=510)
    assert np.abs(out - ref).max() < 2e-6
    k = rng.standard_normal((2048, 2, 64)).astype(np.float32)
    v = rng.standard_normal((2048, 2, 64)).astype(np.float32)
    bad = k.copy()
    bad[1500, 1, 7] = np.inf
    with pytest.raises(YvexError) as e:
        run_exact(backend, q, bad, v, query_start=2047)
    assert e.value.code == B.YVEX_ERR_FORMAT
    bad = v.copy()
    bad[3, 0, 63] = np.nan
    with pytest.raises(YvexError) as e:
        run_exact(backend, q, k, bad, query_start=2047)
    assert e.value.code == B.YVEX_ERR_FORMAT
    good, _, facts = run_exact(backend, q, k, v, query_start=2047)
    assert facts.kernel_launches == 1 and facts.temporary_bytes > 0 and np.all(np.isfinite(good))
    # a query in the middle of the history: runs past its visible keys contribute nothing
    mid, _, _ = run_exact(backend, q, k, v, query_start=700)
    rc, ref, _ = ORACLE.gqa(q, k[:701], v[:701], query_start=700)
    assert np.abs(mid - ref).max() < 2e-6
