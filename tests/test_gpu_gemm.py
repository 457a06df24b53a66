"""GPU parity of the MFMA GEMM paths of `linear` (M > 16) against the CPU oracle.

Two numerics classes (stated in the kernels):
* exact-operand kernels (K a multiple of 32; KRM_COMPUTE_F16, and KRM_COMPUTE_F32 with the f32
  activations split into fp16 hi + lo, in groups of 16 and 32 into three bf16): weights enter as
  exact integers, the group scale multiplies f32 group sums — gated at the GEMV's tolerance
  (`row_gate`: atol 3e-5 times the row's largest |x|, rtol 1e-5); the small groups, which keep every
  bit of x, also at a bound that grows with what is summed.
* fp16-weight kernels (other shapes under KRM_COMPUTE_F16): x rounded to fp16, each weight
  dequantised to fp16 as fp16((u-8) * scale) — one fp16 rounding, relative error <= 2^-11 — and
  products accumulated in f32.  With K terms of typical size t the error of an output behaves
  like sqrt(K) * t * 2^-11 / sqrt(3); those tests scale their tolerance with the RMS of the
  oracle's output:  |got - want| <= 2e-3 * rms(want) + 1e-3 * |want|  (measured worst case about
  a third of that).  When every scale is a power of two the dequantised weights are exact and
  the gate tightens to f32-accumulation level (atol 3e-5 * rms, measured ~5e-6).
"""
import numpy as np
import pytest

import helpers
import karume_amd as ka
from helpers import oracle
from test_gpu_linear import run_linear

pytestmark = pytest.mark.gpu


def sampled_oracle(x, packed, scale, bias, n, k, g, cols):
    """Oracle output restricted to a sample of output columns (weight rows)."""
    rows = packed.reshape(n, k // 2)[cols]
    return oracle.linear_i4(x, rows.reshape(-1), scale[cols], bias[cols], len(cols), k, g)


def check(got, want, exact_weights=False):
    rms = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    err = np.abs(got.astype(np.float64) - want)
    if exact_weights:
        bound = 3e-5 * rms + 1e-6 * np.abs(want)
    else:
        bound = 2e-3 * rms + 1e-3 * np.abs(want)
    worst = float(np.max(err / bound))
    assert worst <= 1.0, (worst, float(err.max()), rms)
    return worst


@pytest.mark.parametrize("m,n,k,g", [(512, 11008, 4096, 128), (512, 4096, 11008, 128)])
@pytest.mark.parametrize("io", [np.float16, np.float32])
def test_config1_prefill_gemm(gpu_ctx, m, n, k, g, io):
    """benchmark config 1 at full size (up- and down-projection); 192 sampled output columns
    are checked against the f64 oracle, all rows."""
    rng = np.random.default_rng(n + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(m, k)).astype(np.float16)
    bias = rng.normal(size=n).astype(np.float16)
    got = run_linear(gpu_ctx, x.astype(io), packed, scale, bias, n, k, g, compute=ka.COMPUTE_F16)
    cols = np.sort(rng.choice(n, size=192, replace=False))
    cols[:3] = [0, 1, 63]
    cols[-3:] = [n - 65, n - 2, n - 1]
    cols = np.unique(cols)
    want = sampled_oracle(x.astype(np.float32), packed, scale.astype(np.float32),
                          bias.astype(np.float32), n, k, g, cols)
    got_cols = got[:, cols].astype(np.float32)
    if io == np.float16:  # add the output rounding to the budget: half an fp16 ulp of |want|
        rms = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
        err = np.abs(got_cols - want)
        bound = 2e-3 * rms + 1.5e-3 * np.abs(want) + 1e-3
        assert np.all(err <= bound), float(np.max(err / bound))
    else:
        check(got_cols, want)


@pytest.mark.parametrize("shape", [(17, 64, 64, 16), (65, 68, 48, 16), (130, 200, 96, 32),
                                   (100, 129, 320, 64), (300, 1000, 2048, 128),
                                   (64, 256, 512, 128), (33, 8, 128, 128),
                                   # enough 128 x 256 tiles for the packed-weights form, with
                                   # ragged edges in M, N and K (K ends inside a 128-code stage)
                                   (300, 13349, 320, 64),
                                   # the same with a K long enough for the (tile, stage) units to
                                   # be dealt over the CUs: tiles shared by 2-3 workgroups
                                   (300, 13349, 2624, 64)])
def test_gemm_edges_exact_weights(gpu_ctx, shape):
    """Tile edges in M, N and K (K not a multiple of the 64-code stage, N not a multiple of
    the tile) with power-of-two scales: dequantised weights are exact in fp16, x is fp16, so
    only the f32 accumulation order differs from the oracle."""
    m, n, k, g = shape
    rng = np.random.default_rng(m * 1000 + n)
    q = rng.integers(-8, 8, size=(n, k), dtype=np.int8)
    scale = (2.0 ** rng.integers(-8, -3, size=(n, k // g))).astype(np.float32)
    packed = oracle.pack_i4(q)
    x = rng.normal(size=(m, k)).astype(np.float16).astype(np.float32)
    bias = rng.normal(size=n).astype(np.float32)
    want = oracle.linear_i4(x, packed, scale, bias, n, k, g)
    got = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g, compute=ka.COMPUTE_F16)
    check(got, want, exact_weights=True)
    got_h = run_linear(gpu_ctx, x.astype(np.float16), packed, scale.astype(np.float16),
                       bias.astype(np.float16), n, k, g, compute=ka.COMPUTE_F16)
    want_h = oracle.linear_i4(x, packed, scale, bias.astype(np.float16).astype(np.float32), n, k,
                              g)
    assert np.max(np.abs(got_h.astype(np.float32) - want_h)
                  - 1e-3 * np.abs(want_h)) <= 2e-3  # fp16 output rounding


def test_gemm_with_tiles_shared_between_workgroups_is_reproducible(gpu_ctx):
    """86 tiles of 32 stages on 256 CUs: the (tile, stage) units are dealt 10 or 11 to a
    workgroup, so every tile is the sum of 3-4 partials added by whichever workgroup arrives
    last.  The sum is taken in K order whoever that is: repeated runs give the same bits, and
    the result meets the exact-weights gate."""
    m, n, k, g = 256, 11008, 4096, 128
    rng = np.random.default_rng(77)
    q = rng.integers(-8, 8, size=(n, k), dtype=np.int8)
    scale = (2.0 ** rng.integers(-8, -3, size=(n, k // g))).astype(np.float32)
    packed = oracle.pack_i4(q)
    x = rng.normal(size=(m, k)).astype(np.float16).astype(np.float32)
    bias = rng.normal(size=n).astype(np.float32)
    first = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g, compute=ka.COMPUTE_F16)
    for _ in range(4):
        again = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g, compute=ka.COMPUTE_F16)
        assert np.array_equal(first.view(np.uint32), again.view(np.uint32))
    check(first, oracle.linear_i4(x, packed, scale, bias, n, k, g), exact_weights=True)


def test_gemm_reference_cases(gpu_ctx):
    """The reference's tile-edge shapes with its own generators (M = 65 and 17 take the MFMA
    path with KRM_COMPUTE_F16); arbitrary f32 scales, f32 x that is not fp16-representable."""
    for case in helpers.I4_LINEAR_CASES[:2]:
        x, packed, _q, scale, bias = helpers.make_i4_linear(case)
        want = oracle.linear_i4(x, packed, scale, bias, case.n, case.k, case.group)
        got = run_linear(gpu_ctx, x, packed, scale, bias, case.n, case.k, case.group,
                         compute=ka.COMPUTE_F16)
        check(got, want)


def test_gemm_f32_mode_stays_on_f32_arithmetic(gpu_ctx):
    """KRM_COMPUTE_F32 with M > 16 keeps f32 products and accumulation (the GEMV over row
    blocks): same gate as the GEMV tests (atol 3e-5, rtol 1e-5), far tighter than fp16."""
    rng = np.random.default_rng(5)
    m, n, k, g = 40, 512, 1024, 128
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(m, k)).astype(np.float32)  # not fp16-representable
    bias = rng.normal(size=n).astype(np.float32)
    want = oracle.linear_i4(x, packed, scale.astype(np.float32), bias, n, k, g)
    got = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g, compute=ka.COMPUTE_F32)
    ok, fails, max_abs, worst = oracle.allclose(got, want, atol=3e-5, rtol=1e-5)
    assert ok, (fails, max_abs, worst)


def row_gate(x):
    """Absolute tolerance per output row of the exact-operand forms: the GEMV's gate
    (atol 3e-5 for activations of unit size, rtol 1e-5) scaled with the row's largest |x|."""
    top = np.max(np.abs(np.where(np.isfinite(x), x, 0.0)), axis=1, keepdims=True)
    return 3e-5 * np.maximum(top, 1e-30)


@pytest.mark.parametrize("m,n,k,g", [(512, 11008, 4096, 128), (512, 4096, 11008, 128)])
def test_config1_f32_class_runs_on_the_matrix_cores_within_the_gemv_gate(gpu_ctx, m, n, k, g):
    """KRM_COMPUTE_F32 with f32 activations at benchmark config 1's shapes: the activations are
    split into fp16 hi + lo (22 bits, scaled per row), the weights enter as exact integers, the
    group scale multiplies f32 group sums.  Rows of very different magnitude (1e5, 1e-6, beyond
    the fp16 range in both directions), a row of zeros and values that are not
    fp16-representable; 160 sampled columns against the f64 oracle at the GEMV's gate."""
    rng = np.random.default_rng(n * 3 + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(m, k)).astype(np.float32)
    x[3] *= 1e5
    x[4] *= 3e7
    x[5] *= 1e-6
    x[6] *= 1e-30
    x[7] = 0.0
    x[8, ::2] *= 1e-4          # wide dynamic range inside one row
    bias = rng.normal(size=n).astype(np.float32)
    got = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g, compute=ka.COMPUTE_F32)
    cols = np.unique(np.concatenate([[0, 1, 63, 64, 511, 512, n - 513, n - 65, n - 2, n - 1],
                                     rng.choice(n, size=150, replace=False)]))
    want = sampled_oracle(x, packed, scale.astype(np.float32), bias, n, k, g, cols)
    err = np.abs(got[:, cols].astype(np.float64) - want)
    bound = row_gate(x) + 1e-5 * np.abs(want)
    assert np.all(err <= bound), float(np.max(err / bound))
    assert np.all(got[7] == bias)      # the row of zeros: exactly the bias


@pytest.mark.parametrize("io", [np.float16, np.float32])
def test_config1_f16_operands_are_exact_integers_times_fp16_x(gpu_ctx, io):
    """KRM_COMPUTE_F16 at config 1's up-projection: with fp16-representable activations every
    product is exact and the group scale multiplies f32 sums, so the result meets the GEMV's
    gate (the per-weight fp16 rounding of the small-shape kernels is gone here)."""
    m, n, k, g = 512, 11008, 4096, 128
    rng = np.random.default_rng(91)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(m, k)).astype(np.float16)
    bias = rng.normal(size=n).astype(np.float16)
    got = run_linear(gpu_ctx, x.astype(io), packed, scale, bias.astype(io), n, k, g,
                     compute=ka.COMPUTE_F16)
    cols = np.unique(rng.choice(n, size=128, replace=False))
    want = sampled_oracle(x.astype(np.float32), packed, scale.astype(np.float32),
                          bias.astype(np.float32), n, k, g, cols)
    err = np.abs(got[:, cols].astype(np.float64) - want)
    bound = row_gate(x.astype(np.float32)) + 1e-5 * np.abs(want)
    if io == np.float16:                # the output rounding: half an fp16 ulp of |want|
        bound = bound + 2.0 ** -11 * np.abs(want) + 1e-7
    assert np.all(err <= bound), float(np.max(err / bound))


def test_f32_class_gemm_edges_and_non_finite_rows(gpu_ctx):
    """Ragged M, N and K (K ends inside a 128-code stage, two scale groups a stage), f32 scales,
    and rows holding Inf / NaN: those rows come out non-finite where the oracle's do, every
    other row meets the gate."""
    m, n, k, g = 300, 13349, 2624, 64
    rng = np.random.default_rng(12)
    q = rng.integers(-8, 8, size=(n, k), dtype=np.int8)
    scale = np.abs(rng.normal(0, 0.02, size=(n, k // g))).astype(np.float32) + 1e-4
    packed = oracle.pack_i4(q)
    x = rng.normal(size=(m, k)).astype(np.float32)
    x[11, 5] = np.inf
    x[12, 2000] = np.nan
    bias = rng.normal(size=n).astype(np.float32)
    got = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g, compute=ka.COMPUTE_F32)
    cols = np.unique(np.concatenate([[0, 511, 512, n - 1], rng.choice(n, size=60, replace=False)]))
    want = sampled_oracle(x, packed, scale, bias, n, k, g, cols)
    finite = np.ones(m, dtype=bool)
    finite[[11, 12]] = False
    err = np.abs(got[finite][:, cols].astype(np.float64) - want[finite])
    bound = row_gate(x[finite]) + 1e-5 * np.abs(want[finite])
    assert np.all(err <= bound), float(np.max(err / bound))
    assert not np.any(np.isfinite(got[[11, 12]][:, cols]))
    assert not np.any(np.isfinite(want[[11, 12]]))


# ---------------------------------------------------------------- few rows (a prefill chunk)

def run_rows(ctx, x, packed, scale, bias, n, k, group, compute, residual=None,
             epilogue=ka.EPILOGUE_NONE):
    x = np.ascontiguousarray(x)
    m = x.shape[0]
    n_out = n // 2 if epilogue == ka.EPILOGUE_SILU_PAIRS else n
    dx, dw, ds = ctx.upload(x), ctx.upload(packed), ctx.upload(np.ascontiguousarray(scale))
    db = ctx.upload(np.ascontiguousarray(bias, dtype=x.dtype)) if bias is not None else None
    dr = ctx.upload(np.ascontiguousarray(residual, dtype=x.dtype)) if residual is not None else None
    out = ctx.alloc(max(m * n_out * x.itemsize, 16))
    ctx.linear_i4_rows(dx, dw, ds, out, m, n, k, group, bias=db, residual=dr,
                       io_dtype=ka.dtype_code(x.dtype), scale_dtype=ka.dtype_code(scale.dtype),
                       compute=compute, epilogue=epilogue)
    got = out.download(x.dtype, (m, n_out))
    for b in (dx, dw, ds, out, db, dr):
        if b is not None:
            b.free()
    return got


ROWS_SHAPES = [(128, 2560, 2048, 128),   # a 128-row chunk of the benchmark decoder: [q; k; v]
               (128, 2048, 5632, 128),   # its down-projection: 44 groups over 8 waves
               (40, 512, 1024, 128), (100, 129, 320, 64), (257, 96, 4096, 256),
               (100, 2700, 1088, 64),    # 64-column tiles; K ends inside a chunk's second half
               (17, 33, 192, 64),        # fewer 64-code chunks than waves
               (1, 64, 2048, 128)]


@pytest.mark.parametrize("m,n,k,g", ROWS_SHAPES)
@pytest.mark.parametrize("mode", ["f32", "f16 on f32", "f16"])
def test_few_row_products_meet_the_gemv_gate(gpu_ctx, m, n, k, g, mode):
    """Shapes too small for the 64 x 512 deal run on the few-row kernel (eight waves split K):
    exact integer weights and f32 group sums, so the f32 class (x split hi + lo) and the fp16
    class (x rounded to fp16 once: the oracle is given the rounded x) both meet the GEMV's
    gate.  Ragged M, N, K, a single row and a K shorter than eight chunks included."""
    rng = np.random.default_rng(m * 7 + n + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(m, k)).astype(np.float32)
    x[0] *= 300.0
    if m > 2:
        x[2] *= 1e-3
    bias = rng.normal(size=n).astype(np.float32)
    if mode == "f32":
        got = run_rows(gpu_ctx, x, packed, scale, bias, n, k, g, ka.COMPUTE_F32)
        seen = x
    elif mode == "f16 on f32":
        got = run_rows(gpu_ctx, x, packed, scale, bias, n, k, g, ka.COMPUTE_F16)
        seen = x.astype(np.float16).astype(np.float32)
    else:
        got = run_rows(gpu_ctx, x.astype(np.float16), packed, scale, bias, n, k, g,
                       ka.COMPUTE_F16)
        seen = x.astype(np.float16).astype(np.float32)
        bias = bias.astype(np.float16).astype(np.float32)
    if m > 16 and mode != "f16":   # krm_linear_i4 takes the same kernel for these shapes
        compute = ka.COMPUTE_F32 if mode == "f32" else ka.COMPUTE_F16
        same = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g, compute=compute)
        assert np.array_equal(got.view(np.uint32), same.view(np.uint32))
    want = oracle.linear_i4(seen, packed, scale.astype(np.float32), bias, n, k, g)
    err = np.abs(got.astype(np.float64) - want)
    bound = row_gate(seen) + 1e-5 * np.abs(want)
    if mode == "f16":
        bound = bound + 2.0 ** -11 * np.abs(want) + 1e-7
    assert np.all(err <= bound), float(np.max(err / bound))


def test_few_row_epilogues_against_the_oracle_and_the_separate_ops(gpu_ctx):
    """residual add and the gate/up pairs folded into the few-row kernel: equal to the plain
    call followed by the oracle's add / silu-mul within one rounding of the stored type, and
    the oracle's own chain within the gate."""
    rng = np.random.default_rng(404)
    m, n, k, g = 96, 1408, 2048, 128
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(m, k)).astype(np.float32)
    bias = rng.normal(size=n).astype(np.float32)
    residual = rng.normal(size=(m, n)).astype(np.float32)
    plain = run_rows(gpu_ctx, x, packed, scale, bias, n, k, g, ka.COMPUTE_F32)
    via_linear = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g, compute=ka.COMPUTE_F32)
    assert np.array_equal(plain.view(np.uint32), via_linear.view(np.uint32))
    with_res = run_rows(gpu_ctx, x, packed, scale, bias, n, k, g, ka.COMPUTE_F32, residual=residual)
    assert np.array_equal(with_res.view(np.uint32), (plain + residual).view(np.uint32))
    # pairs: rows (2i, 2i+1) of w are (gate_i, up_i)
    paired = run_rows(gpu_ctx, x, packed, scale, bias, n, k, g, ka.COMPUTE_F32,
                      epilogue=ka.EPILOGUE_SILU_PAIRS)
    want = oracle.linear_i4(x, packed, scale.astype(np.float32), bias, n, k, g)
    chain = oracle.silu_mul(want[:, 0::2].astype(np.float32), want[:, 1::2].astype(np.float32))
    scale_of = np.abs(want[:, 0::2]) * np.abs(want[:, 1::2]) + np.abs(want[:, 1::2]) + 1.0
    assert np.all(np.abs(paired.astype(np.float64) - chain) <= 1e-4 * scale_of)
    separate = oracle.silu_mul(plain[:, 0::2].copy(), plain[:, 1::2].copy())
    assert np.all(np.abs(paired - separate) <= 4e-6 * scale_of)
    # fp16 storage, the wide (64-column) tiles: n / 32 x m / 64 workgroups beyond two a CU
    m, n, k, g = 128, 11264, 2048, 128
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(m, k)).astype(np.float16)
    paired = run_rows(gpu_ctx, x, packed, scale, None, n, k, g, ka.COMPUTE_F16,
                      epilogue=ka.EPILOGUE_SILU_PAIRS)
    cols = np.unique(rng.choice(n // 2, size=96, replace=False))
    rows = np.stack([2 * cols, 2 * cols + 1], axis=1).reshape(-1)
    want = sampled_oracle(x.astype(np.float32), packed, scale.astype(np.float32),
                          np.zeros(n, dtype=np.float32), n, k, g, rows)
    chain = oracle.silu_mul(want[:, 0::2].astype(np.float32), want[:, 1::2].astype(np.float32))
    err = np.abs(paired[:, cols].astype(np.float64) - chain)
    assert np.all(err <= 1e-3 * np.abs(chain) + 1e-3), float(err.max())


def test_few_row_kernel_rejects_what_it_does_not_cover(gpu_ctx):
    rng = np.random.default_rng(1)
    packed, _q, scale = helpers.synthetic_int4(rng, 64, 64, 16)
    x = rng.normal(size=(20, 64)).astype(np.float32)
    with pytest.raises(ka.GpuValidationError, match="group_size >= 64"):
        run_rows(gpu_ctx, x, packed, scale, None, 64, 64, 16, ka.COMPUTE_F32)
    with pytest.raises(ka.GpuValidationError, match="even n"):
        packed, _q, scale = helpers.synthetic_int4(rng, 33, 128, 64)
        run_rows(gpu_ctx, rng.normal(size=(20, 128)).astype(np.float32), packed, scale, None, 33,
                 128, 64, ka.COMPUTE_F32, epilogue=ka.EPILOGUE_SILU_PAIRS)


@pytest.mark.parametrize("compute", [ka.COMPUTE_F32, ka.COMPUTE_F16])
def test_few_row_results_do_not_depend_on_the_batch(gpu_ctx, compute):
    """In the reference an output row has the same bits whatever M is
    (packages/runtime/tests/gpu_gemm_skinny_test.ts:11-15,156-198).  The few-row kernel keeps
    that: a row's products, its split over the eight waves (a function of K) and the order of the
    final sum do not depend on the other rows, on the row's place in the chunk, or on the tile
    width chosen for the chunk (32 or 64 columns)."""
    rng = np.random.default_rng(808)
    n, k, g = 4224, 1024, 128      # 128 rows: 4 x 132 tiles > 256 CUs -> 64-column tiles
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(128, k)).astype(np.float32)
    x[5] *= 1e4
    bias = rng.normal(size=n).astype(np.float32)
    whole = run_rows(gpu_ctx, x, packed, scale, bias, n, k, g, compute)
    for rows in ([5], [0, 5, 77], list(range(40, 73))):   # 1, 3 and 33 rows: 32-column tiles
        part = run_rows(gpu_ctx, x[rows], packed, scale, bias, n, k, g, compute)
        assert np.array_equal(part.view(np.uint32), whole[rows].view(np.uint32)), rows


# (m, n, k, group): one tile of 32 x 32 / its neighbours, K of one unit, of an odd half unit (ends
# on 32 of 64 codes), fewer blocks than waves, slices of unequal length, every tile size of the
# dispatch on 256 CUs (32 x 32, 32 x 64, 32 x 96, 64 x 32, 64 x 64, 64 x 96), the smallest groups
SLICES_SHAPES = [(17, 31, 64, 16), (32, 33, 96, 16), (33, 64, 96, 32), (77, 300, 2080, 32),
                 (65, 2049, 160, 32), (64, 129, 1056, 16), (129, 1600, 192, 64), (40, 97, 2624, 64),
                 (100, 2500, 640, 128), (200, 2500, 1024, 128), (64, 8100, 384, 128),
                 (512, 2044, 512, 128), (200, 5003, 1024, 256)]


@pytest.mark.parametrize("m,n,k,g", SLICES_SHAPES)
@pytest.mark.parametrize("mode", ["f32", "f16 on f32", "f16"])
def test_k_slices_kernel_at_the_edges_of_its_tiles(gpu_ctx, m, n, k, g, mode):
    """krm_linear_i4 for M > 16 at every group size, ragged tiles and K tails, f32 and fp16
    scales, against the oracle at the gate of the exact-operand kernels."""
    rng = np.random.default_rng(m + n * 3 + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    scale = scale.astype(np.float32 if (m + k) % 3 else np.float16)
    x = rng.normal(size=(m, k)).astype(np.float32)
    x[m // 2] *= 1e3
    bias = rng.normal(size=n).astype(np.float32)
    seen = x if mode == "f32" else x.astype(np.float16).astype(np.float32)
    if mode == "f16":
        x, bias = x.astype(np.float16), bias.astype(np.float16)
    compute = ka.COMPUTE_F32 if mode == "f32" else ka.COMPUTE_F16
    got = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g, compute=compute)
    want = oracle.linear_i4(seen, packed, scale.astype(np.float32), bias.astype(np.float32), n, k, g)
    err = np.abs(got.astype(np.float64) - want)
    bound = row_gate(seen) + 1e-5 * np.abs(want)
    if mode == "f16":
        bound = bound + 2.0 ** -11 * np.abs(want) + 1e-7
    assert np.all(err <= bound), float(np.max(err / bound))


# (one to four column tiles of 32 a workgroup in groups of 32, one to three in groups of 16, two row
# tiles, on 256 CUs)
SMALL_GROUP_SHAPES = [(17, 33, 96, 32), (77, 300, 2080, 32), (100, 200, 2048, 16), (300, 2500, 512, 32),
                      (77, 3001, 96, 16), (100, 9001, 96, 16), (100, 9001, 96, 32),
                      (512, 11003, 160, 32), (512, 2050, 96, 32)]


@pytest.mark.parametrize("m,n,k,g", SMALL_GROUP_SHAPES)
def test_small_groups_keep_entries_beside_an_outlier(gpu_ctx, m, n, k, g):
    """The f32 class in groups of 16 and 32 takes every bit of x: entries of 1e-3 count in full
    beside entries of 1e6 that meet a zero code.  The bound grows with what is summed, not with the
    row's maximum: at most 64 roundings of 2^-24 act on a part of sum |x w| each (a wave's flushes,
    the steps of a group, the waves' sums)."""
    rng = np.random.default_rng(m + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    packed = packed.reshape(n, k // 2).copy()
    at = np.arange(5, k, 3 * g)
    packed[:, at // 2] = (packed[:, at // 2] & 0x0F) | 0x80     # odd columns: the high nibble, code 0
    x = (rng.normal(size=(m, k)) * 1e-3).astype(np.float32)
    x[:, at] = 1e6
    got = run_linear(gpu_ctx, x, packed, scale, None, n, k, g)
    codes = np.stack([packed & 15, packed >> 4], axis=-1).reshape(n, k).astype(np.float64) - 8.0
    w = codes * np.repeat(scale.astype(np.float64).reshape(n, k // g), g, axis=1)
    want, size = x.astype(np.float64) @ w.T, np.abs(x).astype(np.float64) @ np.abs(w).T
    assert np.all(np.abs(got - want) <= 64 * 2.0 ** -24 * size), \
        float(np.max(np.abs(got - want) / size))


@pytest.mark.parametrize("m,n,k,g", SMALL_GROUP_SHAPES)
def test_small_groups_give_what_the_gemv_gives_for_values_that_are_not_finite(gpu_ctx, m, n, k, g):
    """Infinities (against codes of either sign and zero codes), two that cancel, a NaN whose payload
    lies in its low bits, 1e37 (the largest f32 overflows the GEMV's sums), subnormals (whose parts
    may count as zeros): the same rows, 16 at a time, run the GEMV."""
    rng = np.random.default_rng(n + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(m, k)).astype(np.float32)
    x[0, 3] = np.inf
    x[1, k - 1] = -np.inf
    x[2, [1, k // 2]] = np.inf, -np.inf
    x[3, 7] = np.array([0x7F800001], dtype=np.uint32).view(np.float32)[0]
    x[4, 9] = 1e37
    x[5] = 1e-42
    got = run_linear(gpu_ctx, x, packed, scale, None, n, k, g)
    want = run_linear(gpu_ctx, x[:16], packed, scale, None, n, k, g)
    for kind in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(kind(got[:16]), kind(want)), kind.__name__
    assert np.isfinite(got[16:]).all() and np.isfinite(got[4]).all()
    finite = np.isfinite(want)
    err = np.abs(got[:16][finite].astype(np.float64) - want[finite])
    size = np.broadcast_to(np.abs(np.where(np.isfinite(x[:16]), x[:16], 0)).sum(1, keepdims=True)
                           * 8.0 * float(np.abs(scale).max()), want.shape)[finite]
    assert np.all(err <= 64 * 2.0 ** -24 * size + 1e-37)
    if m > 22:     # a row's bits do not depend on the others
        assert np.array_equal(got[6:], run_linear(gpu_ctx, x[6:], packed, scale, None, n, k, g))


def test_small_groups_need_no_scratch(gpu_ctx):
    """A side branch of a graph takes the f32 class in groups of 32, as it took the GEMV."""
    ctx, (m, n, k, g) = gpu_ctx, SMALL_GROUP_SHAPES[1]
    rng = np.random.default_rng(3)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(m, k)).astype(np.float32)
    want = run_linear(ctx, x, packed, scale, None, n, k, g)
    dx, dw, ds = ctx.upload(x), ctx.upload(packed), ctx.upload(np.ascontiguousarray(scale))
    out = ctx.alloc(m * n * 4)
    with ctx.record() as rec:
        rec.branch(1)
        ctx.linear_i4(dx, dw, ds, None, out, m, n, k, g, ka.F32, ka.dtype_code(scale.dtype),
                      ka.COMPUTE_F32)
    for _ in range(3):
        out.zero()
        rec.graph.launch()
        assert np.array_equal(out.download(np.float32, (m, n)), want)
    rec.graph.destroy()
    for b in (dx, dw, ds, out):
        b.free()


@pytest.mark.parametrize("m,n,k,g", [(330, 11300, 448, 64), (400, 20011, 512, 128), (65, 31000, 704, 64)])
@pytest.mark.parametrize("mode", ["f32", "f16 on f32", "f16"])
def test_wide_short_products_on_either_form(gpu_ctx, m, n, k, g, mode):
    """Two to twelve stages a workgroup of the unit-dealt form: whichever form the estimates pick, and
    the one without scratch that a side branch takes, meet the gate of the exact-operand kernels."""
    ctx = gpu_ctx
    rng = np.random.default_rng(m + n + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(m, k)).astype(np.float32)
    if mode == "f16":
        x = x.astype(np.float16)
    compute = ka.COMPUTE_F32 if mode == "f32" else ka.COMPUTE_F16
    seen = x if mode == "f32" else x.astype(np.float16).astype(np.float32)
    dx, dw, ds = ctx.upload(x), ctx.upload(packed), ctx.upload(np.ascontiguousarray(scale))
    out = ctx.alloc(m * n * x.itemsize)
    call = lambda: ctx.linear_i4(dx, dw, ds, None, out, m, n, k, g, ka.dtype_code(x.dtype),  # noqa: E731
                                 ka.dtype_code(scale.dtype), compute)
    call()
    results = [out.download(x.dtype, (m, n))]
    if mode != "f32":      # (hi and lo planes need scratch)
        with ctx.record() as rec:
            rec.branch(1)
            call()
        for _ in range(2):
            out.zero()
            rec.graph.launch()
            results.append(out.download(x.dtype, (m, n)))
        rec.graph.destroy()
        assert np.array_equal(results[1], results[2])
    cols = np.unique(np.concatenate([rng.choice(n, size=96), [0, 1, 511, 512, n - 2, n - 1]]))
    want = sampled_oracle(seen, packed, scale.astype(np.float32), np.zeros(n, np.float32), n, k, g, cols)
    bound = row_gate(seen) + 1e-5 * np.abs(want)
    if mode == "f16":
        bound = bound + 2.0 ** -11 * np.abs(want) + 1e-7
    for got in results:
        err = np.abs(got[:, cols].astype(np.float64) - want)
        assert np.all(err <= bound), float(np.max(err / bound))
    for b in (dx, dw, ds, out):
        b.free()


# (fp16: 128 x 256 tiles with a K that ends half-way through a stage; 64 x 512 tiles of M = 64; the f32
# class: 64 x 512 tiles at ranges of a few stages and, with K of 16384, rows in two blocks because the hi
# and lo planes of all do not fit their scratch, the second block overlapping the first)
@pytest.mark.parametrize("m,n,k,g,mode", [(330, 20011, 1344, 64, "f16"), (257, 24577, 1408, 128, "f16"),
                                          (64, 25001, 8128, 64, "f16"), (330, 11300, 448, 64, "f32"),
                                          (257, 7001, 2048, 128, "f32"), (129, 16300, 1344, 64, "f32"),
                                          (1100, 1601, 16384, 256, "f32")])
def test_unit_dealt_products_at_the_edges_of_their_tiles(gpu_ctx, m, n, k, g, mode):
    """Ragged tiles, shared tiles and K tails of the unit-dealt forms, f32 and fp16 scales, with bias, at
    the gate of the exact-operand kernels; the same bits from every run."""
    rng = np.random.default_rng(m + n + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    scale = scale.astype(np.float32 if m % 2 else np.float16)
    x = rng.normal(size=(m, k)).astype(np.float32)
    x[m // 2] *= 1e3 if mode == "f32" else 10
    bias = rng.normal(size=n).astype(np.float32)
    if mode == "f16":
        x, bias = x.astype(np.float16), bias.astype(np.float16)
    seen = x.astype(np.float32)
    compute = ka.COMPUTE_F32 if mode == "f32" else ka.COMPUTE_F16
    got = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g, compute=compute)
    again = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g, compute=compute)
    assert np.array_equal(got.view(np.uint8), again.view(np.uint8))
    cols = np.unique(np.concatenate([rng.choice(n, size=64), [0, 255, 256, 511, 512, n - 2, n - 1]]))
    want = sampled_oracle(seen, packed, scale.astype(np.float32), bias.astype(np.float32), n, k, g, cols)
    bound = row_gate(seen) + 1e-5 * np.abs(want)
    if mode == "f16":
        bound = bound + 2.0 ** -11 * np.abs(want) + 1e-7
    err = np.abs(got[:, cols].astype(np.float64) - want)
    assert np.all(err <= bound), float(np.max(err / bound))


@pytest.mark.parametrize("m,n,k,g,mode", [(228, 25350, 3072, 128, "f16"), (200, 26999, 2048, 128, "f32"),  # one a tile
                                          (280, 10758, 6592, 64, "f16"), (333, 6001, 4992, 64, "f16"),   # two, three
                                          (250, 8190, 6272, 128, "f32"), (300, 5000, 8192, 128, "f32")])  # four, five
def test_tiles_with_workgroups_of_their_own(gpu_ctx, m, n, k, g, mode):
    """One to five workgroups share a tile and no other, in equal and in unequal parts of its K."""
    test_unit_dealt_products_at_the_edges_of_their_tiles(gpu_ctx, m, n, k, g, mode)


@pytest.mark.parametrize("io", [ka.F16, ka.F32])
@pytest.mark.parametrize("compute", [ka.COMPUTE_F16, ka.COMPUTE_F32])
@pytest.mark.parametrize("m,n,k,silu", [(17, 4, 64, False), (33, 64, 128, True), (50, 96, 576, False),
                                        (128, 2048, 2048, False), (128, 11264, 256, True),
                                        (300, 260, 1152, True)])
def test_quads_and_pairs_of_columns_are_finished_alike(gpu_ctx, io, compute, m, n, k, silu):
    """A finished sum is stored four columns at a time where rows and buffers are aligned to that, two
    at a time elsewhere: the same bits, with a bias and (in place) a residual, for one tile of a few
    columns, tiles that are cut off and waves that own no codes (k of 64 and 128)."""
    rng = np.random.default_rng(m + n + k)
    group = 64
    io_np = np.float32 if io == ka.F32 else np.float16
    eb, n_out = np.dtype(io_np).itemsize, n // 2 if silu else n
    packed, _codes, scales = helpers.synthetic_int4(rng, n, k, group)
    x = rng.normal(size=(m, k)).astype(io_np)
    bias, residual = rng.normal(size=n).astype(io_np), rng.normal(size=m * n_out).astype(io_np)
    dx, dw, ds = map(gpu_ctx.upload, (x, packed, scales))
    got = []
    for shift in (0, 1):     # in elements
        pad = np.zeros(shift, dtype=io_np)
        db = gpu_ctx.upload(np.concatenate([pad, bias]))
        out = gpu_ctx.upload(np.concatenate([pad, residual]))
        at = out.offset(shift * eb)
        gpu_ctx.linear_i4_rows(dx, dw, ds, at, m, n, k, group, bias=db.offset(shift * eb), residual=at,
                               io_dtype=io, scale_dtype=ka.F16, compute=compute,
                               epilogue=ka.EPILOGUE_SILU_PAIRS if silu else ka.EPILOGUE_NONE)
        got.append(out.download(io_np, (shift + m * n_out,))[shift:].reshape(m, n_out))
    bits = np.uint32 if io == ka.F32 else np.uint16
    assert np.isfinite(got[0]).all()
    assert np.array_equal(got[0].view(bits), got[1].view(bits))
    if not silu:
        want = oracle.linear_i4(x.astype(np.float32), packed, scales.astype(np.float32),
                                bias.astype(np.float32), n, k, group) + residual.reshape(m, n)
        # (f32 sums of exact products; x rounded to fp16 in that class, and the fp16 result)
        half = io == ka.F16 or compute == ka.COMPUTE_F16
        err, rms = np.abs(got[0] - want), float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
        assert float(np.max(err - (2e-3 if half else 3e-5) * (np.abs(want) + rms))) <= 0.0


@pytest.mark.parametrize("io", [ka.F16, ka.F32])
@pytest.mark.parametrize("m,heads,kv_heads,d", [(17, 1, 1, 4), (40, 3, 1, 12), (128, 32, 4, 64),
                                                (130, 4, 2, 6)])
def test_rope_of_a_fused_projection_by_quads_and_by_pairs(gpu_ctx, io, m, heads, kv_heads, d):
    """The rotation reads its table rows two dims at a time where the tables are aligned to that:
    the bits of one dim at a time (tables a float off; a head dim of 6 has no quads at all)."""
    rng = np.random.default_rng(m + d)
    n, k, group, table = (heads + 2 * kv_heads) * d, 256, 64, 50
    io_np = np.float32 if io == ka.F32 else np.float16
    eb = np.dtype(io_np).itemsize
    packed, _codes, scales = helpers.synthetic_int4(rng, n, k, group)
    x = rng.normal(size=(m, k)).astype(io_np)
    bias = rng.normal(size=n).astype(io_np)
    ang = rng.normal(size=table * d)
    pos = rng.integers(0, table, size=m).astype(np.int32)
    pos[m // 2] = table                           # outside the table: NaN in q and k
    dx, dw, ds, db, dp = map(gpu_ctx.upload, (x, packed, scales, bias, pos))
    got = []
    for shift in (0, 1):
        pad = np.zeros(shift, dtype=np.float32)
        cos, sin = (gpu_ctx.upload(np.concatenate([pad, f(ang).astype(np.float32)]))
                    for f in (np.cos, np.sin))
        q, kk, v = (gpu_ctx.zeros(m * planes * d * eb) for planes in (heads, kv_heads, kv_heads))
        gpu_ctx.prefill_qkv(dx, dw, ds, dp, cos.offset(4 * shift), sin.offset(4 * shift), q, kk, v,
                            bias=db, m=m, heads=heads, kv_heads=kv_heads, depth=d, k=k, group=group,
                            table_rows=table, io_dtype=io, scale_dtype=ka.F16, compute=ka.COMPUTE_F32)
        got.append([b.download(io_np, (planes, m, d)) for b, planes in
                    ((q, heads), (kk, kv_heads), (v, kv_heads))])
    bits = np.uint32 if io == ka.F32 else np.uint16
    for a, b in zip(*got):
        assert np.array_equal(a.view(bits), b.view(bits))
    assert np.isnan(got[0][0][:, m // 2]).all() and np.isfinite(got[0][2]).all()
    assert np.isfinite(np.delete(got[0][0], m // 2, 1)).all()


@pytest.mark.parametrize("k", [64, 2048, 2112, 4096, 4160, 8192, 8256, 16384, 16448])
def test_hi_and_lo_of_rows_of_any_length(gpu_ctx, k):
    """The lengths at which the pass that splits f32 rows has other threads: every row at the gate of its class, the
    largest magnitude in its last piece."""
    rng = np.random.default_rng(k)
    m, n, g = 18, 70, 64
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(m, k)).astype(np.float32)
    x[::2, k - 1] = 300
    got = run_linear(gpu_ctx, x, packed, scale, None, n, k, g, compute=ka.COMPUTE_F32)
    want = sampled_oracle(x, packed, scale.astype(np.float32), np.zeros(n, np.float32), n, k, g, np.arange(n))
    bound = row_gate(x) + 1e-5 * np.abs(want)
    err = np.abs(got.astype(np.float64) - want)
    assert np.all(err <= bound), float(np.max(err / bound))


# (unit-dealt tiles of 128 x 256 and of 64 x 512; tiles staged through registers; tiles that split K)
@pytest.mark.parametrize("m,n,k,g", [(348, 8164, 4608, 128), (199, 19207, 4160, 64), (64, 25001, 8128, 64),
                                     (463, 5555, 3200, 128), (104, 8583, 1152, 128), (148, 4751, 6656, 64),
                                     (113, 6077, 2112, 32)])
def test_f32_rows_rounded_to_fp16_once(gpu_ctx, m, n, k, g):
    """f32 x in fp16 arithmetic with its rows rounded by a pass of their own: the gate of the exact-operand kernels
    on the rounded x, f32 bias and result; a magnitude past fp16 is infinite, and so is its row's result."""
    rng = np.random.default_rng(m + n + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    scale = scale.astype(np.float32 if m % 2 else np.float16)
    x = rng.normal(size=(m, k)).astype(np.float32)
    x[m - 1, k - 1] = 7e4
    bias = rng.normal(size=n).astype(np.float32)
    with np.errstate(over="ignore"):
        seen = x.astype(np.float16).astype(np.float32)
    got = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g, compute=ka.COMPUTE_F16)
    assert not np.isfinite(got[m - 1]).any()
    cols = np.unique(np.concatenate([rng.choice(n, size=64), [0, 255, 256, 511, 512, n - 2, n - 1]]))
    want = sampled_oracle(seen[:-1], packed, scale.astype(np.float32), bias, n, k, g, cols)
    bound = row_gate(seen[:-1]) + 1e-5 * np.abs(want)
    err = np.abs(got[:-1, cols].astype(np.float64) - want)
    assert np.all(err <= bound), float(np.max(err / bound))


@pytest.mark.parametrize("io", [ka.F16, ka.F32])
@pytest.mark.parametrize("m,n,k", [(17, 8, 64), (40, 96, 576), (128, 2048, 256)])
def test_the_residual_of_a_silu_is_read_at_any_element(gpu_ctx, io, m, n, k):
    """Two residuals are read at once, wherever they lie: the same bits from a buffer that is a whole number of
    pairs and from one that is an element off, with `out` aligned in both."""
    rng = np.random.default_rng(m + n)
    io_np = np.float32 if io == ka.F32 else np.float16
    packed, _codes, scales = helpers.synthetic_int4(rng, n, k, 64)
    x, residual = rng.normal(size=(m, k)).astype(io_np), rng.normal(size=m * n // 2).astype(io_np)
    dx, dw, ds = map(gpu_ctx.upload, (x, packed, scales))
    zero = gpu_ctx.zeros(m * n // 2 * np.dtype(io_np).itemsize)
    gpu_ctx.linear_i4_rows(dx, dw, ds, zero, m, n, k, 64, io_dtype=io, scale_dtype=ka.F16,
                           compute=ka.COMPUTE_F32, epilogue=ka.EPILOGUE_SILU_PAIRS)
    product = zero.download(io_np, (m, n // 2)).astype(np.float64)
    got = []
    for shift in (0, 1):
        res = gpu_ctx.upload(np.concatenate([np.zeros(shift, dtype=io_np), residual]))
        out = gpu_ctx.zeros(m * n // 2 * np.dtype(io_np).itemsize)
        gpu_ctx.linear_i4_rows(dx, dw, ds, out, m, n, k, 64, residual=res.offset(shift * np.dtype(io_np).itemsize),
                               io_dtype=io, scale_dtype=ka.F16, compute=ka.COMPUTE_F32,
                               epilogue=ka.EPILOGUE_SILU_PAIRS)
        got.append(out.download(io_np, (m, n // 2)))
    bits = np.uint32 if io == ka.F32 else np.uint16
    assert np.array_equal(got[0].view(bits), got[1].view(bits))
    # (the product rounded to `io` here, not in the kernel; then one rounding of the sum)
    eps = 2.0 ** -22 if io == ka.F32 else 2.0 ** -10
    want = product + residual.reshape(m, n // 2)
    assert np.all(np.abs(got[0] - want) <= eps * (np.abs(product) + np.abs(want)) + 1e-7)


# (exact tiles of hi + lo and of rounded rows, in both group forms; tiles staged through registers; hi + lo of the
# tiles that split K)
@pytest.mark.parametrize("m,n,k,g,compute", [
    (330, 11300, 448, 64, "f32"), (257, 7001, 2048, 128, "f32"), (333, 6001, 4992, 64, "f16"),
    (348, 8164, 4608, 128, "f16"), (338, 18849, 1280, 128, "f16"), (330, 20011, 448, 64, "f16"),
    (50, 96, 576, 64, "f32"), (33, 64, 512, 128, "f32"), (128, 2048, 1024, 64, "f32")])
def test_f32_scales_keep_their_range(gpu_ctx, m, n, k, g, compute):
    """Whole numbers in x and one f32 scale of 2^-145 for all codes: every sum is a whole number of them below 2^24
    on the way, and so is the result, a subnormal or small normal f32, exactly.  (Totals kept 1024 times smaller
    until their end would lose their last bits.)"""
    rng = np.random.default_rng(m + n + k)
    packed = rng.integers(0, 256, size=(n, k // 2), dtype=np.uint8)
    scale = np.full((n, k // g), 2.0 ** -145, dtype=np.float32)
    top = 1800 if compute == "f16" else 7000     # exact in fp16, in hi + lo
    x = rng.integers(-top, top + 1, size=(m, k)).astype(np.float32)
    got = run_linear(gpu_ctx, x, packed, scale, None, n, k, g,
                     compute=ka.COMPUTE_F16 if compute == "f16" else ka.COMPUTE_F32)
    cols = np.unique(np.concatenate([rng.choice(n, size=64), [0, n // 2, n - 1]]))
    q = np.stack([packed[cols] & 15, packed[cols] >> 4], axis=2).reshape(len(cols), k).astype(np.float64) - 8
    want = x.astype(np.float64) @ q.T
    assert np.abs(want).max() < 2 ** 23
    assert np.array_equal(got[:, cols].astype(np.float64) * 2.0 ** 145, want)


@pytest.mark.parametrize("m,n,k,g", [(333, 6001, 4992, 64), (348, 8164, 4608, 128), (338, 18849, 1280, 128),
                                     (330, 20011, 448, 64)])
def test_f32_scales_of_both_ends_of_their_range(gpu_ctx, m, n, k, g):
    """f32 rows rounded to fp16, columns with a scale of 2^118 beside columns with one of 2^-130, codes of zero in some
    groups: whole numbers of a thousandth of the scale, exactly."""
    rng = np.random.default_rng(m + n + k)
    packed = rng.integers(0, 256, size=(n, k // 2), dtype=np.uint8)
    packed[:, g // 2:g] = 0x88
    scale = np.full((n, k // g), 2.0 ** 118, dtype=np.float32)
    scale[1::2] = 2.0 ** -130
    x = rng.integers(-60, 61, size=(m, k)).astype(np.float32) * np.float32(2.0 ** -10)
    got = run_linear(gpu_ctx, x, packed, scale, None, n, k, g, compute=ka.COMPUTE_F16)
    cols = np.unique(np.concatenate([rng.choice(n, size=64), [0, 1, n // 2, n - 2, n - 1]]))
    q = np.stack([packed[cols] & 15, packed[cols] >> 4], axis=2).reshape(len(cols), k).astype(np.float64) - 8
    want = (x.astype(np.float64) @ q.T) * scale[cols, 0].astype(np.float64)
    assert np.abs(want).max() < 2.0 ** 127 and np.array_equal(got[:, cols].astype(np.float64), want)
