"""GPU parity of the int4 dequant kernel and the `linear` op (through the C ABI) against the
CPU oracle.  Tolerances are written where they are used and follow the reference's rule for
kernels whose reduction order differs from the oracle's: measure, then add margin
(docs/decisions/0022-gemm-register-blocking.md:22-24)."""
import numpy as np
import pytest

import helpers
import karume_amd as ka
from helpers import oracle

pytestmark = pytest.mark.gpu


def run_dequant(ctx, packed, scale, rows, width, group):
    scale = np.ascontiguousarray(scale)
    w = ctx.upload(packed)
    s = ctx.upload(scale)
    out = ctx.alloc(rows * width * 4)
    ctx.dequant_i4(w, s, out, rows, width, group, ka.dtype_code(scale.dtype))
    got = out.download(np.float32, (rows, width))
    for b in (w, s, out):
        b.free()
    return got


def run_linear(ctx, x, packed, scale, bias, n, k, group, compute=ka.COMPUTE_F32):
    """x: [m, k] float32 or float16 array (its dtype selects the io dtype)."""
    x = np.ascontiguousarray(x)
    scale = np.ascontiguousarray(scale)
    m = x.shape[0]
    dx, dw, ds = ctx.upload(x), ctx.upload(packed), ctx.upload(scale)
    db = ctx.upload(np.ascontiguousarray(bias, dtype=x.dtype)) if bias is not None else None
    out = ctx.alloc(max(m * n * x.itemsize, 16))
    ctx.linear_i4(dx, dw, ds, db, out, m, n, k, group, ka.dtype_code(x.dtype),
                  ka.dtype_code(scale.dtype), compute)
    got = out.download(x.dtype, (m, n))
    for b in (dx, dw, ds, out) + ((db,) if db is not None else ()):
        b.free()
    return got


def test_dequant_bit_exact_all_codes_all_positions(gpu_ctx):
    """All 16 codes x 8 in-word positions with row x group varying scales: GPU bits == decodeI4
    bits (packages/runtime/tests/gpu_i4_weights_test.ts:404-459, extended to u = 0)."""
    rows, width, g = 16, 32, 16
    q = np.array([(r + c) % 16 - 8 for r in range(rows) for c in range(width)], dtype=np.int8)
    scale = np.array([[0.1 + 0.017 * r + 0.31 * gi for gi in range(width // g)]
                      for r in range(rows)], dtype=np.float32)
    packed = oracle.pack_i4(q)
    want = oracle.decode_i4(packed, [rows, width], scale, [rows, width // g], g)
    got = run_dequant(gpu_ctx, packed, scale, rows, width, g)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("scale_dtype", [np.float32, np.float16])
def test_dequant_bit_exact_random(gpu_ctx, scale_dtype):
    rng = np.random.default_rng(21)
    rows, width, g = 67, 384, 128
    packed, _q, scale = helpers.synthetic_int4(rng, rows, width, g, scale_f16=True)
    scale = scale.astype(scale_dtype)
    if scale_dtype == np.float32:  # arbitrary f32 scales: the product rounds, once
        scale = (scale.astype(np.float32) * np.float32(1.2345678)).astype(np.float32)
    want = oracle.decode_i4(packed, [rows, width], scale.astype(np.float32),
                            [rows, width // g], g)
    got = run_dequant(gpu_ctx, packed, scale, rows, width, g)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("case", helpers.I4_LINEAR_CASES, ids=lambda c: c.name)
def test_linear_reference_cases_f32(gpu_ctx, case):
    """The reference's tile-edge shapes (gpu_i4_weights_test.ts:116-145), f32 in/out, f32
    scales.  |out| reaches ~1e3 here; gate: the reference's default allclose (atol 1e-5,
    rtol 1e-3) AND a tighter atol 2e-3 / rtol 2e-6 derived from f32 accumulation of ~1e3-sized
    partial sums (measured worst 2.4e-4)."""
    x, packed, _q, scale, bias = helpers.make_i4_linear(case)
    want = oracle.linear_i4(x, packed, scale, bias, case.n, case.k, case.group)
    got = run_linear(gpu_ctx, x, packed, scale, bias, case.n, case.k, case.group)
    ok, fails, max_abs, worst = oracle.allclose(got, want, atol=1e-5, rtol=1e-3)
    assert ok, (fails, max_abs, worst)
    ok, fails, max_abs, worst = oracle.allclose(got, want, atol=2e-3, rtol=2e-6)
    assert ok, (fails, max_abs, worst)


def test_linear_packed_equals_preexpanded_through_same_kernel(gpu_ctx):
    """Invariant of gpu_i4_weights_test.ts:262-298 restated for this backend: weights with
    scale 1 and the same codes must give exactly sum(q * x) — integer arithmetic, bit-exact —
    and scaling every group by a power of two must scale the output exactly."""
    rng = np.random.default_rng(2)
    n, k, g = 40, 256, 32
    q = rng.integers(-8, 8, size=(n, k), dtype=np.int8)
    x = rng.integers(-4, 5, size=(3, k)).astype(np.float32)
    packed = oracle.pack_i4(q)
    ones = np.ones((n, k // g), dtype=np.float32)
    got = run_linear(gpu_ctx, x, packed, ones, None, n, k, g)
    want = (x.astype(np.int64) @ q.astype(np.int64).T).astype(np.float32)
    assert np.array_equal(got, want)
    got4 = run_linear(gpu_ctx, x, packed, ones * 0.25, None, n, k, g)
    assert np.array_equal(got4, want * 0.25)


@pytest.mark.parametrize("io", [np.float16, np.float32])
def test_linear_config0_gemv(gpu_ctx, io):
    """benchmark config 0: M=1, K=N=4096, int4 g128, fp16 scales |N(0,0.02)|, x ~ N(0,1) in fp16.
    f32 output: atol 2e-5 (|out| ~ 5, f32 accumulation; measured worst 4e-6), rtol 0.
    fp16 output: the oracle's f32 result rounded to fp16, within 1 fp16 ulp."""
    rng = np.random.default_rng(40960)
    n = k = 4096
    g = 128
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(1, k)).astype(np.float16)
    want = oracle.linear_i4(x.astype(np.float32), packed, scale.astype(np.float32),
                            np.zeros(n, dtype=np.float32), n, k, g)
    got = run_linear(gpu_ctx, x.astype(io), packed, scale, None, n, k, g)
    if io == np.float32:
        ok, fails, max_abs, worst = oracle.allclose(got, want, atol=2e-5, rtol=0)
        assert ok, (fails, max_abs, worst)
    else:
        want16 = want.astype(np.float16)
        ulp = np.abs(np.nextafter(want16, np.float16(np.inf)).astype(np.float32)
                     - want16.astype(np.float32))
        assert np.all(np.abs(got.astype(np.float32) - want16.astype(np.float32)) <= ulp)


@pytest.mark.parametrize("io", [np.float16, np.float32])
def test_linear_batched_rows_equal_single_rows_bitwise(gpu_ctx, io):
    """benchmark config 3 (GEMV part): M = 16 in one launch vs the rows in smaller launches.
    f32 activations: the per-row reduction order does not depend on M, so the bits agree with
    single-row launches.  fp16 activations: batches of 2..16 rows run on the matrix cores,
    where a row's bits do not depend on the batch it sits in; a single row takes the
    dot-product kernel and agrees to the output's rounding."""
    rng = np.random.default_rng(16)
    n = k = 4096
    g = 128
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(16, k)).astype(np.float16).astype(io)
    batched = run_linear(gpu_ctx, x, packed, scale, None, n, k, g)
    for m_sub in (2, 5):
        part = run_linear(gpu_ctx, x[:m_sub], packed, scale, None, n, k, g)
        assert np.array_equal(part.view(np.uint8), batched[:m_sub].view(np.uint8)), m_sub
    pair = run_linear(gpu_ctx, x[10:12], packed, scale, None, n, k, g)
    assert np.array_equal(pair.view(np.uint8), batched[10:12].view(np.uint8))
    single = run_linear(gpu_ctx, x[11:12], packed, scale, None, n, k, g)
    if io == np.float32:
        assert np.array_equal(single.view(np.uint8), batched[11:12].view(np.uint8))
    else:
        a, b = single.astype(np.float32), batched[11:12].astype(np.float32)
        # both round an f32-accurate sum (each within 2e-5 of the exact one): at most one fp16
        # ulp apart, plus that noise where the output is tiny
        assert np.all(np.abs(a - b) <= 2.0 ** -10 * np.maximum(np.abs(a), np.abs(b)) + 4e-5)
    want = oracle.linear_i4(x.astype(np.float32), packed, scale.astype(np.float32),
                            np.zeros(n, dtype=np.float32), n, k, g)
    tol = 2e-5 if io == np.float32 else 8e-3  # fp16 output: half an ulp at |out| < 16
    assert np.max(np.abs(batched.astype(np.float32) - want)) <= tol


@pytest.mark.parametrize("m,n,k,g,scale_f16,with_bias", [
    (2, 16, 1024, 128, True, False), (16, 4096, 4096, 128, True, True),
    (7, 100, 2048, 128, False, True), (16, 33, 8192, 256, True, False),
    (3, 250, 3072, 128, True, True), (16, 64, 5120, 1024, False, False),
    # K a multiple of 256 only: the chunks are dealt unevenly to the waves (some get none)
    (16, 2048, 5632, 128, True, True), (5, 100, 11008, 128, True, False),
    (3, 40, 256, 128, False, True), (16, 64, 768, 256, True, False)])
def test_batched_fp16_rows_on_matrix_cores_match_oracle(gpu_ctx, m, n, k, g, scale_f16, with_bias):
    """2..16 fp16 rows take the MFMA kernel (K a multiple of 256, group >= 128): ragged N,
    every compile-time chunk count and the loop form (K = 3072, 5120), group sizes up to
    1024, f32 and fp16 scales, bias.  Gate: the oracle's f32 result rounded to fp16, one ulp."""
    rng = np.random.default_rng(m * 1000 + n)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g, scale_f16=scale_f16)
    x = rng.normal(size=(m, k)).astype(np.float16)
    bias = rng.normal(size=n).astype(np.float16) if with_bias else None
    got = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g)
    want = oracle.linear_i4(x.astype(np.float32), packed, scale.astype(np.float32),
                            (bias if with_bias else np.zeros(n)).astype(np.float32), n, k, g)
    err = np.abs(got.astype(np.float32) - want)
    assert np.all(err <= 2.0 ** -10 * np.abs(want) + 4e-5), float(err.max())


@pytest.mark.parametrize("m,n,k,g,scale_f16,with_bias", [
    (2, 4097, 2048, 128, True, True), (16, 4128, 2304, 128, False, False),
    (5, 8193, 4096, 256, False, True), (16, 8300, 5632, 128, True, False),
    (9, 12400, 6144, 128, True, True)])
def test_batched_fp16_rows_with_more_tiles_than_cus(gpu_ctx, m, n, k, g, scale_f16, with_bias):
    """A workgroup walks several tiles of 16 weight rows (two, three and four rounds, the last one
    ragged), even and uneven shares of K: the oracle's gate, and the bits of the narrow form."""
    rng = np.random.default_rng(m + n + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g, scale_f16=scale_f16)
    x = rng.normal(size=(m, k)).astype(np.float16)
    bias = rng.normal(size=n).astype(np.float16) if with_bias else None
    got = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g)
    few = 64
    first = n - few  # the last rows, the ragged tile among them
    codes = np.ascontiguousarray(packed.reshape(-1).view(np.uint8).reshape(n, k // 2)[first:])
    narrow = run_linear(gpu_ctx, x, codes, scale[first:], bias[first:] if with_bias else None, few, k, g)
    assert np.ascontiguousarray(got[:, first:]).tobytes() == narrow.tobytes()
    want = oracle.linear_i4(x.astype(np.float32), packed, scale.astype(np.float32),
                            (bias if with_bias else np.zeros(n)).astype(np.float32), n, k, g)
    err = np.abs(got.astype(np.float32) - want)
    assert np.all(err <= 2.0 ** -10 * np.abs(want) + 4e-5), float(err.max())


@pytest.mark.parametrize("shape", [(1, 256, 2048, 128), (3, 2048, 5632, 128), (1, 100, 11008, 128),
                                   (7, 33, 96, 32), (2, 5, 64, 16), (16, 32000, 2048, 128)])
def test_linear_shapes_of_the_decoder(gpu_ctx, shape):
    """The GEMV over the layer shapes of the 1.1B decoder (N x K) and ragged edges; f32 io,
    gate atol 3e-5 rtol 1e-5 against the f64 oracle (measured worst 6e-6)."""
    m, n, k, g = shape
    rng = np.random.default_rng(n * 7 + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(m, k)).astype(np.float16).astype(np.float32)
    bias = rng.normal(size=n).astype(np.float32)
    want = oracle.linear_i4(x, packed, scale.astype(np.float32), bias, n, k, g)
    got = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g)
    ok, fails, max_abs, worst = oracle.allclose(got, want, atol=3e-5, rtol=1e-5)
    assert ok, (fails, max_abs, worst)


@pytest.mark.parametrize("k,io,many", [(2048, np.float32, 8256), (5632, np.float32, 8256),
                                       (4096, np.float16, 8256), (4096, np.float16, 16512)])
def test_row_bits_do_not_depend_on_rows_per_wave(gpu_ctx, k, io, many):
    """A narrow output gives a wave one row, a wide one two (K = 5632, or fp16) or four
    (K = 2048 with f32 activations, fp16 activations from 16384 rows) that are reduced together:
    the same weight row and x give the same bits either way (one fixed order of additions for
    every form of the wave reduction)."""
    g, few = 128, 64
    rng = np.random.default_rng(k)
    packed, _q, scale = helpers.synthetic_int4(rng, many, k, g)
    x = rng.normal(size=(1, k)).astype(io)
    wide = run_linear(gpu_ctx, x, packed, scale, None, many, k, g)
    narrow = run_linear(gpu_ctx, x, packed.reshape(-1)[:few * k // 2], scale[:few], None, few, k, g)
    assert wide[:, :few].tobytes() == narrow.tobytes()


@pytest.mark.parametrize("n,k", [(3, 6272), (1031, 8192), (2100, 10272), (17, 12320), (2049, 14368),
                                 (5, 16384), (7, 16416)])
@pytest.mark.parametrize("io", [np.float32, np.float16])
def test_single_row_of_a_long_k_is_requested_whole(gpu_ctx, n, k, io):
    """4 to 8 steps of 2048 codes (the last one full, or a single group), one and two rows a wave,
    and the first K that is walked step by step again."""
    g = 32
    rng = np.random.default_rng(n + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(1, k)).astype(np.float16).astype(io)
    bias = rng.normal(size=n).astype(np.float16).astype(io)
    want = oracle.linear_i4(x.astype(np.float32), packed, scale.astype(np.float32),
                            bias.astype(np.float32), n, k, g)
    got = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g).astype(np.float32)
    rel = 1e-5 if io == np.float32 else 2.0 ** -10
    assert np.all(np.abs(got - want) <= rel * np.abs(want) + 5e-5), float(np.abs(got - want).max())


def test_linear_rejections(gpu_ctx):
    """Unsupported combinations fail before launch (never approximated)."""
    buf = gpu_ctx.zeros(4096)
    with pytest.raises(ka.GpuValidationError):  # group does not divide k
        gpu_ctx.linear_i4(buf, buf, buf, None, buf, 1, 4, 48, 32)
    with pytest.raises(ka.GpuValidationError):  # group not a power of two >= 16
        gpu_ctx.linear_i4(buf, buf, buf, None, buf, 1, 4, 48, 24)
    with pytest.raises(ka.GpuValidationError):
        gpu_ctx.linear_i4(buf, buf, buf, None, buf, 1, 4, 64, 8)
    with pytest.raises(ka.GpuValidationError):  # NULL weights
        gpu_ctx.linear_i4(buf, None, buf, None, buf, 1, 4, 64, 32)
    with pytest.raises(ka.GpuValidationError):
        gpu_ctx.dequant_i4(buf, buf, buf, 2, 8, 3)
    buf.free()


def test_linear_fused_decode_forms(gpu_ctx):
    """krm_linear_i4_fused: rms_norm folded in front, residual and silu(gate)*up folded behind,
    against the oracle's op chain rms_norm -> linear -> (+ residual | silu*mul).  f32 io: atol
    3e-5 rtol 2e-5 (the normalised row is not rounded between the ops here, so the result sits
    slightly closer to the f64 chain than the unfused launches do)."""
    rng = np.random.default_rng(8)
    # (1, 72, 8192, 128): K too long for registers, the prefetching loop with the norm in front
    for m, n, k, g in [(1, 2560, 2048, 128), (3, 512, 1024, 128), (1, 64, 256, 32), (2, 40, 96, 16),
                       (1, 72, 8192, 128)]:
        packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
        x = (rng.normal(size=(m, k)) * 5).astype(np.float32)
        gamma = rng.normal(size=k).astype(np.float32)
        res = rng.normal(size=(m, n)).astype(np.float32)
        sf = scale.astype(np.float32)
        zeros = np.zeros(n, dtype=np.float32)
        xn = oracle.rms_norm(x, gamma, 1e-5)
        lin = oracle.linear_i4(xn, packed, sf, zeros, n, k, g)
        bufs = [gpu_ctx.upload(a) for a in (x, packed, scale, gamma, res)]
        dx, dw, ds, dg, dr = bufs
        out = gpu_ctx.alloc(m * n * 4)
        # norm + linear + residual
        gpu_ctx.linear_i4_fused(dx, dw, ds, out, m, n, k, g, norm_weight=dg, norm_eps=1e-5,
                                residual=dr, scale_dtype=ka.F16)
        got = out.download(np.float32, (m, n))
        ok, fails, max_abs, worst = oracle.allclose(got, lin + res, atol=3e-5, rtol=2e-5)
        assert ok, (m, n, k, fails, max_abs, worst)
        # in place on the residual buffer
        gpu_ctx.linear_i4_fused(dx, dw, ds, dr, m, n, k, g, residual=dr, scale_dtype=ka.F16)
        plain = oracle.linear_i4(x, packed, sf, zeros, n, k, g)
        ok, fails, max_abs, worst = oracle.allclose(dr.download(np.float32, (m, n)), plain + res,
                                                    atol=2e-4, rtol=2e-5)
        assert ok, (fails, max_abs, worst)
        # norm + interleaved gate/up + silu*mul
        gpu_ctx.linear_i4_fused(dx, dw, ds, out, m, n, k, g, norm_weight=dg, norm_eps=1e-5,
                                scale_dtype=ka.F16, epilogue=ka.EPILOGUE_SILU_PAIRS)
        got = out.download(np.float32, (m, n // 2))
        want = oracle.silu_mul(lin[:, 0::2], lin[:, 1::2])
        ok, fails, max_abs, worst = oracle.allclose(got, want, atol=3e-5, rtol=5e-5)
        assert ok, (fails, max_abs, worst)
        for b in bufs + [out]:
            b.free()
    buf = gpu_ctx.zeros(1 << 16)
    with pytest.raises(ka.GpuValidationError):  # prefill chunks use the separate ops
        gpu_ctx.linear_i4_fused(buf, buf, buf, buf, 17, 64, 128, 128)
    with pytest.raises(ka.GpuValidationError):
        gpu_ctx.linear_i4_fused(buf, buf, buf, buf, 1, 63, 128, 128,
                                epilogue=ka.EPILOGUE_SILU_PAIRS)
    buf.free()


def test_linear_from_a_model_file(gpu_ctx):
    """File -> reader -> device: an int4 `linear` weight written as an I4 tensor with its F32
    group scale is handed to the kernel as the reader's views of the file (no re-packing) and
    must match the oracle run on the same bytes.  Gate as in the reference cases above."""
    import json
    from karume_amd.format_model import (build_safetensors, i4_resident_initializers, open_model,
                                         packed_int4)
    rng = np.random.default_rng(11)
    n, k, g, m = 96, 512, 64, 3
    q = rng.integers(-8, 8, size=(n, k), dtype=np.int8)
    scale = rng.uniform(0.005, 0.05, size=(n, k // g)).astype(np.float32)
    bias = rng.normal(size=n).astype(np.float32)
    graph = {
        "format": "karume-ir", "version": 1, "requires": {"ops": ["linear"]}, "symbols": [],
        "inputs": [{"name": "x", "dtype": "f32", "shape": [m, k]}], "outputs": ["y"],
        "initializers": {
            "w": {"tensor": "proj.weight",
                  "storage": {"dtype": "i4", "scale": "karume.scale.proj.weight", "group_size": g}},
            "b": {"tensor": "proj.bias", "storage": {"dtype": "f32"}}},
        "values": {"w": {"dtype": "f32", "shape": [n, k]}, "b": {"dtype": "f32", "shape": [n]},
                   "y": {"dtype": "f32", "shape": [m, n]}},
        "nodes": [{"op": "linear", "ins": ["x", "w", "b"], "outs": ["y"], "attrs": {}}]}
    blob = build_safetensors(
        [("karume.scale.proj.weight", "F32", [n, k // g], scale.tobytes()),
         ("proj.bias", "F32", [n], bias.tobytes()),
         ("proj.weight", "I4", [n, k], oracle.pack_i4(q).tobytes())],
        {"karume_ir": json.dumps(graph)})
    model = open_model(blob)
    assert i4_resident_initializers(model) == {"w"}
    weight = packed_int4(model, "w")
    x = rng.normal(size=(m, k)).astype(np.float32)
    want = oracle.linear_i4(x, weight.packed, weight.scales, bias, n, k, g)
    got = run_linear(gpu_ctx, x, weight.packed, weight.scales, bias, n, k, g)
    ok, fails, max_abs, worst = oracle.allclose(got, want, atol=1e-5, rtol=1e-3)
    assert ok, (fails, max_abs, worst)


def test_probe_linear_series_is_a_loop_of_linear_calls(gpu_ctx):
    """krm_probe_linear_series queues `count` plain linear_i4 launches over rotating weights:
    the output is that of the last launch's weights, bit for bit; it refuses to be recorded."""
    n, k, g = 256, 512, 128
    rng = np.random.default_rng(77)
    sets = [helpers.synthetic_int4(rng, n, k, g) for _ in range(3)]
    x = rng.normal(size=(1, k)).astype(np.float16)
    dx = gpu_ctx.upload(x)
    dws = [gpu_ctx.upload(p) for p, _q, _s in sets]
    dss = [gpu_ctx.upload(s) for _p, _q, s in sets]
    out, ref = gpu_ctx.alloc(n * 2), gpu_ctx.alloc(n * 2)
    gpu_ctx.probe_linear_series(dx, dws, dss, out, 5, 1, n, k, g, ka.F16, ka.F16)
    last = (5 - 1) % 3
    gpu_ctx.linear_i4(dx, dws[last], dss[last], None, ref, 1, n, k, g, ka.F16, ka.F16)
    assert out.download(np.uint16, (n,)).tobytes() == ref.download(np.uint16, (n,)).tobytes()
    with gpu_ctx.record() as rec:
        with pytest.raises(ka.GpuValidationError):
            gpu_ctx.probe_linear_series(dx, dws, dss, out, 2, 1, n, k, g, ka.F16, ka.F16)
        gpu_ctx.linear_i4(dx, dws[0], dss[0], None, ref, 1, n, k, g, ka.F16, ka.F16)
    rec.graph.destroy()
    for b in [dx, out, ref] + dws + dss:
        b.free()


def test_probe_exchange_is_bounded_and_clean(gpu_ctx):
    """The in-kernel hand-over probe: every wait in it is bounded, so the launch ends whatever
    the spin limit is and the fault word is 0 (every poll succeeded) or 1 (some poll gave up).
    A generous limit gives 0 only while all 256 workgroups are resident together, which the
    probe cannot guarantee on a GPU it shares with another process: the value is reported, the
    assertion is on termination and on the word being one of the two."""
    entries = 2048
    work = gpu_ctx.alloc(2 * entries * 4 + 1040)
    fault_at = 2 * entries * 4 + 1024
    for phases, limit in ((200, None), (200, 1), (50, None)):  # clean again after a faulted run
        if limit is None:
            gpu_ctx.probe_exchange(work, entries, phases)
        else:
            gpu_ctx.probe_exchange(work, entries, phases, spin_limit=limit)
        gpu_ctx.sync()
        fault = int(work.download(np.uint32, (1,), byte_offset=fault_at)[0])
        print(f"[probe exchange] phases {phases}, spin limit {limit}: fault word {fault}")
        assert fault in (0, 1)
    with pytest.raises(ka.GpuValidationError):
        gpu_ctx.probe_exchange(work, 1000, 10)
    work.free()


@pytest.mark.parametrize("n,k,g", [(8200, 2080, 32), (12000, 1152, 128), (9000, 576, 64), (16001, 832, 64),
                                   (1772, 4672, 32), (30000, 96, 32)])
@pytest.mark.parametrize("scale_type", [np.float16, np.float32])
def test_few_fp16_rows_have_the_same_bits_in_every_batch(gpu_ctx, n, k, g, scale_type):
    """2 to 16 fp16 rows where the GEMV has no matrix instructions: a row does not depend on its batch, and
    every result is the oracle's to one fp16 ulp."""
    rng = np.random.default_rng(n + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    scale = scale.astype(scale_type)
    x = rng.normal(size=(16, k)).astype(np.float16)
    bias = rng.normal(size=n).astype(np.float16)
    whole = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g)
    for rows in (slice(0, 2), slice(3, 8), slice(7, 16)):
        part = run_linear(gpu_ctx, x[rows], packed, scale, bias, n, k, g)
        assert np.array_equal(part.view(np.uint16), whole[rows].view(np.uint16)), rows
    cols = np.unique(np.concatenate([[0, 1, n - 2, n - 1], rng.choice(n, size=200)]))
    want = oracle.linear_i4(x.astype(np.float32), packed.reshape(n, k // 2)[cols].reshape(-1),
                            scale[cols].astype(np.float32), bias[cols].astype(np.float32), len(cols), k, g)
    got = whole[:, cols].astype(np.float32)
    # an fp16 ulp of the result beside the f32 sums (3e-5 of the row's typical product sum)
    assert np.all(np.abs(got - want) <= 2.0 ** -10 * np.abs(want) + 4e-5)


@pytest.mark.parametrize("n,k,g", [(7, 2048, 64), (130, 2080, 32), (1000, 4128, 32), (37, 6272, 128),
                                   (2100, 2176, 128)])
@pytest.mark.parametrize("scale_type", [np.float16, np.float32])
def test_several_f32_rows_brought_to_lds_have_the_bits_of_one_row(gpu_ctx, n, k, g, scale_type):
    """2 to 8 rows of f32 x over a K of a step and more, from 3 rows on dealt, 2 by shape: the bits of a row alone (K of
    one step, of a last step that is nearly empty; blocks of rows that are cut off; rows of N past the last).  (Rows
    brought to LDS: 2 of them here, and what follows a fusion below.)"""
    rng = np.random.default_rng(n * 3 + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    scale = scale.astype(scale_type)
    x = rng.normal(size=(8, k)).astype(np.float32)
    x[2, 5] = np.inf                     # stays in its row
    x[6, k - 1] = np.nan
    bias = rng.normal(size=n).astype(np.float32)
    alone = [run_linear(gpu_ctx, x[r:r + 1], packed, scale, bias, n, k, g)[0] for r in range(8)]
    for m in (2, 3, 4, 5, 7, 8):
        got = run_linear(gpu_ctx, x[:m], packed, scale, bias, n, k, g)
        for r in range(m):
            if r == 6:
                assert np.isnan(got[r]).all()
            else:
                assert np.array_equal(got[r].view(np.uint32), alone[r].view(np.uint32)), (m, r)


@pytest.mark.parametrize("scale_type", [np.float16, np.float32])
@pytest.mark.parametrize("n,k,g", [(66, 2048, 64), (130, 2080, 32), (2100, 2176, 128), (38, 6272, 128)])
@pytest.mark.parametrize("silu", [False, True])
def test_several_f32_rows_of_a_fusion_have_the_bits_of_one_row(gpu_ctx, silu, n, k, g, scale_type):
    """2 to 16 rows of f32 x over a K of a step and more with a residual or silu pairs behind them (blocks of 2, 4 and 8
    rows brought to LDS, 9 and more not): the bits of the same call on a row alone, an infinity in its row only."""
    rng = np.random.default_rng(n + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    scale = scale.astype(scale_type)
    n_out = n // 2 if silu else n
    x = rng.normal(size=(16, k)).astype(np.float32)
    x[2, 5] = np.inf
    residual, bias = rng.normal(size=(16, n_out)).astype(np.float32), rng.normal(size=n).astype(np.float32)
    bufs = [gpu_ctx.upload(a) for a in (x, packed, scale, residual, bias)]
    dx, dw, ds, dr, db = bufs
    out = gpu_ctx.alloc(16 * n_out * 4)

    def run(first, m):
        gpu_ctx.linear_i4_fused(dx.offset(first * k * 4), dw, ds, out, m, n, k, g, bias=db,
                                residual=None if silu else dr.offset(first * n_out * 4), scale_dtype=ka.dtype_code(scale.dtype),
                                epilogue=ka.EPILOGUE_SILU_PAIRS if silu else ka.EPILOGUE_NONE)
        return out.download(np.float32, (m, n_out))

    alone = np.concatenate([run(r, 1) for r in range(16)])
    assert np.isfinite(np.delete(alone, 2, axis=0)).all()
    for m in (2, 3, 4, 5, 8, 9, 16):
        got = run(0, m)
        same = (got.view(np.uint32) == alone[:m].view(np.uint32)) | (np.isnan(got) & np.isnan(alone[:m]))
        assert same.all(), (m, np.argwhere(~same)[:3])
    for b in bufs + [out]:
        b.free()


@pytest.mark.parametrize("n,k,g", [(70, 1152, 32), (300, 2048, 64), (1000, 4160, 64), (33, 8320, 128)])
@pytest.mark.parametrize("m", [9, 12, 13, 16])
def test_nine_to_sixteen_f32_rows_have_the_bits_of_one_row(gpu_ctx, n, k, g, m):
    """Nine rows and more, which are dealt: the bits of a row alone."""
    rng = np.random.default_rng(n + k + m)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    x = rng.normal(size=(m, k)).astype(np.float32)
    bias = rng.normal(size=n).astype(np.float32)
    got = run_linear(gpu_ctx, x, packed, scale, bias, n, k, g)
    for r in (0, 7, 8, m - 1):
        alone = run_linear(gpu_ctx, x[r:r + 1], packed, scale, bias, n, k, g)
        assert np.array_equal(got[r:r + 1].view(np.uint32), alone.view(np.uint32)), r


@pytest.mark.parametrize("n,k,g", [(8200, 2080, 32), (12000, 1152, 128), (9000, 576, 64), (16001, 832, 64),
                                   (1772, 4672, 32), (30000, 96, 32), (4096, 4096, 64)])
@pytest.mark.parametrize("scale_type", [np.float16, np.float32])
def test_few_fp16_rows_have_the_bits_of_one_row_alone(gpu_ctx, n, k, g, scale_type):
    """fp16 rows without matrix instructions in the GEMV (groups below 128, or a K that is no multiple of 256):
    one reduction order for one row and for 2 to 16, and for the fused entry point without a fusion."""
    rng = np.random.default_rng(n + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, g)
    scale = scale.astype(scale_type)
    x = rng.normal(size=(16, k)).astype(np.float16)
    bias = rng.normal(size=n).astype(np.float16)
    alone = [run_linear(gpu_ctx, x[r:r + 1], packed, scale, bias, n, k, g).view(np.uint16) for r in (0, 3, 15)]
    for m in (2, 5, 9, 16):
        got = run_linear(gpu_ctx, x[:m], packed, scale, bias, n, k, g).view(np.uint16)
        for r, want in zip((0, 3, 15), alone):
            assert r >= m or np.array_equal(got[r:r + 1], want), (m, r)
        buffers = [gpu_ctx.upload(a) for a in (x[:m], packed, scale, bias)]
        out = gpu_ctx.alloc(m * n * 2)
        gpu_ctx.linear_i4_fused(*buffers[:3], out, m, n, k, g, bias=buffers[3], io_dtype=ka.F16,
                                scale_dtype=ka.dtype_code(scale.dtype))
        assert np.array_equal(out.download(np.uint16, (m, n)), got), m
        for b in buffers + [out]:
            b.free()


@pytest.mark.parametrize("scale_type", [np.float16, np.float32])
@pytest.mark.parametrize("m, n, k", [(2, 40, 1024), (16, 33, 2048), (5, 17, 4096), (16, 16, 8192), (3, 50, 768),
                                     (16, 20, 2304), (7, 24, 5120), (16, 4112, 2048), (9, 4225, 4096),
                                     (16, 4500, 6144), (4, 4128, 2304), (16, 4100, 4352), (2, 4700, 5888)])
def test_scales_of_a_share_read_together(gpu_ctx, m, n, k, scale_type):
    """Batched fp16 rows in groups of 128, whose scales a wave reads at once (every form of the shares of K, a tile
    a workgroup and several), at a scale address of no more than four bytes' alignment: one fp16 ulp and
    the GEMV's gate against the oracle, and the bits of the same weights in groups of 256 (neighbouring groups of
    128 share a scale here)."""
    rng = np.random.default_rng(n + k)
    packed, _q, scale = helpers.synthetic_int4(rng, n, k, 128, scale_type is np.float16)
    scale[:, 1::2] = scale[:, 0::2]
    scale = scale.astype(scale_type)
    x = rng.normal(size=(m, k)).astype(np.float16)
    want = oracle.linear_i4(x.astype(np.float32), packed, scale.astype(np.float32), np.zeros(n, dtype=np.float32),
                            n, k, 128)
    dx, dw, out = gpu_ctx.upload(x), gpu_ctx.upload(packed), gpu_ctx.alloc(m * n * 2)
    skewed = np.concatenate([np.zeros(4 // scale.itemsize, dtype=scale_type), scale.reshape(-1)])
    ds, d256 = gpu_ctx.upload(skewed), gpu_ctx.upload(np.ascontiguousarray(scale[:, ::2]))
    got = []
    for at, group in ((ds.offset(4), 128), (d256, 256)):
        gpu_ctx.linear_i4(dx, dw, at, None, out, m, n, k, group, ka.F16, ka.dtype_code(scale.dtype))
        got.append(out.download(np.uint16, (m, n)))
    for b in (dx, dw, ds, d256, out):
        b.free()
    assert np.array_equal(got[0], got[1])
    ulp = np.spacing(np.abs(want).astype(np.float16)).astype(np.float32)
    assert np.all(np.abs(got[0].view(np.float16).astype(np.float32) - want) <= ulp + 4e-5)


@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("n,k,g,scale_type,offset", [
    (1030, 32, 32, np.float32, 0), (6200, 96, 32, np.float16, 0), (1025, 2048, 128, np.float16, 1),
    (1040, 4160, 32, np.float32, 3), (6145, 2144, 32, np.float16, 1), (20011, 160, 32, np.float16, 0),
    (9000, 1088, 64, np.float32, 0), (17, 8256, 64, np.float16, 0), (64, 6272, 128, np.float32, 1),
    (20, 65536, 32, np.float32, 0), (1, 1152, 32, np.float16, 0)])
def test_dealt_rows_have_the_bits_of_one_row_alone(gpu_ctx, dtype, n, k, g, scale_type, offset):
    """2 to 16 rows at the edges of what they are dealt by: K of one segment, of a part of a quad, of a step and past
    it; N off the tile; scales that are not aligned, or too many for LDS.  Bits of each row alone, also where x has
    infinities, zeros and subnormals.  (The forms: the test below.)"""
    rng = np.random.default_rng(n + k)
    packed = rng.integers(0, 2**32, size=n * k // 8, dtype=np.uint32)
    scale = (rng.random(size=n * (k // g) + offset) * .02 + .001).astype(scale_type)
    bias = rng.normal(size=n).astype(dtype)
    x = rng.normal(size=(16, k)).astype(dtype)
    x[1] *= dtype(1e-7 if dtype == np.float16 else 1e-42)
    x[2, ::3] = 0
    x[3, k // 2] = np.inf
    d_w, d_s, d_b = gpu_ctx.upload(packed), gpu_ctx.upload(scale), gpu_ctx.upload(bias)
    at = d_s.offset(offset * scale.itemsize)
    io, sd = ka.dtype_code(np.dtype(dtype)), ka.dtype_code(np.dtype(scale_type))

    def run(rows):
        d_x, out = gpu_ctx.upload(np.ascontiguousarray(rows)), gpu_ctx.alloc(len(rows) * n * rows.itemsize)
        gpu_ctx.linear_i4(d_x, d_w, at, d_b, out, len(rows), n, k, g, io, sd, ka.COMPUTE_F32)
        got = out.download(dtype, (len(rows), n))
        d_x.free()
        out.free()
        return got

    alone = np.concatenate([run(x[r:r + 1]) for r in range(16)])
    for m in (2, 3, 4, 5, 7, 9, 12, 16):
        got = run(x[:m])
        same = (got == alone[:m]) | (np.isnan(got) & np.isnan(alone[:m]))
        assert same.all() and (np.signbit(got) == np.signbit(alone[:m]))[~np.isnan(got)].all(), m
    for b in (d_w, d_s, d_b):
        b.free()


@pytest.mark.parametrize("x_size,scale_size,m,n,k,g", helpers.DEALT_ROWS)
def test_every_form_of_dealt_rows_has_the_bits_of_one_row_alone(gpu_ctx, x_size, scale_size, m, n, k, g):
    """64 or 16 rows of W a wave, 1 to 8 of x, one, two or four quads of segments in turn (test_rows_plan.py holds the
    list against the plan); infinities and subnormals stay in their rows."""
    dtype, scale_type = (np.float32 if b == 4 else np.float16 for b in (x_size, scale_size))
    rng = np.random.default_rng(m + n + k)
    packed = rng.integers(0, 256, size=(n, k // 2), dtype=np.uint8)
    scale = (rng.random(size=(n, k // g)) * .02 + .001).astype(scale_type)
    bias = rng.normal(size=n).astype(dtype)
    x = rng.normal(size=(m, k)).astype(dtype)
    x[0] *= dtype(1e-7 if x_size == 2 else 1e-42)
    x[m - 1, k // 2] = np.inf
    dw, ds, db, dx = (gpu_ctx.upload(a) for a in (packed, scale, bias, x))
    out = gpu_ctx.alloc(m * n * x_size)
    io, sd = ka.dtype_code(np.dtype(dtype)), ka.dtype_code(np.dtype(scale_type))
    gpu_ctx.linear_i4(dx, dw, ds, db, out, m, n, k, g, io, sd)
    got = out.download(dtype, (m, n))
    for r in range(m):
        gpu_ctx.linear_i4(dx.offset(r * k * x_size), dw, ds, db, out, 1, n, k, g, io, sd)
        alone = out.download(dtype, (n,))
        same = (got[r] == alone) & (np.signbit(got[r]) == np.signbit(alone))
        assert (same | (np.isnan(got[r]) & np.isnan(alone))).all(), r
    for b in (dw, ds, db, dx, out):
        b.free()
