"""GPU parity of states-form attention, state_append and the ragged decode batch (through the
C ABI) against the CPU oracle."""
import numpy as np
import pytest

import helpers
import karume_amd as ka
from helpers import PARITY_CASES, StateCase, make_state_inputs, oracle, oracle_state_attention

pytestmark = pytest.mark.gpu

# The reference's own gate for this op: atol 5e-6, rtol 0, outputs O(1)
# (packages/runtime/tests/gpu_state_attention_test.ts:41-54; its measured worst is 6.6e-7).
STATE_ATOL = 5e-6


def run_attention(ctx, case: StateCase, x: dict, io=np.float32, kv=np.float32, scale=None,
                  workspace_bytes=None):
    bufs = {k: ctx.upload(np.ascontiguousarray(v, dtype=io if k in ("q", "ins_k", "ins_v") else kv))
            for k, v in x.items()}
    out_elems = case.batch * case.heads * case.chunk_rows * case.depth
    out = ctx.upload(np.full(out_elems, 123.0, dtype=io))  # every element must be overwritten
    ws_bytes = ctx.attention_state_workspace(case.batch, case.heads, case.kv_heads,
                                             case.chunk_rows, case.depth, case.window,
                                             min(case.past, 1 << 20), case.query)
    if workspace_bytes is not None:
        ws_bytes = workspace_bytes
    ws = ctx.alloc(max(ws_bytes, 16))
    ctx.attention_state(
        bufs["q"], bufs["ins_k"], bufs["ins_v"], bufs["slot_k"], bufs["slot_v"], out,
        half_scale=oracle.half_scale(case.depth) if scale is None else scale,
        io_dtype=ka.dtype_code(io), kv_dtype=ka.dtype_code(kv), workspace=ws,
        workspace_bytes=ws_bytes, **case.kwargs())
    got = out.download(io, (case.batch, case.heads, case.chunk_rows, case.depth))
    for b in list(bufs.values()) + [out, ws]:
        b.free()
    return got


@pytest.mark.parametrize("case", PARITY_CASES, ids=lambda c: c.name)
def test_parity_grid(gpu_ctx, case):
    """The reference's 17-case grid with poison in every place that must not be read
    (gpu_state_attention_test.ts:119-347): atol 5e-6 rtol 0, pad rows exact +0."""
    x = make_state_inputs(case)
    want = oracle_state_attention(case, x)
    got = run_attention(gpu_ctx, case, x)
    ok, fails, max_abs, worst = oracle.allclose(got, want, atol=STATE_ATOL, rtol=0)
    assert ok, (fails, max_abs, worst)
    pad = got[:, :, case.query:, :]
    assert np.all(pad == 0.0) and not np.any(np.signbit(pad))


DECODE_CASES = [
    StateCase("decode r4 D128 P300", 1, 8, 2, 1, 128, 512, 0, 300, 1),
    StateCase("decode r4 D128 P127 one split", 2, 8, 2, 1, 128, 128, 0, 127, 1),
    StateCase("decode r4 D128 P128 boundary", 1, 8, 2, 1, 128, 256, 0, 128, 1),
    StateCase("decode r8 D64 P383", 1, 32, 4, 1, 64, 512, 0, 383, 1),
    StateCase("decode r1 D64 P0", 1, 4, 4, 1, 64, 16, 0, 0, 1),
    StateCase("decode r1 D128 P700 six splits", 1, 4, 4, 1, 128, 1024, 0, 700, 1),
    StateCase("decode r1 D64 P300 chunks together", 1, 4, 4, 1, 64, 512, 0, 300, 1),
    StateCase("decode r2 D32 B3 P77", 3, 4, 2, 1, 32, 96, 0, 77, 1),
    StateCase("decode sliding W100 P1000 C128", 1, 8, 2, 1, 128, 128, 100, 1000, 1),
    StateCase("decode sliding W300 P299", 1, 8, 2, 1, 64, 300, 300, 299, 1),
    StateCase("decode sliding W256 P5000", 2, 8, 8, 1, 64, 256, 256, 5000, 1),
]


def random_state_inputs(case: StateCase, seed: int, f16_values: bool):
    rng = np.random.default_rng(seed)
    b, h, hkv, m, d, c = (case.batch, case.heads, case.kv_heads, case.chunk_rows, case.depth,
                          case.capacity)
    x = dict(q=rng.normal(size=(b, h, m, d)), ins_k=rng.normal(size=(b, hkv, m, d)),
             ins_v=rng.normal(size=(b, hkv, m, d)), slot_k=rng.normal(size=(b, hkv, c, d)),
             slot_v=rng.normal(size=(b, hkv, c, d)))
    cast = (lambda a: a.astype(np.float16).astype(np.float32)) if f16_values else \
        (lambda a: a.astype(np.float32))
    x = {k: cast(v) for k, v in x.items()}
    # poison what must not be read: non-resident slot rows
    base = oracle.state_column_base(case.window, case.past)
    resident = {col % case.window if case.window else col for col in range(base, case.past)}
    for row in range(c):
        if row not in resident:
            x["slot_k"][:, :, row] = 9.0
            x["slot_v"][:, :, row] = 400.0
    return x


@pytest.mark.parametrize("case", DECODE_CASES, ids=lambda c: c.name)
@pytest.mark.parametrize("io,kv", [(np.float32, np.float32), (np.float16, np.float16),
                                   (np.float32, np.float16)])
def test_decode_split_k(gpu_ctx, case, io, kv):
    """The split-K decode path (Q = 1, M = 1) over one or several splits, full and sliding.
    f32 output: atol 5e-6 rtol 0 (the reference's gate).  fp16 output: the oracle's value
    rounded to fp16, +-1 fp16 ulp."""
    x = random_state_inputs(case, seed=case.past + case.depth, f16_values=True)
    want = oracle_state_attention(case, x)
    got = run_attention(gpu_ctx, case, x, io=io, kv=kv)
    if io == np.float32:
        ok, fails, max_abs, worst = oracle.allclose(got, want, atol=STATE_ATOL, rtol=0)
        assert ok, (fails, max_abs, worst)
    else:
        want16 = want.astype(np.float16)
        ulp = np.abs(np.nextafter(want16, np.float16(np.inf)).astype(np.float32)
                     - want16.astype(np.float32))
        err = np.abs(got.astype(np.float32) - want16.astype(np.float32))
        assert np.all(err <= ulp), float(np.max(err))


@pytest.mark.parametrize("depth", [32, 64, 128, 256])
@pytest.mark.parametrize("repeat,past", [(8, 0), (4, 1), (8, 65), (2, 129), (1, 127), (4, 600)])
@pytest.mark.parametrize("io,kv", [(np.float32, np.float32), (np.float16, np.float16),
                                   (np.float32, np.float16)])
def test_decode_wave_states_with_several_heads_a_workgroup(gpu_ctx, depth, repeat, past, io, kv):
    """Enough sequences that a workgroup carries up to four heads of a kv head: waves without a
    column, one row past a wave's share, the own column alone, several splits; every head dim
    (groups of 4 to 64 lanes)."""
    batch = 520 if past < 600 else 64
    case = StateCase("", batch, repeat, 1, 1, depth, past + 8, 0, past, 1)
    x = random_state_inputs(case, seed=past + depth + repeat, f16_values=True)
    want = oracle_state_attention(case, x)
    got = run_attention(gpu_ctx, case, x, io=io, kv=kv)
    if io == np.float32:
        ok, fails, max_abs, worst = oracle.allclose(got, want, atol=STATE_ATOL, rtol=0)
        assert ok, (fails, max_abs, worst)
    else:
        ulp = np.spacing(np.abs(want.astype(np.float16))).astype(np.float32)
        assert np.all(np.abs(got.astype(np.float32) - want.astype(np.float16)) <= ulp + STATE_ATOL)


ROWS_CASES = [
    # chunks of rows with D = 64 / 128: the matrix-core form (16 query rows a workgroup, key
    # blocks of 32 dealt to the waves: eight for D = 64, four for D = 128)
    StateCase("rows D64 M128 P0 r8 (decoder prefill)", 1, 32, 4, 128, 64, 256, 0, 0, 128),
    StateCase("rows D64 M40 Q33 P100 pad + slot/ins straddle", 2, 8, 2, 40, 64, 192, 0, 100, 33),
    StateCase("rows D128 M64 P31 r1", 1, 4, 4, 64, 128, 128, 0, 31, 64),
    StateCase("rows D128 M33 Q2 P0", 1, 2, 1, 33, 128, 64, 0, 0, 2),
    StateCase("rows D64 sliding W48 P200 wrap", 2, 4, 2, 70, 64, 48, 48, 200, 70),
    StateCase("rows D64 sliding W16 M64 Q50 gt W", 1, 4, 4, 64, 64, 16, 16, 7, 50),
    StateCase("rows D128 sliding W100 C128 P1000", 1, 8, 2, 35, 128, 128, 100, 1000, 20),
    StateCase("rows D64 M2 Q1 P5", 1, 4, 2, 2, 64, 16, 0, 5, 1),
    # more key blocks than waves, D = 64
    StateCase("rows D64 M64 P300, 12 blocks", 1, 8, 2, 64, 64, 512, 0, 300, 64),
    StateCase("rows D64 M40 Q37 P1000, 33 blocks", 2, 4, 1, 40, 64, 1100, 0, 1000, 37),
    StateCase("rows D64 sliding W300 P900", 1, 4, 2, 48, 64, 300, 300, 900, 48),
]


@pytest.mark.parametrize("case", ROWS_CASES, ids=lambda c: c.name)
@pytest.mark.parametrize("io,kv", [(np.float32, np.float32), (np.float16, np.float16),
                                   (np.float32, np.float16)])
def test_chunks_of_rows_on_the_matrix_cores(gpu_ctx, case, io, kv):
    """M > 1 with D = 64 / 128 (f32 MFMA, online softmax per lane): the reference's gate for
    f32 output (atol 5e-6, rtol 0); for fp16 output the same gate plus one fp16 ulp of the
    oracle's value (the rounding of the stored result); pad rows exact +0; poison in every slot
    row that must not be read and in the ins pad rows."""
    x = random_state_inputs(case, seed=case.past + case.depth + case.chunk_rows, f16_values=True)
    x["ins_k"][:, :, case.query:] = 9.0
    x["ins_v"][:, :, case.query:] = 400.0
    want = oracle_state_attention(case, x)
    got = run_attention(gpu_ctx, case, x, io=io, kv=kv)
    pad = got[:, :, case.query:, :]
    assert np.all(pad == 0.0) and not np.any(np.signbit(pad))
    if io == np.float32:
        ok, fails, max_abs, worst = oracle.allclose(got, want, atol=STATE_ATOL, rtol=0)
        assert ok, (fails, max_abs, worst)
    else:
        want16 = want.astype(np.float16)
        ulp = np.abs(np.nextafter(want16, np.float16(np.inf)).astype(np.float32)
                     - want16.astype(np.float32))
        err = np.abs(got.astype(np.float32) - want16.astype(np.float32))
        assert np.all(err <= ulp + STATE_ATOL), float(np.max(err - ulp))


@pytest.mark.parametrize("case", [
    StateCase("D128 more blocks than waves", 1, 4, 2, 40, 128, 800, 0, 700, 37),
    StateCase("D256 more blocks than waves", 1, 4, 1, 20, 256, 400, 0, 290, 20),
    StateCase("D256 straddle at the first key", 1, 2, 1, 33, 256, 64, 0, 1, 31),
    StateCase("D128 window wraps inside a block", 1, 4, 2, 24, 128, 90, 90, 155, 24),
    StateCase("D256 window below a block", 1, 2, 1, 18, 256, 20, 20, 70, 18),
    StateCase("D64 window whole blocks", 1, 4, 2, 17, 64, 512, 512, 999, 17),
], ids=lambda c: c.name)
@pytest.mark.parametrize("io,kv", [(np.float32, np.float32), (np.float16, np.float16),
                                   (np.float32, np.float16)])
def test_chunk_key_blocks_from_slot_and_step(gpu_ctx, case, io, kv):
    """Key blocks wholly in the slot, wholly in this step's rows, straddling both, and wrapping in
    the window, for every head dim's wave count."""
    x = random_state_inputs(case, seed=case.past + case.depth, f16_values=True)
    x["ins_k"][:, :, case.query:] = 9.0
    x["ins_v"][:, :, case.query:] = 400.0
    want = oracle_state_attention(case, x)
    got = run_attention(gpu_ctx, case, x, io=io, kv=kv).astype(np.float32)
    if io == np.float32:
        ok, fails, max_abs, worst = oracle.allclose(got, want, atol=STATE_ATOL, rtol=0)
        assert ok, (fails, max_abs, worst)
    else:
        ulp = np.spacing(np.abs(want.astype(np.float16))).astype(np.float32)
        assert np.all(np.abs(got - want.astype(np.float16)) <= ulp + STATE_ATOL)


def test_chunk_rows_do_not_depend_on_the_batch(gpu_ctx):
    """A large grid puts two blocks of 16 query rows into one workgroup (the parked K / V blocks
    serve both); a row's arithmetic is the same, so one sequence alone and the same sequence as
    the first of eight give the same bits."""
    big = StateCase("rows D64 M64 P70 B8", 8, 32, 32, 64, 64, 160, 0, 70, 61)
    x = random_state_inputs(big, seed=3, f16_values=False)
    whole = run_attention(gpu_ctx, big, x)
    one = StateCase("rows D64 M64 P70 B1", 1, 32, 32, 64, 64, 160, 0, 70, 61)
    first = {k: np.ascontiguousarray(v[:1]) for k, v in x.items()}
    alone = run_attention(gpu_ctx, one, first)
    assert np.array_equal(alone.view(np.uint32), whole[:1].view(np.uint32))
    ok, fails, max_abs, worst = oracle.allclose(alone, oracle_state_attention(one, first),
                                                atol=STATE_ATOL, rtol=0)
    assert ok, (fails, max_abs, worst)


def test_chunks_of_rows_with_device_lengths_and_mutation_witness(gpu_ctx):
    """The device-lengths form of a chunk equals the scalar form bit for bit, and a dropped
    window bound, a ring taken modulo the capacity, or an ignored kv repeat (the oracle's
    mutations) would each be seen at this gate."""
    case = StateCase("rows D64 sliding W40 C48 P200 Q33", 2, 8, 2, 40, 64, 48, 40, 200, 33)
    x = random_state_inputs(case, seed=5, f16_values=False)
    got = run_attention(gpu_ctx, case, x)
    want = oracle_state_attention(case, x)
    ok, fails, max_abs, worst = oracle.allclose(got, want, atol=STATE_ATOL, rtol=0)
    assert ok, (fails, max_abs, worst)
    for mutation in (oracle.MUT_DROP_LOWER_BOUND, oracle.MUT_RING_MOD_CAPACITY,
                     oracle.MUT_IGNORE_KV_REPEAT):
        wrong = oracle_state_attention(case, x, mutation=mutation)
        assert not oracle.allclose(got, wrong, atol=STATE_ATOL, rtol=0)[0], mutation
    bufs = {k: gpu_ctx.upload(np.ascontiguousarray(v, dtype=np.float32)) for k, v in x.items()}
    out = gpu_ctx.upload(np.full(got.size, 7.0, dtype=np.float32))
    lengths = gpu_ctx.zeros(16)
    gpu_ctx.lengths_set(lengths, case.past, case.query)
    spec = {k: v for k, v in case.kwargs().items() if k not in ("past", "query")}
    gpu_ctx.attention_state_lengths(bufs["q"], bufs["ins_k"], bufs["ins_v"], bufs["slot_k"],
                                    bufs["slot_v"], out, half_scale=oracle.half_scale(case.depth),
                                    lengths=lengths, max_past=case.capacity - 1, **spec)
    again = out.download(np.float32, got.shape)
    assert np.array_equal(again.view(np.uint32), got.view(np.uint32))
    assert lengths.download(np.uint32, (4,))[2] == 0


@pytest.mark.parametrize("case", DECODE_CASES, ids=lambda c: c.name)
@pytest.mark.parametrize("io,kv", [(np.float32, np.float32), (np.float16, np.float16)])
def test_decode_with_device_lengths_equals_scalar_form(gpu_ctx, case, io, kv):
    """pastLength read on the device (a recorded decode step) gives the bits of the call that
    carries it as an argument.  Without a window the device form asks for the first chunk's
    rows before the lengths arrive, bounded by the capacity only: every slot row the step must
    not see (columns >= pastLength) holds NaN here and must not reach the result."""
    x = random_state_inputs(case, seed=case.past * 3 + case.depth, f16_values=True)
    if case.window == 0:
        x["slot_k"][:, :, case.past:] = np.nan
        x["slot_v"][:, :, case.past:] = np.nan
    want = run_attention(gpu_ctx, case, x, io=io, kv=kv)
    assert np.all(np.isfinite(want.astype(np.float32)))
    bufs = {k: gpu_ctx.upload(np.ascontiguousarray(
        v, dtype=io if k in ("q", "ins_k", "ins_v") else kv)) for k, v in x.items()}
    out = gpu_ctx.upload(np.full(want.size, 123.0, dtype=io))
    max_past = case.past if case.window else case.capacity - 1
    ws = gpu_ctx.alloc(max(16, gpu_ctx.attention_state_workspace(
        case.batch, case.heads, case.kv_heads, 1, case.depth, case.window, max_past, 1)))
    lengths = gpu_ctx.zeros(16)
    gpu_ctx.lengths_set(lengths, case.past, 1)
    gpu_ctx.attention_state_lengths(
        bufs["q"], bufs["ins_k"], bufs["ins_v"], bufs["slot_k"], bufs["slot_v"], out,
        batch=case.batch, heads=case.heads, kv_heads=case.kv_heads, chunk_rows=1,
        depth=case.depth, capacity=case.capacity, window=case.window,
        half_scale=oracle.half_scale(case.depth), lengths=lengths, max_past=max_past,
        io_dtype=ka.dtype_code(io), kv_dtype=ka.dtype_code(kv), workspace=ws)
    got = out.download(io, want.shape)
    assert lengths.download(np.uint32, (4,))[2] == 0
    assert got.tobytes() == want.tobytes()
    for b in list(bufs.values()) + [out, ws, lengths]:
        b.free()


@pytest.mark.parametrize("max_past,device_past", [(600, 900), (100, 700)])
def test_replay_beyond_the_sized_past_raises_the_fault_word(gpu_ctx, max_past, device_past):
    """A launch sized for `max_past` (5 splits, or a single split without a workspace) meets a
    device-side pastLength that needs more splits: the fault word is raised, `out` keeps its
    bytes, and the arrival counters stay clean — the same launch with a legal pastLength
    afterwards still equals the scalar form bitwise.  Every workgroup exits normally."""
    case = StateCase("guard", 1, 8, 2, 1, 128, 1024, 0, device_past, 1)
    x = random_state_inputs(case, seed=11, f16_values=True)
    io = kv = np.float16
    bufs = {k: gpu_ctx.upload(np.ascontiguousarray(v, dtype=np.float16)) for k, v in x.items()}
    sentinel = np.full(case.heads * case.depth, 123.0, dtype=io)
    out = gpu_ctx.upload(sentinel)
    ws = gpu_ctx.alloc(max(16, gpu_ctx.attention_state_workspace(
        1, case.heads, case.kv_heads, 1, case.depth, 0, max_past, 1)))
    lengths = gpu_ctx.zeros(16)

    def launch():
        gpu_ctx.attention_state_lengths(
            bufs["q"], bufs["ins_k"], bufs["ins_v"], bufs["slot_k"], bufs["slot_v"], out,
            batch=1, heads=case.heads, kv_heads=case.kv_heads, chunk_rows=1, depth=case.depth,
            capacity=case.capacity, window=0, half_scale=oracle.half_scale(case.depth),
            lengths=lengths, max_past=max_past, io_dtype=ka.F16, kv_dtype=ka.F16,
            workspace=ws if max_past > 512 else None)

    gpu_ctx.lengths_set(lengths, device_past, 1)
    launch()
    state = lengths.download(np.uint32, (4,))
    assert state[2] == 1 and state[0] == device_past
    assert out.download(io, sentinel.shape).tobytes() == sentinel.tobytes()
    # a legal pastLength through the same launch shape afterwards
    legal = StateCase("legal", 1, 8, 2, 1, 128, 1024, 0, max_past, 1)
    want = run_attention(gpu_ctx, legal, x, io=io, kv=kv)
    gpu_ctx.lengths_set(lengths, max_past, 1)
    launch()
    assert lengths.download(np.uint32, (4,))[2] == 0
    assert out.download(io, want.shape).tobytes() == want.tobytes()
    for b in list(bufs.values()) + [out, ws, lengths]:
        b.free()


def test_config2_decode_attention(gpu_ctx):
    """benchmark config 2: B=1, H=32, Hkv=8, D=128, 4095 slot rows + this step's row, fp16."""
    case = StateCase("config 2", 1, 32, 8, 1, 128, 4096, 0, 4095, 1)
    x = random_state_inputs(case, seed=2, f16_values=True)
    want = oracle_state_attention(case, x)
    got32 = run_attention(gpu_ctx, case, x, io=np.float32, kv=np.float16)
    ok, fails, max_abs, worst = oracle.allclose(got32, want, atol=STATE_ATOL, rtol=0)
    assert ok, (fails, max_abs, worst)
    got16 = run_attention(gpu_ctx, case, x, io=np.float16, kv=np.float16)
    want16 = want.astype(np.float16).astype(np.float32)
    assert np.max(np.abs(got16.astype(np.float32) - want16)) <= 2.5e-4  # 1 ulp at |out| < 0.25
    # identical bits for a larger capacity: the work never depends on C
    big = StateCase("config 2 C8192", 1, 32, 8, 1, 128, 8192, 0, 4095, 1)
    xb = {k: v.copy() for k, v in x.items()}
    for name in ("slot_k", "slot_v"):
        grown = np.full((1, 8, 8192, 128), 9.0 if name == "slot_k" else 400.0, dtype=np.float32)
        grown[:, :, :4096] = x[name]
        xb[name] = grown
    got_big = run_attention(gpu_ctx, big, xb, io=np.float32, kv=np.float16)
    assert np.array_equal(got_big.view(np.uint32), got32.view(np.uint32))


def test_mutations_would_be_caught(gpu_ctx):
    """The GPU result sits within tolerance of the faithful oracle and far from every mutated
    oracle on that mutation's witness case."""
    witnesses = {
        oracle.MUT_DROP_LOWER_BOUND: "sliding W4 P10 wrap",
        oracle.MUT_RING_MOD_CAPACITY: "sliding W4 C8 wrap",
        oracle.MUT_PAD_ROWS_COMPUTED: "full r2 pad B2 D6",
        oracle.MUT_IGNORE_KV_REPEAT: "full r2 pad B2 D6",
        oracle.MUT_SCALE_ONE_SIDE: "full r1 prefill B2",
        oracle.MUT_OVERFLOW_FORM: "sliding W2 P near u32 max",
    }
    for mutation, name in witnesses.items():
        case = next(c for c in PARITY_CASES if c.name == name)
        x = make_state_inputs(case)
        got = run_attention(gpu_ctx, case, x)
        bad = oracle_state_attention(case, x, mutation=mutation)
        assert np.max(np.abs(got - bad)) > 1e-3, name


def test_attention_rejections(gpu_ctx):
    buf = gpu_ctx.zeros(1 << 16)
    base = dict(batch=1, heads=4, kv_heads=2, chunk_rows=2, depth=8, capacity=8, window=0,
                half_scale=0.5, past=0, query=1)
    call = lambda **kw: gpu_ctx.attention_state(buf, buf, buf, buf, buf, buf,  # noqa: E731
                                                **{**base, **kw})
    with pytest.raises(ka.GpuValidationError):
        call(heads=3)
    with pytest.raises(ka.GpuValidationError):
        call(window=9)
    with pytest.raises(ka.ExecutionError):  # capacity overflow is rejected before launch
        call(past=7, query=2)
    with pytest.raises(ka.ExecutionError):
        call(query=3)
    with pytest.raises(ka.ExecutionError):
        call(query=0)
    with pytest.raises(ka.GpuValidationError):
        call(half_scale=float("nan"))
    # split-K needs a workspace when there is more than one split
    big = dict(batch=1, heads=8, kv_heads=2, chunk_rows=1, depth=128, capacity=4096, window=0,
               half_scale=0.3, past=4000, query=1, io_dtype=ka.F16, kv_dtype=ka.F16)
    huge = gpu_ctx.zeros(2 * 4096 * 128 * 2)
    with pytest.raises(ka.GpuValidationError):
        gpu_ctx.attention_state(buf, buf, buf, huge, huge, buf, **big)
    huge.free()
    buf.free()


# ---------------------------------------------------------------------------- state_append

def run_append(ctx, x, slot, xd=np.float32, sd=np.float32, **spec):
    dx = ctx.upload(np.ascontiguousarray(x, dtype=xd))
    ds = ctx.upload(np.ascontiguousarray(slot, dtype=sd))
    ctx.state_append(dx, ds, x_dtype=ka.dtype_code(xd), slot_dtype=ka.dtype_code(sd), **spec)
    got = ds.download(sd, np.shape(slot))
    dx.free()
    ds.free()
    return got


def test_append_reference_vectors(gpu_ctx):
    # packages/runtime/tests/kernel_state_attention_test.ts:481-503
    spec = dict(kv_planes=1, chunk_rows=4, depth=1, capacity=4, window=4)
    slot = np.array([-1, -2, -3, -4], dtype=np.float32)
    x = np.array([100, 200, 300, 400], dtype=np.float32)
    assert run_append(gpu_ctx, x, slot, past=2, query=2, **spec).tolist() == [-1, -2, 100, 200]
    assert run_append(gpu_ctx, x, slot, past=3, query=3, **spec).tolist() == [200, 300, -3, 100]
    collide = run_append(gpu_ctx, x, np.array([-1, -2], dtype=np.float32), kv_planes=1,
                         chunk_rows=4, depth=1, capacity=2, window=2, past=0, query=4)
    assert collide.tolist() == [300, 400]


@pytest.mark.parametrize("window,capacity,past,query,m", [(0, 64, 5, 7, 9), (6, 6, 13, 3, 5),
                                                          (4, 8, 9, 2, 3), (2, 2, 5, 4, 4),
                                                          (0, 40, 39, 1, 1)])
def test_append_matches_oracle_bytes(gpu_ctx, window, capacity, past, query, m):
    rng = np.random.default_rng(past)
    planes, d = 6, 16
    x = rng.normal(size=(planes, m, d)).astype(np.float32)
    x[:, query:] = 9.0  # pad rows must never reach the slot
    slot = rng.normal(size=(planes, capacity, d)).astype(np.float32)
    spec = dict(kv_planes=planes, chunk_rows=m, depth=d, capacity=capacity, window=window,
                past=past, query=query)
    want = oracle.state_append(x, slot, **spec)
    got = run_append(gpu_ctx, x, slot, **spec)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    # f32 -> f16 slot: round to nearest even of the same values
    got16 = run_append(gpu_ctx, x, slot.astype(np.float16), sd=np.float16, **spec)
    want16 = oracle.state_append(x.astype(np.float16).astype(np.float32),
                                 slot.astype(np.float16).astype(np.float32), **spec)
    assert np.array_equal(got16, want16.astype(np.float16))


def test_append_rejections(gpu_ctx):
    buf = gpu_ctx.zeros(4096)
    spec = dict(kv_planes=1, chunk_rows=2, depth=4, capacity=4, window=0, past=0, query=1)
    with pytest.raises(ka.ExecutionError):
        gpu_ctx.state_append(buf, buf, **{**spec, "past": 3, "query": 2})
    with pytest.raises(ka.ExecutionError):
        gpu_ctx.state_append(buf, buf, **{**spec, "query": 3})
    with pytest.raises(ka.GpuValidationError):
        gpu_ctx.state_append(buf, buf, **{**spec, "window": 5})
    buf.free()


def test_chain_prefill_then_decode_on_device(gpu_ctx):
    """Prefill -> decode chain with slots that live on the device and start as zeros
    (packages/runtime/tests/gpu_state_execution_test.ts:152-212,268-350): readers first, then
    append; equals ONE full-history causal attention in float64."""
    heads, kv_heads, depth, capacity = 8, 2, 64, 64
    r = heads // kv_heads
    rng = np.random.default_rng(77)
    slot_k = gpu_ctx.zeros(kv_heads * capacity * depth * 4)
    slot_v = gpu_ctx.zeros(kv_heads * capacity * depth * 4)
    ws = gpu_ctx.alloc(gpu_ctx.attention_state_workspace(1, heads, kv_heads, 8, depth, 0, capacity))
    past = 0
    outs, qs, ks, vs = [], [], [], []
    for m, query in [(8, 8), (8, 3)] + [(1, 1)] * 20:
        q = rng.normal(size=(1, heads, m, depth)).astype(np.float32)
        k = rng.normal(size=(1, kv_heads, m, depth)).astype(np.float32)
        v = rng.normal(size=(1, kv_heads, m, depth)).astype(np.float32)
        k[:, :, query:] = 9.0
        v[:, :, query:] = 400.0
        dq, dk, dv = gpu_ctx.upload(q), gpu_ctx.upload(k), gpu_ctx.upload(v)
        out = gpu_ctx.alloc(q.nbytes)
        gpu_ctx.attention_state(dq, dk, dv, slot_k, slot_v, out, batch=1, heads=heads,
                                kv_heads=kv_heads, chunk_rows=m, depth=depth, capacity=capacity,
                                window=0, half_scale=oracle.half_scale(depth), past=past,
                                query=query, workspace=ws)
        spec = dict(kv_planes=kv_heads, chunk_rows=m, depth=depth, capacity=capacity, window=0,
                    past=past, query=query)
        gpu_ctx.state_append(dk, slot_k, **spec)
        gpu_ctx.state_append(dv, slot_v, **spec)
        outs.append(out.download(np.float32, q.shape)[:, :, :query])
        qs.append(q[:, :, :query])
        ks.append(k[:, :, :query])
        vs.append(v[:, :, :query])
        past += query
        for b in (dq, dk, dv, out):
            b.free()
    cat = lambda parts: np.concatenate(parts, axis=2)  # noqa: E731
    total = past
    i = np.arange(total)
    s = float(oracle.half_scale(depth))
    want = helpers.dense_attention_f64(cat(qs), np.repeat(cat(ks), r, axis=1),
                                       np.repeat(cat(vs), r, axis=1), i[None, :] <= i[:, None],
                                       s * s)
    assert np.max(np.abs(cat(outs) - want)) <= STATE_ATOL
    # the slot holds exactly the valid rows; rows past `total` are still the initial zeros
    got_k = slot_k.download(np.float32, (kv_heads, capacity, depth))
    assert np.array_equal(got_k[:, :total], cat(ks)[0])
    assert np.all(got_k[:, total:] == 0.0)
    for b in (slot_k, slot_v, ws):
        b.free()


# ---------------------------------------------------------------------------- ragged batch

def test_config3_ragged_batch_equals_one_at_a_time(gpu_ctx):
    """benchmark config 3: 16 sequences, KV lengths ~ U{128..4096} (seeded), packed with
    prefix-sum offsets, H=32, Hkv=8, D=128, fp16 KV.  One launch; every sequence is then run
    alone through krm_attention_state and the bits must agree; a few are checked against the
    oracle (atol 5e-6 on f32 output)."""
    rng = np.random.default_rng(3)
    nseq, heads, kv_heads, depth = 16, 32, 8, 128
    lengths = rng.integers(128, 4097, size=nseq)
    cu = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    total = int(cu[-1])
    f16 = lambda a: a.astype(np.float16)  # noqa: E731
    slot_k = f16(rng.normal(size=(kv_heads, total, depth)))
    slot_v = f16(rng.normal(size=(kv_heads, total, depth)))
    q = f16(rng.normal(size=(nseq, heads, depth))).astype(np.float32)
    ins_k = f16(rng.normal(size=(nseq, kv_heads, depth))).astype(np.float32)
    ins_v = f16(rng.normal(size=(nseq, kv_heads, depth))).astype(np.float32)
    half = oracle.half_scale(depth)

    d = {name: gpu_ctx.upload(arr) for name, arr in
         dict(q=q, ins_k=ins_k, ins_v=ins_v, slot_k=slot_k, slot_v=slot_v).items()}
    out = gpu_ctx.alloc(q.nbytes)
    ws = gpu_ctx.alloc(gpu_ctx.attention_varlen_workspace(nseq, heads, kv_heads, depth, total))
    gpu_ctx.attention_varlen(d["q"], d["ins_k"], d["ins_v"], d["slot_k"], d["slot_v"], out, cu,
                             heads=heads, kv_heads=kv_heads, depth=depth, total_rows=total,
                             half_scale=half, io_dtype=ka.F32, kv_dtype=ka.F16, workspace=ws)
    batched = out.download(np.float32, q.shape)
    for b in list(d.values()) + [out, ws]:
        b.free()

    for i in range(nseq):
        past = int(lengths[i])
        case = StateCase(f"seq {i}", 1, heads, kv_heads, 1, depth, past + 1, 0, past, 1)
        sk = np.zeros((1, kv_heads, past + 1, depth), dtype=np.float32)
        sv = np.zeros_like(sk)
        sk[0, :, :past] = slot_k[:, cu[i]:cu[i + 1]]
        sv[0, :, :past] = slot_v[:, cu[i]:cu[i + 1]]
        x = dict(q=q[i].reshape(1, heads, 1, depth), ins_k=ins_k[i].reshape(1, kv_heads, 1, depth),
                 ins_v=ins_v[i].reshape(1, kv_heads, 1, depth), slot_k=sk, slot_v=sv)
        alone = run_attention(gpu_ctx, case, x, io=np.float32, kv=np.float16)
        assert np.array_equal(alone.reshape(heads, depth).view(np.uint32),
                              batched[i].view(np.uint32)), i
        if i % 5 == 0:
            want = oracle_state_attention(case, x)
            ok, fails, max_abs, worst = oracle.allclose(alone, want, atol=STATE_ATOL, rtol=0)
            assert ok, (i, fails, max_abs, worst)


def test_varlen_edges(gpu_ctx):
    """Empty past (a sequence whose only column is its own) and single-split sequences."""
    heads, kv_heads, depth = 8, 2, 64
    lengths = np.array([0, 5, 256, 257, 0, 1])
    cu = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    total = int(cu[-1])
    rng = np.random.default_rng(9)
    nseq = len(lengths)
    slot_k = rng.normal(size=(kv_heads, total, depth)).astype(np.float32)
    slot_v = rng.normal(size=(kv_heads, total, depth)).astype(np.float32)
    q = rng.normal(size=(nseq, heads, depth)).astype(np.float32)
    ins_k = rng.normal(size=(nseq, kv_heads, depth)).astype(np.float32)
    ins_v = rng.normal(size=(nseq, kv_heads, depth)).astype(np.float32)
    d = {name: gpu_ctx.upload(arr) for name, arr in
         dict(q=q, ins_k=ins_k, ins_v=ins_v, slot_k=slot_k, slot_v=slot_v).items()}
    out = gpu_ctx.alloc(q.nbytes)
    ws = gpu_ctx.alloc(gpu_ctx.attention_varlen_workspace(nseq, heads, kv_heads, depth, total))
    gpu_ctx.attention_varlen(d["q"], d["ins_k"], d["ins_v"], d["slot_k"], d["slot_v"], out, cu,
                             heads=heads, kv_heads=kv_heads, depth=depth, total_rows=total,
                             half_scale=oracle.half_scale(depth), workspace=ws)
    got = out.download(np.float32, q.shape)
    for i in range(nseq):
        past = int(lengths[i])
        case = StateCase(f"seq {i}", 1, heads, kv_heads, 1, depth, past + 1, 0, past, 1)
        sk = np.zeros((1, kv_heads, past + 1, depth), dtype=np.float32)
        sv = np.zeros_like(sk)
        sk[0, :, :past] = slot_k[:, cu[i]:cu[i + 1]]
        sv[0, :, :past] = slot_v[:, cu[i]:cu[i + 1]]
        x = dict(q=q[i].reshape(1, heads, 1, depth), ins_k=ins_k[i].reshape(1, kv_heads, 1, depth),
                 ins_v=ins_v[i].reshape(1, kv_heads, 1, depth), slot_k=sk, slot_v=sv)
        want = oracle_state_attention(case, x)
        assert np.max(np.abs(got[i].reshape(want.shape) - want)) <= STATE_ATOL, i
    with pytest.raises(ka.GpuValidationError):  # not ascending
        gpu_ctx.attention_varlen(d["q"], d["ins_k"], d["ins_v"], d["slot_k"], d["slot_v"], out,
                                 [0, 5, 3], heads=heads, kv_heads=kv_heads, depth=depth,
                                 total_rows=total, half_scale=0.3, workspace=ws)
    for b in list(d.values()) + [out, ws]:
        b.free()


def test_varlen_planned_on_the_device_is_recordable(gpu_ctx):
    """The ragged step with its tables built on the device: equals the host-table form bitwise;
    recorded once and replayed while the sequences grow (the offsets are rewritten between the
    replays, with eager work and synchronisations in between) every replay equals the eager
    host-table result of the same lengths; offsets that are not ascending raise the plan's
    fault word and leave `out` untouched."""
    heads, kv_heads, depth, nseq = 8, 2, 128, 5
    capacity_rows = [700, 300, 900, 140, 20]           # rows each sequence owns in the slot
    starts = np.concatenate([[0], np.cumsum(capacity_rows)]).astype(np.int64)
    total = int(starts[-1])
    rng = np.random.default_rng(17)
    f16 = lambda a: a.astype(np.float16)  # noqa: E731
    slot_k, slot_v = (f16(rng.normal(size=(kv_heads, total, depth))) for _ in range(2))
    q, ins_k, ins_v = (f16(rng.normal(size=(nseq, h, depth))) for h in (heads, kv_heads, kv_heads))
    d = {name: gpu_ctx.upload(arr) for name, arr in
         dict(q=q, ins_k=ins_k, ins_v=ins_v, slot_k=slot_k, slot_v=slot_v).items()}
    half = oracle.half_scale(depth)
    out, out_host = gpu_ctx.alloc(q.nbytes), gpu_ctx.alloc(q.nbytes)
    ws = gpu_ctx.alloc(gpu_ctx.attention_varlen_workspace(nseq, heads, kv_heads, depth, total))
    ws_host = gpu_ctx.alloc(gpu_ctx.attention_varlen_workspace(nseq, heads, kv_heads, depth, total))
    plan = gpu_ctx.alloc(gpu_ctx.attention_varlen_plan_bytes(nseq))
    max_splits = gpu_ctx.attention_varlen_max_splits(nseq, depth, ka.F16, total)
    assert max_splits == total // 128 + nseq
    cu_dev = gpu_ctx.alloc(4 * (nseq + 1))
    common = dict(heads=heads, kv_heads=kv_heads, depth=depth, total_rows=total, half_scale=half,
                  io_dtype=ka.F16, kv_dtype=ka.F16)

    # each replay sees other (ascending) offsets: sequence i holds fill * capacity_rows[i] rows
    def offsets(fill):
        cu = np.zeros(nseq + 1, dtype=np.int32)
        for i in range(nseq):
            cu[i + 1] = cu[i] + int(capacity_rows[i] * fill)
        return cu

    with gpu_ctx.record() as rec:
        gpu_ctx.attention_varlen_plan(cu_dev, plan, nseq=nseq, depth=depth, kv_dtype=ka.F16,
                                      total_rows=total, max_splits=max_splits)
        gpu_ctx.attention_varlen_planned(d["q"], d["ins_k"], d["ins_v"], d["slot_k"], d["slot_v"],
                                         out, plan, nseq=nseq, max_splits=max_splits,
                                         workspace=ws, **common)
    for fill in (0.25, 0.6, 1.0, 0.4):
        cu = offsets(fill)
        cu_dev.upload(cu)
        out.upload(np.full(q.size, 77.0, dtype=np.float16))
        rec.graph.launch()
        got = out.download(np.float16, q.shape)
        assert plan.download(np.int32, (2 * (nseq + 1) + 1,))[-1] == 0
        gpu_ctx.attention_varlen(d["q"], d["ins_k"], d["ins_v"], d["slot_k"], d["slot_v"],
                                 out_host, cu, workspace=ws_host, **common)
        want = out_host.download(np.float16, q.shape)
        assert got.tobytes() == want.tobytes(), fill
    rec.graph.destroy()

    # offsets that break the contract: fault word, no store
    for bad in ([0, 50, 40, 60, 70, 80], [0, 10, 20, 30, 40, total + 1], [-1, 10, 20, 30, 40, 50]):
        cu_dev.upload(np.array(bad, dtype=np.int32))
        sentinel = np.full(q.size, 55.0, dtype=np.float16)
        out.upload(sentinel)
        gpu_ctx.attention_varlen_plan(cu_dev, plan, nseq=nseq, depth=depth, kv_dtype=ka.F16,
                                      total_rows=total, max_splits=max_splits)
        gpu_ctx.attention_varlen_planned(d["q"], d["ins_k"], d["ins_v"], d["slot_k"], d["slot_v"],
                                         out, plan, nseq=nseq, max_splits=max_splits,
                                         workspace=ws, **common)
        assert plan.download(np.int32, (2 * (nseq + 1) + 1,))[-1] == 1, bad
        assert out.download(np.float16, (q.size,)).tobytes() == sentinel.tobytes(), bad
    # a legal plan afterwards still works (the counters were left clean)
    cu = offsets(1.0)
    cu_dev.upload(cu)
    gpu_ctx.attention_varlen_plan(cu_dev, plan, nseq=nseq, depth=depth, kv_dtype=ka.F16,
                                  total_rows=total, max_splits=max_splits)
    gpu_ctx.attention_varlen_planned(d["q"], d["ins_k"], d["ins_v"], d["slot_k"], d["slot_v"],
                                     out, plan, nseq=nseq, max_splits=max_splits, workspace=ws,
                                     **common)
    gpu_ctx.attention_varlen(d["q"], d["ins_k"], d["ins_v"], d["slot_k"], d["slot_v"], out_host,
                             cu, workspace=ws_host, **common)
    assert out.download(np.float16, q.shape).tobytes() == out_host.download(np.float16, q.shape).tobytes()
    for b in list(d.values()) + [out, out_host, ws, ws_host, plan, cu_dev]:
        b.free()


@pytest.mark.parametrize("splits", [5, 8, 9, 16, 24, 25, 32, 33, 40, 57, 64])
def test_decode_merges_any_number_of_splits(gpu_ctx, splits):
    """Passes of 32 partials, short ones in blocks of eight: the class's gate against the oracle."""
    case = StateCase("splits", 1, 2, 1, 1, 128, splits * 64 + 1, 0, splits * 64, 1)  # f32: 64 columns a split
    x = random_state_inputs(case, seed=splits, f16_values=False)
    got = run_attention(gpu_ctx, case, x)
    ok, fails, max_abs, worst = oracle.allclose(got, oracle_state_attention(case, x), atol=STATE_ATOL, rtol=0)
    assert ok, (fails, max_abs, worst)


@pytest.mark.parametrize("batch,heads,kv_heads,depth,past,window", [
    (1, 12, 3, 128, 641, 0), (2, 20, 5, 128, 1100, 0), (1, 24, 12, 64, 2300, 0), (3, 8, 1, 256, 600, 0),
    (1, 18, 9, 128, 3000, 1100)])
def test_decode_of_splits_that_share_rows_on_an_xcd(gpu_ctx, batch, heads, kv_heads, depth, past, window):
    """Several splits and several head groups a kv head (the folded grid): splits no multiple of eight, kv heads
    past eight, a batch, a window; the class's gate against the oracle."""
    case = StateCase("folded", batch, heads, kv_heads, 1, depth, window or past + 1, window, past, 1)
    x = random_state_inputs(case, seed=past, f16_values=False)
    got = run_attention(gpu_ctx, case, x)
    ok, fails, max_abs, worst = oracle.allclose(got, oracle_state_attention(case, x), atol=STATE_ATOL, rtol=0)
    assert ok, (fails, max_abs, worst)


@pytest.mark.parametrize("batch,heads,kv_heads,depth,past", [(4, 12, 3, 128, 620), (3, 8, 2, 128, 1300),
                                                             (3, 32, 4, 64, 1200), (2, 32, 8, 128, 700)])
def test_decode_deals_the_last_splits_of_a_batch_over_all_xcds(gpu_ctx, batch, heads, kv_heads, depth, past):
    """The folded grid's last row, which begins on another XCD for every batch entry and kv head."""
    test_decode_of_splits_that_share_rows_on_an_xcd(gpu_ctx, batch, heads, kv_heads, depth, past, 0)


@pytest.mark.parametrize("nseq", [1, 62, 63, 64, 65, 127, 128, 300])
def test_varlen_plan_tables_past_a_wave(gpu_ctx, nseq):
    """The tables of a plan, by steps of 64 sequences: offsets as given, splits of 128 columns summed before each
    sequence (one up to 512 columns); one wrong offset anywhere leaves no splits and raises the fault word."""
    rng = np.random.default_rng(nseq)
    rows = rng.choice([0, 1, 511, 512, 513, 2000], size=nseq)
    cu = np.concatenate([[3], 3 + np.cumsum(rows)]).astype(np.int32)
    total = int(cu[-1])
    max_splits = gpu_ctx.attention_varlen_max_splits(nseq, 128, ka.F16, total)
    chunks = -(-rows // 128)
    prefix = np.concatenate([[0], np.cumsum(np.where(chunks <= 4, 1, chunks))])
    cu_dev, plan = gpu_ctx.alloc(cu.nbytes), gpu_ctx.alloc(gpu_ctx.attention_varlen_plan_bytes(nseq))

    def tables(offsets, total_rows, splits):
        cu_dev.upload(offsets)
        plan.upload(np.full(2 * (nseq + 1) + 1, -7, dtype=np.int32))
        gpu_ctx.attention_varlen_plan(cu_dev, plan, nseq=nseq, depth=128, kv_dtype=ka.F16,
                                      total_rows=total_rows, max_splits=splits)
        got = plan.download(np.int32, (2 * (nseq + 1) + 1,))
        return got[:nseq + 1], got[nseq + 1:-1], got[-1]

    got_cu, got_prefix, fault = tables(cu, total, max_splits)
    assert (got_cu == cu).all() and (got_prefix == prefix).all() and fault == 0
    broken = [(cu, total - 1, max_splits), (cu, total, int(prefix[-1]) - 1)]
    for at in sorted({0, nseq // 2, nseq}):
        wrong = cu.copy()
        wrong[at] = -1 if at < nseq else cu[at - 1] - 1
        broken.append((wrong, total, max_splits))
    for offsets, total_rows, splits in broken:
        got_cu, got_prefix, fault = tables(offsets, total_rows, splits)
        assert (got_cu == offsets).all() and not got_prefix.any() and fault == 1
    for b in (cu_dev, plan):
        b.free()


@pytest.mark.parametrize("io,kv", [(np.float32, np.float32), (np.float16, np.float16),
                                   (np.float32, np.float16)])
@pytest.mark.parametrize("dyn", [False, True])
def test_attention_chunk_equals_attention_transpose_and_appends(gpu_ctx, io, kv, dyn):
    """krm_attention_chunk with the row-major output and the fused append writes the bits of
    krm_attention_state + krm_transpose_01 + two krm_state_append (pad rows: zeros in the output,
    nothing appended; every other slot row untouched); with a window the append is refused and
    the row-major output alone still matches."""
    case = StateCase("chunk D64 M40 Q33 P100", 2, 8, 2, 40, 64, 192, 0, 100, 33)
    x = random_state_inputs(case, seed=77, f16_values=True)
    b, h, hkv, m, d, c = (case.batch, case.heads, case.kv_heads, case.chunk_rows, case.depth,
                          case.capacity)
    io_code, kv_code = ka.dtype_code(io), ka.dtype_code(kv)

    def upload():
        return {k: gpu_ctx.upload(np.ascontiguousarray(v, dtype=io if k in ("q", "ins_k", "ins_v")
                                                       else kv)) for k, v in x.items()}
    ref = upload()
    want_hm = gpu_ctx.upload(np.full(b * h * m * d, 5.0, dtype=io))
    gpu_ctx.attention_state(ref["q"], ref["ins_k"], ref["ins_v"], ref["slot_k"], ref["slot_v"],
                            want_hm, half_scale=oracle.half_scale(d), io_dtype=io_code,
                            kv_dtype=kv_code, **case.kwargs())
    spec = dict(kv_planes=b * hkv, chunk_rows=m, depth=d, capacity=c, window=0, x_dtype=io_code,
                slot_dtype=kv_code)
    gpu_ctx.state_append(ref["ins_k"], ref["slot_k"], past=case.past, query=case.query, **spec)
    gpu_ctx.state_append(ref["ins_v"], ref["slot_v"], past=case.past, query=case.query, **spec)
    want = want_hm.download(io, (b, h, m, d)).transpose(0, 2, 1, 3)

    got = upload()
    out = gpu_ctx.upload(np.full(b * h * m * d, 7.0, dtype=io))
    lengths = None
    if dyn:
        lengths = gpu_ctx.zeros(16)
        gpu_ctx.lengths_set(lengths, case.past, case.query)
    geometry = {k: v for k, v in case.kwargs().items() if k not in ("past", "query")}
    gpu_ctx.attention_chunk(got["q"], got["ins_k"], got["ins_v"], got["slot_k"], got["slot_v"],
                            out, half_scale=oracle.half_scale(d), past=0 if dyn else case.past,
                            query=0 if dyn else case.query, lengths=lengths, io_dtype=io_code,
                            kv_dtype=kv_code, row_major=True, append=True, **geometry)
    bits = np.uint32 if io == np.float32 else np.uint16
    kbits = np.uint32 if kv == np.float32 else np.uint16
    assert np.array_equal(out.download(io, (b, m, h, d)).view(bits), np.ascontiguousarray(want).view(bits))
    for name in ("slot_k", "slot_v"):
        assert np.array_equal(got[name].download(kv, (b, hkv, c, d)).view(kbits),
                              ref[name].download(kv, (b, hkv, c, d)).view(kbits)), name
    if dyn:
        assert lengths.download(np.uint32, (4,))[2] == 0
    with pytest.raises(ka.GpuValidationError, match="window == 0"):
        gpu_ctx.attention_chunk(got["q"], got["ins_k"], got["ins_v"], got["slot_k"], got["slot_v"],
                                out, half_scale=oracle.half_scale(d), past=case.past,
                                query=case.query, io_dtype=io_code, kv_dtype=kv_code, append=True,
                                **{**geometry, "window": 64})
    with pytest.raises(ka.GpuValidationError, match="D = 64, 128 or 256"):
        gpu_ctx.attention_chunk(got["q"], got["ins_k"], got["ins_v"], got["slot_k"], got["slot_v"],
                                out, half_scale=0.5, past=0, query=1, io_dtype=io_code,
                                kv_dtype=kv_code, **{**geometry, "depth": 32})


# ---- KV-sharing layers: two readers, one append -------------------------------------------------

SHARED_SERIES = [
    # packages/runtime/tests/gpu_state_acceptance_test.ts:846-864
    dict(name="full", heads=2, kv_heads=2, depth=4, capacity=16, window=0, chunk=3,
         steps=[(3, 3), (3, 3), (3, 3), (1, 1)], order_probe=None),
    # a ring of W = C = 4: the append of step 1 (past 3, Q 3) writes physical rows 3, 0, 1, two of
    # which the readers of the same step still have to read — the one place where the order of
    # readers and append shows in the values
    dict(name="sliding W=4", heads=2, kv_heads=2, depth=4, capacity=4, window=4, chunk=3,
         steps=[(3, 3), (3, 3), (3, 3), (1, 1)], order_probe=1),
]


@pytest.mark.parametrize("series", SHARED_SERIES, ids=lambda s: s["name"])
def test_two_readers_one_append(gpu_ctx, series):
    """Two attention calls with different queries read the same K / V rows and the same state
    slots, then ONE pair of appends follows (packages/runtime/tests/
    gpu_state_acceptance_test.ts:866-977): both outputs equal the oracle on the slots as they
    were BEFORE the append (atol 5e-6), differ from each other, and — where the ring wraps into
    rows of the same step — differ from an oracle that appended first; the slot bytes after
    every step equal the oracle's chained slots."""
    ctx = gpu_ctx
    H, Hkv, D, C, W, M = (series[k] for k in ("heads", "kv_heads", "depth", "capacity", "window",
                                              "chunk"))
    scale = oracle.half_scale(D)
    slot_k = np.zeros((1, Hkv, C, D), dtype=np.float32)
    slot_v = np.zeros((1, Hkv, C, D), dtype=np.float32)
    dk, dv = ctx.upload(slot_k), ctx.upload(slot_v)
    past = 0
    for index, (rows, query) in enumerate(series["steps"]):
        salt = 17 + index * 23
        count = Hkv * rows * D
        qs = [helpers.seeded(H * rows * D, lambda i, s=salt + 101 * r: helpers.QUERY(i + s))
              .reshape(1, H, rows, D) for r in range(2)]
        k = helpers.seeded(count, lambda i: helpers.KEY(i + salt)).reshape(1, Hkv, rows, D)
        v = helpers.seeded(count, lambda i: helpers.VALUE(i + salt)).reshape(1, Hkv, rows, D)
        common = dict(chunk_rows=rows, depth=D, capacity=C, window=W, past=past, query=query)

        def read(q, sk, sv):
            return oracle.state_attention(q, k, v, sk, sv, batch=1, heads=H, kv_heads=Hkv,
                                          scale=scale, **common)

        bk, bv = ctx.upload(k), ctx.upload(v)
        outs = []
        for q in qs:   # both readers first ...
            bq, out = ctx.upload(q), ctx.alloc(q.nbytes)
            ws = ctx.alloc(ctx.attention_state_workspace(1, H, Hkv, rows, D, W, past, query))
            ctx.attention_state(bq, bk, bv, dk, dv, out, batch=1, heads=H, kv_heads=Hkv,
                                half_scale=scale, workspace=ws, **common)
            outs.append(out.download(np.float32, q.shape))
            for b in (bq, out, ws):
                b.free()
        for src, slot in ((bk, dk), (bv, dv)):   # ... then the one pair of appends
            ctx.state_append(src, slot, kv_planes=Hkv, **common)
        for q, got in zip(qs, outs):
            want = read(q, slot_k, slot_v)
            assert np.any(np.abs(want) > 1e-3), "the expected output is trivial"
            ok, fails, max_abs, worst = oracle.allclose(got, want, atol=STATE_ATOL, rtol=0)
            assert ok, (series["name"], index, fails, max_abs, worst)
        assert outs[0].tobytes() != outs[1].tobytes()
        new_k = oracle.state_append(k, slot_k, kv_planes=Hkv, **common)
        new_v = oracle.state_append(v, slot_v, kv_planes=Hkv, **common)
        if series["order_probe"] == index:
            for q, got in zip(qs, outs):
                wrong = read(q, new_k, new_v)
                ok, *_ = oracle.allclose(got, wrong, atol=STATE_ATOL, rtol=0)
                assert not ok, "the probe step does not tell reader-first from append-first"
        slot_k, slot_v = new_k, new_v
        past += query
        assert dk.download(np.float32, slot_k.shape).tobytes() == slot_k.tobytes()
        assert dv.download(np.float32, slot_v.shape).tobytes() == slot_v.tobytes()
        bk.free()
        bv.free()
    dk.free()
    dv.free()


# ---- head dims of 256 (a sliding layer of a Gemma-4-style decoder) -------------------------------

@pytest.mark.parametrize("case,io,kv", [
    (StateCase("chunk 40 rows, past 70, D 256", 1, 4, 2, 40, 256, 128, 0, 70, 37), np.float32, np.float32),
    (StateCase("chunk 33 rows, window 48, D 256", 2, 2, 1, 33, 256, 64, 48, 90, 33), np.float32, np.float32),
    (StateCase("chunk 16 rows, D 256, fp16 state", 1, 8, 1, 16, 256, 64, 0, 20, 16), np.float32, np.float16),
    (StateCase("decode, past 300, D 256", 1, 8, 2, 1, 256, 512, 0, 300, 1), np.float32, np.float32),
    (StateCase("decode, 8:1, past 700, D 256", 1, 8, 1, 1, 256, 1024, 0, 700, 1), np.float32, np.float32),
    (StateCase("decode, window 128, D 256", 2, 4, 4, 1, 256, 128, 128, 1000, 1), np.float32, np.float32),
    (StateCase("decode, past 900, D 512 fp16", 1, 8, 1, 1, 512, 1024, 0, 900, 1), np.float16, np.float16),
], ids=lambda v: v.name if isinstance(v, StateCase) else None)
def test_head_dim_256_forms(gpu_ctx, case, io, kv):
    """The chunk kernel's D = 256 form (two waves a workgroup) and the decode kernel with rows
    that span a whole wave (f32 D = 256, fp16 D = 512) against the oracle: atol 5e-6 for f32
    output (the reference's gate), one fp16 ulp for fp16 output; pad rows exact +0."""
    x = random_state_inputs(case, seed=case.past + case.depth, f16_values=True)
    want = oracle_state_attention(case, x)
    got = run_attention(gpu_ctx, case, x, io=io, kv=kv)
    if io == np.float32:
        ok, fails, max_abs, worst = oracle.allclose(got, want, atol=STATE_ATOL, rtol=0)
        assert ok, (case.name, fails, max_abs, worst)
    else:
        ref = want.astype(np.float16).astype(np.float32)
        assert np.all(np.abs(got.astype(np.float32) - ref) <= np.abs(ref) * 2.0 ** -10 + 1e-6)
    pad = got[:, :, case.query:, :]
    assert not pad.size or (np.all(pad == 0) and not np.any(np.signbit(pad)))


@pytest.mark.parametrize("depth", [64, 128, 256])
def test_chunk_probabilities_far_below_the_maximum_are_exact_exponentials(gpu_ctx, depth):
    """Row r of a chunk sees column 0 at a score d_r and its own columns at 0; only column 0 has a
    value, large enough to show its probability e^d_r.  The scores are exact (one product with 1), so
    the output's relative error is that of the exponential (2 ulp), the value's product, the sum's
    reciprocal and the last product: 2^-22 + 3 * 2^-24."""
    rng = np.random.default_rng(depth)
    m = 40
    d = -rng.uniform(0.5, 84.0, size=m).astype(np.float32)
    d[:3] = -83.7, -84.0, -0.5
    q = np.zeros((1, 1, m, depth), dtype=np.float32)
    q[0, 0, :, 0] = d                 # against k = (1, 0, ..): the score is d_r itself
    ins = np.zeros((1, 1, m, depth), dtype=np.float32)
    slot_k = np.zeros((1, 1, 64, depth), dtype=np.float32)
    slot_v = np.zeros((1, 1, 64, depth), dtype=np.float32)
    slot_k[0, 0, 0, 0] = 1.0
    slot_v[0, 0, 0, :] = 1e30
    bufs = [gpu_ctx.upload(a) for a in (q, ins, ins, slot_k, slot_v)]
    out = gpu_ctx.alloc(q.nbytes)
    gpu_ctx.attention_chunk(*bufs, out, batch=1, heads=1, kv_heads=1, chunk_rows=m, depth=depth,
                            capacity=64, window=0, half_scale=1.0, past=1, query=m)
    got = out.download(np.float32, (m, depth)).astype(np.float64)
    p = np.exp(d.astype(np.float64))
    want = (p * np.float32(1e30) / (p + np.arange(1, m + 1)))[:, None]
    error = np.abs(got / want - 1.0).max(axis=1)
    assert error.max() <= 2.0 ** -22 + 3 * 2.0 ** -24, (float(error.max()), float(d[error.argmax()]))
    for b in bufs + [out]:
        b.free()


def test_chunk_scores_that_are_not_finite(gpu_ctx):
    """A NaN among a row's scores makes that row NaN, one at -inf counts as nothing, and rows whose
    differences overflow f32 keep the maximum's value alone."""
    m, depth = 20, 64
    rng = np.random.default_rng(5)
    q = np.zeros((1, 1, m, depth), dtype=np.float32)
    q[0, 0, :, 0] = 1.0
    ins_k = np.zeros((1, 1, m, depth), dtype=np.float32)
    ins_v = rng.normal(size=ins_k.shape).astype(np.float32)
    ins_k[0, 0, 0, 0] = 3e38
    ins_k[0, 0, 1, 0] = -3e38         # a difference of -6e38: -inf
    ins_k[0, 0, 2, 0] = -np.inf
    ins_k[0, 0, 10, 0] = np.nan
    slots = [np.zeros((1, 1, 32, depth), dtype=np.float32) for _ in range(2)]
    bufs = [gpu_ctx.upload(a) for a in (q, ins_k, ins_v, *slots)]
    out = gpu_ctx.alloc(q.nbytes)
    gpu_ctx.attention_chunk(*bufs, out, batch=1, heads=1, kv_heads=1, chunk_rows=m, depth=depth,
                            capacity=32, window=0, half_scale=1.0, past=0, query=m)
    got = out.download(np.float32, (m, depth))
    assert np.array_equal(got[:10], np.repeat(ins_v[0, 0, :1], 10, axis=0))
    assert np.isnan(got[10:]).all()
    for b in bufs + [out]:
        b.free()


@pytest.mark.parametrize("shift", [1, 2, 3, 7])
@pytest.mark.parametrize("past", [3, 300])
def test_decode_takes_this_steps_rows_at_any_element(gpu_ctx, shift, past):
    """ins_k and ins_v need the alignment of an element only: rows that start `shift` elements into
    their buffers give the bits of aligned ones, in both the single and the ragged form."""
    heads, kv_heads, depth, cap = 8, 2, 128, 320
    rng = np.random.default_rng(shift + past)
    half = lambda *s: rng.normal(size=s).astype(np.float16)  # noqa: E731
    q, slot_k, slot_v = half(heads, depth), half(kv_heads, cap, depth), half(kv_heads, cap, depth)
    ins = [half(kv_heads, depth), half(kv_heads, depth)]
    pad = lambda a: np.concatenate([np.full(shift, np.nan, np.float16), a.reshape(-1)])  # noqa: E731
    dq, dk, dv = (gpu_ctx.upload(a) for a in (q, slot_k, slot_v))
    plain = [gpu_ctx.upload(a) for a in ins]
    moved = [gpu_ctx.upload(pad(a)) for a in ins]
    out = gpu_ctx.alloc(q.nbytes)
    ws = gpu_ctx.alloc(max(gpu_ctx.attention_varlen_workspace(1, heads, kv_heads, depth, cap),
                           gpu_ctx.attention_state_workspace(1, heads, kv_heads, 1, depth, 0, cap)))
    scale = oracle.half_scale(depth)
    results = []
    for k, v in (plain, [b.offset(2 * shift) for b in moved]):
        gpu_ctx.attention_state(dq, k, v, dk, dv, out, batch=1, heads=heads, kv_heads=kv_heads,
                                chunk_rows=1, depth=depth, capacity=cap, window=0,
                                half_scale=scale, past=past, query=1, io_dtype=ka.F16,
                                kv_dtype=ka.F16, workspace=ws)
        results.append(out.download(np.uint16, (heads, depth)))
        gpu_ctx.attention_varlen(dq, k, v, dk, dv, out, np.array([0, past], np.int32), heads=heads,
                                 kv_heads=kv_heads, depth=depth, total_rows=cap, half_scale=scale,
                                 io_dtype=ka.F16, kv_dtype=ka.F16, workspace=ws)
        results.append(out.download(np.uint16, (heads, depth)))
    assert np.isfinite(results[0].view(np.float16)).all()
    for other in results[1:]:
        assert np.array_equal(results[0], other)
    for b in [dq, dk, dv, out, ws] + plain + moved:
        b.free()


def attention_in_64_bits(q, k, v, past, scale):
    """One head, no window: rows of q over keys 0 .. past + row."""
    q, k, v = (a.astype(np.float64) for a in (q, k, v))
    out = np.empty_like(q)
    with np.errstate(invalid="ignore"):
        for r in range(q.shape[0]):
            s = (k[:past + r + 1] @ q[r]) * scale * scale
            p = np.exp(s - s.max())
            out[r] = (p[:, None] * v[:past + r + 1]).sum(axis=0) / p.sum()
    return out


def chunk_over_fp16_state(ctx, q, ik, iv, sk, sv, past, scale):
    m, depth = q.shape
    bufs = [ctx.upload(np.ascontiguousarray(a)) for a in (q, ik, iv, sk, sv)]
    out = ctx.zeros(q.nbytes)
    ctx.attention_chunk(*bufs, out, batch=1, heads=1, kv_heads=1, chunk_rows=m, depth=depth,
                        capacity=sk.shape[0], window=0, half_scale=scale, past=past, query=m,
                        io_dtype=ka.dtype_code(q.dtype), kv_dtype=ka.F16)
    return out.download(q.dtype, q.shape)


@pytest.mark.parametrize("depth", [64, 128, 256])
@pytest.mark.parametrize("past", [31, 32, 33, 320])
@pytest.mark.parametrize("io", [np.float32, np.float16])
def test_chunks_over_an_fp16_state_keep_the_bits_of_f32(gpu_ctx, depth, past, io):
    """Blocks of 32 fp16 keys run with fp16 operands (the queries and the probabilities in parts): no
    further from 64 bits than f32 operands are, for rows of 1e4 and of 1e-7 beside ordinary ones and a row
    with entries eight decades apart (a small probability shows where it alone has a value:
    test_small_probabilities_over_an_fp16_state_keep_their_bits).  f32 operands: every product of
    a score is rounded three times, 3 * 2^-24 of sum |q k| scale^2 at most, which moves a probability by
    as much of itself; the rest (exponential, sums over the keys) stays below 2^-20."""
    rng = np.random.default_rng(depth + past)
    m, scale = 18, float(np.float32(np.sqrt(1.0 / np.sqrt(float(depth)))))
    q, ik, iv = (rng.normal(size=(m, depth)).astype(io) for _ in range(3))
    sk, sv = (rng.normal(size=(past + m + 14, depth)).astype(np.float16) for _ in range(2))
    if io == np.float32:
        q[3] *= 1e-7
        q[4, ::2] *= 1e-8
        q[5] *= 1e4
    got = chunk_over_fp16_state(gpu_ctx, q, ik, iv, sk, sv, past, scale)
    k = np.concatenate([sk[:past].astype(io).astype(np.float64), ik.astype(np.float64)])
    v = np.concatenate([sv[:past].astype(np.float64), iv.astype(np.float64)])
    want = attention_in_64_bits(q, k, v, past, scale)
    moved = 3 * 2.0 ** -24 * (np.abs(q.astype(np.float64)) @ np.abs(k).T).max(axis=1) * scale * scale + 2.0 ** -20
    bound = 2 * moved[:, None] * np.abs(v).max() + (2.0 ** -10 * np.abs(want) + 1e-7 if io == np.float16 else 0.0)
    assert np.all(np.abs(got.astype(np.float64) - want) <= bound)
    if io == np.float32:       # ordinary rows: measured 2.0e-7 to 4.3e-7, f32 operands 3.0e-7 to 7.0e-7
        rows = [r for r in range(m) if r not in (3, 4, 5)]
        assert np.linalg.norm(got[rows] - want[rows]) <= 6e-7 * np.linalg.norm(want[rows])


@pytest.mark.parametrize("depth", [64, 128, 256])
@pytest.mark.parametrize("io", [np.float32, np.float16])
def test_infinities_in_an_fp16_state_reach_what_they_reach_in_f32(gpu_ctx, depth, io):
    """A key whose score is -inf has no weight, a value of inf is the infinity of its dim, alone: parts of
    a query or of a probability that are zero (here q of few bits, and the row whose largest probability
    is 1) do not turn either into a NaN."""
    rng = np.random.default_rng(depth)
    past, m, scale = 96, 17, 0.25
    q = np.abs(rng.integers(1, 3, size=(m, depth))).astype(io)
    ik, iv = (rng.normal(size=(m, depth)).astype(io) for _ in range(2))
    sk, sv = (rng.normal(size=(past + m, depth)).astype(np.float16) for _ in range(2))
    sk[40, 5] = -np.inf
    sv[70, 9] = np.inf
    sv[3, 11] = -np.inf
    got = chunk_over_fp16_state(gpu_ctx, q, ik, iv, sk, sv, past, scale)
    k = np.concatenate([sk[:past].astype(np.float64), ik.astype(np.float64)])
    v = np.concatenate([sv[:past].astype(np.float64), iv.astype(np.float64)])
    want = attention_in_64_bits(q, k, v, past, scale)
    assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.isposinf(want[:, 9]).all()
    assert np.array_equal(np.isneginf(got), np.isneginf(want)) and np.isneginf(want[:, 11]).all()
    rest = np.delete(np.arange(depth), (9, 11))
    assert np.all(np.abs(got[:, rest].astype(np.float64) - want[:, rest]) <=
                  1e-5 + (2e-3 if io == np.float16 else 0.0))


@pytest.mark.parametrize("depth", [64, 128, 256])
@pytest.mark.parametrize("past", [8, 40, 96])
@pytest.mark.parametrize("infinite", [False, True])
def test_large_f32_rows_of_a_chunk_beside_an_fp16_state(gpu_ctx, depth, past, infinite):
    """This step's f32 value rows of 1e36 stay finite beside an fp16 state, also where an infinity of the
    state sends the wave over its keys once more.  |v| <= 3e36 over at most 116 keys: no sum reaches
    f32's largest.  The bound is that of f32 operands: a score's product is rounded three times, which moves
    a probability by 3 * 2^-24 of sum |q k| scale^2; exponential and sums stay below 2^-20."""
    rng = np.random.default_rng(depth + past)
    m, scale = 20, float(np.float32(np.sqrt(1.0 / np.sqrt(float(depth)))))
    q, ik = (rng.normal(size=(m, depth)).astype(np.float32) for _ in range(2))
    iv = (np.clip(rng.normal(size=(m, depth)), -3, 3) * 1e36).astype(np.float32)
    sk, sv = (rng.normal(size=(past + m, depth)).astype(np.float16) for _ in range(2))
    if infinite:
        sv[3, 9] = np.inf
    got = chunk_over_fp16_state(gpu_ctx, q, ik, iv, sk, sv, past, scale).astype(np.float64)
    k = np.concatenate([sk[:past].astype(np.float64), ik.astype(np.float64)])
    v = np.concatenate([sv[:past].astype(np.float64), iv.astype(np.float64)])
    want = attention_in_64_bits(q, k, v, past, scale)
    if infinite:
        assert np.isposinf(got[:, 9]).all()
        got, want, v = (np.delete(a, 9, axis=1) for a in (got, want, v))
    moved = 3 * 2.0 ** -24 * (np.abs(q.astype(np.float64)) @ np.abs(k).T).max(axis=1) * scale * scale + 2.0 ** -20
    assert np.all(np.abs(got - want) <= 2 * moved[:, None] * np.abs(v).max())


@pytest.mark.parametrize("depth", [64, 128, 256])
@pytest.mark.parametrize("past", [32, 33, 96])
@pytest.mark.parametrize("lowest", [-11.0, -40.0, -80.0])
@pytest.mark.parametrize("io", [np.float32, np.float16])
def test_small_probabilities_over_an_fp16_state_keep_their_bits(gpu_ctx, depth, past, lowest, io):
    """Eight keys of the state score down to `lowest` under the rest, and each alone has a value in its dim: the
    dim shows that key's probability, however small.  (From 2^-16 = e^-11.1 on a probability is three fp16 parts,
    below that an f32 operand.)  Scores are exact, one product with 1.  Exponentials are within 2^-22 in the
    dim and in the sum, and about 20 sums and products round once each; fp16 results once more."""
    rng = np.random.default_rng(depth + past)
    m = 18
    q = np.zeros((m, depth), dtype=io)
    q[:, :8] = rng.uniform(lowest, -0.5, size=(m, 8)).astype(io)
    q[:, 0] = lowest
    ins = np.zeros((m, depth), dtype=io)
    sk, sv = (np.zeros((past + m, depth), dtype=np.float16) for _ in range(2))
    keys = rng.choice(past, size=8, replace=False)
    sk[keys, np.arange(8)] = 1.0
    sv[keys, np.arange(8)] = 32768.0
    got = chunk_over_fp16_state(gpu_ctx, q, ins, ins, sk, sv, past, 1.0).astype(np.float64)
    p = np.exp(q[:, :8].astype(np.float64))
    want = 32768.0 * p / (p.sum(axis=1) + past - 8 + np.arange(1, m + 1))[:, None]
    bound = (2 * 2.0 ** -22 + 20 * 2.0 ** -24) * want
    if io == np.float16:
        bound = bound + 2.0 ** -11 * want + 2.0 ** -25
    assert np.all(np.abs(got[:, :8] - want) <= bound)
    assert not got[:, 8:].any()


@pytest.mark.parametrize("depth", [64, 128, 256])
@pytest.mark.parametrize("past", [32, 33, 320])
@pytest.mark.parametrize("io", [np.float32, np.float16])
def test_a_row_over_an_fp16_state_has_the_same_bits_beside_a_steep_row(gpu_ctx, depth, past, io):
    """A query whose probabilities are small (its scores spread over hundreds) takes f32 operands for them; the
    rows beside it in a block of sixteen keep their bits."""
    rng = np.random.default_rng(depth + past)
    m, scale = 20, float(np.float32(np.sqrt(1.0 / np.sqrt(float(depth)))))
    q, ik, iv = (rng.normal(size=(m, depth)).astype(io) for _ in range(3))
    sk, sv = (rng.normal(size=(past + m, depth)).astype(np.float16) for _ in range(2))
    q *= io(0.5)
    alone = chunk_over_fp16_state(gpu_ctx, q, ik, iv, sk, sv, past, scale)
    q[5] *= io(100)
    beside = chunk_over_fp16_state(gpu_ctx, q, ik, iv, sk, sv, past, scale)
    rest = np.delete(np.arange(m), 5)
    assert np.isfinite(beside).all() and not np.array_equal(alone[5], beside[5])
    assert alone[rest].tobytes() == beside[rest].tobytes()


@pytest.mark.parametrize("depth", [64, 128, 256])
@pytest.mark.parametrize("past", [32, 33, 320])
@pytest.mark.parametrize("io", [np.float32, np.float16])
@pytest.mark.parametrize("entry", [np.nan, np.inf])
def test_a_row_over_an_fp16_state_has_the_same_bits_beside_a_row_that_is_not_finite(gpu_ctx, depth, past, io, entry):
    """A row whose sums are not finite is formed once more with f32 operands, alone: the rows beside it in a block
    of sixteen keep their bits."""
    rng = np.random.default_rng(depth + past)
    m, scale = 20, float(np.float32(np.sqrt(1.0 / np.sqrt(float(depth)))))
    q, ik, iv = (rng.normal(size=(m, depth)).astype(io) for _ in range(3))
    sk, sv = (rng.normal(size=(past + m, depth)).astype(np.float16) for _ in range(2))
    alone = chunk_over_fp16_state(gpu_ctx, q, ik, iv, sk, sv, past, scale)
    q[5, 3] = io(entry)
    beside = chunk_over_fp16_state(gpu_ctx, q, ik, iv, sk, sv, past, scale)
    rest = np.delete(np.arange(m), 5)
    assert np.isnan(beside[5]).all() and np.isfinite(beside[rest]).all()
    assert alone[rest].tobytes() == beside[rest].tobytes()


@pytest.mark.parametrize("depth", [64, 128, 256])
@pytest.mark.parametrize("past", [32, 96])
@pytest.mark.parametrize("power", [12, 20, 30, 60])
def test_small_entries_of_an_f32_query_over_an_fp16_state_keep_their_bits(gpu_ctx, depth, past, power):
    """An entry of 2^power stands where every key is zero, so that the others decide the scores: they keep the bits
    that f32 operands keep (a product is rounded three times: 3 * 2^-24 of sum |q k|; exponential and sums
    stay below 2^-20).  Down to 2^-36 of the largest they fit three fp16 parts, below that the row takes f32
    operands."""
    rng = np.random.default_rng(depth + past)
    m = 18
    q, ik, iv = (rng.normal(size=(m, depth)).astype(np.float32) for _ in range(3))
    sk, sv = (rng.normal(size=(past + m, depth)).astype(np.float16) for _ in range(2))
    q[::2, 0] = 2.0 ** power
    sk[:, 0] = ik[:, 0] = 0.0
    scale = float(np.float32(np.sqrt(1.0 / np.sqrt(float(depth)))))
    got = chunk_over_fp16_state(gpu_ctx, q, ik, iv, sk, sv, past, scale).astype(np.float64)
    k = np.concatenate([sk[:past].astype(np.float64), ik.astype(np.float64)])
    v = np.concatenate([sv[:past].astype(np.float64), iv.astype(np.float64)])
    want = attention_in_64_bits(q, k, v, past, scale)
    moved = 3 * 2.0 ** -24 * (np.abs(q.astype(np.float64)) @ np.abs(k).T).max(axis=1) * scale * scale + 2.0 ** -20
    assert np.all(np.abs(got - want) <= 2 * moved[:, None] * np.abs(v).max())


@pytest.mark.parametrize("io", [np.float32, np.float16])
@pytest.mark.parametrize("infinite", [False, True])
def test_two_row_blocks_a_workgroup_have_the_bits_of_one_over_an_fp16_state(gpu_ctx, io, infinite):
    """512 heads of 20 rows are workgroups of two blocks of sixteen rows, one head two workgroups: the same bits, also
    for a steep row, a row that is not finite (alone in the second turn) and, with an infinity in the state, rows
    that all take the second turn."""
    rng = np.random.default_rng(int(infinite))
    heads, m, depth, past, scale = 512, 20, 64, 96, 0.5
    q, ik, iv = (rng.normal(size=(m, depth)).astype(io) for _ in range(3))
    sk, sv = (rng.normal(size=(past + m, depth)).astype(np.float16) for _ in range(2))
    q[2] *= io(50)
    q[17] *= io(50)
    q[18, 3] = np.nan
    if infinite:
        sv[40, 9] = np.inf
    one = chunk_over_fp16_state(gpu_ctx, q, ik, iv, sk, sv, past, scale)
    bufs = [gpu_ctx.upload(np.ascontiguousarray(a)) for a in (np.broadcast_to(q, (heads, m, depth)), ik, iv, sk, sv)]
    out = gpu_ctx.zeros(heads * q.nbytes)
    gpu_ctx.attention_chunk(*bufs, out, batch=1, heads=heads, kv_heads=1, chunk_rows=m, depth=depth,
                            capacity=past + m, window=0, half_scale=scale, past=past, query=m,
                            io_dtype=ka.dtype_code(q.dtype), kv_dtype=ka.F16)
    many = out.download(q.dtype, (heads, m, depth))
    finite = np.delete(np.arange(m), 18)
    assert np.isnan(one[18]).all() and np.isnan(many[:, 18]).all()
    assert np.isfinite(one[finite, 9]).any() != infinite  # (a steep row's zero times the infinity is a NaN)
    if infinite:
        one, many = np.delete(one, 9, axis=1), np.delete(many, 9, axis=2)
    assert np.isfinite(one[finite]).all()
    assert all(head[finite].tobytes() == one[finite].tobytes() for head in many)
