"""Performance cases of karume_amd: the calls a program makes of it, over the sizes it serves.

Three kinds of program use this package: one that runs single ops of a graph through the
context (`linear_i4`, `attention_*`, `linear_w4a8_fused`), one that serves several sequences a
step (16-row products, the ragged attention), and one that runs a whole decoder through a
session (a prompt in chunks, a replayed greedy decode, the step-by-step greedy loop).  Sizes are
those of the benchmark configurations and of the default 1.1B-parameter decoder shape; `draw`
spreads over the same ranges, with sizes that are no multiples of a tile among them.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import karume_amd as ka
from karume_amd.decoder import LlamaConfig, LlamaDecoderSession, random_weights

_DTYPES = {"f16": (ka.F16, torch.float16, 2), "f32": (ka.F32, torch.float32, 4)}
_COMPUTE = {"f16": ka.COMPUTE_F16, "f32": ka.COMPUTE_F32}
_MAX_FLOPS = 2 * 512 * 11008 * 4096
_MAX_KV_BYTES = 512 << 20


# ---------------------------------------------------------------------------------- the cases
def _linear(name, m, n, k, group, io, scale, compute, bias=False):
    return {"name": name, "op": "linear", "m": m, "n": n, "k": k, "group": group, "io": io,
            "scale": scale, "compute": compute, "bias": bias}


def _attention(name, op, heads, kv_heads, depth, rows, past, window, io, kv, **more):
    return {"name": name, "op": op, "heads": heads, "kv_heads": kv_heads, "depth": depth,
            "rows": rows, "past": past, "window": window, "io": io, "kv": kv, **more}


def _model(name, op, layers, heads, kv_heads, prompt, chunk, new, kv, compute):
    return {"name": name, "op": op, "layers": layers, "heads": heads, "kv_heads": kv_heads,
            "prompt": prompt, "chunk": chunk, "new": new, "kv": kv, "compute": compute}


def listed():
    return [
        # down-projection of one decode row, the smallest kind of call that a host makes
        _linear("gemv_m1", 1, 4096, 11008, 128, "f16", "f16", "f32"),
        # up-projection of 16 sequences that decode together
        _linear("gemv_m16", 16, 11008, 4096, 128, "f16", "f16", "f32"),
        # up-projection of a 512-row prompt, fp16 activations (benchmark config 1)
        _linear("gemm_up_f16", 512, 11008, 4096, 128, "f16", "f16", "f16"),
        # down-projection of a 512-row prompt in the default arithmetic class: f32 activations
        _linear("gemm_down_f32", 512, 4096, 11008, 128, "f32", "f16", "f32"),
        # a model file's own storage (f32 scales, a bias, small groups) on a prompt of odd length
        _linear("linear_ragged_g32", 77, 3000, 2080, 32, "f32", "f32", "f32", True),
        # one decode row over a long context (benchmark config 2)
        _attention("attention_decode", "attn_decode", 32, 8, 128, 1, 4095, 0, "f16", "f16"),
        # a decode step of 16 sequences of 128 to 4096 cached rows: the step's tables, then the
        # attention of four layers (benchmark config 3)
        _attention("attention_ragged", "attn_ragged", 32, 8, 128, 16, 4096, 0, "f16", "f16", layers=4),
        # a 128-row chunk in the middle of a long prompt, attention and appends to the state
        _attention("attention_chunk", "attn_chunk", 32, 4, 64, 128, 1024, 0, "f32", "f32"),
        # the integer-dot form of the up-projection, quantiser included
        {"name": "w4a8_up", "op": "w4a8", "m": 512, "n": 11008, "k": 4096, "group": 128,
         "scale": "f16", "bias": False},
        # a 300-token prompt of the 1.1B-parameter shape in chunks of 128 (the last one padded),
        # fp16 products and state
        _model("prompt_f16", "model_prompt", 22, 32, 4, 300, 128, 0, "f16", "f16"),
        # 64 tokens of replayed decode behind a 128-token prompt
        _model("decode_replayed", "model_decode", 22, 32, 4, 128, 128, 64, "f32", "f32"),
        # the greedy loop with defaults: a 128-token prompt in f32 arithmetic, then one run and
        # one read-back a token
        _model("greedy_loop", "model_greedy", 22, 32, 4, 128, 128, 32, "f32", "f32"),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw_linear_sizes(rng):
    """m, n, k, group of a projection: up to the multiply-adds of the largest listed one."""
    group = rng.choice((32, 64, 128, 128))
    while True:
        m = _log_int(rng, 1, 512)
        n, k = _log_int(rng, 256, 32000), max(4, _log_int(rng, 512, 11008) // 128) * 128
        if group < 128:
            k += group * rng.randrange(0, 128 // group)
        if 2 * m * n * k <= _MAX_FLOPS:
            return m, n, k, group


def draw(rng):
    op = rng.choice(("linear", "linear", "linear", "attn_decode", "attn_ragged", "attn_chunk", "w4a8",
                     "model_prompt", "model_decode", "model_greedy"))
    if op == "linear":
        m, n, k, group = _draw_linear_sizes(rng)
        case = _linear("", m, n, k, group, rng.choice(("f16", "f32")), rng.choice(("f16", "f32")),
                       rng.choice(("f16", "f32")), rng.random() < 0.3)
    elif op == "w4a8":
        m, n, k, group = _draw_linear_sizes(rng)
        case = {"op": "w4a8", "m": m, "n": n, "k": k, "group": group,
                "scale": rng.choice(("f16", "f32")), "bias": rng.random() < 0.3}
    elif op.startswith("attn"):
        heads, kv_heads, depth = rng.choice(((32, 8, 128), (32, 4, 64), (16, 16, 64), (8, 2, 128),
                                             (8, 1, 256)))
        io, kv = rng.choice((("f16", "f16"), ("f32", "f32"), ("f32", "f16")))
        window = rng.choice((0, 0, 0, 512)) if op != "attn_ragged" else 0
        if op == "attn_decode":
            case = _attention("", op, heads, kv_heads, depth, 1, _log_int(rng, 16, 8191), window,
                              io, kv)
        elif op == "attn_chunk":
            case = _attention("", op, heads, kv_heads, depth, _log_int(rng, 17, 512),
                              rng.choice((0, _log_int(rng, 16, 2048))), window, io, kv)
        else:
            case = _attention("", op, heads, kv_heads, depth, _log_int(rng, 2, 32),
                              _log_int(rng, 256, 4096), 0, io, kv, layers=rng.randrange(1, 5))
            while _kv_bytes(case) > _MAX_KV_BYTES:
                case["past"] //= 2
    else:
        heads, kv_heads = rng.choice(((32, 4), (16, 4), (8, 2)))
        chunk = rng.choice((32, 64, 128))
        layers, prompt = _log_int(rng, 2, 22), _log_int(rng, 8, 300)
        new = {"model_prompt": 0, "model_decode": _log_int(rng, 8, 64),
               "model_greedy": _log_int(rng, 4, 32)}[op]
        case = _model("", op, layers, heads, kv_heads, prompt, chunk, new,
                      rng.choice(("f32", "f16")),
                      rng.choice(("f32", "f16")) if op == "model_prompt" else "f32")
        if op == "model_greedy" and case["prompt"] > 128:
            case["prompt"] = 128
    case.pop("name", None)
    return case


# --------------------------------------------------------------------------------- preparation
_gpu = None
_session = None  # (key, LlamaDecoderSession): a server keeps its model, requests come and go


def _context():
    global _gpu
    if _gpu is None:
        _gpu = ka.acquire_gpu(0)
    return _gpu


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, shape, dtype):
    return torch.randn(shape, generator=gen, device="cuda").to(dtype)


def _int4(gen, n, k, group, scale):
    """Packed codes uniform in [-8, 7] and group scales |N(0, 0.02)|, as a quantiser leaves them."""
    packed = torch.randint(0, 256, (n, k // 2), generator=gen, device="cuda", dtype=torch.uint8)
    scales = torch.randn((n, k // group), generator=gen, device="cuda").mul_(0.02).abs_()
    return packed, scales.clamp_(min=6.104e-05).to(_DTYPES[scale][1])


def _half_scale(depth):
    return float(np.float32(np.sqrt(1.0 / np.sqrt(float(depth)))))


def _ragged_lengths(case, seed):
    """One cached length per sequence, from a thirty-second of the longest to the longest."""
    low = max(1, case["past"] // 32)
    return np.random.default_rng(seed).integers(low, case["past"] + 1, size=case["rows"])


def _prepare_linear(case, seed):
    gen, (_, io, _) = _generator(seed), _DTYPES[case.get("io", "f32")]
    m, n, k = case["m"], case["n"], case["k"]
    packed, scales = _int4(gen, n, k, case["group"], case["scale"])
    state = {"case": case, "gpu": _context(), "w": packed, "s": scales,
             "x": _normal(gen, (m, k), io), "bias": None,
             "out": torch.empty((m, n), dtype=io, device="cuda")}
    if case["bias"]:
        state["bias"] = _normal(gen, (n,), io)
    if case["op"] == "w4a8":
        state["xq"] = torch.empty((m, k), dtype=torch.int8, device="cuda")
        state["xs"] = torch.empty((m,), dtype=torch.float32, device="cuda")
    return state


def _prepare_attention(case, seed):
    gen, gpu = _generator(seed), _context()
    (io_code, io, _), (kv_code, kv, _) = _DTYPES[case["io"]], _DTYPES[case["kv"]]
    h, hkv, d, rows = case["heads"], case["kv_heads"], case["depth"], case["rows"]
    state = {"case": case, "gpu": gpu}
    if case["op"] == "attn_ragged":
        lengths = _ragged_lengths(case, seed)
        cu = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
        total = int(cu[-1])
        shape = dict(nseq=rows, depth=d, kv_dtype=kv_code, total_rows=total)
        splits = gpu.attention_varlen_max_splits(rows, d, kv_code, total)
        state.update(
            layers=[(_normal(gen, (rows, h, d), io), _normal(gen, (rows, hkv, d), io),
                     _normal(gen, (rows, hkv, d), io), _normal(gen, (hkv, total, d), kv),
                     _normal(gen, (hkv, total, d), kv),
                     torch.empty((rows, h, d), dtype=io, device="cuda"))
                    for _ in range(case["layers"])],
            cu=torch.from_numpy(cu).cuda(), shape=dict(shape, max_splits=splits),
            plan=torch.empty(gpu.attention_varlen_plan_bytes(rows), dtype=torch.uint8,
                             device="cuda"),
            ws=torch.empty(gpu.attention_varlen_workspace(rows, h, hkv, d, total),
                           dtype=torch.uint8, device="cuda"),
            kw=dict(heads=h, kv_heads=hkv, half_scale=_half_scale(d), io_dtype=io_code))
        return state
    window, past = case["window"], case["past"]
    capacity = window if window else (past + rows + 127) // 128 * 128
    state.update(
        q=_normal(gen, (h, rows, d), io), k=_normal(gen, (hkv, rows, d), io),
        v=_normal(gen, (hkv, rows, d), io), slot_k=_normal(gen, (hkv, capacity, d), kv),
        slot_v=_normal(gen, (hkv, capacity, d), kv),
        out=torch.empty((rows, h, d) if case["op"] == "attn_chunk" else (h, rows, d), dtype=io,
                        device="cuda"),
        kw=dict(batch=1, heads=h, kv_heads=hkv, chunk_rows=rows, depth=d, capacity=capacity,
                window=window, half_scale=_half_scale(d), past=past, query=rows,
                io_dtype=io_code, kv_dtype=kv_code))
    if case["op"] == "attn_decode":
        need = gpu.attention_state_workspace(1, h, hkv, rows, d, window, past)
        state["ws"] = torch.empty(max(16, need), dtype=torch.uint8, device="cuda")
    return state


class _Context:
    """A generation context that is disposed when nothing looks at its state any more."""

    def __init__(self, context):
        self.context = context

    def __del__(self):
        if not self.context.disposed:
            self.context.dispose()


class _Borrowed:
    """A device buffer of the package as something torch can view; keeps its owner."""

    def __init__(self, owner, buffer, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "version": 2,
                                         "data": (buffer.address, False)}


class _Request:
    """One request on the kept session: its prompt and the context with its state."""

    def __init__(self, case, seed):
        self.case = case
        self.session = _kept_session(case)
        config = self.session.config
        self.prompt = np.random.default_rng(seed).integers(
            0, config.vocab, size=case["prompt"]).astype(np.int32)
        self.context, self.slots, self.token = None, [], 0
        if case["op"] == "model_greedy":
            return
        self.context = self.session.create_generation_context(
            capacity=config.max_position, chunk_length=case["chunk"])
        owner = _Context(self.context)
        shape = (config.kv_heads, config.max_position, config.head_dim)
        kind = "<f2" if case["kv"] == "f16" else "<f4"
        self.slots = [torch.as_tensor(_Borrowed(owner, b, shape, kind), device="cuda")
                      for b in self.context.slots_k + self.context.slots_v]
        if case["op"] == "model_decode":
            self.token = int(self.prefill()[0, 0, 0])

    def prefill(self):
        c = self.case["chunk"]
        for piece in ka.plan_prefill_chunks(len(self.prompt), c):
            n = piece.query_length
            ids, pos = np.zeros((1, c), dtype=np.int32), np.zeros((1, c), dtype=np.int32)
            ids[0, :n] = self.prompt[piece.position:piece.position + n]
            pos[0, :n] = np.arange(piece.position, piece.position + n)
            token = self.session.run(ids, pos, n - 1, context=self.context, query_length=n)
        return token


def _config(case):
    d = case["heads"] * 64
    return LlamaConfig(layers=case["layers"], d_model=d, ffn=d * 11 // 4, heads=case["heads"],
                       kv_heads=case["kv_heads"])


def _kept_session(case):
    """The model is the program's own and outlives its requests: its weights do not depend on a
    request's seed."""
    global _session
    key = tuple(case[name] for name in ("layers", "heads", "kv_heads", "chunk", "kv", "compute"))
    if _session is None or _session[0] != key:
        if _session is not None:
            _session[1].close()
            _session = None
        # f32 activations: with scales of this size the residual stream leaves the fp16 range
        session = LlamaDecoderSession(_context(), random_weights(_config(case), seed=4),
                                      io_dtype=ka.F32, kv_dtype=_DTYPES[case["kv"]][0],
                                      chunk_length=case["chunk"],
                                      prefill_compute=_COMPUTE[case["compute"]])
        _session = (key, session)
    return _session[1]


def prepare(case, seed):
    if case["op"] in ("linear", "w4a8"):
        return _prepare_linear(case, seed)
    if case["op"].startswith("attn"):
        return _prepare_attention(case, seed)
    return _Request(case, seed)


# ------------------------------------------------------------------------------------- one pass
def run(state):
    if isinstance(state, _Request):
        return _run_request(state)
    case, gpu = state["case"], state["gpu"]
    if case["op"] == "linear":
        bias = state["bias"]
        gpu.linear_i4(state["x"].data_ptr(), state["w"].data_ptr(), state["s"].data_ptr(),
                      None if bias is None else bias.data_ptr(), state["out"].data_ptr(),
                      case["m"], case["n"], case["k"], case["group"], _DTYPES[case["io"]][0],
                      _DTYPES[case["scale"]][0], _COMPUTE[case["compute"]])
        return state["out"]
    if case["op"] == "w4a8":
        bias = state["bias"]
        gpu.linear_w4a8_fused(state["x"].data_ptr(), state["w"].data_ptr(), state["s"].data_ptr(),
                              None if bias is None else bias.data_ptr(), state["out"].data_ptr(),
                              case["m"], case["n"], case["k"], case["group"],
                              _DTYPES[case["scale"]][0], xq_i8=state["xq"].data_ptr(),
                              xs_f32=state["xs"].data_ptr())
        return state["out"]
    if case["op"] == "attn_ragged":
        plan, ws = state["plan"].data_ptr(), state["ws"]
        gpu.attention_varlen_plan(state["cu"].data_ptr(), plan, **state["shape"])
        for q, k, v, slot_k, slot_v, out in state["layers"]:
            gpu.attention_varlen_planned(q.data_ptr(), k.data_ptr(), v.data_ptr(),
                                         slot_k.data_ptr(), slot_v.data_ptr(), out.data_ptr(),
                                         plan, workspace=ws.data_ptr(), workspace_bytes=ws.numel(),
                                         **state["shape"], **state["kw"])
        return [layer[5] for layer in state["layers"]]
    buffers = [state[name].data_ptr() for name in ("q", "k", "v", "slot_k", "slot_v", "out")]
    if case["op"] == "attn_decode":
        ws = state["ws"]
        gpu.attention_state(*buffers, workspace=ws.data_ptr(), workspace_bytes=ws.numel(),
                            **state["kw"])
        return state["out"]
    # (without a window the chunk's keys and values are appended by the same call)
    gpu.attention_chunk(*buffers, row_major=True, append=case["window"] == 0, **state["kw"])
    if case["window"]:
        return state["out"]
    return [state["out"], state["slot_k"], state["slot_v"]]


def _run_request(request):
    case = request.case
    if case["op"] == "model_greedy":
        tokens = ka.generate_greedy(request.session, prompt=[int(t) for t in request.prompt],
                                    max_new_tokens=case["new"], chunk_length=case["chunk"],
                                    max_position=request.session.config.max_position)
        return np.array(tokens, dtype=np.int32)
    if case["op"] == "model_prompt":
        request.context.rewind(0)
        return [request.prefill()] + request.slots
    request.context.rewind(case["prompt"])
    tokens = request.session.decode_tokens(request.context, request.token, case["new"])
    return [np.array(tokens, dtype=np.int32)] + request.slots


# -------------------------------------------------------------------------- work and tolerance
def _attended(case):
    """(columns read, columns summed over the rows) of one attention call."""
    rows, past, window = case["rows"], case["past"], case["window"]
    seen = [min(past + r + 1, window) if window else past + r + 1 for r in range(rows)]
    return min(past, window - 1 if window else past) + rows, sum(seen)


def _kv_bytes(case):
    """Mean state bytes of a ragged step."""
    mean = (max(1, case["past"] // 32) + case["past"]) / 2
    return (case["layers"] * case["rows"] * mean * 2 * case["kv_heads"] * case["depth"]
            * _DTYPES[case["kv"]][2])


def work(case):
    op = case["op"]
    if op in ("linear", "w4a8"):
        m, n, k = case["m"], case["n"], case["k"]
        eb = _DTYPES[case.get("io", "f32")][2]
        size = (n * k // 2 + n * (k // case["group"]) * _DTYPES[case["scale"]][2]
                + (m * k + m * n + (n if case["bias"] else 0)) * eb)
        return {"bytes": size, "flops": 2 * m * n * k}
    if op.startswith("attn"):
        h, hkv, d, rows = case["heads"], case["kv_heads"], case["depth"], case["rows"]
        eb, kb = _DTYPES[case["io"]][2], _DTYPES[case["kv"]][2]
        if op == "attn_ragged":
            io = case["layers"] * rows * (2 * h + 2 * hkv) * d * eb
            return {"bytes": int(_kv_bytes(case)) + io,
                    "flops": int(4 * h * _kv_bytes(case) / (2 * hkv * kb))}
        columns, pairs = _attended(case)
        size = 2 * hkv * (columns - rows) * d * kb + rows * (2 * h + 2 * hkv) * d * eb
        if op == "attn_chunk" and not case["window"]:
            size += 2 * hkv * rows * d * kb
        return {"bytes": size, "flops": 4 * h * d * pairs}
    c = _config(case)
    kv_row = 2 * c.kv_heads * c.head_dim
    layer = (c.d_model * (2 * c.d_model + kv_row) + 3 * c.d_model * c.ffn)
    weight = lambda codes: codes // 2 + codes // c.group_size * 2  # noqa: E731
    head = c.vocab * c.d_model
    kb = _DTYPES[case["kv"]][2]
    size = flops = 0
    if op in ("model_prompt", "model_greedy"):
        for piece in ka.plan_prefill_chunks(case["prompt"], case["chunk"]):
            seen = piece.position + piece.query_length
            size += weight(layer) * c.layers + seen * kv_row * kb * c.layers + weight(head)
            flops += c.layers * piece.query_length * (2 * layer + 2 * seen * 2 * c.d_model) + 2 * head
    for step in range(case["new"] if op == "model_decode" else case["new"] - 1):
        seen = case["prompt"] + step + 1
        size += weight(layer) * c.layers + weight(head) + seen * kv_row * kb * c.layers
        flops += c.layers * (2 * layer + 2 * seen * 2 * c.d_model) + 2 * head
    return {"bytes": size, "flops": flops}


def tolerance(case):
    op = case["op"]
    if op == "w4a8":
        return "exact"  # integer sums, then f32 operations in a fixed order
    if op == "linear":
        # fp16 results, fp16 activations or (small groups in that class) fp16 weights against
        # f32 sums of exact products
        half = case["io"] == "f16" or (case["compute"] == "f16" and case["m"] > 16)
        return {"rel": 1e-3 if half else 1e-5}
    if op.startswith("attn"):
        return {"rel": 1e-3 if case["io"] == "f16" else 1e-5}
    if op == "model_greedy":
        return "exact"  # whole tokens
    # the state behind a chain of 22 layers: f32 sums in another order, or fp16 roundings
    half = case["kv"] == "f16" or case["compute"] == "f16"
    return {"rel": 1e-3 if half else 2e-5}
