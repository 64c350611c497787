"""The work a program has this library do, as cases to time: what a local model runtime asks of it between
loading a model and answering - read the weights, read the prompt, write tokens, import new tensors - over the
sizes, row counts, types and modes that the entry points take.

`kind` says which entry points a case goes through:
  step     a node list as a decoder walks it (plan_many / matmul_many): per layer norm + q/k/v, o + residual,
           norm + gate/up with SwiGLU, down + residual, each layer reading the residual stream of the one before
           it.  Attention itself is not part of the library: o_proj reads an input of its own.
  linear   one node (matmul, matmul_ex, matmul_norm)
  import   f32 tensor -> quantize -> weight_from_device -> dequant (what the import stage checks its output with)
  load     a .model container on disk -> load_into -> dequant of every tensor, replacing the model loaded before
"""
import os
import tempfile

import torch

from cyb_amd import Backend, container, formats, stack

TYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
SIZE = {"f16": 2, "bf16": 2, "f32": 4}

_backends = {}


def _backend(mode):
    """One context per numeric mode for the life of the process, as a runtime keeps it."""
    if mode not in _backends:
        torch.cuda.init()
        be = Backend(0)
        if mode == "exact":
            be.set_prefill_mode("exact")
            be.set_decode_mode("exact")
        _backends[mode] = be
    return _backends[mode]


def _step(**kw):
    return dict({"kind": "step", "bits": 4, "layers": 32, "hidden": 4096, "qkv": 6144, "ffn": 14336, "rows": 1, "act": "f16"}, **kw)


def _linear(**kw):
    return dict({"kind": "linear", "bits": 4, "N": 4096, "K": 4096, "rows": 1, "x": "f16", "y": "f32", "mode": "fast",
                 "norm": False, "epilogue": "none"}, **kw)


def listed():
    return [
        # one token of one conversation through all linears of an 8B-class model: what the user waits for, per token
        _step(name="token"),
        # the same step for eight conversations at once
        _step(name="token_batch_8", rows=8),
        # a full 512-token chunk of a prompt being read
        _step(name="prompt_chunk_512", rows=512, act="bf16"),
        # what is left of a prompt after its full chunks, or a short question: an odd number of rows
        _step(name="prompt_tail_45", rows=45, act="bf16"),
        # the smallest linear of that model, called by itself by a runtime that walks its own graph: latency
        _linear(name="kv_proj_row", N=1024),
        # a small Q8 model on f32 activations, as a CPU-style runtime hands them over
        _linear(name="q8_row_f32", bits=8, N=2048, K=2048, x="f32"),
        # the output head: the largest tensor, once per token
        _linear(name="lm_head_row", N=128256),
        # drafted tokens checked in one go on a model of odd sizes: Q8, 27 rows, a vocabulary that no tile divides
        _linear(name="draft_rows_27_odd", bits=8, N=32003, K=2560, rows=27),
        # a prompt chunk where the caller asked for the operands the CPU path has (exact mode)
        _linear(name="exact_chunk_256", N=14336, rows=256, x="bf16", mode="exact"),
        # a long prompt in one call on a Q8 down projection, bf16 in and out
        _linear(name="prompt_2048_q8_down", bits=8, N=4096, K=14336, rows=2048, x="bf16", y="bf16"),
        # one tensor of a model being imported
        {"name": "import_tensor", "kind": "import", "bits": 4, "N": 14336, "K": 4096},
        # switching to another model: the file's tensors of one layer, Q4 blocks, page cache warm
        {"name": "load_layer", "kind": "load", "bits": 4, "layout": "block_aos", "hidden": 4096, "kv": 1024, "ffn": 14336},
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` between lo and hi, even over the logarithm."""
    v = lo * (hi / lo) ** rng.random()
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["step", "step", "rows", "rows", "prompt", "prompt", "exact", "import", "load"])
    bits = rng.choice([4, 4, 8])
    if kind == "step":
        rows = rng.choice([1, 1, rng.randint(2, 16), _log(rng, 17, 512)])
        hidden = _log(rng, 1024, 4096, 128)
        return _step(bits=bits, layers=rng.randint(4, 16), hidden=hidden, qkv=_log(rng, hidden, 2 * hidden, 64),
                     ffn=_log(rng, 2 * hidden, 14336, 64), rows=rows, act="f16" if rows <= 16 else "bf16")
    if kind == "import":
        return {"kind": "import", "bits": bits, "N": _log(rng, 512, 16384), "K": _log(rng, 512, 14336, 32)}
    if kind == "load":
        hidden = _log(rng, 512, 4096, 64)
        return {"kind": "load", "bits": bits, "layout": rng.choice(["block_aos", "planar"]), "hidden": hidden,
                "kv": _log(rng, 128, 1024, 16), "ffn": _log(rng, 1024, 8192, 32)}
    K = _log(rng, 256, 14336, 32)
    c = _linear(bits=bits, K=K, N=_log(rng, 256, 32768), y=rng.choice(["f32", "f32", "f16", "bf16"]))
    if kind == "rows":              # decode: one row, a batch, a draft
        c.update(rows=rng.choice([1, 1, 2, rng.randint(3, 16), rng.randint(17, 32)]), x=rng.choice(["f16", "f16", "bf16", "f32"]),
                 mode=rng.choice(["fast", "fast", "fast", "exact"]))
    elif kind == "prompt":
        c.update(rows=_log(rng, 33, 2048), x=rng.choice(["bf16", "bf16", "f16", "f32"]))
    else:
        c.update(rows=_log(rng, 33, 512), x=rng.choice(["bf16", "f16", "f32"]), mode="exact")
    extra = rng.choice(["none", "none", "norm", "add", "swiglu"])
    c["norm"] = extra == "norm"
    if extra == "add":
        c["epilogue"] = "add"
    elif extra == "swiglu":
        c.update(epilogue="swiglu", N=max(32, c["N"] // 32 * 32))
    return c


# ---- inputs -------------------------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed & 0x7FFFFFFF)
    return g


def _randn(g, shape, dtype=torch.float32, std=1.0):
    return torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, std, generator=g).to(dtype)


def _packed(be, g, bits, N, K):
    """N(0, 0.02) weights quantised on the device: (q plane, scales) in the PLANAR layout."""
    w = _randn(g, (N, K), std=0.02)
    q = torch.empty(N * K * bits // 8, dtype=torch.uint8, device="cuda")
    s = torch.empty(N * (K // 32), dtype=torch.int16, device="cuda")
    be.quantize(bits, w, N, K, q, s)
    return q, s


def _weight(be, g, bits, N, K):
    q, s = _packed(be, g, bits, N, K)
    w = be.weight_from_device(bits, N, K, q, s)
    torch.cuda.synchronize()
    return w


def _blocks(q, s, bits, N, K):
    """PLANAR device buffers -> the container's block form (f16 scale, then 16 or 32 bytes per group)."""
    if bits == formats.Q8:
        body = q.view(-1, 32)
    else:
        b = q.view(-1, 16)                                   # byte j holds weights 2j and 2j + 1, as signed nibbles
        u = torch.stack([b & 15, b >> 4], dim=2).reshape(-1, 32) ^ 8
        body = u[:, :16] | (u[:, 16:] << 4)
    return torch.cat([s.view(torch.uint8).view(-1, 2), body], dim=1).reshape(-1)


def _prepare_step(case, seed):
    be = _backend("fast")
    L, H, F, M, dt = case["layers"], case["hidden"], case["ffn"], case["rows"], TYPES[case["act"]]
    shapes = {"qkv_proj": (H, case["qkv"]), "o_proj": (H, H), "gate_up_proj": (H, 2 * F), "down_proj": (F, H)}
    st = stack.build(be, layers=L, bits=case["bits"], seed=seed, shapes=shapes, order=list(shapes), epilogues=True, norms=True)
    be.weights.clear()                                       # (the stack owns them)
    g = _gen(seed)
    first, attn = _randn(g, (M, H), dt), _randn(g, (L, M, H), dt)
    out = {"qkv": torch.empty((L, M, case["qkv"]), dtype=dt, device="cuda"), "mid": torch.empty((L, M, H), dtype=dt, device="cuda"),
           "act": torch.empty((L, M, F), dtype=dt, device="cuda"), "res": torch.empty((L, M, H), dtype=dt, device="cuda")}
    xs, ys, residuals = [], [], []
    for i in range(L):
        h = first if i == 0 else out["res"][i - 1]
        xs += [h, attn[i], out["mid"][i], out["act"][i]]
        ys += [out["qkv"][i], out["mid"][i], out["act"][i], out["res"][i]]
        residuals += [None, h, None, out["mid"][i]]
    plan = be.plan_many(st.weights, xs, ys, st.epilogues, residuals, gammas=st.gammas, eps=st.eps)
    return {"be": be, "plan": plan, "rows": M, "out": out}


def _prepare_linear(case, seed):
    be, g = _backend(case["mode"]), _gen(seed)
    N, K, M = case["N"], case["K"], case["rows"]
    cols = N
    if case["epilogue"] == "swiglu":
        cols = N // 2
        gate, up = _weight(be, g, case["bits"], cols, K), _weight(be, g, case["bits"], cols, K)
        w = be.fuse_pairs(gate, up)
    else:
        w = _weight(be, g, case["bits"], N, K)
    return {"be": be, "w": w, "x": _randn(g, (M, K), TYPES[case["x"]]), "y": torch.empty((M, cols), dtype=TYPES[case["y"]], device="cuda"),
            "gamma": (1.0 + 0.1 * _randn(g, (K,))).to(torch.float16) if case["norm"] else None, "epilogue": case["epilogue"],
            "residual": _randn(g, (M, N), TYPES[case["y"]]) if case["epilogue"] == "add" else None}


def _prepare_import(case, seed):
    be, N, K, bits = _backend("fast"), case["N"], case["K"], case["bits"]
    return {"be": be, "bits": bits, "N": N, "K": K, "src": _randn(_gen(seed), (N, K), std=0.02),
            "q": torch.empty(N * K * bits // 8, dtype=torch.uint8, device="cuda"),
            "scales": torch.empty(N * (K // 32), dtype=torch.int16, device="cuda"),
            "check": torch.empty((N, K), dtype=torch.float32, device="cuda")}


def _tensors(case):
    H, F = case["hidden"], case["ffn"]
    return {"q_proj": (H, H), "k_proj": (case["kv"], H), "v_proj": (case["kv"], H), "o_proj": (H, H), "gate_proj": (F, H),
            "up_proj": (F, H), "down_proj": (H, F)}


def _prepare_load(case, seed):
    be, g, bits = _backend("fast"), _gen(seed), case["bits"]
    entries, check = [], {}
    for lin, (N, K) in _tensors(case).items():
        q, s = _packed(be, g, bits, N, K)
        e = {"name": stack.tensor_name(0, lin), "bits": bits, "layout": case["layout"], "shape": (N, K), "scales": b""}
        if case["layout"] == "planar":
            e.update(payload=q.cpu().numpy().tobytes(), scales=s.cpu().numpy().tobytes())
        else:
            e["payload"] = _blocks(q, s, bits, N, K).cpu().numpy().tobytes()
        entries.append(e)
        check[e["name"]] = torch.empty((N, K), dtype=torch.float32, device="cuda")
    folder = tempfile.TemporaryDirectory(prefix="cyb_model_")
    path = os.path.join(folder.name, "layer.model")
    container.write_container(path, "layer", "", entries)
    return {"be": be, "folder": folder, "path": path, "check": check}


def prepare(case, seed):
    return {"kind": case["kind"], **{"step": _prepare_step, "linear": _prepare_linear, "import": _prepare_import,
                                     "load": _prepare_load}[case["kind"]](case, seed)}


def run(state):
    be, kind = state["be"], state["kind"]
    if kind == "step":
        be.matmul_many(state["plan"], state["rows"])
        return state["out"]
    if kind == "linear":
        w, x, y = state["w"], state["x"], state["y"]
        if state["gamma"] is not None:
            be.matmul_norm(w, x, state["gamma"], 1e-5, y, state["epilogue"], state["residual"])
        elif state["epilogue"] != "none":
            be.matmul_ex(w, x, y, state["epilogue"], state["residual"])
        else:
            be.matmul(w, x, y)
        return y
    if kind == "import":
        bits, N, K = state["bits"], state["N"], state["K"]
        be.quantize(bits, state["src"], N, K, state["q"], state["scales"])
        w = be.weight_from_device(bits, N, K, state["q"], state["scales"])
        be.dequant(w, state["check"])
        w.free()
        return [state["q"], state["scales"], state["check"]]
    container.load_into(be, state["path"])
    for name, out in state["check"].items():
        be.dequant(be.weights[name], out)
    return state["check"]


# ---- what a pass cannot do without ----------------------------------------------------------------------------

def work(case):
    kind, bits = case["kind"], case["bits"]
    if kind == "step":
        L, H, Q, F, M = case["layers"], case["hidden"], case["qkv"], case["ffn"], case["rows"]
        weights = sum(formats.weight_bytes(bits, n, k) for n, k in ((Q, H), (H, H), (2 * F, H), (H, F)))
        # per layer: the attention output read, q/k/v, both residuals and the activations written (what one node
        # writes and a later one reads is counted once, as an output); gammas
        acts = M * (H + Q + 2 * H + F) * 2 + 2 * H * 2
        return {"bytes": L * (weights + acts) + M * H * 2, "flops": L * 2 * M * (Q * H + H * H + 2 * F * H + H * F)}
    if kind == "linear":
        N, K, M = case["N"], case["K"], case["rows"]
        cols = N // 2 if case["epilogue"] == "swiglu" else N
        b = formats.weight_bytes(bits, N, K) + M * K * SIZE[case["x"]] + M * cols * SIZE[case["y"]] * (2 if case["epilogue"] == "add" else 1)
        return {"bytes": b + (2 * K if case["norm"] else 0), "flops": 2 * M * N * K}
    if kind == "import":                                     # f32 in, packed tensor and its dequantised values out
        N, K = case["N"], case["K"]
        return {"bytes": 8 * N * K + formats.weight_bytes(bits, N, K), "flops": 0}
    shapes = _tensors(case).values()                         # the file in, the resident weights and the values out
    return {"bytes": sum(2 * formats.weight_bytes(bits, n, k) + 4 * n * k for n, k in shapes), "flops": 0}


def tolerance(case):
    if case["kind"] in ("import", "load"):
        return "exact"
    if case["kind"] == "step":                               # 16-bit activations between the nodes of a chain
        return {"rel": 1e-2 if case["act"] == "bf16" else 3e-3}
    r = {"f32": 0.0, "f16": 5e-4, "bf16": 4e-3}[case["y"]]   # one rounding of the result
    if case["norm"] or case["epilogue"] == "swiglu":         # x * gamma is rounded to the operand type
        r += {"f32": 1e-5, "f16": 3e-4, "bf16": 2.5e-3}[case["x"]]
    fast = case["mode"] == "fast" and (case["rows"] > 32 or (case["rows"] > 16 and (case["x"] == "f32" or case["norm"])))
    return {"rel": r + (5e-4 if fast else 1e-5)}             # fast prefill rounds scale * q (and f32 rows) to f16 once
