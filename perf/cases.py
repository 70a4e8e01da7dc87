"""The work that a user of this framework has it do, as measurable cases.

Every case goes through the public entry points (the C ABI of include/*.h by way of the
ctypes bindings) as a user's program calls them: a linear layer's synchronous call with
its copies, multi-row jobs on device buffers, prepared and fused batches, and the model
engine's prefill, decode and classify calls.

  listed()          the named cases
  draw(rng)         one more case of the same ranges
  prepare(case, s)  what a program holds before the call (device, matrices, buffers, batches,
                    model and context), its inputs made from seed s
  run(state)        one pass; the outputs
  work(case)        bytes and operations the pass cannot do without
  tolerance(case)   every result is pinned bit for bit by the API (quantisation, group dots and
                    the order of every FP32 sum), so two correct implementations agree exactly
  exact(case, s)    the same results with the sums in 64 bits, in plain torch

Distributions: sign bits uniform, fp16 scales U[0.01, 0.1), int8 rows uniform in [-127, 127],
FP32 rows N(0, 1) with one value in a thousand 20 times larger (activation outliers).
"""
from __future__ import annotations

import importlib.util
import math
import os
import sys
import tempfile
from pathlib import Path

import numpy as np
import torch

ROOT = Path(os.getcwd())


def _package():
    name = "bnn_train_infer_amd"
    if name not in sys.modules:
        home = ROOT / "bnn-train-infer_amd"
        spec = importlib.util.spec_from_file_location(name, home / "__init__.py",
                                                      submodule_search_locations=[str(home)])
        module = importlib.util.module_from_spec(spec)
        sys.modules[name] = module
        spec.loader.exec_module(module)
    return sys.modules[name]


pkg = _package()
api, engine, gguf = pkg.api, pkg.engine, pkg.gguf

# Whole decoder (28 layers of width 2048, FFN 6144, 16 heads of 128 over 8 key/value heads,
# vocabulary 151669) and a block of it: two layers under a small vocabulary.
MODELS = {"whole": {"layers": 28, "vocab": 151669}, "block": {"layers": 2, "vocab": 8192}}
HIDDEN, FFN, HEADS, KV_HEADS, HEAD_DIM = 2048, 6144, 16, 8, 128
KV = KV_HEADS * HEAD_DIM
MLP_DIMS, MLP_PIXELS = (896, 512, 512, 10), 784
MAX_CONTEXT = 4096


def listed():
    return [
        # one linear layer of a decode step in the reference engine's call pattern (write the row,
        # execute, read the result): the k/v projection, the smallest call, all latency
        {"name": "call_gemv_f32_2048x1024", "kind": "call", "op": "GEMV_F32", "k": 2048, "n": 1024},
        # group dots of a handful of rows with odd sizes (accelerator bring-up and checking)
        {"name": "rows_dot_896x1000_r37", "kind": "rows", "op": "DOT_GROUPS", "k": 896, "n": 1000, "rows": 37},
        # gate/up projection of a 64-token prompt, rows resident on the device
        {"name": "rows_gemm_f32_2048x6144_r64", "kind": "rows", "op": "GEMM_F32", "k": 2048, "n": 6144, "rows": 64},
        # a ragged prompt through the vocabulary's last chunk (151669 - 18 x 8192 outputs)
        {"name": "rows_gemm_f32_2048x4213_r250", "kind": "rows", "op": "GEMM_F32", "k": 2048, "n": 4213, "rows": 250},
        # down projection of a large int8 batch, throughput
        {"name": "rows_gemm_i8_6144x2048_r1024", "kind": "rows", "op": "GEMM", "k": 6144, "n": 2048, "rows": 1024},
        # many independent resident layers in one prepared launch: a weight stream from HBM
        {"name": "batch_gemv_f32_2048x6144_j256", "kind": "batch", "k": 2048, "n": 6144, "jobs": 256, "rows": 1},
        # q, k and v projections of a 48-token prompt as one prepared batch
        {"name": "batch_qkv_r48", "kind": "qkv", "rows": 48},
        # the feed-forward block of one generated token: two fused launches on resident rows
        {"name": "ffn_2048x6144", "kind": "ffn", "k": 2048, "n": 6144},
        # one generated token early in a conversation, whole model
        {"name": "decode_whole_ctx64", "kind": "decode", "model": "whole", "context": 64},
        # one generated token deep in a conversation: attention over a long cache, two layers
        {"name": "decode_block_ctx3000", "kind": "decode", "model": "block", "context": 3000},
        # a prompt of ragged length in one call, whole model
        {"name": "prefill_whole_t389", "kind": "prefill", "model": "whole", "tokens": 389},
        # one classify call of the small classifier's benchmark: 64 samples from host memory
        {"name": "classify_r64", "kind": "classify", "rows": 64},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["call", "rows", "rows", "batch", "qkv", "ffn", "decode", "prefill", "classify"])
    if kind == "call":
        return {"kind": kind, "op": rng.choice(["GEMV_F32", "GEMV_F32", "GEMV", "DOT_GROUPS"]),
                "k": 128 * _log_int(rng, 3, 64), "n": _log_int(rng, 64, 8192)}
    if kind == "rows":
        op = rng.choice(["GEMM_F32", "GEMM_F32", "GEMM", "DOT_GROUPS"])
        k, n = 128 * _log_int(rng, 3, 64), _log_int(rng, 64, 8192)
        most = 1024 if op != "DOT_GROUPS" else max(2, min(1024, (64 << 20) // (2 * n * (k // 128))))
        return {"kind": kind, "op": op, "k": k, "n": n, "rows": _log_int(rng, 2, most)}
    if kind == "batch":
        rows = _log_int(rng, 1, 64) if rng.random() < 0.5 else 1
        k, n = 128 * _log_int(rng, 8, 48), _log_int(rng, 500, 6144)
        most = min(256, 256 * 2048 * 6144 // (k * n)) if rows == 1 else 8
        return {"kind": kind, "k": k, "n": n, "jobs": _log_int(rng, 1, most), "rows": rows}
    if kind == "qkv":
        return {"kind": kind, "rows": _log_int(rng, 1, 512)}
    if kind == "ffn":
        return {"kind": kind, "k": 128 * _log_int(rng, 2, 24), "n": 128 * _log_int(rng, 4, 48)}
    if kind == "decode":
        return {"kind": kind, "model": "block", "context": _log_int(rng, 16, 3000)}
    if kind == "prefill":
        if rng.random() < 0.5:
            return {"kind": kind, "model": "whole", "tokens": _log_int(rng, 8, 388)}
        return {"kind": kind, "model": "block", "tokens": _log_int(rng, 16, 1500)}
    return {"kind": kind, "rows": _log_int(rng, 1, 1000)}


# ---------------------------------------------------------------------------- inputs


def _rng(seed, stream):
    return np.random.default_rng([int(seed) & 0xFFFFFFFF, stream])


def _bits(rng, n, k):
    return np.frombuffer(rng.bytes(n * (k // 8)), np.uint8).reshape(n, k // 8)


def _matrix(rng, n, k):
    return _bits(rng, n, k), rng.uniform(0.01, 0.1, (n, k // 128)).astype(np.float16)


def _f32_rows(rng, rows, k):
    x = rng.standard_normal((rows, k), dtype=np.float32)
    x[rng.random((rows, k), dtype=np.float32) < 1e-3] *= np.float32(20)
    return x


def _rows(rng, op, rows, k):
    if op.endswith("F32"):
        return _f32_rows(rng, rows, k)
    return rng.integers(-127, 128, (rows, k), dtype=np.int8)


class _DeviceArray:
    """An array over a buffer's device memory; keeps the memory's owner."""

    def __init__(self, owner, buffer, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "version": 2,
                                         "data": (buffer.device_pointer(), False)}


_hip = None


def _device():
    global _hip
    if _hip is None:
        _hip = api.load_hip()
    return api.Device(_hip, 0)


class _Resources:
    """A device with its matrices, buffers and batches, given back with the last state or output."""

    def __init__(self):
        self.dev = _device()
        self.matrices, self.buffers, self.batches = [], [], []

    def matrix(self, bits, scales):
        self.matrices.append(self.dev.matrix(bits, scales))
        return self.matrices[-1]

    def buffer(self, nbytes, data=None):
        b = self.dev.buffer(nbytes)
        self.buffers.append(b)
        if data is not None:
            b.write(data)
        return b

    def tensor(self, buffer, shape, typestr="<f4"):
        """The buffer as a tensor (no copy)."""
        return torch.as_tensor(_DeviceArray(self, buffer, shape, typestr), device="cuda")

    def __del__(self):
        for b in self.batches:
            self.dev.api.BNNX_BatchDestroy(b)
        for m in self.matrices:
            m.destroy()
        for b in self.buffers:
            b.free()
        self.dev.close()


class _State:
    def __init__(self):
        self.res = _Resources()
        self.dev, self.matrix, self.buffer, self.tensor = self.res.dev, self.res.matrix, self.res.buffer, self.res.tensor

    def check(self, status, what):
        if status != api.Status.OK:
            raise api.BnnError(status, what)


def _job(op, matrix, x, y, rows):
    in_t, out_t = api.OP_TYPES[op]
    return api.Job(int(op), matrix.handle.value, x.view(in_t), y.view(out_t), rows)


# ---------------------------------------------------------------------------- accelerator cases


class _Call(_State):
    """BNN_BufferWrite, BNN_Execute, BNN_BufferRead of one row."""

    def __init__(self, case, seed):
        super().__init__()
        k, n, op = case["k"], case["n"], api.Op[case["op"]]
        m = self.matrix(*_matrix(_rng(seed, 1), n, k))
        self.x = _rows(_rng(seed, 2), case["op"], 1, k)
        self.shape, self.dtype = ((1, n, k // 128), np.int16) if case["op"] == "DOT_GROUPS" else ((1, n), np.float32)
        self.out_bytes = int(np.prod(self.shape)) * np.dtype(self.dtype).itemsize
        self.bin, self.bout = self.buffer(self.x.nbytes), self.buffer(self.out_bytes)
        self.job = _job(op, m, self.bin, self.bout, 1)

    def run(self):
        self.bin.write(self.x)
        self.check(self.dev.execute(self.job), "BNN_Execute")
        return self.bout.read(self.out_bytes).view(self.dtype).reshape(self.shape)


class _Rows(_State):
    """BNN_Execute of a multi-row job on resident buffers."""

    def __init__(self, case, seed):
        super().__init__()
        k, n, rows, op = case["k"], case["n"], case["rows"], api.Op[case["op"]]
        m = self.matrix(*_matrix(_rng(seed, 1), n, k))
        x = _rows(_rng(seed, 2), case["op"], rows, k)
        dots = case["op"] == "DOT_GROUPS"
        shape = (rows, n, k // 128) if dots else (rows, n)
        bin_ = self.buffer(x.nbytes, x)
        bout = self.buffer(int(np.prod(shape)) * (2 if dots else 4))
        self.out = self.tensor(bout, shape, "<i2" if dots else "<f4")
        self.job = _job(op, m, bin_, bout, rows)

    def run(self):
        self.check(self.dev.execute(self.job), "BNN_Execute")
        return self.out


class _Batch(_State):
    """BNNX_BatchLaunch of prepared GEMV_F32 / GEMM_F32 jobs; the caller goes on without waiting."""

    def __init__(self, case, seed):
        super().__init__()
        jobs = self.jobs(case, seed)
        arr = (api.Job * len(jobs))(*jobs)
        h = api.ctypes.c_void_p()
        self.check(self.dev.api.BNNX_BatchCreate(self.dev.handle, arr, len(jobs), api.ctypes.byref(h)),
                   "BNNX_BatchCreate")
        self.res.batches.append(h)

    def jobs(self, case, seed):
        k, n, rows, count = case["k"], case["n"], case["rows"], case["jobs"]
        op = api.Op.GEMV_F32 if rows == 1 else api.Op.GEMM_F32
        wr = _rng(seed, 1)
        x = _f32_rows(_rng(seed, 2), count * rows, k)
        bin_, bout = self.buffer(x.nbytes, x), self.buffer(count * rows * n * 4)
        self.out = self.tensor(bout, (count, rows, n))
        return [api.Job(int(op), self.matrix(*_matrix(wr, n, k)).handle.value,
                        bin_.view(api.Type.F32, i * rows * k * 4), bout.view(api.Type.F32, i * rows * n * 4), rows)
                for i in range(count)]

    def run(self):
        self.check(self.dev.api.BNNX_BatchLaunch(self.res.batches[0]), "BNNX_BatchLaunch")
        return self.out


class _Qkv(_Batch):
    """The q, k and v projections of one block of rows, sharing the input."""

    def jobs(self, case, seed):
        rows = case["rows"]
        op = api.Op.GEMV_F32 if rows == 1 else api.Op.GEMM_F32
        wr = _rng(seed, 1)
        x = _f32_rows(_rng(seed, 2), rows, HIDDEN)
        bin_ = self.buffer(x.nbytes, x)
        jobs, self.out = [], []
        for n in (HIDDEN, KV, KV):
            bout = self.buffer(rows * n * 4)
            self.out.append(self.tensor(bout, (rows, n)))
            jobs.append(_job(op, self.matrix(*_matrix(wr, n, HIDDEN)), bin_, bout, rows))
        return jobs


class _Ffn(_State):
    """A decode step's feed-forward block as two fused launches: x = a + b kept, RMSNorm, gate
    and up with SiLU(gate) * up; then the down projection of that row."""

    def __init__(self, case, seed):
        super().__init__()
        k, n = case["k"], case["n"]
        gate_w, up_w, down_w, (a, b, gain) = _ffn_inputs(case, seed)
        ba, bb, bg = (self.buffer(v.nbytes, v) for v in (a, b, gain))
        bx, row, bgate, bup, bh, by = (self.buffer(4 * size) for size in (k, k, n, n, n, k))
        op = api.Op.GEMV_F32
        pre = api.PreOp(api.PreOp.RMSNORM, k, ba.device_pointer(), bb.device_pointer(), bg.device_pointer(),
                        bx.device_pointer(), 1e-6, None, 0)
        post = api.PostOp(api.PostOp.SILU_MUL, bh.device_pointer())
        self.fuse([_job(op, self.matrix(*gate_w), row, bgate, 1), _job(op, self.matrix(*up_w), row, bup, 1)], pre, post)
        self.fuse([_job(op, self.matrix(*down_w), bh, by, 1)], api.PreOp(api.PreOp.ROW, n), api.PostOp())
        self.out = [self.tensor(bx, (k,)), self.tensor(bgate, (n,)), self.tensor(bup, (n,)), self.tensor(bh, (n,)),
                    self.tensor(by, (k,))]

    def fuse(self, jobs, pre, post):
        h, byref = api.ctypes.c_void_p(), api.ctypes.byref
        arr = (api.Job * len(jobs))(*jobs)
        self.check(self.dev.api.BNNX_BatchCreateFusedPost(self.dev.handle, arr, len(jobs), byref(pre), byref(post),
                                                          byref(h)), "BNNX_BatchCreateFusedPost")
        self.res.batches.append(h)

    def run(self):
        for batch in self.res.batches:
            self.check(self.dev.api.BNNX_BatchLaunch(batch), "BNNX_BatchLaunch")
        return self.out


def _ffn_inputs(case, seed):
    k, n = case["k"], case["n"]
    wr, xr = _rng(seed, 1), _rng(seed, 2)
    gate, up, down = ((_bits(wr, o, i), np.full((o, i // 128), 1 / math.sqrt(i), np.float16))
                      for i, o in ((k, n), (k, n), (n, k)))
    a, b = _f32_rows(xr, 1, k)[0], xr.standard_normal(k, dtype=np.float32)
    return gate, up, down, (a, b, (1 + 0.02 * xr.standard_normal(k)).astype(np.float32))


# ---------------------------------------------------------------------------- engine cases

_models: dict = {}  # a program loads its model once and opens a context per conversation


class _Model:
    def __init__(self, name):
        self.tensors = {}

        def keep(tensor, data):
            self.tensors[tensor] = data
            return data

        folder = tempfile.mkdtemp(prefix="cases_")
        path = os.path.join(folder, "model.gguf")
        try:
            if name == "mlp":
                gguf.bnn_mlp_random(path, dims=MLP_DIMS, seed=1, input_pixels=MLP_PIXELS)
            else:
                gguf.qwen3_random(path, hidden=HIDDEN, heads=HEADS, kv_heads=KV_HEADS, head_dim=HEAD_DIM, ffn=FFN,
                                  context=MAX_CONTEXT, seed=5, tweak=keep, **MODELS[name])
            self.dev = _device()
            self.model = engine.Model(engine.EngineLib(), self.dev, path)
            if name == "mlp":
                self.tensors = _mlp_tensors(path)
        finally:
            os.unlink(path)
            os.rmdir(folder)


def _mlp_tensors(path):
    """The classifier's tensors: the file's data section holds them in the order they are written."""
    sizes = []
    for i in range(len(MLP_DIMS) - 1):
        k, n = MLP_DIMS[i], MLP_DIMS[i + 1]
        sizes += [("w", i, n * (k // 128) * 18), ("scale", i, 4 * n), ("bias", i, 4 * n)]
    data = Path(path).read_bytes()
    total = 0
    for _, _, size in sizes:
        total = -(-total // 32) * 32 + size
    at, out = len(data) - total, {}
    start = at
    for what, i, size in sizes:
        at = start + -(-(at - start) // 32) * 32
        raw = data[at:at + size]
        at += size
        out[what, i] = gguf.q1_0_split(raw, MLP_DIMS[i], MLP_DIMS[i + 1]) if what == "w" else np.frombuffer(raw, "<f4")
    return out


def _model(name):
    if name not in _models:
        _models[name] = _Model(name)
    return _models[name]


class _Conversation:
    """A context of a resident model; a pass decodes `ids` at position `start`."""

    def __init__(self, case, seed):
        self.owner = _model(case["model"])
        self.eng = self.owner.model.eng
        history, self.ids = _tokens(case, seed)
        self.start = len(history)
        self.ctx = engine.Context(self.owner.model, n_ctx=-(-(self.start + len(self.ids)) // 128) * 128)
        if self.start:
            self.ctx.decode(history, want_logits=False)

    def run(self):
        self.eng.check(self.eng.BNNE_ContextTruncate(self.ctx.handle, self.start), "BNNE_ContextTruncate")
        return self.ctx.decode(self.ids)

    def __del__(self):
        if hasattr(self, "ctx"):
            self.ctx.free()


def _tokens(case, seed):
    count = case["context"] + 1 if case["kind"] == "decode" else case["tokens"]
    ids = _rng(seed, 3).integers(0, MODELS[case["model"]]["vocab"], count, dtype=np.int32)
    return (ids[:-1], ids[-1:]) if case["kind"] == "decode" else (ids[:0], ids)


class _Classify:
    def __init__(self, case, seed):
        self.owner = _model("mlp")
        self.x = _samples(case, seed)
        self.ctx = engine.Context(self.owner.model, n_batch=case["rows"])

    def run(self):
        return self.ctx.classify(self.x)

    def __del__(self):
        if hasattr(self, "ctx"):
            self.ctx.free()


def _samples(case, seed):
    x = np.zeros((case["rows"], MLP_DIMS[0]), np.float32)
    x[:, :MLP_PIXELS] = _rng(seed, 4).standard_normal((case["rows"], MLP_PIXELS), dtype=np.float32)
    return x


_KINDS = {"call": _Call, "rows": _Rows, "batch": _Batch, "qkv": _Qkv, "ffn": _Ffn, "decode": _Conversation,
          "prefill": _Conversation, "classify": _Classify}


def prepare(case, seed):
    return _KINDS[case["kind"]](case, seed)


def run(state):
    return state.run()


# ---------------------------------------------------------------------------- work and tolerance


def _linear_bytes(k, n):
    return n * k // 8 + n * (k // 128) * 2


def work(case):
    kind = case["kind"]
    if kind in ("call", "rows"):
        k, n, rows = case["k"], case["n"], case.get("rows", 1)
        out = rows * n * (k // 128) * 2 if case["op"] == "DOT_GROUPS" else rows * n * 4
        x = rows * k * (4 if case["op"].endswith("F32") else 1)
        return {"bytes": _linear_bytes(k, n) + x + out, "flops": 2 * rows * k * n}
    if kind == "batch":
        k, n, jobs, rows = case["k"], case["n"], case["jobs"], case["rows"]
        return {"bytes": jobs * (_linear_bytes(k, n) + rows * 4 * (k + n)), "flops": 2 * jobs * rows * k * n}
    if kind == "qkv":
        n = HIDDEN + 2 * KV
        return {"bytes": _linear_bytes(HIDDEN, n) + case["rows"] * 4 * (HIDDEN + n),
                "flops": 2 * case["rows"] * HIDDEN * n}
    if kind == "ffn":
        k, n = case["k"], case["n"]
        return {"bytes": 2 * _linear_bytes(k, n) + _linear_bytes(n, k) + 4 * (5 * k + 3 * n), "flops": 6 * k * n}
    if kind == "classify":
        layers = list(zip(MLP_DIMS[:-1], MLP_DIMS[1:]))
        return {"bytes": sum(_linear_bytes(k, n) + 8 * n for k, n in layers)
                + case["rows"] * 4 * (MLP_DIMS[0] + MLP_DIMS[-1]),
                "flops": sum(2 * case["rows"] * k * n for k, n in layers)}
    m = MODELS[case["model"]]
    past, new = (case["context"], 1) if kind == "decode" else (0, case["tokens"])
    per_layer = 2 * HIDDEN * HIDDEN + 2 * HIDDEN * KV + 3 * HIDDEN * FFN
    weights = m["layers"] * per_layer + m["vocab"] * HIDDEN
    seen = sum(past + i + 1 for i in range(new))  # (query, key) pairs of a head
    return {"bytes": weights // 8 + weights // 64 + m["layers"] * 2 * KV * 4 * (past + new) + 4 * m["vocab"],
            "flops": 2 * new * m["layers"] * per_layer + 2 * m["vocab"] * HIDDEN
            + m["layers"] * HEADS * 4 * HEAD_DIM * seen}


def tolerance(case):
    return "exact"


# ---------------------------------------------------------------------------- 64-bit results


def _weights64(bits, scales):
    """[n][k] float64 on the GPU: +scale where the sign bit is 1, -scale where it is 0."""
    b = torch.from_numpy(np.unpackbits(np.ascontiguousarray(bits), axis=1, bitorder="little")).cuda().double()
    s = torch.from_numpy(np.asarray(scales).view(np.float16).astype(np.float64)).cuda()
    return (2 * b - 1) * s.repeat_interleave(128, dim=1)


def _quantised64(x):
    """The API's row quantisation: Q (as float64) and the row scale, both defined in binary32."""
    x = x.float()
    a = x.abs().amax(dim=-1, keepdim=True)
    s = torch.where(a == 0, torch.ones_like(a), a / 127)
    s = torch.where(s == 0, torch.full_like(s, 2.0 ** -149), s)
    t = x / s
    r = t.trunc()
    q = (r + torch.sign(t) * ((t - r).abs() >= 0.5)).clamp(-127, 127)
    return q.double(), s.double()


def _linear64(x, w):
    q, s = _quantised64(x)
    return (q @ w.t()) * s


def _norm64(x, gain, eps=1e-6):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps) * gain


def _silu64(gate, up):
    return gate / (1 + torch.exp(-gate)) * up


def _accel64(case, seed):
    k, n, rows, op = case["k"], case["n"], case.get("rows", 1), case["op"]
    bits, scales = _matrix(_rng(seed, 1), n, k)
    x = torch.from_numpy(_rows(_rng(seed, 2), op, rows, k)).cuda()
    if op == "DOT_GROUPS":
        signs = _weights64(bits, np.ones((n, k // 128), np.float16))
        d = [x[:, g:g + 128].double() @ signs[:, g:g + 128].t() for g in range(0, k, 128)]
        return torch.stack(d, dim=2).to(torch.int16)
    w = _weights64(bits, scales)
    return _linear64(x, w) if op.endswith("F32") else x.double() @ w.t()


def _qwen64(case, seed):
    t = _model(case["model"]).tensors
    gpu = lambda name: torch.from_numpy(np.asarray(t[name], np.float64)).cuda()  # noqa: E731
    lin = lambda x, name: _linear64(x, _weights64(*t[name]))  # noqa: E731
    ids = np.concatenate(_tokens(case, seed))
    count, half = len(ids), HEAD_DIM // 2
    bits, scales = t["token_embd.weight"]
    x = _weights64(bits[ids], scales[ids])
    # the rotation angles are binary32 products
    freq = np.power(np.float32(1e6), (-2 * np.arange(half) / HEAD_DIM).astype(np.float32)).astype(np.float32)
    angle = torch.from_numpy((np.arange(count, dtype=np.float32)[:, None] * freq).astype(np.float64)).cuda()
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def heads(v, width, gain):
        v = _norm64(v.view(count, width, HEAD_DIM), gain)
        a, b = v[..., :half], v[..., half:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], dim=-1)

    later = torch.ones(count, count, dtype=torch.bool, device="cuda").triu(1)
    for layer in range(MODELS[case["model"]]["layers"]):
        p = f"blk.{layer}."
        h = _norm64(x, gpu(p + "attn_norm.weight"))
        q = heads(lin(h, p + "attn_q.weight"), HEADS, gpu(p + "attn_q_norm.weight"))
        k = heads(lin(h, p + "attn_k.weight"), KV_HEADS, gpu(p + "attn_k_norm.weight"))
        v = lin(h, p + "attn_v.weight").view(count, KV_HEADS, HEAD_DIM)
        y = torch.empty(count, HEADS, HEAD_DIM, dtype=torch.float64, device="cuda")
        for head in range(HEADS):
            kv = head * KV_HEADS // HEADS
            score = (q[:, head] @ k[:, kv].t()) / math.sqrt(HEAD_DIM)
            y[:, head] = torch.softmax(score.masked_fill(later, -math.inf), dim=-1) @ v[:, kv]
        x = x + lin(y.view(count, HIDDEN), p + "attn_output.weight")
        h = _norm64(x, gpu(p + "ffn_norm.weight"))
        x = x + lin(_silu64(lin(h, p + "ffn_gate.weight"), lin(h, p + "ffn_up.weight")), p + "ffn_down.weight")
    h = _norm64(x[-1:], gpu("output_norm.weight"))
    chunks = [_linear64(h, _weights64(bits[i:i + 16384], scales[i:i + 16384])) for i in range(0, len(bits), 16384)]
    return torch.cat(chunks, dim=1)[0].cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "call":
        return _accel64(case, seed).cpu().numpy()
    if kind == "rows":
        return _accel64(case, seed)
    if kind in ("batch", "qkv"):
        rows = case["rows"]
        wr, xr = _rng(seed, 1), _rng(seed, 2)
        if kind == "qkv":
            x = torch.from_numpy(_f32_rows(xr, rows, HIDDEN)).cuda()
            return [_linear64(x, _weights64(*_matrix(wr, n, HIDDEN))) for n in (HIDDEN, KV, KV)]
        k, n, jobs = case["k"], case["n"], case["jobs"]
        x = torch.from_numpy(_f32_rows(xr, jobs * rows, k)).cuda().view(jobs, rows, k)
        return torch.stack([_linear64(x[i], _weights64(*_matrix(wr, n, k))) for i in range(jobs)])
    if kind == "ffn":
        gate_w, up_w, down_w, vectors = _ffn_inputs(case, seed)
        a, b, gain = (torch.from_numpy(v).cuda().double() for v in vectors)
        x = a + b
        h = _norm64(x, gain)[None]
        gate, up = _linear64(h, _weights64(*gate_w)), _linear64(h, _weights64(*up_w))
        h = _silu64(gate, up)
        return [x, gate[0], up[0], h[0], _linear64(h, _weights64(*down_w))[0]]
    if kind == "classify":
        t = _model("mlp").tensors
        x = torch.from_numpy(_samples(case, seed)).cuda().double()
        for i in range(len(MLP_DIMS) - 1):
            scale, bias = (torch.from_numpy(t[what, i].astype(np.float64)).cuda() for what in ("scale", "bias"))
            x = _linear64(x, _weights64(*t["w", i])) * scale + bias
            if i + 2 < len(MLP_DIMS):
                x = x.clamp(min=0)
        return x.cpu().numpy()
    return _qwen64(case, seed)
