"""Blocks of rows: BNNX_LaunchRows against the CPU oracle fed with host-computed rows, and the
engine's prompt blocks against the same tokens decoded one call at a time (whose logits the
fixtures of test_engine.py pin to the reference).  All comparisons bit for bit."""
from __future__ import annotations

import ctypes
import subprocess
import sys

import numpy as np
import pytest

from bnn_cases import first_mismatch
from conftest import ROOT, load_pkg
from test_engine import ERR, _engine_lib, write_error_model
from test_fused import f32, host_rmsnorm, host_silu_mul

pytestmark = pytest.mark.gpu
PreOp = load_pkg().api.PreOp


class Rows:
    def __init__(self, pkg, dev, k, ns, rows, kind, with_b, seed=3):
        self.pkg, self.dev, self.kind, self.k, self.rows, self.with_b = pkg, dev, kind, k, rows, with_b
        rng = np.random.default_rng(seed + k + rows)
        self.chunks = [pkg.synth.matrix(n, k, seed=seed, stream=i) for i, n in enumerate(ns)]
        self.mats = [dev.matrix(b, s) for b, s in self.chunks]
        self.a, self.b = f32(rng, (rows, k), 3.0), f32(rng, (rows, k), 0.5)
        self.gain = (1.0 + 0.02 * rng.standard_normal(k)).astype(np.float32)
        self.bufs = {name: dev.buffer(4 * rows * k) for name in ("a", "b", "gain", "x")}
        self.outs = [dev.buffer(4 * rows * n) for n in ns]
        self.err = dev.buffer(4)
        self.write()
        self.err.write(np.zeros(1, np.int32))
        for o, n in zip(self.outs, ns):
            o.write(np.full(rows * n, 5.0, np.float32))

    def write(self):
        for name in ("a", "b", "gain"):
            self.bufs[name].write(getattr(self, name))

    def launch(self):
        pkg, T = self.pkg, self.pkg.Type.F32
        jobs = (pkg.Job * len(self.mats))(*[
            pkg.Job(int(pkg.Op.GEMM_F32), m.handle.value, self.bufs["a"].view(T), o.view(T), self.rows)
            for m, o in zip(self.mats, self.outs)])
        ptr = {name: b.device_pointer() for name, b in self.bufs.items()}
        pre = PreOp(self.kind, self.k)
        if self.kind != PreOp.ROW:
            pre.a, pre.b = ptr["a"], ptr["b"] if self.with_b else None
        if self.kind == PreOp.RMSNORM:
            pre.gain, pre.a_out, pre.eps, pre.err, pre.err_code = ptr["gain"], ptr["x"], 1e-6, self.err.device_pointer(), 7
        st = self.dev.api.BNNX_LaunchRows(self.dev.handle, jobs, len(self.mats), ctypes.byref(pre))
        return st, self.dev.api.BNNX_DeviceSynchronize(self.dev.handle)

    def row(self, r):
        b = self.b[r] if self.with_b else None
        if self.kind == PreOp.RMSNORM:
            return host_rmsnorm(self.a[r], b, self.gain, 1e-6)[1]
        return host_silu_mul(self.a[r], b) if self.kind == PreOp.SILU_MUL else self.a[r]

    def free(self):
        for m in self.mats:
            m.destroy()
        for b in self.outs + list(self.bufs.values()) + [self.err]:
            b.free()


@pytest.mark.parametrize("k,ns,rows,kind,with_b", [
    (128, [70], 1, PreOp.RMSNORM, True),
    (2048, [256, 100, 64], 3, PreOp.RMSNORM, True),
    (2176, [65], 5, PreOp.RMSNORM, False),
    (6144, [130], 2, PreOp.RMSNORM, True),
    (8192, [64], 17, PreOp.RMSNORM, True),
    (6144, [200], 9, PreOp.SILU_MUL, True),
    (384, [1000], 66, PreOp.SILU_MUL, True),
    (2048, [96, 33], 40, PreOp.ROW, False),
    # more jobs than one launch's parts
    (512, [64, 33, 70, 128, 100], 20, PreOp.RMSNORM, True),
    (256, [64, 5, 70, 64, 130, 64, 1, 33], 9, PreOp.SILU_MUL, True),
    (384, [65, 64, 63, 62, 61, 60], 35, PreOp.ROW, False),
])
def test_launch_rows(pkg, hipdev, oracle, k, ns, rows, kind, with_b):
    f = Rows(pkg, hipdev, k, ns, rows, kind, with_b)
    try:
        print(f"rows {rows} x {k}, kind {kind}", flush=True)
        assert f.launch() == (0, 0)
        x = np.stack([f.row(r) for r in range(rows)])
        with pkg.Device(oracle, 0) as ref:
            for (bits, scales), out in zip(f.chunks, f.outs):
                m = ref.matrix(bits, scales)
                want = ref.run(pkg.Op.GEMM_F32, m, x)
                m.destroy()
                got = out.read().view(np.float32).reshape(want.shape)
                assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), first_mismatch(got, want)
        if kind == PreOp.RMSNORM:
            stored = f.bufs["x"].read().view(np.float32).reshape(rows, k)
            assert np.array_equal(stored, f.a + f.b if with_b else f.a)
    finally:
        f.free()


@pytest.mark.parametrize("kind", [PreOp.ROW, PreOp.RMSNORM, PreOp.SILU_MUL])
def test_launch_rows_illegal_row(pkg, hipdev, kind):
    """One non-finite row: nothing of the block is written, the next synchronisation says so."""
    f = Rows(pkg, hipdev, 256, [70], 20, kind, True)
    try:
        f.a[13, 200] = np.inf
        f.write()
        assert f.launch() == (0, pkg.Status.ERANGE)
        assert (f.outs[0].read().view(np.float32) == 5.0).all()
        assert f.err.read().view(np.int32)[0] == (7 if kind == PreOp.RMSNORM else 0)
        f.a[13, 200] = 1.0
        f.write()
        assert f.launch() == (0, 0)
    finally:
        f.free()


def test_launch_rows_argument_checks(pkg, hipdev):
    """What a call refuses, with its status; nothing is launched."""
    S, T, api = pkg.Status, pkg.Type, hipdev.api
    f = Rows(pkg, hipdev, 256, [70, 64], 6, PreOp.RMSNORM, True)
    ptr = {name: b.device_pointer() for name, b in f.bufs.items()}
    out = [o.device_pointer() for o in f.outs]
    other = hipdev.matrix(*pkg.synth.matrix(64, 128, seed=1))

    def call(kind=PreOp.RMSNORM, count=2, width=256, pre=True, job=None, **fields):
        jobs = (pkg.Job * 9)(*[pkg.Job(int(pkg.Op.GEMM_F32), m.handle.value, f.bufs["a"].view(T.F32), o.view(T.F32), 6)
                               for m, o in zip(f.mats, f.outs)])
        for name, value in (job or {}).items():
            setattr(jobs[1], name, value)
        p = PreOp(kind, width)
        if kind != PreOp.ROW:
            p.a, p.b = ptr["a"], ptr["b"]
        if kind == PreOp.RMSNORM:
            p.gain, p.a_out, p.eps = ptr["gain"], ptr["x"], 1e-6
        for name, value in fields.items():
            setattr(p, name, value)
        return api.BNNX_LaunchRows(hipdev.handle, jobs, count, ctypes.byref(p) if pre else None)

    try:
        assert call(count=0) == S.EINVAL and call(pre=False) == S.EINVAL
        assert call(count=9) == S.ENOTSUP  # more than 8 jobs
        assert call(kind=3) == S.EINVAL
        assert call(width=0) == S.EINVAL and call(width=200) == S.EINVAL and call(width=128) == S.EINVAL
        for missing in ("a", "gain"):
            assert call(**{missing: None}) == S.EINVAL
        for missing in ("a", "b"):
            assert call(PreOp.SILU_MUL, **{missing: None}) == S.EINVAL
        # jobs that differ in rows, K or (plain rows) the input view
        assert call(job={"rows": 5}) == S.EINVAL
        assert call(job={"matrix": other.handle.value, "output": f.outs[1].view(T.F32)}) == S.EINVAL
        assert call(PreOp.ROW, job={"input": f.bufs["b"].view(T.F32)}) == S.EINVAL
        # int8 rows, an output at an odd address; then a call that runs
        assert call(job={"operation": int(pkg.Op.GEMM), "input": f.bufs["a"].view(T.I8)}) == S.ENOTSUP
        assert call(job={"output": f.bufs["x"].view(T.F32, 2)}, a_out=None) == S.ENOTSUP
        assert call(PreOp.ROW, count=1, job={}) == S.OK
        # an output over another output, over an operand, over the stored sum; the sum over an operand
        assert call(job={"output": f.outs[0].view(T.F32)}) == S.EINVAL
        assert call(job={"output": f.bufs["b"].view(T.F32)}) == S.EINVAL
        assert call(job={"output": f.bufs["gain"].view(T.F32)}) == S.EINVAL
        assert call(job={"output": f.bufs["x"].view(T.F32)}) == S.EINVAL
        assert call(a_out=ptr["a"]) == S.EINVAL and call(a_out=out[0] + 4) == S.EINVAL
        assert call(PreOp.ROW, job={"output": f.bufs["a"].view(T.F32)}) == S.EINVAL
        f.outs[0].write(np.full(6 * 70, 5.0, np.float32))  # after the one call that ran
        assert call(job={"rows": 5}) == S.EINVAL
        assert api.BNNX_DeviceSynchronize(hipdev.handle) == S.OK
        assert all((o.read().view(np.float32) == 5.0).all() for o in f.outs)
    finally:
        other.destroy()
        f.free()


def test_launch_rows_limits(pkg, hipdev):
    """4096 rows a call, and no more than the 32 MiB scratch holds."""
    S, T = pkg.Status, pkg.Type.F32
    a, out = hipdev.buffer(4 * 4096 * 8192), hipdev.buffer(4 * 4097 * 8)
    wide, narrow = (hipdev.matrix(*pkg.synth.matrix(8, k, seed=k)) for k in (8192, 128))

    def call(m, k, rows):
        job = (pkg.Job * 1)(pkg.Job(int(pkg.Op.GEMM_F32), m.handle.value, a.view(T), out.view(T), rows))
        return hipdev.api.BNNX_LaunchRows(hipdev.handle, job, 1, ctypes.byref(PreOp(PreOp.ROW, k)))

    assert call(narrow, 128, 4097) == S.ENOTSUP
    assert call(wide, 8192, 4096) == S.ENOTSUP
    a.write(np.ones(4096 * 128, np.float32))
    assert call(narrow, 128, 4096) == S.OK
    assert hipdev.api.BNNX_DeviceSynchronize(hipdev.handle) == S.OK
    got = out.read().view(np.float32)[:4096 * 8].reshape(4096, 8)
    assert (got == got[0]).all() and np.isfinite(got).all()
    wide.destroy()
    narrow.destroy()
    a.free()
    out.free()


@pytest.mark.parametrize("k", [128, 384, 640, 2048, 2176, 4096, 8192])
def test_launch_rows_sum_of_squares(pkg, hipdev, oracle, k):
    """RMSNorm rows whose running sums leave the speculative windows: the sequential loop's bits."""
    f = Rows(pkg, hipdev, k, [65], 6, PreOp.RMSNORM, False)
    try:
        ramp = np.exp2(np.linspace(-60, 40, k)).astype(np.float32)
        f.a[0] = 1.1
        f.a[1], f.a[2] = ramp, ramp[::-1]
        f.a[3] = 0
        f.a[3, k - 1] = 3
        f.a[4] = np.where(np.arange(k) % 2, np.float32(1e-20), np.float32(777.7))
        f.a[5] = np.float32(1e-22)
        f.a[5, k // 2] = 1
        f.write()
        print(f"sum of squares, {k}", flush=True)
        assert f.launch() == (0, 0)
        x = np.stack([f.row(r) for r in range(6)])
        with pkg.Device(oracle, 0) as ref:
            m = ref.matrix(*f.chunks[0])
            want = ref.run(pkg.Op.GEMM_F32, m, x)
            m.destroy()
        got = f.outs[0].read().view(np.float32).reshape(want.shape)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), first_mismatch(got, want)
    finally:
        f.free()


TINY = {"layers": 2, "hidden": 256, "heads": 2, "kv_heads": 1, "ffn": 512, "vocab": 512, "context": 4352}


@pytest.mark.parametrize("count,split", [
    (3, 0), (7, 2), (16, 0), (33, 1), (64, 0), (65, 0), (127, 63), (200, 0),
    (1025, 0),      # a second block of one token
    (1300, 40),     # two blocks behind a started cache
    (2500, 1400),   # softmax rows of more than one LDS chunk
    (4200, 4150),   # single tokens whose in-order softmax sum spans two rounds of segments
])
def test_prompt_blocks_match_single_tokens(pkg, hip, tmp_path, count, split):
    path = tmp_path / "m.gguf"
    pkg.gguf.qwen3_random(path, **TINY)
    ids = np.random.default_rng(count).integers(0, TINY["vocab"], count, dtype=np.int32)
    with pkg.Device(hip, 0) as dev:
        m = pkg.engine.Model(_engine_lib(pkg), dev, path)
        one, block = (pkg.engine.Context(m, n_ctx=TINY["context"]) for _ in range(2))
        print(f"prompt of {count} tokens, {split} of them before the block", flush=True)
        for t in ids[:-1]:
            one.decode([t], want_logits=False)
        want = one.decode(ids[-1:])
        if split:
            block.decode(ids[:split], want_logits=False)
        got = block.decode(ids[split:])
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        # the caches are the same too: the next steps read every row
        nxt = int(want.argmax())
        assert block.decode_greedy(nxt, 3) == one.decode_greedy(nxt, 3)
        for c in (one, block):
            c.free()
        m.free()


def last_step_and_block(pkg, hip, path, ids, context, singles):
    """The last logits with the last `singles` tokens decoded one by one behind a prompt block,
    and with every token in blocks."""
    with pkg.Device(hip, 0) as dev:
        m = pkg.engine.Model(_engine_lib(pkg), dev, path)
        step, block = (pkg.engine.Context(m, n_ctx=context) for _ in range(2))
        step.decode(ids[:-singles], want_logits=False)
        for t in ids[-singles:-1]:
            step.decode([t], want_logits=False)
        got = step.decode(ids[-1:])
        want = block.decode(ids)
        for c in (step, block):
            c.free()
        m.free()
    return got, want


def test_step_past_the_kept_exponentials(pkg, hip, tmp_path):
    """Steps around 16384 positions: past them k_attn_pv forms its exponentials again."""
    path, context = tmp_path / "m.gguf", 16400
    pkg.gguf.qwen3_random(path, **{**TINY, "context": context})
    ids = np.random.default_rng(2).integers(0, TINY["vocab"], 16388, dtype=np.int32)
    print("16388 positions", flush=True)
    got, want = last_step_and_block(pkg, hip, path, ids, context, 6)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("count", [400, 4300])
def test_softmax_sum_off_the_windows(pkg, hip, tmp_path, count):
    """A softmax whose first term is 1 and whose others lie below half an ulp of 1: the in-order
    sum stays at 1 while the prefix sums in 64 bits leave it by more than the candidates reach,
    so k_attn_pv adds every segment term by term."""
    hidden, hd, vocab = TINY["hidden"], 128, TINY["vocab"]
    kept = {}

    def signs(bits):
        return np.unpackbits(bits, axis=1, bitorder="little").astype(np.float64) * 2 - 1

    def note(name, data):  # the first layer's weights, its input norm without gains
        if name == "blk.0.attn_norm.weight":
            return np.ones_like(data)
        if name in ("token_embd.weight", "blk.0.attn_q.weight", "blk.0.attn_k.weight"):
            kept[name] = signs(data[0])
        return data

    pkg.gguf.qwen3_random(tmp_path / "weights.gguf", **{**TINY, "context": 4608}, tweak=note)
    # head 0's queries and keys of every token: signs times signs; norm to RMS 1; of them only the
    # pair of dims that turns least with the position
    pair = [hd // 2 - 1, hd - 1]

    def heads(w):
        y = kept["token_embd.weight"] @ w[:hd].T
        return (y / np.sqrt((y * y).mean(axis=1, keepdims=True)))[:, pair]

    q, key = heads(kept["blk.0.attn_q.weight"]), heads(kept["blk.0.attn_k.weight"])
    # a token x ahead of many y: score(y, x) - score(y, y) = 16.9, so a term of y is 4.6e-8
    lead = q @ key.T - (q * key).sum(axis=1)[:, None]
    y, x = np.unravel_index(lead.argmax(), lead.shape)
    assert lead[y, x] > 1.0 and x != y
    gain = np.float32(np.sqrt(16.9 / (lead[y, x] / np.sqrt(hd))))

    def tweak(name, data):
        if name in ("blk.0.attn_q_norm.weight", "blk.0.attn_k_norm.weight"):
            data = np.zeros_like(data)
            data[pair] = gain
            return data
        return note(name, data)

    path = tmp_path / "m.gguf"
    pkg.gguf.qwen3_random(path, **{**TINY, "context": 4608}, tweak=tweak)
    ids = np.full(count, y, np.int32)
    ids[0] = x
    term = np.exp(-float(gain) ** 2 * lead[y, x] / np.sqrt(hd))
    # (with the position's turn: below 6e-3, a few percent of a term)
    assert 0.8 * 128 * term > 33 * 2.0 ** -23 and term * 1.25 < 2.0 ** -24
    print(f"{count} positions, tokens {x} and {y}, a term {term:.3g}", flush=True)
    got, want = last_step_and_block(pkg, hip, path, ids, 4608, 3)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_prompt_block_error_then_prompt(pkg, hip, tmp_path):
    """A prompt whose middle token fails: the status of the single-token step, the position
    unchanged; afterwards the clean prompt gives the reference's tokens."""
    model_path, _, _ = write_error_model(pkg, tmp_path)
    prompt = list(ERR["prompt"])
    bad = prompt[:2] + [ERR["error_token"]] + prompt[2:]
    with pkg.Device(hip, 0) as dev:
        m = pkg.engine.Model(_engine_lib(pkg), dev, model_path)
        c = pkg.engine.Context(m, n_ctx=ERR["ctx"])
        with pytest.raises(pkg.engine.EngineError) as e:
            c.decode(bad)
        assert e.value.status == -7 and "RMSNorm" in str(e.value)
        assert c.pos() == 0
        first = int(c.decode(prompt).argmax())
        want = [row[1] for row in ERR["steps"]]
        assert [first] + c.decode_greedy(first, len(want) - 1) == want
        c.free()
        m.free()


def test_growing_block_keeps_batches(pkg, hip, tmp_path):
    """Longer and longer prompts grow the context's block memory; a program's own prepared batch
    on the same device stays valid."""
    path = tmp_path / "m.gguf"
    pkg.gguf.qwen3_random(path, **TINY)
    bits, scales = pkg.synth.matrix(70, 256, seed=2)
    with pkg.Device(hip, 0) as dev:
        m = pkg.engine.Model(_engine_lib(pkg), dev, path)
        c = pkg.engine.Context(m, n_ctx=TINY["context"])
        mat, bi, bo = dev.matrix(bits, scales), dev.buffer(4 * 256), dev.buffer(4 * 70)
        bi.write(np.ones(256, np.float32))
        T = pkg.Type.F32
        jobs = (pkg.Job * 1)(pkg.Job(int(pkg.Op.GEMV_F32), mat.handle.value, bi.view(T), bo.view(T), 1))
        batch = ctypes.c_void_p()
        assert dev.api.BNNX_BatchCreate(dev.handle, jobs, 1, ctypes.byref(batch)) == pkg.Status.OK
        for count in (5, 65, 130, 600, 1100):
            print(f"prompt of {count} tokens", flush=True)
            c.decode(np.arange(count, dtype=np.int32) % TINY["vocab"], want_logits=False)
            assert dev.api.BNNX_BatchLaunch(batch) == pkg.Status.OK
        assert dev.api.BNNX_DeviceSynchronize(dev.handle) == pkg.Status.OK
        dev.api.BNNX_BatchDestroy(batch)
        c.free()
        m.free()
        mat.destroy()
        bi.free()
        bo.free()


def test_block_growth_without_memory(pkg, tmp_path):
    """A block buffer that finds no memory: the prompt runs token by token, same logits, and the
    program's own prepared batch on the device stays valid."""
    path = tmp_path / "m.gguf"
    pkg.gguf.qwen3_random(path, **TINY)
    r = subprocess.run([sys.executable, str(ROOT / "tests" / "block_growth_run.py"), str(path)], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.endswith("OK\n"), r.stdout[-500:] + r.stderr[-1500:]


# Batches whose multi-row jobs run on the matrix cores: groups of up to four alike jobs (one k,
# rows and operation), shared and own input views, beside jobs that stay with the dots.
@pytest.mark.parametrize("specs,shared", [
    ([("GEMM_F32", 2048, 2048, 48), ("GEMM_F32", 2048, 1024, 48), ("GEMM_F32", 2048, 1030, 48)], True),
    ([("GEMM_F32", 2048, 2048, 64)] * 9, False),                        # groups of four, four and one
    ([("GEMM_F32", 256, 70, 4)], False),                                # a small group alone
    ([("GEMM_F32", 256, 70, 4), ("GEMM", 256, 70, 4)], False),          # two small groups: the dots
    ([("GEMM_F32", 4096, 3000, 17), ("GEMV_F32", 512, 100, 1), ("GEMM", 4096, 200, 17),
      ("DOT_GROUPS", 4096, 1000, 33), ("GEMM_F32", 128, 5, 3), ("GEMM_F32", 4096, 65, 17)], False),
    ([("DOT_GROUPS", 1024, 1000, 40)] * 4, False),                      # dots of few groups, four parts
    ([("DOT_GROUPS", 640, 1301, 64), ("DOT_GROUPS", 640, 65, 64), ("DOT_GROUPS", 640, 4001, 64)], False),
], ids=["shared", "nine", "small", "small-two", "mixed", "dots", "dots-odd"])
def test_batch_jobs_on_the_matrix_cores(pkg, hipdev, oracle_fast, specs, shared):
    from test_hip_batch import _free, _mk_batch, _oracle, _outputs
    mats, xs, bi, bo, jobs, out_off, layouts = _mk_batch(pkg, hipdev, specs, seed=11)
    if shared:  # one view for all
        for i in range(len(specs)):
            jobs[i].input, xs[i] = jobs[0].input, xs[0]
    wants = _oracle(pkg, oracle_fast, specs, mats, xs)
    print(f"batch of {len(specs)} jobs", flush=True)

    def check():
        for i, (got, want) in enumerate(zip(_outputs(bo, out_off, layouts), wants)):
            assert np.array_equal(got.view(np.uint8), want.view(np.uint8)), (i, specs[i], first_mismatch(got, want))
        bo.write(np.zeros(bo.nbytes, np.uint8))

    api = hipdev.api
    for _ in range(2):  # planned, then from the cached tables
        assert api.BNNX_ExecuteBatch(hipdev.handle, jobs, len(specs)) == pkg.Status.OK
        check()
    batch = ctypes.c_void_p()
    assert api.BNNX_BatchCreate(hipdev.handle, jobs, len(specs), ctypes.byref(batch)) == pkg.Status.OK
    for _ in range(2):
        assert api.BNNX_BatchLaunch(batch) == pkg.Status.OK
        assert api.BNNX_DeviceSynchronize(hipdev.handle) == pkg.Status.OK
        check()
    # an illegal value in the last job's last row: no job writes anything
    t, at = pkg.Type.F32, jobs[len(specs) - 1].input.offset
    row_bytes = specs[-1][1] * 4
    if jobs[len(specs) - 1].input.type == int(t):
        bi.write(np.full(1, np.nan, np.float32), at + (specs[-1][3] - 1) * row_bytes)
        assert api.BNNX_BatchLaunch(batch) == pkg.Status.OK
        assert api.BNNX_DeviceSynchronize(hipdev.handle) == pkg.Status.ERANGE
        assert not bo.read().any()
    api.BNNX_BatchDestroy(batch)
    _free(mats, bi, bo)


@pytest.mark.parametrize("op,k,n,rows", [
    ("GEMM_F32", 384, 70, 1), ("GEMM_F32", 384, 70, 7), ("GEMM_F32", 384, 70, 8), ("GEMM", 1152, 65, 5),
    ("DOT_GROUPS", 256, 70, 7), ("DOT_GROUPS", 1024, 33, 2), ("DOT_GROUPS", 1024, 33, 9),
])
def test_outputs_at_any_address(pkg, hipdev, oracle_fast, op, k, n, rows):
    """Outputs that are not naturally aligned, by the dots and on the matrix cores."""
    from bnn_cases import fast_oracle
    host = pkg.synth.matrix(n, k, seed=k + n)
    in_t, out_t = pkg.api.OP_TYPES[pkg.Op[op]]
    x = pkg.synth.normal_f32(rows, k, seed=6) if op == "GEMM_F32" else pkg.synth.int8_uniform(rows, k, seed=6)
    row = n * (2 * (k // 128) if op == "DOT_GROUPS" else 4)
    m, bi, bo = hipdev.matrix(*host), hipdev.buffer(x.nbytes), hipdev.buffer(1 + rows * (row + 3))
    bi.write(x)
    bo.write(np.full(bo.nbytes, 0x5a, np.uint8))
    job = pkg.Job(int(pkg.Op[op]), m.handle.value, bi.view(in_t), bo.view(out_t, 1, row + 3), rows)
    assert hipdev.execute(job) == pkg.Status.OK
    want = np.full((rows, row + 3), 0x5a, np.uint8)
    want[:, :row] = fast_oracle(pkg, oracle_fast, op, *host, x).reshape(rows, -1).view(np.uint8)
    assert np.array_equal(bo.read()[1:], want.reshape(-1))
    m.destroy()
    bi.free()
    bo.free()


@pytest.mark.parametrize("n,rows", [(1024, 4), (1024, 5), (1000, 16), (6144, 64)])
def test_call_and_read_in_turn(pkg, hipdev, oracle_fast, n, rows):
    """Write, call and read in turn, reads by the copy kernel (16 KB) and the copy engine, calls
    with and without a read before: every read holds the results of the call before it."""
    from bnn_cases import fast_oracle
    k, T = 2048, pkg.Type.F32
    host = pkg.synth.matrix(n, k, seed=9)
    xs = [pkg.synth.normal_f32(rows, k, seed=40 + i) for i in range(3)]
    wants = [fast_oracle(pkg, oracle_fast, "GEMM_F32", *host, x).reshape(-1) for x in xs]
    m, bi, bo = hipdev.matrix(*host), hipdev.buffer(xs[0].nbytes), hipdev.buffer(4 * n * rows)
    job = pkg.Job(int(pkg.Op.GEMM_F32), m.handle.value, bi.view(T), bo.view(T), rows)
    for turn in range(12):
        bi.write(xs[turn % 3])
        assert hipdev.execute(job) == pkg.Status.OK
        if turn % 4 != 3:
            got = bo.read().view(np.float32)
            assert np.array_equal(got.view(np.uint32), wants[turn % 3].view(np.uint32)), (turn, first_mismatch(got, wants[turn % 3]))
    m.destroy()
    bi.free()
    bo.free()


@pytest.mark.parametrize("specs,gemms,dots", [
    ([("GEMM_F32", 2048, 1024, 64)] * 3, 1, 0),
    ([("GEMM_F32", 2048, 1024, 64)] * 32, 8, 0),
    ([("GEMM_F32", 2048, 1024, 16)] * 32, 0, 1),   # eight launches against one: 41.9 us a pass, 32.4 as dots
    ([("GEMM_F32", 512, 512, 8)], 0, 1),
    ([("GEMM_F32", 4096, 512, 4)], 1, 0),
    ([("DOT_GROUPS", 1024, 1000, 40)] * 4, 1, 0),
    ([("DOT_GROUPS", 1024, 1000, 40)] * 16, 0, 1),
    ([("GEMM_F32", 2048, 2048, 64)] * 4 + [("GEMV_F32", 2048, 64, 1)] * 3, 1, 1),
], ids=["qkv", "many-rows", "many-jobs", "one-small", "one-long", "dots-four", "dots-many", "beside"])
def test_batch_routes(pkg, hipdev, specs, gemms, dots):
    """Few jobs of many rows take launches on the matrix cores, many jobs of few rows the one dot
    launch (what each gives is compared above and in test_hip_batch.py)."""
    host = {(k, n): pkg.synth.matrix(n, k, seed=4) for _, k, n, _ in specs}
    mats = [hipdev.matrix(*host[k, n]) for _, k, n, _ in specs]
    jobs, bufs = (pkg.Job * len(specs))(), []
    for i, (op, k, n, rows) in enumerate(specs):
        in_t, out_t = pkg.api.OP_TYPES[pkg.Op[op]]
        bi = hipdev.buffer(rows * k * (4 if in_t == pkg.Type.F32 else 1))
        bo = hipdev.buffer(rows * n * (2 * (k // 128) if op == "DOT_GROUPS" else 4))
        bi.write(np.zeros(bi.nbytes, np.uint8))
        bufs += [bi, bo]
        jobs[i] = pkg.Job(int(pkg.Op[op]), mats[i].handle.value, bi.view(in_t), bo.view(out_t), rows)
    batch = ctypes.c_void_p()
    assert hipdev.api.BNNX_BatchCreate(hipdev.handle, jobs, len(specs), ctypes.byref(batch)) == pkg.Status.OK
    hipdev.kernel_timing(True)
    before = [hipdev.kernel_timing_read(kind)[1] for kind in (3, 1)]
    assert hipdev.api.BNNX_BatchLaunch(batch) == pkg.Status.OK
    assert hipdev.api.BNNX_DeviceSynchronize(hipdev.handle) == pkg.Status.OK
    ran = [hipdev.kernel_timing_read(kind)[1] - b for kind, b in zip((3, 1), before)]
    hipdev.kernel_timing(False)
    hipdev.api.BNNX_BatchDestroy(batch)
    for m in mats:
        m.destroy()
    for b in bufs:
        b.free()
    assert ran == [gemms, dots]


@pytest.mark.parametrize("k,n,rows,off,pad", [
    (896, 1000, 37, 0, 0),      # 7 groups, 16-byte rows
    (896, 1001, 20, 0, 0),      # rows that start at odd multiples of 2 bytes
    (128, 33, 17, 2, 0),        # one group, a view at offset 2
    (2048, 100, 16, 0, 0),      # 16 groups: 16-byte pieces, a partial column tile
    (512, 70, 49, 8, 8),        # 4 groups, 8-byte aligned rows
    (2048, 70, 9, 2, 6),        # 16 groups from an odd address: two values at a time
    (2176, 65, 18, 0, 0),       # 17 groups, an odd number of values in a tile's row
    (8192, 40, 33, 0, 16),      # 64 groups
    (1280, 5000, 130, 0, 0),    # more than two tiles per CU: 64-column tiles
    # the blocks for few groups: one group, pairs, fours; a last group alone; odd addresses
    (128, 8000, 300, 0, 0),     # 64 x 128 blocks, more workgroups than signal
    (256, 2417, 70, 2, 0),
    (384, 1001, 65, 0, 2),
    (512, 301, 130, 4, 4),      # fours at addresses that are no multiples of 8
    (640, 5065, 27, 0, 0),
    (768, 1223, 119, 0, 0),
    (896, 6046, 106, 2, 2),
    (1024, 6421, 170, 0, 0),    # fours in 64 x 128 blocks
    (1024, 3001, 63, 0, 8),
])
def test_dot_groups_rows(pkg, hipdev, oracle_fast, k, n, rows, off, pad):
    """DOT_GROUPS of many rows: every store width; padding and neighbours untouched."""
    from bnn_cases import fast_oracle
    host = pkg.synth.matrix(n, k, seed=k + n)
    x = pkg.synth.int8_uniform(rows, k, seed=3)
    m = hipdev.matrix(*host)
    row = n * (k // 128) * 2
    bi, bo = hipdev.buffer(x.nbytes), hipdev.buffer(off + rows * (row + pad) + 64)
    bi.write(x)
    bo.write(np.full(bo.nbytes, 0x5a, np.uint8))
    T = pkg.Type
    job = pkg.Job(int(pkg.Op.DOT_GROUPS), m.handle.value, bi.view(T.I8), bo.view(T.I16, off, row + pad), rows)
    print(f"dots {k}->{n} x {rows}", flush=True)
    assert hipdev.execute(job) == pkg.Status.OK
    raw = bo.read()
    want = np.full(bo.nbytes, 0x5a, np.uint8)
    dots = fast_oracle(pkg, oracle_fast, "DOT_GROUPS", *host, x).reshape(rows, -1).view(np.uint8)
    for r in range(rows):
        want[off + r * (row + pad):off + r * (row + pad) + row] = dots[r]
    assert np.array_equal(raw, want)
    bi.free()
    bo.free()
    m.destroy()


# k_gemm_mx in each of its tiles, at group counts around its pipeline's depth, ragged both ways
@pytest.mark.parametrize("op", ["GEMM_F32", "GEMM"])
@pytest.mark.parametrize("k,n,rows,pad", [
    (128, 1500, 500, 0),      # 64 x 64, one group
    (2176, 701, 650, 12),     # 64 x 64, 17 groups, rows that are not 16-byte aligned
    (256, 2100, 641, 0),      # 64 x 128
    (384, 4000, 642, 16),     # 64 x 192
    (640, 3999, 1000, 0),     # 128 x 128
    (512, 5001, 770, 4),      # 128 x 192
    (2048, 4213, 250, 0),     # 64 x 128, half a round
    (2048, 5900, 400, 0),     # 64 x 192
    (896, 8000, 1000, 0),     # 128 x 128, more workgroups than signal
    (6144, 2048, 289, 0),     # 64 x 64, 48 groups
    (4224, 4001, 99, 8),      # 32 x 64, 33 groups
    (8192, 1000, 130, 0),     # 32 x 64, 64 groups
])
def test_gemm_tiles(pkg, hipdev, oracle_fast, op, k, n, rows, pad):
    from bnn_cases import fast_oracle
    host = pkg.synth.matrix(n, k, seed=k + n)
    f32_in = op == "GEMM_F32"
    x = pkg.synth.normal_f32(rows, k, seed=5) if f32_in else pkg.synth.int8_uniform(rows, k, seed=5)
    m = hipdev.matrix(*host)
    bi, bo = hipdev.buffer(x.nbytes), hipdev.buffer(rows * (4 * n + pad))
    bi.write(x)
    bo.write(np.full(bo.nbytes, 0x5a, np.uint8))
    T = pkg.Type
    job = pkg.Job(int(pkg.Op[op]), m.handle.value, bi.view(T.F32 if f32_in else T.I8), bo.view(T.F32, 0, 4 * n + pad), rows)
    print(f"{op} {k}->{n} x {rows}", flush=True)
    assert hipdev.execute(job) == pkg.Status.OK
    raw = bo.read().reshape(rows, 4 * n + pad)
    want = fast_oracle(pkg, oracle_fast, op, *host, x).reshape(rows, n)
    assert np.array_equal(raw[:, :4 * n].copy().view(np.uint32), want.view(np.uint32))
    assert (raw[:, 4 * n:] == 0x5a).all()
    bi.free()
    bo.free()
    m.destroy()
