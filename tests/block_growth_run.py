"""Run by test_rows.py::test_block_growth_without_memory in a process of its own: the engine
library has to be loaded behind oracle/lib/liballoc_fail.so."""
from __future__ import annotations

import ctypes
import sys

import numpy as np

from conftest import ROOT, load_pkg

CONTEXT = 2304


def main(path: str) -> None:
    fail = ctypes.CDLL(str(ROOT / "oracle" / "lib" / "liballoc_fail.so"), mode=ctypes.RTLD_GLOBAL)
    pkg = load_pkg()
    hip = pkg.load_hip()

    def arm(countdown: int) -> None:
        fail.alloc_fail_arm(ctypes.cast(hip.lib.BNN_BufferAlloc, ctypes.c_void_p), countdown)

    arm(0)
    with pkg.Device(hip, 0) as dev:
        m = pkg.engine.Model(pkg.engine.EngineLib(), dev, path)
        one, block = (pkg.engine.Context(m, n_ctx=CONTEXT) for _ in range(2))
        bits, scales = pkg.synth.matrix(70, 256, seed=2)
        mat, bi, bo = dev.matrix(bits, scales), dev.buffer(4 * 256), dev.buffer(4 * 70)
        bi.write(np.ones(256, np.float32))
        T = pkg.Type.F32
        jobs = (pkg.Job * 1)(pkg.Job(int(pkg.Op.GEMV_F32), mat.handle.value, bi.view(T), bo.view(T), 1))
        batch = ctypes.c_void_p()
        assert hip.BNNX_BatchCreate(dev.handle, jobs, 1, ctypes.byref(batch)) == pkg.Status.OK
        # a block's two buffers in turn find no memory, for the first block and for larger ones
        turns = [(5, 1), (5, 2), (5, 1), (5, 0), (70, 2), (90, 1), (140, 1), (140, 2), (300, 2), (300, 0), (1100, 0)]
        for turn, (count, countdown) in enumerate(turns):
            print(f"prompt of {count} tokens, allocation {countdown} fails", flush=True)
            ids = np.random.default_rng(turn).integers(0, 512, count, dtype=np.int32)
            arm(countdown)
            got = block.decode(ids)
            assert fail.alloc_fail_left() == 0, "the block made fewer buffers than that"
            for t in ids[:-1]:
                one.decode([t], want_logits=False)
            want = one.decode(ids[-1:])
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
            assert hip.BNNX_BatchLaunch(batch) == pkg.Status.OK, "the program's own batch is stale"
            assert hip.BNNX_DeviceSynchronize(dev.handle) == pkg.Status.OK
        hip.BNNX_BatchDestroy(batch)
        one.free()
        block.free()
        m.free()
        mat.destroy()
        bi.free()
        bo.free()
    print("OK", flush=True)


if __name__ == "__main__":
    main(sys.argv[1])
