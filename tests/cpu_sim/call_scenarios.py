"""Device calls of several blocks replayed on the CPU simulation build
(tests/test_sim_calls.py): `python call_scenarios.py NAME [key=int ...]`, exit
status as scenarios.py's."""
import ctypes
import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)
sys.path.insert(0, os.path.dirname(HERE))
import simlib  # noqa: E402

lib = simlib.load()
import tan_amd as T  # noqa: E402

UNIFORM = T.TAN_CONVOLUTION_METHOD_FFT_UNIFORM_PARTITIONED
NONUNIFORM = T.TAN_CONVOLUTION_METHOD_FFT_PARTITIONED_NONUNIFORM
TIME_DOMAIN = T.TAN_CONVOLUTION_METHOD_TIME_DOMAIN
METHODS = (UNIFORM, NONUNIFORM, TIME_DOMAIN)
_done = ctypes.c_size_t(0)


def call(conv, x, y, t, n, B):
    """Blocks t .. t + n - 1 of x into y (simlib.Dev; the same one: in place)."""
    rc = lib.tanx_conv_process_device(conv.handle, x.at(t * B), x.stride, y.at(t * B), y.stride, n * B, None,
                                      ctypes.byref(_done))
    assert rc == T.AMF_OK and _done.value == n * B, (rc, _done.value)


def update(conv, h):
    dev = simlib.Dev(*h.shape, h)
    assert lib.tanx_conv_update_td_device(conv.handle, dev.ptr, dev.stride, h.shape[1], None, 0) == T.AMF_OK
    dev.free()


def in_place(method=0, L=4096, B=64, C=3):
    """Calls whose output is their input's buffer give what separate buffers
    do: a crossfade inside a call, calls of more blocks than one launch takes."""
    calls = [4, 8, 1, 8, 40, 3, 16, 2, 24]
    nb, ups = sum(calls), {0: 0, 3: 1, 6: 2}
    x = T.signals.input_bank(C, nb * B, base_seed=11)
    irs = [T.signals.ir_bank(C, L, k, base_seed=12) for k in range(len(ups))]
    ctx = T.TANContext(device=0)
    ys = []
    for same in (False, True):
        conv = T.TANConvolution(ctx)
        assert conv.InitGpu(METHODS[method], L, B, C) == T.AMF_OK
        xd = simlib.Dev(C, nb * B, x)
        yd = xd if same else simlib.Dev(C, nb * B, 0.0)
        t = 0
        for i, n in enumerate(calls):
            if i in ups:
                update(conv, irs[ups[i]])
            call(conv, xd, yd, t, n, B)
            t += n
        ys.append(yd.a.copy())
    assert np.abs(ys[0]).max() > 0.1
    err = np.abs(ys[0] - ys[1]).max(0).reshape(nb, B).max(1)
    print("in place against separate buffers:", err.max(), "from block", int(np.argmax(err > 0)), flush=True)
    assert np.array_equal(ys[0], ys[1])


def few_partitions(P=4, kp=8, B=64, C=2):
    """Objects with fewer partitions than their calls have blocks, a response
    issued before some calls: as one block per call."""
    calls = [5, 24, 1, 16, 8, 33, 4, 7]
    nb, ups = sum(calls), {0: 0, 3: 1, 5: 2}
    x = T.signals.input_bank(C, nb * B, base_seed=21)
    irs = [T.signals.ir_bank(C, P * B, k, base_seed=22) for k in range(len(ups))]
    at = dict(zip(np.cumsum([0] + calls), range(len(calls) + 1)))
    ctx = T.TANContext(device=0)
    ys = []
    for sizes in (calls, [1] * nb):
        conv = T.TANConvolution(ctx, pass_blocks=kp)
        assert conv.InitGpu(UNIFORM, P * B, B, C) == T.AMF_OK
        assert conv.Info()["partitions"] == P
        xd, yd = simlib.Dev(C, nb * B, x), simlib.Dev(C, nb * B, 0.0)
        t = 0
        for n in sizes:
            if at.get(t) in ups:
                update(conv, irs[ups[at[t]]])
            call(conv, xd, yd, t, n, B)
            t += n
        ys.append(yd.a.copy())
    err = float(np.abs(ys[0].astype(np.float64) - ys[1]).max())
    print(f"P={P} K={kp}: calls vs one block per call {err:.3e}", flush=True)
    assert np.abs(ys[1]).max() > 0.1 and err <= 2e-6  # outputs up to 3, as in test_gpu_passes.py


def chunk_changes(method=1, L=32768, B=64, C=3):
    """The tail chunk count set between a call of several blocks and the next
    block: as one block per call with the default count."""
    # (the first call: a non-uniform object's response fades in up to three frames later)
    calls, chunks = [200, 8, 1, 7, 1, 1, 9, 1, 6, 2, 12, 1], {2: 4, 4: 1, 5: 0, 7: 3, 9: 2, 11: 8}
    nb = sum(calls)
    x = T.signals.input_bank(C, nb * B, base_seed=31)
    h = T.signals.ir_bank(C, L, 0, base_seed=32)
    ctx = T.TANContext(device=0)
    ys = []
    for sizes in (calls, [1] * nb):
        conv = T.TANConvolution(ctx, nu_multiple=64 if method == 1 else 0)
        assert conv.InitGpu(METHODS[method], L, B, C) == T.AMF_OK
        update(conv, h)
        xd, yd = simlib.Dev(C, nb * B, x), simlib.Dev(C, nb * B, 0.0)
        t = 0
        for i, n in enumerate(sizes):
            if sizes is calls and i in chunks:
                assert lib.tanx_conv_set_tail_chunks(conv.handle, chunks[i]) == T.AMF_OK
            call(conv, xd, yd, t, n, B)
            t += n
        ys.append(yd.a.copy())
    err = float(np.abs(ys[0].astype(np.float64) - ys[1]).max())
    print(f"chunk count changed between calls: {err:.3e}", flush=True)
    assert np.abs(ys[1]).max() > 0.1 and err <= 2e-6  # outputs up to 3, as in test_gpu_passes.py


if __name__ == "__main__":
    globals()[sys.argv[1]](**{k: int(v) for k, v in (a.split("=") for a in sys.argv[2:])})
    print("scenario complete", flush=True)
