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


def mixed(seed=1, method=0, kp=0, precision=0, steps=40):
    """Random orders of calls of several blocks, single blocks, host and group
    blocks, updates, flushes, stops and chunk counts: as the same object a
    block at a time on separate launches."""
    rng = np.random.default_rng(1000 * seed + 10 * kp + method)
    B = int(rng.choice([64, 128, 512]))
    parts = int(rng.choice([4, 16, 64])) if method == 0 else 128
    C, L = int(rng.integers(1, 5)), parts * B - int(rng.integers(0, B // 2))
    opt = dict(ir_precision=precision)
    if method == 0:
        opt.update(pass_blocks=kp, pass_phase=int(rng.integers(0, 16)), ir_slots=int(rng.choice([2, 3])),
                   max_tail_chunks=int(rng.choice([0, 0, 1, 2])))
    else:
        opt.update(nu_multiple=min(int(rng.choice([8, 16])), 4096 // B), nu_phase=int(rng.integers(0, 16)))
    ctx = T.TANContext(device=0)
    objs = [T.TANConvolution(ctx, **opt) for _ in range(2)]
    for o in objs:
        assert o.InitGpu(METHODS[method], L, B, C) == T.AMF_OK
    assert lib.tanx_conv_set_fused(objs[1].handle, 0) == T.AMF_OK
    cap = 24 * steps
    x = rng.uniform(-1, 1, (C, cap * B)).astype(np.float32)
    xd, ys = simlib.Dev(C, cap * B, x), [simlib.Dev(C, cap * B, 0.0) for _ in objs]
    host = [np.zeros((C, B), np.float32) for _ in objs]
    vp, sz = ctypes.c_void_p, ctypes.c_size_t
    t, k = 0, 0
    for step in range(steps):
        if step == 0 or rng.random() < 0.3:
            h = T.signals.ir_bank(C, L, k, base_seed=50 + seed)
            k += 1
            dev = simlib.Dev(C, L, h)
            rcs = [lib.tanx_conv_update_td_device(o.handle, dev.ptr, L, L, None, 0) for o in objs]
            assert rcs[0] == rcs[1] and rcs[0] in (T.AMF_OK, T.AMF_INPUT_FULL), rcs
            dev.free()
        if rng.random() < 0.15:
            assert lib.tanx_conv_set_tail_chunks(objs[0].handle, int(rng.integers(0, 9))) == T.AMF_OK
        if rng.random() < 0.08:
            ch = int(rng.integers(0, C))
            for o in objs:
                assert lib.tanx_conv_flush(o.handle, ch) == T.AMF_OK
        what = rng.choice(["call", "call", "call", "one", "one", "host", "group", "stop"])
        n = int(rng.integers(2, 24)) if what == "call" else 1
        if what == "stop":
            flags = np.zeros(C, np.uint32)
            flags[int(rng.integers(0, C))] = T.TAN_CONVOLUTION_CHANNEL_FLAG_STOP_INPUT
            n = int(rng.integers(1, 4))
        for i, (o, y) in enumerate(zip(objs, ys)):
            if what in ("call", "one", "stop"):
                fp = flags.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)) if what == "stop" else None
                for b in range(t, t + n, n if i == 0 else 1):
                    rc = lib.tanx_conv_process_device(o.handle, xd.at(b * B), xd.stride, y.at(b * B), y.stride,
                                                      (n if i == 0 else 1) * B, fp, ctypes.byref(_done))
                    assert rc == T.AMF_OK or (what == "stop" and rc == T.AMF_WRONG_STATE), (what, rc)
            elif what == "host":
                rc, _ = o.Process(np.ascontiguousarray(x[:, t * B:(t + 1) * B]), host[i], B)
                assert rc == T.AMF_OK
                y.a[:, t * B:(t + 1) * B] = host[i]
            else:
                assert lib.tanx_group_process_device(1, (vp * 1)(o.handle.value), (vp * 1)(xd.at(t * B)),
                                                     (sz * 1)(xd.stride), (vp * 1)(y.at(t * B)), (sz * 1)(y.stride),
                                                     None) == T.AMF_OK
        t += n
        e = float(np.abs(ys[0].a[:, :t * B].astype(np.float64) - ys[1].a[:, :t * B]).max())
        assert e <= 2e-6, (step, what, n, t, e)  # outputs up to 3, as in test_gpu_passes.py
    assert [o.Info()["ticks"] for o in objs][0] == objs[1].Info()["ticks"]
    assert objs[0].Info()["crossfades"] == objs[1].Info()["crossfades"]
    assert np.abs(ys[1].a).max() > 0.1
    print(f"seed {seed}: {t} blocks of {C} channels, B={B}, {parts} partitions, {opt}", flush=True)


def next_block(method=0, L=65536, B=256, C=3, kp=0):
    """A call leaves the sums of the block after it computed: that block is
    one launch, whatever the call's length."""
    ctx = T.TANContext(device=0)
    conv = T.TANConvolution(ctx, **({"pass_blocks": kp} if method == 0 else {"nu_multiple": 16}))
    assert conv.InitGpu(METHODS[method], L, B, C) == T.AMF_OK
    update(conv, T.signals.ir_bank(C, L, 0, base_seed=61))
    assert conv.EnableTiming(True) == T.AMF_OK
    xd, yd = simlib.Dev(C, 70 * B, 0.5), simlib.Dev(C, 70 * B, 0.0)
    for n in (1, 2, 4, 5, 8, 11, 16, 17, 24, 64, 70):
        call(conv, xd, yd, 0, n, B)
        conv.ReadTiming(reset=True)
        call(conv, xd, yd, 0, 1, B)
        rt = conv.ReadTiming(reset=True)
        assert rt["head_launches"] + rt["tail_launches"] == 1, (n, rt)


if __name__ == "__main__":
    globals()[sys.argv[1]](**{k: int(v) for k, v in (a.split("=") for a in sys.argv[2:])})
    print("scenario complete", flush=True)
