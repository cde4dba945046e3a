"""Kernels at the sizes where their tiling can go wrong, against FP64."""
import numpy as np
import pytest

import tan_amd as T

pytestmark = pytest.mark.gpu
U = 2.0 ** -24  # unit roundoff of FP32


# lanes compute 2 outputs each below 1,024 waves of 4, 4 each from there on
@pytest.mark.parametrize("L,B,C,calls", [(64, 64, 3, (64, 1, 63, 7)), (500, 256, 2, (255, 3, 250)),
                                         (4096, 1024, 1, (1021, 1024)), (64, 256, 1027, (250, 64, 63)),
                                         (128, 1024, 300, (1021, 5))])
def test_time_domain_ragged_calls_and_tap_ranges(gpu_ctx, L, B, C, calls):
    rng = np.random.default_rng(L + B + C)
    conv = T.TANConvolution(gpu_ctx)
    assert conv.InitGpu(T.TAN_CONVOLUTION_METHOD_TIME_DOMAIN, L, B, C) == T.AMF_OK
    n_ir = conv.Info()["ir_len"]
    h = rng.standard_normal((C, n_ir)).astype(np.float32)
    first = rng.integers(0, 9, C)
    last = n_ir - rng.integers(0, 9, C)
    last[0] = first[0] + 3  # fewer taps than one step of the sums
    if C > 1:
        last[1] = first[1]  # none
    nz = np.stack([first, last], 1).astype(np.int32)
    hz = h.astype(np.float64)
    for c in range(C):
        hz[c, :first[c]] = 0
        hz[c, last[c]:] = 0
    hist = np.zeros((C, n_ir - 1))
    for n in calls:
        n = min(n, n_ir)
        x = rng.uniform(-1, 1, (C, n)).astype(np.float32)
        y = np.full((C, n), 7.0, np.float32)
        rc, done = conv.ProcessDirect(h, x, y, n, nz)
        assert rc == T.AMF_OK and done == n
        full = np.concatenate([hist, x], 1)
        hist = full[:, full.shape[1] - (n_ir - 1):]
        win = np.lib.stride_tricks.sliding_window_view(full, n_ir, axis=1)[:, :, ::-1]
        ref = np.einsum("cnk,ck->cn", win, hz)
        # eight interleaved sums of at most n_ir / 8 products and their tree
        bound = (n_ir / 8 + 4) * U * np.einsum("cnk,ck->cn", np.abs(win), np.abs(hz))
        assert np.all(np.abs(y - ref) <= bound + 1e-30), np.abs(y - ref).max()
    conv.Terminate()


@pytest.mark.parametrize("n,channels", [(1, 1), (63, 15), (64, 16), (65, 17), (256, 32), (1000, 33)])
def test_mix_sums_in_channel_order(gpu_ctx, n, channels):
    import torch
    rng = np.random.default_rng(n + channels)
    x = rng.standard_normal((channels, n + 3)).astype(np.float32)
    ref = x[0, :n].copy()
    for c in range(1, channels):
        ref = ref + x[c, :n]
    m = T.TANMixer(gpu_ctx)
    assert m.Init(n, channels) == T.AMF_OK
    d = torch.from_numpy(x).cuda()
    for inputs in (d, [d[c] for c in range(channels)]):
        out = torch.full((n + 2,), 5.0, device="cuda")
        assert m.Mix(inputs, out) == T.AMF_OK
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy()[:n], ref)
        assert (out[n:] == 5.0).all()
    m.Terminate()


# (taps, block, pass_blocks, max_tail_chunks, precision): as many blocks as
# partitions, rows of several slices, one chunk, 16-bit rows
@pytest.mark.parametrize("L,B,K,chunks,precision", [(16 * 64, 64, 4, 0, 0), (16 * 1024, 1024, 4, 0, 0),
                                                    (300 * 128, 128, 8, 0, 0), (64 * 512, 512, 12, 1, 0),
                                                    (80 * 256, 256, 16, 1, 0), (20 * 1024, 1024, 4, 2, 1),
                                                    (20 * 128, 128, 4, 0, 2)])
def test_calls_of_many_blocks(gpu_ctx, L, B, K, chunks, precision):
    """Calls of 1 to 33 blocks, with a response issued before some of them
    (its crossfade falls into the call, on its first block, or in the next
    one), against the FP64 crossfade model."""
    import torch

    from helpers import crossfade_model, snr_db
    calls = [4, 5, 1, 16, 8, 2, 9, 12, 1, 13, 33, 3, 17]
    at = {0: 0, 3: 1, 4: 2, 5: 3, 7: 4, 9: 5, 10: 6}  # call -> response
    C, nb = 3, sum(calls)
    starts = np.cumsum([0] + calls)
    x = T.signals.input_bank(C, nb * B, base_seed=41)
    irs = [T.signals.ir_bank(C, L, k, base_seed=43) for k in range(len(at))]
    conv = T.TANConvolution(gpu_ctx, ir_precision=precision, pass_blocks=K, max_tail_chunks=chunks)
    assert conv.InitGpu(T.TAN_CONVOLUTION_METHOD_FFT_UNIFORM_PARTITIONED, L, B, C) == T.AMF_OK
    xd = torch.from_numpy(x).cuda()
    yd = torch.zeros_like(xd)
    for i, n in enumerate(calls):
        b = int(starts[i])
        if i in at:
            assert conv.UpdateResponseTD(irs[at[i]], L) == T.AMF_OK
        rc, done = conv.Process(xd[:, b * B:(b + n) * B], yd[:, b * B:(b + n) * B])
        assert rc == T.AMF_OK and done == n * B
    conv.Synchronize()
    conv.Terminate()
    y = yd.cpu().numpy()
    # every switch falls two blocks after its update (none is issued while another is armed)
    sw = [int(starts[i]) + 2 for i in at]
    for c in range(C):
        ref = crossfade_model(x[c], [h[c] for h in irs], sw, B)
        if precision == 0:
            assert np.abs(y[c] - ref).max() <= 1e-5
        assert snr_db(ref, y[c]) >= (120.0, 60.0, 45.0)[precision]


# sizes of each stage plan, channel counts that leave a workgroup part empty,
# rows whose pairs of floats are not 8-byte aligned
@pytest.mark.parametrize("log2m,C,pad,off", [(6, 17, 0, 0), (6, 3, 3, 1), (7, 9, 1, 0), (8, 5, 0, 1), (9, 3, 2, 0),
                                             (10, 2, 5, 1), (11, 3, 1, 1)])
@pytest.mark.parametrize("direction", range(6))
def test_fft_row_layouts(gpu_ctx, log2m, C, pad, off, direction):
    import torch
    log2n = log2m if direction < 2 else log2m + 1
    n, m = 1 << log2n, 1 << (log2n - 1)
    rng = np.random.default_rng(100 * log2m + direction)
    x = rng.standard_normal((C, 2 * n + pad)).astype(np.float32)
    base = torch.zeros(C * (2 * n + pad) + off, device="cuda")
    base[off:] = torch.from_numpy(x).cuda().reshape(-1)
    ob = torch.full_like(base, 9.0)
    xin = base[off:].view(C, 2 * n + pad)
    out = ob[off:].view(C, 2 * n + pad)
    f = T.TANFFT(gpu_ctx)
    assert f.Init() == T.AMF_OK
    assert f.Transform(direction, log2n, C, xin, out) == T.AMF_OK
    got = out.cpu().numpy().astype(np.float64)
    x64 = x.astype(np.float64)
    if direction < 2:
        z = x64[:, 0:2 * n:2] + 1j * x64[:, 1:2 * n:2]
        ref = np.fft.fft(z) if direction == 0 else np.fft.ifft(z)
        g, used = got[:, 0:2 * n:2] + 1j * got[:, 1:2 * n:2], 2 * n
    elif direction in (2, 4):
        ref = np.fft.rfft(x64[:, :n])
        if direction == 2:
            g, used = got[:, 0:n + 2:2] + 1j * got[:, 1:n + 2:2], n + 2
        else:
            g, used = got[:, :m + 1] + 1j * got[:, m + 8:2 * m + 9], 2 * m + 9
            assert np.all(got[:, m + 1:m + 8] == 9.0)
    else:
        z = (x64[:, 0:n + 2:2] + 1j * x64[:, 1:n + 2:2] if direction == 3
             else x64[:, :m + 1] + 1j * x64[:, m + 8:2 * m + 9])
        z[:, 0], z[:, m] = z[:, 0].real, z[:, m].real
        ref, g, used = np.fft.irfft(z, n), got[:, :n], n
    assert np.abs(g - ref).max() <= 3e-7 * np.abs(ref).max() * log2n  # the bound of test_gpu_fft.py
    assert np.all(got[:, used:] == 9.0)


# more cells along x than the table holds; more reflections along y or z than
# the power tables hold; one window and several, ending inside one
@pytest.mark.parametrize("dims,n", [((0.4, 30.0, 40.0), 17000), ((30.0, 0.2, 40.0), 16500), ((40.0, 30.0, 0.2), 9001),
                                    ((3.0, 2.5, 4.0), 8193)])
def test_room_tables_and_windows(gpu_ctx, dims, n):
    import oracle_lib as O
    from tan_amd import room as R
    room = R.make_room(*dims, 0.8, damp_top=0.4)
    src = R.MonoSource(*[0.3 * d for d in dims])
    lst = R.make_listener(tuple(0.6 * d for d in dims), 0.16, 20.0)
    left, right = np.zeros(n, np.float32), np.zeros(n, np.float32)
    assert R.generateRoomResponse(gpu_ctx, room, src, lst, 48000, n, left, right) == T.AMF_OK
    rc, oleft, oright = O.room_response(room, src, lst, 48000, n, 0, 0)
    assert rc == 0
    np.testing.assert_array_equal(left, oleft)
    np.testing.assert_array_equal(right, oright)
    assert np.count_nonzero(left) > 0


# frames of 16, 8 and 64 blocks, a shifted frame clock, one tail chunk, 16-bit rows
@pytest.mark.parametrize("L,B,mult,phase,precision,chunks", [(16384, 64, 16, 0, 0, 0), (20000, 128, 8, 3, 0, 0),
                                                             (9000, 64, 64, 5, 1, 1), (40000, 256, 16, 0, 2, 0),
                                                             (250007, 128, 0, 0, 0, 0), (30000, 1024, 4, 1, 0, 0)])
def test_nonuniform_calls_of_many_blocks(gpu_ctx, L, B, mult, phase, precision, chunks):
    """Calls that cross frame ends and switches equal one block per call (the
    sums of a block are added in another order)."""
    import torch
    calls = [1, 20, 5, 3, 40, 16, 1, 1, 33, 4, 7, 64, 2, 50]
    C, nb = 3, sum(calls)
    starts = np.cumsum([0] + calls)
    ups = {int(starts[i]): T.signals.ir_bank(C, L, k, base_seed=61) for k, i in enumerate((0, 4, 8, 11))}
    x = torch.from_numpy(T.signals.input_bank(C, nb * B, base_seed=70)).cuda()
    ys = []
    for sizes in (calls, [1] * nb):
        conv = T.TANConvolution(gpu_ctx, ir_precision=precision, nu_multiple=mult, nu_phase=phase,
                                max_tail_chunks=chunks)
        assert conv.InitGpu(T.TAN_CONVOLUTION_METHOD_FFT_PARTITIONED_NONUNIFORM, L, B, C) == T.AMF_OK
        y, t = torch.zeros_like(x), 0
        for n in sizes:
            if t in ups:
                assert conv.UpdateResponseTD(ups[t], L) == T.AMF_OK
            rc, done = conv.Process(x[:, t * B:(t + n) * B], y[:, t * B:(t + n) * B])
            assert rc == T.AMF_OK and done == n * B
            t += n
        conv.Synchronize()
        conv.Terminate()
        ys.append(y.cpu().numpy())
    assert np.abs(ys[1]).max() > 1.0
    assert np.abs(ys[0].astype(np.float64) - ys[1]).max() <= 2e-6  # outputs up to 3, as in test_gpu_passes.py
