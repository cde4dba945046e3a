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
