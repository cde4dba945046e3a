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
