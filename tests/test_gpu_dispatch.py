"""Transforms, mixes and time-domain blocks at the sizes where their dispatch
turns from one kernel to another, against FP64."""
import numpy as np
import pytest

import tan_amd as T

pytestmark = pytest.mark.gpu


# (complex points, channels): below and above the lines of each direction,
# channel counts that leave a workgroup part empty
@pytest.mark.parametrize("log2m,C", [(6, 1001), (7, 1535), (7, 1537), (8, 767), (8, 769), (8, 3907), (9, 383), (9, 385),
                                     (9, 1955), (10, 191), (10, 977), (11, 97), (11, 489)])
@pytest.mark.parametrize("direction", range(6))
def test_fft_dispatch(gpu_ctx, log2m, C, direction):
    import torch
    log2n = log2m if direction < 2 else log2m + 1
    n, m = 1 << log2n, 1 << (log2n - 1)
    g = torch.Generator(device="cuda").manual_seed(100 * log2m + direction)
    x = torch.zeros(C, 2 * n, device="cuda")
    if direction < 3 or direction == 4:
        x[:, :2 * n if direction < 2 else n].normal_(generator=g)
    else:
        re = torch.randn(C, m + 1, device="cuda", generator=g)
        im = torch.randn(C, m + 1, device="cuda", generator=g)
        im[:, 0] = im[:, m] = 0
        if direction == 3:
            x[:, 0:n + 2:2], x[:, 1:n + 2:2] = re, im
        else:
            x[:, :m + 1], x[:, m + 8:2 * m + 9] = re, im
    out = torch.full_like(x, 9.0)
    f = T.TANFFT(gpu_ctx)
    assert f.Init() == T.AMF_OK
    assert f.Transform(direction, log2n, C, x, out) == T.AMF_OK
    # every channel through torch's FP64 transforms
    d = x.double()
    if direction < 2:
        z = torch.view_as_complex(d.reshape(C, n, 2))
        ref = torch.view_as_real(torch.fft.fft(z) if direction == 0 else torch.fft.ifft(z)).reshape(C, 2 * n)
        got = out.double()
    elif direction in (2, 4):
        z = torch.fft.rfft(d[:, :n])
        ref = torch.cat([z.real, z.imag], 1)
        got = (torch.cat([out[:, 0:n + 2:2], out[:, 1:n + 2:2]], 1) if direction == 2
               else torch.cat([out[:, :m + 1], out[:, m + 8:2 * m + 9]], 1)).double()
    else:
        ref, got = torch.fft.irfft(torch.complex(re.double(), im.double()), n), out[:, :n].double()
    assert (got - ref).abs().max() <= 3e-7 * ref.abs().max() * log2n  # the bound of test_gpu_fft.py


@pytest.mark.parametrize("n,channels", [(1, 2), (255, 1), (257, 3), (1000, 4), (64, 5), (256, 8), (300, 9), (65, 17),
                                        (1048577, 1), (1050000, 3), (1048577, 18)])
def test_mix_batches(gpu_ctx, n, channels):
    import torch
    d = torch.randn(channels, n + 3, device="cuda", generator=torch.Generator(device="cuda").manual_seed(n))
    ref = d[0, :n].clone()
    for c in range(1, channels):
        ref = ref + d[c, :n]
    m = T.TANMixer(gpu_ctx)
    assert m.Init(n, channels) == T.AMF_OK
    for inputs in (d, [d[c] for c in range(channels)]):
        out = torch.full((n + 2,), 5.0, device="cuda")
        assert m.Mix(inputs, out) == T.AMF_OK
        torch.cuda.synchronize()
        assert torch.equal(out[:n], ref) and (out[n:] == 5.0).all()
    m.Terminate()


# one, two and four outputs per lane, taps shared between idle lanes
@pytest.mark.parametrize("L,B,C", [(64, 64, 3), (128, 64, 1030), (256, 64, 5), (128, 128, 2), (256, 128, 1030),
                                   (512, 64, 2)])
def test_time_domain_blocks(gpu_ctx, L, B, C):
    """Blocks with a switch in between, against the FP64 crossfade model."""
    import torch

    from helpers import crossfade_model
    nb, pick = 12, sorted({0, C // 2, C - 1})
    g = torch.Generator(device="cuda").manual_seed(L + B)
    x = torch.empty(C, nb * B, device="cuda").uniform_(-1, 1, generator=g)
    irs = [torch.randn(C, L, device="cuda", generator=g) / L ** 0.5 for _ in range(2)]
    conv = T.TANConvolution(gpu_ctx)
    assert conv.InitGpu(T.TAN_CONVOLUTION_METHOD_TIME_DOMAIN, L, B, C) == T.AMF_OK
    y = torch.zeros_like(x)
    for b in range(nb):
        if b in (0, 6):
            assert conv.UpdateResponseTD(irs[b // 6], L) == T.AMF_OK
        rc, done = conv.Process(x[:, b * B:(b + 1) * B], y[:, b * B:(b + 1) * B])
        assert rc == T.AMF_OK and done == B
    conv.Synchronize()
    conv.Terminate()
    for c in pick:
        ref = crossfade_model(x[c].cpu().numpy(), [h[c].cpu().numpy() for h in irs], [2, 8], B)
        # eight sums of at most L / 8 products of magnitude below 4 / sqrt(L), and their tree
        assert np.abs(y[c].cpu().numpy() - ref).max() <= 2 * (L / 8 + 4) * 2.0 ** -24 * 4 * L ** 0.5
