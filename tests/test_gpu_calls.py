"""Device calls of several blocks: buffers, shapes and orders of calls at which
the call path and the paths for single blocks have to agree."""
import numpy as np
import pytest

import tan_amd as T

pytestmark = pytest.mark.gpu
UNIFORM = T.TAN_CONVOLUTION_METHOD_FFT_UNIFORM_PARTITIONED
NONUNIFORM = T.TAN_CONVOLUTION_METHOD_FFT_PARTITIONED_NONUNIFORM
TIME_DOMAIN = T.TAN_CONVOLUTION_METHOD_TIME_DOMAIN


def _run(conv, x, y, calls, B, before=None):
    """Calls of the given lengths on conv (x is y: in place); before: call ->
    function of the object run before it."""
    t = 0
    for i, n in enumerate(calls):
        if before and i in before:
            before[i](conv)
        rc, done = conv.Process(x[:, t * B:(t + n) * B], y[:, t * B:(t + n) * B])
        assert rc == T.AMF_OK and done == n * B
        t += n
    conv.Synchronize()
    return y.cpu().numpy()


def _update(h):
    def issue(conv):
        assert conv.UpdateResponseTD(h, h.shape[1]) == T.AMF_OK
    return issue


# waves and whole workgroups per block, a ring of frames, several launches per call
@pytest.mark.parametrize("method,L,B", [(UNIFORM, 4096, 64), (UNIFORM, 65536, 512), (NONUNIFORM, 16384, 64),
                                        (NONUNIFORM, 65536, 1024), (TIME_DOMAIN, 500, 128)])
def test_in_place(gpu_ctx, method, L, B):
    """Calls whose output is their input's buffer give what separate buffers do."""
    import torch
    calls = [4, 8, 1, 8, 40, 3, 16, 2, 24]
    C, nb = 5, sum(calls)
    x = torch.from_numpy(T.signals.input_bank(C, nb * B, base_seed=11)).cuda()
    before = {i: _update(T.signals.ir_bank(C, L, k, base_seed=12)) for k, i in enumerate((0, 3, 6))}
    ys = []
    for same in (False, True):
        conv = T.TANConvolution(gpu_ctx)
        assert conv.InitGpu(method, L, B, C) == T.AMF_OK
        xd = x.clone()
        ys.append(_run(conv, xd, xd if same else torch.zeros_like(xd), calls, B, before))
        conv.Terminate()
    assert np.abs(ys[0]).max() > 0.1
    np.testing.assert_array_equal(ys[0], ys[1])


@pytest.mark.parametrize("P,kp,B", [(1, 4, 64), (2, 4, 64), (4, 16, 64), (8, 4, 128), (4, 4, 1024), (8, 12, 512)])
def test_few_partitions(gpu_ctx, P, kp, B):
    """Objects with fewer partitions than their calls have blocks, a response
    issued before some calls: as one block per call."""
    import torch
    calls = [5, 24, 1, 16, 8, 33, 4, 7]
    C, nb = 3, sum(calls)
    starts = np.cumsum([0] + calls)
    x = torch.from_numpy(T.signals.input_bank(C, nb * B, base_seed=21)).cuda()
    ups = {i: _update(T.signals.ir_bank(C, P * B, k, base_seed=22)) for k, i in enumerate((0, 3, 5))}
    ys = []
    for sizes, before in ((calls, ups), ([1] * nb, {int(starts[i]): u for i, u in ups.items()})):
        conv = T.TANConvolution(gpu_ctx, pass_blocks=kp)
        assert conv.InitGpu(UNIFORM, P * B, B, C) == T.AMF_OK
        ys.append(_run(conv, x, torch.zeros_like(x), sizes, B, before))
        conv.Terminate()
    assert np.abs(ys[1]).max() > 0.1
    assert np.abs(ys[0].astype(np.float64) - ys[1]).max() <= 2e-6  # outputs up to 3, as in test_gpu_passes.py


@pytest.mark.parametrize("method,L,B,mult", [(UNIFORM, 32768, 64, 0), (NONUNIFORM, 32768, 64, 64),
                                             (NONUNIFORM, 65536, 256, 16)])
def test_chunk_changes(gpu_ctx, method, L, B, mult):
    """The tail chunk count set between a call of several blocks and the next
    block: as one block per call with the default count."""
    import torch
    # (the first call: a non-uniform object's response fades in up to three frames later)
    calls, chunks = [200, 8, 1, 7, 1, 1, 9, 1, 6, 2, 12, 1], {2: 4, 4: 1, 5: 0, 7: 3, 9: 2, 11: 8}
    C, nb = 3, sum(calls)
    x = torch.from_numpy(T.signals.input_bank(C, nb * B, base_seed=31)).cuda()
    h = T.signals.ir_bank(C, L, 0, base_seed=32)

    def chunk(n):
        def issue(conv):
            assert conv.SetTailChunks(n) == T.AMF_OK
        return issue

    ys = []
    for sizes, before in ((calls, {i: chunk(n) for i, n in chunks.items()}), ([1] * nb, None)):
        conv = T.TANConvolution(gpu_ctx, nu_multiple=mult)
        assert conv.InitGpu(method, L, B, C) == T.AMF_OK
        _update(h)(conv)
        ys.append(_run(conv, x, torch.zeros_like(x), sizes, B, before))
        conv.Terminate()
    assert np.abs(ys[1]).max() > 0.1
    assert np.abs(ys[0].astype(np.float64) - ys[1]).max() <= 2e-6  # outputs up to 3, as in test_gpu_passes.py


# one bin and two per lane, one filter and a crossfade, chunks of one object's and of many channels
@pytest.mark.parametrize("C,L,B,n,switch", [(64, 65536, 256, 16, False), (256, 65536, 256, 16, False),
                                            (200, 65536, 128, 9, False), (250, 65536, 256, 12, True),
                                            (300, 65536, 512, 16, False), (100, 65536, 512, 9, True)])
def test_error_of_calls(gpu_ctx, C, L, B, n, switch):
    """Calls of several blocks are no further from FP64 than one block per
    call.  Both errors are sums of tens of millions of roundings, which vary
    by a few percent with the order of the sums: 5% is allowed."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(C + n)
    decay = torch.exp(-torch.arange(L, device="cuda") / 12000.0)
    irs = [torch.randn(C, L, device="cuda", generator=g) * decay for _ in range(2)]
    warm = L // B + 4
    x = torch.empty(C, (warm + n) * B, device="cuda").uniform_(-1, 1, generator=g)
    ys = [[], []]
    for way in range(2):
        conv = T.TANConvolution(gpu_ctx)
        assert conv.InitGpu(UNIFORM, L, B, C) == T.AMF_OK
        assert conv.UpdateResponseTD(irs[0], L) == T.AMF_OK
        y = torch.zeros_like(x)
        _run(conv, x, y, [warm], B)
        if switch:
            assert conv.UpdateResponseTD(irs[1], L) == T.AMF_OK
        tail = slice(warm * B, None)
        _run(conv, x[:, tail], y[:, tail], [n] if way == 0 else [1] * n, B)
        ys[way] = y[:, tail].double()
        conv.Terminate()

    def exact(h):
        hist = x[:, -(L + n * B):].double()
        size = 1 << (hist.shape[1] + L).bit_length()
        out = torch.empty(C, n * B, dtype=torch.float64, device="cuda")
        for c in range(0, C, 50):
            f = torch.fft.rfft(hist[c:c + 50], size) * torch.fft.rfft(h[c:c + 50].double(), size)
            out[c:c + 50] = torch.fft.irfft(f, size)[:, L:L + n * B]
        return out

    ref = exact(irs[0])
    if switch:  # the update is handed off by the first block and crossfades in the third
        new, at = exact(irs[1]), 2 * B
        j = torch.arange(B, device="cuda", dtype=torch.float64) / B
        ref[:, at:at + B] = new[:, at:at + B] * j + ref[:, at:at + B] * (1 - j)
        ref[:, at + B:] = new[:, at + B:]
    err = [float((y - ref).norm() / ref.norm()) for y in ys]
    assert err[1] <= 1e-6
    assert err[0] <= 1.05 * err[1], err


@pytest.mark.parametrize("opt", [{}, {"pass_blocks": 8}, {"pass_blocks": 12}, {"nu_multiple": 16}])
def test_next_block(gpu_ctx, opt):
    """A call leaves the sums of the block after it computed: that block is
    one launch, whatever the call's length."""
    import torch
    L, B, C = 65536, 256, 3
    conv = T.TANConvolution(gpu_ctx, **opt)
    assert conv.InitGpu(NONUNIFORM if "nu_multiple" in opt else UNIFORM, L, B, C) == T.AMF_OK
    _update(T.signals.ir_bank(C, L, 0, base_seed=61))(conv)
    assert conv.EnableTiming(True) == T.AMF_OK
    x = torch.rand(C, 70 * B, device="cuda")
    y = torch.empty_like(x)
    for n in (1, 2, 4, 5, 8, 11, 16, 17, 24, 64, 70):
        _run(conv, x, y, [n], B)
        conv.ReadTiming(reset=True)
        _run(conv, x, y, [1], B)
        t = conv.ReadTiming(reset=True)
        assert t["head_launches"] + t["tail_launches"] == 1, (n, t)
    conv.Terminate()
