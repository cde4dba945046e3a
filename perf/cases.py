"""The work this framework is measured on: its public entry points as an audio
renderer calls them, over the sizes they are used at.

Every case is a dict of plain values with a "kind":

  host      Process on host arrays, one block per call (the reference's own
            usage: a caller without a GPU pipeline of its own)
  stream    Process on device arrays, `blocks` blocks per call, optionally with
            UpdateResponseTD to a fresh response before the call (a switch with
            its crossfade falls into the call)
  render    one block through the whole output chain: Process, TANMixer to two
            ears, TANConverter to interleaved 16-bit samples
  rig       a node full of channels: objects of equal size on staggered pass
            phases, `pass_blocks` ticks of group launches, with three objects'
            responses replaced along the way
  streams   uneven streams (own response length and block size each), one
            cycle of group launches
  td        the time-domain method (HRTF-length responses)
  fft       TANFFT, one transform of a batch
  room      image-source responses for a batch of listeners

The programs share torch's stream with the context (TANContext(conv_stream=)),
so inputs written by torch and the library's launches follow each other in
stream order.  Responses are Gaussian noise with a 0.25 s decay and unit norm,
inputs uniform white noise in [-1, 1].
"""
import math

import numpy as np
import torch

import tan_amd as T
from tan_amd import batching
from tan_amd import room as R

FS = 48000
UNIFORM = T.TAN_CONVOLUTION_METHOD_FFT_UNIFORM_PARTITIONED
NONUNIFORM = T.TAN_CONVOLUTION_METHOD_FFT_PARTITIONED_NONUNIFORM
TIME_DOMAIN = T.TAN_CONVOLUTION_METHOD_TIME_DOMAIN
BLOCKING = T.TAN_CONVOLUTION_OPERATION_FLAG_BLOCK_UNTIL_READY
METHODS = {"uniform": UNIFORM, "nonuniform": NONUNIFORM, "time": TIME_DOMAIN}
PRECISIONS = {"fp32": T.TAN_IR_PRECISION_FP32, "fp16": T.TAN_IR_PRECISION_FP16, "bf16": T.TAN_IR_PRECISION_BF16}
IR_BYTES = {"fp32": 4, "fp16": 2, "bf16": 2}  # stored bytes per real value of a spectrum
LONGEST_PASS = 16      # blocks one sweep over an object's partitions serves at most
SWITCH_BLOCKS = 2      # an update issued before block b crossfades at block b + 2
WARM_CYCLES = 16       # cycles of 512 samples the uneven streams have run for
ROOM = (10.0, 4.0, 8.0)


def listed():
    return [
        # the reference's own test program: stereo, host buffers, one block at a time
        {"name": "host_stereo", "kind": "host", "channels": 2, "taps": 16384, "block": 1024},
        # a VR scene's audio callback: 32 sources x 2 ears, mixed and converted every block
        {"name": "render_64ch", "kind": "render", "channels": 64, "taps": 65536, "block": 256},
        # offline or buffered rendering: several blocks per call
        {"name": "stream_64ch_16blk", "kind": "stream", "method": "uniform", "precision": "fp32", "channels": 64,
         "taps": 65536, "block": 256, "blocks": 16, "update": False},
        # moving sources: a fresh response and its crossfade within a short call
        {"name": "switch_64ch_8blk", "kind": "stream", "method": "uniform", "precision": "fp32", "channels": 64,
         "taps": 65536, "block": 256, "blocks": 8, "update": True},
        # a node that carries as many channels as it can, the largest work here
        {"name": "rig_12x1024", "kind": "rig", "objects": 12, "channels": 1024, "taps": 65536, "block": 256,
         "pass_blocks": 12},
        # many independent mono streams of uneven response length and block size
        {"name": "streams_512", "kind": "streams", "count": 512, "min_taps": 4096, "max_taps": 262144, "plan": 7},
        # long responses stored in 16 bits
        {"name": "long_1024ch_fp16", "kind": "stream", "method": "uniform", "precision": "fp16", "channels": 1024,
         "taps": 131072, "block": 256, "blocks": 8, "update": False},
        # cathedral-length responses at low latency: odd channel count, ragged length
        {"name": "nonuniform_63ch", "kind": "stream", "method": "nonuniform", "precision": "fp32", "channels": 63,
         "taps": 250007, "block": 128, "blocks": 16, "update": False},
        # binaural filters of many sources
        {"name": "hrtf_512ch", "kind": "td", "channels": 512, "taps": 512, "block": 256, "blocks": 1},
        # spectra of blocks of audio, the planar layout the reference's engine uses
        {"name": "fft_2k_1000ch", "kind": "fft", "direction": 4, "log2len": 11, "channels": 1000},
        # whole recordings, there and back in one buffer layout
        {"name": "fft_256k_12ch", "kind": "fft", "direction": 0, "log2len": 18, "channels": 12},
        # responses of a moving listener group in one shoebox room
        {"name": "room_32", "kind": "room", "count": 32, "taps": 65536},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _odd(rng, n):
    return max(1, n | 1) if rng.random() < 0.5 else n


def draw(rng):
    kind = rng.choice(["host", "stream", "stream", "stream", "render", "rig", "streams", "td", "fft", "fft", "room"])
    if kind == "host":
        return {"kind": kind, "channels": _odd(rng, _log_int(rng, 1, 32)), "taps": _log_int(rng, 1000, 100000),
                "block": rng.choice([64, 128, 256, 512, 1024])}
    if kind == "render":
        return {"kind": kind, "channels": 2 * _log_int(rng, 4, 128), "taps": _log_int(rng, 8192, 131072),
                "block": rng.choice([128, 256, 512])}
    if kind == "stream":
        method = rng.choice(["uniform", "uniform", "nonuniform"])
        taps = _log_int(rng, 4096, 262144)
        return {"kind": kind, "method": method, "precision": rng.choice(["fp32", "fp32", "fp16", "bf16"]),
                "channels": _odd(rng, _log_int(rng, 1, min(1024, (1 << 26) // taps))), "taps": taps,
                "block": rng.choice([64, 128, 256, 256, 512, 1024]), "blocks": _log_int(rng, 1, 24),
                "update": method == "uniform" and rng.random() < 0.4}
    if kind == "rig":
        return {"kind": kind, "objects": rng.randint(4, 12), "channels": _odd(rng, _log_int(rng, 64, 800)),
                "taps": _log_int(rng, 16384, 65536), "block": rng.choice([128, 256, 512]),
                "pass_blocks": rng.choice([4, 8, 12])}
    if kind == "streams":
        return {"kind": kind, "count": _log_int(rng, 32, 700), "min_taps": 4096,
                "max_taps": _log_int(rng, 16384, 262144), "plan": rng.randint(1, 1 << 20)}
    if kind == "td":
        return {"kind": kind, "channels": _odd(rng, _log_int(rng, 2, 2048)), "taps": _log_int(rng, 64, 2048),
                "block": rng.choice([64, 128, 256, 512, 1024]), "blocks": rng.randint(1, 4)}
    if kind == "fft":
        direction, log2len = rng.randint(0, 5), rng.randint(6, 19)
        return {"kind": kind, "direction": direction, "log2len": log2len,
                "channels": _odd(rng, _log_int(rng, 1, min(4096, (1 << 23) >> log2len)))}
    return {"kind": kind, "count": rng.randint(1, 40), "taps": _log_int(rng, 8192, 65536)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _generator(seed, stage=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * (int(seed) + 1) + stage)
    return g


def _responses(gen, channels, taps):
    t = torch.arange(taps, device="cuda", dtype=torch.float32)
    h = torch.randn(channels, taps, device="cuda", generator=gen).mul_(torch.exp(-t / (0.25 * FS)))
    return h.div_(h.norm(dim=1, keepdim=True))


def _noise(gen, channels, n):
    return torch.empty(channels, n, device="cuda").uniform_(-1.0, 1.0, generator=gen)


def _warm_blocks(case):
    """Blocks run before the measured pass: the delay line is full and the
    first response has faded in (for frames too: at most 4,096 samples)."""
    n = -(-case["taps"] // case["block"]) + 4
    if case.get("method") == "nonuniform":
        n += 3 * (4096 // case["block"] + 1)
    return n


def _stream_inputs(case, seed):
    """(old responses, new responses or None, input of the warm-up, input of the pass)"""
    gen = _generator(seed)
    c, b = case["channels"], case["block"]
    old = _responses(gen, c, case["taps"])
    new = _responses(gen, c, case["taps"]) if case.get("update") else None
    return old, new, _noise(gen, c, _warm_blocks(case) * b), _noise(gen, c, case.get("blocks", 1) * b)


def _rig_updates(case):
    """{tick: object} of the responses replaced in one pass (the next pass takes the next three objects)."""
    n = case["pass_blocks"]
    return {0: 0, n // 3: 1, 2 * n // 3: 2}


def _rig_inputs(case, seed, o):
    """Responses, warm-up input and the pass's input of object o."""
    gen = _generator(seed, 1 + o)
    c, b = case["channels"], case["block"]
    return (_responses(gen, c, case["taps"]), _noise(gen, c, _warm_blocks(case) * b),
            _noise(gen, c, case["pass_blocks"] * b))


def _rig_bank(case, seed, k):
    return _responses(_generator(seed, 1000 + k), case["channels"], case["taps"])


def _streams_plan(case):
    return batching.draw_streams(case["count"], seed=case["plan"], min_len=case["min_taps"], max_len=case["max_taps"])


def _fft_inputs(case, seed):
    """Rows of 2^(log2len + 1) floats as TANFFT takes them: complex noise, real
    noise, or (inverse real directions) the spectrum of real noise."""
    gen = _generator(seed)
    n, c, d = 1 << case["log2len"], case["channels"], case["direction"]
    x = torch.zeros(c, 2 * n, device="cuda")
    if d < 2:
        x.normal_(generator=gen)
    elif d in (2, 4):
        x[:, :n].normal_(generator=gen)
    else:
        m = n // 2
        re = torch.randn(c, m + 1, device="cuda", generator=gen)
        im = torch.randn(c, m + 1, device="cuda", generator=gen)
        im[:, 0] = 0.0
        im[:, m] = 0.0
        if d == 3:
            x[:, 0:n + 2:2], x[:, 1:n + 2:2] = re, im
        else:
            x[:, :m + 1], x[:, m + 8:2 * m + 9] = re, im
    return x


def _room_scene(case, seed):
    rng = np.random.default_rng(seed)
    room = R.make_room(*ROOM, 0.9, damp_bottom=0.6, damp_top=0.7)
    n = case["count"]
    sources = [R.MonoSource(*rng.uniform([0.5, 0.5, 0.5], [9.5, 3.5, 7.5])) for _ in range(n)]
    listeners = [R.make_listener(tuple(rng.uniform([1.0, 1.2, 1.0], [9.0, 2.0, 7.0])), 0.16,
                                 float(rng.uniform(-180, 180))) for _ in range(n)]
    return [room] * n, sources, listeners


# ---------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------
_stream = None


def _context():
    """A context on the stream the program works on (made torch's current one)."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    torch.cuda.set_stream(_stream)
    return T.TANContext(conv_stream=_stream, general_stream=_stream)


def _ok(rc):
    if isinstance(rc, tuple):
        rc = rc[0]
    if rc != T.AMF_OK:
        raise RuntimeError(f"AMF_RESULT {rc}")


def _convolution(ctx, method, taps, block, channels, **options):
    conv = T.TANConvolution(ctx, **options)
    _ok(conv.InitGpu(method, taps, block, channels))
    return conv


def prepare(case, seed):
    kind = case["kind"]
    ctx = _context()
    s = {"case": case, "ctx": ctx}
    if kind in ("host", "stream", "render", "td"):
        method = METHODS["time" if kind == "td" else case.get("method", "uniform")]
        conv = _convolution(ctx, method, case["taps"], case["block"], case["channels"],
                            ir_precision=PRECISIONS[case.get("precision", "fp32")])
        old, new, warm, x = _stream_inputs(case, seed)
        if kind == "host":
            # host arrays throughout, as such a program has nothing on the device
            _ok(conv.UpdateResponseTD(old.cpu().numpy(), case["taps"], None, BLOCKING))
            b, w = case["block"], warm.cpu().numpy()
            out = np.zeros((case["channels"], b), np.float32)
            for k in range(w.shape[1] // b):
                _ok(conv.Process(np.ascontiguousarray(w[:, k * b:(k + 1) * b]), out, b))
            s.update(conv=conv, x=x.cpu().numpy(), y=out)
            return s
        _ok(conv.UpdateResponseTD(old, case["taps"], None, BLOCKING))
        _ok(conv.Process(warm, torch.empty_like(warm)))
        s.update(conv=conv, x=x, y=torch.empty_like(x), new=new)
        if kind == "render":
            half = case["channels"] // 2
            s["mixers"] = [T.TANMixer(ctx), T.TANMixer(ctx)]
            for m in s["mixers"]:
                _ok(m.Init(case["block"], half))
            s["converter"] = T.TANConverter(ctx)
            s["ears"] = [torch.empty(case["block"], device="cuda") for _ in range(2)]
            s["pcm"] = torch.empty(2 * case["block"], device="cuda", dtype=torch.int16)
    elif kind == "rig":
        b, n = case["block"], case["pass_blocks"]
        s["convs"], s["x"], s["y"] = [], [], []
        for o in range(case["objects"]):
            conv = _convolution(ctx, UNIFORM, case["taps"], b, case["channels"], pass_blocks=n, pass_phase=o % n,
                                max_tail_chunks=1, ir_slots=2)
            h, warm, x = _rig_inputs(case, seed, o)
            _ok(conv.UpdateResponseTD(h, case["taps"], None, BLOCKING))
            _ok(conv.Process(warm, torch.empty_like(warm)))
            s["convs"].append(conv)
            s["x"].append(x)
            s["y"].append(torch.empty_like(x))
        s["calls"] = [batching.GroupCall(s["convs"], [x[:, t * b:(t + 1) * b] for x in s["x"]],
                                         [y[:, t * b:(t + 1) * b] for y in s["y"]]) for t in range(n)]
        s["banks"] = [_rig_bank(case, seed, k) for k in range(3)]
        s["turn"] = 0
    elif kind == "streams":
        specs = _streams_plan(case)
        gen = _generator(seed)
        _, periods, phases, cycle = batching.phase_plan([b for _, b in specs])
        n, span = len(specs), max(b for _, b in specs)
        warm, x = _noise(gen, n, WARM_CYCLES * span), _noise(gen, n, span)
        arena, y = torch.empty(n, span, device="cuda"), torch.empty(n, span, device="cuda")
        convs = []
        for taps, b in specs:
            conv = _convolution(ctx, UNIFORM, taps, b, 1)
            _ok(conv.UpdateResponseTD(_responses(gen, 1, taps), taps, None, BLOCKING))
            convs.append(conv)

        def call(t):
            due = [j for j in range(n) if t % periods[j] == phases[j]]
            at = {j: (t // periods[j]) * specs[j][1] for j in due}
            return batching.GroupCall([convs[j] for j in due],
                                      [arena[j:j + 1, at[j]:at[j] + specs[j][1]] for j in due],
                                      [y[j:j + 1, at[j]:at[j] + specs[j][1]] for j in due])

        s.update(convs=convs, arena=arena, y=y, calls=[call(t) for t in range(cycle)])
        for k in range(WARM_CYCLES):
            arena.copy_(warm[:, k * span:(k + 1) * span])
            run(s)
        arena.copy_(x)
    elif kind == "fft":
        s["fft"] = T.TANFFT(ctx)
        _ok(s["fft"].Init())
        s["x"] = _fft_inputs(case, seed)
        s["y"] = torch.zeros_like(s["x"])
    else:
        s["scene"] = _room_scene(case, seed)
        s["y"] = torch.zeros(2 * case["count"], case["taps"], device="cuda")
    return s


# ---------------------------------------------------------------------------
# run
# ---------------------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("host", "stream", "td"):
        if s.get("new") is not None:
            _ok(s["conv"].UpdateResponseTD(s["new"]))
        _ok(s["conv"].Process(s["x"], s["y"]))
        return s["y"]
    if kind == "render":
        half, b = case["channels"] // 2, case["block"]
        _ok(s["conv"].Process(s["x"], s["y"]))
        for ear in range(2):
            _ok(s["mixers"][ear].Mix(s["y"][ear * half:(ear + 1) * half], s["ears"][ear]))
            _ok(s["converter"].Convert(s["ears"][ear], 1, b, s["pcm"], 2, 0.25, 0, ear, want_clipped=False))
        return {"channels": s["y"], "ears": s["ears"], "pcm": s["pcm"]}
    if kind == "rig":
        updates = _rig_updates(case)
        for t, call in enumerate(s["calls"]):
            if t in updates:
                o = (s["turn"] + updates[t]) % case["objects"]
                _ok(T.GroupUpdateResponseTD([s["convs"][o]], [s["banks"][updates[t]]]))
            _ok(call.launch())
        s["turn"] = (s["turn"] + 3) % case["objects"]
        return s["y"]
    if kind == "streams":
        for call in s["calls"]:
            _ok(call.launch())
        return s["y"]
    if kind == "fft":
        _ok(s["fft"].Transform(case["direction"], case["log2len"], case["channels"], s["x"], s["y"]))
        return s["y"]
    _ok(R.GenerateRoomResponses(s["ctx"], *s["scene"], FS, case["taps"], s["y"]))
    return s["y"]


# ---------------------------------------------------------------------------
# work: what one pass cannot do without
# ---------------------------------------------------------------------------
def _conv_work(channels, taps, block, blocks, ir_bytes, update):
    # a response and the history it multiplies, read once per longest pass;
    # input and output of every block; an update reads a response and writes its spectra
    rows = channels * taps * (ir_bytes + 4) * blocks / LONGEST_PASS
    io = 8 * channels * block * blocks
    new = channels * taps * (4 + 2 * ir_bytes) if update else 0
    transforms = 2 * 2.5 * 2 * block * math.log2(2 * block) * channels * blocks
    return {"bytes": rows + io + new, "flops": 8 * channels * taps * blocks / LONGEST_PASS + transforms}


def work(case):
    kind = case["kind"]
    if kind in ("host", "stream", "render"):
        return _conv_work(case["channels"], case["taps"], case["block"], case.get("blocks", 1),
                          IR_BYTES[case.get("precision", "fp32")], case.get("update", False))
    if kind == "rig":
        one = _conv_work(case["channels"], case["taps"], case["block"], case["pass_blocks"], 4, False)
        new = _conv_work(case["channels"], case["taps"], case["block"], 0, 4, True)
        return {k: case["objects"] * one[k] + 3 * new[k] for k in one}
    if kind == "streams":
        specs = _streams_plan(case)
        span = max(b for _, b in specs)
        each = [_conv_work(1, taps, b, span // b, 4, False) for taps, b in specs]
        return {k: sum(e[k] for e in each) for k in ("bytes", "flops")}
    if kind == "td":
        n = case["block"] * case["blocks"]
        return {"bytes": 4 * case["channels"] * (2 * case["taps"] + 2 * n),
                "flops": 2 * case["channels"] * case["taps"] * n}
    if kind == "fft":
        n, real = 1 << case["log2len"], case["direction"] >= 2
        return {"bytes": case["channels"] * (8 * n if real else 16 * n),
                "flops": case["channels"] * (2.5 if real else 5) * n * case["log2len"]}
    # images within the sphere the response's length reaches, about 40 operations each
    reach = case["taps"] / FS * R.SPEED_OF_SOUND
    images = 4 / 3 * math.pi * reach ** 3 / (ROOM[0] * ROOM[1] * ROOM[2])
    rows = 2 * case["count"]
    return {"bytes": 4 * rows * case["taps"], "flops": 40 * rows * images}


# ---------------------------------------------------------------------------
# exact: the same outputs in 64 bits
# ---------------------------------------------------------------------------
def _convolve(h, history, n):
    """The last n samples of history * h, per row, in 64 bits (rows in slices
    that keep the transforms' memory small)."""
    out = torch.empty(h.shape[0], n, dtype=torch.float64, device=h.device)
    keep = min(history.shape[1], h.shape[1] - 1 + n)
    size = 1 << (keep + h.shape[1] - 2).bit_length()
    rows = max(1, (1 << 24) // size)
    for r in range(0, h.shape[0], rows):
        x = torch.fft.rfft(history[r:r + rows, -keep:].double(), size)
        y = torch.fft.irfft(x * torch.fft.rfft(h[r:r + rows].double(), size), size)
        out[r:r + rows] = y[:, keep - n:keep]
    return out


def _switched(old, new, history, n, block, at):
    """The last n samples with the crossfade from old to new in the block that starts `at` samples into them."""
    y = _convolve(old, history, n)
    if new is not None and at < n:
        z = _convolve(new, history, n)
        j = torch.arange(block, device=y.device, dtype=torch.float64) / block
        y[:, at:at + block] = z[:, at:at + block] * j + y[:, at:at + block] * (1 - j)
        y[:, at + block:] = z[:, at + block:]
    return y


def exact(case, seed):
    kind = case["kind"]
    if kind in ("host", "stream", "render", "td"):
        old, new, warm, x = _stream_inputs(case, seed)
        y = _switched(old, new, torch.cat([warm, x], 1), x.shape[1], case["block"], SWITCH_BLOCKS * case["block"])
        if kind == "render":
            half = case["channels"] // 2
            return {"channels": y, "ears": [y[:half].sum(0), y[half:].sum(0)], "pcm": None}
        return y
    if kind == "rig":
        # the three objects whose responses change, and one that keeps its own
        b, outs = case["block"], [None] * case["objects"]
        ticks = {o: t for t, o in _rig_updates(case).items()}
        for o in (0, 1, 2, 3):
            h, warm, x = _rig_inputs(case, seed, o)
            bank = _rig_bank(case, seed, o) if o in ticks else None
            outs[o] = _switched(h, bank, torch.cat([warm, x], 1), x.shape[1], b,
                                (ticks.get(o, 0) + SWITCH_BLOCKS) * b)
        return outs
    if kind == "streams":
        specs = _streams_plan(case)
        gen = _generator(seed)
        n, span = len(specs), max(b for _, b in specs)
        warm, x = _noise(gen, n, WARM_CYCLES * span), _noise(gen, n, span)
        history = torch.cat([warm, x], 1)
        return torch.cat([_convolve(_responses(gen, 1, taps), history[j:j + 1], span)
                          for j, (taps, _) in enumerate(specs)])
    if kind == "fft":
        x, n, d = _fft_inputs(case, seed).double(), 1 << case["log2len"], case["direction"]
        y, m = torch.zeros_like(x), n // 2
        if d < 2:
            z = torch.view_as_complex(x.reshape(-1, n, 2))
            z = torch.fft.fft(z) if d == 0 else torch.fft.ifft(z)
            return torch.view_as_real(z).reshape(-1, 2 * n)
        if d in (2, 4):
            z = torch.fft.rfft(x[:, :n])
            if d == 2:
                y[:, 0:n + 2:2], y[:, 1:n + 2:2] = z.real, z.imag
            else:
                y[:, :m + 1], y[:, m + 8:2 * m + 9] = z.real, z.imag
            return y
        z = (torch.complex(x[:, 0:n + 2:2], x[:, 1:n + 2:2]) if d == 3
             else torch.complex(x[:, :m + 1], x[:, m + 8:2 * m + 9]))
        y[:, :n] = torch.fft.irfft(z, n)
        return y
    # a room response is a sum of single-precision arrival times and fixed-point gains: no 64-bit value
    return None
