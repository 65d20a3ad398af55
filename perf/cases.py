"""Performance cases of the SuBSENSE / LOBSTER background subtractors: what a program that uses
litiv_amd has it do, through the package's public entry points.

A case is a dict of plain values:
  op        "apply"       apply_device() + synchronize(): one frame that is already in device memory
            "host"        apply(): one frame in host memory, mask back in host memory (the reference's call)
            "batch"       Batch.apply_device() + synchronize(): one frame of every stream of a batch
            "serve"       Server.submit() of one frame per stream, drain(), poll()
            "background"  getBackgroundImage() of a running model
            "initialize"  initialize() of a subtractor from a host frame (opening or resetting a stream)
            "score"       BinClassif.accumulate_device() of a mask against ground truth and ROI
  algo      "subsense" or "lobster"
  width, height, channels; streams and mix (batch, serve: number of streams, choice of their sizes)
  groups    member groups stepped concurrently (batch)
  lr        learning-rate override of apply(), 0 = the algorithm's default
  roi       True: a custom elliptic ROI given to initialize()

A running model is what a program has in hand: prepare() initializes it on the first frame of a
synthetic sequence and steps it over the next WARM frames, so its samples, maps and thresholds are those of
a stream under way (moving objects, sensor noise, a flickering patch, an illumination ramp). A pass
then takes the next frame of a ring of RING consecutive frames. The objects cross a pixel within a few
frames and come back only after the ring, so the model does not absorb them: 3 to 10% of the pixels are
foreground, as in the generator's long sequences, however often the ring goes round.
"""
import math
import random

import numpy as np
import torch

from litiv_amd import BackgroundSubtractorLOBSTER, BackgroundSubtractorSuBSENSE, Batch, BinClassif, Server, synth

RING, WARM = 48, 120
ALGOS = {"subsense": BackgroundSubtractorSuBSENSE, "lobster": BackgroundSubtractorLOBSTER}
# sizes of mixed batches and served streams: (width, height, channels)
MIX = ((320, 240, 3), (640, 480, 3), (640, 512, 1), (1920, 1080, 3))
SERVED = ((320, 240, 3), (320, 240, 3), (320, 240, 3), (640, 480, 3), (640, 480, 3), (640, 480, 3), (1280, 720, 3),
          (1280, 720, 3), (1920, 1080, 3), (1920, 1080, 3))


def _case(name, op, algo="subsense", width=0, height=0, channels=3, streams=1, mix=0, groups=1, lr=0.0, roi=False):
    c = {"op": op, "algo": algo, "width": width, "height": height, "channels": channels, "streams": streams,
         "mix": mix, "groups": groups, "lr": lr, "roi": roi}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: one frame of a thumbnail-size thermal sensor, all latency and launches
        _case("lobster_160x120_gray", "apply", "lobster", 160, 120, 1),
        # one surveillance camera of the classic test size, frame after frame
        _case("subsense_320x240_rgb", "apply", "subsense", 320, 240, 3),
        # the reference's own call on an HD camera: frames arrive and masks leave in host memory
        _case("subsense_1920x1080_rgb_host", "host", "subsense", 1920, 1080, 3),
        # a thermal camera at its full size
        _case("lobster_640x512_gray", "apply", "lobster", 640, 512, 1),
        # an odd-size crop with a region of interest, as dataset sequences have
        _case("subsense_721x577_rgb_roi", "apply", "subsense", 721, 577, 3, roi=True),
        # one HD camera
        _case("subsense_1920x1080_rgb", "apply", "subsense", 1920, 1080, 3),
        # one UHD camera: the largest single frame
        _case("subsense_3840x2160_rgb", "apply", "subsense", 3840, 2160, 3),
        # 64 cameras of four sizes stepped together: the throughput configuration (16 streams of each size)
        _case("batch64_mixed", "batch", streams=64, groups=3),
        # 24 served cameras whose frames arrive together
        _case("serve24_mixed", "serve", streams=24, mix=7),
        # looking at the learned background of an HD stream
        _case("background_1920x1080_rgb", "background", "subsense", 1920, 1080, 3),
        # opening a 720p stream
        _case("initialize_1280x720_rgb", "initialize", "subsense", 1280, 720, 3),
        # scoring an HD mask against labelled ground truth
        _case("score_1920x1080", "score", width=1920, height=1080, channels=1),
    ]


def _size(rng, lo, hi):
    """width and height of about lo..hi pixels (log-uniform) in the aspects cameras and crops have."""
    area = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    aspect = rng.choice((4 / 3, 16 / 9, 5 / 4, 1.0, rng.uniform(0.6, 2.2)))
    w = max(64, int(math.sqrt(area * aspect)))
    h = max(48, int(w / aspect))
    kind = rng.random()
    if kind < 0.5:  # sensor sizes: multiples of 8 or 16
        step = rng.choice((8, 16))
        w, h = w // step * step, h // step * step
    return w, h


def draw(rng):
    op = rng.choice(("apply",) * 8 + ("host",) * 4 + ("batch",) * 3 + ("serve",) * 2 + ("background", "initialize", "score"))
    if op == "batch":
        return _case(None, op, streams=int(math.exp(rng.uniform(math.log(2), math.log(40)))), mix=rng.randrange(1, 1 << 30),
                     groups=rng.choice((1, 2, 3)))
    if op == "serve":
        return _case(None, op, streams=int(math.exp(rng.uniform(math.log(1.01), math.log(24)))), mix=rng.randrange(1, 1 << 30))
    if op == "score":
        w, h = _size(rng, 64 * 48, 3840 * 2160)
        return _case(None, op, width=w, height=h, channels=1, roi=rng.random() < 0.5)
    algo = "subsense" if op == "background" or rng.random() < 0.65 else "lobster"
    w, h = _size(rng, 96 * 72, {"apply": 3840 * 2160, "host": 1920 * 1080}.get(op, 1280 * 720))
    lr = 0.0
    if op in ("apply", "host") and rng.random() < 0.25:
        lr = rng.choice((2.0, 8.0, 32.0))
    return _case(None, op, algo, w, h, rng.choice((3, 3, 1)), lr=lr, roi=op == "apply" and w * h < 1500000 and rng.random() < 0.3)


def _stream_sizes(case):
    n, op = case["streams"], case["op"]
    if case["mix"] == 0:  # equal shares of the four sizes
        return [MIX[i * len(MIX) // n] for i in range(n)]
    r = random.Random(case["mix"])
    sizes = [r.choice(SERVED if op == "serve" else MIX) for _ in range(n)]
    if op == "batch":  # and some cropped ones
        sizes = [(w - r.randrange(1, 60), h - r.randrange(1, 40), c) if r.random() < 0.3 else (w, h, c) for w, h, c in sizes]
    return sizes


def _sequence(algo, w, h, c, seed):
    """a scene of the size: the nearest preset's content, its objects scaled to the frame"""
    if algo == "lobster" and c == 1:
        kind = synth.THERMAL
    else:
        kind = synth.QVGA if w * h < 500000 else synth.HD1080 if w * h < 4000000 else synth.UHD4K
    cfg = synth.preset(kind)
    side = min(w, h)
    cfg.width, cfg.height, cfg.channels = w, h, c
    cfg.seed = (cfg.seed + 2654435761 * (seed + 1)) & 0x7FFFFFFF
    cfg.obj_max = max(4, min(cfg.obj_max, side // 4))
    cfg.obj_min = max(3, min(cfg.obj_min, cfg.obj_max))
    cfg.speed_min, cfg.speed_max = max(1, w // 96), max(2, w // 32)
    if cfg.flicker_size:
        cfg.flicker_size = max(4, min(cfg.flicker_size, side // 4))
    return synth.Sequence(cfg)


class _Feed:
    """RING consecutive frames of one stream in device memory; the first WARM passes walk them too."""

    def __init__(self, algo, w, h, c, seed):
        self.shape = (h, w, c) if c > 1 else (h, w)
        self.bytes = w * h * c
        self.frames = torch.empty((RING,) + self.shape, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        _sequence(algo, w, h, c, seed).frames_device(0, RING, self.frames.data_ptr())
        self.mask = torch.empty((h, w), dtype=torch.uint8, device="cuda")

    def at(self, t):
        return self.frames[t % RING].data_ptr()


def _ellipse(w, h):
    y, x = np.ogrid[:h, :w]
    return np.where(((x - w / 2) / (0.45 * w)) ** 2 + ((y - h / 2) / (0.42 * h)) ** 2 <= 1.0, 255, 0).astype(np.uint8)


def _lr(case):
    return case["lr"] if case["lr"] else None


def _running(case, feed, stream=0):
    """a subtractor initialized on the sequence's first frame and stepped over WARM frames"""
    w, h, c = case["width"], case["height"], case["channels"]
    bgs = ALGOS[case["algo"]](stream_id=stream)
    first = feed.frames[0].cpu().numpy()
    bgs.initialize(first, _ellipse(w, h)) if case["roi"] else bgs.initialize(first)
    for t in range(WARM):
        bgs.apply_device(feed.at(t), feed.mask.data_ptr(), _lr(case))
    bgs.synchronize()
    return bgs


def _labels(w, h, seed):
    """mask, ground truth with every label, ROI: patches of about 16 pixels, as segmentations have"""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    values = torch.tensor([0, 0, 0, 0, 255, 255, 50, 85, 170], dtype=torch.uint8, device="cuda")

    def patches(n):
        k = torch.randint(0, n, ((h + 15) // 16, (w + 15) // 16), device="cuda", generator=g)
        return k.repeat_interleave(16, 0)[:h].repeat_interleave(16, 1)[:, :w]

    gt = values[patches(len(values))].contiguous()
    noise = torch.randint(0, 50, (h, w), device="cuda", generator=g) == 0
    mask = (((gt == 255) | (gt == 50)) ^ noise).to(torch.uint8) * 255
    roi = (patches(10) > 0).to(torch.uint8) * 255
    return mask.contiguous(), gt, roi.contiguous()


def prepare(case, seed):
    op, w, h, c = case["op"], case["width"], case["height"], case["channels"]
    s = {"case": case, "t": WARM}
    if op in ("apply", "background"):
        s["feed"] = _Feed(case["algo"], w, h, c, seed)
        s["bgs"] = _running(case, s["feed"])
    elif op == "host":
        feed = _Feed(case["algo"], w, h, c, seed)
        s["bgs"] = _running(case, feed)
        s["frames"] = [f.copy() for f in feed.frames.cpu().numpy()]
    elif op == "batch":
        sizes = _stream_sizes(case)
        s["feeds"] = [_Feed("subsense", *z, seed * 64 + i) for i, z in enumerate(sizes)]
        s["members"] = [BackgroundSubtractorSuBSENSE(stream_id=i) for i in range(len(sizes))]
        torch.cuda.synchronize()
        for m, f, z in zip(s["members"], s["feeds"], sizes):
            m.initialize_device(f.at(0), *z)
        s["batch"] = Batch(s["members"], groups=case["groups"])
        for t in range(WARM):
            s["batch"].apply_device([f.at(t) for f in s["feeds"]], [f.mask.data_ptr() for f in s["feeds"]])
        s["batch"].synchronize()
    elif op == "serve":
        sizes = _stream_sizes(case)
        s["feeds"] = [_Feed("subsense", *z, seed * 64 + i) for i, z in enumerate(sizes)]
        torch.cuda.synchronize()
        s["server"] = Server(hbm_budget=64 << 30)
        s["ids"] = [s["server"].open(f.at(0), *z, stream_id=i) for i, (f, z) in enumerate(zip(s["feeds"], sizes))]
        for t in range(WARM):
            _serve(s, t)
    elif op == "initialize":
        s["frames"] = _Feed(case["algo"], w, h, c, seed).frames.cpu().numpy()
        s["bgs"] = ALGOS[case["algo"]]()
        s["bgs"].initialize(s["frames"][0].copy())
    elif op == "score":
        s["mask"], s["gt"], s["roi"] = _labels(w, h, seed)
    torch.cuda.synchronize()
    return s


def _serve(s, t):
    server = s["server"]
    for sid, f in zip(s["ids"], s["feeds"]):
        server.submit(sid, f.at(t), f.mask.data_ptr(), tag=sid)
    server.drain()
    return server.poll()


def run(state):
    case, t = state["case"], state["t"]
    op = case["op"]
    state["t"] = t + 1
    if op == "apply":
        feed, bgs = state["feed"], state["bgs"]
        bgs.apply_device(feed.at(t), feed.mask.data_ptr(), _lr(case))
        bgs.synchronize()
        return feed.mask
    if op == "host":
        return state["bgs"].apply(state["frames"][t % RING], learningRate=_lr(case))
    if op == "batch":
        feeds = state["feeds"]
        state["batch"].apply_device([f.at(t) for f in feeds], [f.mask.data_ptr() for f in feeds])
        state["batch"].synchronize()
        return [f.mask for f in feeds]
    if op == "serve":
        done = _serve(state, t)
        if (done["status"] != 0).any():
            raise RuntimeError("a served frame failed")
        return [f.mask for f in state["feeds"]]
    if op == "background":
        return state["bgs"].getBackgroundImage()
    if op == "initialize":
        state["bgs"].initialize(state["frames"][t % RING])
        return state["bgs"].getBackgroundImage()
    b = BinClassif()
    b.accumulate_device(state["mask"].data_ptr(), state["gt"].data_ptr(), state["roi"].data_ptr() if case["roi"] else None,
                        case["width"], case["height"])
    return b.counts()


def _frame_bytes(algo, w, h, c):
    """Bytes of one frame step that no arrangement of it avoids, per pixel. SuBSENSE: the frame (c), ten f32 maps
    read and written (80), the last colour and descriptor read and written (6c), six u8 maps read and written
    (12), the ROI (1) and the mask (1), two examined samples (2 matches are needed) and three written
    samples per four pixels at 3c bytes. LOBSTER: the frame, ROI, previous raw mask, mask, two examined samples and
    one written per eight pixels (learning rate 16)."""
    if algo == "subsense":
        return w * h * (c + 80 + 6 * c + 12 + 2 + 3 * c * 2.75)
    return w * h * (2 * c + 4 + 3 * c * 2.125)


def work(case):
    op, w, h, c = case["op"], case["width"], case["height"], case["channels"]
    if op in ("apply", "host"):
        n = _frame_bytes(case["algo"], w, h, c)
    elif op in ("batch", "serve"):
        n = sum(_frame_bytes("subsense", *z) for z in _stream_sizes(case))
    elif op == "background":  # the samples' colours, once
        n = w * h * c * 51
    elif op == "initialize":  # every sample written, every map set, then the background image read
        samples = 50 if case["algo"] == "subsense" else 35
        n = w * h * (3 * c * samples + c * samples + 2 * c + (40 if case["algo"] == "subsense" else 0))
    else:
        n = w * h * (3 if case["roi"] else 2)
    return {"bytes": float(n), "flops": 0.0}


def exact(case, seed):
    """The counts of the scoring cases from plain torch. Every other output is a byte mask or image of an
    integer algorithm run over many frames."""
    if case["op"] != "score":
        return None
    mask, gt, roi = _labels(case["width"], case["height"], seed)
    valid = (gt != 85) & (gt != 170)
    if case["roi"]:
        valid &= roi != 0
    pos, true = mask == 255, gt == 255
    count = lambda m: int((m & valid).sum())  # noqa: E731
    return {"tp": count(pos & true), "tn": count(~pos & ~true), "fp": count(pos & ~true), "fn": count(~pos & true),
            "se": count(pos & (gt == 50)), "dc": int((~valid).sum())}
