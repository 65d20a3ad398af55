"""GPU parity of the frame step's dispatch branches and list edges against the sequential oracle:
contents and sizes at which the worklists, tiles and zones of the kernels have their remainders."""
import numpy as np
import pytest

from litiv_amd import synth
from oracle_lib import LOBSTER, SUBSENSE
from test_gpu_parity import run_sequence

pytestmark = pytest.mark.gpu


def flashing(w, h, c, n, seed=0):
    """blocks that jump between two textures from frame to frame: raw decisions change everywhere, so
    many pixels push to the fix-point worklists, some to the same target"""
    r = np.random.default_rng(seed)
    shape = (h, w) if c == 1 else (h, w, c)
    a, b = r.integers(0, 256, (2,) + shape)
    out = []
    for _ in range(n):
        m = np.kron(r.integers(0, 4, ((h + 4) // 5, (w + 6) // 7)) == 0, np.ones((5, 7), bool))[:h, :w]
        f = np.where(m if c == 1 else m[..., None], b, a) + r.integers(-4, 5, shape)
        out.append(np.clip(f, 0, 255).astype(np.uint8))
    return out


@pytest.mark.parametrize("algo,c", [(SUBSENSE, 3), (SUBSENSE, 1), (LOBSTER, 3)])
@pytest.mark.parametrize("w,h", [(200, 141), (67, 9)])
@pytest.mark.parametrize("schedule", [(0, 1024, 2, 256), (4, 3, 0, 1), (255, 1024, 1, 2)])
def test_first_worklist_stripes(algo, c, w, h, schedule):
    # more tiles than stripes and fewer; read by a full-grid iteration, by few blocks, by the tail alone
    run_sequence(algo, flashing(w, h, c, 10), schedule=schedule, lr=None if algo == SUBSENSE else 2.0)


@pytest.mark.parametrize("algo,c,schedule", [(SUBSENSE, 3, (1, 1024, 2, 256)), (SUBSENSE, 3, (1, 3, 1, 5)),
                                             (SUBSENSE, 1, (1, 1024, 2, 256)), (LOBSTER, 3, (1, 2, 2, 256)),
                                             (LOBSTER, 1, (6, 1, 1, 1)), (SUBSENSE, 3, (11, 1, 1, 1))])
def test_continuation_lanes_and_groups(algo, c, schedule):
    # seq_limit 1 on 60 K pixels leaves more entries than phase B takes in lane groups (32 K), later limits
    # fewer; few blocks make the list loops run several rounds with a ragged last one
    run_sequence(algo, flashing(301, 205, c, 6), schedule=schedule, lr=None if algo == SUBSENSE else 2.0)


@pytest.mark.parametrize("lr,limit", [(1.0, 255), (1.0, 3)])
def test_more_overwritten_slots_than_entries(lr, limit):
    # learning rate 1 with 5x5 diffusion: every background pixel writes a neighbour, so some pixels have more
    # than four overwritten slots and go to the fix point unmatched
    gpu, _ = run_sequence(SUBSENSE, flashing(484, 325, 3, 7), lr=lr, schedule=(limit, 1024, 2, 256))
    assert gpu.stats()["fixpoint_work"][1] > 0


@pytest.mark.parametrize("pad_in,pad_out", [(0, 0), (7, 0), (0, 5), (3, 9)])
def test_host_rows_packed_and_padded(pad_in, pad_out):
    # packed rows take one linear copy, padded rows the 2-D copy, in and out independently
    import ctypes as C

    from litiv_amd import BackgroundSubtractorSuBSENSE
    from litiv_amd.bgs import lib
    w, h = 83, 45
    frames = flashing(w, h, 3, 4)
    a, b = BackgroundSubtractorSuBSENSE(), BackgroundSubtractorSuBSENSE()
    a.initialize(frames[0])
    b.initialize(frames[0])
    for f in frames:
        src = np.zeros((h, 3 * w + pad_in), np.uint8)
        src[:, :3 * w] = f.reshape(h, 3 * w)
        out = np.full((h, w + pad_out), 7, np.uint8)
        assert lib().lvbgs_apply(b._h, src.ctypes.data, src.strides[0], out.ctypes.data, out.strides[0], C.c_double(0.0)) == 0
        assert np.array_equal(out[:, :w], a.apply(f)) and (out[:, w:] == 7).all()
    bg = np.full((h, 3 * w + pad_out), 7, np.uint8)
    assert lib().lvbgs_get_background_image(b._h, bg.ctypes.data, bg.strides[0]) == 0
    assert np.array_equal(bg[:, :3 * w].reshape(h, w, 3), a.getBackgroundImage()) and (bg[:, 3 * w:] == 7).all()


@pytest.mark.parametrize("w,h", [(4, 9), (5, 5), (9, 4), (8, 6)])
def test_validate_roi_border(w, h):
    from litiv_amd import BackgroundSubtractorSuBSENSE
    roi = BackgroundSubtractorSuBSENSE.validateROI(np.full((h, w), 255, np.uint8))
    want = np.zeros((h, w), np.uint8)
    want[2:max(2, h - 2), 2:max(2, w - 2)] = 255
    assert np.array_equal(roi, want)


@pytest.mark.parametrize("algo,c,w,h", [(SUBSENSE, 3, 131, 70), (SUBSENSE, 1, 64, 48), (LOBSTER, 3, 70, 67),
                                        (LOBSTER, 1, 129, 5)])
def test_reinitialize_over_an_old_model(algo, c, w, h):
    # the arena is reused and its samples are not cleared: a second initialize with a smaller ROI writes them
    # all (zeros outside the ROI), and a partial refresh then keeps the foreground's
    from test_gpu_parity import LOB_STATE, SUB_STATE, _pair
    frames = flashing(w, h, c, 6, seed=w)
    roi = np.zeros((h, w), np.uint8)
    roi[3:h - 1, 9:w - 20] = 255
    gpu, orc = _pair(algo)
    for m in (gpu, orc):
        m.initialize(frames[0])
        for f in frames[:3]:
            m.apply(f)
        m.initialize(frames[3], roi)
    names = SUB_STATE if algo == SUBSENSE else LOB_STATE
    for name in names:
        assert np.array_equal(gpu.state(name), orc.state(name)), name
    assert np.array_equal(gpu.getBackgroundImage(), orc.background_image())
    assert np.array_equal(gpu.getBackgroundDescriptorsImage(), orc.background_descriptors())
    for k, f in enumerate(frames[3:]):
        assert np.array_equal(gpu.apply(f), orc.apply(f))
        gpu.refreshModel(0.3, bool(k & 1))
        orc.refresh_model(0.3, bool(k & 1))
    for name in names:
        assert np.array_equal(gpu.state(name), orc.state(name)), name


@pytest.mark.parametrize("groups", [1, 2])
def test_batch_model_reset(groups):
    # a brightness jump triggers the automatic reset of two members (odd and even sizes): their
    # dilation blocks refresh the model, the third member's (grey, no jump) must not
    import torch

    from litiv_amd import BackgroundSubtractorSuBSENSE, Batch
    from oracle_lib import Oracle
    from test_gpu_parity import SUB_STATE
    specs = [(333, 247, 3, 120), (320, 240, 3, 120), (322, 240, 1, 0)]
    gpus, orcs, seqs = [], [], []
    for i, (w, h, c, jump) in enumerate(specs):
        s = synth.Sequence(synth.preset(synth.QVGA, i, width=w, height=h, channels=c))
        frames = [s.frame(t) for t in range(52)]
        for t in range(28, 52):
            frames[t] = np.clip(frames[t].astype(np.int16) + jump, 0, 255).astype(np.uint8)
        seqs.append(frames)
        for cls, to in ((BackgroundSubtractorSuBSENSE, gpus), (lambda **k: Oracle(SUBSENSE, **k), orcs)):
            m = cls(stream_id=i)
            m.initialize(frames[0])
            to.append(m)
    batch = Batch(gpus, groups=groups)
    masks = [torch.empty(f[0].shape[:2], dtype=torch.uint8, device="cuda") for f in seqs]
    for t in range(52):
        d = [torch.from_numpy(f[t]).cuda() for f in seqs]
        torch.cuda.synchronize()
        batch.apply_device([x.data_ptr() for x in d], [m.data_ptr() for m in masks])
        batch.synchronize()
        for i in range(3):
            assert np.array_equal(masks[i].cpu().numpy(), orcs[i].apply(seqs[i][t])), (i, t)
    assert [o.scalars()["refresh_seq"] >= 2 for o in orcs] == [True, True, False]
    for i in range(3):
        for name in SUB_STATE:
            assert np.array_equal(gpus[i].state(name), orcs[i].state(name)), (i, name)


@pytest.mark.parametrize("algo,c", [(SUBSENSE, 3), (SUBSENSE, 1), (LOBSTER, 3), (LOBSTER, 1)])
@pytest.mark.parametrize("w,h", [(5, 5), (6, 7), (63, 5), (65, 6), (67, 9), (131, 10)])
def test_tile_rows_at_small_and_ragged_sizes(algo, c, w, h):
    # tile rows are read in words at any alignment: frames whose rows and whole size are no multiple of a word,
    # tiles with one to three columns
    run_sequence(algo, flashing(w, h, c, 6, seed=w * h), lr=None if algo == SUBSENSE else 2.0)


@pytest.mark.parametrize("offset", [1, 2, 3])
@pytest.mark.parametrize("c", [1, 3])
def test_unaligned_device_frames(offset, c):
    import torch

    from test_gpu_parity import _pair
    w, h = 77, 21
    gpu, orc = _pair(SUBSENSE)
    frames = flashing(w, h, c, 5, seed=offset)
    gpu.initialize(frames[0])
    orc.initialize(frames[0])
    buf = torch.zeros(w * h * c + 8, dtype=torch.uint8, device="cuda")
    mask = torch.zeros(w * h + 8, dtype=torch.uint8, device="cuda")
    for f in frames:
        buf[offset:offset + f.size].copy_(torch.from_numpy(f.reshape(-1)))
        torch.cuda.synchronize()
        gpu.apply_device(buf.data_ptr() + offset, mask.data_ptr() + offset)
        gpu.synchronize()
        m = mask.cpu().numpy()
        assert np.array_equal(m[offset:offset + w * h].reshape(h, w), orc.apply(f))
        assert not m[:offset].any() and not m[offset + w * h:].any()


@pytest.mark.parametrize("lr", [1.0, 5.0, 4194303.5, 4194304.0, 4194304.5, 3e9, 1e12])
@pytest.mark.parametrize("algo", [SUBSENSE, LOBSTER])
def test_learning_rates_around_the_divisibility_range(algo, lr):
    run_sequence(algo, flashing(90, 40, 1, 5), lr=lr)


@pytest.mark.parametrize("n", [1, 2, 3, 32, 33, 64, 65, 127, 128, 255])
def test_sample_counts(n):
    # the slot draw's reciprocal (powers of two and their neighbours), slots past 64
    run_sequence(SUBSENSE, flashing(70, 30, 3, 5), bg_samples=n, required_bg_samples=min(n, 2), lr=1.0)


@pytest.mark.parametrize("w,h", [(5, 5), (6, 63), (63, 6), (64, 65), (65, 64), (127, 130), (129, 9), (192, 67)])
@pytest.mark.parametrize("density", [0.05, 0.4])
def test_zone_rows_and_floods(w, h, density):
    """rows of 64 that end inside, at or past the image, and hole fills that cross zone edges both ways"""
    from litiv_amd import BackgroundSubtractorSuBSENSE
    from test_gpu_kernels import _annuli, _oracle_post
    rng = np.random.default_rng(w * 1000 + h)
    raw = np.where(rng.random((h, w)) < density, 255, 0).astype(np.uint8) | _annuli(rng, h, w, 6, 45)
    sub = BackgroundSubtractorSuBSENSE()
    sub.initialize(np.zeros((h, w, 3), np.uint8))
    exp, n_holes = _oracle_post(raw, int(sub.scalars()["median_k"]))
    assert np.array_equal(sub.debug_postprocess(raw), exp), "%d hole px" % n_holes


@pytest.mark.parametrize("c", [3, 1])
@pytest.mark.parametrize("w,h", [(15, 23), (23, 15), (71, 65), (95, 79), (64, 71), (71, 64), (17, 17)])
def test_frame_level_cells_of_ragged_sizes(w, h, c):
    """cells of 8 to 15 pixels a side: ten columns as words or the plain loop, up to the frame's last byte"""
    run_sequence(SUBSENSE, flashing(w, h, c, 8, seed=w + h))


@pytest.mark.parametrize("w,h", [(16, 1), (17, 1), (4096, 1), (4097, 1), (4096, 1024), (4096, 1025), (4099, 1027)])
def test_score_chunks_and_words(w, h):
    """every pair of a result and a ground-truth value in words of four, and sizes around a chunk and a grid"""
    import torch
    from litiv_amd import BinClassif
    from oracle_lib import binclassif
    i = np.arange(h * w, dtype=np.uint32)
    res = np.where(i % 3 == 0, 255, i & 255).astype(np.uint8).reshape(h, w)
    gt = np.where(i % 5 == 0, np.array([50, 85, 170, 255])[i // 5 % 4], i >> 8 & 255).astype(np.uint8).reshape(h, w)
    roi = (np.random.default_rng(w + h).integers(0, 9, (h, w)) * 16).astype(np.uint8)
    d = [torch.from_numpy(x).cuda() for x in (res, gt, roi)]
    torch.cuda.synchronize()
    for k in (2, 3):
        b = BinClassif().accumulate_device(d[0].data_ptr(), d[1].data_ptr(), d[2].data_ptr() if k == 3 else None, w, h)
        got = tuple(b.counts()[n] for n in ("tp", "tn", "fp", "fn", "se", "dc"))
        assert got == binclassif(res, gt, roi if k == 3 else None)


@pytest.mark.parametrize("c", [1, 3])
@pytest.mark.parametrize("t", [0, 1, 2, 126, 127, 128, 129, 253, 254, 255])
def test_lbsp_limits_of_every_byte(t, c):
    """centres and taps of every value, with differences just at, below and above the threshold"""
    from test_gpu_kernels import _lbsp_gpu, orc
    h, w = 40, 130
    r = np.random.default_rng(t)
    img = r.integers(0, 256, (h, w, c), dtype=np.uint8)
    near = r.random((h, w, c)) < 0.7  # values at distance t - 1, t, t + 1 of a common centre, and the extremes
    centre = int(r.integers(0, 256))
    d = centre + r.choice([-t - 1, -t, 1 - t, 0, t - 1, t, t + 1, -256, 256], (h, w, c))
    img[near] = np.clip(d, 0, 255).astype(np.uint8)[near]
    ref = np.zeros((h, w, c), np.uint16)
    orc().orc_lbsp_compute_abs(img, w, h, c, t, ref)
    assert np.array_equal(_lbsp_gpu(img, t, packed=True), ref)


@pytest.mark.parametrize("k", [1, 3, 11, 13])
@pytest.mark.parametrize("w,h", [(64, 16), (65, 17), (127, 33), (200, 47)])
def test_median_windows_and_mask_bits(w, h, k):
    """the smallest and largest windows at tile edges, and erosions whose words end inside or past the image"""
    from litiv_amd import BackgroundSubtractorSuBSENSE
    from test_gpu_kernels import _oracle_post
    rng = np.random.default_rng(w + k)
    coarse = np.kron(rng.random((h // 9 + 1, w // 11 + 1)) < 0.55, np.ones((9, 11), bool))[:h, :w]
    raw = np.where(coarse ^ (rng.random((h, w)) < 0.04), 255, 0).astype(np.uint8)
    sub = BackgroundSubtractorSuBSENSE(median_blur_kernel=k)
    sub.initialize(np.zeros((h, w, 3), np.uint8))
    assert int(sub.scalars()["median_k"]) == k
    exp, n_holes = _oracle_post(raw, k)
    assert np.array_equal(sub.debug_postprocess(raw), exp), "%d hole px" % n_holes


def test_schedules_return_to_automatic():
    """after any override the calls that name the automatic values leave a context as it was created"""
    import inspect

    from litiv_amd import BackgroundSubtractorSuBSENSE
    from litiv_amd.bgs import LvbgsError
    from test_gpu_parity import SUB_STATE
    assert inspect.signature(BackgroundSubtractorSuBSENSE.set_match_schedule).parameters["cont_blocks"].default == 0
    frames = flashing(150, 90, 3, 8)
    a, b = BackgroundSubtractorSuBSENSE(), BackgroundSubtractorSuBSENSE()
    for m in (a, b):
        m.initialize(frames[0])
    a.set_match_schedule(7, 3)
    a.set_fixpoint_schedule(0, 1)
    for t, f in enumerate(frames):
        if t == 4:
            a.set_match_schedule(0)
            a.set_fixpoint_schedule(-1, 0)
        assert np.array_equal(a.apply(f), b.apply(f)), t
        if t >= 4:  # what phase A examined and handed on follows from its limit
            sa, sb = a.stats(), b.stats()
            assert (sa["examined_speculative"], sa["fixpoint_work"][0]) == (sb["examined_speculative"], sb["fixpoint_work"][0])
    for name in SUB_STATE:
        assert np.array_equal(a.state(name), b.state(name)), name
    for bad in ((-1, 1), (256, 1), (1, -1), (1, 65536)):
        with pytest.raises(LvbgsError):
            a.set_match_schedule(*bad)
    for bad in ((-2, 1), (65, 1), (1, -1), (1, 65536)):
        with pytest.raises(LvbgsError):
            a.set_fixpoint_schedule(*bad)


def _distinct_slots(rec, raw):
    """per pixel, how many sample slots its raster-earlier neighbours overwrite if those that were background in
    the mask `raw` write: the record's target is the pixel and its forward gate is open"""
    h, w = rec.shape
    gate = ((rec >> 5) & 1 | (rec >> 6) & (rec >> 7) & 1).astype(bool) & (raw == 0)
    slots = np.full((12, h, w), -1, np.int64)
    for i in range(12):
        dx, dy = i % 5 - 2, i // 5 - 2  # the writer stands at (x + dx, y + dy)
        hit = np.where(gate & ((rec & 31) == (2 - dy) * 5 + 2 - dx), rec >> 24, -1)
        slots[i, 2:, 2:-2] = hit[2 + dy:h + dy, 2 + dx:w - 2 + dx]
    slots.sort(axis=0)
    return (slots[0] >= 0).astype(int) + ((slots[1:] != slots[:-1]) & (slots[1:] >= 0)).sum(axis=0)


@pytest.mark.parametrize("limit", [4, 255])
def test_pixels_past_the_entries_of_a_thread_occur(limit):
    # five or more overwritten slots: such pixels keep their guess and list themselves. They must occur in the
    # frames, and the masks must be the oracle's
    from test_gpu_parity import _pair
    frames = flashing(484, 325, 3, 5)
    gpu, orc = _pair(SUBSENSE)
    gpu.set_match_schedule(limit)
    gpu.initialize(frames[0])
    orc.initialize(frames[0])
    unmatched = 0
    for f in frames:
        raw = gpu.state("last_raw")
        assert np.array_equal(gpu.apply(f, learningRate=1.0), orc.apply(f, 1.0))
        n = _distinct_slots(gpu.state("rec"), raw)
        past = (n > 4) & (gpu.state("roi") != 0)
        unmatched += int(past.sum())
        assert (gpu.state("mres")[past] >> 24).all()  # the fix point matched them
    assert unmatched >= 5, unmatched


def test_iteration_cap_is_reported_by_synchronize():
    """the steps' error bits reach lvbgs_synchronize and lvbgs_batch_synchronize through the context's pinned word,
    stay until the next initialize, and stay with the context that they belong to"""
    import torch

    from litiv_amd import BackgroundSubtractorSuBSENSE, Batch, Server
    from litiv_amd.bgs import ERR_DEVICE, LvbgsError
    frames = flashing(96, 72, 3, 8)
    d = [torch.from_numpy(f).cuda() for f in frames]
    mask = torch.empty((72, 96), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    srv = Server(hbm_budget=1 << 30, fixpoint_launches=0)
    srv.debug_fixpoint_cap(0)
    sid = srv.open(d[0].data_ptr(), 96, 72, 3)
    member = srv.member(sid)
    member.synchronize()
    failed = False
    for t in range(8):
        srv.submit(sid, d[t].data_ptr(), mask.data_ptr(), tag=t)
        srv.drain()
        failed = any(int(s) == ERR_DEVICE for _, _, s in srv.poll())
        if failed:
            break
    assert failed, "no frame needed the fix point"
    # the server has closed the stream; its context waits in the server's pool
    other = BackgroundSubtractorSuBSENSE()
    other.initialize(frames[0])
    other.apply(frames[1])
    batch = Batch([other, member])
    for call in (member.synchronize, batch.synchronize, member.synchronize):
        with pytest.raises(LvbgsError) as e:
            call()
        assert e.value.code == ERR_DEVICE
    other.synchronize()
    member.initialize(frames[0])
    member.synchronize()
    batch.synchronize()
    batch.close()
    srv.close_server()
