"""Stand-alone LBSP maps of images below a word, below a patch, and past 2^31 bytes: the reads of a tile stay inside the
image (checked on the host), and the maps are the oracle's."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tile_reads_stay_inside_the_image(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    exe = str(tmp_path / "word_place")
    r = subprocess.run([hipcc, "-x", "hip", "--cuda-host-only", "-O1", "-std=c++17",
                        os.path.join(ROOT, "tests", "cpp", "word_place.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("w,h,c", [(1, 1, 1), (2, 1, 1), (3, 1, 1), (1, 3, 1), (1, 1, 3), (4, 4, 1), (4, 70, 3), (70, 4, 3), (5, 5, 3)])
def test_lbsp_of_the_smallest_images(w, h, c, packed):
    from oracle_lib import lib as orc
    from test_gpu_kernels import _lbsp_gpu
    img = np.random.default_rng(w * 100 + h).integers(0, 256, (h, w, c), dtype=np.uint8)
    ref = np.zeros((h, w, c), np.uint16)
    if w >= 5 and h >= 5:
        orc().orc_lbsp_compute_abs(img, w, h, c, 9, ref)
    assert np.array_equal(_lbsp_gpu(img, 9, packed), ref)


@pytest.mark.gpu
@pytest.mark.parametrize("w,h,c", [(26755, 26755, 3), (46341, 46341, 1)])
def test_lbsp_past_two_gigabytes(w, h, c):
    # bands of the large image's map equal the maps of the bands alone
    import torch

    from litiv_amd import lbsp_compute_abs
    g = torch.Generator(device="cuda")
    g.manual_seed(w)
    img = torch.randint(0, 256, (h, w * c), dtype=torch.uint8, device="cuda", generator=g)
    out = torch.full((h, w * c), -1, dtype=torch.int16, device="cuda")
    torch.cuda.synchronize()
    lbsp_compute_abs(img.data_ptr(), w, h, c, 30, out.data_ptr())
    torch.cuda.synchronize()
    for y in (0, h // 2, h - 40):
        band, want = img[y:y + 40].clone(), torch.empty((40, w * c), dtype=torch.int16, device="cuda")
        torch.cuda.synchronize()
        lbsp_compute_abs(band.data_ptr(), w, 40, c, 30, want.data_ptr())
        torch.cuda.synchronize()
        assert torch.equal(out[y + 2:y + 38], want[2:38]), y
    assert not out[:2].any() and not out[h - 2:].any()
