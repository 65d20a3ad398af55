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
