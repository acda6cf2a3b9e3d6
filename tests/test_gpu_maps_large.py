"""Maps of a bunch with more particles than one launch takes threads (2^32;
57 bytes each fit the card's memory up to about 5e9)."""
import gc

import numpy as np
import pytest

import synergia2_amd as sc
from helpers import GAMMA, gaussian_parts

pytestmark = pytest.mark.gpu


def test_more_particles_than_threads(gpu):
    import torch
    n, few = 2 ** 32 + 300, 4096
    gc.collect()
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 57 * n + (4 << 30):
        pytest.skip("needs 250 GB of free device memory")
    print("case maps of 2^32 + 300 particles", flush=True)
    cell = [(sc.MAP_DRIFT, 0.37, 0.0), (sc.MAP_QUADRUPOLE, 0.2, 0.6)]
    p = torch.from_numpy(gaussian_parts(few, (1e-3,) * 6, seed=1))
    small = sc.Bunch(few, 1e11, gamma=GAMMA)
    small.set_host(p.numpy())
    slices = sc.make_slices(cell, small.p, small.mass)
    sc.apply_maps(small, slices)
    want = small.host()[0]

    b = sc.Bunch(1, 1e11, gamma=GAMMA)
    b.n = n
    b.parts = torch.empty((7, n), dtype=torch.float64, device="cuda")
    b.masks = torch.zeros(n, dtype=torch.uint8, device="cuda")
    # active: the first particles, those around the middle and the last
    places = [0, 2 ** 31 - few // 2, n - few]
    for at in places:
        b.parts[:, at:at + few] = p.cuda()
        b.masks[at:at + few] = 1
    sc.apply_maps(b, slices)
    got = [b.parts[:, at:at + few].cpu().numpy() for at in places]
    del b
    gc.collect()
    torch.cuda.empty_cache()
    for g in got:
        assert np.array_equal(g, want)
