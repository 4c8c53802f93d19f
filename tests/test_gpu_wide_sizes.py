"""The grid of the wide step at the edges of its one-load pass: flocks of one
agent more than eight per thread (the rest are read again), of several such
passes, and smaller ones.  Fields and poses equal the full scan's bit for bit."""
import pytest

import test_gpu_large_flock as large

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N, R, side, r", [(2049, 250, 2000.0, 5), (8193, 512, 3000.0, 4), (17000, 300, 5000.0, 6)])
def test_grid_of_flocks_beyond_one_load(gpu, N, R, side, r):
    large.test_wide_grid_path_matches_full_scan(gpu, N, R, side, r, False)
