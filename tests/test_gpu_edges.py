"""Kernels at the sizes where their tilings can go wrong: edges of tiles,
remainders, the smallest and largest of their ranges, against the oracle or a
64-bit restatement."""
import numpy as np
import pytest

import oracle_lib as OL
import trajgen

pytestmark = pytest.mark.gpu


# Active counts around the 256-row tile; L = 130 takes 13000 bins, three
# passes of the LDS histogram.
@pytest.mark.parametrize("na,L", [(0, 9.0), (1, 9.0), (255, 9.0), (256, 9.0), (257, 130.0), (513, 9.0), (700, 130.0)])
def test_guu_tile_edges(gpu, na, L):
    n, frames = 700, trajgen.case_frames(5, 40)
    X, Y, Z, _ = trajgen.make_frames(n, frames, 31 + na, 0.3, 1.0)
    act = np.zeros(n, dtype=np.int32)
    act[np.random.default_rng(na).permutation(n)[:na]] = 1
    fr = gpu.Frames(n, L, len(frames))
    for k, t in enumerate(frames):
        fr.push(X[k], Y[k], Z[k], t)
    h, fn, no = fr.guu(act, 40, 0.06)
    fr.close()
    ho, fno, noo = OL.guu(n, L, X, Y, Z, act, frames, 40, 0.06)
    assert (fn, no) == (fno, noo)
    assert np.array_equal(h[0], ho[0])
    # a bin sums at most a few thousand FP64 terms: n_terms * 2^-53 of their absolute sum
    scale = max(1.0, np.abs(ho[1]).max())
    assert np.abs(h[1:] - ho[1:]).max() <= 1e-12 * scale
