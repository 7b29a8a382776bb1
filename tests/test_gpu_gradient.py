"""The network's gradient kernels at the edges of their row groups against the
oracle, through the C ABI.

A block of the rows' kernel takes 16 rows; a wavefront of the weights' kernel
takes parts of 8 such groups (128 rows), two groups to an instruction, at most 64
parts at once (8192 rows), and batches go in chunks of 32768 rows.  So: one
group, an odd number of groups, a full pair, a part and one group more, a second
round of the first parts, and a second chunk.  Both sides round activations
and dZ to BF16 at the same places, so they differ by FP32 sums and by the
roundings those flip: 1e-4 of the loss, 1e-2 of a layer's gradient norm, at any
row count.
"""
import numpy as np
import pytest

from oracle import surrogate as S
from test_gpu_surrogate import box, lattice, scaled_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [16, 48, 64, 80, 16384 + 16, 128 + 16, 8192 + 16, 32768 + 16])
def test_gradient_matches_oracle_at_row_group_edges(rows):
    lat = lattice(box())
    params = scaled_params(9, 1.2)
    lat.set_surrogate_params(params)
    rng = np.random.default_rng(rows)
    X = np.zeros((rows, 16), np.float32)
    X[:, :S.NIN] = rng.standard_normal((rows, S.NIN))
    T = np.zeros((rows, 16), np.float32)
    T[:, :S.NOUT] = rng.standard_normal((rows, S.NOUT))
    loss, g = lat.surrogate_gradient(X, T)
    again = lat.surrogate_gradient(X, T)
    lref, gref = S.loss_and_grad(params, X, T)
    assert loss == again[0] and np.array_equal(g, again[1])
    assert abs(loss - lref) / lref < 1e-4
    for L, ((gw, gb), (rw, rb)) in enumerate(zip(S.unpack(g), S.unpack(gref))):
        ew = np.linalg.norm(gw - rw) / np.linalg.norm(rw)
        eb = np.linalg.norm(gb - rb) / np.linalg.norm(rb)
        assert ew < 1e-2 and eb < 1e-2, (L, ew, eb)
