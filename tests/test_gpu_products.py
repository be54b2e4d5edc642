"""The FP64 contractions (KB projection and apply, overlaps, constraint) at the
edges of their tiles: orbital counts around 16, 64, 96 and 128, projector
counts that leave a 96- or 128-row tile partly empty, and more than one tile
row and column, through the SD step against the oracle."""
import pytest

from test_gpu_shapes import run_pair, say

pytestmark = pytest.mark.gpu

# molecules (6 projectors each), orbitals; the carried overlap runs at 128
EDGES = [(1, 15), (1, 16), (2, 17), (3, 31), (5, 32), (11, 33), (4, 48), (6, 49), (16, 63), (17, 64), (22, 65),
         (3, 95), (16, 96), (11, 97), (2, 127), (22, 128), (3, 129), (2, 191)]


@pytest.mark.parametrize("nmol,ne", EDGES)
def test_products_at_tile_edges_vs_oracle(gpu, nmol, ne):
    say("%d projectors, %d orbitals at 16^3" % (6 * nmol, ne))
    run_pair(nmol, 12.0, 16, ne, steps=2, inner=2, seed=11)
