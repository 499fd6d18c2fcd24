"""Pairwise three-body energies of cells, summed per pair of atoms in the LDS
for every tile pair, against the oracle: hardly an image per atom in a list (as
many LDS cells as slot pairs), about two (some tile pairs have more pairs of
atoms than cells), many, a slab, and a batch of all of them."""
import sys

import numpy as np
import pytest
import torch

import oracle as O
from helpers import BJ, ZERO, cell

pytestmark = pytest.mark.gpu

# seed, atoms, edge (bohr), three-body cutoff, directions
CELLS = [(31, 110, 24.0, 11.0, [True] * 3), (32, 140, 24.0, 19.5, [True] * 3), (33, 5, 8.5, 20.0, [True] * 3),
         (34, 70, 20.0, 16.0, [True, True, False])]


def _check(systems, precision):
    from dftd3 import torch_api
    spec, pos = torch_api.batch_spec(systems)
    out = torch_api.run_pairwise(spec, torch.as_tensor(pos, dtype=torch.float64, device="cuda").contiguous(),
                                 precision=precision)
    got = out["pair3"].cpu().numpy().reshape(-1)
    off = 0
    for s in systems:
        n = len(s["numbers"])
        x = got[off:off + n * n].reshape(n, n)
        off += n * n
        cut = (*O.DEFAULT_CUTOFF[:2], s["cutoff"]["disp3"], *O.DEFAULT_CUTOFF[3:])
        _, ref = O.pairwise(s["numbers"], s["positions"], s["lattice"], s["periodic"],
                            O.ZERO if s["kind"] == "zero" else O.RATIONAL, s["param"], cut)
        np.testing.assert_allclose(x, ref, rtol=0, atol=1e-10 if precision == "fp64" else 1e-5)
        np.testing.assert_array_equal(x, x.T)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("which", [0, 1, 2, 3, None])
def test_cells_vs_oracle(which, precision):
    print(f"[gpu-pairwise-cells] {which} {precision}", flush=True)
    sys.stdout.flush()
    systems = []
    for k, (seed, n, edge, cut3, pbc) in enumerate(CELLS):
        num, pos, lat = cell(seed, n, edge)
        systems.append(dict(numbers=num, positions=pos, lattice=lat, periodic=pbc, kind="zero" if k % 2 else "rational",
                            param=ZERO if k % 2 else BJ, cutoff=dict(disp3=cut3)))
    _check(systems if which is None else [systems[which]], precision)
