"""Pair sums of molecules longer than the cutoffs: tile pairs and third atoms
out of range are left out, and their records are neither written nor read.
Compared with the oracle at the bars of the parity tests."""
import sys

import numpy as np
import pytest
import torch

import oracle as O
from helpers import BJ

pytestmark = pytest.mark.gpu


def _step(msg):
    print(f"[gpu-pair-sum-range] {msg}", flush=True)
    sys.stdout.flush()


def _molecule(seed, n, shape, spacing=4.07):
    rng = np.random.default_rng(seed)
    grid = np.stack(np.meshgrid(*[np.arange(m) for m in shape], indexing="ij"), axis=-1).reshape(-1, 3)[:n]
    pos = spacing * (rng.permutation(grid) + rng.uniform(-0.23, 0.23, (n, 3)))
    return rng.choice([1, 6, 7, 8], size=n, p=[0.5, 0.3, 0.1, 0.1]), pos


def _check(out, num, pos, cutoff, mixed, grad=True):
    c = {**dict(disp2=60.0, disp3=40.0, cn=40.0, width2=0.0, width3=0.0), **cutoff}
    cut = (c["cn"], c["disp2"], c["disp3"], c["width2"], c["width3"])
    ref = O.dispersion(num, pos, None, None, O.RATIONAL, BJ, cut, grad=grad)
    n, e, er = len(num), out["energy"][0].item(), ref["energy"]
    assert abs(e - er) <= (1e-8 * n if mixed else 1e-10 * abs(er)), (e, er)
    if grad:
        assert np.abs(out["gradient"].cpu().numpy() - ref["gradient"]).max() <= (1e-7 if mixed else 1e-9)
        assert np.abs(out["sigma"][0].cpu().numpy() - ref["virial"]).max() <= (1e-7 * n if mixed else 1e-9)


SHAPES = [  # tiles of 8 and of 16 positions; a last tile of one atom, of a part, whole
    (130, (1, 1, 130), dict(disp3=20.0)),
    (513, (1, 1, 513), {}),
    (577, (2, 2, 145), dict(disp3=25.0, disp2=30.0)),
    (640, (1, 26, 26), dict(disp3=12.0)),
    (705, (9, 9, 9), dict(disp3=8.0, disp2=20.0, width3=3.0)),
    (900, (2, 2, 225), dict(disp2=15.0)),  # the three-body cutoff is the longer one
]


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,shape,cutoff", SHAPES)
def test_extended_molecules(n, shape, cutoff, precision, grad):
    from dftd3 import torch_api
    _step(f"{n} atoms {shape} {cutoff} {precision} grad={grad}")
    num, pos = _molecule(n, n, shape)
    s = dict(numbers=num, positions=pos, param=BJ, cutoff=cutoff)
    _check(torch_api.get_dispersion_batch([s], precision=precision, grad=grad), num, pos, cutoff,
           precision == "mixed", grad)


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("n", [100, 640])
def test_records_of_an_earlier_geometry(n, grad):
    """A plan evaluates a compact molecule, whose pairs all have records, then
    the same atoms drawn apart, then parts of it out of each other's range."""
    from dftd3 import torch_api
    _step(f"{n} atoms, compact then drawn apart, grad={grad}")
    m = int(np.ceil(n ** (1.0 / 3.0)))
    num, pos = _molecule(n, n, (m, m, m))
    spec, p = torch_api.batch_spec([dict(numbers=num, positions=pos, param=BJ)])
    p = torch.as_tensor(p, dtype=torch.float64, device="cuda").contiguous()
    plan = torch_api.BatchPlan(spec, p, precision="fp64", grad=grad)
    _check(plan.execute(), num, pos, {}, False, grad)
    apart = pos * np.array([1.0, 1.0, 9.0])
    parts = pos + 150.0 * np.floor(np.arange(n) * 3 / n)[:, None]
    for x in (apart, parts, pos):
        t = torch.as_tensor(x, dtype=torch.float64, device="cuda").contiguous()
        _check(plan.execute(t), num, x, {}, False, grad)
        _check(torch_api.run_batch(spec, t, precision="fp64", grad=grad), num, x, {}, False, grad)


@pytest.mark.parametrize("n,shape", [(130, (1, 1, 130)), (640, (2, 2, 160))])
def test_pair_energies(n, shape):
    from dftd3 import torch_api
    _step(f"pair energies, {n} atoms {shape}")
    num, pos = _molecule(n, n, shape)
    spec, p = torch_api.batch_spec([dict(numbers=num, positions=pos, param=BJ)])
    p = torch.as_tensor(p, dtype=torch.float64, device="cuda").contiguous()
    out = torch_api.run_pairwise(spec, p, precision="fp64")
    r2, r3 = O.pairwise(num, pos, None, None, O.RATIONAL, BJ, O.DEFAULT_CUTOFF)
    for key, ref in (("pair2", r2), ("pair3", r3)):
        np.testing.assert_allclose(torch_api.blocks(out, key)[0].cpu().numpy(), ref, rtol=0, atol=1e-10)


def test_cost_follows_the_range():
    """The three-body kernels of a wire of 3,000 atoms, in which a pair has
    some 80 third atoms in range, cost less than a twentieth of those of a
    cube, in which it has all: a fixed cost per pair of tiles or per atom
    beyond the range shows here (0.08 when every third atom's record was
    fetched, 0.012 now)."""
    from dftd3 import library, torch_api
    _step("cost of a wire against a cube")
    ms = []
    for shape in ((2, 2, 750), (15, 15, 14)):
        num, pos = _molecule(1, 3000, shape)
        spec, p = torch_api.batch_spec([dict(numbers=num, positions=pos, param=BJ)])
        p = torch.as_tensor(p, dtype=torch.float64, device="cuda").contiguous()
        ws = library.new_workspace()
        torch_api.run_batch(spec, p, precision="fp64", ws=ws)
        library.set_kernel_timing(ws, True)
        for _ in range(5):
            torch_api.run_batch(spec, p, precision="fp64", ws=ws)
        total, calls = library.get_kernel_time(ws, "atm")
        assert calls == 5
        ms.append(total)
    assert ms[0] < 0.05 * ms[1], ms


# atoms of a molecule, three-body cutoff, precision, gradient, molecules in the
# batch, lists: the edges of the rule by the cutoff (0.75 atoms per squared cutoff,
# 0.055 per cubed cutoff, 250 and 500 atoms, 4,096 atoms a batch)
ROUTES = [
    (250, 12.0, "mixed", True, 17, False), (251, 12.0, "mixed", True, 17, True),
    (251, 12.0, "mixed", True, 16, False), (251, 12.0, "mixed", False, 17, False),
    (600, 28.4, "mixed", True, 7, False), (600, 28.2, "mixed", True, 7, True),
    (500, 12.0, "fp64", True, 9, False), (501, 12.0, "fp64", True, 9, True),
    (501, 12.0, "fp64", False, 9, False), (600, 22.3, "fp64", True, 7, False),
    (600, 22.1, "fp64", True, 7, True), (600, 12.0, "fp64", True, 6, False),
]


@pytest.mark.parametrize("n,disp3,precision,grad,m,lists", ROUTES)
def test_short_cutoffs_in_batches(n, disp3, precision, grad, m, lists):
    """Which route a batch of equal molecules takes, and its results against
    each molecule alone (pair sums)."""
    from dftd3 import library, torch_api
    _step(f"{m} x {n} atoms, cutoff {disp3}, {precision}, grad={grad}")
    k = int(np.ceil(n ** (1.0 / 3.0)))
    systems = []
    for seed in range(m):
        num, pos = _molecule(seed, n, (k, k, k))
        systems.append(dict(numbers=num, positions=pos, param=BJ, cutoff=dict(disp3=disp3)))
    spec, p = torch_api.batch_spec(systems)
    p = torch.as_tensor(p, dtype=torch.float64, device="cuda").contiguous()
    ws = library.new_workspace()
    library.set_kernel_timing(ws, True)
    out = torch_api.run_batch(spec, p, precision=precision, grad=grad, ws=ws)
    assert (library.get_kernel_time(ws, "atm_list")[1] > 0) == lists
    # mixed lists form the three-body term in FP32, the pair sums in FP64
    mixed = precision == "mixed"
    for q in (0, m - 1):
        one = torch_api.get_dispersion_batch([systems[q]], precision=precision, grad=grad)
        e, er = out["energy"][q].item(), one["energy"][0].item()
        assert abs(e - er) <= (1e-8 * n if mixed else 1e-10 * abs(er)), (e, er)
        if grad:
            g, s = out["gradient"][q * n:(q + 1) * n], out["sigma"][q]
            assert (g - one["gradient"]).abs().max().item() <= (1e-7 if mixed else 1e-9)
            assert (s - one["sigma"][0]).abs().max().item() <= (1e-7 * n if mixed else 1e-9)
