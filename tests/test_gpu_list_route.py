"""Three-body lists of molecules above the sizes of the pair sums: lists by
storage order, with the dense form of the kernel for tile pairs that are mostly
within the cutoff.  Compared with the oracle at the bars of the parity tests."""
import sys

import numpy as np
import pytest
import torch

import oracle as O
from helpers import BJ, ZERO, cell

pytestmark = pytest.mark.gpu


def _step(msg):
    print(f"[gpu-list-route] {msg}", flush=True)
    sys.stdout.flush()


def _molecule(seed, n, shape):
    """n atoms at about 0.1 per cubic Angstrom in random order, at least 1 Angstrom apart."""
    rng = np.random.default_rng(seed)
    grid = np.stack(np.meshgrid(*[np.arange(m) for m in shape], indexing="ij"), axis=-1).reshape(-1, 3)[:n]
    pos = 4.07 * (rng.permutation(grid) + rng.uniform(-0.23, 0.23, (n, 3)))
    return rng.choice([1, 6, 7, 8], size=n, p=[0.5, 0.3, 0.1, 0.1]), pos


def _reference(s, grad=True):
    c = {**dict(disp2=60.0, disp3=40.0, cn=40.0, width2=0.0, width3=0.0), **s.get("cutoff", {})}
    return O.dispersion(s["numbers"], s["positions"], s.get("lattice"), [True] * 3 if "lattice" in s else None,
                        O.ZERO if s.get("kind") == "zero" else O.RATIONAL, s["param"],
                        (c["cn"], c["disp2"], c["disp3"], c["width2"], c["width3"]), grad=grad)


def _compare(out, off, k, ref, n, mixed, grad):
    e, er = out["energy"][k].item(), ref["energy"]
    assert abs(e - er) <= (1e-8 * n if mixed else 1e-10 * abs(er)), (k, e, er)
    if grad:
        assert np.abs(out["gradient"][off:off + n].cpu().numpy() - ref["gradient"]).max() <= (1e-7 if mixed else 1e-9)
        assert np.abs(out["sigma"][k].cpu().numpy() - ref["virial"]).max() <= (1e-7 * n if mixed else 1e-9)


@pytest.mark.parametrize("n,shape,disp3,m", [(1751, (13, 13, 11), 40.0, 1), (300, (7, 7, 7), 12.0, 14)])
def test_capture_without_an_evaluation_before(n, shape, disp3, m):
    """A plan holds every buffer of an evaluation, so that its first one can
    be recorded: lists of a large molecule, and of a batch of small ones with
    a short cutoff."""
    from dftd3 import library, torch_api
    _step(f"capture first, {m} x {n} atoms")
    num, pos = _molecule(n, n, shape)
    s = dict(numbers=num, positions=pos, param=BJ, cutoff=dict(disp3=disp3))
    spec, p = torch_api.batch_spec([s] * m)
    p = torch.as_tensor(p, dtype=torch.float64, device="cuda").contiguous()
    plan = torch_api.BatchPlan(spec, p, precision="mixed")
    plan.capture()
    ref = _reference(s)
    for _ in range(3):
        for v in plan.out.values():
            v.zero_()
        _compare(plan.replay(), 0, 0, ref, n, True, True)


def _noalloc(systems, precision, grad, lists=True):
    """The allocation-free entry point, which keeps the lists when the records
    and sums of the pair sums (48 bytes a pair of atoms) exceed 16 MiB."""
    from dftd3 import library, torch_api
    assert not lists or 48 * sum(len(s["numbers"]) ** 2 for s in systems if "lattice" not in s) > 16 << 20
    spec, pos = torch_api.batch_spec(systems)
    p = torch.as_tensor(pos, dtype=torch.float64, device="cuda").contiguous()
    out = dict(energy=torch.empty(len(spec), dtype=torch.float64, device="cuda"),
               gradient=torch.empty(len(pos), 3, dtype=torch.float64, device="cuda"),
               sigma=torch.empty(len(spec), 3, 3, dtype=torch.float64, device="cuda"))
    prec = {"fp64": library.PRECISION_FP64, "mixed": library.PRECISION_MIXED}[precision]
    library.get_dispersion_batch_noalloc(
        spec.natoms, spec.numbers, spec.lattices, spec.periodic, spec.params, spec.cutoffs, prec, p.data_ptr(),
        out["energy"].data_ptr(), out["gradient"].data_ptr() if grad else None,
        out["sigma"].data_ptr() if grad else None, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("scale", [1.0, 1.0 + 3e-10, 1.0 - 3e-10])
@pytest.mark.parametrize("k", [4, 54])
def test_distances_at_the_cutoff(k, scale, precision, grad):
    """A 10 x 9 x 8 grid of spacing 3 bohr in random order with a three-body
    cutoff of 3 sqrt(k) bohr, at the cutoff to the last bit, or inside the band
    that the reference's arithmetic decides, for listed pairs and for the third
    side of the triples: short lists (4) and a cutoff that most tile pairs are
    within (54, a distance of 10,144 pairs)."""
    _step(f"cutoff band, k={k}, scale 1{scale - 1.0:+.0e}, {precision}, grad={grad}")
    rng = np.random.default_rng(9)
    g = np.array([[x, y, z] for x in range(10) for y in range(9) for z in range(8)], dtype=float)
    pos = 3.0 * scale * rng.permutation(g) + np.array([0.1, 0.7, -0.3])
    cut = 3.0 * np.sqrt(float(k))
    s = dict(numbers=rng.choice([1, 6], size=len(pos)), positions=pos, param=BJ, cutoff=dict(disp3=cut))
    _compare(_noalloc([s], precision, grad), 0, 0, _reference(s, grad), len(pos), precision == "mixed", grad)


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,kind,alp,width3", [(640, "rational", 14.0, 0.0), (641, "zero", 14.0, 8.0),
                                               (703, "rational", 16.0, 0.0)])
def test_long_lists_among_others(n, kind, alp, width3, precision, grad):
    """One large molecule (whole tiles, one atom past them, a ragged last
    tile) with a small molecule and a cell, whose lists keep the reference's
    triangle."""
    _step(f"{n} atoms {kind} alp={alp} width3={width3} {precision} grad={grad}")
    num, pos = _molecule(n, n, (9, 9, 9))
    cutoff = dict(width3=width3)
    systems = [dict(numbers=num, positions=pos, param=dict(ZERO if kind == "zero" else BJ, alp=alp), kind=kind,
                    cutoff=cutoff)]
    num, pos = _molecule(3, 30, (4, 4, 4))
    systems.append(dict(numbers=num, positions=pos, param=BJ, cutoff=cutoff))
    num, pos, lat = cell(17, 12, 13.0)
    systems.append(dict(numbers=num, positions=pos, lattice=lat, periodic=[True] * 3, param=BJ, cutoff=cutoff))
    out, off = _noalloc(systems, precision, grad), 0
    for k, s in enumerate(systems):
        _compare(out, off, k, _reference(s, grad), len(s["numbers"]), precision == "mixed", grad)
        off += len(s["numbers"])


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,shape,cutoff", [(640, (4, 4, 40), dict(disp3=20.0, disp2=30.0)),
                                            (611, (1, 25, 25), dict(disp3=15.0, disp2=12.0, width3=4.0)),
                                            (777, (1, 1, 777), dict())])
def test_tile_culling(n, shape, cutoff, precision, grad):
    """Molecules longer than the cutoffs: tiles out of range in the loops of
    the lists and of the two-body term, tile pairs mostly out of range."""
    _step(f"{n} atoms {shape} {cutoff} {precision} grad={grad}")
    num, pos = _molecule(n, n, shape)
    s = dict(numbers=num, positions=pos, param=BJ, cutoff=cutoff)
    _compare(_noalloc([s], precision, grad), 0, 0, _reference(s, grad), n, precision == "mixed", grad)


@pytest.mark.parametrize("n,shape,disp3,runs", [(1751, (13, 13, 11), 40.0, [("mixed", True)]),
                                                (3501, (16, 16, 14), 24.0, [("fp64", True), ("fp64", False),
                                                                            ("mixed", False)])])
def test_every_launch_shape(n, shape, disp3, runs):
    """Every launch shape of the kernels with the dense form, through plans
    above the sizes of the pair sums, and graph replays of the last."""
    from dftd3 import library, torch_api
    num, pos = _molecule(n, n, shape)
    s = dict(numbers=num, positions=pos, param=BJ, cutoff=dict(disp3=disp3))
    ref = _reference(s)
    spec, p = torch_api.batch_spec([s])
    p = torch.as_tensor(p, dtype=torch.float64, device="cuda").contiguous()
    for precision, grad in runs:
        ws = library.new_workspace()
        library.set_kernel_timing(ws, True)
        _compare(torch_api.run_batch(spec, p, precision=precision, grad=grad, ws=ws), 0, 0, ref, n,
                 precision == "mixed", grad)
        assert library.get_kernel_time(ws, "atm_list")[1] > 0
        plan = torch_api.BatchPlan(spec, p, precision=precision, grad=grad)
        for waves, bpc in library.plan_candidate_shapes():
            _step(f"{n} atoms {precision} grad={grad} waves={waves} blocks/CU={bpc}")
            plan.set_shape(waves, bpc)
            out = {k: torch.zeros_like(v) for k, v in plan.out.items()}
            _compare(plan.execute(out=out), 0, 0, ref, n, precision == "mixed", grad)
        plan.capture()
        for _ in range(3):
            for v in plan.out.values():
                v.zero_()
            _compare(plan.replay(), 0, 0, ref, n, precision == "mixed", grad)
        assert not plan.overflowed()


def test_work_area_that_holds_the_lists_only():
    """A molecule and a cell that exceed the work area of the allocation-free
    entry point (65 MiB) with the records and sums of the molecule's pair sums
    (48 bytes a pair of atoms) and fit it with lists (72 bytes a slot)."""
    _step("work area that holds the lists only")
    n, nc = 590, 310
    num, pos = _molecule(n, n, (9, 9, 9))
    cnum, cpos, lat = cell(41, nc, 28.0)
    img = np.array([[i, j, k] for i in range(-2, 3) for j in range(-2, 3) for k in range(-2, 3)]) @ lat
    slots = 0
    for t in img:
        d2 = ((cpos[None] + t - cpos[:, None]) ** 2).sum(-1)
        slots += int(np.tril((d2 <= 1600.0) & (d2 > 1e-12)).sum())
    area, records = 65 << 20, 32 * (n * n + nc * nc)
    assert 48 * n * n <= 16 << 20
    assert records + 72 * (slots + n * (n - 1) // 2) + (1 << 20) < area < records + 72 * slots + 48 * n * n, slots
    systems = [dict(numbers=num, positions=pos, param=BJ),
               dict(numbers=cnum, positions=cpos, lattice=lat, periodic=[True] * 3, param=BJ)]
    from dftd3 import torch_api
    ref = torch_api.get_dispersion_batch(systems, precision="fp64")
    out = _noalloc(systems, "fp64", True, lists=False)
    assert ((out["energy"] - ref["energy"]).abs() <= 1e-12 * ref["energy"].abs()).all()
    for key in ("gradient", "sigma"):
        assert (out[key] - ref[key]).abs().max() <= 1e-11 * ref[key].abs().max(), key
