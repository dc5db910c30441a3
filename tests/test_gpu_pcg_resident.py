"""The resident Jacobi-PCG loop (one kernel for the whole solve) against the
launch-per-kernel loop, over the forms both accept: every cell-centred BC type,
periodic directions, rows and planes that do not divide into the blocks, one
block and many, both operators, and a solve whose waits are given up.

The two loops round every cell's arithmetic alike and differ only in the order
in which the dot products' block sums are added, so they take the same number
of iterations and agree to the 1e-10 that the solvers' parity tests ask."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N6, D6 = ["Neumann"] * 6, ["Dirichlet"] * 6
PER = ["Periodic", "Periodic"]
# (cells, BC types): planes 1, 2, 4, 8 and 16 a thread, ragged last blocks, one row a block, rows of 2 and of 300 cells
CASES = [
    ((16, 16, 16), N6), ((18, 15, 17), PER + ["Neumann", "Dirichlet", "Symmetric", "Antisymmetric"]),
    ((2, 9, 5), N6), ((5, 2, 7), D6), ((6, 7, 2), N6),  # a direction of 2 cells is the least a mesh may have
    ((32, 32, 32), ["Dirichlet", "Neumann"] + PER + PER), ((300, 5, 9), ["Neumann", "Dirichlet"] + N6[:4]),
    ((50, 39, 45), PER + PER + PER), ((64, 63, 65), D6), ((100, 67, 70), ["Robin"] * 2 + ["Neumann"] * 4),
    ((128, 96, 101), PER + N6[:4]),
    ((80, 81, 77), N6), ((130, 59, 50), PER + ["Neumann", "Dirichlet", "Symmetric", "Antisymmetric"]),
]


def nodes(gpu, n, beta):
    if beta is None or n < 4:
        return gpu.nodes_uniform(0.0, 1.0, n)
    return gpu.nodes_roberts_both(0.0, 1.0, n, beta)


def solve(gpu, monkeypatch, spins, n, types, op, isp):
    if spins is None:
        monkeypatch.delenv("MOONS_RESIDENT_SPINS", raising=False)
    else:
        monkeypatch.setenv("MOONS_RESIDENT_SPINS", str(spins))
    rng = np.random.default_rng(sum(n))
    periodic = [types[2 * d] == "Periodic" for d in range(3)]
    m = gpu.mesh(*[nodes(gpu, n[d], None if periodic[d] else 1.1) for d in range(3)])
    alln = op == "Lap_uniform_SF" and all(t in ("Neumann", "Periodic", "Symmetric") for t in types)
    b = gpu.SF(m, "CC").upload(np.asfortranarray(rng.standard_normal(m.shape(0))))
    x = gpu.SF(m, "CC").upload(np.asfortranarray(rng.standard_normal(m.shape(0))))
    x.set_BCs(types, list(rng.random(6)) if not alln else None, all_Neumann=alln, c_w=[0.3] * 6)
    P = gpu.PCG_solver_SF(m, x, gpu.iter_solver_params(*isp), op=op)
    if op == "nrg_diffusion":
        P.set_k([gpu.SF(m, 1 << d).upload(np.asfortranarray(1.0 + 0.2 * rng.random(m.shape(1 << d)))) for d in range(3)])
        P.update_MFP(-1e-3)
    info = P.solve(x, b)
    # the loop that ran: resident unless the bound of its waits is 0 (no plan) or 1 (given up)
    planes, blocks, given_up = P.resident()
    assert (planes > 0 and blocks > 0, given_up) == {None: (True, 0), 0: (False, 0), 1: (False, 1)}[spins]
    return info, x.download()


def agree(a, b):
    (ia, xa), (ib, xb) = a, b
    assert (ia.iterations, ia.exit_loop) == (ib.iterations, ib.exit_loop), (ia, ib)
    assert ia.res_norm0 == ib.res_norm0
    assert np.linalg.norm(xa - xb) <= 1e-10 * np.linalg.norm(xb), np.linalg.norm(xa - xb) / np.linalg.norm(xb)


@pytest.mark.parametrize("op", ["Lap_uniform_SF", "nrg_diffusion"])
@pytest.mark.parametrize("n,types", CASES)
def test_resident_loop_equals_launched_loop(gpu, monkeypatch, n, types, op):
    print(f"resident PCG {n} {types} {op}", flush=True)
    isp = (40, 1e-9, 1e-300, 1)
    agree(solve(gpu, monkeypatch, None, n, types, op, isp), solve(gpu, monkeypatch, 0, n, types, op, isp))


def test_cases_take_every_plane_count(gpu, monkeypatch):
    monkeypatch.delenv("MOONS_RESIDENT_SPINS", raising=False)
    planes = set()
    for n, types in CASES:
        m = gpu.mesh(*[nodes(gpu, q, None) for q in n])
        x = gpu.SF(m, "CC").set_BCs(types)
        planes.add(gpu.PCG_solver_SF(m, x, gpu.iter_solver_params(1, 1e-9, 1e-300, 1)).resident()[0])
    assert planes == {1, 2, 4, 8, 16}


def test_exits_of_the_resident_loop(gpu, monkeypatch):
    """Both loops stop at the same iteration for the same reason: either tolerance, the iteration limit, a check every
    third iteration, and a start that already meets the absolute tolerance.  (The x of a solve stopped at a residual is
    defined to that residual only; the x of equal iterations is compared above.)"""
    for isp in [(2000, 1e-8, 1e-300, 1), (2000, 1e-300, 1e-9, 1), (2000, 1e-6, 1e-300, 3), (7, 1e-30, 1e-300, 3),
                (50, 1e-8, 1e9, 1)]:
        print(f"resident PCG exits {isp}", flush=True)
        (ia, _), (ib, _) = (solve(gpu, monkeypatch, s, (20, 18, 22), N6, "Lap_uniform_SF", isp) for s in (None, 0))
        assert (ia.iterations, ia.exit_loop, ia.res_norm0) == (ib.iterations, ib.exit_loop, ib.res_norm0), (ia, ib)
        for i in (ia, ib):
            assert bool(i.exit_loop & 1) == (i.res_norm / i.res_norm0 < isp[1])
            assert bool(i.exit_loop & 2) == (i.res_norm < isp[2])


def test_given_up_wait_solves_by_launches(gpu, monkeypatch):
    """With a bound of one look at a slot the resident kernel returns at once and the launched loop gives the result."""
    print("resident PCG given up", flush=True)
    isp = (200, 1e-9, 1e-300, 1)
    ia, xa = solve(gpu, monkeypatch, 1, (64, 63, 65), D6, "Lap_uniform_SF", isp)
    ib, xb = solve(gpu, monkeypatch, 0, (64, 63, 65), D6, "Lap_uniform_SF", isp)
    assert (ia.iterations, ia.res_norm) == (ib.iterations, ib.res_norm)
    np.testing.assert_array_equal(xa, xb)


def test_given_up_once_is_not_tried_again(gpu, monkeypatch):
    """After one given-up solve the solver's next ones are launched, with the launched loop's bits, and do not wait."""
    print("resident PCG given up, solved again", flush=True)
    m = gpu.mesh(*[gpu.nodes_uniform(0.0, 1.0, 20)] * 3)
    b = gpu.SF(m, "CC").upload(np.asfortranarray(np.random.default_rng(2).standard_normal(m.shape(0))))
    got = []
    for spins in ("1", "0"):
        monkeypatch.setenv("MOONS_RESIDENT_SPINS", spins)
        x = gpu.SF(m, "CC").set_BCs(D6)
        P = gpu.PCG_solver_SF(m, x, gpu.iter_solver_params(200, 1e-9, 1e-300, 1))
        assert (P.resident()[0] > 0) == (spins == "1")
        for _ in range(3):
            x.fill(0.0)
            info = P.solve(x, b)
            got.append((info.iterations, info.res_norm, x.download().tobytes()))
            assert P.resident() == (0, 0, int(spins))
    assert len(set(got)) == 1
