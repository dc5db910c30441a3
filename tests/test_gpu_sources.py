"""The fused source kernels at the sizes where their numbering can go wrong:
the smallest grids, remainders of a block, one long direction, against the
oracle (bit equality), and calls that only the sequence of passes covers."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (3, 2, 5), (64, 2, 2), (2, 67, 3), (2, 3, 130), (17, 13, 9)]


def _rand(shape, seed):
    return np.asfortranarray(np.random.default_rng(seed).standard_normal(shape))


def _grid(gpu, n):
    hs = [O.roberts_both_nodes(0, 1 + d, n[d], 1.1) for d in range(3)]
    return O.Grid(*hs), gpu.mesh(*hs)


@pytest.mark.parametrize("n", SHAPES)
def test_advect_b_sizes(gpu, n):
    g, m = _grid(gpu, n)
    U_E = [_rand(g.shape(dl), q) for q, dl in enumerate((6, 6, 5, 5, 3, 3))]
    B = [_rand(g.shape(1 << d), 10 + d) for d in range(3)]
    gU = [gpu.SF(m, dl).upload(u) for u, dl in zip(U_E, (6, 6, 5, 5, 3, 3))]
    gB = [gpu.SF(m, 1 << d).upload(B[d]) for d in range(3)]
    tmp = [gpu.SF(m, dl) for dl in (5, 3, 6, 3, 6, 5)]
    E = [gpu.SF(m, dl) for dl in (6, 5, 3)]
    adv = [gpu.SF(m, 1 << d) for d in range(3)]
    ref = O.advect_B(g, U_E, B)
    gpu.advect_B(adv, gU, gB, tmp, E)
    for d in range(3):
        np.testing.assert_array_equal(adv[d].download(), ref[d])
    # the six interpolants are results as well
    for q, (c, dl) in enumerate(((0, 5), (0, 3), (1, 6), (1, 3), (2, 6), (2, 5))):
        orth = next(d for d in range(3) if ((1 << c) ^ dl) == 1 << d)
        np.testing.assert_array_equal(tmp[q].download(), O.interp(g, B[c], 1 << c, dl, orth))
    # in place: E over U_E's first entry of each edge, adv over B
    Ea = [gU[0], gU[2], gU[4]]
    gpu.advect_B(gB, gU, gB, tmp, Ea)
    for d in range(3):
        np.testing.assert_array_equal(gB[d].download(), ref[d])


@pytest.mark.parametrize("n", SHAPES)
@pytest.mark.parametrize("periodic", [None, 0, 2])
def test_div_is_three_del_passes(gpu, n, periodic):
    g, m = _grid(gpu, n)
    u = [gpu.SF(m, 1 << d).upload(_rand(g.shape(1 << d), 20 + d)) for d in range(3)]
    types = ["Neumann"] * 6
    if periodic is not None:
        types[2 * periodic] = types[2 * periodic + 1] = "Periodic"
    out, ref = gpu.SF(m, "CC").set_BCs(types), gpu.SF(m, "CC")
    gpu.div(out, *u)
    for d in range(3):
        gpu.del_op(ref, u[d], 1, d, 0, 1 if d == 0 else 2)
    want = ref.download()
    for d in range(3):
        if d != periodic:
            np.moveaxis(want, d, 0)[[0, -1]] = 0.0
    np.testing.assert_array_equal(out.download(), want)


BC_SETS = [
    (["Dirichlet", "Neumann", "Neumann", "Dirichlet", "Robin", "Symmetric"], [0.3, -0.2, 0.7, 1.0, 0.5, 0.1]),
    (["Periodic", "Periodic", "Robin", "Robin", "Antisymmetric", "Dirichlet"], [0, 0, 0.2, -0.4, 0.1, 0.6]),
    (["Robin", "Dirichlet", "Periodic", "Periodic", "Periodic", "Periodic"], [0.4, 1.5, 0, 0, 0, 0]),
    (["none", "Dirichlet", "Neumann", "none", "none", "none"], [0, 0.3, 0.2, 0, 0, 0]),
]


@pytest.mark.parametrize("n", SHAPES)
@pytest.mark.parametrize("bc", range(len(BC_SETS)))
@pytest.mark.parametrize("implicit", [False, True])
def test_apply_bcs_sizes(gpu, n, bc, implicit):
    """Every face's rule in one launch: edges and corners as the face sequence leaves them."""
    g, m = _grid(gpu, n)
    types, vals = BC_SETS[bc]
    cw = [0.01, 0.02, 0.5, 1.0, 3.0, 0.07]
    for dl in range(8):
        u = _rand(g.shape(dl), 30 + dl)
        ref = u.copy(order="F")
        O.apply_bcs(g, ref, dl, O.BCs.make(types, vals, cw), implicit)
        U = gpu.SF(m, dl).upload(u).set_BCs(types, vals, c_w=cw)
        (gpu.apply_BCs_implicit if implicit else gpu.apply_BCs)(U)
        np.testing.assert_array_equal(U.download(), ref, err_msg=f"dl={dl}")
