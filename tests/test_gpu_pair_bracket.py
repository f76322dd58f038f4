"""Direct Coulomb force of single pairs, 0.75 A to the cutoff, from the
force-only rows with and without LJ and from the soft-core module, against 64
bits: within 2e-6 relative where beta r < 1 and 2e-5 up to the cutoff, where the
force factor has fallen to 1e-3 of q q / r^3 (the bracket's own bounds, in
test_ewald_bracket_fit, with up to three ulps of 1/r and, at the far end, 18 times
the rounding of r).  Coordinates are multiples of 2^-10, so that displacements
are exact."""
import numpy as np
import pytest
from scipy.special import erfc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", ["coulomb", "lj", "soft_core"])
@pytest.mark.parametrize("tolerance", [1e-4, 1e-5])
def test_pairs(dev, rows, tolerance):
    import torch
    from oracle import oracle as O
    from sponge_amd import abi
    print(f"case: {rows} rows, tolerance {tolerance}", flush=True)
    rng = np.random.default_rng(17)
    m, L, cutoff = 5, 125.0, 10.0
    g = (np.stack(np.meshgrid(*(np.arange(m),) * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5) * L / m
    r = np.linspace(0.75, cutoff - 0.02, len(g))
    u = rng.normal(size=g.shape)
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    grid = lambda a: np.round(a * 1024.0) / 1024.0  # noqa: E731
    x = np.stack([grid(g), grid(g + r[:, None] * u)], 1).reshape(-1, 3).astype(np.float32)
    q = np.tile(np.array([3.25, -5.5], np.float32), len(g))
    N = len(x)
    beta = float(O.get_beta(cutoff, tolerance))
    t = lambda a: torch.tensor(a, device=dev)  # noqa: E731
    xd, qd, f = t(x), t(q), torch.zeros(N, 3, device=dev)
    box = abi.Box([L] * 3)
    nl = abi.NeighborList(N, cutoff, 2.0, box)
    # packed pairs (0,0), (1,0), (1,1): the atoms are of type 0, whose
    # coefficients with the absent type 1 decide whether its rows evaluate LJ
    A = np.array([0.0, 1.0 if rows == "lj" else 0.0, 0.0], np.float32)
    types = np.zeros(N, np.int32)
    torch.cuda.synchronize()
    nl.update(xd, update=abi.NL_FORCED)
    if rows == "soft_core":
        sc = abi.LJSoftCore(N, A, A, A, A, types, types, cutoff, **{"lambda": 0.5})
        sc.direct_force(nl, xd, qd, f, box, beta)
    else:
        lj = abi.LennardJones(N, 2, A, A, types, cutoff)
        lj.direct_force(nl, xd, qd, f, box, beta)
    torch.cuda.synchronize()
    f = f.cpu().numpy().astype(np.float64).reshape(-1, 2, 3)
    d = np.diff(x.astype(np.float64).reshape(-1, 2, 3), axis=1)[:, 0]
    R = np.linalg.norm(d, axis=1)
    b = beta * R
    want = (float(q[0]) * float(q[1]) * (erfc(b) + 2 / np.sqrt(np.pi) * b * np.exp(-b * b)) / R ** 3)[:, None] * d
    for side, sign in ((0, -1.0), (1, 1.0)):
        e = np.linalg.norm(f[:, side] - sign * want, axis=1) / np.linalg.norm(want, axis=1)
        print(f"    largest relative error {e[b < 1].max():.2e} below beta r = 1, {e.max():.2e}")
        assert e[b < 1].max() < 2e-6
        assert e.max() < 2e-5
