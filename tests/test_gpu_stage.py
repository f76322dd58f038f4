"""The stage of the pair kernels holds the streams that exist: sheared cells and
axes of four cells (streams of the whole stencil) from the start, a liquid in a
half or an eighth of its box (streams of twice the mean and more) and one that
condenses after the first build once a force call has met them, with the same
forces on both sides of it (FP64 oracle, test_gpu_streams.check_force); in the
step driver with captured steps as without."""
import dataclasses

import numpy as np
import pytest

from gpu_helpers import DevSystem
from test_gpu_streams import box_case, check_force

pytestmark = pytest.mark.gpu


def stretched(s, n):
    """The liquid of s in a corner of a box n times as long."""
    return dataclasses.replace(s, box=(s.box * np.array(n)).astype(np.float32))


def sheared(s):
    """A lower-triangular cell of the same lengths and its inverse, with the
    molecules moved to their fractional coordinates in it."""
    from sponge_amd import abi
    L = s.box.astype(np.float64)
    M = np.array([[L[0], 0, 0], [0.2 * L[0], L[1], 0], [0.1 * L[0], -0.15 * L[1], L[2]]])
    o = s.crd.reshape(-1, 3, 3)[:, :1].astype(np.float64)
    crd = (s.crd.reshape(-1, 3, 3) + ((o / L) @ M - o)).reshape(-1, 3).astype(np.float32)
    low = (np.array([0, 1, 1, 2, 2, 2]), np.array([0, 0, 1, 0, 1, 2]))
    return crd, abi.Box.from_cell(M[low], np.linalg.inv(M)[low])


def case(name):
    from sponge_amd import abi
    from sponge_amd import system as S
    if name in ("4_cells", "elongated", "uneven"):
        s = box_case(name)
    elif name == "sheared":
        s = S.water_box(1381, cutoff=8.0, seed=8)
        return (s,) + sheared(s)
    else:
        n = {"half": (1, 1, 2), "eighth": (2, 2, 2)}[name]
        s = stretched(S.water_box(1381, cutoff=8.0, seed=9), n)
    return s, s.crd, abi.Box(s.box)


def force(nl, lj, d, box, beta):
    import torch
    f = d.zeros(d.N, 3)
    torch.cuda.synchronize()
    lj.direct_force(nl, d.crd, d.charge, f, box, beta)
    torch.cuda.synchronize()
    return f.cpu().numpy()


@pytest.mark.parametrize("name", ["uneven", "4_cells", "elongated", "sheared", "half", "eighth"])
def test_streams_are_staged(dev, name):
    import torch
    from oracle import oracle as O
    from sponge_amd import abi
    s, crd, box = case(name)
    d = DevSystem(s, dev, crd)
    beta = O.get_beta(s.cutoff, s.tolerance)
    nl = abi.NeighborList(d.N, s.cutoff, s.skin, box)
    lj = abi.LennardJones(d.N, s.n_types, s.lj_A, s.lj_B, s.lj_type, s.cutoff)
    torch.cuda.synchronize()
    nl.update(d.crd, update=abi.NL_FORCED, excl=d.excl)
    longest, before = nl.stream_info()
    f = force(nl, lj, d, box, beta)
    longest, staged = nl.stream_info()
    print(f"case: {name}: longest stream {longest}, staged {before}, then {staged}", flush=True)
    assert 0 < longest <= staged <= 3584
    if name not in ("half", "eighth"):
        assert longest <= before
    if name != "sheared":
        check_force(f, s)
        check_force(force(nl, lj, d, box, beta), s)


def test_condensing_liquid(dev):
    import torch
    from oracle import oracle as O
    from sponge_amd import abi
    from sponge_amd import system as S
    s = stretched(S.water_box(1381, cutoff=8.0, seed=10), (2, 2, 2))
    oxygen = np.repeat(s.crd[::3], 3, axis=0)
    print("case: liquid in an eighth of its box after a gas", flush=True)
    d = DevSystem(s, dev)
    gas = torch.tensor(s.crd + oxygen, device=dev)  # twice the distances: an eighth of the density
    box = abi.Box(s.box)
    nl = abi.NeighborList(d.N, s.cutoff, s.skin, box)
    lj = abi.LennardJones(d.N, s.n_types, s.lj_A, s.lj_B, s.lj_type, s.cutoff)
    beta = O.get_beta(s.cutoff, s.tolerance)
    torch.cuda.synchronize()
    nl.update(gas, update=abi.NL_FORCED, excl=d.excl)
    lj.direct_force(nl, gas, d.charge, d.zeros(d.N, 3), box, beta)
    longest, staged = nl.stream_info()
    assert longest <= staged
    nl.update(d.crd, update=abi.NL_FORCED, excl=d.excl)
    longest, staged = nl.stream_info()
    assert longest > staged
    check_force(force(nl, lj, d, box, beta), s)
    longest, staged = nl.stream_info()
    assert longest <= staged <= 3584
    check_force(force(nl, lj, d, box, beta), s)


def test_step_driver(dev):
    import ctypes as C
    from sponge_amd import abi
    from sponge_amd import system as S
    s = stretched(S.water_box(700, cutoff=8.0, seed=11), (1, 1, 2))
    print("case: captured steps of a liquid in half of its box", flush=True)
    eager, captured = abi.MDSystem(s), abi.MDSystem(s)
    eager.run(41)
    for n in (1, 20, 20):
        captured.run(n, use_graph=True)
    x, y = eager.state()[0], captured.state()[0]
    assert np.abs(x.astype(np.float64) - y).max() < 1e-3
    nl, _, _ = captured.handles()
    longest, staged = C.c_int(), C.c_int()
    assert captured.lib.sponge_nl_stream_info(nl, C.byref(longest), C.byref(staged)) == 0
    assert longest.value <= staged.value
