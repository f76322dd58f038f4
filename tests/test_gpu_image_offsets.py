"""Direct Coulomb forces (no LJ) of the module's force-only call, whose partners
are staged as offsets from a cell's centre: no further from the FP64 oracle than
the FP32 restatement of the reference, which rounds the minimum image of the
coordinates; wrapped coordinates, and molecules a box length or two away."""
import dataclasses

import numpy as np
import pytest

from gpu_helpers import DevSystem, rel_rms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("unwrapped", [False, True])
@pytest.mark.parametrize("cutoff", [8.0, 9.0, 10.0])
def test_coulomb_force(dev, cutoff, unwrapped):
    import torch
    from oracle import oracle as O
    from sponge_amd import abi
    from sponge_amd import system as S
    s = S.water_box(1381, cutoff=cutoff, seed=5)
    s = dataclasses.replace(s, lj_A=0 * s.lj_A, lj_B=0 * s.lj_B)
    crd = s.crd
    if unwrapped:
        n = np.random.default_rng(13).integers(-2, 3, (s.n_waters, 3))
        crd = (crd + np.repeat(n, 3, axis=0) * s.box).astype(np.float32)
    print(f"case: cutoff {cutoff}, unwrapped {unwrapped}", flush=True)
    beta = O.get_beta(cutoff, s.tolerance)
    c, ser, _ = O.nl_build(s, crd=crd)
    ref64 = O.direct64_list(s, beta, c, ser, crd=crd)["frc"]
    ref32 = O.lj_direct(s, c, ser, beta, crd=crd, need_energy=False, need_virial=False)["frc"]
    d = DevSystem(s, dev, crd)
    box = abi.Box(s.box)
    nl = abi.NeighborList(d.N, cutoff, s.skin, box)
    lj = abi.LennardJones(d.N, s.n_types, s.lj_A, s.lj_B, s.lj_type, cutoff)
    f = d.zeros(d.N, 3)
    torch.cuda.synchronize()
    nl.update(d.crd, update=abi.NL_FORCED, excl=d.excl)
    lj.direct_force(nl, d.crd, d.charge, f, box, beta)
    torch.cuda.synchronize()
    e, e32 = rel_rms(f.cpu().numpy(), ref64), rel_rms(ref32, ref64)
    print(f"    force error {e:.2e}, of the FP32 restatement {e32:.2e}")
    assert e <= e32
