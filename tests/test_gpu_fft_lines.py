"""The PME line transforms at every radix of the two-factor form (1..10, 12,
14, 15, 16 on either side), at lengths without two factors up to 16 (125,
162: the Stockham passes), mixed between axes, and at the smallest, ragged and
largest tilings, on a grid of whole planes (where only the z tiling reaches a
kernel), on one of two factors beyond them and on Stockham lengths on x and on
y: the convolved grid and the forces against the oracle within 1e-5 relative
RMS, reciprocal energy and virial against the FP64 oracle (gpu_helpers.
check_total)."""
import numpy as np
import pytest

from gpu_helpers import DevSystem, check_total, rel_rms

pytestmark = pytest.mark.gpu

GRIDS = [(70, 75, 98), (128, 27, 50), (125, 32, 45), (48, 125, 36), (30, 42, 162), (15, 16, 14),
         (7, 8, 12), (5, 6, 9), (20, 35, 24), (63, 64, 120)]


@pytest.fixture(scope="module")
def cfg1():
    from sponge_amd import system as S
    return S.config(1)


@pytest.mark.parametrize("fft", GRIDS, ids=["x".join(map(str, g)) for g in GRIDS])
def test_grid_force_energy_virial(dev, cfg1, fft):
    import torch
    from oracle import oracle as O
    from sponge_amd import abi
    s = cfg1
    print(f"case: fft {fft}", flush=True)
    beta = O.get_beta(s.cutoff, s.tolerance)
    p = O.PME(s, fft, beta)
    ref = p.reciprocal()
    ref64 = O.pme64(s.crd, s.charge, s.box, beta, fft)
    grids = p.grids()
    d = DevSystem(s, dev)
    pm = abi.ParticleMesh(d.N, abi.Box(s.box), s.cutoff, fftx=fft[0], ffty=fft[1], fftz=fft[2])
    frc, vir, pot, plain = d.zeros(d.N, 3), d.zeros(6), d.zeros(1), d.zeros(d.N, 3)
    F = d.zeros(int(np.prod(fft)))
    pm.reciprocal_force(d.crd, d.charge, frc, virial=vir, potential=pot)
    pm.reciprocal_force(d.crd, d.charge, plain)
    pm.grids(None, F)
    torch.cuda.synchronize()
    rec = pm.step_print()["reciprocal"]
    assert rel_rms(F.cpu().numpy(), grids["FBCFQ"]) < 1e-5
    assert rel_rms(frc.cpu().numpy(), ref["frc"]) < 1e-5
    assert rel_rms(plain.cpu().numpy(), ref["frc"]) < 1e-5
    check_total("reciprocal", rec, ref["reciprocal"], ref64["reciprocal"])
    check_total("virial", vir.cpu().numpy(), ref["virial"], ref64["virial"])


@pytest.mark.parametrize("fft", [(27, 50, 125), (70, 75, 45), (125, 36, 45), (36, 125, 45)],
                         ids=["plane", "three_passes", "stockham_x", "stockham_y"])
@pytest.mark.parametrize("tiles", [(2, 2, 2), (4, 6, 10), (16, 16, 16), (14, 8, 12)])
def test_tilings(dev, cfg1, tiles, fft):
    import ctypes as C
    import torch
    from oracle import oracle as O
    from sponge_amd import abi
    s = cfg1
    print(f"case: fft {fft}, tiles {tiles}", flush=True)
    beta = O.get_beta(s.cutoff, s.tolerance)
    ref = O.PME(s, fft, beta).reciprocal()
    ref64 = O.pme64(s.crd, s.charge, s.box, beta, fft)
    d = DevSystem(s, dev)
    pm = abi.ParticleMesh(d.N, abi.Box(s.box), s.cutoff, fftx=fft[0], ffty=fft[1], fftz=fft[2])
    t = (C.c_int * 3)(*tiles)
    assert pm.lib.sponge_pme_set_fft_tiling(pm.h, t) == 0
    frc, plain, vir, pot = d.zeros(d.N, 3), d.zeros(d.N, 3), d.zeros(6), d.zeros(1)
    pm.reciprocal_force(d.crd, d.charge, plain)
    pm.reciprocal_force(d.crd, d.charge, frc, virial=vir, potential=pot)
    torch.cuda.synchronize()
    assert rel_rms(plain.cpu().numpy(), ref["frc"]) < 1e-5
    assert rel_rms(frc.cpu().numpy(), ref["frc"]) < 1e-5
    check_total("reciprocal", pm.step_print()["reciprocal"], ref["reciprocal"], ref64["reciprocal"])
    check_total("virial", vir.cpu().numpy(), ref["virial"], ref64["virial"])
