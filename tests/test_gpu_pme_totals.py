"""Energies and virial of the reciprocal part from the per-workgroup partial
sums: atom counts around the bin pass's 256, each of energy and virial alone,
and, on a grid of the three passes, FFT tilings with the fewest and the most
workgroups (on a grid of whole planes there is one per plane).  Against the FP64
oracle within 1e-5 (the charge grid and its transform are FP32; a partial sum
left out or taken twice shows at 1e-3 or more); the self and neutralizing
energy, FP64 sums of exact FP32 products rounded once, within 1e-6."""
import ctypes as C

import numpy as np
import pytest

from gpu_helpers import DevSystem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fft", [(36, 40, 45), (70, 75, 45)], ids=["plane", "three_passes"])
@pytest.mark.parametrize("n, tiles", [(1, None), (255, (2, 2, 2)), (256, (16, 16, 16)), (257, None),
                                      (1944, (4, 8, 14))])
def test_totals(dev, n, tiles, fft):
    import torch
    from oracle import oracle as O
    from sponge_amd import abi
    from sponge_amd import system as S
    s = S.config(1)
    print(f"case: {n} atoms, tiling {tiles}, fft {fft}", flush=True)
    d = DevSystem(s, dev)
    crd, charge = d.crd[:n].contiguous(), d.charge[:n].contiguous()
    pm = abi.ParticleMesh(n, abi.Box(s.box), s.cutoff, fftx=fft[0], ffty=fft[1], fftz=fft[2])
    if tiles:
        assert pm.lib.sponge_pme_set_fft_tiling(pm.h, (C.c_int * 3)(*tiles)) == 0
    beta = O.get_beta(s.cutoff, s.tolerance)
    ref = O.pme64(s.crd[:n], s.charge[:n], s.box, beta, fft)
    q = s.charge[:n].astype(np.float64)
    self_energy = (-beta / np.sqrt(np.pi) * (q * q).sum()
                   - 0.5 * np.pi / (beta ** 2 * np.prod(s.box.astype(np.float64))) * q.sum() ** 2)
    for energy, virial in ((True, True), (True, False), (False, True)):
        frc, pot, vir = d.zeros(n, 3), d.zeros(1), d.zeros(6)
        pm.reciprocal_force(crd, charge, frc, virial=vir if virial else None,
                            potential=pot if energy else None)
        torch.cuda.synchronize()
        if energy:
            e = pm.step_print()
            assert abs(e["reciprocal"] - ref["reciprocal"]) < 1e-5 * abs(ref["reciprocal"])
            assert abs(e["self_energy"] - self_energy) < 1e-6 * abs(self_energy)
            assert abs(float(pot.cpu()[0]) - (e["reciprocal"] + e["self_energy"])) < 1e-6 * abs(self_energy)
        if virial:
            v = vir.cpu().numpy().astype(np.float64)
            assert np.linalg.norm(v - ref["virial"]) < 1e-5 * np.linalg.norm(ref["virial"])
