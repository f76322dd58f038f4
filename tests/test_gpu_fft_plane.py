"""The x-y planes of the spectrum transformed in LDS: every radix of a factor
on both axes, very uneven planes, the largest plane that fits, and planes just
beyond it (three passes); convolved grid and forces against the oracle within
1e-5 relative RMS, the energy within 1e-6 of the FP64 sum over the FP64 spectrum
of the charge grid the pass read.  (The virial is held to the oracle on usual
grids in test_gpu_fft_lines; on uneven ones its terms cancel.)  A batch of
systems of both forms takes one of them and agrees with single runs."""
import dataclasses

import numpy as np
import pytest

from gpu_helpers import DevSystem, check_total, rel_rms

pytestmark = pytest.mark.gpu

GRIDS = [(256, 16, 8), (16, 256, 12), (225, 20, 9), (20, 225, 10), (196, 24, 8), (24, 144, 15),
         (100, 35, 12), (81, 48, 7), (63, 64, 16), (4, 5, 6), (7, 9, 5), (196, 25, 8), (96, 80, 12),
         (70, 112, 16)]


def spectrum(Q, s, beta):
    """Per point of a charge grid's spectrum, in FP64: frequencies m, m^2, the
    squared amplitude and the influence function."""
    n, box = Q.shape, s.box.astype(np.float64)
    P = np.abs(np.fft.fftn(Q.astype(np.float64))) ** 2
    k = [np.arange(m) for m in n]
    m = np.meshgrid(*(np.where(a > b // 2, a - b, a) / L for a, b, L in zip(k, n, box)), indexing="ij")
    m2 = m[0] ** 2 + m[1] ** 2 + m[2] ** 2
    m2[0, 0, 0] = 1.0
    b = [1 / np.abs(sum(w * np.exp(2j * np.pi * a * i / c) for i, w in enumerate((1 / 6, 4 / 6, 1 / 6)))) ** 2
         for a, c in zip(k, n)]
    bc = np.exp(-np.pi ** 2 * m2 / beta ** 2) / (np.pi * m2 * box.prod())
    bc *= b[0][:, None, None] * b[1][None, :, None] * b[2][None, None, :]
    bc[0, 0, 0] = 0.0
    return m, m2, P, bc


def spectrum_energy(Q, s, beta):
    """Reciprocal energy of a charge grid."""
    _, _, P, bc = spectrum(Q, s, beta)
    return 0.5 * (bc * P).sum()


def spectrum_virial(Q, s, beta):
    """Reciprocal virial (xx, xy, yy, xz, yz, zz) of a charge grid over the half
    spectrum, its first and last planes at half weight (PM_force.cpp:1024-1068),
    and the sums of its terms' magnitudes."""
    m, m2, P, bc = spectrum(Q, s, beta)
    half = Q.shape[2] // 2 + 1
    (x, y, z), m2, P, bc = [a[:, :, :half] for a in m], *(a[:, :, :half] for a in (m2, P, bc))
    w = np.ones(half)
    w[0] = w[-1] = 0.5
    f = 0.5 * w * bc * P
    t = 2.0 / m2 * (1.0 + np.pi ** 2 / beta ** 2 * m2)
    terms = [-f * (1 - t * x * x), f * t * x * y, -f * (1 - t * y * y), f * t * x * z,
             f * t * y * z, -f * (1 - t * z * z)]
    return (np.array([a.sum() for a in terms]),
            np.array([(f * (1 + t * c)).sum() for c in (x * x, abs(x * y), y * y, abs(x * z),
                                                         abs(y * z), z * z)]))


@pytest.mark.parametrize("fft", GRIDS, ids=["x".join(map(str, g)) for g in GRIDS])
def test_grid_force_energy(dev, fft):
    import torch
    from oracle import oracle as O
    from sponge_amd import abi
    from sponge_amd import system as S
    s = S.config(1)
    print(f"case: fft {fft}", flush=True)
    beta = O.get_beta(s.cutoff, s.tolerance)
    p = O.PME(s, fft, beta)
    ref = p.reciprocal()
    grids = p.grids()
    d = DevSystem(s, dev)
    pm = abi.ParticleMesh(d.N, abi.Box(s.box), s.cutoff, fftx=fft[0], ffty=fft[1], fftz=fft[2])
    frc, vir, pot, plain = d.zeros(d.N, 3), d.zeros(6), d.zeros(1), d.zeros(d.N, 3)
    Q, F = d.zeros(int(np.prod(fft))), d.zeros(int(np.prod(fft)))
    pm.reciprocal_force(d.crd, d.charge, frc, virial=vir, potential=pot)
    # the charge grid of this evaluation (the next one's differs in the order of
    # the bins' sums)
    pm.grids(Q, None)
    pm.reciprocal_force(d.crd, d.charge, plain)
    pm.grids(None, F)
    torch.cuda.synchronize()
    assert rel_rms(F.cpu().numpy(), grids["FBCFQ"]) < 1e-5
    assert rel_rms(frc.cpu().numpy(), ref["frc"]) < 1e-5
    assert rel_rms(plain.cpu().numpy(), ref["frc"]) < 1e-5
    energy = spectrum_energy(Q.cpu().numpy().reshape(fft), s, beta)
    check_total("reciprocal", pm.step_print()["reciprocal"], energy, energy)


@pytest.mark.parametrize("fft", GRIDS, ids=["x".join(map(str, g)) for g in GRIDS])
def test_virial(dev, fft):
    import torch
    from oracle import oracle as O
    from sponge_amd import abi
    from sponge_amd import system as S
    s = S.config(1)
    d = DevSystem(s, dev)
    pm = abi.ParticleMesh(d.N, abi.Box(s.box), s.cutoff, fftx=fft[0], ffty=fft[1], fftz=fft[2])
    frc, vir, Q = d.zeros(d.N, 3), d.zeros(6), d.zeros(int(np.prod(fft)))
    pm.reciprocal_force(d.crd, d.charge, frc, virial=vir)
    pm.grids(Q, None)
    torch.cuda.synchronize()
    want, size = spectrum_virial(Q.cpu().numpy().reshape(fft), s, O.get_beta(s.cutoff, s.tolerance))
    e = np.abs(vir.cpu().numpy() - want) / size
    print(f"case: fft {fft}: virial {want}, error of its terms {e.max():.2e}", flush=True)
    assert e.max() < 1e-6


@pytest.mark.parametrize("grids", [((28, 30, 32), (125, 28, 30)), ((28, 30, 32), (36, 25, 27))],
                         ids=["mixed", "planes"])
def test_batch(dev, grids):
    from sponge_amd import abi
    from sponge_amd import system as S
    boxes = [dataclasses.replace(S.water_box(n, seed=n), fft=g) for n, g in zip((600, 700), grids)]
    print(f"case: batch {grids}", flush=True)
    singles = [abi.MDSystem(s) for s in boxes]
    batched = [abi.MDSystem(s) for s in boxes]
    b = abi.Batch(batched)
    for m in singles:
        m.run(1)
    b.run(1)
    b.synchronize()
    for m1, m2 in zip(singles, batched):
        assert rel_rms(m2.state()[2], m1.state()[2]) < 1e-5
    for m in singles:
        m.run(9, use_graph=True)
    b.run(9, steps_per_launch=8)
    b.synchronize()
    for m1, m2 in zip(singles, batched):
        assert np.abs(m1.state()[0].astype(np.float64) - m2.state()[0]).max() < 1e-3
    b.clear()
