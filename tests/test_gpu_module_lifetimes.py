"""Soft-core and learned modules outlive the step driver whose stream they
worked on: their later calls and their release use a live stream."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_soft_core_after_the_driver(dev):
    from sponge_amd import abi
    from sponge_amd import system as S
    print("case: soft-core module cleared after its driver", flush=True)
    s = S.water_box(600, cutoff=8.0, seed=3)
    m = abi.MDSystem(s)
    sc = abi.LJSoftCore(s.n_atoms, s.lj_A, s.lj_B, s.lj_A, s.lj_B, s.lj_type, s.lj_type, s.cutoff,
                        **{"lambda": 0.5})
    m.set_soft_core(sc)
    m.run(2, energy_interval=1)
    short = m.energies()["LJ_short"]
    m.clear()
    assert sc.step_print() == pytest.approx(short, rel=1e-6)
    sc.clear()


def test_learned_form_after_the_driver(dev):
    from sponge_amd import abi
    from sponge_amd import system as S
    print("case: learned module trained and cleared after its driver", flush=True)
    s = S.water_box(600, cutoff=8.0, seed=3)
    m = abi.MDSystem(s)
    beta = float(abi.load().sponge_amd_get_beta(s.cutoff, s.tolerance))
    rs = abi.ReciprocalSurrogate(s.n_atoms, beta, feature_cutoff=s.cutoff, max_frames=2)
    m.collect_frames(rs, 2, 1)
    m.clear()
    rs.fit_normalization(2)
    loss, grad = rs.gradient(0)
    assert np.isfinite(loss) and np.isfinite(grad).all()
    rs.clear()
