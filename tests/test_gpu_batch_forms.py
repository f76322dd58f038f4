"""The form of the x and y transforms that a batch takes ends with it: a system
whose planes fit in LDS runs the three passes beside one whose planes do not,
and its plane transform again in steps of its own, on the same trajectory."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def launches(abi, m, steps):
    """Launches of the plane transform and of the y pass over steps of m."""
    abi.set_kernel_timing(True)
    try:
        abi.reset_kernel_timing()
        m.run(steps)
        return abi.kernel_timing("pme_fft_plane")[1], abi.kernel_timing("pme_fft_y")[1]
    finally:
        abi.set_kernel_timing(False)


def test_single_steps_after_a_mixed_batch(dev):
    from sponge_amd import abi
    from sponge_amd import system as S
    print("case: plane grid beside a grid of three passes", flush=True)
    boxes = [dataclasses.replace(S.water_box(n, seed=n), fft=g)
             for n, g in ((600, (28, 30, 32)), (700, (125, 28, 30)))]
    small, large = (abi.MDSystem(s) for s in boxes)
    single = abi.MDSystem(boxes[0])
    b = abi.Batch([small, large])
    b.run(4, steps_per_launch=3)
    b.synchronize()
    assert launches(abi, small, 2) == (2, 0)
    assert launches(abi, large, 2) == (0, 2)
    b.run(3, steps_per_launch=3)
    b.clear()
    assert launches(abi, small, 1) == (1, 0)
    single.run(10)
    x, y = small.state()[0], single.state()[0]
    assert np.abs(x.astype(np.float64) - y).max() < 1e-3
