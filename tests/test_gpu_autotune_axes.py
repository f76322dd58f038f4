"""The tuner of the FFT passes times the tilings that reach a kernel: on a grid
whose planes are transformed in LDS the y and x tilings keep their values
(values that are no candidate of the tuner), of a module as of a batch; on one
that takes the three passes every axis is a candidate's or the former one."""
import ctypes as C
import dataclasses

import pytest

from gpu_helpers import DevSystem

pytestmark = pytest.mark.gpu

TILES = (4, 6, 10)


@pytest.mark.parametrize("fft, plane", [((28, 30, 32), True), ((125, 28, 30), False)])
def test_module(dev, fft, plane):
    from sponge_amd import abi
    from sponge_amd import system as S
    print(f"case: grid {fft}", flush=True)
    s = S.config(1)
    d = DevSystem(s, dev)
    pm = abi.ParticleMesh(d.N, abi.Box(s.box), s.cutoff, fftx=fft[0], ffty=fft[1], fftz=fft[2])
    for _ in range(3):
        assert pm.lib.sponge_pme_set_fft_tiling(pm.h, (C.c_int * 3)(*TILES)) == 0
        t = (C.c_int * 3)()
        assert pm.lib.sponge_pme_autotune(pm.h, d.crd.data_ptr(), d.charge.data_ptr(), 3, t) == 0
        if plane:
            assert tuple(t)[1:] == TILES[1:]
        for a in range(3):
            assert t[a] in (2, 4, 8, 16, TILES[a])


def test_batch(dev):
    from sponge_amd import abi
    from sponge_amd import system as S
    print("case: batch of plane grids", flush=True)
    boxes = [dataclasses.replace(S.water_box(n, seed=n), fft=g)
             for n, g in ((600, (28, 30, 32)), (700, (36, 25, 27)))]
    md = [abi.MDSystem(s) for s in boxes]
    for m in md:
        pme = m.handles()[2]
        assert m.lib.sponge_pme_set_fft_tiling(pme, (C.c_int * 3)(*TILES)) == 0
    b = abi.Batch(md)
    b.run(1)
    for t in b.autotune(2):
        assert t[1:] == TILES[1:]
    b.clear()
