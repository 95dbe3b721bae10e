"""The sweep shape of meshes that step in one launch: setting what was read keeps that
step, any other shape takes the launches, and the autotuner's rows hold every candidate."""
import ctypes

import numpy as np
import pytest

from physicsbasedanimationtoolkit_amd import _native, pbat

from test_gpu_local import DT, build, grid, loose

pytestmark = pytest.mark.gpu


def launches(g):
    g.set_timing(True)
    g.sweep_timing(reset=True)
    g.step(DT, 3, 2)
    return g.sweep_timing(reset=True)[1]


def configure(g, c):
    g.set_sweep_config(c["lanes_per_vertex"], c["incidences_per_lane"], c["xcd_remap"], c["nontemporal"],
                       c["fixed_stride"])


@pytest.mark.parametrize("mesh", [loose(3), loose(70), grid(4, 3, 5), grid(8, 9, 7)],
                         ids=["tets", "tets70", "grid", "grid8"])
def test_setting_what_was_read(gpu_device, mesh):
    d = build(*mesh)[0]
    g, ref = pbat.gpu.vbd.Integrator(d), pbat.gpu.vbd.Integrator(d)
    c = g.sweep_config()
    configure(g, c)
    assert g.sweep_config() == c
    assert launches(g) == launches(ref) == 1
    assert np.array_equal(g.x, ref.x)
    g.set_sweep_config(16, 2)
    read = g.sweep_config()
    configure(g, read)
    assert g.sweep_config() == read
    assert launches(g) == 3 * 2 * g.counts()[0]
    configure(g, c)  # an explicit shape, now that the automatic one is gone
    assert launches(g) == 3 * 2 * g.counts()[0]
    g.set_sweep_config()
    assert launches(g) == 1


@pytest.mark.parametrize("mesh,one_launch,candidates",
                         [(grid(4, 3, 5), True, 17), (grid(9, 9, 9), True, 32), (grid(12, 11, 13), False, 32)],
                         ids=["grid", "grid9", "launches"])
def test_autotune_rows(gpu_device, mesh, one_launch, candidates):
    """Degree 24 has 32 launch shapes, 16 without fixed-stride rows; every candidate has a row."""
    g = pbat.gpu.vbd.Integrator(build(*mesh)[0])
    rows, n = np.zeros(192), ctypes.c_int32()
    _native.check(g._lib.pbat_vbd_integrator_autotune(g._h, DT, 2, _native.ptr(rows, ctypes.c_double),
                                                      ctypes.byref(n)))
    assert n.value == candidates
    rows = rows.reshape(-1, 6)[:n.value]
    assert (rows[:, 5] > 0).all()
    assert [r[0] == 0 for r in rows] == [one_launch] + (candidates - 1) * [False]
