"""The per step lookups of an engine compiled for one energy loss scheme, on
the row tables as the library packs them, against the general engine's on the
columns, on the host: the same bits in the grid, below and above it, and at
values that are not finite."""
import ctypes

import numpy as np
import pytest

import pumas_amd as pa
import restatement
from test_host_engine import build_host

LOOKUPS = ("grammage", "energy_loss", "straggling", "del_cross_section",
           "ehs_length", "msc_mu0", "msc_inverse_path", "kinetic_energy",
           "event_energy_loss")


@pytest.fixture(scope="module")
def host():
    lib = build_host()
    vp, i = ctypes.c_void_p, ctypes.c_int
    lib.host_lookups.argtypes = [i, i, i, i, vp, vp, vp, ctypes.c_int64]
    return lib


def arguments(grid, rng):
    inner = np.concatenate([
        grid, np.nextafter(grid, -np.inf), np.nextafter(grid, np.inf),
        0.5 * (grid[1:] + grid[:-1]),
        rng.choice(grid[1:], 2000) * rng.uniform(0.5, 2.0, 2000)])
    return np.concatenate([inner, grid[-1] * np.array([1.5, 10.0, 1e3]),
                           [-1.0, -1e-300, 0.0, 5e-324, 1e300, np.inf,
                            -np.inf, np.nan]])


@pytest.mark.parametrize("physics", ["standard_c005", "iron_c001"])
@pytest.mark.parametrize("scheme", [pa.Mode.CSDA, pa.Mode.MIXED,
                                    pa.Mode.STRAGGLED])
@pytest.mark.parametrize("which", range(len(LOOKUPS)), ids=LOOKUPS)
def test_lean_lookups_equal_general(host, physics, scheme, which):
    path = pa.physics_path(physics)
    assert host.host_load(path.encode()) == 0
    t = restatement.Tables(path)
    n, nm = t.n_energies, t.n_materials
    rng = np.random.default_rng(4)
    for material in range(nm):
        table = (min(int(scheme), 1) * nm + material) * n
        grid = t.sections["X"][table:table + n] if which == 7 else t.K
        x = arguments(np.asarray(grid), rng)
        guess = rng.integers(0, n - 1, len(x)).astype(np.int32)
        out = []
        for lean in (0, 1):
            y = np.full(len(x), -7.0)
            assert host.host_lookups(lean, which, int(scheme), material,
                                     x.ctypes.data, guess.ctypes.data,
                                     y.ctypes.data, len(x)) == 0
            out.append(y)
        a, b = out
        same = (a.view(np.uint64) == b.view(np.uint64)) | \
            (np.isnan(a) & np.isnan(b))
        assert same.all(), (x[~same][:5], a[~same][:5], b[~same][:5])
