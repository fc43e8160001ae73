"""Row tables of the lean stepping kernels against the per column lookups, on
the host: the same row and the same bits, from any first guess, at every grid
value and its neighbours, between them, and outside of the grid."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import pumas_amd as pa
import restatement

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "pumas_amd", "csrc")
COLUMNS = ("X", "X_dK", "K_dX", "dE", "dE_dK", "Omega", "Omega_dK", "CS",
           "CS_dK", "Mu0", "Mu0_dK", "Ms1", "Ms1_dK", "Lb", "K")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("rows") / "librows.so")
    subprocess.check_call(
        ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off",
         "-mfma", "-I", CSRC, "-o", path, os.path.join(HERE, "rows_check.cpp")])
    lib = ctypes.CDLL(path)
    p, i = ctypes.c_void_p, ctypes.c_int
    lib.rows_check.argtypes = [p, i, i, p, p, p, p, p, ctypes.c_long]
    lib.rows_check.restype = ctypes.c_long
    return lib


def column(t, name, scheme, material):
    if name == "K":
        return t.K
    if name in ("Omega", "Omega_dK", "CS", "CS_dK", "Mu0", "Mu0_dK", "Lb"):
        return t.col1(name, material)
    table = (scheme + (1 if name.startswith("Ms1") else 0)) * t.n_materials
    n = t.n_energies
    return t.sections[name][(table + material) * n:(table + material + 1) * n]


def arguments(grid, rng):
    inner = np.concatenate([grid, np.nextafter(grid, -np.inf),
                            np.nextafter(grid, np.inf),
                            0.5 * (grid[1:] + grid[:-1]),
                            rng.choice(grid[1:], 20000) *
                            rng.uniform(0.5, 2.0, 20000)])
    return np.concatenate([inner, [-1.0, 0.0, np.inf, 2 * grid[-1]]])


@pytest.mark.parametrize("physics", ["standard_c005", "iron_c001"])
def test_row_tables_equal_columns(lib, physics):
    t = restatement.Tables(pa.physics_path(physics))
    rng = np.random.default_rng(3)
    n = t.n_energies
    for scheme in (0, 1):
        for material in range(t.n_materials):
            c = {name: np.ascontiguousarray(column(t, name, scheme, material))
                 for name in COLUMNS}
            rows = np.ascontiguousarray(np.stack(
                [c[name] for name in COLUMNS], axis=1))

            def bad(index, grid, y, m):
                x = arguments(grid, rng)
                near = np.clip(np.searchsorted(grid, x) - 1 +
                               rng.integers(-2, 3, len(x)), 0, n - 2)
                far = rng.integers(0, n - 1, len(x))
                guess = np.where(rng.random(len(x)) < 0.8, near,
                                 far).astype(np.int32)
                return lib.rows_check(
                    rows.ctypes.data, n, index, grid.ctypes.data,
                    y.ctypes.data, m.ctypes.data, x.ctypes.data,
                    guess.ctypes.data, len(x))

            for y, m in (("X", "X_dK"), ("dE", "dE_dK"), ("Omega", "Omega_dK"),
                         ("CS", "CS_dK"), ("Mu0", "Mu0_dK"),
                         ("Ms1", "Ms1_dK")):
                assert bad(COLUMNS.index(y), c["K"], c[y], c[m]) == 0, y
            assert bad(-1, c["X"], c["K"], c["K_dX"]) == 0
