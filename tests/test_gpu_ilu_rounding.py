"""Rounding of an ILU(0) application on the device: no larger than that of the
plain triangular solves in the same precision, on the same factors."""
import numpy as np
import pytest

import sysu_cfd_parallel_amd as s
from helpers import params, push, random_state

pytestmark = pytest.mark.gpu

CASES = {
    "hex": lambda: s.channel(16, 10, 10, jitter=0.1, seed=2, re=400.0),
    "tets": lambda: s.cavity(7, tets=True, jitter=0.1, seed=3),
    "split": lambda: s.channel(14, 9, 9, jitter=0.12, split=0.25, seed=6, re=400.0),
}


def ilu0(ptr, col, diag, a):
    """The IKJ elimination on the pattern, in the type of a."""
    lu = a.copy()
    at = [{int(col[k]): k for k in range(ptr[i], ptr[i + 1])} for i in range(len(ptr) - 1)]
    for i in range(len(ptr) - 1):
        for k in range(ptr[i], diag[i]):
            j = col[k]
            lu[k] = lu[k] / lu[diag[j]]
            for q in range(diag[j] + 1, ptr[j + 1]):
                t = at[i].get(int(col[q]))
                if t is not None:
                    lu[t] = lu[t] - lu[k] * lu[q]
    return lu


def apply(ptr, col, diag, lu, r):
    """Both triangular solves row by row, in the type of r (every product and
    sum rounded to it)."""
    n, z = len(r), r.copy()
    for i in range(n):
        for k in range(ptr[i], diag[i]):
            z[i] = z[i] - lu[k] * z[col[k]]
    for i in range(n - 1, -1, -1):
        for k in range(diag[i] + 1, ptr[i + 1]):
            z[i] = z[i] - lu[k] * z[col[k]]
        z[i] = z[i] / lu[diag[i]]
    return z


@pytest.mark.parametrize("precision", [s.FP64, s.MIXED])
@pytest.mark.parametrize("name", sorted(CASES))
def test_rounding_is_that_of_plain_solves_at_most(name, precision):
    kind = np.float32 if precision == s.MIXED else np.float64
    p = params(restart=30, pc=s.PC_ILU0)
    p.precision = precision
    d = s.Solver(CASES[name](), p)
    st = random_state(d.sizes.n_cell, d.sizes.n_bnd, d.sizes.n_face, 7)
    push(d, {k: st[k] for k in ("U", "V", "W", "P", "R", "APR", "DPDX", "RUFACE")})
    d.call("build_velocity_matrix")
    push(d, {k: np.zeros(d.sizes.n_cell) for k in "UVW"})
    rng = np.random.default_rng(11)
    push(d, {"B%s_RHS" % k: rng.standard_normal(d.sizes.n_cell) for k in "UVW"})
    # one GMRES step from a zero guess: each solution is a multiple of (LU)^-1 b;
    # a later component is solved only where the earlier ones have ended, so the
    # cap is for the first one
    try:
        d.solve_velocity(1e-30, 1)
    except s.NotConverged:
        pass
    ptr, col, diag = d.ints("CSR_ROWPTR"), d.ints("CSR_COL"), d.ints("CSR_DIAG")
    b = d.get("BU_RHS").astype(kind)
    lu = ilu0(ptr, col, diag, d.get("AU").astype(kind))
    plain = apply(ptr, col, diag, lu, b).astype(np.float64)
    wide = np.longdouble if kind is np.float64 else np.float64
    exact = apply(ptr, col, diag, lu.astype(wide), b.astype(wide))

    def error(x):
        """x against the multiple of the exact vector nearest to it, in the 2-norm"""
        x = x.astype(wide)
        c = (x @ exact) / (exact @ exact)
        return float(np.sqrt(((x - c * exact) ** 2).sum() / (x ** 2).sum())), float(c)

    got, c = error(d.get("U"))
    # the plain solve's vector times the same number, rounded as the update rounds it
    want, _ = error(plain * c)
    print(name, kind.__name__, got, want)
    assert 0 < got <= want
    d.close()
