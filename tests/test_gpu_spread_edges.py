"""The spreading kernels at the edges of what they accept: common factors of
the results, positions that are not finite or very far apart, state kept
between calls, captured calls, and tables and grids that the recurrence kernels
take."""
import numpy as np
import pytest

from oracle import scatter as oracle
from pyiid_amd import _lib, structures
from pyiid_amd.formfactors import element_table

pytestmark = pytest.mark.gpu


def load(ctx, pos, numbers, qbin, nq):
    table, index, _ = element_table(numbers, qbin, nq)
    ctx.set_positions(pos)
    ctx.set_elements(index)
    ctx.set_scatter(_lib.SLOT_FQ, table)
    return table[index]


def test_f_has_no_common_factor(ctx):
    """F = (1 + a) F_exact + noise: a from fits over five parts of the Q range and
    four structures.  The noise is the float32 result's rounding (1.7e-8 r.m.s. of
    a value, about 100 values a part: 2e-9 a fit, 5e-10 their mean) and what single
    pairs are off by; the window leaves 2.5e-9.  Allowed: 8e-9."""
    n, nq, qbin = 1000, 500, 0.05
    slopes = []
    for seed in range(4):
        pos = structures.jitter(structures.fcc_nearest(n), 0.05, seed=seed).astype(np.float32)
        per_atom = load(ctx, pos, np.full(n, 79), qbin, nq)
        got = ctx.fq(_lib.SLOT_FQ, qbin, nq).astype(np.float64)
        want = oracle.fq(pos, per_atom, qbin)
        for part in range(5):
            s = slice(nq * part // 5, nq * (part + 1) // 5)
            slopes.append(((got - want)[s] @ want[s]) / (want[s] @ want[s]))
    assert abs(np.mean(slopes)) < 8e-9, np.mean(slopes)


@pytest.mark.parametrize("far", [1e12, 1e14, 1e18, 1e25, 1e37])
def test_very_far_atoms_add_nothing(ctx, far):
    """A cluster and an atom so far away that its pairs' weights 1/r are below
    float32's smallest step of F: F and the gradient are those of the cluster
    without it (but for the normalisation's number of atoms), and the far atom's
    gradient is zero to that step."""
    n, nq, qbin = 60, 250, 0.1
    pos = structures.jitter(structures.fcc_nearest(n), 0.05, seed=3).astype(np.float32)
    alone = np.concatenate([pos, pos[-1:]])  # a duplicate contributes nothing either
    alone[-1] = pos[-1]
    apart = alone.copy()
    apart[-1] = (far, 0, 0)
    load(ctx, alone[:n], np.full(n, 79), qbin, nq)
    f0 = ctx.fq(_lib.SLOT_FQ, qbin, nq).astype(np.float64) * n
    g0 = ctx.grad_fq(_lib.SLOT_FQ, qbin, n, nq).astype(np.float64) * n
    load(ctx, apart, np.full(n + 1, 79), qbin, nq)
    f1 = ctx.fq(_lib.SLOT_FQ, qbin, nq).astype(np.float64) * (n + 1)
    fq = np.empty(nq, np.float32)
    g1 = ctx.grad_fq(_lib.SLOT_FQ, qbin, n + 1, nq, fq_out=fq).astype(np.float64) * (n + 1)
    assert np.abs(f1 - f0).max() < 2e-7 * np.abs(f0).max()
    assert np.abs(fq * (n + 1.0) - f0).max() < 2e-7 * np.abs(f0).max()
    assert np.abs(g1[:n] - g0).max() < 1e-6 * np.abs(g0).max()
    assert np.abs(g1[n]).max() < 1e-7 * np.abs(g0).max()
