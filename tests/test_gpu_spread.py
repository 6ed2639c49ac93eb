"""The spreading kernels (F(Q) from pair distances put onto a fine grid)
against the FP64 oracle where they can go wrong: tile and bin remainders,
distances folded at the grid's period, close contacts, duplicated atoms,
several elements, batches.

Tolerance, derived from the kernel's arithmetic: a pair's term sin(Qr)/r is
off by at most 6.6e-8 / r (window 2.3e-8 and its single-precision values), so
F by 6.6e-8 of the sum of its pair weights 1/r, plus the rounding of the
float32 result; twice that is allowed."""
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


def bound(pos, per_atom, want):
    """Twice the error the arithmetic allows, per bin."""
    p = pos.astype(np.float64)
    i, j = np.tril_indices(len(pos), -1)
    r = np.linalg.norm(p[i] - p[j], axis=1)
    inv = np.divide(1.0, r, out=np.zeros_like(r), where=r > 0)
    f = per_atom.astype(np.float64)
    w = np.einsum("k,kq,kq->q", inv, np.abs(f[i]), np.abs(f[j]))
    na = np.abs(oracle.normalization(per_atom))
    return 2 * (6.6e-8 * 2 * w / na + 6e-8 * np.abs(want)) + 1e-30


def debye(pos, per_atom, qbin):
    """The oracle's F(Q); with duplicated atoms (for which the oracle zeroes
    every bin, as the reference's NaN does) the FP64 sum over the other pairs."""
    i, j = np.tril_indices(len(pos), -1)
    p, f = pos.astype(np.float64), per_atom.astype(np.float64)
    r = np.linalg.norm(p[i] - p[j], axis=1)
    if np.all(r > 0):
        return oracle.fq(pos, per_atom, qbin)
    i, j, r = i[r > 0], j[r > 0], r[r > 0]
    q = oracle.q_values(qbin, per_atom.shape[1])
    return 2.0 / oracle.normalization(per_atom) * np.sum(
        f[i] * f[j] * np.sin(np.outer(r, q)) / r[:, None], axis=0)


def check(ctx, pos, numbers, qbin, nq):
    per_atom = load(ctx, pos, numbers, qbin, nq)
    got = ctx.fq(_lib.SLOT_FQ, qbin, nq)
    want = debye(pos, per_atom, qbin)
    off = np.abs(got - want) / bound(pos, per_atom, want)
    assert np.all(np.isfinite(got)) and off.max() < 1.0, (off.argmax(), off.max())


@pytest.mark.parametrize("n", [2, 3, 63, 64, 65, 129, 300])
@pytest.mark.parametrize("nq", [1, 2, 7, 32, 65, 330])
def test_tiles_and_bins(ctx, n, nq):
    pos = structures.jitter(structures.fcc_nearest(n), 0.05, seed=n).astype(np.float32)
    check(ctx, pos, np.full(n, 79), 25.0 / nq, nq)


def test_largest_grid(ctx):
    pos = structures.jitter(structures.fcc_nearest(40), 0.05, seed=1).astype(np.float32)
    for nq in (3400, 3420):  # the last with a grid in LDS, and past it (recurrence kernel)
        check(ctx, pos, np.full(len(pos), 79), 0.008, nq)


@pytest.mark.parametrize("length", [30.0, 314.0, 4e3, 3e5])
def test_distances_beyond_the_period(ctx, length):
    """Periods of the 0.1 bins: 62.8 A; the distances span many of them, and
    one is an exact multiple."""
    rs = np.random.RandomState(3)
    pos = rs.uniform(-length, length, (90, 3)).astype(np.float32)
    pos[0], pos[1] = 0.0, (np.float32(4 * np.pi / np.float32(0.1)), 0, 0)
    check(ctx, pos, np.full(90, 79), 0.1, 250)


@pytest.mark.parametrize("r", [1e-6, 1e-3, 0.02, 0.0418, 0.042, 0.2, 0.355, 0.36, 1.0])
def test_close_contacts(ctx, r):
    """A pair at each of the kernel's short ranges (grid spacing 0.0209 A:
    interpolation below 2, 64-bit conversion below 17 of them), beside a
    duplicated atom, which contributes nothing."""
    pos = structures.jitter(structures.fcc_nearest(50), 0.05, seed=5).astype(np.float32)
    pos[7] = 0.0
    pos[20] = (r, 0, 0)
    pos[31] = pos[30]
    check(ctx, pos, np.full(50, 79), 0.1, 250)


def test_elements_and_batch(ctx):
    """Three elements in one particle, and a batch whose chains hold one
    atom, one element, and all three; a second call sees cleared grids."""
    rs = np.random.RandomState(8)
    zs = np.array([28, 78, 79])
    pos = structures.jitter(structures.fcc_nearest(210), 0.05, seed=9).astype(np.float32)
    check(ctx, pos, zs[rs.randint(0, 3, 210)], 0.05, 500)
    qbin, nq = 0.0756865, 330
    numbers = [np.array([79]), np.full(70, 28), zs[rs.randint(0, 3, 131)], np.array([78, 79])]
    chains = [structures.jitter(structures.fcc_nearest(len(z)), 0.05, seed=len(z)).astype(np.float32)
              for z in numbers]
    table, index, elems = element_table(np.concatenate(numbers), qbin, nq)
    ctx.set_batch(chains)
    ctx.set_elements(index)
    ctx.set_scatter(_lib.SLOT_FQ, table)
    first = ctx.fq(_lib.SLOT_FQ, qbin, nq, n_chain=4)
    again = ctx.fq(_lib.SLOT_FQ, qbin, nq, n_chain=4)
    np.testing.assert_array_equal(first, again)
    assert not np.any(first[0])
    for b in (1, 2, 3):
        per_atom = table[np.searchsorted(elems, numbers[b])]
        want = oracle.fq(chains[b], per_atom, qbin)
        assert np.all(np.abs(first[b] - want) < bound(chains[b], per_atom, want))


def test_infinite_position_is_not_a_number(ctx):
    pos = structures.fcc_nearest(20).astype(np.float32)
    pos[3, 0] = np.inf
    load(ctx, pos, np.full(20, 79), 0.1, 100)
    assert np.all(np.isnan(ctx.fq(_lib.SLOT_FQ, 0.1, 100)[1:]))


def force_check(ctx, pos, base, numbers, qbin, nq, upload=None):
    """F(Q)-Rw energy and forces against the oracle.  Allowed: 4e-7 of the sum
    of the amplitudes of an atom's pair forces (table polynomial 4.2e-8, its
    single-precision coefficients and evaluation about 3e-7), and 2e-6 of the
    largest force for the error of F in the residual."""
    n, first = len(pos), 5
    per_atom = load(ctx, base if upload else pos, numbers, qbin, nq)
    target = oracle.fq((pos * np.float32(0.98)).astype(np.float32), per_atom, qbin)[first:]
    if upload:
        ctx.fq_energy_forces(_lib.SLOT_FQ, qbin, first, target, _lib.POT_RW, 10.0, n)
        upload(pos)
    e, f = ctx.fq_energy_forces(_lib.SLOT_FQ, qbin, first, target, _lib.POT_RW, 10.0, n)
    fq = oracle.fq(pos, per_atom, qbin)[first:]
    g = oracle.grad_fq(pos, per_atom, qbin)[:, :, first:]
    want = 10.0 * oracle.wrap_grad_rw(g, fq, target)
    rw, a = oracle.get_rw(target, fq)
    w = 10.0 * np.abs(rw / np.sum((target - a * fq) ** 2) * a * (target - a * fq))
    q = oracle.q_values(qbin, nq)[first:]
    x, ff = pos.astype(np.float64), per_atom.astype(np.float64)[:, first:]
    r = np.linalg.norm(x[:, None] - x[None], axis=-1)
    inv = np.divide(1.0, r, out=np.zeros_like(r), where=r > 0)
    na = np.abs(oracle.normalization(per_atom))[first:]
    amp = np.einsum("q,iq,jq,ij->i", w * q / na, ff, ff, inv) + \
        np.einsum("q,iq,jq,ij->i", w / na, ff, ff, inv * inv)
    allowed = 4e-7 * amp[:, None] + 2e-6 * np.abs(want).max()
    assert abs(e - 10.0 * rw) < 1e-5
    off = (np.abs(f - want) / allowed).max()
    assert off < 1.0, off


@pytest.mark.parametrize("n", [2, 3, 64, 65, 150, 400])
def test_force_table_tiles(ctx, n):
    base = structures.fcc_nearest(n)
    pos = structures.jitter(base, 0.05, seed=n).astype(np.float32)
    force_check(ctx, pos, base, np.full(n, 79), 0.1, 250)
    zs = np.random.RandomState(n).permutation(np.array([28, 78, 79])[np.arange(n) % 3])
    force_check(ctx, pos, base, zs, 0.05, 330)


def test_force_past_the_table(ctx):
    """Positions moved on the device after the table's length was taken: the
    pairs past its end are summed directly, and the next call has a longer
    table."""
    import torch
    base = structures.fcc_nearest(90).astype(np.float32)
    pos = structures.jitter(base, 0.05, seed=2).astype(np.float32)
    pos[40:] += np.float32(17.3)

    def upload(p):
        ctx.set_positions(torch.from_numpy(p).cuda(), flags=_lib.PYIID_DEVICE)
    for _ in range(2):
        force_check(ctx, pos, base, np.full(90, 79), 0.1, 250, upload)


def test_long_force_table(ctx):
    """A structure whose table fills most of LDS, and one past it (which runs
    the recurrence kernel)."""
    for length in (140.0, 400.0):
        pos = np.random.RandomState(4).uniform(0, length, (70, 3)).astype(np.float32)
        force_check(ctx, pos, pos, np.full(70, 79), 0.05, 600)


def grad_check(ctx, pos, numbers, qbin, nq, f64=False, per_atom=None):
    """The gradient against the oracle.  Allowed per entry: the window's worst
    errors (3.2e-7 of the largest Q for the cosine term, 3.5e-7 for the sine
    term, single-precision values included) for every pair, and 2^-20 of the
    largest entry for the two-half products."""
    if per_atom is None:
        per_atom = load(ctx, pos, numbers, qbin, nq)
    got = ctx.grad_fq(_lib.SLOT_FQ, qbin, len(pos), nq, f64=f64)
    assert ctx.grad_shape() == (False, 0, 0)
    want = oracle.grad_fq(pos, per_atom, qbin)
    x, f = pos.astype(np.float64), np.abs(per_atom.astype(np.float64))
    r = np.linalg.norm(x[:, None] - x[None], axis=-1)
    inv = np.divide(1.0, r, out=np.zeros_like(r), where=r > 0)
    na = np.abs(oracle.normalization(per_atom))
    pair = 3.2e-7 * qbin * nq * inv + 3.5e-7 * inv * inv
    allowed = np.einsum("iq,jq,ij->iq", f, f, pair) / na + 2.0 ** -20 * np.abs(want).max() + 1e-30
    assert np.all(np.isfinite(got))
    off = (np.abs(got - want) / allowed[:, None, :]).max()
    assert off < 1.0, off


@pytest.mark.parametrize("n", [2, 3, 42, 43, 65, 300])
@pytest.mark.parametrize("nq", [1, 2, 31, 127, 128, 129, 330])
def test_gradient_tiles(ctx, n, nq):
    pos = structures.jitter(structures.fcc_nearest(n), 0.05, seed=n).astype(np.float32)
    numbers = np.full(n, 79) if nq != 129 else np.array([28, 78, 79])[np.arange(n) % 3]
    grad_check(ctx, pos, numbers, 25.0 / nq, nq, f64=nq % 2 == 1)


def test_gradient_largest_grid(ctx):
    pos = structures.jitter(structures.fcc_nearest(25), 0.05, seed=1).astype(np.float32)
    grad_check(ctx, pos, np.full(25, 79), 0.009, 3010)


@pytest.mark.parametrize("r", [1e-3, 0.02, 0.1116, 0.1118, 0.5, 1.07, 1.08])
def test_gradient_close_contacts(ctx, r):
    """A pair at the kernel's short ranges (grid spacing 0.0558 A)."""
    pos = structures.jitter(structures.fcc_nearest(50), 0.05, seed=5).astype(np.float32)
    pos[7], pos[20] = 0.0, (r, 0, 0)
    grad_check(ctx, pos, np.full(50, 79), 0.1, 250)


@pytest.mark.parametrize("length", [30.0, 314.0, 4e3])
def test_gradient_beyond_the_period(ctx, length):
    rs = np.random.RandomState(3)
    pos = rs.uniform(-length, length, (90, 3)).astype(np.float32)
    pos[0], pos[1] = 0.0, (np.float32(4 * np.pi / np.float32(0.1)), 0, 0)
    grad_check(ctx, pos, np.full(90, 79), 0.1, 250)


def test_gradient_of_positions_moved_on_the_device(ctx):
    """The reach of the grid comes from the device after an upload there: a
    larger structure of the same size, then a smaller one, equal to host mode."""
    import torch
    base = structures.jitter(structures.fcc_nearest(150), 0.05, seed=6).astype(np.float32)
    per_atom = load(ctx, base, np.full(150, 79), 0.05, 400)
    for scale in (1.0, 2.5, 0.8):
        pos = (base * np.float32(scale)).astype(np.float32)
        ctx.set_positions(torch.from_numpy(pos).cuda(), flags=_lib.PYIID_DEVICE)
        got = ctx.grad_fq(_lib.SLOT_FQ, 0.05, 150, 400)
        grad_check(ctx, pos, None, 0.05, 400, per_atom=per_atom)
        ctx.set_positions(pos)
        np.testing.assert_array_equal(got, ctx.grad_fq(_lib.SLOT_FQ, 0.05, 150, 400))


@pytest.mark.parametrize("n,nq", [(193, 512), (300, 100), (505, 164), (2048, 65), (2049, 65)])
def test_gradient_with_f_in_its_launches(ctx, n, nq):
    """F that rides along with a gradient equals F asked for alone, again on a
    second call (its grids are cleared by the gradient's last launch), and both
    match the oracle."""
    pos = structures.jitter(structures.fcc_nearest(n), 0.05, seed=n).astype(np.float32)
    per_atom = load(ctx, pos, np.full(n, 79), 0.1, nq)
    alone = ctx.fq(_lib.SLOT_FQ, 0.1, nq)
    for _ in range(2):
        fq = np.empty(nq, np.float32)
        g = ctx.grad_fq(_lib.SLOT_FQ, 0.1, n, nq, fq_out=fq)
        # one transform block per 64 bins instead of several parts: FP64 rounding
        np.testing.assert_allclose(fq, alone, rtol=3e-7, atol=1e-9)
    rows = np.arange(0, n, 37)
    want = oracle.grad_fq(pos, per_atom, 0.1, atom_index=rows)
    assert np.abs(g[rows] - want).max() < 2e-6 * np.abs(want).max()
    np.testing.assert_array_equal(ctx.fq(_lib.SLOT_FQ, 0.1, nq), alone)


@pytest.mark.parametrize("m", [60, 118, 119, 120, 400])
@pytest.mark.parametrize("cap", [np.pi, 0.35])
def test_gradient_of_a_shell(ctx, m, cap):
    """Atoms at one distance from atom 0, all around it or on one side, where
    their entries add up to more than 31 bits: 32-bit grids of up to about 118
    atoms at 10 A, 64-bit ones beyond."""
    z = 1.0 - (1.0 - np.cos(cap)) * (np.arange(m) + 0.5) / m
    phi = np.arange(m) * np.pi * (3.0 - np.sqrt(5.0))
    s = np.sqrt(1.0 - z * z)
    shell = 10.0 * np.stack([s * np.cos(phi), s * np.sin(phi), z], 1)
    pos = np.concatenate([np.zeros((1, 3)), shell]).astype(np.float32)
    grad_check(ctx, pos, np.full(m + 1, 79), 0.1, 250)


@pytest.mark.parametrize("r", [0.2675, 0.268, 0.2685])
@pytest.mark.parametrize("far", [40.0, 114.2, 114.4])
def test_gradient_choice_of_grid(ctx, r, far):
    """A pair at the least distance of the 32-bit grids, and a structure at
    their largest extent (4.8 and 2,048 spacings of 0.0558 A)."""
    pos = structures.jitter(structures.fcc_nearest(50), 0.05, seed=5).astype(np.float32)
    pos[7], pos[20], pos[30] = 0.0, (r, 0, 0), (0, 0, far)
    grad_check(ctx, pos, np.full(50, 79), 0.1, 250)


@pytest.mark.parametrize("n,nq,n_r", [(86, 128, 4000), (86, 129, 63), (100, 330, 1001), (343, 160, 2001),
                                      (700, 200, 3969), (701, 130, 4001)])
@pytest.mark.parametrize("f64", [False, True])
def test_gradient_transform_on_split_operands(ctx, n, nq, n_r, f64):
    """Tiles of 128 x 64 and (from 700 atoms here) 128 x 128 against the FP64
    product, with rows of zeros, of far magnitudes and with an infinity or a
    NaN.  Each operand is left 2^-22 of itself off by its split and by the
    product of the low halves; 2^-20 of the sum of magnitudes covers the three
    and the FP32 sums."""
    dq = 0.05
    r = 0.01 * np.arange(n_r)
    ctx.set_transform(0.01, dq, r, 0.0, nq)
    eye = np.zeros((66, 3, nq), np.float32)  # too few entries for the split
    t = np.empty((n_r, nq))
    for m0 in range(0, nq, 66):
        m1 = min(m0 + 66, nq)
        eye[:] = 0.0
        eye[np.arange(m1 - m0), 0, np.arange(m0, m1)] = 1.0
        for m in range(m0, m1, 22):
            k = min(22, m1 - m)
            t[:, m:m + k] = ctx.grad_pdf(eye[m - m0:m - m0 + k], n_r)[:, 0].T
    rs = np.random.RandomState(n + nq)
    a = rs.standard_normal((n, 3, nq)).astype(np.float32)
    a *= np.exp(rs.uniform(-8, 8, (n, 3, 1))).astype(np.float32)
    a[0, 0], a[1, 1], a[2, 2] = 0.0, a[1, 1] * np.float32(1e25), a[2, 2] * np.float32(1e-25)
    a[3, 0, 5], a[4, 1, nq - 1] = np.inf, np.nan
    got = ctx.grad_pdf(a.astype(np.float64) if f64 else a, n_r)
    x = a.astype(np.float64).reshape(-1, nq)
    ok = np.isfinite(x).all(1)
    want = x[ok] @ t.T
    allowed = 2.0 ** -20 * (np.abs(x[ok]) @ np.abs(t).T) + 2.0 ** -30 * (
        np.abs(x[ok]).max(1, keepdims=True) * np.abs(t).sum(1)) + 1e-38
    off = np.abs(got.reshape(-1, n_r)[ok] - want) / allowed
    assert off.max() < 1.0, off.max()
    with np.errstate(invalid="ignore"):
        bad = x[~ok] @ t.T
    assert np.isnan(got[4, 1]).all()
    np.testing.assert_array_equal(np.isnan(got[3, 0]), np.isnan(bad[0]))
    np.testing.assert_array_equal(np.isposinf(got[3, 0]), np.isposinf(bad[0]))


@pytest.mark.parametrize("n", [2, 55, 70, 71, 85, 86, 128, 129])
@pytest.mark.parametrize("nq", [64, 65, 270, 400, 830])
def test_one_launch_with_two_elements(ctx, n, nq):
    """F of small structures, one to three elements, up to and past the sizes that
    one launch takes (128, 85 and 70 atoms, 80 KB of grids)."""
    pos = structures.jitter(structures.fcc_nearest(n), 0.05, seed=n).astype(np.float32)
    check(ctx, pos, np.full(n, 79), 25.0 / nq, nq)
    check(ctx, pos, np.array([28, 79])[np.random.RandomState(n).randint(0, 2, n)], 25.0 / nq, nq)
    check(ctx, pos, np.array([28, 78, 79])[np.random.RandomState(n).randint(0, 3, n)], 25.0 / nq, nq)


@pytest.mark.parametrize("n_r", [15, 16, 17, 63, 1000])
@pytest.mark.parametrize("zs", [(79,), (28, 79)])
def test_energy_and_forces_of_g(ctx, n_r, zs):
    """Energy and forces against G(r) from the gradient of G(r), for one chain,
    and for each of 17 (a tile of 16 and one more).  Each entry of the gradient
    may be off by 2^-20 of the largest, which the adjoint's weights add up; the
    two numbers of tables in a launch round alike to 1e-6."""
    nq, qbin, sizes = 200, 0.1, 20 + np.arange(17)
    r = 2.0 + 0.02 * np.arange(n_r)
    chains = [structures.jitter(structures.fcc_nearest(n), 0.05, seed=n).astype(np.float32) for n in sizes]
    numbers = [np.array(zs)[np.arange(n) % len(zs)] for n in sizes]
    table, index, _ = element_table(np.concatenate(numbers), qbin, nq)
    ctx.set_transform(0.02, qbin, r, 0.0, nq)
    alone, targets, at = [], [], 0
    for pos, n in zip(chains, sizes):
        ctx.set_positions(pos)
        ctx.set_elements(index[at:at + n])
        ctx.set_scatter(_lib.SLOT_PDF, table)
        at += n
        fq = ctx.fq(_lib.SLOT_PDF, qbin, nq)
        g = ctx.pdf(fq, n_r)
        target = g * (1.0 + 0.3 * np.sin(np.arange(n_r))) + 0.1
        gg = ctx.grad_pdf(ctx.grad_fq(_lib.SLOT_PDF, qbin, n, nq), n_r)
        e, f = ctx.pdf_energy_forces(_lib.SLOT_PDF, qbin, target, _lib.POT_RW, 10.0, n)
        rw, a = oracle.get_rw(target, g)
        want = 10.0 * oracle.wrap_grad_rw(gg, g, target)
        res = target - a * g
        w = 10.0 * np.abs(rw / np.sum(res ** 2) * a * res).sum()
        assert abs(e - 10.0 * rw) < 1e-5
        assert np.abs(f - want).max() < 2.0 ** -20 * w * np.abs(gg).max() + 1e-6 * np.abs(want).max()
        alone.append((e, f))
        targets.append(target)
    ctx.set_batch(chains)
    ctx.set_elements(index)
    ctx.set_scatter(_lib.SLOT_PDF, table)
    e, f = ctx.pdf_energy_forces(_lib.SLOT_PDF, qbin, np.array(targets), _lib.POT_RW, 10.0, len(index))
    at = 0
    for b, n in enumerate(sizes):
        scale = np.abs(alone[b][1]).max()
        assert abs(e[b] - alone[b][0]) < 1e-6 * abs(alone[b][0])
        assert np.abs(f[at:at + n] - alone[b][1]).max() < 1e-6 * scale
        at += n


@pytest.mark.parametrize("kinds", [2, 3])
def test_uploads_in_element_order(ctx, kinds):
    """From the second upload of a structure on the packing puts the atoms in
    element order: F, gradient and forces equal a new context's, also after the
    elements have changed and after a sampler has moved the atoms."""
    n, nq, qbin, zs = 150, 300, 0.08, np.array([28, 78, 79])[:kinds]
    rs = np.random.RandomState(kinds)
    base = structures.fcc_nearest(n)
    target = 0.5 + 0.1 * np.cos(np.arange(400))

    def elements(c, numbers):
        table, index, _ = element_table(numbers, qbin, nq)
        c.set_elements(index)
        c.set_scatter(_lib.SLOT_FQ, table)
        c.set_scatter(_lib.SLOT_PDF, table)
        c.set_transform(0.02, qbin, 2.0 + 0.02 * np.arange(400), 0.0, nq)

    def results(c, pos):
        c.set_positions(pos)
        fq = np.empty(nq, np.float32)
        g = c.grad_fq(_lib.SLOT_FQ, qbin, n, nq, fq_out=fq)
        e, f = c.pdf_energy_forces(_lib.SLOT_PDF, qbin, target, _lib.POT_RW, 10.0, n)
        return c.fq(_lib.SLOT_FQ, qbin, nq), fq, g, np.float64(e), f

    def fresh(numbers, pos):
        c = _lib.Context(0)
        c.set_positions(pos)
        elements(c, numbers)
        out = results(c, pos)
        c.close()
        return out

    ctx.set_positions(base.astype(np.float32))
    for step in range(6):
        numbers = zs[np.random.RandomState(step // 3).permutation(np.arange(n) % kinds)]
        pos = (base + rs.normal(0, 0.05, (n, 3))).astype(np.float32)
        if step % 3 == 0:
            elements(ctx, numbers)
        for got, want in zip(results(ctx, pos), fresh(numbers, pos)):
            np.testing.assert_array_equal(got, want)
        if step == 4:
            ctx.hmc_setup(_lib.SLOT_PDF, qbin, target, _lib.POT_RW, 10.0, np.full(n, 100.0))
            ctx.hmc_run(2, 2, 0.5, 1.0, 1, 1)
            after, want = ctx.fq(_lib.SLOT_FQ, qbin, nq), fresh(numbers, ctx.get_positions(n))[0]
            # the sampler's positions are FP64, those handed out float32 (6e-7 A)
            assert np.abs(after - want).max() < 1e-4 * np.abs(want).max()
            assert np.abs(ctx.get_positions(n) - pos).max() > 1e-3


@pytest.mark.parametrize("chains", [61, 66])
@pytest.mark.parametrize("nq", [200, 201])
def test_forces_of_many_chains(ctx, chains, nq):
    """Tables made four to a block (more than 2,048 blocks of 64 cells; the last
    four are not whole) against one chain alone, whose table rounds alike to
    1e-6."""
    qbin, n, r = 25.0 / nq, 24, 2.0 + 0.02 * np.arange(200)
    base = structures.fcc_nearest(n)
    pos = [structures.jitter(base, 0.05, seed=b).astype(np.float32) for b in range(chains)]
    for p in pos:
        p[0] += np.float32(55.0)  # a wide extent: about 2,200 cells
    table, index, _ = element_table(np.full(n * chains, 79), qbin, nq)
    target = np.tile(0.5 + 0.1 * np.cos(np.arange(200)), (chains, 1))
    ctx.set_batch(pos)
    ctx.set_elements(index)
    ctx.set_scatter(_lib.SLOT_PDF, table)
    ctx.set_transform(0.02, qbin, r, 0.0, nq)
    e, f = ctx.pdf_energy_forces(_lib.SLOT_PDF, qbin, target, _lib.POT_RW, 10.0, n * chains)
    for b in (0, 1, chains // 2, chains - 2, chains - 1):
        ctx.set_positions(pos[b])
        ctx.set_elements(index[:n])
        ctx.set_scatter(_lib.SLOT_PDF, table)
        want_e, want = ctx.pdf_energy_forces(_lib.SLOT_PDF, qbin, target[b], _lib.POT_RW, 10.0, n)
        assert abs(e[b] - want_e) < 1e-6 * abs(want_e)
        assert np.abs(f[b * n:(b + 1) * n] - want).max() < 1e-6 * np.abs(want).max()
