"""The spreading kernels at the edges of what they accept: common factors of
the results, positions that are not finite or very far apart, state kept
between calls, captured calls, and tables and grids that the recurrence kernels
take."""
import numpy as np
import pytest

from oracle import scatter as oracle
from pyiid_amd import _lib, structures
from pyiid_amd.formfactors import element_table
from test_gpu_spread import force_check

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


def test_gradient_after_a_sampler_and_new_elements(ctx):
    """A sampler brings the atoms closer together, which the next gradient takes
    note of; new elements then put the atoms back to where they were uploaded,
    farther apart, and the gradient has to reach that far again."""
    n, nq, qbin = 3, 250, 0.1
    pos = np.array([(0, 0, 0), (10, 0, 0), (0, 10, 0)], np.float32)
    r = 1.0 + 0.02 * np.arange(100)
    per_atom = load(ctx, pos, np.full(n, 79), qbin, nq)
    ctx.set_scatter(_lib.SLOT_PDF, per_atom[:1])
    ctx.set_transform(0.02, qbin, r, 0.0, nq)
    want = ctx.grad_fq(_lib.SLOT_FQ, qbin, n, nq)

    def spread():
        p = ctx.get_positions(n)
        return max(np.linalg.norm(p[a] - p[b]) for a in range(n) for b in range(a))
    for seed in range(200):  # nearly free flight: every proposal is accepted
        ctx.set_positions(pos)
        ctx.hmc_setup(_lib.SLOT_PDF, qbin, np.cos(r), _lib.POT_RW, 1e-9, np.full(n, 1.0))
        ctx.hmc_run(1, 1, 3.0, 1.0, seed, 1, use_graph=False)
        if spread() < 8.0:
            break
    assert spread() < 8.0
    closer = ctx.grad_fq(_lib.SLOT_FQ, qbin, n, nq)
    assert np.abs(closer - want).max() > 0.1 * np.abs(want).max()
    ctx.set_elements(np.zeros(n, np.int32))
    np.testing.assert_array_equal(ctx.get_positions(n), pos)
    np.testing.assert_array_equal(ctx.grad_fq(_lib.SLOT_FQ, qbin, n, nq), want)


@pytest.mark.parametrize("where", [0, 7])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_host_and_device_positions_that_are_not_finite(fixed_shapes, where, value):
    """One atom's x is not finite: from host arrays, where the extent is taken on
    the host, F, gradient, energy and forces are those of a device upload, where
    it is taken on the GPU; the pairs of the other atoms are all there."""
    import torch
    n, nq, qbin = 60, 250, 0.1
    pos = structures.jitter(structures.fcc_nearest(n), 0.05, seed=4).astype(np.float32)
    rest = np.arange(n) != where
    table, index, _ = element_table(np.full(n, 79), qbin, nq)
    r = 2.0 + 0.02 * np.arange(300)

    def results(device, p):
        c = _lib.Context(0)
        try:
            c.set_positions(torch.from_numpy(p).cuda() if device else p,
                            flags=_lib.PYIID_DEVICE if device else 0)
            c.set_elements(np.zeros(len(p), np.int32))
            c.set_scatter(_lib.SLOT_FQ, table)
            c.set_scatter(_lib.SLOT_PDF, table)
            c.set_transform(0.02, qbin, r, 0.0, nq)
            g = c.grad_fq(_lib.SLOT_FQ, qbin, len(p), nq)
            e, f = c.pdf_energy_forces(_lib.SLOT_PDF, qbin, np.cos(r), _lib.POT_RW, 1.0, len(p))
            return g, c.fq(_lib.SLOT_FQ, qbin, nq), np.float64(e), f
        finally:
            c.close()
    moved = pos.copy()
    moved[where, 0] = value
    host, device = results(False, moved), results(True, moved)
    for a, b in zip(host, device):
        np.testing.assert_array_equal(a, b)
    if np.isnan(value):  # y and z: the pairs of the others, none with the atom itself
        want = results(False, pos[rest])[0] * ((n - 1.0) / n)
        off = np.abs(host[0][rest][:, 1:] - want[:, 1:])
        assert off.max() < 1e-6 * np.abs(want).max()


@pytest.mark.parametrize("kinds", [1, 3])
@pytest.mark.parametrize("bad", [(0, (0,)), (3, (1,)), (69, (0, 2)), (5, (0, 1, 2))])
def test_gradient_shows_positions_that_are_not_numbers(ctx, kinds, bad):
    """One atom has components that are not numbers: so have the same components of
    every atom's gradient, on the spreading kernel as on the recurrence kernels,
    and the other components are those of the remaining pairs.  Duplicated atoms
    are no such case."""
    n, nq, qbin = 70, 250, 0.1
    which, where = bad
    pos = structures.jitter(structures.fcc_nearest(n), 0.05, seed=6).astype(np.float32)
    pos[40] = pos[41]
    numbers = np.array([79, 28, 78])[np.arange(n) % kinds]
    load(ctx, pos, numbers, qbin, nq)
    assert np.isfinite(ctx.grad_fq(_lib.SLOT_FQ, qbin, n, nq)).all()
    pos[which, list(where)] = np.nan
    got = {}
    try:
        for kernel in (_lib.GRAD_AUTO, _lib.GRAD_ORDERED, _lib.GRAD_SYMMETRIC):
            ctx.set_grad_kernel(kernel)
            ctx.set_positions(pos)
            got[kernel] = ctx.grad_fq(_lib.SLOT_FQ, qbin, n, nq)
            assert (ctx.grad_shape() == (False, 0, 0)) == (kernel == _lib.GRAD_AUTO)
    finally:
        ctx.set_grad_kernel(_lib.GRAD_AUTO)
    new, old = got[_lib.GRAD_AUTO], got[_lib.GRAD_ORDERED]
    for c in range(3):
        assert np.isnan(new[:, c]).all() == (c in where)
        np.testing.assert_array_equal(np.isnan(new[:, c]), np.isnan(old[:, c]))
        np.testing.assert_array_equal(np.isnan(new[:, c]), np.isnan(got[_lib.GRAD_SYMMETRIC][:, c]))
        if c not in where:
            assert np.abs(new[:, c] - old[:, c]).max() < 2e-6 * np.abs(old[:, c]).max()
    import torch
    ctx.set_positions(torch.from_numpy(pos).cuda(), flags=_lib.PYIID_DEVICE)
    np.testing.assert_array_equal(ctx.grad_fq(_lib.SLOT_FQ, qbin, n, nq), new)


class Captured:
    """A context on a stream of torch's, whose gradient (with F) goes to `grad` and
    `fq`; `capture` records calls into a graph."""

    def __init__(self, n, kinds, qbin, nq):
        import torch
        self.torch, self.n, self.qbin, self.nq = torch, n, qbin, nq
        self.stream = torch.cuda.Stream()
        self.c = _lib.Context(0)
        self.c.set_stream(self.stream.cuda_stream)
        self.numbers = np.array([79, 28, 78])[np.random.RandomState(n).permutation(n) % kinds]
        self.table, self.index, _ = element_table(self.numbers, qbin, nq)
        self.grad = torch.zeros((n, 3, nq), device="cuda")
        self.fq = torch.zeros(nq, device="cuda")
        self.buf = torch.zeros((n, 3), device="cuda")
        torch.cuda.synchronize()

    def load(self, pos):
        self.c.set_positions(pos)
        self.c.set_elements(self.index)
        for slot in (_lib.SLOT_FQ, _lib.SLOT_PDF):
            self.c.set_scatter(slot, self.table)

    def eager(self):
        self.c.grad_fq(_lib.SLOT_FQ, self.qbin, self.n, self.nq, out=self.grad, fq_out=self.fq,
                       flags=_lib.PYIID_DEVICE)

    def upload(self):
        self.c.set_positions(self.buf, flags=_lib.PYIID_DEVICE)

    def capture(self, calls):
        g = self.torch.cuda.CUDAGraph()
        self.torch.cuda.synchronize()
        with self.torch.cuda.graph(g, stream=self.stream):
            for f in calls:
                f()
        return g

    def replay(self, g):
        with self.torch.cuda.stream(self.stream):
            g.replay()

    def result(self):
        self.torch.cuda.synchronize()
        out = self.grad.cpu().numpy(), self.fq.cpu().numpy()
        with self.torch.cuda.stream(self.stream):
            self.grad.zero_()
            self.fq.zero_()
        return out

    def fill(self, pos):
        self.buf.copy_(self.torch.from_numpy(pos))
        self.torch.cuda.synchronize()

    def fresh(self, pos):
        other = Captured(self.n, 1, self.qbin, self.nq)
        other.table, other.index = self.table, self.index
        other.load(pos)
        other.eager()
        out = other.result()
        other.c.close()
        return out


def same(got, want):
    for a, b in zip(got, want):
        assert np.any(b)
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("n,kinds,qbin,nq", [(60, 1, 0.1, 250), (300, 1, 0.1, 250), (300, 3, 0.1, 250),
                                             (5000, 1, 0.02, 300)])
def test_captured_gradient_follows_the_positions(n, kinds, qbin, nq):
    """A gradient in a graph, captured when the extent, the reach and the element
    order of the positions were known, replayed after uploads of larger and smaller
    structures from the host and the device: each time a new context's result."""
    base = structures.jitter(structures.fcc_nearest(n), 0.05, seed=n).astype(np.float32)
    s = Captured(n, kinds, qbin, nq)
    s.load(base)
    for _ in range(2):
        s.fill(base)
        s.upload() if n > 4096 else s.c.set_positions(base)
        s.eager()
        s.eager()
    g = s.capture([s.eager])
    s.result()
    for scale, device in ((1.0, True), (2.0, False), (0.8, True), (1.7, True), (1.3, False)):
        pos = (base * np.float32(scale)).astype(np.float32)
        s.fill(pos)
        s.upload() if device else s.c.set_positions(pos)
        s.replay(g)
        want = s.fresh(pos)
        same(s.result(), want)
        s.eager()
        same(s.result(), want)
    del g
    s.c.close()


@pytest.mark.parametrize("n,kinds", [(60, 1), (300, 3)])
def test_captured_upload_and_gradient(n, kinds):
    """An upload and a gradient in a graph, replayed with other positions in the
    buffer; an eager gradient between the replays finds the atoms where the replay
    has put them.  Positions in host memory cannot be captured."""
    nq = 250
    base = structures.jitter(structures.fcc_nearest(n), 0.05, seed=n).astype(np.float32)
    s = Captured(n, kinds, 0.1, nq)
    s.load(base)
    s.fill(base)
    for _ in range(2):
        s.upload()
        s.eager()

    def refused():
        with pytest.raises(Exception, match="captured"):
            s.c.set_positions(base)
    g = s.capture([s.upload, s.eager, refused])
    s.result()
    for scale in (1.0, 1.9, 0.8, 1.6):
        pos = (base * np.float32(scale)).astype(np.float32)
        s.fill(pos)
        s.replay(g)
        want = s.fresh(pos)
        same(s.result(), want)
        s.eager()
        same(s.result(), want)
        s.fill((base * np.float32(0.9)).astype(np.float32))
        s.upload()
        s.eager()
        same(s.result(), s.fresh((base * np.float32(0.9)).astype(np.float32)))
    del g
    s.c.close()


def test_captured_gradient_after_a_sampler():
    """Atoms of three elements that a sampler has moved since the capture, by up to
    a hundred A: the replay finds them there.  The extent has grown past 114 A, up
    to which the gradient's grids are of 32 bits; the graph keeps its choice, the
    eager call does not, so the two agree to rounding (2^-20 of the largest entry,
    as the product's two halves allow), not bit for bit."""
    n, nq, qbin = 300, 250, 0.1
    base = structures.jitter(structures.fcc_nearest(n), 0.05, seed=n).astype(np.float32)
    s = Captured(n, 3, qbin, nq)
    s.load(base)
    r = 2.0 + 0.02 * np.arange(300)
    s.c.set_transform(0.02, qbin, r, 0.0, nq)
    for _ in range(3):
        s.c.set_positions(base)
        s.eager()
    g = s.capture([s.eager])
    s.replay(g)
    same(s.result(), s.fresh(base))
    s.c.hmc_setup(_lib.SLOT_PDF, qbin, np.cos(r), _lib.POT_RW, 1.0, np.full(n, 100.0))
    s.c.hmc_run(3, 3, 1.0, 1e-3, 1, 1)
    assert np.abs(s.c.get_positions(n) - base).max() > 0.01
    s.replay(g)
    got = s.result()
    s.eager()
    for a, b in zip(got, s.result()):
        assert np.abs(a - b).max() < 2.0 ** -20 * np.abs(b).max()
    del g
    s.c.close()


def device_forces(c, n, target, chains=1):
    """Forces alone, all arrays on the GPU: no energy that the host would wait for."""
    import torch
    out = torch.zeros((n, 3), dtype=torch.float64, device="cuda")
    _lib.check(c.lib.pyiid_pdf_energy_forces(c.handle, _lib.SLOT_PDF, 0.1, target.data_ptr(),
                                             _lib.POT_RW, 1.0, None, out.data_ptr(),
                                             _lib.PYIID_DEVICE))
    return out


def test_force_table_grows_after_calls_without_energy():
    """Atoms moved past the force table's end on the device: their pairs are summed
    directly, and the next call has a table for their extent, whether or not the
    host asks for energies: the same bits as a new context's."""
    import torch
    n, nq, qbin = 90, 250, 0.1
    base = structures.jitter(structures.fcc_nearest(n), 0.05, seed=2).astype(np.float32)
    pos = base.copy()
    pos[40:] += np.float32(17.3)
    table, _, _ = element_table(np.full(n, 79), qbin, nq)
    r = 2.0 + 0.02 * np.arange(300)
    target = torch.from_numpy(np.cos(r)).cuda()

    def context(p):
        c = _lib.Context(0)
        c.set_positions(torch.from_numpy(p).cuda(), flags=_lib.PYIID_DEVICE)
        c.set_elements(np.zeros(n, np.int32))
        c.set_scatter(_lib.SLOT_PDF, table)
        c.set_transform(0.02, qbin, r, 0.0, nq)
        c.set_autotune(True)
        out = device_forces(c, n, target)
        c.synchronize()
        return c, out.cpu().numpy()
    c, _ = context(base)
    moved = torch.from_numpy(pos).cuda()
    got = []
    for _ in range(2):
        c.set_positions(moved, flags=_lib.PYIID_DEVICE)
        out = device_forces(c, n, target)
        c.synchronize()
        got.append(out.cpu().numpy())
    fresh, want = context(pos)
    assert np.abs(got[0] - want).max() < 1e-6 * np.abs(want).max()
    np.testing.assert_array_equal(got[1], want)
    c.close()
    fresh.close()


def test_batch_after_a_larger_one_keeps_its_extent():
    """Energies of eight chains, then of four: nothing of the first batch's results
    is taken for a pair past the force table, which would make the next call wait
    for the extent, and so fail in a capture."""
    import torch
    nq, qbin, r = 250, 0.1, 2.0 + 0.02 * np.arange(300)
    chains = [structures.jitter(structures.fcc_nearest(40), 0.05, seed=b).astype(np.float32)
              for b in range(8)]
    stream = torch.cuda.Stream()
    c = _lib.Context(0)
    c.set_stream(stream.cuda_stream)
    table, _, _ = element_table(np.full(40, 79), qbin, nq)
    target = np.tile(np.cos(r) + 0.5, (8, 1))
    c.set_transform(0.02, qbin, r, 0.0, nq)
    for b in (8, 4):
        c.set_batch(chains[:b])
        c.set_elements(np.zeros(40 * b, np.int32))
        c.set_scatter(_lib.SLOT_PDF, table)
        e, f = c.pdf_energy_forces(_lib.SLOT_PDF, qbin, target[:b], _lib.POT_RW, 1.0, 40 * b)
        assert np.all(e > 0.0)
    dev = torch.from_numpy(target).cuda()
    out = torch.zeros((160, 3), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        _lib.check(c.lib.pyiid_pdf_energy_forces(c.handle, _lib.SLOT_PDF, qbin, dev.data_ptr(),
                                                 _lib.POT_RW, 1.0, None, out.data_ptr(),
                                                 _lib.PYIID_DEVICE))
    for _ in range(3):
        with torch.cuda.stream(stream):
            out.zero_()
            g.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy(), f)
        np.testing.assert_array_equal(
            c.pdf_energy_forces(_lib.SLOT_PDF, qbin, target[:4], _lib.POT_RW, 1.0, 160)[1], f)
    del g
    c.close()


@pytest.mark.parametrize("rows", [361, 362, 400, 1000])
def test_tables_of_many_rows(ctx, rows):
    """A table with a row for every atom and more (element pairs up to and past what
    one launch of the transform takes): F, gradient and forces against the oracle."""
    n, nq, qbin = 80, 60, 0.25
    rs = np.random.RandomState(rows)
    pos = structures.jitter(structures.fcc_nearest(n), 0.05, seed=rows).astype(np.float32)
    q = np.arange(nq) * qbin
    table = (rs.uniform(20, 80, (rows, 1)) * np.exp(-rs.uniform(0.5, 3.0, (rows, 1)) * (q / 12.6) ** 2)
             ).astype(np.float32)
    index = rs.permutation(rows)[:n].astype(np.int32)
    ctx.set_positions(pos)
    ctx.set_elements(index)
    ctx.set_scatter(_lib.SLOT_FQ, table)
    per_atom = table[index]
    want, gwant = oracle.fq(pos, per_atom, qbin), oracle.grad_fq(pos, per_atom, qbin)
    # (a structure 2% smaller: near a fit the residual would magnify F's rounding)
    target = oracle.fq((pos * np.float32(0.98)).astype(np.float32), per_atom, qbin)
    for _ in range(2):
        fq = np.empty(nq, np.float32)
        g = ctx.grad_fq(_lib.SLOT_FQ, qbin, n, nq, fq_out=fq)
        assert np.abs(ctx.fq(_lib.SLOT_FQ, qbin, nq) - want).max() < 1e-6 * np.abs(want).max()
        assert np.abs(fq - want).max() < 1e-6 * np.abs(want).max()
        assert np.abs(g - gwant).max() < 2e-6 * np.abs(gwant).max()
        e, f = ctx.fq_energy_forces(_lib.SLOT_FQ, qbin, 0, target, _lib.POT_RW, 10.0, n)
        fwant = 10.0 * oracle.wrap_grad_rw(gwant, want, target)
        assert np.abs(f - fwant).max() < 5e-6 * np.abs(fwant).max()


@pytest.mark.parametrize("n,kinds", [(40, 1), (40, 2), (300, 1)])
def test_energies_of_negative_bins(ctx, n, kinds):
    """Energies and forces take a bin width of either sign: F(-Q) = -F(Q), so that
    the energy against a target is that of the positive bins against its negative
    (to the 1e-6 that two kernels differ by; the target is that of a structure 2%
    smaller, Rw 0.7: near a fit the residual would magnify F's rounding).  F and the
    gradient refuse it."""
    nq, qbin, r = 250, 0.1, 2.0 + 0.02 * np.arange(300)
    pos = structures.jitter(structures.fcc_nearest(n), 0.05, seed=n).astype(np.float32)
    numbers = np.array([79, 28])[np.arange(n) % kinds]
    table, index, _ = element_table(numbers, qbin, nq)
    load(ctx, (pos * np.float32(0.98)).astype(np.float32), numbers, qbin, nq)
    ctx.set_scatter(_lib.SLOT_PDF, table)
    ctx.set_transform(0.02, qbin, r, 0.0, nq)
    fq = ctx.fq(_lib.SLOT_FQ, qbin, nq)
    ctx.set_positions(pos)
    for target, call in (
            (ctx.pdf(fq, 300),
             lambda q, t: ctx.pdf_energy_forces(_lib.SLOT_PDF, q, t, _lib.POT_RW, 10.0, n)),
            (fq.astype(np.float64),
             lambda q, t: ctx.fq_energy_forces(_lib.SLOT_FQ, q, 0, t, _lib.POT_RW, 10.0, n))):
        e, f = call(qbin, target)
        en, fn = call(-qbin, -target)
        assert abs(en - e) < 1e-5 * abs(e)
        assert np.abs(fn - f).max() < 1e-5 * np.abs(f).max()
        assert call(-qbin, target)[0] > 1.01 * e
    for width in (-qbin, 0.0, np.nan):
        with pytest.raises(ValueError):
            ctx.fq(_lib.SLOT_FQ, width, nq)
        with pytest.raises(ValueError):
            ctx.grad_fq(_lib.SLOT_FQ, width, n, nq)


@pytest.mark.parametrize("n,kinds,nq,q_max,spread", [
    (400, 1, 40, 1.01, True), (401, 1, 40, 1.01, False), (400, 1, 40, 0.9, False),
    (650, 1, 129, 1.01, False), (650, 1, 130, 1.01, True), (650, 1, 16, 12.0, True),
    (650, 1, 16, 11.0, False), (900, 1, 90, 9.9, False), (900, 1, 90, 10.1, True),
    (900, 1, 257, 1.01, True), (1300, 1, 105, 3.9, False), (1300, 1, 105, 4.1, True),
    (100, 3, 100, 25.0, True), (100, 4, 100, 25.0, False), (210, 4, 250, 25.0, True),
    (210, 6, 250, 25.0, False)])
def test_gradient_beside_the_lines_between_kernels(ctx, n, kinds, nq, q_max, spread):
    """Both sides of the rule's lines (atoms, bins, largest Q, elements): the kernel
    it names runs, and F and the gradient are the oracle's (1e-6 and 2e-6 of the
    largest, as everywhere)."""
    qbin = q_max / nq
    pos = structures.jitter(structures.fcc_nearest(n), 0.05, seed=n).astype(np.float32)
    q = np.arange(nq) * qbin
    table = np.stack([(20 + 10 * e) * np.exp(-(1 + 0.2 * e) * (q / 12.6) ** 2)
                      for e in range(kinds)]).astype(np.float32)
    index = (np.arange(n) % kinds).astype(np.int32)
    ctx.set_positions(pos)
    ctx.set_elements(index)
    ctx.set_scatter(_lib.SLOT_FQ, table)
    fq = np.empty(nq, np.float32)
    g = ctx.grad_fq(_lib.SLOT_FQ, qbin, n, nq, fq_out=fq)
    assert (ctx.grad_shape() == (False, 0, 0)) == spread
    want = oracle.fq(pos, table[index], qbin)
    rows = np.arange(0, n, 29)
    gwant = oracle.grad_fq(pos, table[index], qbin, atom_index=rows)
    assert np.abs(fq - want).max() < 1e-6 * np.abs(want).max()
    assert np.abs(ctx.fq(_lib.SLOT_FQ, qbin, nq) - want).max() < 1e-6 * np.abs(want).max()
    assert np.abs(g[rows] - gwant).max() < 2e-6 * np.abs(gwant).max()


@pytest.mark.parametrize("chains,n,kinds", [(1, 90, 12), (1, 90, 40), (40, 45, 3), (40, 130, 3), (20, 100, 6)])
def test_batches_beside_the_lines_between_kernels(ctx, chains, n, kinds):
    """F, energies and forces of batches on either side of the rules, against each
    chain alone in float64."""
    nq, qbin, r = 100, 0.2, 2.0 + 0.02 * np.arange(120)
    pos = [structures.jitter(structures.fcc_nearest(n), 0.05, seed=b).astype(np.float32)
           for b in range(chains)]
    q = np.arange(nq) * qbin
    table = np.stack([(20 + 3 * e) * np.exp(-(1 + 0.05 * e) * (q / 12.6) ** 2)
                      for e in range(kinds)]).astype(np.float32)
    index = (np.arange(n) % kinds).astype(np.int32)
    target = np.tile(np.cos(r) + 0.2, (chains, 1))
    ctx.set_batch(pos)
    ctx.set_elements(np.tile(index, chains))
    for slot in (_lib.SLOT_FQ, _lib.SLOT_PDF):
        ctx.set_scatter(slot, table)
    ctx.set_transform(0.02, qbin, r, 0.0, nq)
    for _ in range(2):
        fq = ctx.fq(_lib.SLOT_FQ, qbin, nq, n_chain=chains).reshape(chains, nq)
        e, f = ctx.pdf_energy_forces(_lib.SLOT_PDF, qbin, target, _lib.POT_RW, 10.0, n * chains)
    want_fq = [oracle.fq(p, table[index], qbin) for p in pos]
    for b in (0, chains // 2, chains - 1):
        assert np.abs(fq[b] - want_fq[b]).max() < 1e-6 * np.abs(want_fq[b]).max()
    for b in (0, chains - 1):
        ctx.set_positions(pos[b])
        ctx.set_elements(index)
        ctx.set_transform(0.02, qbin, r, 0.0, nq)
        g = ctx.pdf(want_fq[b].astype(np.float32), len(r))
        gg = ctx.grad_pdf(oracle.grad_fq(pos[b], table[index], qbin), len(r))
        want = 10.0 * oracle.wrap_grad_rw(gg, g, target[0])
        assert abs(np.atleast_1d(e)[b] - 10.0 * oracle.get_rw(target[0], g)[0]) < 1e-5
        assert np.abs(f[b * n:(b + 1) * n] - want).max() < 1e-5 * np.abs(want).max()


def upload_device(c, pos):
    import torch
    c.set_positions(torch.from_numpy(pos).cuda(), flags=_lib.PYIID_DEVICE)


@pytest.mark.parametrize("n,device", [(300, True), (4097, False), (4097, True)])
def test_fixed_shapes_forget_earlier_positions(fixed_shapes, n, device):
    """Without the autotuner, F and gradient have the same bits in a context that has
    seen the same atoms sixty times farther apart (whose scale sums most pairs in
    another way) as in a new one."""
    nq, qbin = 130, 0.2
    pos = structures.jitter(structures.fcc_nearest(n), 0.05, seed=1).astype(np.float32)
    table, index, _ = element_table(np.full(n, 79), qbin, nq)
    got = []
    for earlier in (True, False):
        c = _lib.Context(0)
        for p in ([60 * pos] if earlier else []) + [pos]:
            if device:
                upload_device(c, p)
            else:
                c.set_positions(p)
            if p is not pos or not earlier:  # the layout stays
                c.set_elements(index)
                c.set_scatter(_lib.SLOT_FQ, table)
            fq = np.empty(nq, np.float32)
            out = [c.fq(_lib.SLOT_FQ, qbin, nq),
                   c.grad_fq(_lib.SLOT_FQ, qbin, n, nq, fq_out=fq), fq]
        got.append(out)
        c.close()
    same(*got)


@pytest.mark.parametrize("earlier,device,graph", [(0.4, True, False), (3, True, True), (1, False, True)])
def test_fixed_shapes_forget_earlier_forces(fixed_shapes, earlier, device, graph):
    """The same of forces and of the sampler, 16 chains: the tables' length, past
    which pairs are summed directly, must not be that of earlier positions (0.4 times
    as far apart, or 3 times, which makes the tables in another way), nor that of
    a proposal's graph."""
    n, chains, nq, qbin, r = 40, 16, 250, 0.1, 2.0 + 0.02 * np.arange(300)
    base = np.concatenate([structures.jitter(structures.fcc_nearest(n), 0.05, seed=b)
                           for b in range(chains)]).astype(np.float32)
    table, _, _ = element_table(np.full(n, 79), qbin, nq)
    target = np.tile(np.cos(r) + 0.2, (chains, 1))

    def results(earlier, device, graph):
        import torch
        c = _lib.Context(0)
        off = np.arange(chains + 1, dtype=np.int64) * n

        def upload(p):
            dev = torch.from_numpy(p).cuda()
            _lib.check(c.lib.pyiid_set_batch(c.handle, dev.data_ptr() if device else p.ctypes.data,
                                             n * chains, off.ctypes.data, chains,
                                             _lib.PYIID_DEVICE if device else 0))
            c.synchronize()

        def forces():
            return c.pdf_energy_forces(_lib.SLOT_PDF, qbin, target, _lib.POT_RW, 1.0, n * chains)
        upload(np.float32(earlier) * base)
        c.set_elements(np.zeros(n * chains, np.int32))
        c.set_scatter(_lib.SLOT_PDF, table)
        c.set_transform(0.02, qbin, r, 0.0, nq)
        out = []
        forces()
        for scale in (1, 2):
            upload(np.float32(scale) * base)
            out += forces()
            if scale == 1:
                c.hmc_setup(_lib.SLOT_PDF, qbin, target, _lib.POT_RW, 10.0, np.full(n * chains, 1.0))
            # (from the forces of the setup or of the run before)
            for _ in range(2):
                out.append(c.hmc_run(4, 5, 0.1, 1.0, 1, chains, use_graph=graph)[0])
            out += [c.get_positions(n * chains), *forces()]
        c.close()
        return out
    want = results(1, False, False)
    same(results(earlier, device, graph), want)


@pytest.mark.parametrize("cells", [6825, 6826, 6827])
def test_longest_force_table(ctx, cells):
    """Force tables that fill the 160 KB of LDS but for 40 and 16 bytes, and a
    structure that would need a cell more than fits (the recurrence kernel).  The
    outermost pair then moves on the device to where it reads the table's last
    cell, a tenth beyond the extent that the table was made for."""
    nq, qbin = 600, 0.05
    h = np.pi / (5 * nq * np.float64(np.float32(qbin)))
    inner = structures.jitter(structures.fcc_nearest(68), 0.05, seed=4)
    inner -= 0.5 * (inner.min(0) + inner.max(0))

    def structure(length):
        ends = np.array([(0.5 * length, 0, 0), (-0.5 * length, 0, 0)])
        return np.concatenate([inner, ends]).astype(np.float32)

    def table_cells(pos):
        x = pos.astype(np.float64)
        mid = 0.5 * (x.min(0) + x.max(0))
        reach = min(np.linalg.norm(x.max(0) - x.min(0)), 2 * np.linalg.norm(x - mid, axis=1).max())
        return int(1.1 * reach / h + 8)
    base = structure((cells - 7.5) * h / 1.1)
    assert table_cells(base) == cells
    assert (24 * cells <= 160 * 1024) == (cells <= 6826)
    force_check(ctx, base, base, np.full(70, 79), qbin, nq)
    pos = structure((cells - 0.6) * h)
    assert int(np.linalg.norm(pos[-1].astype(np.float64) - pos[-2]) / h) == cells - 1
    force_check(ctx, pos, base, np.full(70, 79), qbin, nq, lambda p: upload_device(ctx, p))
