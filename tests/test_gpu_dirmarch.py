"""The direction march: stencils whose points lie on straight lines through
the centre, against the oracle, over cells, boundaries, data types, odd
sides, tile remainders and every epilogue."""
import contextlib

import numpy as np
import pytest

import oracle
from gpaw_amd import _lib, bands
from gpaw_amd.fd_operators import (FDOperator, Gradient, Laplace, LaplaceA,
                                   LaplaceB)
from gpaw_amd.grid_descriptor import GridDescriptor
from gpu_util import dev, host, say
from helpers import bloch_phases, rand, relerr, spec

pytestmark = pytest.mark.gpu
TOL = 1e-13

HEX = np.array([[1, 0, 0], [-0.5, 0.75**0.5, 0], [0, 0, 1.1]])
FCC = np.array([[0, 1, 1], [1, 0, 1], [1, 1, 0]]) * 0.5**0.5
BCC = np.array([[-1, 1, 1], [1, -1, 1], [1, 1, -1]]) * 0.5
SKEW = np.array([[1, 0.13, 0.04], [0.2, 1.05, -0.11], [-0.1, 0.15, 0.95]])
CELLS = {'box': np.eye(3), 'hex': HEX, 'fcc': FCC, 'bcc': BCC, 'skew': SKEW}


@contextlib.contextmanager
def path(p):
    lib = _lib.load()
    _lib.check(lib.gfd_set_tuning(b'force_path', p), 'force_path')
    try:
        yield
    finally:
        lib.gfd_set_tuning(b'force_path', 0)


def grid(N, cell, pbc):
    return GridDescriptor(N, CELLS[cell] * 0.3 * np.array(N)[:, None], pbc)


def both(*steps):
    """Each offset and its opposite."""
    return [(0, 0, 0)] + [o for s in steps
                          for o in (s, tuple(-i for i in s))]


def family(op, dtype=0, nin=1, epilogue=0):
    """Kernel family of a pass (1 general, 2 march, 3 full rows, 4 point)."""
    return _lib.load().gfd_operator_family(op._handle(), dtype, nin, epilogue)


@pytest.mark.parametrize('cell', list(CELLS))
@pytest.mark.parametrize('nn', [1, 2, 3, 4])
@pytest.mark.parametrize('N,pbc', [((8, 7, 9), True),
                                   ((13, 22, 71), (True, True, False)),
                                   ((24, 19, 130), False)])
@pytest.mark.parametrize('dtype', [float, complex])
def test_laplace(cell, nn, N, pbc, dtype):
    rng = np.random.default_rng(nn)
    gd = grid(N, cell, pbc)
    op = Laplace(gd, -0.7, nn, dtype)
    a = rand(rng, (3,) + tuple(gd.n_c), dtype)
    ph = bloch_phases(rng, gd.pbc_c) if dtype == complex else None
    out = dev(np.zeros_like(a))
    say('dirmarch laplace', cell, nn, N, pbc, dtype)
    # the march holds the directions of every cell, at radius 4 the axes only
    takes = 2 if cell == 'box' or nn < 4 else 1
    with path(2):
        assert family(op, int(dtype == complex), 3) == takes
        op.apply(dev(a), out, ph)
    ref = oracle.fd_apply(op.coef_p, op.offset_pc, gd.n_c, gd.neighbor_cd, a,
                          ph)
    assert relerr(host(out), ref) < TOL


def edges(gd):
    """Every in-plane and off-axis direction the march holds."""
    steps = [(0, 0, 1), (0, 1, 0), (0, 1, 1), (1, 0, 0), (1, 1, 0),
             (1, -1, 0), (1, 0, 1), (1, 0, -1)]
    off = both(*steps)
    return FDOperator([-3.0] + [0.1 + 0.2 * i for i in range(1, len(off))],
                      off, gd)


@pytest.mark.parametrize('make,takes', [
    (lambda gd: Gradient(gd, 1, 1.0, 3), 2), (edges, 2),
    (lambda gd: LaplaceA(gd, 0.3), 1), (lambda gd: LaplaceB(gd), 2),
    (lambda gd: FDOperator([1.0, 0.5], [(0, 0, 0), (0, 2, 2)], gd), 2)])
def test_other_stencils(make, takes):
    """One axis only; edges of the cube, and one in-plane direction more than
    the march holds (the Mehrstellen operator: the general kernel); points on
    one side of the centre."""
    rng = np.random.default_rng(3)
    gd = grid((9, 20, 33), 'box', (True, False, True))
    op = make(gd)
    a = rand(rng, (2,) + tuple(gd.n_c))
    out = dev(np.zeros_like(a))
    say('dirmarch stencil', op.description)
    with path(2):
        assert family(op, nin=2) == takes
        op.apply(dev(a), out)
    ref = oracle.fd_apply(op.coef_p, op.offset_pc, gd.n_c, gd.neighbor_cd, a)
    assert relerr(host(out), ref) < TOL


@pytest.mark.parametrize('axis', [0, 1, 2])
@pytest.mark.parametrize('nn', [1, 2, 3, 4])
@pytest.mark.parametrize('N,pbc', [((4, 5, 6), True), ((9, 12, 70), False),
                                   ((21, 37, 16), (False, True, True)),
                                   ((16, 4, 131), (True, False, False))])
@pytest.mark.parametrize('dtype', [float, complex])
def test_gradient(axis, nn, N, pbc, dtype):
    """One axis: its line alone, over tile remainders and sides down to the
    radius."""
    rng = np.random.default_rng(nn)
    gd = grid(tuple(n + 1 - p for n, p in
                    zip(N, np.broadcast_to(pbc, 3))), 'box', pbc)
    op = Gradient(gd, axis, 1.0, nn, dtype)
    a = rand(rng, (3,) + N, dtype)
    ph = bloch_phases(rng, gd.pbc_c) if dtype == complex else None
    ref = oracle.fd_apply(op.coef_p, op.offset_pc, gd.n_c, gd.neighbor_cd, a,
                          ph)
    say('dirmarch gradient', axis, nn, N, pbc, dtype)
    for p in (2, 0):
        out = dev(np.zeros_like(a))
        with path(p):
            assert p == 0 or family(op, int(dtype == complex), 3) == 2
            op.apply(dev(a), out, ph)
        assert relerr(host(out), ref) < TOL


def test_which_kernel():
    """The rule's lines: few real points, complex Laplacians and gradients,
    the passes with other epilogues."""
    even, odd = (grid(N, 'box', True) for N in ((48,) * 3, (47, 48, 49)))
    for R, most in ((1, 5), (2, 4), (3, 5), (4, 4)):
        op = Laplace(even, 1.0, R)
        next = 2 if R == 3 else 3
        assert [family(op, nin=most + i) for i in (0, 1)] == [4, next]
        assert [family(op, nin=i) for i in (8, 9)] == [next, 3]
        op = Gradient(even, 0, 1.0, R)
        assert [family(op, nin=i) for i in (6, 7)] == [4, 3]
        op = Laplace(odd, 1.0, R)
        assert [family(op, nin=i) for i in (5, 8)] == [4, 2]
        lap = [Laplace(gd, 1.0, R, complex) for gd in (even, odd)]
        grad = [[Gradient(gd, c, 1.0, R, complex) for c in range(3)]
                for gd in (even, odd)]
        want = 2 if R >= 3 else 3
        assert [family(op, 1) for op in lap] == [want] * 2
        assert [family(op, 1) for op in grad[0]] == [3, want, want]
        assert [family(op, 1) for op in grad[1]] == [want] * 3
        for epilogue in (2, 3, 4):
            assert family(grad[0][1], 1, 1, epilogue) == 3
            assert family(lap[0], 1, 1, epilogue) == (
                2 if epilogue == 4 else want)


def test_infinities_stay_on_their_lines():
    """A direction without points does not multiply its neighbours."""
    gd = grid((8, 9, 12), 'box', True)
    op = Gradient(gd, 2, 1.0, 2)
    a = np.ones((1, 8, 9, 12))
    a[0, 4, 4, :] = np.inf
    out = dev(np.zeros_like(a))
    with path(2):
        op.apply(dev(a), out)
    bad = ~np.isfinite(host(out)[0])
    assert bad[4, 4].all() and bad.sum() == 12


@pytest.mark.parametrize('offsets', [
    # one side of a diagonal, the first step left out
    [(0, 0, 0), (0, 2, 2)], [(0, 0, 0), (2, 2, 0), (-1, 0, 1)],
    # equal coefficients, one line shorter than the others
    both((1, 0, 0), (0, 1, 0), (0, 2, 0), (0, 0, 1), (0, 0, 2)),
    both((1, 0, 0), (2, 0, 0), (0, 1, 0), (0, 2, 0), (0, 0, 1), (0, 0, 2),
         (1, 1, 0))])
@pytest.mark.parametrize('pbc', [True, False])
def test_infinities_on_partly_filled_lines(offsets, pbc):
    """Points that a line does not have are not read: an infinity there
    leaves the sum finite."""
    rng = np.random.default_rng(6)
    gd = grid((9, 11, 15), 'box', pbc)
    op = FDOperator([1.0] + [0.5] * (len(offsets) - 1), offsets, gd)
    a = rand(rng, (2,) + tuple(gd.n_c))
    a[rng.random(a.shape) < 0.02] = np.inf
    out = dev(np.zeros_like(a))
    with path(2):
        op.apply(dev(a), out)
    ref = oracle.fd_apply(op.coef_p, op.offset_pc, gd.n_c, gd.neighbor_cd, a)
    got, fin = host(out), np.isfinite(ref)
    assert 0 < (~fin).sum() < 0.5 * fin.size
    assert (np.isfinite(got) == fin).all()
    assert (np.isnan(got) == np.isnan(ref)).all()
    assert relerr(got[fin], ref[fin]) < TOL


@pytest.mark.parametrize('cell,N,pbc', [('box', (14, 23, 47), False),
                                        ('hex', (12, 12, 21), True)])
def test_epilogues(cell, N, pbc):
    """Jacobi sweeps, residual with its norm, H psi - eps psi, on the shapes
    the full-row kernel does not take."""
    rng = np.random.default_rng(11)
    gd = grid(N, cell, pbc)
    n = tuple(gd.n_c)
    op = Laplace(gd, -0.5, 3)
    sp = spec(op)
    f, src = rand(rng, n), rand(rng, n)
    say('dirmarch epilogues', cell, N)
    with path(2):
        for w in (2.0 / 3.0, 1.0):
            g = dev(f.copy())
            op.relax(2, g, dev(src), 3, w)
            ref = oracle.fd_relax(2, op.coef_p, op.offset_pc, gd.n_c,
                                  gd.neighbor_cd, f.copy(), src, 3, w)
            assert relerr(host(g), ref) < TOL
        lib = _lib.load()
        r = dev(np.zeros_like(f))
        df, ds = dev(f), dev(src)
        norm = _lib.ctypes.c_double()
        _lib.check(lib.gfd_operator_residual(
            op._handle(), df.data_ptr(), ds.data_ptr(), r.data_ptr(), 1,
            None, _lib.ctypes.byref(norm), None), 'residual')
        want = oracle.fd_apply(sp.coef_p, sp.offset_pc, gd.n_c,
                               gd.neighbor_cd, f) - src
        assert relerr(host(r), want) < TOL
        assert abs(norm.value / (want**2).sum() - 1) < 1e-12
        for dtype, nn in ((float, 3), (complex, 3),
                          (complex, 4 if cell == 'box' else 2)):
            kin = Laplace(gd, -0.5, nn, dtype)
            assert family(kin, int(dtype == complex), 3, 4) == 2
            psi = rand(rng, (3,) + n, dtype)
            vt, eps = rng.uniform(-2, 0, n), rng.uniform(-1, 1, 3)
            ph = bloch_phases(rng, gd.pbc_c) if dtype == complex else None
            out = dev(np.zeros_like(psi))
            bands.apply_hamiltonian(kin, dev(vt), dev(psi), out, ph,
                                    eps=dev(eps))
            want = oracle.fd_apply(kin.coef_p, kin.offset_pc, gd.n_c,
                                   gd.neighbor_cd, psi, ph) + \
                (vt - eps[:, None, None, None]) * psi
            assert relerr(host(out), want) < TOL


@pytest.mark.parametrize('cell,N,pbc', [('box', (20, 28, 36), False),
                                        ('hex', (16, 16, 24), True)])
@pytest.mark.parametrize('dtype', [float, complex])
@pytest.mark.parametrize('fp32', [False, True])
def test_preconditioner(cell, N, pbc, dtype, fp32):
    """The UPDATE epilogues, FP32 data with FP64 residual and result among
    them, against the general kernel (2e-6: the FP32 chain's bar)."""
    from types import SimpleNamespace

    from gpaw_amd.preconditioner import Preconditioner
    rng = np.random.default_rng(5)
    gd = grid(N, cell, pbc)
    kin = Laplace(gd, -0.5, 3, dtype)
    pc = Preconditioner(gd, kin, dtype, block=3, fp32=fp32)
    res = dev(rand(rng, (3,) + tuple(gd.n_c), dtype))
    ph = bloch_phases(rng, gd.pbc_c) if dtype == complex else None
    kpt = SimpleNamespace(phase_cd=ph)
    outs = []
    say('dirmarch preconditioner', cell, N, dtype, fp32)
    for p in (2, 1):
        with path(p):
            outs.append(host(pc(res, kpt)))
    assert relerr(outs[0], outs[1]) < (2e-6 if fp32 else TOL)


@pytest.mark.parametrize('N', [(8, 4, 14), (8, 4, 16), (5, 5, 12),
                               (4, 4, 4), (9, 6, 70)])
@pytest.mark.parametrize('dtype', [float, complex])
def test_radius_4(N, dtype):
    """Planes of a few short rows, whose halo at radius 4 is more than four
    points per tile point; sides equal to the radius; a z remainder."""
    rng = np.random.default_rng(4)
    gd = grid(N, 'box', True)
    count = 3 if dtype == complex else -(-620_000 // np.prod(N))
    a = rand(rng, (count,) + N, dtype)
    ph = bloch_phases(rng, gd.pbc_c) if dtype == complex else None
    for op in (Laplace(gd, -0.7, 4, dtype), Gradient(gd, 1, 1.0, 4, dtype)):
        out = dev(np.zeros_like(a))
        say('dirmarch radius 4', N, dtype, op.description)
        for p in (0, 2):
            with path(p):
                op.apply(dev(a), out, ph)
            ref = oracle.fd_apply(op.coef_p, op.offset_pc, gd.n_c,
                                  gd.neighbor_cd, a, ph)
            assert relerr(host(out), ref) < TOL


def test_tiles_are_looked_up():
    """A batch searches for its tile once, with the residual's block bound;
    batches beyond the number kept still run right."""
    rng = np.random.default_rng(8)
    gd = grid((9, 13, 17), 'hex', True)
    op = Laplace(gd, -0.7, 2, complex)
    searches = _lib.load().gfd_march_tile_searches
    a = rand(rng, (40,) + tuple(gd.n_c), complex)
    da, out = dev(a), dev(np.zeros_like(a))
    ref = oracle.fd_apply(op.coef_p, op.offset_pc, gd.n_c, gd.neighbor_cd, a)
    op.apply(da[:3], out[:3])
    n = searches()
    for _ in range(3):
        op.apply(da[:3], out[:3])
    assert searches() == n
    norm, lib = _lib.ctypes.c_double(), _lib.load()
    for new in (1, 0, 0):      # one halo more, with and without a norm
        n = searches()
        _lib.check(lib.gfd_operator_residual(
            op._handle(), da.data_ptr(), da.data_ptr(), out.data_ptr(), 2,
            None, _lib.ctypes.byref(norm), None), 'residual')
        assert searches() == n + new
    for nb in (*range(1, 41), 1, 40):
        out.zero_()
        op.apply(da[:nb], out[:nb])
        assert relerr(host(out)[:nb], ref[:nb]) < TOL


def test_many_tiny_skew_cells():
    """A residual on fixed scratch of more cells than it has partial sums
    for one block each: the general kernel, with one per 256 points."""
    import torch
    gd = grid((4, 4, 4), 'hex', True)
    op = Laplace(gd, -0.7, 1)
    lib = _lib.load()
    nb = lib.gfd_operator_residual_noalloc_max_blocks() + 60
    g = torch.Generator(device='cuda').manual_seed(2)
    a, b = (torch.randn((nb, 4, 4, 4), generator=g, dtype=torch.float64,
                        device='cuda') for _ in range(2))
    r, norm = torch.empty_like(a), _lib.ctypes.c_double()
    _lib.check(lib.gfd_operator_residual_noalloc(
        op._handle(), a.data_ptr(), b.data_ptr(), r.data_ptr(), nb, None,
        _lib.ctypes.byref(norm), None), 'residual')
    ref = oracle.fd_apply(op.coef_p, op.offset_pc, gd.n_c, gd.neighbor_cd,
                          host(a)) - host(b)
    assert relerr(host(r), ref) < TOL
    assert abs(norm.value / (ref**2).sum() - 1) < 1e-12
