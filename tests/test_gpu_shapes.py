"""Launch shapes of the kernels that split the grid by a rule on its sizes,
against the oracle at the sizes where a split can go wrong: segments of one
cell, a last segment or workgroup that is nearly empty, rows that are no
multiple of a wavefront, block edges inside and at the ends of a segment.

FP64 is held to 1e-12 per field after one step (the bound of the other
parity tests: the operations are the oracle's, the transcendentals may
differ by an ulp); mixed precision to 1e-5 (FP32 rates and states)."""
import numpy as np
import pytest

import oracle
from code_tohoku_amd import ics, mcf, surrogate
from code_tohoku_amd.restart import Input3D
from helpers import interior, rel_linf, worst

pytestmark = pytest.mark.gpu


def box(nx, ny, nz, periodic):
    q = 0.25  # cell size: a power of two, so every spacing is the same bits
    p = Input3D(np1x=nx // 2, np2x=nx - nx // 2, np1y=ny // 2, np2y=ny - ny // 2, np1z=nz // 2, np2z=nz - nz // 2,
                ql1x=q * (nx // 2), ql2x=q * (nx - nx // 2), ql1y=q * (ny // 2), ql2y=q * (ny - ny // 2),
                ql1z=q * (nz // 2), ql2z=q * (nz - nz // 2))
    if periodic:
        p.bcx1 = p.bcx2 = 3
    return p


def check_step(p, st, nsplit, precision):
    o = oracle.Oracle(p, st, nsplit=nsplit)
    g = mcf.Domain(p, nsplit=nsplit, precision=precision)
    g.upload(st)
    dts, _ = o.run(1)
    assert len(dts) == 1
    if precision == mcf.PREC_FP64:
        np.testing.assert_allclose(g.run(1), dts, rtol=1e-13)
    else:
        g.step(dts[0])
    got, ref = interior(g.download(), p), interior(o.state(), p)
    g.close()
    if precision == mcf.PREC_FP64:
        errs = rel_linf(got, ref)
        assert worst(errs) <= 1e-12, errs
    else:
        for f in range(8):
            assert np.abs(got[f] - ref[f]).max() <= 1e-5 * np.abs(ref[f]).max(), f


@pytest.mark.parametrize("precision", [mcf.PREC_FP64, mcf.PREC_MIXED])
@pytest.mark.parametrize("n,nsplit,periodic", [
    ((12, 8, 9), (1, 1, 1), False),     # one-cell segments, fewer columns than a workgroup takes
    ((33, 17, 23), (1, 1, 1), True),    # odd sides, unequal halves
    ((66, 18, 40), (3, 2, 4), False),   # rows of 64 + 2 cells; blocks of 9 and 10 cells
    ((130, 65, 31), (5, 5, 1), True),   # the last segment shorter than the others
    ((61, 122, 10), (1, 2, 2), False),  # x rows of exactly one CT tile; blocks of 5 cells along z
])
def test_step_shapes_vs_oracle(n, nsplit, periodic, precision):
    p = box(*n, periodic)
    print("shape", n, nsplit, precision, flush=True)
    check_step(p, ics.random_state(p, seed=sum(n)), nsplit, precision)


@pytest.mark.parametrize("precision", [mcf.PREC_FP64, mcf.PREC_MIXED])
@pytest.mark.parametrize("value", [np.nan, -np.nan, np.inf])
@pytest.mark.parametrize("field", [0, 1, 6])
def test_non_finite_cell_stays_visible(field, value, precision):
    """A blown-up cell does not turn into plausible numbers: with a NaN or an
    infinity in rho, v_x or B_y of one cell, that cell and its neighbours
    along each axis hold one after a step."""
    p = box(24, 20, 16, True)
    st = ics.random_state(p, seed=5)
    k, j, i = 9, 11, 13
    st[field, k, j, i] = value
    g = mcf.Domain(p, nsplit=(2, 2, 2), precision=precision)
    g.upload(st)
    g.step(1.0e-4)
    got = g.download()
    g.close()
    for dk, dj, di in ((0, 0, 0), (0, 0, 1), (0, 0, -1), (0, 1, 0), (0, -1, 0), (1, 0, 0), (-1, 0, 0)):
        assert not np.isfinite(got[:, k + dk, j + dj, i + di]).all(), (dk, dj, di)


def test_sweep_of_a_flat_box():
    """4104 x 8 x 4100 cells: 65729 workgroups of columns along y, more than
    the y axis of a launch grid takes (65536).  The sweep is launched on the
    zero state and has to come to its end without an error; the shapes above
    hold its values."""
    d = mcf.Domain(box(4104, 8, 4100, True), nsplit=(1, 1, 1))
    print("flat box allocated", flush=True)
    d.sweep(1, 1.0e-3)
    d.sync()
    d.close()


@pytest.mark.parametrize("n,nsplit", [
    (16, (1, 2, 2)),   # all levels but the finest in one workgroup
    (16, (1, 4, 4)),   # the coarsest split level is the highest that one takes
    (64, (4, 1, 2)),   # its sweeps: blocks of 2 x 8 x 4 and 4 x 16 x 8 cells, a barrier per plane at 16 x 8
    (64, (4, 4, 4)),   # 1024 columns of blocks, two whole-domain levels below
    (128, (8, 2, 1)),  # two columns of blocks per thread, a barrier per plane
])
def test_gravity_small_levels_vs_oracle(n, nsplit):
    check_gravity(n, nsplit)


@pytest.mark.parametrize("n,nsplit", [
    (32, (2, 4, 1)),   # blocks of 17 x 9 x 33 nodes: in LDS and streamed, unequal axes
    (32, (1, 1, 2)),   # one block along x and y: a block is its own neighbour
    (64, (1, 2, 2)),   # 65 x 33 x 33 nodes: four columns per thread
    (64, (2, 8, 1)),   # 33 x 9 x 65 nodes, three whole-domain levels
])
def test_gravity_blocks_vs_oracle(n, nsplit):
    """Self-gravity on block shapes that take each relaxation kernel: state and
    Phi after a step, at 1e-12, then Phi of a second solve of the same
    density, bit for bit (a solve starts from the same potential whatever the
    previous one left)."""
    check_gravity(n, nsplit)


@pytest.mark.parametrize("n", [16, 32, 64, 128])
def test_gravity_unsplit_vs_oracle(n):
    """One block: mglin's V-cycles end at level 2, above the coarsest split
    level (level 1), and every y and z ghost is the block's own.  The finest
    levels take the four relaxation kernels in turn (17, 33, 65 and 129 nodes
    a side).  The reference's fixtures have 8 and 16 ranks: parity with its
    build on one block is unpinned, the oracle's schedule is the measure."""
    check_gravity(n, (1, 1, 1))


def check_gravity(n, nsplit):
    p = box(n, n, n, False)
    p.ifgrv = 2
    st = ics.random_state(p, seed=n + sum(nsplit))
    o = oracle.Oracle(p, st, nsplit=nsplit)
    g = mcf.Domain(p, nsplit=nsplit)
    g.upload(st)
    print("gravity", n, nsplit, flush=True)
    dts, _ = o.run(1)
    np.testing.assert_allclose(g.run(1), dts, rtol=1e-13)
    errs = rel_linf(interior(g.download(), p), interior(o.state(), p))
    assert worst(errs) <= 1e-12, errs
    a, b = g.phi(), o.phi()
    assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max()
    g.gravty(0.0, 2)
    c = g.phi()
    g.gravty(0.0, 2)
    np.testing.assert_array_equal(g.phi(), c)
    g.close()


def test_cool_solve_batch_sizes():
    """The stiff-cell solve on batches that end inside a wave, a block and a
    block's share of cells: every cell's result and fallback flag are those of
    the whole batch, bit for bit, in both modes (a cell's solve does not depend
    on its place)."""
    d = mcf.Domain(ics.converging_flow_input(16), nsplit=(1, 1, 1))
    d.mlp_set_weights(surrogate.load_weights())
    args = surrogate.stiff_batch(300001, 77)
    for mode in (0, 1):
        P, fl, _ = d.cool_solve(*args, mode)
        for n in (1, 63, 257, 2048, 2049, 131073):
            p, f, _ = d.cool_solve(*[a[:n] for a in args], mode)
            np.testing.assert_array_equal(p, P[:n])
            np.testing.assert_array_equal(f, fl[:n])
    d.close()


def test_cool_solve_full_blocks():
    """A batch past two full shares a compute unit (2048 cells a block, the
    last block one cell), in both modes: results and flags as in its prefixes.
    Then a network whose prediction overflows: every cell of every block is
    rejected, the reject lists are full, and the fallback's results are mode
    0's, bit for bit."""
    n = (1 << 20) + 2049
    d = mcf.Domain(ics.converging_flow_input(16), nsplit=(1, 1, 1))
    d.mlp_set_weights(surrogate.load_weights())
    args = surrogate.stiff_batch(n, 78)
    imc = None
    for mode in (0, 1):
        P, fl, _ = d.cool_solve(*args, mode)
        imc = P if mode == 0 else imc
        for m in (1 << 20, 2049):
            p, f, _ = d.cool_solve(*[a[:m] for a in args], mode)
            np.testing.assert_array_equal(p, P[:m])
            np.testing.assert_array_equal(f, fl[:m])
            p, f, _ = d.cool_solve(*[a[n - m:] for a in args], mode)
            np.testing.assert_array_equal(p, P[n - m:])
            np.testing.assert_array_equal(f, fl[n - m:])
    w = np.zeros(mcf.MLP_NPARAM, np.float32)
    w[-1] = 1.0e30  # the output's bias
    d.mlp_set_weights(w)
    P, fl, _ = d.cool_solve(*args, 1)
    d.close()
    assert fl.all()
    np.testing.assert_array_equal(P, imc)
