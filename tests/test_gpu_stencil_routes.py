"""The launch rules of the stencil kernels at the sizes where they change:
each route against the oracle, bit for bit (no tolerance: the kernels evaluate
the oracle's float expressions in its order)."""
import numpy as np
import pytest
import torch

from util import oracle_run

pytestmark = pytest.mark.gpu


def _gradient(w, obs, prepare=None):
    """(syn, res, gradients) of every shot's run through one propagator."""
    from efwi.propagator import Propagator
    print(f"[gpu] grid={w.grid.shape} nt={w.grid.nt} form={w.grid.formulation} npml={w.grid.npml}", flush=True)
    with Propagator(w.grid) as P:
        if prepare:
            prepare(P)
        P.set_model(*(torch.from_numpy(a) for a in w.model))
        P.zero_gradient()
        syns, ress = [], []
        for s, o in zip(w.shots, obs):
            _, syn, res = P.run_shot(s, 1, torch.from_numpy(o), want_syn=True, want_res=True)
            syns.append(syn.cpu().numpy())
            ress.append(res.cpu().numpy())
        return syns, ress, [g.cpu().numpy() for g in P.gradient()]


def _check(orc, w, prepare=None):
    obs = [s.astype(np.float32) for s in oracle_run(orc, w, model=w.true, calc_id=2).syn]
    syns, ress, grads = _gradient(w, obs, prepare)
    ref = oracle_run(orc, w, model=w.model, obs=obs, calc_id=1)
    for k in range(len(w.shots)):
        assert np.array_equal(syns[k], ref.syn[k].astype(np.float32))
        assert np.array_equal(ress[k], ref.res[k].astype(np.float32))
    for a, b in zip(grads, (ref.glam, ref.gmu, ref.grho)):
        assert np.abs(b).max() > 0
        assert np.array_equal(a, b.astype(np.float32))


# padded y sizes: one 32-cell segment (2..31), a last segment of 4 cells, one
# of 18, and one whole; 65 rows over 8 strips leave an odd row in every strip
@pytest.mark.parametrize("ny,formulation", [(34, 0), (70, 1), (84, 0), (98, 0)])
def test_two_rows_per_wavefront(orc, ny, formulation):
    """Grids whose rows waste lanes of 64-cell segments run 32 lanes on each of
    two rows per wavefront; rows of both halves differ in their C-PML slabs."""
    from efwi import synth
    npml = 6
    w = synth.small(n=69 - 2 * npml, npml=npml, nt=24, ny=ny - 2 * npml, formulation=formulation)
    assert w.grid.shape == (69, 69, ny)
    _check(orc, w)


def test_folded_receivers(orc):
    """Receivers in the velocity kernels: several in one cell, in the C-PML, on
    the first and last cells of the stencil box, at 64-cell segment edges."""
    from efwi import synth
    w = synth.small(n=24, npml=6, nt=60, ny=68)
    nz, nx, ny = w.grid.shape
    assert ny == 80
    rec = [(8, 8, y) for y in (2, 5, 31, 32, 63, 64, ny - 3)] + [(2, 2, 2), (nz - 3, nx - 3, ny - 3), (2, nx - 3, 40)]
    rec += [(9, 10, 40)] * 3 + [(8, 8, 63)]
    w.shots[0].rec = np.array(rec, np.int32)
    _check(orc, w)


def test_receivers_outside_the_stencil_box(orc):
    """One receiver on the outermost cells sends the shot's receivers to the gather and scatter launches."""
    from efwi import synth
    w = synth.small(n=24, npml=6, nt=60)
    nz, nx, ny = w.grid.shape
    w.shots[0].rec = np.array([(8, 8, 8), (10, 12, 20), (1, 8, 8), (8, nx - 2, 8), (8, 8, ny - 1)], np.int32)
    _check(orc, w)


@pytest.mark.parametrize("nt", [18, 33, 40])
def test_batch_steps_replayed_and_launched(nt):
    """A batch replays captured graphs of sixteen time steps and launches the
    rest directly: nt - 1 = one graph and one step, two graphs, two graphs and
    seven steps, on narrow rows (two per wavefront); equal to single shots."""
    from efwi import synth
    from efwi.propagator import Propagator, ShotSpec
    w = synth.small(n=69 - 12, npml=6, nt=nt, ny=70 - 12)
    base = w.shots[0]
    rec = np.array([[9, 20, 30], [9, 20, 30], [10, 2, 2]], np.int32)
    shots = [base, ShotSpec((12, 30, 40), base.stf, rec), ShotSpec((20, 10, 12), base.stf, rec[:1])]
    print(f"[gpu] batch grid={w.grid.shape} nt={nt}", flush=True)
    with Propagator(w.grid) as P:
        P.set_model(*(torch.from_numpy(a) for a in w.true))
        obs = [P.run_shot(s, 2)[1] for s in shots]
        P.set_model(*(torch.from_numpy(a) for a in w.model))
        mis, syns = P.run_batch(shots, 1, obs, want_syn=True)
        grads = [P.batch_gradient(k) for k in range(len(shots))]
        again, _ = P.run_batch(shots, 1, obs)
        for k, s in enumerate(shots):
            P.zero_gradient()
            j, syn, _ = P.run_shot(s, 1, obs[k], want_syn=True)
            assert mis[k] == j and again[k] == j
            assert torch.equal(syns[k], syn)
            for a, b, c in zip(grads[k], P.gradient(), P.batch_gradient(k)):
                assert torch.equal(a, b) and torch.equal(c, b)


@pytest.mark.parametrize("ny,depth", [(61 * 64, 2), (60 * 64, 1)])
def test_backward_shape_of_large_grids(ny, depth):
    """From 256 wavefronts per CU on, the backward kernels take two z planes per
    workgroup (an odd number of planes here); results are those of one."""
    from efwi import synth
    npml = 4
    w = synth.small(n=37 - 2 * npml, npml=npml, nt=40, ny=ny - 2 * npml)
    nz, nx, _ = w.grid.shape
    z, x, y = w.shots[0].src
    w.shots[0].rec = np.array([(z + 1, x, y), (z + 2, x + 1, y - 2)], np.int32)
    assert ((nz - 4) * (nx - 4) * ((ny - 3) // 64 + 1) >= 65536) == (depth == 2)
    shapes = []

    def one_plane(P):
        for k in ("velocity_bwd", "stress_bwd"):
            shapes.append(P.tiles()[k])
            P.set_tile(k, 1, 1)

    rng = np.random.default_rng(1)
    obs = [rng.standard_normal((3, len(s.rec), w.grid.nt)).astype(np.float32) for s in w.shots]
    a = _gradient(w, obs)
    b = _gradient(w, obs, one_plane)
    assert shapes == [(1, depth)] * 2
    for x, y in zip(a[2], b[2]):
        assert np.abs(x).max() > 0 and np.array_equal(x, y)
