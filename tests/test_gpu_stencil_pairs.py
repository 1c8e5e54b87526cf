"""Where the stencil kernels put two rows of 32 cells into a wavefront: grids on
both sides of the rule, forward and backward kernels apart, against the oracle
bit for bit, and the time of a grid whose strips of rows pair up badly."""
import time

import numpy as np
import pytest
import torch

from util import oracle_run

pytestmark = pytest.mark.gpu


def _workload(n, npml, ny, nt):
    from efwi import synth
    w = synth.small(n=n - 2 * npml, npml=npml, nt=nt, ny=ny - 2 * npml)
    assert w.grid.shape == (n, n, ny)
    return w


# 7 rows per strip and a C-PML edge inside a pair: the forward kernels take two rows, the backward ones one; 12 rows and
# an edge inside a pair of both outer strips: both take two; 7 rows of 3 segments: both take one
@pytest.mark.parametrize("n,npml,ny", [(60, 10, 84), (100, 9, 84), (60, 10, 148)])
def test_pairs_of_rows(orc, n, npml, ny):
    from efwi.propagator import Propagator
    w = _workload(n, npml, ny, 24)
    print(f"[gpu] pairs of rows on {w.grid.shape}, C-PML {npml}", flush=True)
    obs = [s.astype(np.float32) for s in oracle_run(orc, w, model=w.true, calc_id=2).syn]
    ref = oracle_run(orc, w, model=w.model, obs=obs, calc_id=1)
    with Propagator(w.grid) as P:
        P.set_model(*(torch.from_numpy(a) for a in w.model))
        P.zero_gradient()
        _, syn, _ = P.run_shot(w.shots[0], 1, torch.from_numpy(obs[0]), want_syn=True)
        single = [g.cpu().numpy() for g in P.gradient()]
        _, syns = P.run_batch(w.shots * 2, 1, [torch.from_numpy(obs[0])] * 2, want_syn=True)
        batch = [g.cpu().numpy() for g in P.batch_gradient(1)]
    for s in (syn, syns[1]):
        assert np.array_equal(s.cpu().numpy(), ref.syn[0].astype(np.float32))
    for a, c, b in zip(single, batch, (ref.glam, ref.gmu, ref.grho)):
        assert np.abs(b).max() > 0
        assert np.array_equal(a, b.astype(np.float32)) and np.array_equal(c, b.astype(np.float32))


# 128 x 128 rows of two segments are 128 wavefronts per CU: receivers in both velocity kernels; one row more: in the
# forward one; 128 x 256 rows: as many as there; one more: gather and scatter launches
@pytest.mark.parametrize("nx", [132, 133, 260, 261])
def test_receivers_on_both_sides_of_the_limits(orc, nx):
    from efwi import synth
    from efwi.propagator import GridSpec, Propagator, ShotSpec
    g = GridSpec(132, nx, 68, 8, 12, 10.0, 10.0, 10.0, 1e-3, 15.0, 0)
    vp = np.linspace(2000.0, 3000.0, 132, dtype=np.float32)[:, None, None] * np.ones(g.shape, np.float32)
    model = synth.lame(vp, vp / 1.73, 310.0 * vp ** 0.25)
    rec = np.array([(13, nx // 2 + x, 34 + y) for x in (-2, 0, 1) for y in (-30, -1, 0, 29)] + [(13, nx // 2, 34)], np.int32)
    shot = ShotSpec((12, nx // 2, 34), synth.ricker_integrated(15.0, g.nt, 1e-3).astype(np.float32), rec)
    w = synth.Workload("limit", g, [shot], model, model, vp)
    obs = np.random.default_rng(nx).standard_normal((3, len(rec), g.nt)).astype(np.float32)
    print(f"[gpu] receivers on {g.shape}", flush=True)
    with Propagator(g) as P:
        P.set_model(*(torch.from_numpy(a) for a in model))
        P.zero_gradient()
        _, syn, res = P.run_shot(shot, 1, torch.from_numpy(obs), want_syn=True, want_res=True)
        got = [t.cpu().numpy() for t in (syn, res, *P.gradient())]
    ref = oracle_run(orc, w, obs=[obs], calc_id=1)
    for a, b in zip(got, (ref.syn[0], ref.res[0], ref.glam, ref.gmu, ref.grho)):
        assert np.abs(b).max() > 0
        assert np.array_equal(a, b.astype(np.float32))


def test_fewer_rows_take_no_longer():
    """A gradient on 60 x 60 x 148 cells (7 rows per strip) takes about the time
    of 60 x 68 x 148 (8 rows, four full pairs); with half-filled pairs and
    pairs across the C-PML's edge it took 1.14 times as long."""
    from contextlib import ExitStack
    from efwi import synth
    from efwi.propagator import GridSpec, Propagator, ShotSpec
    with ExitStack() as stack:
        runs = {}
        for nx in (60, 68):
            g = GridSpec(60, nx, 148, 10, 200, 10.0, 10.0, 10.0, 1e-3, 15.0, 0)
            vp = np.full(g.shape, 2500.0, np.float32)
            stf = synth.ricker_integrated(15.0, g.nt, 1e-3).astype(np.float32)
            shot = ShotSpec((15, nx // 2, 74), stf, np.array([[13, x, 74] for x in range(12, nx - 12)], np.int32))
            P = stack.enter_context(Propagator(g))
            P.set_model(*(torch.from_numpy(a) for a in synth.lame(vp, vp / 1.73, 310.0 * vp ** 0.25)))
            runs[nx] = (P, shot, torch.zeros(3, len(shot.rec), g.nt), [])
        for _ in range(12):
            for P, shot, obs, times in runs.values():
                torch.cuda.synchronize()
                t = time.perf_counter()
                P.run_shot(shot, 1, obs)
                torch.cuda.synchronize()
                times.append(time.perf_counter() - t)
        ms = {nx: min(r[3]) * 1e3 for nx, r in runs.items()}
    print(f"[gpu] gradient on 60x60x148 {ms[60]:.1f} ms, on 60x68x148 {ms[68]:.1f}", flush=True)
    assert ms[60] < 1.07 * ms[68]


@pytest.mark.parametrize("ny,depth", [(61 * 64, 2), (60 * 64, 1)])
def test_backward_shapes_of_large_grids(orc, ny, depth):
    """On both sides of the rule for two z planes per workgroup: the default
    shape and the other one give the oracle's gradient."""
    from efwi.propagator import Propagator
    w = _workload(37, 4, ny, 16)
    z, x, y = w.shots[0].src
    w.shots[0].rec = np.array([(z + 1, x, y), (z + 2, x + 1, y - 2)], np.int32)
    obs = np.random.default_rng(1).standard_normal((3, 2, w.grid.nt)).astype(np.float32)
    print(f"[gpu] backward shapes on {w.grid.shape}", flush=True)
    ref = oracle_run(orc, w, obs=[obs], calc_id=1)
    for other in (False, True):
        with Propagator(w.grid) as P:
            P.set_model(*(torch.from_numpy(a) for a in w.model))
            for k in ("velocity_bwd", "stress_bwd"):
                assert P.tiles()[k] == (1, depth)
                if other:
                    P.set_tile(k, 1, 3 - depth)
            P.run_shot(w.shots[0], 1, torch.from_numpy(obs))
            got = [t.cpu().numpy() for t in P.gradient()]
        for a, b in zip(got, (ref.glam, ref.gmu, ref.grho)):
            assert np.abs(b).max() > 0
            assert np.array_equal(a, b.astype(np.float32))


def test_marching_backward_kernels_are_alike():
    """The marching backward kernels read and write about the same number of
    fields: velocity_bwd in {4, 16} takes 1.1 times stress_bwd's time (with a
    variant per set of C-PML axes it took 1.75 times)."""
    from efwi.propagator import Propagator
    w = _workload(84, 10, 84, 60)
    obs = torch.zeros(3, len(w.shots[0].rec), w.grid.nt)
    with Propagator(w.grid) as P:
        P.set_model(*(torch.from_numpy(a) for a in w.model))
        for k in ("velocity_bwd", "stress_bwd"):
            P.set_tile(k, 4, 16)
        P.run_shot(w.shots[0], 1, obs)
        P.profile(True)
        P.profile_read(reset=True)
        P.run_shot(w.shots[0], 1, obs)
        us = {k: ms / n * 1e3 for k, (ms, n) in P.profile_read(reset=True).items() if n}
    print(f"[gpu] marching velocity_bwd {us['velocity_bwd']:.1f} us, stress_bwd {us['stress_bwd']:.1f}", flush=True)
    assert us["velocity_bwd"] < 1.4 * us["stress_bwd"]


def test_scattered_receivers_of_a_short_run(orc):
    """8000 receivers all over the grid for 19 steps: their tables would cost
    more than the launches they save (1.17 times the time of the same receivers
    and one on the outermost cells, which sends them to the launches anyway);
    seismograms are the oracle's."""
    from efwi import synth
    from efwi.propagator import GridSpec, Propagator, ShotSpec
    g = GridSpec(60, 60, 300, 8, 20, 10.0, 10.0, 10.0, 1e-3, 15.0, 0)
    vp = np.full(g.shape, 2500.0, np.float32)
    model = synth.lame(vp, vp / 1.73, 310.0 * vp ** 0.25)
    rng = np.random.default_rng(0)
    rec = np.stack([rng.integers(2, n - 2, 8000) for n in g.shape], 1).astype(np.int32)
    rec[:50] = [30, 30, 150] + rng.integers(-4, 5, (50, 3))  # near the source
    stf = synth.ricker_integrated(15.0, g.nt, 1e-3).astype(np.float32)
    shot = ShotSpec((30, 30, 150), stf, rec)
    outer = ShotSpec((30, 30, 150), stf, np.concatenate([rec, [[0, 0, 0]]]).astype(np.int32))
    print(f"[gpu] scattered receivers on {g.shape}", flush=True)
    with Propagator(g) as P:
        P.set_model(*(torch.from_numpy(a) for a in model))
        times = {}
        for _ in range(15):
            for name, s in (("inside", shot), ("outer", outer)):
                torch.cuda.synchronize()
                t = time.perf_counter()
                _, syn, _ = P.run_shot(s, 2)
                torch.cuda.synchronize()
                times.setdefault(name, []).append(time.perf_counter() - t)
                if name == "inside":
                    got = syn.cpu().numpy()
    ref = oracle_run(orc, synth.Workload("scattered", g, [shot], model, model, vp), calc_id=2).syn[0]
    assert np.abs(ref).max() > 0 and np.array_equal(got, ref.astype(np.float32))
    print(f"[gpu] {min(times['inside']) * 1e3:.2f} ms, {min(times['outer']) * 1e3:.2f} with one outside", flush=True)
    assert min(times["inside"]) < 1.08 * min(times["outer"])
