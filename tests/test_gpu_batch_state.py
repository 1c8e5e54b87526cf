"""What a context keeps from one batch to the next (shot table, captured graphs,
boundary rings, launch settings): a batch gives the results of the same shots
run one by one whatever batches ran before it."""
import time

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _workload(nt, n=24, npml=6):
    from efwi import synth
    return synth.small(n=n, npml=npml, nt=nt)


def _shots(w, count, seed, nrec=5):
    """Shots with seeded sources and receivers inside the stencil box."""
    from efwi.propagator import ShotSpec
    rng = np.random.default_rng(seed)
    (nz, nx, ny), p, stf = w.grid.shape, w.grid.npml, w.shots[0].stf
    inner = lambda: tuple(int(rng.integers(p, n - p)) for n in (nz, nx, ny))  # noqa: E731
    box = lambda: [int(rng.integers(2, n - 2)) for n in (nz, nx, ny)]  # noqa: E731
    return [ShotSpec(inner(), stf, np.array([box() for _ in range(nrec)], np.int32)) for _ in range(count)]


def _obs(w, shots, seed):
    rng = np.random.default_rng(seed)
    return [torch.from_numpy(rng.standard_normal((3, len(s.rec), w.grid.nt)).astype(np.float32)) for s in shots]


def _open(w):
    from efwi.propagator import Propagator
    P = Propagator(w.grid)
    P.set_model(*(torch.from_numpy(a) for a in w.model))
    return P


def _check(w, shots, obs, misfits, syns, grads):
    with _open(w) as P:
        for k, s in enumerate(shots):
            P.zero_gradient()
            j, syn, _ = P.run_shot(s, 1, obs[k], want_syn=True)
            assert misfits[k] == j, k
            assert torch.equal(syns[k], syn), k
            for a, b in zip(grads[k], P.gradient()):
                assert b.abs().max() > 0
                assert torch.equal(a, b), k


@pytest.mark.parametrize("use_graph", [True, False])
def test_batch_after_a_larger_one(use_graph):
    """A batch between two others of one size makes the shot table grow: the
    second of them replays no graph of the first one's table."""
    w = _workload(40)
    first, larger, then = _shots(w, 2, 1), _shots(w, 5, 2), _shots(w, 2, 3)
    o1, o2 = _obs(w, first, 4), _obs(w, then, 5)
    print(f"[gpu] batch of 2, of 5 (graph={use_graph}), of 2 on {w.grid.shape}", flush=True)
    with _open(w) as P:
        P.run_batch(first, 1, o1)
        P.run_batch(larger, 2, use_graph=use_graph)
        misfits, syns = P.run_batch(then, 1, o2, want_syn=True)
        grads = [P.batch_gradient(k) for k in range(2)]
        _check(w, then, o2, misfits, syns, grads)


def test_rings_of_a_batch_are_bounded():
    """Shots whose boundary rings are large (11 GB each here) do not each get
    one in the automatic mode: after a batch the context holds less than one
    ring more than after a single shot."""
    w = _workload(4000, n=52, npml=10)
    shots = _shots(w, 3, 6)
    obs = _obs(w, shots, 7)
    print(f"[gpu] rings of a batch of 3 on {w.grid.shape}, nt={w.grid.nt}", flush=True)
    with _open(w) as P:
        before = P.device_bytes
        P.run_shot(shots[0], 1, obs[0])
        after_shot = P.device_bytes
        misfits, _ = P.run_batch(shots, 1, obs)
        assert P.device_bytes - after_shot < after_shot - before
        assert misfits == [P.run_shot(s, 0, o)[0] for s, o in zip(shots, obs)]


def test_batch_config_costs_nothing():
    """Setting the work distribution (its former defaults here) leaves results
    and speed of a batch as they are. Work queues took 1.9 times as long on
    this batch; launches without them repeat within a few percent."""
    w = _workload(120, n=32)
    shots = _shots(w, 12, 8)
    obs = _obs(w, shots, 9)
    print(f"[gpu] 12 shots on {w.grid.shape} with and without batch_config", flush=True)

    ms, misfits = ([], []), [None, None]
    with _open(w) as P, _open(w) as Q:
        Q.batch_config()
        for _ in range(6):
            for k, prop in enumerate((P, Q)):
                torch.cuda.synchronize()
                t = time.perf_counter()
                misfits[k], _ = prop.run_batch(shots, 1, obs)
                ms[k].append((time.perf_counter() - t) * 1e3)
    t, t2 = min(ms[0]), min(ms[1])
    print(f"[gpu] {t:.1f} ms, {t2:.1f} ms after batch_config", flush=True)
    assert misfits[0] == misfits[1] and t2 < 1.4 * t


@pytest.mark.parametrize("use_graph", [True, False])
def test_one_shot_outside_the_stencil_box(use_graph):
    """One shot's receiver on the outermost cells sends the receivers of the
    whole batch to the gather and scatter launches; two replayed graphs of steps
    and seven launched ones, in groups of three and one."""
    w = _workload(40)
    shots = _shots(w, 4, 10)
    nz, nx, ny = w.grid.shape
    shots[1].rec = np.concatenate([shots[1].rec, [[1, 8, 8], [8, nx - 2, 8], [8, 8, ny - 1], [8, 8, ny - 1]]]).astype(np.int32)
    obs = _obs(w, shots, 11)
    print(f"[gpu] batch of 4, one outside the box, graph={use_graph}", flush=True)
    with _open(w) as P:
        P.batch_group(3)
        for _ in range(2):  # the second replays the first one's graphs
            misfits, syns = P.run_batch(shots, 1, obs, want_syn=True, use_graph=use_graph)
        grads = [P.batch_gradient(k) for k in range(4)]
        _check(w, shots, obs, misfits, syns, grads)
        # and the next batch's receivers are in the kernels again
        misfits, syns = P.run_batch(shots[2:4], 1, obs[2:4], want_syn=True, use_graph=use_graph)
        _check(w, shots[2:4], obs[2:4], misfits, syns, [P.batch_gradient(k) for k in range(2)])
