"""GPU tests of the batch engine's blocks of planned steps and of the kernels it chooses per class: every instance's state
bitwise the same as its own run, whatever shares its launches."""
import pytest
import torch

from pfkit import PFSolver, workloads
from pfkit._lib import PFError
from pfkit.allen_cahn import DTYPES
from pfkit.batch import BatchEngine
from pfkit.laser import RosenthalRamp

pytestmark = pytest.mark.gpu


def _solo(w, steps):
    s = PFSolver(w.pf_args, w.polycrystal, dtype=w.dtype, clean=False, tile=-2, zchunk=0)
    return s.run(s.ini_cond(), w.ts(steps), w.laser)


def _make(j, nx, ny, nz, k, dtype, steps, aniso=0.15):
    return workloads.make(f"b{j}", nx, ny, nz, k, 10, steps, dtype, aniso, seed=80 + j, vel=2.0)


@pytest.mark.parametrize("chunk", [0, 1, 5, 8, 11, 16, 20])
def test_step_counts_within_and_across_blocks(cuda, chunk):
    steps = (0, 1, 7, 8, 9, 17, 24)
    W = [_make(j, 18 + j, 11, 9, 6, "float32", n) for j, n in enumerate(steps)]
    eng = BatchEngine(max_instances=8)
    slots = [eng.add(w.instance()) for w in W]
    eng.run(25, chunk)
    left, t, parity = eng.status()
    for w, s, n in zip(W, slots, steps):
        assert left[s] == 0 and t[s] == n * w.dt
        assert torch.equal(eng.state(s, parity[s]), _solo(w, n))
    eng.close()


@pytest.mark.parametrize("dtype,k", [("float32", 10), ("bfloat16", 12), ("float64", 13), ("float32", 27)])
def test_a_class_changes_its_kernel_as_instances_come_and_go(cuda, dtype, k):
    """One small instance runs on channel groups; with large ones in its class on tiles of one, two or three
    fillings and then as asked; alone again, on channel groups: graphs of each are cached."""
    small = _make(0, 24, 20, 13, k, dtype, 40)
    big = [_make(1 + j, 130, 128, 40, k, dtype, 8) for j in range(4)]
    eng = BatchEngine(max_instances=8)
    s0 = eng.add(small.instance())
    done = 0
    for n in (0, 1, 2, 4, 0, 1):
        slots = [eng.add(w.instance()) for w in big[:n]]
        eng.run(6, 6)
        done += 6
        par = eng.status()[2]
        assert torch.equal(eng.state(s0, par[s0]), _solo(small, done))
        for w, s in zip(big, slots):
            assert torch.equal(eng.state(s, par[s]), _solo(w, 6))
            eng.remove(s)
    eng.close()


@pytest.mark.parametrize("ks,dtype,chunk", [((6, 9, 12, 27, 16), "float32", 8), ((6, 9, 12, 27, 16), "bfloat16", 3),
                                            ((10, 13), "float64", 12), ((20,), "float32", 4), ((20,), "float32", 3),
                                            ((20,), "bfloat16", 16), ((16,), "float64", 5)])
def test_classes_and_parts_that_run_side_by_side(cuda, ks, dtype, chunk):
    """More classes than branches, fewer, and a lone class large enough to be split (four instances of uneven size,
    then two, then one): replays with eager steps and host reads between, each instance bitwise its own run."""
    if len(ks) > 1:
        W = [_make(j, 30 + 3 * j, 26, 12, k, dtype, 80) for j, k in enumerate(ks + ks[:2])]
    else:
        W = [_make(j, 96 + 8 * j, 90, 25, ks[0], dtype, 80) for j in range(4)]
    eng = BatchEngine(max_instances=8)
    slots = [eng.add(w.instance()) for w in W]
    done = 0
    for rest in (1, 0, 2):
        eng.run(2 * chunk + rest, chunk)
        done += 2 * chunk + rest
        par = eng.status()[2]
        for w, s in zip(W, slots):
            assert torch.equal(eng.state(s, par[s]), _solo(w, min(done, 80)))
        if rest < 1 or len(ks) == 1:
            for s in slots[len(slots) // 2:]:
                eng.remove(s)
            slots = slots[:len(slots) // 2]
    eng.close()


def _quad_items(dims, k, v=4):
    """Work items of instances of one class on the march of channel groups, as rebuild_work counts them."""
    up = lambda a, b: -(-a // b)  # noqa: E731
    c = 256 // up(k, v)
    runs = [up(up(nx * ny, c), 8) * 8 for nx, ny, _ in dims]
    chunks = max(1, 1024 // sum(runs))
    return sum(r * up(nz, min(up(nz, chunks), 512 // c)) for r, (_, _, nz) in zip(runs, dims))


def test_more_work_items_than_max_tiles(cuda):
    """Slots are charged as they asked to be tiled; shorter marches and channel groups make more work items than that.
    The list of a tiny instance fits and a graph that holds it has run; with two more of the class (the same graph
    key) it grows past max_tiles, and the next replay must not read the old one."""
    dims, k = [(6, 6, 4), (33, 31, 24), (33, 31, 24)], 25
    W = [_make(j, *d, k, "float32", 20) for j, d in enumerate(dims)]
    charge = sum(-(-nx * ny * nz // 256) for nx, ny, nz in dims)
    assert _quad_items(dims[:1], k) <= charge < _quad_items(dims, k)
    eng = BatchEngine(max_instances=4, max_tiles=charge)
    slots = [eng.add(W[0].instance())]
    eng.run(4, 4)
    slots += [eng.add(w.instance()) for w in W[1:]]
    for n in (4, 8):
        eng.run(4, 4)
        par = eng.status()[2]
        for w, s, done in zip(W, slots, (4 + n, n, n)):
            assert torch.equal(eng.state(s, par[s]), _solo(w, done))
    with pytest.raises(PFError, match="max_tiles"):
        eng.add(_make(9, 33, 31, 24, k, "float32", 20).instance())
    eng.close()


@pytest.mark.parametrize("chunk", [3, 16])
def test_source_tables_are_planned_per_step(cuda, chunk):
    """Two instances of one class with source tables of their own and one without, over steps that end within a
    block: each bitwise its own run_toolpath or run."""
    W = [_make(j, 26, 18, 10, 8, "float32", 19) for j in range(3)]
    n, dt = 19, W[0].dt
    ramps = [RosenthalRamp(x0=5.0, y0=9.0, z0=10.0, t_OFF=30 * dt * (1 + 0.1 * j), dt=dt * (1 + 0.1 * j),
                           vel_avg=0.3 / dt, Q_max=2.0e6, Q_min=0.5e6, alpha=5.2) for j in range(2)]
    eng = BatchEngine(max_instances=4)
    slots = []
    for w, r in zip(W, ramps):
        inst = w.instance(toolpath=r)
        slots.append(eng.add(inst))
    slots.append(eng.add(W[2].instance()))
    eng.run(n, chunk)
    left, t, par = eng.status()
    for j, (w, s) in enumerate(zip(W, slots)):
        if j < 2:
            sol = PFSolver(w.pf_args, w.polycrystal, dtype="float32", clean=False)
            want = sol.run_toolpath(sol.ini_cond(), ramps[j], steps=n)
            assert t[s] == ramps[j].step_times()[n]
        else:
            want = _solo(w, n)
        assert left[s] == 0 and torch.equal(eng.state(s, par[s]), want)
    eng.close()


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("side", [False, True])
def test_admission_while_steps_are_queued_takes_the_state_of_its_call(cuda, dtype, side):
    """One buffer refilled in place for each of several requests, admitted behind a long queue of steps: every instance
    starts from what the buffer held at its own add.  The first state is there for the caller's next reads."""
    busy = _make(0, 128, 128, 64, 20, "float32", 300)
    W = [_make(1 + j, 40, 31, 17, 6, dtype, 3) for j in range(4)]
    eng = BatchEngine(max_instances=16)
    eng.add(busy.instance())
    eng.run(16, 16)
    caller = torch.cuda.Stream() if side else torch.cuda.current_stream()
    states = [torch.rand(w.N, w.K, device=cuda, generator=torch.Generator(cuda).manual_seed(j)).to(DTYPES[dtype])
              for j, w in enumerate(W)]
    oris = [torch.as_tensor(w.polycrystal.cell_ori_inds, device=cuda, dtype=torch.int32) for w in W]
    eta0, ori = torch.empty_like(states[0]), torch.empty_like(oris[0])
    caller.wait_stream(torch.cuda.current_stream())
    got, first = [], []
    with torch.cuda.stream(caller):
        for w, state, o in zip(W, states, oris):
            eng.run(32, 16)
            eta0.copy_(state)
            ori.copy_(o)
            for kw in (dict(eta0=eta0), dict()):
                inst = w.instance(**kw)
                if not kw:
                    inst.cell_ori_inds = ori
                got.append(eng.add(inst))
                first.append(eng.state(got[-1], 0).clone())
            eta0.fill_(float("nan"))
            ori.fill_(0)
    torch.cuda.current_stream().wait_stream(caller)
    eng.run_to_completion()
    par = eng.status()[2]
    for j, w in enumerate(W):
        s = PFSolver(w.pf_args, w.polycrystal, dtype=w.dtype, clean=False, tile=-2, zchunk=0)
        for slot, start, e in zip(got[2 * j:], first[2 * j:], (states[j], s.ini_cond())):
            assert torch.equal(start, e)
            assert torch.equal(eng.state(slot, par[slot]), s.run(e, w.ts(3), w.laser))
    eng.close()
