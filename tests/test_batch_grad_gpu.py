"""Batched lower-star .grad (msceer_batch_grad) on the GPU.

One launch per stage for a whole group of volumes, captured in a hipGraph:
every volume's .grad must be the single-volume call's bytes, which the
oracle and the reference goldens pin.  Covered: the goldens (ragged, tied
and two-vertex-thick volumes) under every brick shape and both launch forms
(a work-group per brick; persistent work-groups claiming bricks in chunks);
16 volumes of the 512-volume workload's family (sides 32..160, smoothed
noise and Gaussian mixtures) against the oracle; graph replays with other
GPU work between them, each checked; groups split by a vertex cap; a first
capture with too few flood sweeps, finished eagerly, and the recapture
that follows; more sweeps than a graph holds, and more groups than a context
keeps graphs of."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle_lib
from golden import load_lstar
from msceer_amd import batch, hipmem, lstar, native, synth

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
GOLDEN = ["noise_48x97x31", "ties_10x11x12", "tiny_5x2x3", "smooth_60x50x40"]


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0)
    yield c
    c.close()


def _goldens():
    fs, refs = [], []
    for name in GOLDEN:
        f, ref = load_lstar(name)
        fs.append(np.ascontiguousarray(f, np.float32))
        refs.append(ref)
    return fs, refs


@pytest.mark.parametrize("mode", [0, 1, 2, 3, 4, 5])
def test_goldens_every_shape(ctx, mode):
    """Autotune mode 0 (64x2x2), 1 (measured) and 2 + k (shape k)."""
    fs, refs = _goldens()
    native.check(native.lib().msceer_set_autotune(ctx.handle, mode), "msceer_set_autotune")
    try:
        grads, ms, st = batch.run_batch_grad(fs + fs[::-1], ctx=ctx)
    finally:
        native.lib().msceer_set_autotune(ctx.handle, 1)
    _say(f"mode {mode}: shape {st.shape} blocks {st.blocks} chunk {st.chunk} rounds {st.rounds} "
         f"groups {st.groups} eager {st.eager_rounds}")
    for g, ref in zip(grads, refs + refs[::-1]):
        assert (g == ref).all(), int((g != ref).sum())
    assert st.groups == 1 and st.replays == 1


def _fresh_process(code, env):
    """Run `code` in a new interpreter (the launch form is read from the
    environment when a context first tunes a group)."""
    e = dict(os.environ)
    e.update(env)
    e["PYTHONPATH"] = os.pathsep.join([ROOT, os.path.join(ROOT, "tests"), os.path.join(ROOT, "tests", "golden")])
    r = subprocess.run([sys.executable, "-c", code], env=e, capture_output=True, text=True, timeout=300)
    _say(r.stdout[-2000:])
    assert r.returncode == 0, r.stderr[-4000:]


_PERSISTENT = """
import numpy as np
from golden import load_lstar
from msceer_amd import batch, native
fs, refs = [], []
for name in {golden!r}:
    f, ref = load_lstar(name)
    fs.append(np.ascontiguousarray(f, np.float32)); refs.append(ref)
ctx = native.Context(0)
for rep in range(3):
    grads, ms, st = batch.run_batch_grad(fs * 3, ctx=ctx)
    print("persistent", st.shape, st.blocks, st.chunk, "captures", st.captures, flush=True)
    assert st.blocks > 0
    for g, ref in zip(grads, refs * 3):
        assert (g == ref).all(), int((g != ref).sum())
ctx.close()
"""


@pytest.mark.parametrize("form", ["2:8:1", "0:4:16", "3:2:4"])
def test_persistent_launch_forms(form):
    _fresh_process(_PERSISTENT.format(golden=GOLDEN), {"MSCEER_BATCH_LAUNCH": form})


def _c4_subset():
    """16 volumes of the 512-volume workload spanning its sizes (every 32nd
    by vertex count)."""
    sizes = []
    for i in range(512):
        u = synth.Stream(4000 + i).uniform(5)
        shape = tuple(int(32 + min(128, int(129 * float(u[k])))) for k in range(3))
        sizes.append((shape[0] * shape[1] * shape[2], i))
    sizes.sort()
    return [i for _, i in sizes[::32]]


@pytest.fixture(scope="module")
def c4(ctx):
    ids = _c4_subset()
    vols = [synth.batch_volume(i).astype(np.float32) for i in ids]
    _say(f"c4 subset: {len(vols)} volumes, {sum(v.size for v in vols)} vertices")
    refs = [oracle_lib.steepest_grad(v) for v in vols]
    return ids, vols, refs


def test_c4_subset_against_oracle(ctx, c4):
    ids, vols, refs = c4
    grads, ms, st = batch.run_batch_grad(vols, timing=True, ctx=ctx)
    _say(f"c4 subset: shape {st.shape} blocks {st.blocks} chunk {st.chunk} rounds {st.rounds} "
         f"eager {st.eager_rounds} ms_gpu {st.ms_gpu:.3f} per-volume ms {np.round(ms, 3).tolist()}")
    for i, v, g, ref in zip(ids, vols, grads, refs):
        assert (g == ref).all(), (i, v.shape, int((g != ref).sum()))
    assert (ms > 0).all() and (ms <= st.ms_gpu * 1.5 + 1.0).all()


def test_c4_subset_split_into_groups(ctx, c4):
    ids, vols, refs = c4
    cap = max(v.size for v in vols) + 1
    grads, ms, st = batch.run_batch_grad(vols, max_group_verts=cap, ctx=ctx)
    _say(f"groups {st.groups} with at most {cap} vertices")
    assert st.groups > 2
    for i, g, ref in zip(ids, grads, refs):
        assert (g == ref).all(), i


def test_graph_replays_with_device_buffers(ctx, c4):
    """The same device buffers batched four times; other GPU work (a
    single-volume call, buffer clears) and host synchronisations between the
    replays; every replay checked against the oracle."""
    ids, vols, refs = c4
    vols, refs = vols[:8], refs[:8]
    dv = [hipmem.DeviceBuffer(v.nbytes) for v in vols]
    dg = [hipmem.DeviceBuffer(r.size) for r in refs]
    for d, v in zip(dv, vols):
        d.upload(v)
    arr = batch.volume_table([v.shape for v in vols], [d.addr for d in dv], [d.addr for d in dg])
    other = synth.smoothed_noise((40, 50, 60), 99, 2.0).astype(np.float32)
    other_ref = oracle_lib.steepest_grad(other)
    lib = native.lib()
    for rep in range(4):
        for d in dg:
            d.fill(0xA5)
        hipmem.synchronize()
        native.check(lib.msceer_batch_grad(ctx.handle, arr, len(vols), 0, native.DEVICE_PTRS), "msceer_batch_grad")
        st = native.BatchStats()
        native.check(lib.msceer_last_batch_stats(ctx.handle, ctypes.byref(st)), "msceer_last_batch_stats")
        hipmem.synchronize()
        _say(f"replay {rep}: captures {st.captures} replays {st.replays} eager {st.eager_rounds}")
        if rep > 0:
            assert st.captures == 0 or st.eager_rounds > 0
        for i, (d, ref) in enumerate(zip(dg, refs)):
            g = d.download(np.uint8, ref.size)
            assert (g == ref).all(), (rep, i, int((g != ref).sum()))
        g1 = lstar.steepest_lstar_grad(other, ctx=ctx).ravel()
        assert (g1 == other_ref).all()


def _ridge(nz, seed):
    """A ridge along z between two valleys: the flood of its edges starts at
    one end and takes a sweep per tile of 16 layers."""
    z, y, x = np.meshgrid(np.arange(nz, dtype=np.float64), np.arange(3), np.arange(33), indexing="ij")
    f = -np.cos(2 * np.pi * (x - 16) / 32) + 0.01 * z + 1e-4 * synth.Stream(seed).uniform(x.size).reshape(x.shape)
    f[:, 1] -= 0.5
    return f.astype(np.float32)


def test_group_beyond_the_captured_sweeps_keeps_its_graph(ctx):
    """More sweeps than any graph holds: the rest runs after each replay, and
    the graph is captured again only once, for the limit."""
    f = _ridge(16 * 90, 5)
    ref = oracle_lib.steepest_grad(f)
    captures = []
    for rep in range(4):
        grads, _, st = batch.run_batch_grad([f], ctx=ctx)
        _say(f"ridge call {rep}: sweeps {st.rounds} eager {st.eager_rounds} captures {st.captures}")
        assert (grads[0] == ref).all(), int((grads[0] != ref).sum())
        assert st.eager_rounds > 0
        captures.append(st.captures)
    assert captures == [1, 1, 0, 0], captures


def test_more_groups_than_kept_plans_remember_their_sweeps(ctx):
    """Six groups of one volume each, more than the plans a context keeps:
    every call captures them again, with the sweeps the call before needed."""
    fs = [_ridge(16 * 20 + i, 6 + i) for i in range(6)]
    refs = [oracle_lib.steepest_grad(f) for f in fs]
    eager = []
    for rep in range(3):
        grads, _, st = batch.run_batch_grad(fs, max_group_verts=1, ctx=ctx)
        _say(f"groups call {rep}: {st.groups} groups, eager {st.eager_rounds} captures {st.captures}")
        for g, ref in zip(grads, refs):
            assert (g == ref).all()
        assert st.groups == 6 and st.captures == 6
        eager.append(st.eager_rounds)
    assert eager[0] > 0 and eager[1:] == [0, 0], eager


_FEW_ROUNDS = """
import numpy as np
import oracle_lib
from msceer_amd import batch, native, synth
vols = [synth.smoothed_noise((48, 56, 64), 300 + i, 1.5 + 0.5 * i).astype(np.float32) for i in range(3)]
vols.append(synth.gaussian_mixture((40, 44, 52), 310, 6, 2.0, 6.0, -1.0, 1.0).astype(np.float32))
refs = [oracle_lib.steepest_grad(v) for v in vols]
ctx = native.Context(0)
eager = []
for rep in range(3):
    grads, ms, st = batch.run_batch_grad(vols, ctx=ctx)
    print("rep", rep, "rounds", st.rounds, "eager", st.eager_rounds, "captures", st.captures, flush=True)
    eager.append(st.eager_rounds)
    for g, ref in zip(grads, refs):
        assert (g == ref).all(), int((g != ref).sum())
{check}
assert eager[-1] == 0, eager
ctx.close()
"""


def test_first_capture_without_rounds_sweeps_and_recaptures():
    """No flood sweeps in the first graph: all run after the replay, and the
    next capture takes the sweeps needed."""
    _fresh_process(_FEW_ROUNDS.format(check="assert eager[0] > 0, eager"), {"MSCEER_BATCH_ROUNDS": "0"})


def test_first_capture_with_one_round():
    _fresh_process(_FEW_ROUNDS.format(check=""), {"MSCEER_BATCH_ROUNDS": "1"})


def test_rejects_labels_and_bad_flags(ctx):
    f = np.zeros((4, 4, 4), np.float32)
    g = np.empty(7 * 7 * 7, np.uint8)
    lab = np.empty(64, np.int32)
    arr = batch.volume_table([f.shape], [f.ctypes.data], [g.ctypes.data])
    arr[0].labels_out = lab.ctypes.data
    assert native.lib().msceer_batch_grad(ctx.handle, arr, 1, 0, 0) == native.EINVAL
    arr[0].labels_out = None
    assert native.lib().msceer_batch_grad(ctx.handle, arr, 1, 0, native.SKIP_LDIR) == native.EINVAL
    assert native.lib().msceer_batch_grad(ctx.handle, arr, 1, -1, 0) == native.EINVAL
    assert native.lib().msceer_batch_grad(ctx.handle, arr, 0, 0, 0) == native.OK
