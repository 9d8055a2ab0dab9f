"""What the library asks of the HIP runtime, in order (no GPU: a runtime of host memory answers and logs
the calls, kernels do not run): allocations and the buffers the launches write, streams, launch choices.
Each scenario runs in a process of its own, where that runtime is loaded before the library."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C, re, sys
F = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
F.fake_log.restype, F.fake_log.argtypes = C.c_size_t, [C.c_char_p, C.c_size_t]
F.fake_room.argtypes, F.fake_capture.argtypes = [C.c_size_t], [C.c_void_p]
F.fake_step.argtypes = [C.c_double]
sys.path.insert(0, sys.argv[2])
import numpy as np
import tandem_amd as T
from tandem_amd._lib import lib

def log(pattern=""):
    b = C.create_string_buffer(F.fake_log(None, 0))
    F.fake_log(b, len(b))
    F.fake_clear()
    return [l for l in b.value.decode().splitlines() if re.search(pattern, l)]

def operator(kind, D, n, N):
    op = T.DGOperator(T.Mesh.box(D, n, 1 if D == 3 else 0, 5), kind, N)
    one = np.ones((op.E, op.Nq))
    op.set_material(one, one if kind == 0 else None)
    return op

X, Y = C.c_void_p(1 << 20), C.c_void_p(1 << 21)  # vectors that no host code touches
MULT = {8: lib().tdg_mult, 4: lib().tdg_mult_f32}
BATCH = {8: lib().tdg_mult_batched, 4: lib().tdg_mult_batched_f32}

def traces(lines):
    return {l.split()[-1] for l in lines if "poisson_trace" in l or "poisson_element" in l}

def slots(lines):
    return {l.split()[-1] for l in lines if "facet_kernel" in l or "element_kernel" in l}
"""


@pytest.fixture(scope="session")
def host_hip(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hip") / "host_hip.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I/opt/rocm/include",
                           os.path.join(HERE, "fake_hip.cpp"), "-o", so])

    def run(code):
        r = subprocess.run([sys.executable, "-c", PRELUDE + code, so, ROOT], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout

    return run


def test_batch_that_finds_no_memory_leaves_single_applies_whole(host_hip):
    """A column count whose facet slots do not fit is an error; the applies after it write slots that are
    there, not the lost buffer."""
    host_hip("""
op = operator(0, 3, 2, 4)
for pb in (8, 4):
    assert MULT[pb](op._h, X, Y) == 0
    one = slots(log())
    assert BATCH[pb](op._h, X, Y, 2, op.n) == 0
    F.fake_room(1 << 22)
    assert BATCH[pb](op._h, X, Y, 64, op.n) == -3 and b"out of memory" in lib().tdg_last_error()
    F.fake_room(1 << 40)
    log()
    assert MULT[pb](op._h, X, Y) == 0 and slots(log()) == one
    assert BATCH[pb](op._h, X, Y, 2, op.n) == 0
    lines = log()
    (m,) = [l.split() for l in lines if l.startswith("malloc")]
    assert int(m[2]) == 2 * op.n * 4 * pb and slots(lines) == {m[1]}
""")


def test_poisson_batch_that_finds_no_memory_leaves_single_applies_whole(host_hip):
    """The same for the traces of the matrix-core Poisson apply: no launch writes a buffer that is gone."""
    host_hip("""
op = operator(1, 3, 14, 1)
for pb in (8, 4):
    assert MULT[pb](op._h, X, Y) == 0
    F.fake_room(1 << 22)
    BATCH[pb](op._h, X, Y, 64, op.n)
    F.fake_room(1 << 40)
    log()
    assert MULT[pb](op._h, X, Y) == 0
    used = traces(log())
    assert used and "(nil)" not in used
""")


@pytest.mark.parametrize("pb", [8, 4])
def test_poisson_traces_stay_in_place(host_hip, pb):
    """No apply frees a trace buffer that an earlier one was launched with (a captured apply replays into
    it), and all of them together stay bounded whatever column counts come."""
    host_hip("""
pb = %d
op = operator(1, 3, 14, 1)
op.upload()
log()
one = op.E * 4 * op.nq * 2 * pb
seen = []
for cols in (1, 2, 7, 64, 3, 300, 1, 3000):
    assert (MULT[pb](op._h, X, Y) if cols == 1 else BATCH[pb](op._h, X, Y, cols, op.n)) == 0
    lines = log()
    seen += [int(l.split()[2]) for l in lines if l.startswith("malloc")]
    assert not [l for l in lines if l.startswith("free")], cols
    used = traces(lines)
    assert len(used) == 1
    if cols == 1:
        single = single if cols > 1 or "single" in globals() else used
        assert used == single
    # columns a launch takes fit the buffer that it writes
    assert sum(int(l.split("x")[1].split()[0]) for l in lines if "poisson_trace" in l) == cols
assert sum(seen) <= 2 * (1 << 30) and max(seen) > (1 << 30) - one
op.set_material(np.ones((op.E, op.Nq)))  # a new material gives everything back
assert len(log("^free")) >= len(seen)
""" % pb)


@pytest.mark.parametrize("pb", [8, 4])
def test_poisson_apply_under_capture_needs_nothing_new(host_hip, pb):
    """What could be captured before the operator had any traces still can: after the upload every column
    count, and variants switched in between, by the kernels whose data are there."""
    host_hip("""
pb = %d
S = 1 << 12
for n, cols in ((14, 1), (14, 64), (5, 64)):      # large, and of a size that only batches take the rule
    for reserved in (False, True):
        op = operator(1, 3, n, 1)
        if not reserved:
            lib().tdg_set_variant(op._h, 1)       # uploaded for another variant
        op.upload()
        lib().tdg_set_variant(op._h, 0)
        if reserved:
            assert BATCH[pb](op._h, X, Y, cols, op.n) == 0
        assert lib().tdg_set_stream(op._h, C.c_void_p(S)) == 0
        F.fake_capture(S)
        log()
        assert BATCH[pb](op._h, X, Y, cols, op.n) == 0, (n, cols, reserved, lib().tdg_last_error())
        F.fake_capture(None)
        lines = log("launch")
        assert bool(traces(lines)) == reserved and len(lines) >= 1 and all("stream 0x1000 " in l for l in lines)
""" % pb)


@pytest.mark.parametrize("pb", [8, 4])
def test_poisson_operator_without_memory_for_traces(host_hip, pb):
    """An operator that fits the device without the matrix-core apply's data still works, on the kernel that
    needs none; without memory for a batch's traces the batch goes through those there are."""
    host_hip("""
pb = %d
op = operator(1, 3, 14, 1)
lib().tdg_set_variant(op._h, 1)
op.upload()
lib().tdg_set_variant(op._h, 0)
F.fake_room(op.n * pb * 3)      # the traces of one column are four vectors and more
assert MULT[pb](op._h, X, Y) == 0, lib().tdg_last_error()
assert log("launch") and not log("poisson_trace")
F.fake_room(1 << 40)
op.set_material(np.ones((op.E, op.Nq)))
assert MULT[pb](op._h, X, Y) == 0
one = traces(log())
assert one
F.fake_room(op.E * 4 * op.nq * 2 * pb + 1)
assert BATCH[pb](op._h, X, Y, 3, op.n) == 0
lines = log("launch")
assert traces(lines) == one and len(lines) == 6
""" % pb)


def test_poisson_noalloc_applies_share_nothing(host_hip):
    """tdg_mult_noalloc of two Poisson operators: neither writes memory of the other (they may overlap in
    time on two streams), whatever their size, and nothing is allocated."""
    host_hip("""
used = []
for n in (14, 20):
    op = operator(1, 3, n, 1)
    op.upload()
    globals()["op%d" % n] = op
    log()
    assert lib().tdg_mult_noalloc(op._h, X, Y) == 0
    lines = log()
    assert not [l for l in lines if l.startswith("malloc")]
    used.append(traces(lines))
    assert MULT[8](op._h, X, Y) == 0 and traces(log()) == used[-1]
assert used[0] and used[1] and not used[0] & used[1]
""")


@pytest.mark.parametrize("kind,N,n,shared", [(1, 1, 14, True), (0, 2, 2, True), (1, 1, 3, False)])
def test_new_stream_waits_for_the_old_one(host_hip, kind, N, n, shared):
    """Applies queued on one stream and then on another meet in the operator's buffers: the new stream waits
    for the old one; not under capture, nor where an operator has no such buffers."""
    host_hip("""
op = operator(%d, 3, %d, %d)
shared = %s
A, B = 1 << 12, 1 << 13
def streams(s):
    log()
    assert lib().tdg_set_stream(op._h, C.c_void_p(s)) == 0
    return log("record|wait")
assert streams(A) == []                       # nothing on the device yet
op.upload()
assert MULT[8](op._h, X, Y) == 0
lines = streams(B)
if shared:
    (r, rs, re_), (w, ws, we) = [l.split() for l in lines]
    assert (r, rs, w, ws) == ("record", hex(A), "wait", hex(B)) and re_ == we
else:
    assert lines == []
assert streams(B) == []                       # the same stream again
assert len(streams(None)) == len(lines)
F.fake_capture(A)
assert streams(A) == [] and MULT[8](op._h, X, Y) == 0 and streams(B) == []
""" % (kind, n, N, shared))


@pytest.mark.parametrize("precision,pb", [("fp64", 8), ("fp32", 4)])
def test_shape_search_leaves_the_small_launches(host_hip, precision, pb):
    """A shape searched for many columns governs the launches that the rule for few elements leaves to it: a
    one-column apply of the same mesh keeps its small launches (a facet group a workgroup of five waves), and a
    count for which they were the slower choice does without them."""
    host_hip("""
precision, pb = "%s", %d
op = operator(0, 3, 4, 4)
def small(cols):
    log()
    assert (MULT[pb](op._h, X, Y) if cols == 1 else BATCH[pb](op._h, X, Y, cols, op.n)) == 0
    (f,) = log("facet_kernel")
    return " block 320 " in f
assert small(1) and small(2) and not small(64)
for step in (1.0, -1.0):
    F.fake_step(step)
    shape, ms = op.autotune_shapes(64, precision)
    assert small(1) and small(2) and not small(64)
    assert ms[shape] == min(ms.values())
F.fake_step(1.0)                    # the later a configuration is timed, the slower it is
shape, ms = op.autotune_shapes(1, precision)
assert ms[shape] == min(ms.values()) and not small(1) and small(2)
F.fake_step(-1.0)
shape, ms = op.autotune_shapes(1, precision)
assert ms[shape] == min(ms.values()) and small(1) and small(2)
op.set_shape(precision, *shape)     # chosen by the caller: for every apply
assert not small(1) and not small(2)
F.fake_step(1.0)
assert op.autotune(64, precision)[0] == "auto" and small(1)
""" % (precision, pb))


@pytest.mark.parametrize("precision,order", [("fp64", 2), ("fp64", 0), ("fp32", 1)])
def test_shape_search_for_columns_leaves_the_order(host_hip, precision, order):
    """Several columns take the same launch in the linear and the per-XCD order: noise between equal launches
    does not choose the order of single applies."""
    host_hip("""
precision, order = "%s", %d
op = operator(0, 3, 4, 4)
for step, kept in ((1.0, 1 if order == 2 else order), (-1.0, 2)):   # the first configuration wins, then the last
    op.set_shape(precision, 1, order)
    F.fake_step(step)
    log()
    shape, ms = op.autotune_shapes(64, precision)
    assert shape == (0 if step > 0 else 3, kept)
    assert len(log("elapsed")) == 2 * 8
    assert len(ms) == 12 and all(ms[s, 0] == ms[s, 1] for s in range(4))
    assert ms[shape] == min(ms.values())
F.fake_step(1.0)
assert op.autotune_shapes(1, precision)[0] == (0, 0)   # a single column times every order
""" % (precision, order))


@pytest.mark.parametrize("precision,pb", [("fp64", 8), ("fp32", 4)])
@pytest.mark.parametrize("D,n,N,visits", [(3, 3, 4, False), (3, 5, 2, True), (2, 24, 3, True)])
def test_kernels_of_several_columns(host_hip, D, n, N, visits, precision, pb):
    """The element kernel of several columns is the one of single columns (one with a loop over columns has no
    registers for it), and facet workgroups visit several columns where that pays: every (group, column) once."""
    host_hip("""
D, n, N, visits, precision, pb = %r
op = operator(0, D, n, N)
for shape in range(4):
    for order in range(3):
        op.set_shape(precision, shape, order)
        log()
        assert MULT[pb](op._h, X, Y) == 0
        f1, e1 = log("launch")
        assert BATCH[pb](op._h, X, Y, 800, op.n) == 0
        f, e = log("launch")
        assert "facet" in f and "element" in e and e.split()[1] == e1.split()[1]
        assert (f.split()[1] != f1.split()[1]) == visits
""" % ((D, n, N, visits, precision, pb),))


def test_poisson_search_below_the_size_rule_leaves_the_choice_open(host_hip):
    """Tuned at a size where the automatic choice and "points" are the same kernel, a Poisson operator still
    takes the matrix-core apply for more columns; a faster assembled apply, or a choice at a size where both
    kernels ran, is kept."""
    host_hip("""
op = operator(1, 3, 5, 2)          # 7,500 unknowns; no assembled register kernel
for precision, pb in (("fp64", 8), ("fp32", 4)):
    name, ms = op.autotune(1, precision)
    assert name == "auto" and ms["auto"] == ms["points"]
    log()
    assert MULT[pb](op._h, X, Y) == 0 and not traces(log())
    assert BATCH[pb](op._h, X, Y, 64, op.n) == 0 and traces(log())
    F.fake_step(-1.0)
    assert op.autotune(1, precision)[0] == "auto"
    assert op.autotune(64, precision)[0] == "points"
    F.fake_step(1.0)
    assert op.autotune(64, precision)[0] == "auto"
small = operator(1, 3, 5, 1)       # block size 4: the assembled register kernel
F.fake_step(-1.0)
assert small.autotune(1, "fp64")[0] == "assembled"
F.fake_step(1.0)
assert small.autotune(1, "fp64")[0] == "auto"
assert operator(1, 2, 5, 1).autotune(1, "fp64")[0] == "points"   # no matrix-core apply at any size
""")


def test_right_hand_side_is_one_launch(host_hip):
    """Volume and facet part of a right-hand side in one launch whatever its data (small calls cost their
    launches), with a workgroup for every element that has a face with data."""
    host_hip("""
for D, n, N in ((3, 2, 1), (2, 9, 4)):
    op = operator(0, D, n, N)
    F0, D0 = C.c_void_p(1 << 22), C.c_void_p(1 << 23)
    grid = {}
    for force, data in ((F0, D0), (None, D0), (F0, None), (None, None)):
        log()
        assert lib().tdg_rhs_device(op._h, force, data, Y, 3, op.E * D * op.Nq, op.F * D * op.nq, op.n) == 0
        (l,) = log("launch")
        grid[force is not None, data is not None] = int(l.split("grid ")[1].split("x")[0])
        assert "x3 " in l
    f = op.facets()
    touched = len(set(f[f[:, 4] == 5][:, 0]))
    assert grid[True, True] == grid[False, True] == grid[True, False] + touched and touched > 0
""")


def test_inverse_mass_of_the_smallest_meshes(host_hip):
    """3D P4 up to 512 elements and degrees without an apply take a workgroup an element, all else the
    matrix cores."""
    host_hip("""
for D, n, N, mfma in ((3, 1, 4, False), (3, 4, 4, False), (3, 5, 4, True), (3, 1, 3, True), (2, 1, 6, True), (3, 1, 5, False)):
    op = operator(0, D, n, N)
    op.upload()
    log()
    assert lib().tdg_inverse_mass(op._h, X, Y) == 0
    (l,) = log("launch")
    assert ("mfma" in l) == mfma, (D, n, N, l)
    assert mfma or "grid %dx1" % op.E in l
""")


@pytest.mark.parametrize("pb", [8, 4])
@pytest.mark.parametrize("D,n,N", [(3, 2, 4), (2, 9, 6)])
def test_single_column_slots_stay_in_place(host_hip, D, n, N, pb):
    """A batch of any size leaves the facet slots of single applies where they are (a captured single apply
    replays into them)."""
    host_hip("""
D, n, N, pb = %r
op = operator(0, D, n, N)
op.upload()
assert MULT[pb](op._h, X, Y) == 0
one = slots(log())
assert len(one) == 1
for cols in (2, 5, 3, 40):
    assert BATCH[pb](op._h, X, Y, cols, op.n) == 0
    lines = log()
    assert not one & slots(lines) and not [l for l in lines if l.startswith("free") and l.split()[1] in one]
    assert MULT[pb](op._h, X, Y) == 0
    assert slots(log()) == one
""" % ((D, n, N, pb),))
