"""The library's host side on a stand-in HIP runtime (no GPU): what it does when
the runtime refuses something, and what it asks the runtime for.

tests/hip_stand_in.c takes the place of the HIP runtime in a process of its
own; device memory is host memory there and kernels do not run.  Each test
runs a short script against the C ABI and reads what it prints.
"""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = r"""
import ctypes as C, struct, sys
si = C.CDLL(sys.argv[1], C.RTLD_GLOBAL)       # its symbols come before the runtime's
from starrynight_amd._lib import LIB_PATH, Params, Tuning
L = C.CDLL(LIB_PATH)
vp = C.c_void_p
L.sn_last_error.restype = C.c_char_p
class Launch(C.Structure):
    _fields_ = [("name", C.c_char * 256), ("grid", C.c_uint32 * 3), ("block", C.c_uint32 * 3), ("lds", C.c_size_t),
                ("arg", C.c_ubyte * 128)]
limit, uploaded = C.c_size_t.in_dll(si, "si_malloc_limit"), C.c_size_t.in_dll(si, "si_uploaded")
capturing, copy_fails = C.c_int.in_dll(si, "si_capturing"), C.c_int.in_dll(si, "si_copy_fails")
def launches():
    n, ring = C.c_long.in_dll(si, "si_launches").value, (Launch * 64).in_dll(si, "si_launch")
    return [ring[k % 64] for k in range(max(0, n - 64), n)]
def last(name):
    return [l for l in launches() if name.encode() in l.name][-1]
def create(boxes, rc=3, T=300.0, kernel=0):
    ps = (Params * len(boxes))()
    for p, (p.X, p.Y, p.Z) in zip(ps, boxes):
        p.dipole_cutoff, p.cage_strain, p.temperature = rc, 1.0, T
    t, h = Tuning(kernel=kernel), vp()
    status = L.sn_create(ps, len(boxes), C.byref(t), C.byref(h))
    return status, h
def context(*args, **kw):
    status, h = create(*args, **kw)
    assert status == 0, L.sn_last_error(h)
    return h
D = C.c_double
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    so = tmp_path_factory.mktemp("stand_in") / "hip_stand_in.so"
    subprocess.check_call(["gcc", "-O1", "-Wall", "-shared", "-fPIC", "-o", str(so),
                           os.path.join(ROOT, "tests", "hip_stand_in.c")])

    def script(body):
        r = subprocess.run([sys.executable, "-c", PRELUDE + body, str(so)], cwd=ROOT, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
        return r.stdout.split()
    return script


def test_partial_sums_are_never_a_null_buffer(run):
    """A larger buffer that cannot be had is an error, and so is not forgotten:
    the next call that needs no more than the old size gets a buffer again."""
    out = run(r"""
h = context([(64, 64, 64), (12, 12, 12)])
fe, afe, count, M = (D * 81)(), (D * 81)(), (C.c_int64 * 81)(), (D * 3)()
print(L.sn_moment(h, 0, M))                      # a first buffer
limit.value = 100000
print(L.sn_radial_order(h, 0, fe, afe, count))   # needs a larger one
print(L.sn_moment(h, 1, M), struct.unpack("<Q", bytes(last("moment_kernel").arg[:8]))[0] != 0)
""")
    assert out == ["0", "2", "0", "True"]


@pytest.mark.parametrize("call", ["L.sn_radial_order(h, 0, fe, afe, count)", "L.sn_dipole_potential(h, 0, pot)"])
def test_observable_tables_are_kept_only_when_filled(run, call):
    """A table whose copy to the device failed is made again on the next call."""
    out = run(rf"""
h = context([(12, 12, 12)])
fe, afe, count, pot = (D * 81)(), (D * 81)(), (C.c_int64 * 81)(), (D * 1728)()
copy_fails.value = 1
print({call})
copy_fails.value = 0
before = uploaded.value
print({call}, uploaded.value > before)
before = uploaded.value
print({call}, uploaded.value > before)           # kept from now on
""")
    assert out == ["2", "0", "True", "0", "False"]


def test_refused_parameters_are_not_kept(run):
    """Parameters refused under capture reach the device with no later call."""
    out = run(r"""
h = context([(12, 12, 12)])
lat = (D * (4 * 1728))(*([0.0, 0.0, 1.0, 1.0] * 1728))
def record():                                    # beta, J, L0 of the last parameter record
    a = bytes(last("put_rep_kernel").arg)
    return struct.unpack_from("<2d", a, 24) + struct.unpack_from("<d", a, 48)
capturing.value = 1
print(L.sn_set_params(h, 0, D(600.0), (D * 3)(0, 0, 0.5), D(7.0)))
capturing.value = 0
print(L.sn_set_lattice(h, 0, lat), record() == (1.0, 1.0, 1.0))
print(L.sn_set_params(h, 0, D(600.0), (D * 3)(0, 0, 0.5), D(7.0)), record() == (0.5, 7.0, 1.0))
""")
    assert out == ["2", "0", "True", "0", "True"]


@pytest.mark.parametrize("refusal", ["capturing.value = 1", "limit.value = 100"])
def test_refused_random_lattice_leaves_the_sweep_as_it_was(run, refusal):
    """A random lattice of several lengths that is refused (capture, no memory
    for its species table) leaves the kernel variant and the uniform length."""
    out = run(rf"""
h = context([(12, 12, 12)])
print(L.sn_mc_sweeps(h, 1)); before = last("torus_sweep").name
{refusal}
print(L.sn_init_lattice_random(h, 0, 2, (D * 2)(0.0, 1.0), (D * 2)(0.5, 0.5)) != 0)
capturing.value, limit.value = 0, 1 << 40
print(L.sn_mc_sweeps(h, 1), last("torus_sweep").name == before)
print(any(b"put_rep" in l.name for l in launches()))
""")
    assert out == ["0", "True", "0", "True", "False"]


def test_parameters_are_not_refused_for_an_earlier_error(run):
    """An error another library left behind is not this call's."""
    out = run(r"""
h = context([(12, 12, 12)])
C.c_int.in_dll(si, "si_last_error").value = 1
print(L.sn_set_params(h, 0, D(600.0), None, D(7.0)))
""")
    assert out == ["0"]


def test_round_tables_are_made_for_one_layout_at_a_time(run):
    """A whole-lattice context makes the round tables of uniform lengths (8 + 8
    NPL bytes a lane and round, 16^3 at DipoleCutOff 3: about 3.2 MB) and those
    of mixed lengths with its first such lattice, again after a failure."""
    out = run(r"""
h = context([(16, 16, 16)])
n = 16 ** 3
at_create = uploaded.value
lat = (D * (4 * n))(*([0.0, 0.0, 1.0, 1.0] * (n - 1) + [0.0, 1.0, 0.0, 0.0]))
def tables(call):                                # bytes copied beyond the lattice itself
    before = uploaded.value
    return call(), uploaded.value - before - (32 * n if call is set_lattice else 0)
set_lattice, sweep = lambda: L.sn_set_lattice(h, 0, lat), lambda: L.sn_mc_sweeps(h, 1)
limit.value = 100000
print(*[v for call in (set_lattice, sweep) for v in tables(call)])       # refused, and the sweep with it
limit.value = 1 << 40
first = tables(sweep)
print(first[0], 0.9 * at_create < first[1] < at_create < 3.5e6)
print(*[v for call in (sweep, set_lattice, sweep) for v in tables(call)])
h = context([(16, 16, 16)])
print(*[tables(set_lattice) == (0, first[1]), tables(sweep) == (0, 0)])
""")
    assert out == ["2", "0", "2", "0", "0", "True", "0", "0", "0", "0", "0", "0", "True", "True"]


def test_whole_lattice_kernel_with_static_lds_is_refused(run):
    """Its tables hold LDS addresses that begin at 0: an instance whose sites
    would begin elsewhere is not launched."""
    out = run(r"""
print(create([(25, 25, 1)])[0], create([(25, 25, 1)], kernel=3)[0])
C.c_size_t.in_dll(si, "si_static_lds").value = 16
for kernel in (0, 3):
    status, h = create([(25, 25, 1)], kernel=kernel)
    print(status, b"static LDS" in L.sn_last_error(h))
""")
    assert out == ["0", "0", "2", "True", "2", "True"]
