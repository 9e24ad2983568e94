"""The library's host code without a device (tests/cpp/no_device.c): what a call does when an allocation fails, and objects of the
host mirror that need a context but no result."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def no_device(tmp_path_factory):
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        pytest.skip("no C compiler")
    lib = tmp_path_factory.mktemp("no_device") / "libno_device.so"
    subprocess.check_call([cc, "-O1", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC", "-o", str(lib), os.path.join(ROOT, "tests", "cpp", "no_device.c")])
    return lib


@pytest.fixture(scope="module")
def run(no_device):
    """runs statements in a process of their own in which `dp` is the package and `dev` the runtime without a device"""

    def go(body):
        text = "import ctypes, importlib, sys\nimport numpy as np\n"
        text += "dev = ctypes.CDLL(%r, ctypes.RTLD_GLOBAL)\n" % str(no_device)  # (before the library: its calls are found here)
        text += "for f in ('no_device_in_use', 'no_device_most', 'no_device_launches', 'no_device_first_word'): getattr(dev, f).restype = ctypes.c_int64\n"
        text += "dev.no_device_budget.argtypes = [ctypes.c_int64]\n"
        text += "sys.path.insert(0, %r)\ndp = importlib.import_module('deep-prove_amd')\n" % ROOT + body
        res = subprocess.run([sys.executable, "-c", text], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=300)
        assert res.returncode == 0, res.stdout[-2000:] + res.stderr[-2000:]
        assert "done" in res.stdout

    return go


def test_a_sum_that_is_rewritten_falls_back_when_the_new_tables_do_not_fit(run):
    # X Y + X Z over 2^18 entries runs as X (Y + Z): more memory than the sum as it stands, which is taken where only it fits
    run("""
n = 18
one = np.array([1, 0], dtype=np.uint64)
def tables(ctx):
    z = np.zeros((1 << n, 2), dtype=np.uint64)
    return [ctx.mle_from_ext2(z) for _ in range(3)]
terms = [(one, [0, 1]), (one, [0, 2])]
ctx = dp.Context(0)
tabs = tables(ctx)
before = dev.no_device_in_use()
dev.no_device_most_from_now()
s = ctx.session(n, tabs, terms)
rewritten = dev.no_device_most() - before
assert rewritten > 0
del s, tabs
ctx.close()
ctx = dp.Context(0)
tabs = tables(ctx)
before = dev.no_device_in_use()
dev.no_device_budget(before + rewritten - 1)
s = ctx.session(n, tabs, terms)
as_it_stands = dev.no_device_most() - before
assert s.degree == 2
del s
dev.no_device_budget(before)  # nothing fits beside the tables
try:
    s = ctx.session(n, tabs, terms)
    raise SystemExit("a session without memory")
except dp.DpsError as e:
    assert e.status == 3, e  # out of memory
dev.no_device_budget(1 << 60)
s = ctx.session(n, tabs, terms)
print("done")
""")


def test_a_round_asked_for_again_when_its_descriptors_did_not_fit(run):
    # 8 products over 16 tables, several groups of them: planned to be resident from round 1, so only round 1 is described.  Without a place on the device the
    # launches read descriptors from device memory; where those do not fit the call fails, and the next one finds memory for them
    run("""
n = 9
one = np.array([1, 0], dtype=np.uint64)
ctx = dp.Context(0)
z = np.zeros((1 << n, 2), dtype=np.uint64)
tabs = [ctx.mle_from_ext2(z) for _ in range(16)]
s = ctx.session(n, tabs, [(one, [h, 8 + h]) for h in range(8)])
dp.set_resident_budget(0, 0)
dev.no_device_budget(dev.no_device_in_use())
launches = dev.no_device_launches()
try:
    s.round(None)
    raise SystemExit("a round without memory")
except dp.DpsError as e:
    assert e.status == 3, e  # out of memory
assert dev.no_device_launches() == launches
dev.no_device_budget(1 << 60)
try:
    s.round(None)
    raise SystemExit("a result without a device")
except dp.DpsError as e:
    assert e.status == 2, e
assert dev.no_device_launches() == launches + 1
assert dev.no_device_first_word() != 0, "the launch has no descriptors"
print("done")
""")


def test_sums_over_three_eq_factors_without_a_compute_unit_take_them_as_tables(run):
    # sum_g eq_g P_g over two tables.  In closed form the eq tables are never folded and have no buffers; as tables they do (3/4 of 2^n entries each)
    run("""
n = 16
one = np.array([1, 0], dtype=np.uint64)
ctx = dp.Context(0)
tabs = [ctx.mle_from_ext2(np.zeros((1 << n, 2), dtype=np.uint64)) for _ in range(2)]
eqs = [ctx.eq_build(np.full((n, 2), g + 1, dtype=np.uint64)) for g in range(3)]
polys = {"softmax": [[[0], [0, 1, 1]], [[0], [1, 1, 1]], [[0, 1]]], "two cubics": [[[0], [0, 1, 1]], [[0], [1, 1, 1]]], "activation": [[[0], [0, 1, 1]], [[0], [1]]]}
def taken(ps):
    terms = [(one, fs + [2 + g]) for g, poly in enumerate(ps) for fs in poly]
    before = dev.no_device_in_use()
    s = ctx.session(n, tabs + eqs[:len(ps)], terms)
    bytes_ = dev.no_device_in_use() - before
    ctx.keep = getattr(ctx, "keep", []) + [s]  # (so that no session finds another's memory)
    return bytes_
folded = 16 * (3 << n) // 4
with_units = {k: taken(ps) for k, ps in polys.items()}
dp.set_resident_budget(0, 0)
without = {k: taken(ps) for k, ps in polys.items()}
for k, ps in polys.items():
    more = without[k] - with_units[k]
    assert (more >= folded * len(ps)) == (k != "activation"), (k, more, folded)
print("done")
""")


def test_a_logup_circuit_is_complete_as_its_constructor_leaves_it(no_device, tmp_path):
    exe, lib = tmp_path / "test_logup_circuit", os.path.join(ROOT, "deep-prove_amd", "lib")
    # (linked before the library: its calls are found in the runtime without a device)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-o", str(exe), os.path.join(ROOT, "tests", "cpp", "test_logup_circuit.cpp"), "-Wl,--no-as-needed",
                           "-L" + str(no_device.parent), "-lno_device", "-L" + lib, "-ldpsumcheck", "-Wl,-rpath," + str(no_device.parent) + ":" + lib])
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and "ok" in out.stdout, out.stdout + out.stderr
