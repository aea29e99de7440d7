"""CPU checks of the C ABI: the library loads, exports every symbol the
public header declares, host-side logic agrees with the oracle, and invalid
specs are rejected before any device work."""
import ctypes
import os
import re
import subprocess
import sys
import tempfile

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    txt = open(os.path.join(ROOT, "include", "fpde_hip.h")).read()
    txt = re.sub(r"/\*.*?\*/", "", txt, flags=re.S)
    return sorted(set(re.findall(r"\b(fpde_[A-Za-z0-9_]+)\s*\(", txt)))


def test_library_exports_every_declared_symbol(fpde):
    L = fpde.lib()
    syms = declared_symbols()
    assert len(syms) >= 40
    missing = [s for s in syms if not hasattr(L, s)]
    assert not missing, missing


def test_binding_covers_header(fpde):
    from fpde_hpc_amd._lib import SIGNATURES
    bound = {n for n, _, _ in SIGNATURES}
    assert set(declared_symbols()) == bound


def test_init_conditions_match_oracle(fpde, oracle):
    for n, seed in [(1000, 1000), (10000, 1001), (37, 5)]:
        assert np.array_equal(fpde.init_1d(n, seed), oracle.init_1d(n, seed))
    for n, seed in [(16, 1003), (9, 7)]:
        assert np.array_equal(fpde.init_3d(n, seed), oracle.init_3d(n, seed))


def test_ksat_fourier_matches_oracle(fpde, oracle):
    for ut, h, tau in [(-1.0, 1e-3, 1e-3), (-0.95, 1e-4, 5e-4), (-1.07, 2.5e-4, 1e-3)]:
        a = fpde.lib().fpde_ksat_for_fourier(ut, h, tau, 1.0)
        b = oracle.ksat_for_fourier(ut, h, tau, 1.0)
        assert abs(a - b) <= 1e-14 * abs(b)


def test_product_vgm_matches_closed_form(fpde):
    """The library's K/C at suction P (through fpde_ksat_for_fourier, which
    returns fo h^2 / (tau Kr(P) / C(P))) against the van Genuchten-Mualem
    closed form in 50-digit arithmetic: Kr = Se^(1/2) (1 - (x/(1+x))^m)^2,
    C = (n-1)(s1-s0) x Se / (P (1+x)), x = (100 a P)^n, Se = (1+x)^-m, over
    wet to very dry soil (the dry end is where a difference of logarithms
    would lose digits)."""
    import mpmath
    mpmath.mp.dps = 50
    n, s0, s1, a = mpmath.mpf(5) / 4, mpmath.mpf("0.0736"), mpmath.mpf("0.55"), mpmath.mpf("0.066")
    m = 1 - 1 / n
    for P in np.logspace(-6, 3, 400):
        Pm = mpmath.mpf(float(P))
        x = (100 * a * Pm) ** n
        se = (1 + x) ** (-m)
        kr = mpmath.sqrt(se) * (1 - (x / (1 + x)) ** m) ** 2
        C = (n - 1) * (s1 - s0) * x * se / (Pm * (1 + x))
        ratio = fpde.lib().fpde_ksat_for_fourier(-float(P), 1.0, 1.0, 1.0)     # = 1 / (Kr / C)
        exact = float(C / kr)
        assert abs(ratio - exact) <= 1e-14 * exact, P


@pytest.mark.parametrize("bad", [
    dict(dims=2), dict(nodes=3), dict(steps=0), dict(alpha=0.0), dict(alpha=1.5),
    dict(picard_max=0), dict(hist_mode=9), dict(block=48), dict(dims=3, nodes=300),
    dict(tau=-1.0), dict(nodes=70000), dict(sum_alg=3), dict(sum_alg=1, sum_param=-1.0),
    dict(sum_alg=2, sum_param=0.0, hist_mode=0), dict(sum_alg=2, sum_param=65.0, hist_mode=0),
    dict(sum_alg=2, sum_param=2.5, hist_mode=0), dict(sum_alg=2, sum_param=8.0, hist_mode=1),
    dict(sum_alg=2, sum_param=8.0, hist_mode=0, do_q=4),
    dict(gamma=1.5), dict(gamma=-0.1),
    dict(chunk_rows=16), dict(chunk_rows=300), dict(nodes=20000, chunk_rows=64),
])
def test_invalid_specs_rejected(fpde, bad):
    kw = dict(nodes=100, steps=10, tau=1e-3, alpha=0.5, hist_mode=1, block=64)
    kw.update(bad)
    dims = kw.pop("dims", 1)
    spec = fpde.make_spec(kw.pop("nodes"), kw.pop("steps"), kw.pop("tau"), dims=dims, ksat=1.0, **kw)
    h = ctypes.c_void_p()
    rc = fpde.lib().fpde_solver_create(ctypes.byref(spec), ctypes.byref(h))
    assert rc == 1
    assert fpde.lib().fpde_last_error()


def test_footprint_scales_with_history(fpde):
    a = fpde.footprint(fpde.make_spec(10000, 20000, 5e-4, hist_mode="plain", ksat=1.0))
    b = fpde.footprint(fpde.make_spec(10000, 20000, 5e-4, hist_mode="split_bf16", ksat=1.0))
    assert a >= 8 * 10000 * 20000
    assert b >= a + 4 * 10000 * 20000 - 1
    # series moments (sum_alg 2): P values per node instead of M levels
    c = fpde.footprint(fpde.make_spec(10000, 20000, 5e-4, hist_mode="plain", ksat=1.0, sum_alg=2, sum_param=32))
    assert c < a / 50


def test_unknown_kernel_name_is_reported(fpde):
    # program/kernel objects need no device
    L = fpde.lib()
    prog = ctypes.c_void_p()
    assert L.fpde_cl_program_create(ctypes.c_void_p(1), b"#define OS 64\n", ctypes.byref(prog)) == 0
    k = ctypes.c_void_p()
    assert L.fpde_cl_kernel_create(prog, b"Nope", ctypes.byref(k)) == 4
    assert b"Sum" in L.fpde_last_error()
    assert L.fpde_cl_kernel_create(prog, b"Sum", ctypes.byref(k)) == 0
    L.fpde_cl_kernel_destroy(k)
    L.fpde_cl_program_destroy(prog)


@pytest.mark.parametrize("name", ["fpde_spec", "fpde_stats", "fpde_result_info"])
def test_struct_layout_matches_binding(fpde, name):
    """The ctypes structures have the C header's size and field offsets (gcc)."""
    from fpde_hpc_amd import _lib
    cls = {"fpde_spec": _lib.Spec, "fpde_stats": _lib.Stats, "fpde_result_info": _lib.ResultInfo}[name]
    fields = [f for f, _ in cls._fields_]
    body = "".join(f'printf("%zu\\n", offsetof({name}, {f}));' for f in fields)
    src = ('#include <stdio.h>\n#include "fpde_hip.h"\nint main(void){printf("%zu\\n", sizeof('
           + name + '));' + body + 'return 0;}\n')
    with tempfile.TemporaryDirectory() as d:
        c, exe = os.path.join(d, "l.c"), os.path.join(d, "l")
        open(c, "w").write(src)
        subprocess.check_call(["gcc", "-std=c99", "-I", os.path.join(ROOT, "include"), c, "-o", exe])
        out = [int(v) for v in subprocess.check_output([exe]).split()]
    assert out[0] == ctypes.sizeof(cls)
    assert out[1:] == [getattr(cls, f).offset for f in fields]


@pytest.mark.parametrize("args", [
    (0, 0, 100, 0.01, 0.5, 1, 1e-5), (8, 8, 3, 0.01, 0.5, 1, 1e-5), (8, 8, 100, 0.0, 0.5, 1, 1e-5),
    (8, 8, 100, 0.01, 1.0, 1, 1e-5), (8, 8, 100, 0.01, 0.0, 1, 1e-5), (8, 8, 100, 0.01, 0.5, 2, 1e-5),
])
def test_space_sum_rejects_bad_arguments(fpde, args):
    """Argument checks run before any device call (no GPU needed)."""
    rc = fpde.lib().fpde_space_sum(*args)
    assert rc == 1
    assert fpde.lib().fpde_last_error()


def test_autotune_block_argument_checks_and_plain_form(fpde):
    """Null arguments and invalid specs are refused before any device call;
    hist_mode 0 has no history block, so no trial runs and the block stays."""
    L = fpde.lib()
    spec = fpde.make_spec(64, 300, 1e-3, hist_mode="split_bf16", block=0)
    u0 = np.zeros(64)
    b, ms = ctypes.c_int(-1), ctypes.c_double(-1.0)
    assert L.fpde_autotune_block(None, fpde.solver._p(u0), 0, ctypes.byref(b), None) == 1
    assert L.fpde_autotune_block(ctypes.byref(spec), None, 0, ctypes.byref(b), None) == 1
    assert L.fpde_autotune_block(ctypes.byref(spec), fpde.solver._p(u0), 0, None, None) == 1
    bad = fpde.make_spec(64, 300, 1e-3, hist_mode="split_bf16", block=48)
    assert L.fpde_autotune_block(ctypes.byref(bad), fpde.solver._p(u0), 0, ctypes.byref(b), None) == 1
    plain = fpde.make_spec(64, 300, 1e-3, hist_mode="plain", block=0)
    assert L.fpde_autotune_block(ctypes.byref(plain), fpde.solver._p(u0), 0, ctypes.byref(b), ctypes.byref(ms)) == 0
    assert b.value == 0 and ms.value == 0.0


def test_advance_batch_argument_checks(fpde):
    """A null array, a count outside 1..32 and a null solver are refused
    before any device call."""
    L = fpde.lib()
    null1 = (ctypes.c_void_p * 1)(None)
    assert L.fpde_solver_advance_batch(None, 1, 0) == 1
    assert L.fpde_solver_advance_batch(null1, 0, 0) == 1
    many = (ctypes.c_void_p * 33)()
    assert L.fpde_solver_advance_batch(many, 33, 0) == 1
    assert L.fpde_solver_advance_batch(null1, 1, 0) == 1
    assert b"null solver" in L.fpde_last_error()


def test_correction_table_holds_every_row_of_the_last_block(fpde):
    """The history GEMM of a 3D block reads the two corrections of all its
    rows, also those of steps past the last: the table holds them wherever the
    last block starts."""
    entries = fpde.lib()["_ZN4fpde12corr_entriesEi"]
    entries.argtypes, entries.restype = [ctypes.c_int], ctypes.c_size_t
    for steps in (1, 63, 64, 65, 70, 1000, 20000):
        for block in (16, 32, 64, 128):
            for n0 in (steps - 1, (steps - 1) // block * block):
                assert entries(steps) > 2 * (n0 + block - 1) + 1, (steps, block, n0)


def test_history_plans_of_no_nodes(fpde):
    """A sum over no nodes is a call like any other: its plans (which divide
    the work by tiles of nodes) give one part, no partial row and no crash.  In
    a process of its own, since a division by zero ends it."""
    code = ("import ctypes, fpde_hpc_amd as F\n"
            "L = F.lib()\n"
            "r, h = L['_ZN4fpde14ref_sum_splitsEll'], L['_ZN4fpde15hist_plain_planEiiPii']\n"
            "r.argtypes = [ctypes.c_int64] * 2\n"
            "h.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.POINTER(ctypes.c_int), ctypes.c_int]\n"
            "c = ctypes.c_int(-1)\n"
            "assert all(r(0, n) == 1 for n in (-1, 0, 1, 64, 10 ** 6))\n"
            "assert all(h(0, n, c, 64) == 0 and c.value == 0 for n in (0, 1, 257, 10 ** 6))\n")
    subprocess.run([sys.executable, "-c", code], cwd=ROOT, check=True, timeout=120)


FAKE_DEVICE = r"""
#include <stddef.h>
#include <stdlib.h>
/* the device calls of the scratch pool on host memory: `budget` bytes per device, two devices */
static size_t budget, used[2], size_of[64];
static void *ptr_of[64];
static int dev_of[64], dev;
void fake_budget(size_t b) { budget = b; }
size_t fake_used(int d) { return used[d]; }
int hipGetDevice(int *d) { *d = dev; return 0; }
int hipSetDevice(int d) { dev = d; return 0; }
static int last, launch_error, launches;
void fake_launch_error(int e) { launch_error = e; }
int fake_launches(void) { return launches; }
int hipGetLastError(void) { int e = last; last = 0; return e; }
int hipLaunchKernel(void) { launches++; return last = launch_error; }
int __hipPushCallConfiguration(void) { return 0; }
int __hipPopCallConfiguration(void) { return 0; }
int hipDeviceSynchronize(void) { return 0; }
int hipMalloc(void **p, size_t n) {
    if (used[dev] + n > budget) return 2;
    for (int i = 0; i < 64; i++)
        if (!ptr_of[i]) {
            *p = ptr_of[i] = malloc(1);
            size_of[i] = n; dev_of[i] = dev; used[dev] += n;
            return 0;
        }
    return 2;
}
int hipFree(void *p) {
    for (int i = 0; i < 64; i++)
        if (p && ptr_of[i] == p) { used[dev_of[i]] -= size_of[i]; free(p); ptr_of[i] = 0; return 0; }
    return 1;
}
"""

SCRATCH_POOL = r"""
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1])
import fpde_hpc_amd as F
L = F.lib()
class Lease(ctypes.Structure):
    _fields_ = [("ptr", ctypes.c_void_p), ("bytes", ctypes.c_size_t), ("dev", ctypes.c_int)]
sz, MB, ANY = ctypes.c_size_t, 1 << 20, ctypes.c_size_t(-1).value
fake.fake_budget.argtypes, fake.fake_used.restype = [sz], sz
take, give = L["_ZN4fpde12ScratchLease4takeEmim"], L["_ZN4fpde12ScratchLease4giveEv"]
take.argtypes, give.argtypes = [ctypes.c_void_p, sz, ctypes.c_int, sz], [ctypes.c_void_p]
def lease(n, dev=-1, at_most=ANY):
    l = Lease()
    return take(ctypes.byref(l), n, dev, at_most), l
def keep(n):
    rc, l = lease(n)
    assert rc == 0
    give(ctypes.byref(l))
fake.fake_budget(100 * MB)
# what the pool keeps gives way to a lease it does not fit and to other allocations
keep(60 * MB)
assert fake.fake_used(0) == 60 * MB
rc, l = lease(80 * MB)
assert rc == 0 and fake.fake_used(0) == 80 * MB
assert lease(30 * MB)[0] == 3                     # nothing kept: refused
give(ctypes.byref(l))
b = ctypes.c_void_p()
L.fpde_cl_buf_alloc.argtypes = [ctypes.c_void_p, sz, ctypes.c_void_p, ctypes.POINTER(ctypes.c_void_p)]
assert L.fpde_cl_buf_alloc(1, 90 * MB, None, ctypes.byref(b)) == 0 and fake.fake_used(0) == 90 * MB
assert L.fpde_cl_buf_free(b) == 0
# a lease held for long does not take a far larger buffer, a short one does
keep(60 * MB)
rc, l = lease(MB, -1, 2 * MB)
assert rc == 0 and l.bytes == MB and fake.fake_used(0) == 61 * MB
rc, m = lease(MB)
assert rc == 0 and m.bytes == 60 * MB
# memory of another device, the thread's device left as it was
rc, o = lease(3 * MB, 1)
assert rc == 0 and o.dev == 1 and fake.fake_used(1) == 3 * MB
cur = ctypes.c_int(-1)
fake.hipGetDevice(ctypes.byref(cur))
assert cur.value == 0
for x in (l, m, o):
    give(ctypes.byref(x))
assert L.fpde_shutdown() in (0, 2)                # (its own device calls find no device here)
"""


def _on_fake_device(tmp_path, code):
    c, so = tmp_path / "fake.c", tmp_path / "fake.so"
    c.write_text(FAKE_DEVICE)
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", str(so), str(c)])
    env = dict(os.environ, LD_PRELOAD=" ".join([str(so), os.environ.get("LD_PRELOAD", "")]).strip())
    subprocess.run([sys.executable, "-c", code, str(so)], cwd=ROOT, env=env, check=True, timeout=120)


def test_scratch_pool_gives_way(tmp_path):
    """The scratch pool on a host stand-in for the device calls it makes: kept
    buffers are freed when an allocation is refused, a long lease is about as
    large as its request, and a lease for another device is on that device."""
    _on_fake_device(tmp_path, SCRATCH_POOL)


HISTORY_SUM_CALLS = r"""
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1])
import fpde_hpc_amd as F
L = F.lib()
fake.fake_budget.argtypes, fake.fake_used.restype = [ctypes.c_size_t], ctypes.c_size_t
def call(levels, nodes):
    return L.fpde_history_sum_f64(8, 8, levels, nodes, (nodes + 63) // 64 * 64, 8)
"""


def test_history_sum_takes_the_memory_its_form_needs(tmp_path):
    """A short history's sum is one launch without partial rows; a long one
    takes as many rows as its plan has parts (fewer than 64 on long lines)."""
    _on_fake_device(tmp_path, HISTORY_SUM_CALLS + r"""
fake.fake_budget(0)
rc = call(64, 20000)
assert rc == 0 and fake.fake_launches() == 1, (rc, fake.fake_launches(), L.fpde_last_error())
assert call(2000, 20000) == 3
fake.fake_budget(24 << 20)
assert call(300, 3000000) == 0                    # one row of 24 MB
""")


def test_short_history_sums_of_long_lines_are_streamed(tmp_path):
    """One launch for a short history up to 65536 nodes; beyond, the stream and
    the sum of its parts."""
    _on_fake_device(tmp_path, HISTORY_SUM_CALLS + r"""
fake.fake_budget(1 << 40)
for nodes, launches in ((65536, 1), (65537, 2), (1 << 29, 2), (1 << 30, 2)):
    before = fake.fake_launches()
    assert call(1, nodes) == 0 and fake.fake_launches() - before == launches, nodes
""")


def test_history_sum_reports_a_refused_launch(tmp_path):
    """A launch that the runtime refuses is an error of the call, in the one
    launch of a short history and in the stream."""
    _on_fake_device(tmp_path, HISTORY_SUM_CALLS + r"""
fake.fake_budget(1 << 40)
for levels in (1, 256, 257, 5000):
    fake.fake_launch_error(1)
    assert call(levels, 1000) == 2, levels
    fake.fake_launch_error(0)
    assert call(levels, 1000) == 0, levels
""")
