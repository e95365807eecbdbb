"""libqcu.so's host side on a stand-in for the HIP runtime (tests/host/host_hip.cpp): what
a call leaves behind when an allocation fails, and the bookkeeping of resident fields.
Kernels do not run here; the stand-in logs their launches and finds one that reads links
or clover blocks that no earlier launch wrote.  Each scenario is a process of its own."""
import os
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

PRELUDE = """
import ctypes, sys
H = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)   # before libqcu.so: its symbols win
H.host_hip_wrong.restype = ctypes.c_char_p
H.host_hip_live.restype = ctypes.c_size_t
H.host_hip_fail_after.argtypes, H.host_hip_fail_after.restype = [ctypes.c_long], ctypes.c_long
H.host_hip_cost.argtypes = [ctypes.c_char_p, ctypes.c_double]
import numpy as np
import qcu_cg_inverter_amd as q
ref = ctypes.byref
q.init(0)
L = (4, 4, 4, 4)
VH = q.half_volume(L)
def spinor(): return q.DeviceBuffer(2 * VH * 192)
"""


@pytest.fixture(scope="session")
def host_hip(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "host_hip.so")
    src = os.path.join(ROOT, "tests", "host", "host_hip.cpp")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.path.join(ROCM, "include"), src, "-o", so], check=True)
    return so


def run(host_hip, script, *args, **env):
    e = dict(os.environ, PYTHONPATH=ROOT, QCU_EXIT_ON_ERROR="0", **env)
    p = subprocess.run([sys.executable, "-c", PRELUDE + script, host_hip, *map(str, args)],
                       capture_output=True, text=True, env=e, cwd=ROOT, timeout=300)
    assert p.returncode == 0, p.stdout + p.stderr
    return p.stdout


CALLS = """
op = q.Operator(0.12, 1.0, -1, 12)
a, b = spinor(), spinor()
def call(g, name):
    l = q.lib()
    if name == "apply_m": return l.qcuApplyM(g.handle, ref(op), b.ptr, a.ptr, 0)
    if name == "ainv": return l.qcuApplyComposite(g.handle, ref(op), q.COMP_AINV, b.ptr, a.ptr, 0)
    if name == "export": return l.qcuCloverExport(g.handle, ref(op), A.ptr, Ai.ptr, None)
    if name.startswith("mhat"): return l.qcuApplyMhat(g.handle, ref(op), b.ptr, a.ptr, 0, int(name[-1]))
    return l.qcuSolve(g.handle, ref(op), ref(q.default_solve_params(precision=int(name[-1]))), b.ptr, a.ptr, None)
A, Ai = q.DeviceBuffer(2 * VH * 72 * 16), q.DeviceBuffer(2 * VH * 72 * 16)
"""


@pytest.mark.parametrize("name", ["apply_m", "ainv", "export", "mhat0", "mhat1", "mhat2", "solve0", "solve1", "solve2"])
def test_retry_after_failed_allocation(host_hip, name):
    """Whichever allocation of a call fails, the call says so, and the same call made again
    reads no links and no clover block that was not built."""
    run(host_hip, CALLS + textwrap.dedent("""
    name = sys.argv[2]
    for k in range(100):
        g = q.Gauge.random(L, seed=1, eps=0.2)
        H.host_hip_fail_after(k)
        rc = call(g, name)
        H.host_hip_fail_after(-1)
        if rc == 0: break
        assert rc == 3, (k, rc)
        rcs = [call(g, name) for _ in range(3)]
        assert rcs[-1] == 0, (k, rcs, q.lib().qcuGetLastErrorString())
        assert H.host_hip_wrong() == b"", (k, H.host_hip_wrong())
        g.destroy()
    assert 2 < k < 99, k
    """), name)


def test_error_of_one_call_is_not_the_next_ones(host_hip):
    """A call that runs out of memory leaves no error behind for the calls after it."""
    run(host_hip, textwrap.dedent("""
    g = q.Gauge.random(L, seed=1, eps=0.2)
    a, b = spinor(), spinor()
    p = ctypes.c_void_p()
    assert q.lib().qcuMalloc(ref(p), 1 << 50) == 3
    assert q.lib().qcuHop(g.handle, b.ptr, a.ptr, 0, 0, 1, 12, 0) == 0, q.lib().qcuGetLastErrorString()
    """))


DROPIN = """
prm = q.param(L)
def dropin(name, *args):
    q.lib().qcuClearLastError()
    getattr(q.lib(), name)(*args)
    return q.lib().qcuGetLastError()
def new_links(seed):
    u = np.random.default_rng(seed).standard_normal((4, 2, VH, 3, 3, 2))
    gd.upload(u)
gd = q.DeviceBuffer(4 * 2 * VH * 9 * 16)
a, b = spinor(), spinor()
"""


def test_solver_workspace_goes_with_its_dropin_gauge(host_hip):
    """A drop-in gauge that changed after a solve and is then replaced by one of another
    lattice takes the solve's workspace with it."""
    run(host_hip, DROPIN + textwrap.dedent("""
    big = q.param((4, 4, 4, 8))
    gbig, abig, bbig = (q.DeviceBuffer(2 * n) for n in (gd.nbytes, a.nbytes, b.nbytes))
    def apply_big(): assert dropin("fullDslashQcu", bbig.ptr, abig.ptr, gbig.ptr, ref(big), 0) == 0
    def apply(): assert dropin("fullDslashQcu", b.ptr, a.ptr, gd.ptr, ref(prm), 0) == 0
    new_links(1)
    apply()
    apply_big()
    live = H.host_hip_live()
    apply()
    assert dropin("cg_inverter", a.ptr, b.ptr, gd.ptr, ref(prm)) == 0
    new_links(2)
    apply()
    apply_big()
    assert H.host_hip_live() == live
    """))


def test_dropin_gives_up_kept_allocations_for_a_new_one(host_hip):
    """When an allocation fails, whichever it is, while a changed drop-in gauge keeps old
    ones, they are freed and the call goes on, on fields of the new links."""
    run(host_hip, DROPIN + textwrap.dedent("""
    def solve(prec):
        q.check(q.lib().qcuSetDefaultSolve(ref(q.default_solve_params(precision=prec))))
        return dropin("cg_inverter", a.ptr, b.ptr, gd.ptr, ref(prm))
    for k in range(20):
        new_links(2 * k)
        assert solve(1) == 0
        new_links(2 * k + 1)          # FP32 links and clover are kept for the next of their size
        H.host_hip_fail_after(k)
        assert solve(2) == 0, (k, q.lib().qcuGetLastErrorString())
        if H.host_hip_fail_after(-1) >= 0: break
        assert H.host_hip_wrong() == b"", (k, H.host_hip_wrong())
    assert k > 3, k
    """))


def test_kept_workspace_is_given_back(host_hip):
    """The workspace of a solve on links that have changed since does not stand in the way
    of another allocation."""
    run(host_hip, DROPIN + textwrap.dedent("""
    new_links(1)
    assert dropin("cg_inverter", a.ptr, b.ptr, gd.ptr, ref(prm)) == 0
    new_links(2)
    assert dropin("fullDslashQcu", b.ptr, a.ptr, gd.ptr, ref(prm), 0) == 0
    live = H.host_hip_live()
    H.host_hip_fail_after(0)
    extra = q.DeviceBuffer(64)
    assert H.host_hip_fail_after(-1) == -1 and H.host_hip_live() < live
    assert dropin("cg_inverter", a.ptr, b.ptr, gd.ptr, ref(prm)) == 0
    assert H.host_hip_wrong() == b"", H.host_hip_wrong()
    """))


@pytest.mark.parametrize("shift", [0, 192])
def test_in_place_dropin_operator_sees_new_links_first(host_hip, shift):
    """fullDslashQcu whose output overlaps its input cannot be redone once it has written:
    on links that changed, it imports them before anything of the operator is stored."""
    run(host_hip, DROPIN + textwrap.dedent("""
    shift = int(sys.argv[2])
    buf = q.DeviceBuffer(2 * VH * 192 + shift)
    def apply(out, x): assert dropin("fullDslashQcu", out, x, gd.ptr, ref(prm), 0) == 0
    new_links(1)
    apply(buf.ptr + shift, buf.ptr)
    new_links(2)
    H.host_hip_clear_log()
    apply(buf.ptr + shift, buf.ptr)
    assert H.host_hip_launches(b"gauge_pack_kernelILi0ELi12ELi1E") == 1
    assert H.host_hip_first(b"gauge_pack_kernel") < H.host_hip_first(b"spinor_to_aos_kernel")
    assert H.host_hip_launches(b"spinor_to_aos_kernel") == 2
    H.host_hip_clear_log()           # unchanged links: the operator once, nothing imported
    apply(buf.ptr + shift, buf.ptr)
    assert H.host_hip_launches(b"gauge_pack_kernel") == 0 and H.host_hip_launches(b"spinor_to_aos_kernel") == 2
    """), shift)


@pytest.mark.parametrize("plain", [10.0, 0.01])
@pytest.mark.parametrize("older_line", [False, True])
def test_tuned_kernels_outlive_the_process(host_hip, tmp_path, plain, older_line):
    """The tuner's winners come back from QCU_TUNE_CACHE, also where the leg-split kernel
    won (for every epilogue, or for all but the plain one), and over an older line of the
    same key; a process with QCU_TUNE=1 does not tune them again."""
    cache = tmp_path / "tune.cache"
    if older_line:
        cache.write_text("hop:1:12:128:1 64 1 1 0 0 0 0 0 1 1 1 0 0.1\n")
    script = textwrap.dedent("""
    phase, plain = sys.argv[2], float(sys.argv[3])
    g = q.Gauge.random(L, seed=1, eps=0.2)
    split = b"hop_split_kernelILi1ELi12ELi"
    if phase == "tune":
        H.host_hip_cost(split, 0.01)
        H.host_hip_cost(split + b"0E", plain)    # the plain epilogue
        q.tune_hop(g, 1, 12, 1)
    H.host_hip_clear_log()
    op = q.Operator(0.12, 0.0, -1, 12)
    q.apply_mhat(g, op, np.zeros((VH, 4, 3), complex), precision=1)   # one plain hop, one x + a h
    assert H.host_hip_launches(split + b"1E") == 1
    assert H.host_hip_launches(split + b"0E") == (plain < 1)
    a, b = spinor(), spinor()
    q.check(q.lib().qcuSolve(g.handle, ref(op), ref(q.default_solve_params(precision=1)), b.ptr, a.ptr, None))
    assert H.host_hip_launches(b"hop") < 20
    """)
    run(host_hip, script, "tune", plain, QCU_TUNE_CACHE=str(cache))
    run(host_hip, script, "use", plain, QCU_TUNE_CACHE=str(cache), QCU_TUNE="1")


def test_tuner_times_reducing_hops_as_solves_launch_them(host_hip):
    """The epilogues that read x sum |out|^2 in a solve, which takes one right-hand side per
    wave: the tuner times them that way."""
    run(host_hip, textwrap.dedent("""
    g = q.Gauge.random(L, seed=1, eps=0.2)
    H.host_hip_clear_log()
    q.tune_hop(g, 1, 12, 4)
    # hop_kernel<FP32, 12, epilogue, dagger 0, 1 per thread, several per wave, ...>
    kernel = lambda epi, several: b"10hop_kernelILi1ELi12ELi%dELi0ELi1ELi%dE" % (epi, several)
    assert H.host_hip_launches(kernel(0, 1)) > 0 and H.host_hip_launches(kernel(1, 0)) > 0
    assert H.host_hip_launches(kernel(1, 1)) == 0 and H.host_hip_launches(kernel(3, 1)) == 0
    """))


def test_clover_batches_leave_the_split_kernel_in_time(host_hip):
    """The leg-split kernel reads the clover once per right-hand side: points on both sides
    of where that costs more than it gains, each measured."""
    run(host_hip, textwrap.dedent("""
    f = q.lib()["_ZN3qcu9tuned_hopEiilii"]
    f.restype = None
    def split(prec, L, n, epi):
        t = (ctypes.c_int * 15)()      # struct Tune, returned through memory
        f(t, ctypes.c_int(prec), ctypes.c_int(12), ctypes.c_long(q.half_volume(L)), ctypes.c_int(n), ctypes.c_int(epi))
        return t[14] == 1
    A, B, C, D, E, F = (16,) * 4, (16, 16, 16, 32), (20, 20, 20, 40), (24, 24, 24, 32), (24, 24, 24, 48), (8,) * 4
    for epi in (2, 3):
        for prec, L, n in ((0, A, 8), (0, B, 4), (0, C, 2), (1, B, 8), (1, C, 3), (1, A, 12), (1, E, 2), (2, E, 3),
                           (2, A, 6), (2, B, 4), (0, F, 16), (1, F, 16), (2, F, 16)):
            assert split(prec, L, n, epi), (prec, L, n)
        for prec, L, n in ((0, A, 16), (0, B, 8), (0, B, 6), (1, B, 12), (1, B, 16), (1, C, 4), (1, C, 6), (1, D, 4),
                           (2, E, 4), (2, D, 4), (2, A, 12), (2, B, 8)):
            assert not split(prec, L, n, epi), (prec, L, n)
        assert split(0, A, 16, epi - 2) and split(1, C, 6, epi - 2) and split(2, A, 12, epi - 2)
    """))


def test_tuner_times_the_default_too(host_hip):
    """What the default rule would launch is among the tuner's candidates, per epilogue: here
    eight waves beside a staged clover, which no shape that can be pinned has.  What the
    caller is told can be pinned all the same."""
    run(host_hip, textwrap.dedent("""
    L = (16, 16, 16, 12)
    VH = q.half_volume(L)
    g = q.Gauge.random(L, seed=1, eps=0.2)
    op = q.Operator(0.12, 1.0, -1, 12)
    a, b = ([spinor() for _ in range(12)] for _ in range(2))
    def finish():      # a zero source: set up and finished, with two A x + a h hops of 12
        H.host_hip_clear_log()
        q.solve_batch_device(g, op, a, b, q.default_solve_params(precision=0))
        return H.host_hip_launches(b"/512")
    assert finish() == 2
    H.host_hip_cost(b"/512", 0.01)
    shape, _ = q.tune_hop(g, 0, 12, 12)
    assert finish() == 2
    q.set_hop_shape(g, 0, 12, 12, shape)
    """))


def test_layout_streams_what_is_not_read_next(host_hip):
    """A converted spinor that overflows the Infinity Cache beside its copy is streamed past
    it; a smaller even-odd one is left there for what reads it next."""
    run(host_hip, textwrap.dedent("""
    # lattice, field, complex per site, fields, (loads, stores) streamed to even-odd, and back
    for L, field, nc, nf, there, back in (((24, 24, 24, 48), 0, 12, 1, (0, 0), (0, 1)),
                                          ((24, 24, 24, 48), 1, 9, 4, (1, 1), (1, 1)),
                                          ((24, 24, 24, 64), 0, 12, 1, (1, 1), (1, 1)),
                                          ((20, 20, 20, 40), 0, 12, 1, (0, 0), (0, 0)),
                                          ((16, 16, 16, 32), 1, 9, 4, (1, 1), (1, 1)),
                                          ((16, 16, 16, 16), 1, 9, 4, (0, 0), (0, 0))):
        n = 2 * q.half_volume(L) * nc * nf * 16
        a, b = q.DeviceBuffer(n), q.DeviceBuffer(n)
        for f, to_eo, nt in ((q.lib().qcuLexToEvenOdd, 1, there), (q.lib().qcuEvenOddToLex, 0, back)):
            H.host_hip_clear_log()
            q.check(f(b.ptr, a.ptr, (ctypes.c_int * 4)(*L), field))
            assert H.host_hip_launches(b"lex_eo_kernelILb%dELi%dELi%dELi%dE" % (to_eo, nc, *nt)) == 1, (L, field, to_eo)
        del a, b
    """))


def test_clover_counts_in_a_single_launch(host_hip):
    """One right-hand side: the clover a launch reads counts like its links and spinors, on
    both sides of the line by measured points; without one the line is at 300 MiB (550 for
    FP64 recon-12)."""
    run(host_hip, textwrap.dedent("""
    f = q.lib()["_ZN3qcu9tuned_hopEiilii"]
    f.restype = None
    def split(prec, recon, L, epi):
        t = (ctypes.c_int * 15)()
        f(t, ctypes.c_int(prec), ctypes.c_int(recon), ctypes.c_long(q.half_volume(L)), ctypes.c_int(1), ctypes.c_int(epi))
        return t[14] == 1
    T = lambda t: (24, 24, 24, t)
    for epi in (2, 3):
        for prec, recon, L in ((0, 12, T(40)), (0, 12, T(48)), (1, 12, T(48)), (1, 18, T(40)), (2, 18, T(64))):
            assert split(prec, recon, L, epi), (prec, recon, L)
        for prec, recon, L in ((0, 12, T(56)), (0, 12, T(64)), (1, 12, T(56)), (1, 12, T(64)), (1, 18, T(48)),
                               (1, 18, T(56)), (2, 18, (28, 28, 28, 64))):
            assert not split(prec, recon, L, epi), (prec, recon, L)
            assert prec == 0 and L == T(64) or split(prec, recon, L, epi - 2), (prec, recon, L)
    assert split(0, 12, T(64), 0) and not split(1, 18, T(64), 0) and not split(0, 12, (28, 28, 28, 64), 0)
    """))


def test_failed_solves_leave_no_pinned_memory(host_hip):
    """Whichever device allocation of a first solve fails, the scalars it pins are freed."""
    run(host_hip, CALLS + textwrap.dedent("""
    for k in range(100):
        g = q.Gauge.random(L, seed=1, eps=0.2)
        H.host_hip_fail_after(k)
        rc = call(g, "solve1")
        if H.host_hip_fail_after(-1) >= 0: break
        assert rc == 3, (k, rc)
        g.destroy()
        assert H.host_hip_pinned() == 0, (k, H.host_hip_pinned())
    assert k > 6, k
    """))
