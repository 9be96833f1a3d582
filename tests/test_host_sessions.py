"""The host code of the driver, the sessions, the server and the host copies
against a HIP runtime of plain host memory (tests/host/fake_hip.cpp), on the
CPU: the order between streams, the device of a copy's events, and scalars
that never arrive, none of which a test on a GPU can bring about at will."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "multigrid_amd", "csrc")
OK, EDEVICE = 0, 5
LOST = 719  # hipErrorLaunchFailure
_D = ctypes.POINTER(ctypes.c_double)
_I = ctypes.POINTER(ctypes.c_int)


def _run(*cmd):
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return r.stdout


@pytest.fixture(scope="session")
def host(tmp_path_factory):
    """The host sources and the fake runtime as one library; kernels it does
    not name are functions that return 0."""
    d = str(tmp_path_factory.mktemp("host"))
    flags = ["-D__HIP_PLATFORM_AMD__", "-D__align__(n)=__attribute__((aligned(n)))",
             "-DHIP_SYMBOL(x)=(&x)", "-I/opt/rocm/include", "-std=c++17", "-O1", "-fPIC",
             "-pthread", "-w"]
    jobs, objs = [], []
    for s in [os.path.join(CSRC, f) for f in ("pmg_solver.hip", "pmg_serve.hip",
                                              "pmg_hostcopy.hip")] \
            + [os.path.join(ROOT, "tests", "host", "fake_hip.cpp")]:
        objs.append(os.path.join(d, os.path.basename(s) + ".o"))
        jobs.append(subprocess.Popen(["g++", *flags, "-c", "-x", "c++", "-o", objs[-1], s]))
    assert [j.wait() for j in jobs] == [0] * len(jobs)
    undefined, defined = set(), set()
    for line in _run("nm", *objs).splitlines():
        p = line.split()
        if len(p) >= 2 and not p[-1].endswith(":"):
            (undefined if p[-2] == "U" else defined).add(p[-1])
    names = sorted(n for n in undefined - defined if n.startswith("_ZN3pmg"))
    asm = os.path.join(d, "kernels.s")
    with open(asm, "w") as f:
        f.write(".text\n" + "".join(f".globl {n}\n{n}:\n" for n in names)
                + "xor %eax, %eax\nret\n.section .note.GNU-stack,\"\",@progbits\n")
    so = os.path.join(d, "libhost.so")
    _run("g++", "-shared", "-pthread", "-Wl,--no-undefined", "-Wl,-Bsymbolic", "-o", so, *objs,
         asm)
    L = ctypes.CDLL(so)
    L.fk_set.argtypes = [ctypes.c_int, ctypes.c_double, ctypes.c_double, ctypes.c_int,
                         ctypes.c_int]
    L.fk_copy.argtypes = [ctypes.c_size_t, ctypes.c_int, ctypes.c_int]
    L.pmg_ctx_destroy.argtypes = [ctypes.c_void_p]
    for f in ("pmg_ctx_solve", "pmg_ctx_set_graphs"):
        getattr(L, f).argtypes = [ctypes.c_void_p, ctypes.c_int]
    L.pmg_ctx_pcg.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int]
    L.fk_reset(1)
    return L


def _dp(a):
    return a.ctypes.data_as(_D)


class Ctx:
    def __init__(self, host, mg, n=9, nlev=2, **kw):
        sz = mg.Vmgsz(2, 0, 0, n, n, n, nlev)
        ip, rp = mg.Vpackmg(sz["iretot"], sz["iintot"], n, n, n, nlev, **kw)
        arrays = [np.zeros(n)] * 3 + [np.zeros(4 * n * n)] * 3 + [np.ones(n**3)] * 5
        self.L, self.h = host, ctypes.c_void_p()
        rc = host.pmg_ctx_create(ctypes.byref(self.h), ip.ctypes.data_as(_I), _dp(rp),
                                 *[_dp(a) for a in arrays])
        assert rc == OK

    def close(self):
        self.L.pmg_ctx_destroy(self.h)


@pytest.mark.parametrize("mode", [0, 1])
def test_group_starts_behind_its_members(host, mg, mode):
    """A grouped iteration runs behind all that its members' own streams
    hold: lin_poll may have seen a start's scalar before its work is done."""
    host.fk_reset(1)
    cs = [Ctx(host, mg) for _ in range(3)]
    h = (ctypes.c_void_p * 3)(*[c.h for c in cs])
    assert host.pmg_ctx_solve_group(h, 3, mode) == OK
    assert host.fk_unordered() == 0
    for c in cs:
        c.close()


class Server:
    def __init__(self, host, mg, groups=0, active=4):
        self.L, self.mg, self.h, self.out = host, mg, ctypes.c_void_p(), []
        host.pmg_server_create_grouped.argtypes = [ctypes.c_void_p, ctypes.c_size_t,
                                                   ctypes.c_int, ctypes.c_int]
        host.pmg_server_submit.argtypes = [ctypes.c_void_p, _I, _D, ctypes.c_int,
                                           ctypes.c_double, ctypes.c_double, ctypes.c_int, _D, _D,
                                           ctypes.POINTER(ctypes.c_int64)]
        host.pmg_server_wait.argtypes = [ctypes.c_void_p, ctypes.c_int64, ctypes.c_int,
                                         ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p]
        host.pmg_server_destroy.argtypes = [ctypes.c_void_p]
        assert host.pmg_server_create_grouped(ctypes.byref(self.h), 1 << 33, active,
                                              groups) == OK

    def submit(self, mode, n=9, nlev=2):
        ip, rp = self.mg.make_params(n, nlev)
        at, t = np.array([0.0, 0.0, 0.0, 1.5, 1.0]), ctypes.c_int64()
        self.out.append(np.zeros(n**3))
        assert self.L.pmg_server_submit(self.h, ip.ctypes.data_as(_I), _dp(rp), mode, 0.5, 0.15, 1,
                                        _dp(at), _dp(self.out[-1]), ctypes.byref(t)) == OK
        return t.value

    def wait(self, t, ms=20000):
        return self.L.pmg_server_wait(self.h, t, ms, None, None, None)


@pytest.mark.parametrize("mode", [0, 1])
def test_served_group_starts_behind_its_members(host, mg, mode):
    host.fk_reset(1)
    s = Server(host, mg, groups=2)
    for t in [s.submit(mode) for _ in range(6)]:
        assert s.wait(t) == OK
    assert host.fk_unordered() == 0
    host.pmg_server_destroy(s.h)


@pytest.mark.parametrize("bytes_", [4096, (4 << 20) + 24, (33 << 20) + 8])
@pytest.mark.parametrize("on,cur", [(0, 0), (1, 1), (0, 1), (1, 0)])
def test_copy_from_another_device(host, bytes_, on, cur):
    """A copy takes the device of its stream; the calling thread's current
    device need not be that one, and stays."""
    host.fk_reset(2)
    assert host.fk_copy(bytes_, on, cur) == OK



@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("kind,kw", [("solve", {}), ("pcg", {}), ("newton", dict(nonlin=1)),
                                     ("newton", dict(nonlin=1, mgkey=1))])
@pytest.mark.parametrize("fault", ["none", "no store", "sync", "launch"])
def test_scalar_that_never_lands(host, mg, mode, kind, kw, fault):
    """A stopping scalar that never reaches the host (a failed launch, a lost
    device) ends a solve with PMG_EDEVICE, not with a NaN that passes for
    convergence; and the same context solves again afterwards."""
    host.fk_reset(1)
    c = Ctx(host, mg, **kw)
    graphs = kind == "solve" and fault == "launch"
    host.pmg_ctx_set_graphs(c.h, int(graphs))

    def run():
        return host.pmg_ctx_pcg(c.h, mode, 0) if kind == "pcg" else host.pmg_ctx_solve(c.h, mode)

    if fault == "no store":
        host.fk_set(0, 0.0, 0.0, 0, 0)
    elif fault == "sync":
        host.fk_set(0, 0.0, 0.0, 0, LOST)
    elif fault == "launch":
        host.fk_set(1 if graphs else 0, 0.0, 0.0, LOST, 0)
    rc = run()
    host.fk_set(1, 0.0, 0.0, 0, 0)
    host.pmg_ctx_set_graphs(c.h, 0)
    assert rc == (OK if fault == "none" else EDEVICE)
    assert graphs or run() == OK
    c.close()


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("fault", [(0, 0, 0), (0, LOST, 0), (0, 0, LOST)])
def test_served_scalar_that_never_lands(host, mg, mode, fault):
    """A served request whose scalar never lands is answered with
    PMG_EDEVICE; its worker does not poll for ever."""
    host.fk_reset(1)
    s = Server(host, mg)
    host.fk_set(fault[0], 0.0, 0.0, fault[1], fault[2])
    t = [s.submit(mode) for _ in range(3)]
    assert [s.wait(q, 10000) for q in t] == [EDEVICE] * 3
    host.fk_set(1, 0.0, 0.0, 0, 0)
    host.pmg_server_destroy(s.h)


@pytest.mark.parametrize("group", [False, True])
@pytest.mark.parametrize("zero,iters", [(np.nan, 0), (1.0, 1)])
def test_mixed_first_residual_nan(host, mg, group, zero, iters):
    """A mixed solve whose first cycle gives NaN took no cycle if the
    residual of u = 0 is NaN already (an inf or NaN in the operator), and one
    if the cycle itself overflowed."""
    host.fk_reset(1)
    c = Ctx(host, mg)
    host.pmg_ctx_set_graphs(c.h, 0)
    host.fk_set(1, np.nan, zero, 0, 0)
    h = (ctypes.c_void_p * 1)(c.h)
    assert (host.pmg_ctx_solve_group(h, 1, 1) if group else host.pmg_ctx_solve(c.h, 1)) == OK
    it, rel = ctypes.c_int(), ctypes.c_double()
    host.pmg_ctx_stats(c.h, ctypes.byref(it), None, ctypes.byref(rel), None, None)
    host.pmg_ctx_history.argtypes = [ctypes.c_void_p, _D, ctypes.c_int]
    assert it.value == iters and np.isnan(rel.value)
    assert host.pmg_ctx_history(c.h, None, 0) == iters
    c.close()
