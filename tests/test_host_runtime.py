"""The library's host side against a stand-in runtime (hip_stub.cpp): what it does when a device call fails, which
streams, workspaces and limits it asks for.  Each test runs a short program in a child process with the stand-in
preloaded; the kernels do nothing there, so only control flow is looked at, never a number."""
import os
import subprocess
import sys
import textwrap

import pytest

from conftest import ROOT

HEAD = """
import ctypes as C, sys, threading
sys.path.insert(0, {root!r}); sys.path.insert(0, {pkg!r})
import numpy as np
import __graft_entry__ as entry
hf = entry._load()
import molecules as M
stub = C.CDLL({stub!r})
stub.stub_count.restype = C.c_long
MALLOCS, STREAMS, WATCHED, OUTSIDE, LDS_BEYOND, FAILED, WATCHED_STREAMS, BETWEEN = range(8)
def basis(mol, name):
    return hf.Basis.from_g94(M.basis_text(name), mol.symbols, mol.xyz)
def raises(code, call):
    try:
        call()
    except hf.HfError as e:
        assert e.code == code, (e.code, str(e))
        return str(e)
    raise AssertionError("no error")
water = M.water_config1()
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("stub") / "hip_stub.so")
    src = os.path.join(os.path.dirname(os.path.abspath(__file__)), "hip_stub.cpp")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", so, src, "-lpthread"])
    head = HEAD.format(root=ROOT, pkg=os.path.join(ROOT, "hf-rs_amd"), stub=so)

    def run(body, **env):
        pre = os.environ.get("LD_PRELOAD", "")
        e = dict(os.environ, LD_PRELOAD=(pre + ":" if pre else "") + so, OMP_NUM_THREADS="2", **env)
        r = subprocess.run([sys.executable, "-c", head + textwrap.dedent(body)], env=e, capture_output=True, text=True,
                           timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr

    return run


def test_server_builds_over_two_streams(program):
    """The fleet's two and one per set-up worker, and no more when it has run."""
    program("""
    srv = hf.Server(capacity=2)
    assert stub.stub_count(STREAMS) == 2 + 2, stub.stub_count(STREAMS)
    srv.submit([basis(water, "sto-3g")], [water.zxyz], max_iter=3)
    srv.run()
    assert stub.stub_count(STREAMS) == 2 + 2
    srv.close()
    assert stub.stub_count(STREAMS) == 0
    """)


@pytest.mark.parametrize("kernel", ["k_sad_scatter", "k_symmetrize"])
def test_device_errors_of_the_guess_are_reported(program, kernel):
    """A device call that fails in the SAD guess (its own kernel, or a build of an atomic solve) fails the request or
    the solve with its message: the core-Hamiltonian start is for a guess that is unavailable, not for one that the
    device failed to make."""
    program("""
    b = basis(water, "sto-3g")
    stub.stub_fail_kernel(%r)
    srv = hf.Server(capacity=1)
    rid = srv.submit([b], [water.zxyz], max_iter=3)
    srv.run()
    r = srv.result(rid)
    assert not r["ok"] and r["status"] == hf.HFG_DEVICE and "stub failure" in r["error"], r
    if %r == "k_sad_scatter":  # (a solve's own builds use the other one as well)
        assert "stub failure" in raises(hf.HFG_DEVICE, lambda: hf.scf_rhf(b, water.zxyz, max_iter=3))
    stub.stub_fail_kernel(b"")
    again = srv.submit([b], [water.zxyz], max_iter=3)
    srv.run()
    assert srv.result(again)["ok"]
    """ % (kernel.encode(), kernel))


def test_a_reported_error_is_not_reported_again(program):
    """A failed allocation fails its call with HFG_DEVICE; the runtime keeps the error for the thread's next
    hipGetLastError, but the next call on another handle of the thread, which succeeds, does not report it."""
    program("""
    b = basis(water, "sto-3g")
    ctx = hf.Context(b)
    p = np.eye(b.n)
    ctx.contract_jk(p)
    stub.stub_fail_malloc(2)
    raises(hf.HFG_DEVICE, lambda: hf.Context(b))
    ctx.contract_jk(p)
    """)


@pytest.mark.parametrize("precision", ["fp64", "bf16x3"])
def test_df_workspace_after_a_failed_allocation(program, precision):
    """Every allocation of a first J/K call fails in turn; the next call on the same handle has a whole workspace (J's
    tiles, the buffer of several that is allocated last, lie in an allocation)."""
    program("""
    b, aux = basis(water, "sto-3g"), basis(water, "def2-svp-rifit")
    c = np.ones((b.n, 5))
    k = 0
    while True:
        k += 1
        df = hf.DfTensor(b, aux)
        before = stub.stub_count(FAILED)
        stub.stub_fail_malloc(k)
        try:
            df.jk_precision(c, %r)
        except hf.HfError as e:
            assert e.code == hf.HFG_DEVICE
        if stub.stub_count(FAILED) == before:
            break
        stub.stub_watch(b"k_untile_sym", 0)
        df.jk_precision(c, %r)
        assert stub.stub_count(WATCHED) == 1 and stub.stub_count(OUTSIDE) == 0, k
        df.close()
    assert k > 5
    """ % (precision, precision))


def test_server_slot_after_a_failed_allocation(program):
    """Every allocation of the set-up of a larger molecule fails in turn; the smaller one that takes the slot next has
    a buffer (its density lies in an allocation)."""
    program("""
    small, large = basis(water, "sto-3g"), basis(water, "cc-pvdz")
    k = hit = 0
    while True:
        k += 1
        srv = hf.Server(capacity=1)
        first = srv.submit([small], [water.zxyz], max_iter=2)
        srv.run()
        srv.submit([large], [water.zxyz], max_iter=2)
        before = stub.stub_count(FAILED)
        stub.stub_watch(b"k_clear", 0)
        stub.stub_fail_malloc(k)
        try:
            srv.run()  # the larger one first, then the smaller one again
        except hf.HfError as e:
            assert e.code == hf.HFG_DEVICE
        assert stub.stub_count(OUTSIDE) == 0, k
        stub.stub_fail_malloc(0)
        srv.close()
        if stub.stub_count(FAILED) == before or k == 60:
            break
    assert k > 20
    """)


def test_lds_limit_of_a_kernel_is_shared_by_the_threads(program):
    """The limit that a kernel's launches with much LDS rely on is the kernel's: another thread's builds of a smaller
    molecule leave it, so that no launch asks for more than is allowed."""
    program("""
    small, large = basis(water, "sto-3g"), basis(M.water_cluster_m(6, 1), "6-31g*")
    a = hf.Context(large)
    a.contract_jk(np.eye(large.n))
    def other():
        hf.Context(small).contract_jk(np.eye(small.n))
    t = threading.Thread(target=other)
    t.start(); t.join()
    for _ in range(2):
        a.contract_jk(np.eye(large.n))
    assert stub.stub_count(LDS_BEYOND) == 0, stub.stub_count(LDS_BEYOND)
    """)


@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16x3"])
def test_df_device_time_holds_no_allocation(program, precision):
    """The device time that a J/K call returns is the contraction's, on a handle's first call as on later ones: no
    allocation lies between its two events."""
    program("""
    b, aux = basis(water, "sto-3g"), basis(water, "def2-svp-rifit")
    df = hf.DfTensor(b, aux)
    before = stub.stub_count(MALLOCS), stub.stub_count(BETWEEN)
    df.jk_precision(np.ones((b.n, 5)), %r)
    assert stub.stub_count(MALLOCS) > before[0]
    assert stub.stub_count(BETWEEN) == before[1], stub.stub_count(BETWEEN) - before[1]
    """ % precision)
