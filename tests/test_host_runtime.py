"""The library's host code over a HIP runtime that runs no kernels
(hip_host_stub.cpp): what it does when memory or launches are refused, and
what it asks the runtime for.  Each case is a process of its own, in which
the stub's symbols stand before the real runtime's."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

from conftest import ROOT

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, sys
import numpy as np
sys.path[:0] = [{root!r}, {here!r}]
stub = ctypes.CDLL({stub!r}, mode=ctypes.RTLD_GLOBAL)
stub.stub_device_bytes.restype = ctypes.c_size_t
stub.stub_pinned_device.argtypes = [ctypes.c_uint64]
from cudaprotoplanetarydisks_amd import native
from cudaprotoplanetarydisks_amd.mlp import MLP
from cudaprotoplanetarydisks_amd.native import lib
lib()
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    so = str(tmp_path_factory.mktemp("stub") / "hip_host_stub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", os.path.join(HERE, "hip_host_stub.cpp"), "-o", so],
                   check=True)

    def go(code):
        text = PRELUDE.format(root=ROOT, here=HERE, stub=so) + textwrap.dedent(code)
        r = subprocess.run([sys.executable, "-c", text], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-3000:])
    return go


def test_forward_without_pinned_memory_copies(run):
    """A prediction needs no pinned memory: without it the rows are copied."""
    run("""
    stub.stub_fail_pinned(1)
    with MLP([5, 16, 8], max_batch=4) as net:
        for _ in range(2):
            assert net.forward(np.ones((4, 5))).shape == (4, 8)
        net.train(np.ones((4, 5)), np.ones((4, 8)), batch=4, steps=1, lr=1e-3)
    """)


def test_pinned_rows_belong_to_the_networks_device(run):
    """Whatever device is current when a network predicts, the memory its
    kernel reads the rows from is mapped for the network's own."""
    run("""
    stub.stub_watch(b"k_mlp_rows", 2, 8)
    with MLP([5, 16, 8], max_batch=4, device=1) as net, MLP([5, 16, 8], max_batch=4, device=0):
        net.forward(np.ones((4, 5)))
        rows = ctypes.c_uint64()
        stub.stub_watched(ctypes.byref(rows))
        assert stub.stub_pinned_device(rows) == 1, stub.stub_pinned_device(rows)
    """)


def test_forward_refuses_null(run):
    """A NULL input or output is an error of the call, with the rows in pinned
    memory as with the copies."""
    run("""
    y = np.zeros((2, 8), np.float32)
    p = y.ctypes.data_as(ctypes.POINTER(ctypes.c_float))
    for pinned in (1, 0):
        stub.stub_fail_pinned(1 - pinned)
        with MLP([5, 16, 8], max_batch=4) as net:
            assert lib().fg_mlp_forward(net.h, None, 2, p) == native.FG_E_HIP
            assert lib().fg_mlp_forward(net.h, p, 1, None) == native.FG_E_HIP
    """)


def test_training_gives_large_sample_sets_back(run):
    """What a network holds between training calls is bounded: a sample set
    beyond the bound (64 MB) is freed when the call returns."""
    run("""
    widths, bound = [1024, 8, 1024], 64 << 20
    rows = 2 * bound // (4 * 2048)
    with MLP(widths, max_batch=16) as net:
        held = stub.stub_device_bytes()
        small = np.zeros((16, 1024), np.float32)
        net.train(small, small, batch=16, steps=2, lr=1e-3)
        large = np.zeros((rows, 1024), np.float32)
        for _ in range(2):
            net.train(large, large, batch=16, steps=2, lr=1e-3)
            assert stub.stub_device_bytes() - held < bound, stub.stub_device_bytes() - held
        net.train(small, small, batch=16, steps=2, lr=1e-3)
    assert stub.stub_device_bytes() == 0
    """)


@pytest.mark.parametrize("widths", [[5, 16, 8], [5, 1000, 8]], ids=["rows", "layers"])
@pytest.mark.parametrize("kernel", ["forward", "weights"])
def test_failed_training_step_is_not_counted(run, widths, kernel):
    """The bias corrections of Adam take the steps that were taken: a step
    whose launches failed before its update is none of them."""
    rows = len(widths) == 3 and widths[1] <= 896
    fail = {"forward": "k_mlp_rows" if rows else "k_gemm", "weights": "k_mlp_weights" if rows else "k_colsum"}[kernel]
    # 1 - 0.9: the last but one of adam_args' six floats, or k_adam's argument
    watch, index, size, at = ("k_mlp_weights", 11, 24, 4) if rows else ("k_adam", 10, 4, 0)
    run(f"""
    stub.stub_watch({watch.encode()!r}, {index}, {size})
    x, t = np.ones((4, 5), np.float32), np.ones((4, 8), np.float32)
    with MLP({widths!r}, max_batch=4) as net:
        stub.stub_fail_launches({fail.encode()!r}, 1)
        try:
            net.train(x, t, batch=4, steps=1, lr=1e-3)
            raise SystemExit("the step did not fail")
        except native.FargoError:
            pass
        net.train(x, t, batch=4, steps=1, lr=1e-3)
        arg = (ctypes.c_float * {size // 4})()
        stub.stub_watched(arg)
        assert arg[{at}] == np.float32(1) - np.float32(0.9), list(arg)
    """)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_substep_entries_allocate_no_host_memory(run, deck, precision):
    """A substep's C entries take no memory from the C++ heap, whose failure
    would be an exception that no C caller can catch."""
    path = deck(Nrad=16, Nsec=32)
    run(f"""
    from cudaprotoplanetarydisks_amd import Simulation
    sim = Simulation({path!r}, precision={precision!r}, fused=True)
    planet = native.FgPlanetPot(1.0, 0.0, 1e-3, 1e-4, 1.0)
    for fail in (0, 1):
        stub.stub_fail_new(fail)
        status = [lib().fg_step_fused(sim.ctx.h, 1e-3, 1.0, 0.0, ctypes.byref(planet), 1, 0.0, 0.0, 0.1, 0)]
        status.append(lib().fg_transport(sim.ctx.h, 1e-3, 1.0, None))
        stub.stub_fail_new(0)
        assert status == [0, 0], (status, lib().fg_last_error())
    """)


def test_wide_rings_ask_for_their_lds(run, deck):
    """A launch beyond 64 KB of LDS, dynamic and static together, asks for it
    first: the kernels that stage a ring, at the widest grid."""
    path = deck(Nrad=8, Nsec=8192, InnerBoundary="NONREFLECTING", Viscosity=None, AlphaViscosity=1e-3)
    run(f"""
    from cudaprotoplanetarydisks_amd import Simulation
    sim = Simulation({path!r})
    n, c = ctypes.c_int(), sim.ctx.h
    lib().fg_cfl(c, 0.1, ctypes.byref(n))
    lib().fg_ring_mean_cs(c)
    lib().fg_boundary(c, 1e-3, 1.0)
    for kernel in (b"k_cfl_ring", b"k_ring_mean", b"k_nr_edges"):
        asked, granted = ctypes.c_size_t(), ctypes.c_size_t()
        stub.stub_lds(kernel, ctypes.byref(asked), ctypes.byref(granted))
        assert asked.value >= 8192 * 8, kernel
        assert granted.value >= asked.value, (kernel, asked.value, granted.value)
    """)


def test_single_disks_take_no_batch_tuned_shapes(run, deck):
    """The autotuner times batches; a lone FP32 disk keeps the bands picked for
    its grid, and a batch takes the entry."""
    path = deck(Nrad=16, Nsec=32)
    run(f"""
    from cudaprotoplanetarydisks_amd import Simulation, ensemble, sim
    entry = dict([("16x32", dict(src_rows=16, trad_band=8))])
    ensemble.load_tiles = lambda path=None: entry
    calls = []
    def call(name, *args):
        calls.append(name)
        return native.call(name, *args)
    sim.call = ensemble.call = call
    Simulation({path!r}, precision="fp32").close()
    assert "fg_set_tiles" not in calls
    ensemble.Ensemble([{path!r}]).close()
    assert "fg_batch_set_tiles" in calls
    """)
