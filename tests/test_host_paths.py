"""The host side of liblbmhip.so without a device: which launches a call
makes, what it allocates and what it does when an allocation or a launch
fails.  Each test runs a script in a child process whose HIP runtime is the
stub of tests/stub_hip (device memory out of a budget, launches logged)."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

from conftest import PKG, ROOT

STUB = os.path.join(ROOT, "tests", "stub_hip", "hip_stub.c")
pytestmark = pytest.mark.skipif(shutil.which("gcc") is None or not os.path.exists("/opt/rocm/include/hip"),
                                reason="needs gcc and the HIP headers")

PRELUDE = """
import ctypes as C, sys
sys.path.insert(0, {pkg!r})
import lbm_amd as lbm
S = C.CDLL({stub!r})
S.stub_log.restype = C.c_char_p

def free_bytes(n=None):
    v = C.c_size_t.in_dll(S, "stub_free")
    if n is not None:
        v.value = n
    return v.value

def fail_launch(name):
    C.memmove(C.addressof(C.c_char.in_dll(S, "stub_fail_launch")), name.encode() + bytes(1), len(name) + 1)

def fail_call(name):
    C.memmove(C.addressof(C.c_char.in_dll(S, "stub_fail_call")), name.encode() + bytes(1), len(name) + 1)

def log():
    # lines since the last call
    text = S.stub_log().decode().splitlines()
    S.stub_clear()
    return text

def launches(name):
    return sum(line.startswith("launch") and name in line for line in log())

def kernel(name, dims, args=(), periodic=(1, 0, 0), geo="channel"):
    g = lbm.Geometry.from_string(geo, dims, periodic)
    C.c_uint32.in_dll(S, "stub_count").value = g.n_fluid
    return lbm.Kernel(name, g, ["-quiet"] + list(args))

def case(steps, **kw):
    return lbm.case_data(iterations=steps, **kw)
"""


@pytest.fixture(scope="session")
def stub(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("stub") / "hip_stub.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", STUB, "-o", out,
                    "-lpthread"], check=True, capture_output=True)

    def run(script):
        env = dict(os.environ, LD_PRELOAD=out)
        r = subprocess.run([sys.executable, "-c", PRELUDE.format(pkg=PKG, stub=out) + textwrap.dedent(script)],
                           capture_output=True, text=True, env=env, timeout=120)
        assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-3000:])
    return run


def test_init_reports_a_failed_launch_when_memory_is_short(stub):
    """aa-soa's Init reports a launch that failed also where the arrays of the
    two-step launch do not fit."""
    stub("""
        free_bytes(8 << 20)
        fail_launch("k_aa_info")
        try:
            kernel("aa-soa", (40, 24, 24))
        except RuntimeError as e:
            assert "cell info kernel" in str(e), e
        else:
            raise AssertionError("Init succeeded")
    """)


@pytest.mark.parametrize("name", ["list-aa-pv-soa", "aa-soa"])
def test_two_step_info_says_what_the_call_did(stub, name):
    """LbmHipTwoStepInfo counts the two-step launches that the last call made,
    also from a replayed graph and where the arrays did not fit."""
    stub(f"""
        def check(k, steps, want):
            log()
            k.run(case(steps))
            made = launches("k_pair")
            assert k.two_step().launches == want, (k.two_step().launches, want)
            return made
        name = {name!r}
        k = kernel(name, (20, 20, 20), ["-two-step", "on"])
        i = k.two_step()
        assert i.planned and (i.tileY, i.tileZ, i.segments) == (5, 32, 20) and i.bytes > 0
        assert check(k, 6, 3) == 3 and k.two_step().held == i.bytes
        k.set_launch_events(True)
        assert check(k, 6, 0) == 0
        k = kernel(name, (20, 20, 20), ["-two-step", "on", "-graph", "on"])
        want = 2 if name == "list-aa-pv-soa" else 3          # an odd number of pairs: one in place
        assert check(k, 6, want) == want and check(k, 6, want) == 0
        k = kernel(name, (20, 20, 20), ["-two-step", "off"])
        assert not k.two_step().planned and check(k, 6, 0) == 0
        k = kernel(name, (20, 20, 20), ["-two-step", "on"])
        free_bytes(i.bytes + 4096)                           # more than half of it
        assert k.two_step().planned
        assert check(k, 6, 0) == 0 and k.two_step().held == 0
    """)


def test_aa_init_takes_the_lattice_alone(stub):
    """aa-soa's Init allocates as much with two-step launches as without, and
    a lattice stepped with launch events never takes their arrays."""
    stub("""
        def taken(mode):
            before = free_bytes()
            k = kernel("aa-soa", (20, 20, 20), ["-two-step", mode])
            return k, before - free_bytes()
        a, plain = taken("off")
        b, paired = taken("on")
        assert paired == plain, (paired, plain)
        before = free_bytes()
        b.set_launch_events(True)
        b.run(case(4))
        assert free_bytes() == before
        b.set_launch_events(False)
        b.run(case(4))
        assert before - free_bytes() == b.two_step().held == b.two_step().bytes
    """)


@pytest.mark.parametrize("name", ["list-aa-pv-soa", "aa-soa"])
def test_arrays_are_given_back_to_another_lattice(stub, name):
    """A lattice whose Init fits only without the two-step arrays of another
    one gets their memory; the other goes on with the separate launches and
    takes the arrays again once there is room."""
    stub(f"""
        a = kernel({name!r}, (40, 40, 40), ["-two-step", "on"])
        a.run(case(4))
        held = a.two_step().held
        assert held > 0
        free_bytes(held // (2 if {name!r} == "list-aa-pv-soa" else 8))
        b = kernel({name!r}, (40, 40, 40), ["-two-step", "off"])
        assert a.two_step().held == 0 and a.two_step().planned
        log()
        a.run(case(4))
        assert a.two_step().launches == 0 and launches("k_pair") == 0
        b.close()
        free_bytes(1 << 40)
        a.run(case(4))
        assert a.two_step().launches == 2 and a.two_step().held == held and launches("pair_map") == 1
        a.release_two_step()
        assert a.two_step().held == 0
        a.close()
        c = kernel({name!r}, (40, 40, 40), ["-two-step", "on"])
        d = kernel({name!r}, (40, 40, 40), ["-two-step", "on"])
        c.run(case(4)), d.run(case(4))
        assert lbm.hip_lib().LbmHipTwoStepRelease(None) == 0
        assert c.two_step().held == d.two_step().held == 0
        c.run(case(4)), c.close(), d.close()
    """)


@pytest.mark.parametrize("name", ["list-aa-pv-soa", "aa-soa"])
def test_arrays_in_use_stay_and_graphs_follow_them(stub, name):
    """Arrays that a Kernel() call is using are not given back, and a graph
    captured with arrays that were given back is captured anew."""
    stub(f"""
        name = {name!r}
        k = kernel(name, (20, 20, 20), ["-two-step", "on"])
        HOOK = C.CFUNCTYPE(None)
        hook = HOOK(lambda: lbm.hip_lib().LbmHipTwoStepRelease(None) and None)
        C.c_void_p.in_dll(S, "stub_hook").value = C.cast(hook, C.c_void_p).value
        k.run(case(8))
        C.c_void_p.in_dll(S, "stub_hook").value = None
        assert k.two_step().launches == 4 and k.two_step().held > 0
        k = kernel(name, (20, 20, 20), ["-two-step", "on", "-graph", "on"])
        for release, captures in ((False, 1), (False, 0), (True, 1), (False, 0)):
            if release:
                k.release_two_step()
            log()
            k.run(case(8))
            lines = log()
            assert lines.count("graph capture") == captures and lines.count("graph replay") == 1, lines
            assert k.two_step().launches == 4
    """)


@pytest.mark.parametrize("what", ["launch", "memset"])
def test_list_arrays_are_built_again_after_a_failure(stub, what):
    """A Kernel() call that could not fill the cell map or clear the second
    array fails, and the next call builds both before it uses them."""
    stub(f"""
        k = kernel("list-aa-pv-soa", (20, 20, 20), ["-two-step", "on"])
        what = {what!r}
        fail_launch("k_list_pair_map") if what == "launch" else fail_call("memset")
        try:
            k.run(case(4))
        except RuntimeError as e:
            assert ("cell map kernel" if what == "launch" else "hipMemset") in str(e), e
        else:
            raise AssertionError("no error")
        fail_launch("")
        fail_call("")
        log()
        k.run(case(4))
        lines = [line for line in log() if line.startswith("launch")]
        assert "k_list_pair_map" in lines[0] and all("k_pair" in line for line in lines[1:]), lines
    """)


@pytest.mark.parametrize("name", ["list-aa-pv-soa", "aa-soa"])
def test_arrays_are_taken_on_the_lattice_s_device(stub, name):
    """Kernel() called while another device is current allocates on the
    device that Init ran on, and leaves the current one as it was."""
    stub(f"""
        C.c_int.in_dll(S, "stub_devices").value = 2
        k = kernel({name!r}, (20, 20, 20), ["-two-step", "on"])
        S.hipSetDevice(1)
        k.run(case(4))
        lines = log()
        assert any("k_pair" in line for line in lines)
        assert all(line.endswith(" on 0") for line in lines if line.startswith("malloc")), lines
        d = C.c_int(-1)
        S.hipGetDevice(C.byref(d))
        assert d.value == 1
    """)


def test_plan_of_a_long_lattice_takes_no_time(stub):
    """Init's search for segments visits their distinct lengths alone: along
    8 million cells that is within the noise of Init, where a visit of every
    number of segments took 150 ms."""
    stub("""
        import time
        import numpy as np
        X = 8000000
        g = lbm.Geometry.from_mask(np.ones(X, dtype=np.int32), (X, 1, 1), (0, 0, 0))
        C.c_uint32.in_dll(S, "stub_count").value = X
        best = {"off": 1e9, "on": 1e9}
        for mode in ("off", "on") * 3:
            t = time.process_time()
            with lbm.Kernel("list-aa-pv-soa", g, ["-quiet", "-shadow", "lazy", "-prec", "fp16s", "-two-step", mode]) as k:
                best[mode] = min(best[mode], time.process_time() - t)
                assert k.two_step().segments == (1024 if mode == "on" else 0)
        assert best["on"] - best["off"] < 0.075, best
    """)
