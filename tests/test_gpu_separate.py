"""GPU parity of the separate even and odd launches as they run by default,
with -two-step off alone: lattices above the two-step launch's window, calls
with launch events and calls short of memory take them, while the default of
smaller lattices is the two-step launch.  -two-step off is no option of the
separate launches, so their own defaults (block shapes, non-temporal accesses,
odd-step pairs) apply.

Bar: node views bit-identical to the oracle, or to the golden hash at 256^3.
"""
import hashlib

import numpy as np
import pytest

from conftest import golden

pytestmark = pytest.mark.gpu

LAM = 3 / 16
OFF = ["-two-step", "off", "-quiet"]
NAMES = ["list-aa-pv-soa", "aa-soa"]


def _run(lbm, name, geo, runs, omega, F, args):
    with lbm.Kernel(name, geo, OFF + list(args)) as k:
        k.set_initial_weights()
        for steps in runs:
            k.run(lbm.case_data(omega=omega, xforce=F, iterations=steps))
            assert k.two_step().launches == 0 and k.two_step().planned == 0
        return k.dump()


@pytest.mark.parametrize("name", NAMES)
def test_ragged_lattice(lbm, oracle, name):
    geo = lbm.Geometry.from_string("porous-3-0.75-9", (40, 37, 70))
    want, _ = oracle.list_run(geo.mask.reshape(-1), geo.dims, geo.periodic, 30, 1.25, 3e-5, vsize=1)
    assert np.array_equal(_run(lbm, name, geo, [20, 10], 1.25, 3e-5, []), want)


@pytest.mark.parametrize("name", NAMES)
def test_large_lattice(lbm, oracle, name):
    # above the size where the even step runs one 512-thread block per CU
    geo = lbm.Geometry.from_string("porous-4-0.85-5", (176, 128, 128))
    assert geo.n_fluid > 16 * 512 * 256
    print(f"{name} 176x128x128 nFluid={geo.n_fluid}", flush=True)
    want, _ = oracle.list_run(geo.mask.reshape(-1), geo.dims, geo.periodic, 10, 1.3, 2e-5, vsize=1)
    assert np.array_equal(_run(lbm, name, geo, [10], 1.3, 2e-5, []), want)


@pytest.mark.parametrize("prec", ["fp32s", "fp16s"])
def test_aa_narrow_over_256_mib(lbm, prec):
    """aa-soa above 256 MiB of narrow storage: non-temporal even step at full
    occupancy, and in FP32 the odd step over pairs of z cells; the same bits
    as the cache-friendly launches and as the two-step launch."""
    geo = lbm.Geometry.from_string("channel", (80, 256, 256), (1, 0, 0))   # 309 MiB in FP16, 514 in FP32
    base = ["-prec", prec, "-lambda", repr(LAM)]
    print(f"aa 80x256x256 -prec {prec}", flush=True)
    got = _run(lbm, "aa-soa", geo, [20], 1.2, 1e-5, base)
    assert np.array_equal(got, _run(lbm, "aa-soa", geo, [20], 1.2, 1e-5,
                                    base + ["-nt", "off", "-even-cap", "on", "-odd-pairs", "off"]))
    with lbm.Kernel("aa-soa", geo, base + ["-quiet"]) as k:
        k.set_initial_weights()
        k.run(lbm.case_data(omega=1.2, xforce=1e-5, iterations=20))
        assert k.two_step().launches == 10
        assert np.array_equal(got, k.dump())


@pytest.mark.parametrize("name", NAMES)
def test_graph_replay(lbm, name):
    geo = lbm.Geometry.from_string("porous-3-0.7-5", (40, 36, 34))
    args = OFF + ["-lambda", repr(LAM)]
    with lbm.Kernel(name, geo, args + ["-graph", "on"]) as kg, lbm.Kernel(name, geo, args) as kp:
        for k in (kg, kp):
            k.set_initial_weights()
        x, y, z = [int(v) for v in np.argwhere(geo.mask != 0)[5][::-1]]
        for steps, omega in [(20, 1.2), (20, 1.2), (20, 1.2), (30, 0.9), (20, 1.2)]:
            for k in (kg, kp):
                k.run(lbm.case_data(omega=omega, xforce=2e-5, iterations=steps))
                assert k.two_step().launches == 0
            assert np.array_equal(kg.dump(), kp.dump()), (steps, omega)
            for k in (kg, kp):                      # host work between the replays
                v = k.get_node(x, y, z)
                k.set_node(x, y, z, [a * (1 + 1e-3) for a in v])


def test_porous256_500_steps(lbm):
    g = golden("porous256_500.npz")
    geo = lbm.Geometry.from_string("porous-6-0.8-42", (256, 256, 256))
    print("porous256 list-aa-pv-soa 500 steps, separate launches", flush=True)
    d = _run(lbm, "list-aa-pv-soa", geo, [int(g["steps"])], float(g["omega"]), float(g["xforce"]), ["-lambda", "0.1875"])
    assert hashlib.sha256(np.ascontiguousarray(d).tobytes()).hexdigest() == str(g["orc_l316_sha"])


@pytest.mark.parametrize("name", NAMES)
def test_fp32_mixed_with_two_step_launches(lbm, oracle, name):
    """Calls in two-step and, with launch events, in separate launches in turn
    end in the oracle's state (FP32; the other types are covered beside the
    two-step launch)."""
    dims, per, runs = (17, 15, 35), (1, 0, 0), [2, 2, 6, 4, 2]
    m = (np.random.default_rng(5).random((dims[2], dims[1], dims[0])) < 0.8).astype(np.int32)
    m[0] = m[-1] = 0
    m[:, 0] = m[:, -1] = 0
    m = np.ascontiguousarray(m.reshape(-1))
    geo = lbm.Geometry.from_mask(m, dims, per)
    with lbm.Kernel(name, geo, ["-lambda", repr(LAM), "-prec", "fp32s", "-quiet", "-two-step", "on"]) as k:
        k.set_initial_weights()
        for call, steps in enumerate(runs):
            k.set_launch_events(call in (1, 3))
            k.run(lbm.case_data(omega=1.2, xforce=1e-4, iterations=steps))
            assert k.two_step().launches == (0 if call in (1, 3) else steps // 2)
        got = k.dump()
    run = (lambda *a, **kw: oracle.list_run_shifted(*a, **kw)[0]) if name == "list-aa-pv-soa" else oracle.aa_run_shifted
    assert np.array_equal(got, run(m, dims, per, runs, 1.2, 1e-4, "fp32s", magic=LAM))
