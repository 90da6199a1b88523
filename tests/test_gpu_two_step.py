"""GPU parity of the two-step launch (-two-step): an even and an odd step of a
lattice in one launch over tiles of the y-z plane.

Bar: node views bit-identical to the oracle (the same arithmetic per node), at
the edges of every tile shape and of its segments along x, on random masks
(bounce-back links everywhere), over two Kernel() calls of which the first has
an odd number of step pairs.  Lattices whose boundary the launch does not
cover keep the separate launches.
"""
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAM = 3 / 16
RUNS = [2, 4]
WALLS, PERIODIC, OPEN = (1, 0, 0), (1, 1, 1), (0, 0, 0)
# dims, boundary, and the tile shape (y, z) the launch takes there per type
CASES = [
    ((1, 14, 33), PERIODIC), ((2, 13, 32), PERIODIC), ((3, 5, 64), WALLS), ((4, 1, 40), PERIODIC),
    ((5, 16, 1), PERIODIC), ((7, 6, 35), OPEN), ((20, 27, 66), WALLS), ((33, 29, 31), PERIODIC),
    ((92, 127, 5), WALLS), ((74, 66, 67), PERIODIC), ((58, 58, 70), WALLS), ((80, 80, 80), WALLS),
]
NARROW = [((68, 31, 105), PERIODIC), ((11, 138, 102), WALLS), ((105, 66, 79), PERIODIC), ((63, 106, 101), WALLS),
          ((135, 16, 40), PERIODIC)]


def _mask(dims, per, seed):
    """About 80 % fluid; walls on the non-periodic faces unless all are open."""
    rng = np.random.default_rng(seed)
    m = (rng.random((dims[2], dims[1], dims[0])) < 0.8).astype(np.int32)
    m[dims[2] // 2, dims[1] // 2, dims[0] // 2] = 1
    if per == WALLS:
        m[0] = m[-1] = 0
        m[:, 0] = m[:, -1] = 0
        m[dims[2] // 2, dims[1] // 2, dims[0] // 2] = 1
    return np.ascontiguousarray(m.reshape(-1))


def _run(lbm, name, geo, prec, args, omega, F, runs=RUNS, nodes=None):
    with lbm.Kernel(name, geo, ["-lambda", repr(LAM), "-prec", prec, "-two-step", "on"] + list(args)) as k:
        if nodes is None:
            k.set_initial_weights()
        else:
            k.load(nodes)
        for n in runs:
            k.run(lbm.case_data(omega=omega, xforce=F, iterations=n))
        return k.dump()


def _oracle(oracle, name, mask, dims, per, prec, omega, F, force_on=True):
    if prec == "fp64":
        run = oracle.list_run if name == "list-aa-pv-soa" else oracle.aa_run
        return run(mask, dims, per, sum(RUNS), omega, F, magic=LAM, force_on=force_on)[0]
    if name == "list-aa-pv-soa":
        return oracle.list_run_shifted(mask, dims, per, RUNS, omega, F, prec, magic=LAM, force_on=force_on)[0]
    return oracle.aa_run_shifted(mask, dims, per, RUNS, omega, F, prec, magic=LAM, force_on=force_on)


@pytest.mark.parametrize("prec", ["fp64", "fp32s", "fp16s"])
@pytest.mark.parametrize("name", ["list-aa-pv-soa", "aa-soa"])
def test_tiles_bitexact(lbm, oracle, capfd, name, prec):
    tiles = set()
    for i, (dims, per) in enumerate(CASES + ([] if prec == "fp64" else NARROW)):
        if name == "aa-soa" and per == OPEN:
            continue                                   # ghost cells: separate launches
        mask = _mask(dims, per, 100 + i)
        geo = lbm.Geometry.from_mask(mask, dims, per)
        force_on = i % 3 != 1
        print(f"{name} {prec} {dims} {per} force {force_on}", flush=True)
        got = _run(lbm, name, geo, prec, ["-force", "on" if force_on else "off"], 1.3, 1e-4)
        said = re.search(r"two-step launch: +tiles of (\d+) x (\d+)", capfd.readouterr().out)
        assert said, f"{dims}: no two-step launch"
        tiles.add((int(said.group(1)), int(said.group(2))))
        want = _oracle(oracle, name, mask, dims, per, prec, 1.3, 1e-4, force_on)
        assert np.array_equal(got, want), f"{dims}: max diff {np.abs(got - want).max()}"
    assert tiles == {(13, 32), (5, 32)} | (set() if prec == "fp64" else {(13, 64), (18, 48), (28, 32)})


@pytest.mark.parametrize("name,per", [("aa-soa", OPEN), ("aa-soa", (0, 1, 1)), ("list-aa-pv-soa", (1, 0, 0)),
                                      ("list-aa-pv-soa", (0, 1, 1))])
def test_open_faces_keep_the_separate_launches(lbm, oracle, capfd, name, per):
    dims = (9, 15, 34)
    mask = _mask(dims, OPEN, 7)                        # fluid on every face
    geo = lbm.Geometry.from_mask(mask, dims, per)
    got = _run(lbm, name, geo, "fp64", [], 1.1, 1e-4)
    assert "two-step launch" not in capfd.readouterr().out
    assert np.array_equal(got, _oracle(oracle, name, mask, dims, per, "fp64", 1.1, 1e-4))


@pytest.mark.parametrize("name", ["list-aa-pv-soa", "aa-soa"])
@pytest.mark.parametrize("prec", ["fp64", "fp16s"])
def test_mixed_with_separate_launches(lbm, name, prec):
    """Calls in two-step launches, in separate ones (per-launch events) and
    from a replayed graph in turn, and SetNode between them, end in the state
    of separate launches alone."""
    dims, per = (17, 15, 35), WALLS
    geo = lbm.Geometry.from_mask(_mask(dims, per, 5), dims, per)
    out = []
    for args, events in ((["-two-step", "on"], True), (["-two-step", "on", "-graph", "on"], False),
                         (["-two-step", "off"], False)):
        with lbm.Kernel(name, geo, ["-lambda", repr(LAM), "-prec", prec, "-quiet"] + args) as k:
            k.set_initial_weights()
            for call, steps in enumerate((2, 2, 6, 4, 2, 2)):
                k.set_launch_events(events and call in (1, 3))
                k.run(lbm.case_data(omega=1.2, xforce=1e-4, iterations=steps))
                if call == 3:
                    v = k.dump()
                    k.load(v * 1.01)
            out.append((k.dump(), k.moments()))
    for nodes, moments in out[:2]:
        assert np.array_equal(nodes, out[2][0])
        assert moments == out[2][1]


@pytest.mark.parametrize("graph", ["off", "on"])
@pytest.mark.parametrize("name", ["list-aa-pv-soa", "aa-soa"])
def test_arrays_given_back_between_calls(lbm, oracle, name, graph):
    """Calls before and after the arrays were given back, with SetNode between
    two of them, end in the oracle's state."""
    dims, per = (17, 15, 35), WALLS
    mask = _mask(dims, per, 5)
    geo = lbm.Geometry.from_mask(mask, dims, per)
    with lbm.Kernel(name, geo, ["-lambda", repr(LAM), "-two-step", "on", "-graph", graph, "-quiet"]) as k:
        k.set_initial_weights()
        for call in range(4):
            k.run(lbm.case_data(omega=1.3, xforce=1e-4, iterations=6))
            info = k.two_step()
            assert info.held == info.bytes > 0 and info.launches >= 2
            if call != 1:
                k.release_two_step()
                assert k.two_step().held == 0
            if call == 2:
                k.load(k.dump())
        run = oracle.list_run if name == "list-aa-pv-soa" else oracle.aa_run
        assert np.array_equal(k.dump(), run(mask, dims, per, 24, 1.3, 1e-4, magic=LAM, force_on=True)[0])


@pytest.mark.parametrize("prec,plane", [("fp64", 76_695_840), ("fp32s", 153_391_680), ("fp16s", 226_050_896)])
def test_offsets_up_to_the_window(lbm, oracle, prec, plane):
    """Direction planes as far apart as the launch takes them (the list
    kernel's padding): a store reaches up to six planes behind the window's
    base, 3.7 GB in FP64 and FP32 and 2.7 GB in FP16, where 2^32 PDFs end the
    range.  One padding step further the steps are launched one by one, with
    the same results."""
    dims, per = (17, 15, 35), WALLS
    mask = _mask(dims, per, 5)
    geo = lbm.Geometry.from_mask(mask, dims, per)
    want = _oracle(oracle, "list-aa-pv-soa", mask, dims, per, prec, 1.3, 1e-4)
    elem = {"fp64": 8, "fp32s": 4, "fp16s": 2}[prec]
    assert 6 * plane * elem > 2**31 and 19 * plane < 2**32
    for n in (plane, plane + 16):
        over = 7 * n * elem > 0xfffffff0
        if 19 * n > 2**32 - 1:
            continue
        print(f"list {prec} planes of {n} values", flush=True)
        with lbm.Kernel("list-aa-pv-soa", geo, ["-lambda", repr(LAM), "-prec", prec, "-two-step", "on", "-quiet",
                                                "-shadow", "lazy", "-pad", f"{8 * n}+0"]) as k:
            assert k.list_info().nCells == n
            assert lbm.hip_lib().LbmHipSyncShadow(k.kd) == 0
            k.set_initial_weights()
            for steps in RUNS:
                k.run(lbm.case_data(omega=1.3, xforce=1e-4, iterations=steps))
                assert k.two_step().launches == (0 if over else steps // 2)
            assert np.array_equal(k.dump(), want), (prec, n)
