"""trt_collide of csrc/lbm_device.h, compiled for the host, against the
reference's form of the collision, which halves the sum and the difference of
an opposite pair before it relaxes them (src/BenchKernelD3Q19ListAaPv.c:387-463)."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

from conftest import PKG, ROOT

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not os.path.exists("/opt/rocm/include/hip"),
                                reason="needs g++ and the HIP headers")

SOURCE = """
#include <hip/hip_fp16.h>
template <class H> unsigned short __half_as_ushort(H);      // device code only
#include "lbm_device.h"
template <class R> static void run(R * f, const R * c)      // c: oe, oo, w0, w1, w2
{
	lbm::TrtConsts k{};
	k.oe = c[0]; k.oo = c[1]; k.w0 = c[2]; k.w1 = c[3]; k.w2 = c[4];
	k.w1x3 = c[5]; k.w1nh = c[6]; k.w2x3 = c[7]; k.w2nh = c[8];
	R v[19];
	for (int d = 0; d < 19; ++d) v[d] = f[d];
	lbm::trt_collide(v, lbm::trt_cast<R>(k));
	for (int d = 0; d < 19; ++d) f[d] = v[d];
}
extern "C" void collide_f32(float * f, const float * c, int n) { while (n--) run(f + 19 * n, c); }
extern "C" void collide_f64(double * f, const double * c, int n) { while (n--) run(f + 19 * n, c); }
"""

N, S, E, W, NE, SE, NW, SW, T, TN, TE, TW, TS, B, BS, BN, BW, BE, CC = range(19)


@pytest.fixture(scope="module")
def collide(tmp_path_factory):
    path = tmp_path_factory.mktemp("collide")
    src, out = str(path / "collide.cpp"), str(path / "collide.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-ffp-contract=off", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(PKG, "csrc"), src,
                    "-o", out], check=True, capture_output=True)
    lib = C.CDLL(out)

    def run(f, c):
        g = np.ascontiguousarray(f.copy())
        fn = lib.collide_f32 if f.dtype == np.float32 else lib.collide_f64
        fn(C.c_void_p(g.ctypes.data), C.c_void_p(c.ctypes.data), len(g))
        return g
    return run


def _consts(omega, magic, dtype):
    w1, w2 = 1.0 / 18.0, 1.0 / 36.0
    return np.array([omega, 1.0 / (0.5 + magic / (1.0 / omega - 0.5)), 1.0 / 3.0, w1, w2, w1 * 3.0, w1 * 9.0 / 2.0,
                     w2 * 3.0, w2 * 9.0 / 2.0], dtype=dtype)


def _halved(f, c):
    """The reference's operations in its order, in f's type."""
    t = f.dtype.type
    oe, oo, w0, w1, w2, w1x3, w1nh, w2x3, w2nh = (t(v) for v in c)
    p = [f[:, d] for d in range(19)]
    ux = p[E] + p[NE] + p[SE] + p[TE] + p[BE] - p[W] - p[NW] - p[SW] - p[TW] - p[BW]
    uy = p[N] + p[NE] + p[NW] + p[TN] + p[BN] - p[S] - p[SE] - p[SW] - p[TS] - p[BS]
    uz = p[T] + p[TE] + p[TW] + p[TN] + p[TS] - p[B] - p[BE] - p[BW] - p[BN] - p[BS]
    dens = (p[CC] + p[N] + p[E] + p[S] + p[W] + p[NE] + p[SE] + p[SW] + p[NW]
            + p[T] + p[TN] + p[TE] + p[TS] + p[TW] + p[B] + p[BN] + p[BE] + p[BS] + p[BW])
    dirn = dens - (ux * ux + uy * uy + uz * uz) * t(3.0) / t(2.0)
    q = np.empty_like(f)
    q[:, CC] = p[CC] - oe * (p[CC] - w0 * dirn)
    for a, b, u, wi, wnh, wx3 in ((N, S, uy, w1, w1nh, w1x3), (E, W, ux, w1, w1nh, w1x3), (T, B, uz, w1, w1nh, w1x3),
                                  (NW, SE, -ux + uy, w2, w2nh, w2x3), (NE, SW, ux + uy, w2, w2nh, w2x3),
                                  (TW, BE, -ux + uz, w2, w2nh, w2x3), (TE, BW, ux + uz, w2, w2nh, w2x3),
                                  (TS, BN, -uy + uz, w2, w2nh, w2x3), (TN, BS, uy + uz, w2, w2nh, w2x3)):
        ev = oe * (t(0.5) * (p[a] + p[b]) - u * u * wnh - wi * dirn)
        od = oo * (t(0.5) * (p[a] - p[b]) - u * wx3)
        q[:, a] = p[a] - ev - od
        q[:, b] = p[b] - ev + od
    return q


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("size", [1e-1, 1e-5, 1e-9])
def test_same_bits_as_the_halved_form(collide, dtype, size):
    # deviations; products of two of them at 1e-9 are normal in FP32 too
    f = (np.random.default_rng(3).standard_normal((4000, 19)) * size).astype(dtype)
    for omega, magic in ((1.2, 3.0 / 16.0), (0.5, 1.0 / 12.0), (1.95, 1.0 / 4.0)):
        c = _consts(omega, magic, dtype)
        assert np.array_equal(collide(f, c), _halved(f, c))


def test_subnormal_deviations(collide):
    """Values of up to 2^16 smallest subnormals: sums are exact there, squares
    vanish, and every product rounds by half a unit (of the smallest
    subnormal).  With rates below 2 a pair's two parts are each off by
    rate / 4 + 1/2 < 1 (halved before: rate * (1/2 + 1/2) + 1/2 < 2.5), and a
    value by twice that; the rest value has two products, 2 * 1/2 + 1/2."""
    unit = float(np.float32(2.0) ** -149)
    f = (np.random.default_rng(4).integers(-65536, 65537, (4000, 19)) * unit).astype(np.float32)
    f[0, :] = 0.0
    f[0, N] = np.float32(3 * unit)
    for omega, magic in ((1.2, 3.0 / 16.0), (1.6, 1.0 / 4.0), (1.95, 1.0 / 12.0)):
        c = _consts(omega, magic, np.float32)
        new, halved = collide(f, c).astype(np.float64), _halved(f, c).astype(np.float64)
        exact = _halved(f.astype(np.float64), c.astype(np.float64))
        # the equilibrium's squares are below 2^-250 in the exact result
        assert np.abs(new - exact).max() / unit <= 2.0
        assert np.abs(halved - exact).max() / unit <= 5.0
        assert np.abs(new - exact).max() <= np.abs(halved - exact).max()
        assert np.abs(new - halved).max() / unit <= 7.0
