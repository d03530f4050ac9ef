"""The Boys values of the light classes (vlxmi_device.hpp:boys_lds_fill, boys_lds)
compiled for the host, on the library's own table, against 113-bit arithmetic.

Bars, in units of one rounding (e = 2^-53 = 1.1e-16 relative):
* F_L below T = 40: the constant coefficient carries two roundings (the table's,
  the economisation's), the last step of the polynomial one, everything before it
  is damped by |x c_1| / F_L <= 0.1: 3.6 e = 4e-16 (the degree-8 polynomial's own
  error is below 1e-17);
* F_m, m < L: exp(-T) (three roundings and the coefficient sums, 4e-16) and
  F_{m+1} enter with weights that add to one; a step adds three roundings;
* at and above 40 the roundings are independent except that of 1/T, which enters
  F_m m times: 3 m + 2 independent ones of mean square e^2 / 4 and m coherent
  ones give a mean error below (1 + m / 2) 1e-16."""

import ctypes as C
import subprocess

import numpy as np
import pytest

from _util import PKG
from vlxmi import runtime

HIP = r"""
#pragma once
#include <cmath>
#include <cstddef>
#include <cstdint>
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_rcp(x) (double)(1.0f / (float)(x))
#define __builtin_amdgcn_rsq(x) (double)(1.0f / sqrtf((float)(x)))
#define __builtin_amdgcn_fence(a, b)
#define __builtin_amdgcn_wave_barrier()
#define __expf expf
struct Dim { unsigned x; };
static Dim threadIdx = {0}, blockDim = {1};
static inline void __syncthreads() {}
using std::exp;
using std::fma;
"""

SRC = r"""
#include "vlxmi_device.hpp"
typedef __float128 Q;

static Q qexp(Q x)                       // x <= 0
{
    int n = 0;
    while (x < -0.001Q) { x /= 2; ++n; }
    Q s = 1, t = 1;
    for (int k = 1; k < 16; ++k) { t *= x / k; s += t; }
    while (n--) s *= s;
    return s;
}

static void reference(int L, Q T, Q* F)
{
    const Q et = T > 200 ? 0 : qexp(-T);
    if (T < 40) {
        Q term = 1 / (Q)(2 * L + 1), sum = term;
        for (int k = 1; term > sum * 1e-33Q; ++k) { term *= 2 * T / (Q)(2 * L + 2 * k + 1); sum += term; }
        F[L] = et * sum;
        for (int m = L - 1; m >= 0; --m) F[m] = (2 * T * F[m + 1] + et) / (Q)(2 * m + 1);
    } else {                             // the part of F_0 beyond t = 1 is below 1e-18 of it
        Q y = 1 / std::sqrt((double)T);
        for (int k = 0; k < 4; ++k) y = y * (1.5Q - 0.5Q * T * y * y);
        F[0] = 0.886226925452758013649083741670572591Q * y;
        for (int m = 0; m < L; ++m) F[m + 1] = ((2 * m + 1) * F[m] - et) / (2 * T);
    }
}

template <int L>
static void errors(const double* table, const double* T, int n, double* out)
{
    static double lt[VLX_BOYS_LROWS * VLX_BOYS_LCOLS];
    vlxmi::boys_lds_fill<L>(table, lt);
    for (int i = 0; i < n; ++i) {
        double F[L + 1];
        Q R[L + 1];
        vlxmi::boys_lds<L>(T[i], lt, F);
        reference(L, (Q)T[i], R);
        for (int m = 0; m <= L; ++m) out[i * (L + 1) + m] = std::fabs((double)((F[m] - R[m]) / R[m]));
    }
}

extern "C" void boys_errors(int L, const double* table, const double* T, int n, double* out)
{
    switch (L) {
        case 0: return errors<0>(table, T, n, out);
        case 1: return errors<1>(table, T, n, out);
        case 2: return errors<2>(table, T, n, out);
        case 3: return errors<3>(table, T, n, out);
        case 4: return errors<4>(table, T, n, out);
    }
}
"""


@pytest.fixture(scope="module")
def errors(tmp_path_factory):
    d = tmp_path_factory.mktemp("boys")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    (d / "rows.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=gnu++17", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-I", str(d), "-I", PKG + "/csrc",
                    str(d / "rows.cpp"), "-o", str(d / "rows.so")], check=True)
    L = C.CDLL(str(d / "rows.so"))
    dp = C.POINTER(C.c_double)
    nr, nc, nf = C.c_uint32(), C.c_uint32(), C.c_uint32()
    lib = runtime.lib()
    lib.vlxmi_boys_table_size(C.byref(nr), C.byref(nc), C.byref(nf))
    table, ft = np.zeros((nr.value, nc.value)), np.zeros(nf.value)
    lib.vlxmi_boys_table_fill(table.ctypes.data_as(C.c_void_p), ft.ctypes.data_as(C.c_void_p))

    def run(order, T):
        out = np.zeros((T.size, order + 1))
        L.boys_errors(order, table.ctypes.data_as(dp), T.ctypes.data_as(dp), T.size, out.ctypes.data_as(dp))
        return out
    return run


@pytest.mark.parametrize("order", range(5))
def test_rows(errors, order):
    """Row ends and centres, small arguments and the whole range."""
    rng = np.random.default_rng(order)
    k = np.arange(200)
    T = np.concatenate([0.2 * k, np.nextafter(0.2 * (k + 1), 0), 0.2 * k + 0.1, rng.uniform(0, 1, 4000), rng.uniform(0, 40, 40000),
                        [0.0, 1e-300, 1e-12, np.nextafter(40.0, 0)]])
    e = errors(order, T[T < 40.0]).max(axis=0)
    assert e[order] <= 4e-16
    for m in range(order):
        assert e[m] <= 4e-16 + 3.3e-16 * (order - m), (m, e)


@pytest.mark.parametrize("order", range(5))
def test_large_arguments(errors, order):
    rng = np.random.default_rng(10 + order)
    T = np.concatenate([40.0 + rng.uniform(0, 40, 20000), np.exp(rng.uniform(np.log(40), np.log(1e6), 20000))])
    e = errors(order, T)
    assert (e.mean(axis=0) <= 1e-16 * (1 + 0.5 * np.arange(order + 1))).all(), e.mean(axis=0)
    assert e[:, order].max() <= 4e-16 * (order + 1)
