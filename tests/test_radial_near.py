"""The near-pair kernels of the molecule records and the fast exponential (csrc/pairs.h, csrc/common.h) on the CPU.

The device functions are compiled for the host from the sources (the two hardware approximations they
call are replaced by correctly rounded ones) and compared with float64 incomplete gamma functions:
B_n = (2a/sqrt(pi)) (2a^2)^n F_n(s), F_n(s) = gamma(n + 1/2) P(n + 1/2, s) / (2 s^(n+1/2)), s = (a r)^2.

Bounds.  A record's G1, G2 are differences of two B_n, rounded once: half an ulp of the result, 2^-24.  With a
screening below 6, B_n takes exp(-s) in FP32 (one ulp: two units 2^-24) and the terms of its series from the
sixth on (a fifth of the sum at s = 6), whose Horner steps round about a dozen units; the rest is FP64: 4.5
units 2^-24 of each B_n at most, and 2^-26 on average over a narrow range of s (a fifth of one coefficient's
rounding), since a rigid molecule repeats the same s everywhere.  With a screening at or above 6 that B_n
comes from the FP32 recursion B_n = ((2n-1) B_(n-1) - c) / r^2: erf, 1/sqrt and each step round by 2^-24 a few
times, (4n + 4) 2^-24 of B_n at most.  exp(-s): half an ulp from exp2 and half from the last step.
"""

import ctypes as C
import os
import subprocess

import numpy as np
import pytest
from scipy.special import gamma, gammainc

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pgm-jax_amd", "csrc")
EPS = 2.0**-24

SHIM = r"""
#include <cmath>
#include <hip/hip_runtime.h>
static inline float host_exp2(float x) { return (float)std::exp2((double)x); }
static inline float host_rsq(float x) { return (float)(1.0 / std::sqrt((double)x)); }
static inline float host_rcp(float x) { return (float)(1.0 / (double)x); }
static inline float rsqrtf(float x) { return host_rsq(x); }
#define __builtin_amdgcn_exp2f host_exp2
#define __builtin_amdgcn_rsqf host_rsq
#define __builtin_amdgcn_rcpf host_rcp
// what the kernels of the headers name (never called here)
#define __builtin_amdgcn_fence(...)
#define __builtin_amdgcn_wave_barrier()
#define __builtin_amdgcn_readfirstlane(x) (x)
#define __launch_bounds__(...)
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_load(p, ...) (*(p))
struct Dim { unsigned x, y, z; };
static Dim threadIdx, blockIdx, blockDim, gridDim;
static inline void __syncthreads() {}
template <typename T> T __shfl_xor(T v, int, int) { return v; }
template <typename T> T __shfl_up(T v, int, int) { return v; }
template <typename T> T __shfl(T v, int, int) { return v; }
static inline unsigned long long __ballot(bool b) { return b; }
static inline int __popc(unsigned x) { return __builtin_popcount(x); }
static inline int __popcll(unsigned long long x) { return __builtin_popcountll(x); }
static inline int __ffs(int x) { return __builtin_ffs(x); }
static inline int atomicMax(int *p, int v) { return *p = *p > v ? *p : v; }
static inline unsigned atomicOr(unsigned *p, unsigned v) { return *p |= v; }
static inline int min(int a, int b) { return a < b ? a : b; }
static inline int max(int a, int b) { return a > b ? a : b; }
static inline int __float_as_int(float f) { return (int)f; }
using std::erf; using std::erfc; using std::exp; using std::fabs; using std::floor; using std::fmax; using std::rint; using std::sqrt;
namespace pgm { struct Ext3 { double x, y, z; }; }
#include "pairs.h"
namespace pgm { unsigned mol_bits[1]; }
using namespace pgm;

// G1, G2 that the record pass writes for a pair at distance r of two atoms with Gaussian radii squared w each.
template <typename real> static void record(int n, const double *w, const double *r, double beta, double *out) {
    Box box{};
    for (int a = 0; a < 3; ++a) box.h[4 * a] = 10.0, box.hinv[4 * a] = box.inv_diag[a] = 0.1;
    for (int i = 0; i < n; ++i) {
        double4 xr[6] = {};
        xr[0].w = xr[3].w = w[i];
        xr[3].x = r[i];
        real mg[MCH * MOL_REC] = {};
        mol_near_pair<real>(0, 1, 0, 0, xr, box, 1e30, beta, MCH, mg);
        out[2 * i] = mg[mslot<real>(0, 0)];
        out[2 * i + 1] = mg[mslot<real>(0, 3)];
    }
}
extern "C" void record_f32(int n, const double *w, const double *r, double beta, double *out) { record<float>(n, w, r, beta, out); }
extern "C" void fast_exp(int n, const float *s, float *out) {
    for (int i = 0; i < n; ++i) out[i] = exp_neg(s[i]);
}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("radial")
    src, lib = d / "shim.cpp", d / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["/opt/rocm/llvm/bin/clang++", "-O1", "-std=c++17", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I" + CSRC, str(src), "-o", str(lib)], check=True)
    return C.CDLL(str(lib))


def _p(a):
    return a.ctypes.data_as(C.c_void_p)


def _B(a, r, n):
    s = (a * r) ** 2
    F = 0.5 * gamma(n + 0.5) * gammainc(n + 0.5, s) / s ** (n + 0.5)
    return 2.0 * a / np.sqrt(np.pi) * (2.0 * a * a) ** n * F


# (a r)^2 of the wider screening: inside each branch and either side of its ends
@pytest.mark.parametrize("lo, hi", [(1e-3, 0.5), (0.5, 1.2), (1.2, 3.0), (3.0, 5.0), (5.0, 5.6), (5.6, 5.9999), (6.0001, 20.0)])
def test_record_near_pairs(host, lo, hi):
    rng = np.random.default_rng(1)
    n, beta = 4000, 4.0
    r = rng.uniform(0.05, 0.24, n)  # (beta r)^2 < 1
    a = np.sqrt(rng.uniform(lo, hi, n)) / r
    w = 1.0 / (4.0 * a * a)  # a = 1 / sqrt(2 (w + w))
    out = np.empty((n, 2))
    host.record_f32(n, _p(w), _p(r), C.c_double(beta), _p(out))
    for k in (1, 2):
        Ba, Bb = _B(a, r, k), _B(beta, r, k)
        ref = Ba - Bb
        size = Ba + Bb
        bound = EPS * np.abs(ref) + (4 * k + 4 if lo > 6.0 else 4.5) * EPS * size
        err = out[:, k - 1] - ref
        assert np.all(np.abs(err) <= bound), (k, (np.abs(err) / bound).max())
        assert abs(np.mean(err / size)) <= 2.0**-26, (k, np.mean(err / size))


def test_fast_exponential(host):
    rng = np.random.default_rng(2)
    s = np.concatenate([rng.uniform(0.0, 87.0, 200000), rng.uniform(0.0, 2.0, 100000), [0.0, 1.0]]).astype(np.float32)
    e = np.empty_like(s)
    host.fast_exp(len(s), _p(s), _p(e))
    ref = np.exp(-s.astype(np.float64))
    err = e.astype(np.float64) - ref
    assert np.all(np.abs(err) <= np.spacing(ref.astype(np.float32)).astype(np.float64))
    assert abs(np.mean(err / ref)) < 1e-9  # 0.3 ulp rms over 3e5 values: unbiased to 6e-11
