// Device-side constants and the Boys function for the J/K kernels (gfx950).
//
// Boys function F_m(T) = int_0^1 t^(2m) exp(-T t^2) dt, m = 0..L (L <= 8).
// The reference calls VeloxChem's gpu::computeBoysFunction(F, T, L,
// boys_func_table, boys_func_ft) (gen_coulomb.py:257-259); that function is not
// in the reference tree, so the table format below is this project's own:
//
//   boys_func_table: VLX_BOYS_NROW fine rows x VLX_BOYS_NCOL doubles, row k
//     holds F_0..F_14 at T_k = k * VLX_BOYS_DT (columns 0..14) and exp(-T_k)
//     (column 15); one 128-byte row per grid point; then VLX_BOYS_CROWS coarse
//     rows (below).
//   boys_func_ft: 1/(2m+1), m = 0..31 (the generated kernels fold these
//     constants at compile time; the array is kept for the signature).
//
// For T < VLX_BOYS_TMAX: a 6-term Taylor expansion of F_L about the nearest
// grid point, |T - T_k| <= DT/2 = 0.01, so the remainder is below
// F_L * 0.01^6 / 6! = 1.4e-15 F_L (F_{m+1} <= F_m); the six coefficients
// F_L..F_{L+5}(T_k) are contiguous, three 16-byte loads per lane -- the table
// gather is what limits the light classes, so the row is kept that short.
// exp(-T): for L <= 4 from the device exp (those classes are bound by the
// table gathers, not by instructions); for L >= 5, whose kernels re-evaluate
// the prologue once per component pass and are not gather-bound, as
// exp(-T_k) (column 15) times a 7-term Taylor of exp(T_k - T) (remainder
// < 0.01^7/7! = 2e-18).  Then downward recursion
// F_{m} = (2T F_{m+1} + exp(-T)) / (2m+1).
// For T >= VLX_BOYS_TMAX: F_0 = sqrt(pi/T)/2 (Newton-refined 1/sqrt) and upward recursion
// F_{m+1} = ((2m+1) F_m - exp(-T)) / (2T); there exp(-T) < 5e-18 and the
// single-precision hardware exponential is accurate enough for it.
//
// Coarse rows (after the fine table, VLX_BOYS_CROWS rows of VLX_BOYS_NCOL
// doubles): F_0..F_15 at T_k = k * VLX_BOYS_CDT.  No kernel reads them; they
// stay because the layout is public (callers size and fill their tables with
// vlxmi_boys_table_size / _fill, and check it).  Kernels of the light classes
// make their own rows in LDS from every tenth fine row, once per workgroup
// (boys_lds_fill), and evaluate F_L from there: no global gather per quartet.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "vlxmi_status.h"

// List-order validation the class launchers run when it is switched on
// (vlxmi_lists.cpp).
extern "C" int vlxmi_list_validation(void);
extern "C" int vlxmi_validate_j_list(uint32_t la, uint32_t lb, const uint32_t* first, const uint32_t* second,
                                     const double* mat_Q, const double* mat_D, uint32_t count, void* stream);
extern "C" int vlxmi_validate_ik_list(uint32_t la, uint32_t lc, const uint32_t* ik_i, const uint32_t* ik_k,
                                      uint32_t count, void* stream);
extern "C" int vlxmi_validate_k_csr(uint32_t la, uint32_t lb, uint32_t count_a, const uint32_t* displs,
                                    const uint32_t* counts, const double* Q, const uint32_t* D_inds, void* stream);

// Ket-split partial sums of the launchers (vlxmi_workspace.cpp, vlxmi_capi.cpp).
extern "C" int vlxmi_ket_workspace(size_t ndoubles, void* stream, double** out);
extern "C" int vlxmi_try_workspace(size_t ndoubles, void* stream, double** out);
extern "C" void vlxmi_workspace_hold(int on);
extern "C" int vlxmi_ket_split_reduce(const double* part, uint32_t nsplit, uint32_t count, double* out,
                                      void* stream);

namespace vlxmi {
// Held by a launcher from taking its workspace to enqueueing the reduction that
// reads it: another thread on the same stream neither regrows the buffer nor
// puts its own partial sums between the two launches.
struct WorkspaceHold {
    WorkspaceHold() { vlxmi_workspace_hold(1); }
    ~WorkspaceHold() { vlxmi_workspace_hold(0); }
    WorkspaceHold(const WorkspaceHold&) = delete;
    WorkspaceHold& operator=(const WorkspaceHold&) = delete;
};
}  // namespace vlxmi

#define VLX_BOYS_NCOL 16
#define VLX_BOYS_NROW 2001
#define VLX_BOYS_DT 0.02
#define VLX_BOYS_INV_DT 50.0
#define VLX_BOYS_TMAX 40.0
#define VLX_BOYS_CROWS 101
#define VLX_BOYS_CDT 0.4
#define VLX_BOYS_LROWS 200
#define VLX_BOYS_LCOLS 10
#define VLX_BOYS_COARSE_OFF (VLX_BOYS_NROW * VLX_BOYS_NCOL)

#define MATH_CONST_PI 3.14159265358979323846
#define MATH_CONST_INV_PI 0.31830988618379067154

// one wavefront per workgroup for both kernel families
#define TILE_SIZE_J 64
#define TILE_SIZE_K 64

namespace vlxmi {

// Orders one wavefront's LDS accesses around this point: the ket tile a
// wavefront stages is read only by its own lanes, so kernels that run several
// independent wavefronts per workgroup synchronise each wavefront on its own.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The sum of v over the workgroup's W wavefronts, lane by lane, in wavefront
// order (buf: W * 64 doubles of LDS).  Every thread calls it.
template <int W>
__device__ __forceinline__ double team_sum(double v, double* buf)
{
    __syncthreads();
    buf[threadIdx.x] = v;
    __syncthreads();
    double s = buf[threadIdx.x & 63];
#pragma unroll
    for (int k = 1; k < W; ++k) s += buf[k * 64 + (threadIdx.x & 63)];
    return s;
}

// 1/x and 1/sqrt(x) for positive, normal x well inside the double range (the
// Gaussian exponent sums and Boys arguments these are used on): the hardware
// estimate (relative error below 2^-22) refined by one third-order step, which
// cubes that error, so the result is within a few ulp; no denormal/overflow
// scaling.
__device__ __forceinline__ double rcp_nr(double x)
{
    const double r = __builtin_amdgcn_rcp(x);
    const double e = fma(-x, r, 1.0);
    return fma(r, fma(e, e, e), r);
}

__device__ __forceinline__ double rsq_nr(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}

template <int L>
__device__ __forceinline__ void boys(double T, const double* __restrict__ table, double* F)
{
    if (T < VLX_BOYS_TMAX) {
        const int k = (int)(T * VLX_BOYS_INV_DT + 0.5);
        const double nd = (double)k * VLX_BOYS_DT - T;   // -(T - T_k)
        const double* row = table + k * VLX_BOYS_NCOL;
        // F_L(T) = sum_j F_{L+j}(T_k) (-d)^j / j!, j = 0..5 (Horner)
        double s = row[L + 5];
        s = fma(s, nd * (1.0 / 5.0), row[L + 4]);
        s = fma(s, nd * (1.0 / 4.0), row[L + 3]);
        s = fma(s, nd * (1.0 / 3.0), row[L + 2]);
        s = fma(s, nd * (1.0 / 2.0), row[L + 1]);
        s = fma(s, nd, row[L]);
        F[L] = s;
        if (L > 0) {
            double et;
            if constexpr (L >= 5) {
                double e = 1.0 / 720.0;
                e = fma(e, nd, 1.0 / 120.0);
                e = fma(e, nd, 1.0 / 24.0);
                e = fma(e, nd, 1.0 / 6.0);
                e = fma(e, nd, 0.5);
                e = fma(e, nd, 1.0);
                e = fma(e, nd, 1.0);
                et = row[15] * e;
            } else {
                et = exp(-T);
            }
            const double T2 = 2.0 * T;
#pragma unroll
            for (int m = L - 1; m >= 0; --m) F[m] = fma(T2, F[m + 1], et) * (1.0 / (2.0 * m + 1.0));
        }
    } else {
        const double inv_T = rcp_nr(T);
        F[0] = (0.5 * 1.77245385090551602730) * rsq_nr(T);   // sqrt(pi/T) / 2
        if (L > 0) {
            const double et = (double)__expf(-(float)T);
            const double h = 0.5 * inv_T;
#pragma unroll
            for (int m = 0; m < L; ++m) F[m + 1] = ((2.0 * m + 1.0) * F[m] - et) * h;
        }
    }
}

// The LDS rows of order L: row k covers T in [k/5, (k+1)/5), T_k = k/5 + 1/10 (a
// fine row of the table): columns 0..8 the degree-8 polynomial of F_L in
// x = 10 (T - T_k), |x| <= 1, column 9 exp(-T_k).  The polynomial is the
// degree-10 Taylor expansion F_L = sum_j F_{L+j}(T_k) (-x/10)^j / j! with its
// two highest powers replaced by their Chebyshev economisation (error below
// 0.1^9 / (9! 2^8) F_{L+9} = 1e-17 F_{L+9}); against 113-bit arithmetic F_L is
// within 4.2e-16 relative for L <= 4 (degree 7: 9.7e-16 at one instruction
// less a quartet).
// Ten doubles a row: 16-byte reads of random rows spread over all LDS banks.
// Every thread of the workgroup calls it; the caller synchronises afterwards.
template <int L>
__device__ __forceinline__ void boys_lds_fill(const double* __restrict__ table, double* lt)
{
    static_assert(L + 10 < VLX_BOYS_NCOL - 1, "fine rows hold F_0..F_14");
    for (int r = threadIdx.x; r < VLX_BOYS_LROWS; r += blockDim.x) {
        const double* row = table + (10 * r + 5) * VLX_BOYS_NCOL;
        double c[11], f = 1.0;
#pragma unroll
        for (int j = 0; j <= 10; ++j) {
            c[j] = row[L + j] * f;
            f *= -0.1 / (double)(j + 1);
        }
        c[8] += c[10] * (1280.0 / 512.0);
        c[6] -= c[10] * (1120.0 / 512.0);
        c[4] += c[10] * (400.0 / 512.0);
        c[2] -= c[10] * (50.0 / 512.0);
        c[0] += c[10] * (1.0 / 512.0);
        c[7] += c[9] * (576.0 / 256.0);
        c[5] -= c[9] * (432.0 / 256.0);
        c[3] += c[9] * (120.0 / 256.0);
        c[1] -= c[9] * (9.0 / 256.0);
#pragma unroll
        for (int j = 0; j < 9; ++j) lt[r * VLX_BOYS_LCOLS + j] = c[j];
        lt[r * VLX_BOYS_LCOLS + 9] = row[15];
    }
}

// F_0..F_L from the LDS rows (T < VLX_BOYS_TMAX): F_L by its polynomial,
// exp(-T) = exp(-T_k) exp(-x/10) (degree 8, economised from degree 10: error
// 1e-17) and downward recursion; the T >= VLX_BOYS_TMAX branch is that of
// boys<L>.
template <int L>
__device__ __forceinline__ void boys_lds(double T, const double* lt, double* F)
{
    if (T < VLX_BOYS_TMAX) {
        const int k = (int)(T * 5.0);
        const double x = fma(T, 10.0, -(double)(2 * k + 1));
        const double* row = lt + k * VLX_BOYS_LCOLS;
        double s = row[8];
#pragma unroll
        for (int j = 7; j >= 0; --j) s = fma(s, x, row[j]);
        F[L] = s;
        if (L > 0) {
            constexpr double t9 = -1e-9 / 362880.0, t10 = 1e-10 / 3628800.0;
            double e = 1e-8 / 40320.0 + t10 * (1280.0 / 512.0);
            e = fma(e, x, -1e-7 / 5040.0 + t9 * (576.0 / 256.0));
            e = fma(e, x, 1e-6 / 720.0 - t10 * (1120.0 / 512.0));
            e = fma(e, x, -1e-5 / 120.0 - t9 * (432.0 / 256.0));
            e = fma(e, x, 1e-4 / 24.0 + t10 * (400.0 / 512.0));
            e = fma(e, x, -1e-3 / 6.0 + t9 * (120.0 / 256.0));
            e = fma(e, x, 1e-2 / 2.0 - t10 * (50.0 / 512.0));
            e = fma(e, x, -1e-1 - t9 * (9.0 / 256.0));
            e = fma(e, x, 1.0 + t10 * (1.0 / 512.0));
            const double et = row[9] * e;
            const double T2 = 2.0 * T;
#pragma unroll
            for (int m = L - 1; m >= 0; --m) F[m] = fma(T2, F[m + 1], et) * (1.0 / (2.0 * m + 1.0));
        }
    } else {
        const double y = rsq_nr(T);
        F[0] = (0.5 * 1.77245385090551602730) * y;
        if (L > 0) {
            const double et = (double)__expf(-(float)T);
            // 1/T as y^2 with y's rounding taken out: F_m multiplies it m times
            const double y2 = y * y, h = 0.5 * fma(y2, fma(-T, y2, 1.0), y2);
#pragma unroll
            for (int m = 0; m < L; ++m) F[m + 1] = ((2.0 * m + 1.0) * F[m] - et) * h;
        }
    }
}

// The N-point Rys rule of argument T (tables and their accuracy:
// vlxmi/gen/rys.py): roots times ``su`` to slot[i * 64], weights times ``sw``
// to slot[(N + i) * 64], i < N -- lane-private LDS slots, so that the kernels'
// point loops index them at run time.  T < 64: one degree-7 polynomial per
// value on intervals of width 1/4 (64 contiguous bytes per lane and value);
// above, the half-range Gauss-Hermite rule scaled by T.
#define VLX_RYS_TMAX 64.0
#define VLX_RYS_INV_WIDTH 4.0
#define VLX_RYS_NCOEF 8

template <int N>
__device__ __forceinline__ void rys_points(double T, const double* __restrict__ table, const double* large, double su,
                                           double sw, double* slot)
{
    if (T < VLX_RYS_TMAX) {
        const int k = (int)(T * VLX_RYS_INV_WIDTH);
        const double x = T * (2.0 * VLX_RYS_INV_WIDTH) - (double)(2 * k + 1);
        const double* c = table + k * (2 * N * VLX_RYS_NCOEF);
#pragma unroll
        for (int f = 0; f < 2 * N; ++f) {
            double s = c[f * VLX_RYS_NCOEF + VLX_RYS_NCOEF - 1];
#pragma unroll
            for (int j = VLX_RYS_NCOEF - 2; j >= 0; --j) s = fma(s, x, c[f * VLX_RYS_NCOEF + j]);
            slot[f * 64] = s * (f < N ? su : sw);
        }
    } else {
        const double y = rsq_nr(T), ty = su * (y * y), wy = sw * y;
#pragma unroll
        for (int f = 0; f < N; ++f) {
            slot[f * 64] = large[f] * ty;
            slot[(N + f) * 64] = large[N + f] * wy;
        }
    }
}

}  // namespace vlxmi
