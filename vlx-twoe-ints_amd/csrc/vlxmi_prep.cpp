// Density-dependent inputs of a J/K build in a few launches: the symmetrised
// Cartesian density with the maxima the checks and the exchange screening need
// (gen_exchange.py:229-232 takes max|D| per (b,d) type pair), and the ket copies
// of the Coulomb lists ordered by block bound (gen_coulomb.py:209-212).  For a
// molecule of a few atoms the one-operation-at-a-time form of this was most of
// a build: about 130 launches and ten host synchronisations before the first
// class kernel (8 atoms s/p), now six launches and one.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "vlxmi_device.hpp"
#include "vlxmi_prep.h"

namespace {

// |x| of a double as an integer that orders like it (NaN above infinity)
__device__ __forceinline__ unsigned long long abs_bits(double x)
{
    return (unsigned long long)__double_as_longlong(x) & 0x7fffffffffffffffull;
}

__device__ __forceinline__ void raise_to(unsigned long long* p, unsigned long long v)
{
    if (v > *p) atomicMax(p, v);
}

__global__ void zero_stats_kernel(unsigned long long* stats)
{
    if (threadIdx.x < VLXMI_NDSTATS) stats[threadIdx.x] = 0;
}

// stats: [0] max|Dc|, [1] max|Ds - Ds^T|, [2] max|Ds|, [3 + 3 tb + td] max|Dsym|
// over AO pairs of types (tb, td); Dsym = (Dc + Dc^T) / 2.
__global__ void __launch_bounds__(256)
density_stats_kernel(const double* __restrict__ Dc, const uint8_t* __restrict__ type, uint32_t n,
                     const double* __restrict__ Ds, uint32_t m, double* __restrict__ Dsym,
                     unsigned long long* __restrict__ stats)
{
    __shared__ unsigned long long top[VLXMI_NDSTATS];
    if (threadIdx.x < VLXMI_NDSTATS) top[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t step = (uint64_t)gridDim.x * blockDim.x, first = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    unsigned long long c = 0, asym = 0, s = 0;
    for (uint64_t e = first; e < (uint64_t)n * n; e += step) {
        const uint32_t i = (uint32_t)(e / n), j = (uint32_t)(e - (uint64_t)i * n);
        const double v = Dc[e], d = 0.5 * (v + Dc[(uint64_t)j * n + i]);
        Dsym[e] = d;
        c = max(c, abs_bits(v));
        raise_to(&top[3 + 3 * type[i] + type[j]], abs_bits(d));
    }
    for (uint64_t e = first; e < (uint64_t)m * m; e += step) {
        const uint32_t i = (uint32_t)(e / m), j = (uint32_t)(e - (uint64_t)i * m);
        const double v = Ds[e];
        asym = max(asym, abs_bits(v - Ds[(uint64_t)j * m + i]));
        s = max(s, abs_bits(v));
    }
    raise_to(&top[0], c);
    raise_to(&top[1], asym);
    raise_to(&top[2], s);
    __syncthreads();
    if (threadIdx.x < VLXMI_NDSTATS && top[threadIdx.x]) atomicMax(&stats[threadIdx.x], top[threadIdx.x]);
}

struct KetClasses {
    vlxmi_ket_class c[VLXMI_MAX_KET_CLASSES];
};

// One thread per pair block: mat_D of its entries (0 where keep is 0) and the
// block bound max|Q D|.
__global__ void __launch_bounds__(256)
ket_bounds_kernel(KetClasses K, const double* __restrict__ D, uint32_t n, double* __restrict__ mat_D,
                  double* __restrict__ beta)
{
    const vlxmi_ket_class& c = K.c[blockIdx.y];
    const uint64_t b = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= c.nblk) return;
    unsigned long long top = 0;        // ordered as the values; a NaN leads its list
    for (uint32_t t = 0; t < c.nab; ++t) {
        const uint64_t e = b * c.nab + t;
        const double v = c.keep[e] ? D[(uint64_t)c.ao_first[e] * n + (uint64_t)c.ao_second[e]] : 0.0;
        mat_D[c.entry_offset + e] = v;
        top = max(top, abs_bits(c.mat_Q[e] * v));
    }
    beta[c.block_offset + b] = __longlong_as_double((long long)top);
}

// The ket copy of every list: block p of the output is block order[p] of the
// list, or, without an order (lists of at most VLXMI_KET_RANK_MAX blocks), the
// block with p others before it by (bound descending, position), which each
// thread counts for its own block: n comparisons a thread, fewer microseconds than
// a device sort's launches at this size.
__global__ void __launch_bounds__(256)
ket_order_kernel(KetClasses K, const double* __restrict__ beta, const double* __restrict__ mat_D,
                 uint32_t* __restrict__ first, uint32_t* __restrict__ second, double* __restrict__ pair_data,
                 double* __restrict__ mat_Q, double* __restrict__ ket_D)
{
    __shared__ unsigned long long key[256];
    __shared__ uint32_t place[256];
    const vlxmi_ket_class& c = K.c[blockIdx.y];
    const uint64_t base = (uint64_t)blockIdx.x * 256;
    if (base >= c.nblk) return;
    const uint32_t own = c.nblk - base < 256 ? (uint32_t)(c.nblk - base) : 256u;
    if (c.order == nullptr) {
        const uint64_t b = base + threadIdx.x;
        const unsigned long long mine = threadIdx.x < own ? abs_bits(beta[c.block_offset + b]) : 0;
        uint32_t rank = 0;
        for (uint64_t t0 = 0; t0 < c.nblk; t0 += 256) {
            __syncthreads();
            if (t0 + threadIdx.x < c.nblk) key[threadIdx.x] = abs_bits(beta[c.block_offset + t0 + threadIdx.x]);
            __syncthreads();
            const uint32_t cnt = c.nblk - t0 < 256 ? (uint32_t)(c.nblk - t0) : 256u;
            for (uint32_t k = 0; k < cnt; ++k) rank += (key[k] > mine || (key[k] == mine && t0 + k < b)) ? 1u : 0u;
        }
        place[threadIdx.x] = rank;
        __syncthreads();
    }
    for (uint32_t q = threadIdx.x; q < own * c.nab; q += 256) {
        const uint32_t k = q / c.nab, t = q - k * c.nab;
        const uint64_t src = (c.order ? (uint64_t)c.order[base + k] : base + k) * c.nab + t;
        const uint64_t dst = c.entry_offset + (c.order ? base + k : (uint64_t)place[k]) * c.nab + t;
        first[dst] = c.first[src];
        second[dst] = c.second[src];
        pair_data[dst] = c.pair_data[src];
        mat_Q[dst] = c.mat_Q[src];
        ket_D[dst] = mat_D[c.entry_offset + src];
    }
}

int gather_classes(const vlxmi_ket_class* cls, uint32_t ncls, KetClasses* K, uint64_t* most)
{
    if (ncls > VLXMI_MAX_KET_CLASSES) return VLXMI_ERR_SIZE;
    *most = 0;
    for (uint32_t i = 0; i < ncls; ++i) {
        const vlxmi_ket_class& c = cls[i];
        if (c.nblk && (!c.ao_first || !c.ao_second || !c.keep || !c.mat_Q || !c.pair_data || !c.first || !c.second || !c.nab))
            return VLXMI_ERR_ARG;
        K->c[i] = c;
        if (c.nblk > *most) *most = c.nblk;
    }
    return *most / 256 >= 0x7fffffffull ? VLXMI_ERR_SIZE : VLXMI_OK;
}

}  // namespace

extern "C" int vlxmi_density_stats(const double* Dc, const uint8_t* ao_type, uint32_t n, const double* Ds, uint32_t m,
                                   double* Dsym, double* stats, void* stream)
{
    if (!Dc || !ao_type || !Ds || !Dsym || !stats || n == 0 || m == 0) return VLXMI_ERR_ARG;
    hipStream_t st = (hipStream_t)stream;
    unsigned long long* bits = reinterpret_cast<unsigned long long*>(stats);
    hipLaunchKernelGGL(zero_stats_kernel, dim3(1), dim3(64), 0, st, bits);
    const uint64_t blocks = ((uint64_t)n * n + 1023) / 1024;
    hipLaunchKernelGGL(density_stats_kernel, dim3((unsigned)(blocks < 1024 ? blocks : 1024)), dim3(256), 0, st, Dc, ao_type,
                       n, Ds, m, Dsym, bits);
    return (int)hipGetLastError();
}

extern "C" int vlxmi_ket_bounds(const vlxmi_ket_class* cls, uint32_t ncls, const double* D, uint32_t n, double* mat_D,
                                double* beta, void* stream)
{
    if (ncls == 0) return VLXMI_OK;
    if (!cls || !D || !mat_D || !beta) return VLXMI_ERR_ARG;
    KetClasses K = {};
    uint64_t most;
    const int rc = gather_classes(cls, ncls, &K, &most);
    if (rc != 0 || most == 0) return rc;
    hipLaunchKernelGGL(ket_bounds_kernel, dim3((unsigned)((most + 255) / 256), ncls), dim3(256), 0, (hipStream_t)stream, K, D,
                       n, mat_D, beta);
    return (int)hipGetLastError();
}

extern "C" int vlxmi_ket_order(const vlxmi_ket_class* cls, uint32_t ncls, const double* beta, const double* mat_D,
                               uint32_t* first, uint32_t* second, double* pair_data, double* mat_Q, double* ket_D, void* stream)
{
    if (ncls == 0) return VLXMI_OK;
    if (!cls || !beta || !mat_D || !first || !second || !pair_data || !mat_Q || !ket_D) return VLXMI_ERR_ARG;
    KetClasses K = {};
    uint64_t most;
    const int rc = gather_classes(cls, ncls, &K, &most);
    if (rc != 0 || most == 0) return rc;
    for (uint32_t i = 0; i < ncls; ++i)
        if (cls[i].nblk > VLXMI_KET_RANK_MAX && !cls[i].order) return VLXMI_ERR_SIZE;
    hipLaunchKernelGGL(ket_order_kernel, dim3((unsigned)((most + 255) / 256), ncls), dim3(256), 0, (hipStream_t)stream, K, beta,
                       mat_D, first, second, pair_data, mat_Q, ket_D);
    return (int)hipGetLastError();
}
