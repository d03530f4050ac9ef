/* Density-dependent inputs of a J/K build (csrc/vlxmi_prep.cpp); no counterpart
 * in the reference tree, whose host prepares them.  Return codes as in
 * vlxmi_kernels.h; all pointers device pointers unless said otherwise. */
#ifndef VLXMI_PREP_H
#define VLXMI_PREP_H
#include <stdint.h>

#define VLXMI_NDSTATS 12
#define VLXMI_MAX_KET_CLASSES 6
/* longest list vlxmi_ket_order orders by itself */
#define VLXMI_KET_RANK_MAX 4096

/* One Coulomb pair list in its resident order (nblk blocks of nab entries) and
 * where its share of the concatenated outputs begins. */
typedef struct {
    const int64_t* ao_first;      /* Cartesian AO of every entry's first / second component */
    const int64_t* ao_second;
    const uint8_t* keep;          /* 0: mat_D is 0 (entries below a diagonal block's diagonal) */
    const double* mat_Q;
    const double* pair_data;
    const uint32_t* first;
    const uint32_t* second;
    const int64_t* order;         /* vlxmi_ket_order: block of the list for every output block, or null */
    uint64_t nblk;
    uint64_t entry_offset;
    uint64_t block_offset;
    uint32_t nab;
    uint32_t unused;
} vlxmi_ket_class;

#ifdef __cplusplus
extern "C" {
#endif

/* Dsym = (Dc + Dc^T) / 2 (n x n) and stats[12]: max|Dc|, max|Ds - Ds^T|, max|Ds| (Ds m x m), then
 * max|Dsym| over the AO pairs of each ordered pair of types ss, sp, sd, ps, .. dd (ao_type: 0 s, 1 p, 2 d). */
int vlxmi_density_stats(const double* Dc, const uint8_t* ao_type, uint32_t n, const double* Ds, uint32_t m, double* Dsym,
                        double* stats, void* stream);

/* Every list's mat_D (resident order) from the density D (n x n) and block bounds beta = max|Q D|;
 * cls: HOST array of ncls <= VLXMI_MAX_KET_CLASSES lists. */
int vlxmi_ket_bounds(const vlxmi_ket_class* cls, uint32_t ncls, const double* D, uint32_t n, double* mat_D, double* beta,
                     void* stream);

/* The ket copies of the lists: blocks by non-increasing beta (ties in list order), or by cls[i].order. */
int vlxmi_ket_order(const vlxmi_ket_class* cls, uint32_t ncls, const double* beta, const double* mat_D, uint32_t* first,
                    uint32_t* second, double* pair_data, double* mat_Q, double* ket_D, void* stream);

#ifdef __cplusplus
}
#endif
#endif
