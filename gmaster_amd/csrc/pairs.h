// Launchers of the FP64 ring-pair kernels (pairs.hip) for spin-0 maps.
#pragma once

#include <stdint.h>

namespace gm {

// Ring pairs per workgroup (and per partial slot) of the FP64 spin-0 analyses.
int pairs_chunk(int64_t nside);

// Ring pairs jbeg .. jend - 1 in nblk workgroups per order, one partial slot each.
int ana_pairs_s0(const char* name, const double* spec, int K, int64_t ld, int64_t smap, int64_t nside, int64_t L,
                 const double* alpha, const double* smant, const int32_t* sexp, const int32_t* nact, double* partial,
                 int jbeg, int jend, int nblk, void* stream);
int finish_pairs_s0(const char* name, const double* partial, int K, int64_t nside, int64_t L, const int32_t* nact,
                    const double* P, double* alm, int64_t astride, int mode, int jbeg, int jend, void* stream);
int syn_pairs_s0(const char* name, const double* coef, int K, int64_t nside, int64_t L, const double* alpha,
                 const double* smant, const int32_t* sexp, const int32_t* nact, double* spec, int64_t ld, int64_t smap,
                 void* stream);

}  // namespace gm
