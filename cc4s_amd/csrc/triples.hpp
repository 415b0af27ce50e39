// (T) correction: the connected triples amplitudes and the energy (triples.hip).
#pragma once

#include "tensor.hpp"

namespace cc4s_amd {

// largest grid of the energy kernel (one running sum per block in `acc`);
// the complex kernel uses 512 blocks (two per CU, bound by registers), the real
// one 1024 (four per CU, bound by threads): one resident wave of blocks, no
// tail
constexpr int kTriplesBlocks = 1024;

// hole triples per launch: at most `most` of `all`, at least one
int64_t triples_chunk(int64_t Nv, int64_t all, int64_t most, int parts);

// Connected triples amplitudes of the hole triples t0 ... t0 + count - 1 (number
// tetrahedral(k) + triangular(j) + i, i <= j <= k), in three parts that add up
// (triples.hip): all of them, Y[x1,x2,x3,part,triple], or (part >= 0) one of them
// in W[a,b,c,triple], written (0) or added (1, 2).  Dense operands V_ppph[b,c,d,k],
// T2[a,b,i,j], H[a,l,j,i] = -conj(V_ijla).
void triples_product(hipStream_t s, Field f, const void *Vppph, const void *T2, const void *H,
                     void *Y, int64_t No, int64_t Nv, int64_t t0, int64_t count, int part);

// acc[block] += partial sums of the weighted Re(W Zs)/D over those hole triples;
// W in `parts` (3 or 1) as above; Vpphh [v,v,o,o], T1 [v,o]
void triples_energy(hipStream_t s, Field f, const void *W, const void *Vpphh,
                    const void *T1, const double *eps_h, const double *eps_p,
                    int64_t No, int64_t Nv, int64_t t0, int64_t count, int parts, double *acc);

}  // namespace cc4s_amd
