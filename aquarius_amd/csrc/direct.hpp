// Contractions of small and medium tensors straight from their labelled
// layouts (direct.hip): no permuted operand copies, no output pass.
#pragma once

#include "internal.hpp"

namespace aqamd {

// A group of labels as the digits of one index, first digit fastest, with the
// stride of each digit in two tensors (elements).
constexpr int kDirDigits = 4;
struct DirDigits {
    int nd = 0;
    uint32_t len[kDirDigits] = {1, 1, 1, 1};
    uint32_t s0[kDirDigits] = {0, 0, 0, 0};
    uint32_t s1[kDirDigits] = {0, 0, 0, 0};
    uint32_t mul[kDirDigits] = {0, 0, 0, 0}, shift[kDirDigits] = {0, 0, 0, 0};   // division by len
};

//   C(m,n,b) = alpha * sum_k A(m,k,b) B(k,n,b) + beta * C(m,n,b)
struct DirectArgs {
    const double* A;
    const double* B;
    double* C;
    double* P;             // split partials [batch*tile][split][TM*TN], or null
    double alpha, beta;
    uint32_t M, N, K;
    uint32_t tilesM, tilesN, batch, nsplit;
    uint32_t kchunk;       // k range of one split (a multiple of 16)
    DirDigits m;           // s0: stride in A, s1: in C
    DirDigits n;           // s0: in B, s1: in C
    DirDigits k;           // s0: in A, s1: in B
    uint32_t bsA, bsB, bsC;   // strides of the batch index
};

// Runs the problem if the direct kernels take its sizes; false: not taken.
bool direct_contract(aq_ctx* ctx, DirectArgs a);
// a group of same-kernel problems in one launch (grouping across contexts)
constexpr int kDirGroup = 8;   // problems per launch
void launch_direct_group(int config, const DirectArgs* const* p, int n, hipStream_t s);

// offers a problem for a grouped launch (gemm.hip): true once it ran in one
bool batcher_offer_direct(aq_ctx* ctx, int config, const DirectArgs& a, int64_t blocks);

}  // namespace aqamd
