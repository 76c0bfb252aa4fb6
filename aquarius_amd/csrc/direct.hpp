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
    uint32_t config, tm, tn;  // batched stages: kernel (tile shape * 4 + layout bits) and tile
};

// Blocks of a launch: fewer than 2^32 threads, 256 a block.
constexpr uint64_t kDirBlocks = uint64_t(1) << 24;
constexpr int kDirGroup = 8;   // problems per grouped launch

// Runs the problem if the direct kernels take its sizes; false: not taken.
bool direct_contract(aq_ctx* ctx, DirectArgs a);
// a group of same-kernel problems in one launch (grouping across contexts), each
// of fewer than kDirBlocks / kDirGroup blocks
void launch_direct_group(int config, const DirectArgs* const* p, int n, hipStream_t s);

// ---- batched stages: the contractions of a solver's small iteration, level by
// level (direct.hip, stage.cpp)
struct StageLevel {
    const DirectArgs* prob = nullptr;   // device
    const uint32_t* first = nullptr;    // device: np + 1 block offsets
    uint32_t np = 0, blocks = 0;
};
struct AsmTerm {
    const double* p;
    double coef;
    uint32_t s0[4], s1[4];   // kind 0: strides; kind 1: row / column multipliers of the digits
    uint32_t kind;           // 0 tensor, 1 product tiles, 2 / 3 packed-pair product, symmetric / antisymmetric
    uint32_t ltm, ltn, tilesM, nsplit;
};
struct AsmOut {
    double* out;
    uint32_t len[4], n, first, term, nterms, sym;
};
void plan_stage_level(DirectArgs* const* a, int n);   // tiles, splits and layouts of a level's problems (P is the caller's)
void launch_stage(const StageLevel* const* l, int n, hipStream_t s);
void launch_assemble(hipStream_t s, const AsmOut* outs, const AsmTerm* terms, int nout, uint32_t blocks);
// sum_k A[ia] B[ib] with output labels ic as a problem (sizes, digits, operands);
// mulM / mulN: the multiplier of each ic label in its row / column index.
// False: not of the direct kernels' form.
bool plan_product(const aq_tensor* A, const char* ia, const aq_tensor* B, const char* ib, const char* ic, DirectArgs& a,
                  uint32_t* mulM, uint32_t* mulN);

// offers a level for a grouped launch (gemm.hip): true once it ran in one
bool batcher_offer_stage(aq_ctx* ctx, int level, const StageLevel& l);
// offers a problem for a grouped launch (gemm.hip): true once it ran in one
bool batcher_offer_direct(aq_ctx* ctx, int config, const DirectArgs& a, int64_t blocks);

}  // namespace aqamd
