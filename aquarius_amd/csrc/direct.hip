// FP64 contractions read straight from the operands' labelled layouts.
//
//   C(m,n,b) = alpha * sum_k A(m,k,b) B(k,n,b) + beta * C(m,n,b)
//
// m, n and k are groups of labels with arbitrary strides in A, B and C, so no
// operand is permuted into a matrix first and no result is permuted
// afterwards.  Two kinds of tile:
//  - from registers: FP64 MFMA on gfx950 is slow against its operands, a 16x16x4
//    instruction takes 64 cycles for two 512-byte fragments, so fragments are
//    loaded from global memory (L1/L2) into registers directly, without LDS
//    staging and without a barrier in the k loop; every wave runs on its own;
//  - staged through LDS, 64 x 64 and 128 x 128, for many long tiles (below).
//
// A block of 256 threads = WM x WN x WK waves owns a (16 FM WM) x (16 FN WN)
// output tile; each wave has FM x FN 16x16 MFMA blocks, and WK waves share the
// k range (added in LDS, in wave order, at the end).  Work goes in chunks of
// 16 k: lane group q = lane/16 takes k = 4q..4q+3, so an operand whose k is
// contiguous is read with two 16-byte loads per row and chunk, and one whose
// rows are contiguous with 128-byte runs; the k offsets of both operands come
// from an LDS table built once per block, the row offsets from registers.
// Several chunks are in flight per wave.
//
// When the output has too few tiles, the k range is also split over blocks and
// a second launch adds the partial tiles in split order.  (Having the last
// block of a tile add them in the same launch was measured 5 to 15 times
// slower: each block's device-scope fence writes back its XCD's whole L2; 485
// blocks, M = N = 344: 9 us without a split, 117 us with two.)
#include "direct.hpp"

#include <algorithm>
#include <cstdio>
#include <vector>
#include <cmath>

namespace aqamd {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));   // 16-byte load, 8-byte aligned
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kKT = 1024;   // k offsets held at a time

// offset of index x (below 2^31) through a digit group; the divisions by the
// digit lengths are multiplications (set_divider)
__device__ __forceinline__ uint32_t digit_offset(const DirDigits& d, const uint32_t* st, uint32_t x) {
    uint32_t off = 0;
#pragma unroll
    for (int k = 0; k < kDirDigits; ++k) {   // static indices only: the group stays in scalar registers
        if (k + 1 < kDirDigits && k + 1 < d.nd) {
            const uint32_t q = __umulhi(x, d.mul[k]) >> d.shift[k];
            off += (x - q * d.len[k]) * st[k];
            x = q;
        } else if (k + 1 == d.nd) {
            off += x * st[k];
        }
    }
    return off;
}

// block id -> work id: the dispatcher deals ids to the 8 XCDs round-robin; give
// each XCD a contiguous run, whose tiles share operand rows in its L2
__device__ __forceinline__ uint32_t xcd_order(uint32_t bid, uint32_t nb) {
    const uint32_t full = nb / 8 * 8;
    return bid >= full ? bid : (bid % 8) * (nb / 8) + bid / 8;
}

// LDS of a tile: the k tables, then (WK > 1) the waves' accumulators.
constexpr int direct_lds(int fm, int fn, int wm, int wn, int wk) {
    const int red = wk > 1 ? wk * fm * fn * wm * wn * 256 * 8 : 0, tab = 2 * kKT * 4;
    return red > tab ? red : tab;
}

// The epilogue: the tile into C, or (a split, a batched stage) into its place in
// the partial buffer.
template <int FM, int FN, int WM, int WN, int WK, bool TILE>
__device__ __forceinline__ void store_tile(const DirectArgs& g, const f64x4 (&acc)[FM][FN], uint32_t split, uint32_t bt,
                                           uint32_t m0, uint32_t n0, char* lds) {
    constexpr int TM = 16 * FM * WM, TN = 16 * FN * WN;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave % WK, wm = (wave / WK) % WM, wn = wave / (WK * WM);
    const int l16 = lane & 15, q = lane >> 4;
    const uint32_t b = bt / (g.tilesM * g.tilesN);
    // lane holds tile element (m = l16 of block i, n = q + 4r of block j)
    double* Cb = g.C + uint64_t(b) * g.bsC;
    if (!TILE && WK == 1 && g.nsplit == 1) {
        uint32_t cn[FN][4];
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                cn[j][r] = digit_offset(g.n, g.n.s1, min(n0 + (wn * FN + j) * 16 + q + 4 * r, g.N - 1));
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const uint32_t m = m0 + (wm * FM + i) * 16 + l16;
            const uint32_t cm = digit_offset(g.m, g.m.s1, min(m, g.M - 1));
            // every C value of the row is read before any is written (one round trip)
            double cv[FN][4];
            if (g.beta != 0.0) {
#pragma unroll
                for (int j = 0; j < FN; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) cv[j][r] = Cb[cm + cn[j][r]];
            }
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t n = n0 + (wn * FN + j) * 16 + q + 4 * r;
                    if (m < g.M && n < g.N) {
                        double v = g.alpha * acc[i][j][r];
                        if (g.beta != 0.0) v += g.beta * cv[j][r];
                        Cb[cm + cn[j][r]] = v;
                    }
                }
        }
        return;
    }

    constexpr int TE = TM * TN, NE = TE / 256;   // tile elements, and per thread
    static_assert(TE % 256 == 0, "whole tile per thread count");
    double v[NE];
    if (WK > 1) {
        double* red = reinterpret_cast<double*>(lds);
        __syncthreads();   // the k tables are no longer read
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    red[wk * TE + ((wn * FN + j) * 16 + q + 4 * r) * TM + (wm * FM + i) * 16 + l16] = acc[i][j][r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < NE; ++r) {
            double s = red[tid + 256 * r];
#pragma unroll
            for (int w = 1; w < WK; ++w) s += red[w * TE + tid + 256 * r];
            v[r] = s;
        }
    }
    if (TILE || g.nsplit > 1) {
        double* P = g.P + uint64_t(bt) * g.nsplit * TE;
        double* mine = P + uint64_t(split) * TE;
        if (WK > 1) {
#pragma unroll
            for (int r = 0; r < NE; ++r) mine[tid + 256 * r] = v[r];
        } else {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        mine[((wn * FN + j) * 16 + q + 4 * r) * TM + (wm * FM + i) * 16 + l16] = acc[i][j][r];
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < NE; ++r) {
        const uint32_t e = tid + 256 * r;
        const uint32_t m = m0 + e % TM, n = n0 + e / TM;
        if (m < g.M && n < g.N) {
            double* c = Cb + digit_offset(g.m, g.m.s1, m) + digit_offset(g.n, g.n.s1, n);
            const double x = g.alpha * v[r];
            *c = g.beta != 0.0 ? g.beta * *c + x : x;
        }
    }
}

// TILE: the tile goes to the partial buffer whatever the split (batched stages,
// whose assembly adds the tiles of several products).
template <int FM, int FN, int WM, int WN, int WK, int ST, bool VA, bool VB, bool TILE = false>
__device__ __forceinline__ void direct_tile(const DirectArgs& g, uint32_t bid, char* lds) {
    static_assert(WM * WN * WK == 4, "4 waves");
    constexpr int TM = 16 * FM * WM, TN = 16 * FN * WN;
    uint32_t* ta = reinterpret_cast<uint32_t*>(lds);
    uint32_t* tb = ta + kKT;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave % WK, wm = (wave / WK) % WM, wn = wave / (WK * WM);
    const int l16 = lane & 15, q = lane >> 4;

    // work id -> (split, batch, tile), tiles fastest (m, then n): the run of ids
    // that one XCD gets (xcd_order) then covers few splits of many tiles, so its
    // L2 fetches a k range of the operands once for all of them (110 x
    // 110 x 21560, 16 tiles of 16 splits: 32 us with the splits fastest, 24 so)
    const uint32_t tiles = g.tilesM * g.tilesN;
    const uint32_t split = bid / (tiles * g.batch);
    const uint32_t bt = bid % (tiles * g.batch);
    const uint32_t b = bt / tiles, tile = bt % tiles;
    const uint32_t m0 = (tile % g.tilesM) * TM, n0 = (tile / g.tilesM) * TN;
    const uint32_t kbeg = split * g.kchunk, kend = min(g.K, kbeg + g.kchunk);

    const char* Ab = reinterpret_cast<const char*>(g.A + uint64_t(b) * g.bsA);
    const char* Bb = reinterpret_cast<const char*>(g.B + uint64_t(b) * g.bsB);

    // byte offsets of this lane's operand rows; rows past the edge read the
    // last one (they only feed outputs that are not stored)
    uint32_t ra[FM], rb[FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
        ra[i] = digit_offset(g.m, g.m.s0, min(m0 + (wm * FM + i) * 16 + l16, g.M - 1)) * 8u;
#pragma unroll
    for (int j = 0; j < FN; ++j)
        rb[j] = digit_offset(g.n, g.n.s0, min(n0 + (wn * FN + j) * 16 + l16, g.N - 1)) * 8u;

    f64x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f64x4{0, 0, 0, 0};

    // The k loop issues its loads without conditions, ST - 1 chunks ahead (past
    // the end it reads the last full chunk again): behind a branch the compiler
    // would have to wait for every outstanding load at the join.  The partial
    // last chunk is loaded first, by the wave whose turn it is, and used last.
    double va[ST][4][FM], vb[ST][4][FN], ua[4][FM], ub[4][FN];
    for (uint32_t kb = kbeg; kb < kend; kb += kKT) {
        const uint32_t klen = min(uint32_t(kKT), kend - kb);
        const uint32_t nfull = klen / 16;
        if (kb != kbeg) __syncthreads();   // every wave is done with the previous table
        for (uint32_t k = tid; k < (klen + 15) / 16 * 16; k += 256) {
            const uint32_t kk = kb + min(k, klen - 1);   // past the end: the last k, zeroed after the load
            ta[k] = digit_offset(g.k, g.k.s0, kk) * 8u;
            tb[k] = digit_offset(g.k, g.k.s1, kk) * 8u;
        }
        __syncthreads();

        auto offsets = [&](const uint32_t* t, uint32_t c) { return *reinterpret_cast<const u32x4*>(t + c * 16 + 4 * q); };
        auto each = [&](double* x, const char* base, uint32_t row, const u32x4 o, int step) {
#pragma unroll
            for (int s = 0; s < 4; ++s) x[s * step] = *reinterpret_cast<const double*>(base + (row + o[s]));
        };
        auto run = [&](double* x, const char* base, uint32_t row, const u32x4 o, int step) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const f64x2u y = *reinterpret_cast<const f64x2u*>(base + (row + o[0] + 16u * h));
                x[2 * h * step] = y[0];
                x[(2 * h + 1) * step] = y[1];
            }
        };
        auto load = [&](double (&xa)[4][FM], double (&xb)[4][FN], uint32_t c) {
            const u32x4 oa = offsets(ta, c), ob = offsets(tb, c);
#pragma unroll
            for (int i = 0; i < FM; ++i)
                if constexpr (VA) run(&xa[0][i], Ab, ra[i], oa, FM);
                else each(&xa[0][i], Ab, ra[i], oa, FM);
#pragma unroll
            for (int j = 0; j < FN; ++j)
                if constexpr (VB) run(&xb[0][j], Bb, rb[j], ob, FN);
                else each(&xb[0][j], Bb, rb[j], ob, FN);
        };
        auto mma = [&](const double (&xa)[4][FM], const double (&xb)[4][FN]) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(xb[s][j], xa[s][i], acc[i][j], 0, 0, 0);
        };

        const bool tail = klen % 16 != 0 && nfull % WK == uint32_t(wk);
        if (tail) {
            const u32x4 oa = offsets(ta, nfull), ob = offsets(tb, nfull);
#pragma unroll
            for (int i = 0; i < FM; ++i) each(&ua[0][i], Ab, ra[i], oa, FM);
#pragma unroll
            for (int j = 0; j < FN; ++j) each(&ub[0][j], Bb, rb[j], ob, FN);
        }
        if (nfull > uint32_t(wk)) {
            const uint32_t nw = (nfull - wk + WK - 1) / WK;   // this wave's full chunks
            auto chunk = [&](uint32_t i) { return min(wk + i * WK, nfull - 1); };
#pragma unroll
            for (int s = 0; s < ST - 1; ++s) load(va[s], vb[s], chunk(s));
            uint32_t i = 0;
            for (; i + ST <= nw; i += ST) {
#pragma unroll
                for (int s = 0; s < ST; ++s) {
                    load(va[(s + ST - 1) % ST], vb[(s + ST - 1) % ST], chunk(i + s + ST - 1));
                    __builtin_amdgcn_sched_barrier(0);
                    mma(va[s], vb[s]);
                }
            }
#pragma unroll
            for (int s = 0; s < ST - 1; ++s)
                if (i + s < nw) mma(va[s], vb[s]);
        }
        if (tail) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const bool in = nfull * 16 + 4 * q + s < klen;
#pragma unroll
                for (int i = 0; i < FM; ++i) ua[s][i] = in ? ua[s][i] : 0.0;
#pragma unroll
                for (int j = 0; j < FN; ++j) ub[s][j] = in ? ub[s][j] : 0.0;
            }
            mma(ua, ub);
        }
    }

    store_tile<FM, FN, WM, WN, WK, TILE>(g, acc, split, bt, m0, n0, lds);
}

// 64 x 64 and 128 x 128 tiles staged through LDS: 2 x 2 waves of F x F blocks
// share the operands, each element is loaded once per tile, and an operand is
// read along whichever of its rows (KA, KB false) or k (true) is contiguous.  That
// is what the register path lacks on long contractions: its fragments need 20
// L1 accesses for a 64-lane load when k and rows are both strided in memory, a
// chunk then costs 2300 cycles of the CU instead of the 1024 of its MFMAs
// (64 x 64 from registers and so: 1110^3 in two splits 110 and 80 us, 1600^3 191 and
// 178; 2800^3 943, 837, and 744
// with 128 x 128, which also needs half the LDS and L2 traffic of 64 x 64).  A
// chunk is loaded into registers while the one before it is multiplied; LDS holds
// it as [k][row] or [row][k], padded so that the 32 lanes of a half-wave read 32
// different bank pairs.  What bounds it: the matrix cores are busy 73% of a CU's
// busy cycles at 64 x 64 and 82% at 128 x 128 (2800^3), waves wait for data 17% and
// 11% of their time and for the matrix cores to take an instruction most of the
// rest.  A deeper prefetch (2 or 3 chunks) and stores to LDS between the products
// change nothing.  128 x 128 has no registers left: 256, and 5 to 9 spilled in
// three of its four layouts; what that costs is not known.  Random values run up to
// 9% slower than constants (a power limit on short kernels: the same loop reaches
// 72 TFLOP/s over 15 ms, 59 over 2 ms).
template <int F>
struct Staged {
    static constexpr int T = 32 * F, PR = T + 16, PK = 18;             // tile side, pitches
    static constexpr int kOperand = 16 * PR > T * PK ? 16 * PR : T * PK;   // elements of one chunk
    static constexpr int kTab = 512;                                   // k offsets held at a time
    static constexpr int kLds = 4 * kOperand * 8 + 2 * kTab * 4;
};

template <int F, bool KA, bool KB, bool TILE = false>
__device__ __forceinline__ void staged_tile(const DirectArgs& g, uint32_t bid, char* lds) {
    using S = Staged<F>;
    constexpr int T = S::T, L = T / 16;   // tile side; elements a thread loads of an operand per chunk
    double* const sa = reinterpret_cast<double*>(lds);                    // two chunks of A,
    double* const sb = sa + 2 * S::kOperand;                              // two of B
    uint32_t* ta = reinterpret_cast<uint32_t*>(sb + 2 * S::kOperand);
    uint32_t* tb = ta + S::kTab;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = wave >> 1;
    const int l16 = lane & 15, q = lane >> 4;
    const uint32_t tiles = g.tilesM * g.tilesN;   // work id as in direct_tile
    const uint32_t split = bid / (tiles * g.batch);
    const uint32_t bt = bid % (tiles * g.batch);
    const uint32_t b = bt / tiles, tile = bt % tiles;
    // tiles in bands of 8 rows: those that run side by side on an XCD then share
    // operand rows both ways
    const uint32_t band = tile / (8 * g.tilesN) * 8, in = tile % (8 * g.tilesN);
    const uint32_t rows = min(8u, g.tilesM - band);
    const uint32_t tm = band + in % rows, tn = in / rows;
    const uint32_t m0 = tm * T, n0 = tn * T;
    const uint32_t kbeg = split * g.kchunk, kend = min(g.K, kbeg + g.kchunk);
    const char* Ab = reinterpret_cast<const char*>(g.A + uint64_t(b) * g.bsA);
    const char* Bb = reinterpret_cast<const char*>(g.B + uint64_t(b) * g.bsB);

    // the elements (row, k) = (rX + i, kX) or (rX, kX + i) a thread carries, and
    // the byte offsets of its rows (past the edge: the last one, never stored)
    constexpr int NA = KA ? L : 1, NB = KB ? L : 1;
    const int rA = KA ? tid / 16 : tid % T, kA = KA ? tid % 16 : tid / T;
    const int rB = KB ? tid / 16 : tid % T, kB = KB ? tid % 16 : tid / T;
    uint32_t ra[NA], rb[NB];
#pragma unroll
    for (int i = 0; i < NA; ++i) ra[i] = digit_offset(g.m, g.m.s0, min(m0 + rA + 16 * i, g.M - 1)) * 8u;
#pragma unroll
    for (int i = 0; i < NB; ++i) rb[i] = digit_offset(g.n, g.n.s0, min(n0 + rB + 16 * i, g.N - 1)) * 8u;

    f64x4 acc[F][F];
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j) acc[i][j] = f64x4{0, 0, 0, 0};

    constexpr int KS = 256 / T;   // k step between a thread's elements along k
    for (uint32_t kb = kbeg; kb < kend; kb += S::kTab) {
        const uint32_t klen = min(uint32_t(S::kTab), kend - kb), nch = (klen + 15) / 16;
        for (uint32_t k = tid; k < nch * 16; k += 256) {
            const uint32_t kk = kb + min(k, klen - 1);   // past the end: the last k, zeroed before its use
            ta[k] = digit_offset(g.k, g.k.s0, kk) * 8u;
            tb[k] = digit_offset(g.k, g.k.s1, kk) * 8u;
        }
        __syncthreads();
        double x[L], y[L];         // the next chunk's elements of A and B
        uint32_t oa[L], ob[L];     // k offsets of the chunk to be loaded next
        auto offsets = [&](uint32_t c) {
#pragma unroll
            for (int i = 0; i < L; ++i) {
                if (i == 0 || !KA) oa[i] = ta[c * 16 + kA + (KA ? 0 : KS * i)];
                if (i == 0 || !KB) ob[i] = tb[c * 16 + kB + (KB ? 0 : KS * i)];
            }
        };
        auto load = [&] {
#pragma unroll
            for (int i = 0; i < L; ++i)
                x[i] = *reinterpret_cast<const double*>(Ab + (ra[KA ? i : 0] + oa[KA ? 0 : i]));
#pragma unroll
            for (int i = 0; i < L; ++i)
                y[i] = *reinterpret_cast<const double*>(Bb + (rb[KB ? i : 0] + ob[KB ? 0 : i]));
        };
        auto put = [&](uint32_t c) {
            double* pa = sa + (c & 1) * S::kOperand;
            double* pb = sb + (c & 1) * S::kOperand;
            if (c * 16 + 16 > klen) {   // the partial last chunk
#pragma unroll
                for (int i = 0; i < L; ++i) {
                    x[i] = c * 16 + kA + (KA ? 0 : KS * i) < klen ? x[i] : 0.0;
                    y[i] = c * 16 + kB + (KB ? 0 : KS * i) < klen ? y[i] : 0.0;
                }
            }
#pragma unroll
            for (int i = 0; i < L; ++i) pa[KA ? (rA + 16 * i) * S::PK + kA : (kA + KS * i) * S::PR + rA] = x[i];
#pragma unroll
            for (int i = 0; i < L; ++i) pb[KB ? (rB + 16 * i) * S::PK + kB : (kB + KS * i) * S::PR + rB] = y[i];
        };
        offsets(0);
        load();
        offsets(min(1u, nch - 1));
        put(0);
        __syncthreads();
        for (uint32_t c = 0; c < nch; ++c) {
            const double* pa = sa + (c & 1) * S::kOperand;
            const double* pb = sb + (c & 1) * S::kOperand;
            double fa0[F], fb0[F], fa1[F], fb1[F];
            auto fragments = [&](double (&fa)[F], double (&fb)[F], int s) {
                const int k = 4 * s + q;
#pragma unroll
                for (int i = 0; i < F; ++i) {
                    const int r = (wm * F + i) * 16 + l16;
                    fa[i] = pa[KA ? r * S::PK + k : k * S::PR + r];
                }
#pragma unroll
                for (int j = 0; j < F; ++j) {
                    const int r = (wn * F + j) * 16 + l16;
                    fb[j] = pb[KB ? r * S::PK + k : k * S::PR + r];
                }
            };
            auto mma = [&](const double (&fa)[F], const double (&fb)[F]) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < F; ++i)
#pragma unroll
                    for (int j = 0; j < F; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[j], fa[i], acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            };
            // nothing waits for what was just asked for: the next chunk is loaded
            // with offsets read a chunk ago (past the end: the last chunk again),
            // each step's fragments are read a step ahead
            fragments(fa0, fb0, 0);
            fragments(fa1, fb1, 1);
            load();
            offsets(min(c + 2, nch - 1));
            mma(fa0, fb0);
            fragments(fa0, fb0, 2);
            mma(fa1, fb1);
            fragments(fa1, fb1, 3);
            mma(fa0, fb0);
            mma(fa1, fb1);
            put(c + 1);   // into the buffer whose readers passed the last barrier
            __syncthreads();
        }
    }
    store_tile<F, F, 2, 2, 1, TILE>(g, acc, split, b * tiles + tm + tn * g.tilesM, m0, n0, lds);
}

// C from the partial tiles of a split launch: one thread per tile element, the
// splits added in order, eight loads in flight.
__global__ __launch_bounds__(256) void k_direct_reduce(DirectArgs g, uint32_t tm, uint32_t te) {
    const uint32_t per = te / 256;                      // blocks of 256 elements per tile
    const uint32_t bt = blockIdx.x / per, e = (blockIdx.x % per) * 256 + threadIdx.x;
    const uint32_t tiles = g.tilesM * g.tilesN;
    const uint32_t b = bt / tiles, tile = bt % tiles;
    const uint32_t m = (tile % g.tilesM) * tm + e % tm, n = (tile / g.tilesM) * (te / tm) + e / tm;
    if (m >= g.M || n >= g.N) return;
    const double* P = g.P + uint64_t(bt) * g.nsplit * te + e;
    double v = 0.0;
    uint32_t s = 0;
    for (; s + 8 <= g.nsplit; s += 8) {
        double x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = P[uint64_t(s + u) * te];
#pragma unroll
        for (int u = 0; u < 8; ++u) v += x[u];
    }
    for (; s < g.nsplit; ++s) v += P[uint64_t(s) * te];
    double* c = g.C + uint64_t(b) * g.bsC + digit_offset(g.m, g.m.s1, m) + digit_offset(g.n, g.n.s1, n);
    const double x = g.alpha * v;
    *c = g.beta != 0.0 ? g.beta * *c + x : x;
}

template <int FM, int FN, int WM, int WN, int WK, int ST, bool VA, bool VB>
__global__ __launch_bounds__(256) void k_direct(DirectArgs g) {
    __shared__ __attribute__((aligned(16))) char lds[direct_lds(FM, FN, WM, WN, WK)];
    direct_tile<FM, FN, WM, WN, WK, ST, VA, VB>(g, xcd_order(blockIdx.x, gridDim.x), lds);
}

template <int F, bool KA, bool KB>
__global__ __launch_bounds__(256, F == 2 ? 3 : 2) void k_staged(DirectArgs g) {
    __shared__ __attribute__((aligned(16))) char lds[Staged<F>::kLds];
    staged_tile<F, KA, KB>(g, xcd_order(blockIdx.x, gridDim.x), lds);
}

// The tiles of up to kDirGroup problems of different contexts in one launch;
// each tile is computed exactly as in a launch of its problem alone.
struct DirectGroup {
    DirectArgs p[kDirGroup];
    uint32_t first[kDirGroup + 1];
    int n;
};

template <int FM, int FN, int WM, int WN, int WK, int ST, bool VA, bool VB>
__global__ __launch_bounds__(256) void k_direct_grouped(DirectGroup G) {
    __shared__ __attribute__((aligned(16))) char lds[direct_lds(FM, FN, WM, WN, WK)];
    int p = 0;
    while (p + 1 < G.n && blockIdx.x >= G.first[p + 1]) ++p;
    direct_tile<FM, FN, WM, WN, WK, ST, VA, VB>(G.p[p], xcd_order(blockIdx.x - G.first[p], G.first[p + 1] - G.first[p]), lds);
}

template <int F, bool KA, bool KB>
__global__ __launch_bounds__(256, F == 2 ? 3 : 2) void k_staged_grouped(DirectGroup G) {
    __shared__ __attribute__((aligned(16))) char lds[Staged<F>::kLds];
    int p = 0;
    while (p + 1 < G.n && blockIdx.x >= G.first[p + 1]) ++p;
    staged_tile<F, KA, KB>(G.p[p], xcd_order(blockIdx.x - G.first[p], G.first[p + 1] - G.first[p]), lds);
}

struct DirCfg {
    int fm, fn, wm, wn, wk, stages;   // stages 0: staged through LDS
    int resident;                     // blocks of 256 threads a CU holds (registers)
    int tm() const { return 16 * fm * wm; }
    int tn() const { return 16 * fn * wn; }
};
constexpr DirCfg kDirCfg[] = {
    {1, 1, 1, 1, 4, 4, 4},   // 16 x 16: tiny outputs
    {2, 2, 1, 1, 4, 3, 2},   // 32 x 32, waves share k
    {1, 1, 2, 2, 1, 4, 4},   // 32 x 32, short k
    {2, 2, 2, 2, 1, 0, 3},   // 64 x 64, staged through LDS
    {4, 1, 1, 1, 4, 3, 2},   // 64 x 16
    {1, 4, 1, 1, 4, 3, 2},   // 16 x 64
    {4, 1, 4, 1, 1, 2, 2},   // 256 x 16, short k
    {1, 4, 1, 4, 1, 2, 2},   // 16 x 256, short k
    {4, 4, 2, 2, 1, 0, 2},   // 128 x 128, staged
    {2, 2, 2, 2, 1, 3, 2},   // 64 x 64, from registers: a block alone on its CU
    {4, 2, 4, 1, 1, 2, 2},   // 256 x 32, short k: 607500 x 27 x 150 streams 991 MB in 204 us, 4.9 TB/s
};
constexpr int kNDirCfg = int(sizeof(kDirCfg) / sizeof(kDirCfg[0]));

template <class F>
static void with_layout(int va, int vb, F&& f) {
    if (va && vb) f(std::integral_constant<int, 3>{});
    else if (va) f(std::integral_constant<int, 1>{});
    else if (vb) f(std::integral_constant<int, 2>{});
    else f(std::integral_constant<int, 0>{});
}

template <int FM, int FN, int WM, int WN, int WK, int ST>
static void run_direct(int lay, dim3 grid, hipStream_t s, const DirectArgs* one, const DirectGroup* many) {
    with_layout(lay & 1, lay & 2, [&](auto L) {
        constexpr int l = decltype(L)::value;
        if (one)
            hipLaunchKernelGGL((k_direct<FM, FN, WM, WN, WK, ST, (l & 1) != 0, (l & 2) != 0>), grid, dim3(256), 0, s, *one);
        else
            hipLaunchKernelGGL((k_direct_grouped<FM, FN, WM, WN, WK, ST, (l & 1) != 0, (l & 2) != 0>), grid, dim3(256), 0,
                               s, *many);
    });
    AQ_HIP(hipGetLastError());
}

template <int F>
static void run_staged(int lay, dim3 grid, hipStream_t s, const DirectArgs* one, const DirectGroup* many) {
    with_layout(lay & 1, lay & 2, [&](auto L) {
        constexpr bool ka = (decltype(L)::value & 1) != 0, kb = (decltype(L)::value & 2) != 0;
        if (one) hipLaunchKernelGGL((k_staged<F, ka, kb>), grid, dim3(256), 0, s, *one);
        else hipLaunchKernelGGL((k_staged_grouped<F, ka, kb>), grid, dim3(256), 0, s, *many);
    });
    AQ_HIP(hipGetLastError());
}

// config = shape index * 4 + layout bits
static void dispatch_direct(int config, dim3 grid, hipStream_t s, const DirectArgs* one, const DirectGroup* many) {
    const int lay = config & 3;
    switch (config >> 2) {
        case 0: run_direct<1, 1, 1, 1, 4, 4>(lay, grid, s, one, many); break;
        case 1: run_direct<2, 2, 1, 1, 4, 3>(lay, grid, s, one, many); break;
        case 2: run_direct<1, 1, 2, 2, 1, 4>(lay, grid, s, one, many); break;
        case 3: run_staged<2>(lay, grid, s, one, many); break;
        case 4: run_direct<4, 1, 1, 1, 4, 3>(lay, grid, s, one, many); break;
        case 5: run_direct<1, 4, 1, 1, 4, 3>(lay, grid, s, one, many); break;
        case 6: run_direct<4, 1, 4, 1, 1, 2>(lay, grid, s, one, many); break;
        case 7: run_direct<1, 4, 1, 4, 1, 2>(lay, grid, s, one, many); break;
        case 8: run_staged<4>(lay, grid, s, one, many); break;
        case 9: run_direct<2, 2, 2, 2, 1, 3>(lay, grid, s, one, many); break;
        default: run_direct<4, 2, 4, 1, 1, 2>(lay, grid, s, one, many); break;
    }
}

void launch_direct_group(int config, const DirectArgs* const* p, int n, hipStream_t s) {
    AQ_CHECK(n >= 1 && n <= kDirGroup, AQ_ERR_INVALID, "direct group size");
    DirectGroup G{};
    G.n = n;
    for (int i = 0; i < n; ++i) {
        G.p[i] = *p[i];
        G.first[i + 1] = G.first[i] + p[i]->tilesM * p[i]->tilesN * p[i]->batch * p[i]->nsplit;
    }
    dispatch_direct(config, dim3(G.first[n]), s, nullptr, &G);
}

// Division of x < 2^31 by len >= 2 as (x * mul) >> (32 + shift): with
// s = ceil(log2 len), mul = ceil(2^(31+s) / len) fits 32 bits and is exact
// for those x (Granlund and Montgomery, PLDI 1994).
void set_dividers(DirDigits& d) {
    for (int k = 0; k < d.nd; ++k) {
        uint32_t s = 1;
        while ((uint64_t(1) << s) < d.len[k]) ++s;
        d.mul[k] = uint32_t(((uint64_t(1) << (31 + s)) + d.len[k] - 1) / d.len[k]);
        d.shift[k] = s - 1;
    }
}

// k contiguous over every aligned group of four
static bool k_runs(const DirDigits& k, const uint32_t* st) {
    return k.nd >= 1 && st[0] == 1 && (k.nd == 1 || k.len[0] % 4 == 0);
}

// The layout bits of an operand's kernel, whose k strides are `st`: a staged tile
// reads it along k if that is contiguous; the register path loads pairs of k.
static bool k_layout(const DirCfg& f, const DirDigits& k, const uint32_t* st) {
    return f.stages == 0 ? k.nd >= 1 && st[0] == 1 : k_runs(k, st);
}

// Tile shape and split of one problem: the least modelled time over the
// shapes and power-of-two splits.  Model (clock cycles): a chunk of 16 k costs a
// wave its MFMAs (64 each) or the L1 accesses of its fragments (more where k is
// the contiguous index), and a single wave at least the load latency over the
// chunks in flight; blocks queue on 256 CUs, as many at a time as registers let
// a CU hold; waves that share k are added at the end; operand tiles come in at a
// rate of the whole chip; a split pays a second launch and the traffic of the
// partial tiles.  The constants are a least-regret fit to 515 contractions (the
// forms of the CCSD iteration at o = 4 to 28, v = 17 to 165, and plain products up
// to 1e9 FLOP), each timed in every shape and split; over these and 190 more (long
// inner extents, batches, short products with long sides) the chosen one is 2.2%
// slower than the best on average, 9% at the 90th percentile.  (A model without
// residency and the waves' sum, fitted to 39 contractions, was 3.7% and 15% off:
// 1110^3 in 32 x 32 tiles 102 us, now 64 x 64 in two splits 78; 201600 x 14 x 120 in
// 64 x 16 tiles 52 us, now 256 x 16 43.)
constexpr double kL1Rows = 320.0, kL1K = 369.0, kLatency = 934.0, kStart = 3460.0, kReduce = 905.0, kChip = 4508.0;
constexpr double kLaunch = 1.5, kSplit = 2.955, kSplitBytes = 5148.0, kPerSplit = 0.06, kCyclesPerUs = 2400.0;
constexpr double kStagedWait = 676.0;

struct Pick {
    int cfg = -1;
    uint32_t nsplit = 1;
    double us = 1e300;
};

static Pick pick_shape(const DirectArgs& a) {
    Pick best;
    const uint32_t chunks = (a.K + 15) / 16;
    const uint32_t padM = (a.M + 15) / 16 * 16, padN = (a.N + 15) / 16 * 16;
    auto contiguous = [](const DirDigits& d, const uint32_t* st) { return d.nd > 0 && st[0] == 1; };
    const double l1A = !contiguous(a.m, a.m.s0) && contiguous(a.k, a.k.s0) ? kL1K : kL1Rows;
    const double l1B = !contiguous(a.n, a.n.s0) && contiguous(a.k, a.k.s1) ? kL1K : kL1Rows;
    for (int c = 0; c < kNDirCfg; ++c) {
        const DirCfg& f = kDirCfg[c];
        const uint32_t tm = uint32_t(f.tm()), tn = uint32_t(f.tn()), wk = uint32_t(f.wk);
        // at most a quarter of such a tile is the product (batches of tiny ones)
        if (tm >= 2 * padM && tn >= 2 * padN) continue;
        const uint64_t tiles = uint64_t((a.M + tm - 1) / tm) * ((a.N + tn - 1) / tn) * a.batch;
        // cycles of a CU per chunk of a block (of each wave); 128 x 128 spills 5 to
        // 9 registers in three of its four layouts
        const double mfma = f.fm * f.fn * 256.0;
        const double busy = f.stages ? std::max(mfma, f.fm * l1A + f.fn * l1B) : mfma * (f.fm == 4 ? 1.27 : 1.064);
        const double wait = f.stages ? std::max(kLatency / (f.stages - 1), busy) : busy + kStagedWait;
        const double ends = f.wk > 1 ? kReduce : 0.0, feed = (tm + tn) * 128.0 * f.wk / kChip;
        const double partials = double(tiles) * tm * tn * 8.0 / kSplitBytes / kCyclesPerUs;
        for (uint32_t l = 0, s = 1; l < 8; ++l, s *= 2) {
            const uint64_t blocks = tiles << l;
            if (s > 1 && (chunks < wk * s || blocks > 16384)) break;
            const uint64_t cu = (blocks + 255) / 256, rounds = (cu + uint32_t(f.resident) - 1) / uint32_t(f.resident);
            const double per_wave = ((chunks + s - 1) / s + wk - 1) / wk;
            const double alone = per_wave * wait + kStart + ends;
            const double queued = std::max(double(cu) * (per_wave * busy + ends), double(rounds) * alone);
            double t = kLaunch + std::max({alone, queued, feed * per_wave * double(blocks)}) / kCyclesPerUs;
            if (s > 1) t += kSplit + partials * (2 * s + 1) + s * kPerSplit;
            if (t < best.us) best = {c, s, t};
        }
    }
    return best;
}

// ------------------------------------------------------- batched stages
//
// One launch over the tiles of many independent contractions (of one job, or
// of several jobs' stages merged): block -> (job, problem, tile).  The problem
// descriptors are in device memory, built once per solver; every tile goes to
// its problem's partial buffer and k_assemble forms the tensors from them.
// Bound by latency at the sizes it serves (a block runs a few us, most of it
// waiting for its first operands), so what counts is that all products of a
// level run side by side and that a stage is 8 launches instead of 57.
struct StageGroup {
    const DirectArgs* prob[kDirGroup];
    const uint32_t* first[kDirGroup];   // block offsets of each job's problems (np + 1)
    uint32_t np[kDirGroup];
    uint32_t start[kDirGroup + 1];
    int n;
};

template <int FM, int FN, int WM, int WN, int WK, int ST>
__device__ __forceinline__ void stage_tile(const DirectArgs& g, uint32_t bid, char* lds) {
    switch (g.config & 3) {
        case 0: direct_tile<FM, FN, WM, WN, WK, ST, false, false, true>(g, bid, lds); break;
        case 1: direct_tile<FM, FN, WM, WN, WK, ST, true, false, true>(g, bid, lds); break;
        case 2: direct_tile<FM, FN, WM, WN, WK, ST, false, true, true>(g, bid, lds); break;
        default: direct_tile<FM, FN, WM, WN, WK, ST, true, true, true>(g, bid, lds); break;
    }
}

// Fewer chunks in flight than the single kernels, for three waves per SIMD: the
// blocks of a level are short and mostly wait (o = 8, v = 43: 37 us a launch
// with 4/3/3 chunks and two waves, 29 us with 3/2/2 and three).  The 64 x 64 tile
// takes all of the 168 registers that three waves leave, and 8 are spilled; the
// other shapes need fewer (o = 13, v = 75: 171 us a level, matrix cores busy 60%).
__global__ __launch_bounds__(256, 3) void k_stage(StageGroup G) {
    __shared__ __attribute__((aligned(16))) char lds[Staged<2>::kLds];   // the largest of the shapes
    int j = 0;
    while (j + 1 < G.n && blockIdx.x >= G.start[j + 1]) ++j;
    const uint32_t bid = blockIdx.x - G.start[j];
    const uint32_t* first = G.first[j];
    // np <= 64: one load and a ballot instead of a chain of loads
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t p = __popcll(__ballot(lane + 1 < G.np[j] && bid >= first[min(lane + 1, G.np[j])]));
    const DirectArgs& g = G.prob[j][p];
    const uint32_t id = xcd_order(bid - first[p], first[p + 1] - first[p]);
    switch (g.config >> 2) {
        case 0: stage_tile<1, 1, 1, 1, 4, 3>(g, id, lds); break;
        case 1: stage_tile<2, 2, 1, 1, 4, 2>(g, id, lds); break;
        case 3: stage_tile<4, 1, 1, 1, 4, 2>(g, id, lds); break;
        default:
            switch (g.config & 3) {
                case 0: staged_tile<2, false, false, true>(g, id, lds); break;
                case 1: staged_tile<2, true, false, true>(g, id, lds); break;
                case 2: staged_tile<2, false, true, true>(g, id, lds); break;
                default: staged_tile<2, true, true, true>(g, id, lds); break;
            }
    }
}

void launch_stage(const StageLevel* const* l, int n, hipStream_t s) {
    AQ_CHECK(n >= 1 && n <= kDirGroup, AQ_ERR_INVALID, "stage group size");
    StageGroup G{};
    G.n = n;
    for (int i = 0; i < n; ++i) {
        G.prob[i] = l[i]->prob;
        G.first[i] = l[i]->first;
        G.np[i] = l[i]->np;
        G.start[i + 1] = G.start[i] + l[i]->blocks;
    }
    hipLaunchKernelGGL(k_stage, dim3(G.start[n]), dim3(256), 0, s, G);
    AQ_HIP(hipGetLastError());
}

// Value of a term at digits d (of the output's dimensions): a strided tensor
// element; a tile element of a product at its row and column index; or one of
// the packed-pair products S+ / S- (symmetric / antisymmetric under exchange of
// the pair (d0,d1), and of (d2,d3)).
__device__ __forceinline__ double term_value(const AsmTerm& t, const uint32_t (&d)[4]) {
    uint32_t m = d[0] * t.s0[0] + d[1] * t.s0[1] + d[2] * t.s0[2] + d[3] * t.s0[3];
    if (t.kind == 0) return t.coef * t.p[m];
    uint32_t n = d[0] * t.s1[0] + d[1] * t.s1[1] + d[2] * t.s1[2] + d[3] * t.s1[3];
    double sign = t.coef;
    if (t.kind >= 2) {
        const uint32_t a = min(d[0], d[1]), b = max(d[0], d[1]), i = min(d[2], d[3]), j = max(d[2], d[3]);
        if (t.kind == 2) {
            m = a + b * (b + 1) / 2;
            n = i + j * (j + 1) / 2;
        } else {
            if (a == b || i == j) return 0.0;
            m = a + b * (b - 1) / 2;
            n = i + j * (j - 1) / 2;
            if ((d[0] < d[1]) != (d[2] < d[3])) sign = -sign;
        }
    }
    const uint32_t tile = (m >> t.ltm) + t.tilesM * (n >> t.ltn);
    const uint32_t e = ((n & ((1u << t.ltn) - 1)) << t.ltm) + (m & ((1u << t.ltm) - 1));
    const double* p = t.p + ((uint64_t(tile) * t.nsplit) << (t.ltm + t.ltn)) + e;
    double v = p[0];
    uint32_t s = 1;
    for (; s + 8 <= t.nsplit; s += 8) {   // 8 loads in flight
        double x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = p[uint64_t(s + u) << (t.ltm + t.ltn)];
#pragma unroll
        for (int u = 0; u < 8; ++u) v += x[u];
    }
    for (; s < t.nsplit; ++s) v += p[uint64_t(s) << (t.ltm + t.ltn)];
    return sign * v;
}

__device__ __forceinline__ double terms_at(const AsmTerm* terms, uint32_t n, const uint32_t (&d)[4]) {
    double v = 0.0;
    for (uint32_t k = 0; k < n; ++k) v += term_value(terms[k], d);
    return v;
}

// out[d] = sum of the terms at d; block -> output by prefix, one thread per
// element, first dimension fastest.  A symmetrised output [n1,n1,n2,n2] adds
// the sum at (d1,d0,d3,d2): a block takes the 16 x 16 tile (t0,t1) of slab
// (r,s), r <= s, and its mirror, the tile (t1,t0) of slab (s,r), forms each
// element's sum once, along its first index, and exchanges them through LDS.
// (o = 13, v = 75: the doubles, 11 products and a tensor, 128 -> 37 us.)
__global__ __launch_bounds__(256) void k_assemble(const AsmOut* __restrict__ outs, const AsmTerm* __restrict__ terms,
                                                  int nout) {
    __shared__ double ta[16][17], tb[16][17];
    const int lane = threadIdx.x & 63;   // nout <= 64
    const int o = __popcll(__ballot(lane + 1 < nout && blockIdx.x >= outs[min(lane + 1, nout - 1)].first));
    const AsmOut& q = outs[o];
    const AsmTerm* t = terms + q.term;
    const uint32_t w = blockIdx.x - q.first;
    if (!q.sym) {
        const uint32_t x = w * 256 + threadIdx.x;
        if (x >= q.n) return;
        uint32_t d[4], r = x;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const uint32_t c = r / q.len[k];
            d[k] = r - c * q.len[k];
            r = c;
        }
        d[3] = r;
        q.out[x] = terms_at(t, q.nterms, d);
        return;
    }
    const uint32_t n1 = q.len[0], n2 = q.len[2], nt = (n1 + 15) / 16;
    const uint32_t t0 = w % nt, t1 = w / nt % nt;
    uint32_t pair = w / (nt * nt), s = 0;
    while (pair > s) pair -= ++s;          // pair = (r, s), r <= s
    const uint32_t r = pair;
    if (r == s && t1 < t0) return;         // the mirrored tile's block
    const uint32_t tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    const uint32_t d[4] = {t0 * 16 + tx, t1 * 16 + ty, r, s}, e[4] = {t1 * 16 + tx, t0 * 16 + ty, s, r};
    const bool in_d = d[0] < n1 && d[1] < n1, in_e = e[0] < n1 && e[1] < n1;
    const double x = in_d ? terms_at(t, q.nterms, d) : 0.0, y = in_e ? terms_at(t, q.nterms, e) : 0.0;
    ta[ty][tx] = x;
    tb[ty][tx] = y;
    __syncthreads();
    if (in_d) q.out[d[0] + n1 * (d[1] + uint64_t(n1) * (r + n2 * s))] = x + tb[tx][ty];
    if (in_e) q.out[e[0] + n1 * (e[1] + uint64_t(n1) * (s + n2 * r))] = y + ta[tx][ty];
}

void launch_assemble(hipStream_t s, const AsmOut* outs, const AsmTerm* terms, int nout, uint32_t blocks) {
    hipLaunchKernelGGL(k_assemble, dim3(blocks), dim3(256), 0, s, outs, terms, nout);
    AQ_HIP(hipGetLastError());
}

// Tiles and splits for the problems of one level, which share the chip: with a
// bound T on what any block may take alone, each problem takes its cheapest
// option in CU time within T, and the level takes the larger of T and the sum
// of those; the T that gives the shortest level is kept.  A chunk of a block
// alone takes about 2000 cycles in every tile; a model without that left K =
// 5625 unsplit and its 264 us set the length of the level (o = 13, v = 75: 410 us
// against 322).  The thin products take 64 x 16 tiles (304 us; with 64 x 64 for
// 13 columns 322).
void plan_stage_level(DirectArgs* const* a, int n) {
    struct Option {
        int cfg;
        uint32_t nsplit;
        double alone, share;
    };
    constexpr double kStageBlock = 1000.0;     // CU cycles of a block's start and end
    constexpr double kStageStart = 2337.0, kStageL1 = 286.0, kStageChip = 5534.0, kStageSplitBytes = 3509.0;
    constexpr double kStageLatency = 2000.0;   // a chunk of a block alone, whatever its tile
    constexpr double kStageSplit = 60.0;       // the assembly's cycles per partial tile
    std::vector<std::vector<Option>> opts(static_cast<size_t>(n));
    double lo = 1e300, hi = 0.0;
    for (int i = 0; i < n; ++i) {
        for (int c : {0, 1, 3, 4}) {
            const DirCfg& f = kDirCfg[c];
            const double chunks = std::ceil(a[i]->K / 16.0);
            const double tiles = double((a[i]->M + f.tm() - 1) / f.tm()) * double((a[i]->N + f.tn() - 1) / f.tn());
            for (uint32_t s = 1; s <= 128; s *= 2) {
                if (s > 1 && (chunks / s < f.wk || tiles * s > 16384)) break;
                const double per_wave = std::ceil(std::ceil(chunks / s) / f.wk);
                const double mfma = f.fm * f.fn * 256.0;
                const double busy = f.stages ? std::max(mfma, (f.fm + f.fn) * kStageL1) : mfma * 1.05;
                const double cu = per_wave * busy + kStageBlock;
                const double fed = (f.tm() + f.tn()) * 128.0 * f.wk * per_wave / kStageChip * 256.0;
                const double sums = s > 1 ? f.tm() * f.tn() * 16.0 / kStageSplitBytes * 256.0 : 0.0;
                const double alone = per_wave * std::max(kStageLatency, busy) + kStageStart + kStageSplit * s;
                const double share = tiles * s * (std::max(cu, fed) + sums) / 256.0;
                // not an option that is never the better one
                bool worse = false;
                for (const auto& x : opts[size_t(i)]) worse = worse || (x.alone <= alone && x.share <= share);
                if (!worse) opts[size_t(i)].push_back({c, s, alone, share});
                lo = std::min(lo, alone);
                hi = std::max(hi, alone);
            }
        }
    }
    auto choose = [&](const std::vector<Option>& o, double T) {
        const Option* best = nullptr;
        for (const auto& x : o)   // within T the smallest share; otherwise the shortest
            if (!best || (x.alone <= T ? best->alone > T || x.share < best->share : best->alone > T && x.alone < best->alone))
                best = &x;
        return best;
    };
    double bestT = hi, best_time = 1e300;
    for (double T = lo; T <= hi * 1.15; T *= 1.15) {
        double sum = 0.0, longest = 0.0;
        for (const auto& o : opts) {
            const Option* x = choose(o, T);
            sum += x->share;
            longest = std::max(longest, x->alone);
        }
        if (std::max(sum, longest) < best_time) {
            best_time = std::max(sum, longest);
            bestT = T;
        }
    }
    for (int i = 0; i < n; ++i) {
        const Option* x = choose(opts[size_t(i)], bestT);
        const DirCfg& f = kDirCfg[x->cfg];
        DirectArgs& p = *a[i];
        p.tilesM = (p.M + f.tm() - 1) / f.tm();
        p.tilesN = (p.N + f.tn() - 1) / f.tn();
        p.kchunk = ((p.K + 15) / 16 + x->nsplit - 1) / x->nsplit * 16;
        p.nsplit = (p.K + p.kchunk - 1) / p.kchunk;
        for (DirDigits* d : {&p.m, &p.n, &p.k}) set_dividers(*d);
        const uint32_t shape = x->cfg == 3 ? 2 : x->cfg == 4 ? 3 : uint32_t(x->cfg);   // k_stage's shapes: 16, 32, 64, 64 x 16
        p.config = shape * 4 + (k_layout(f, p.k, p.k.s0) ? 1 : 0) + (k_layout(f, p.k, p.k.s1) ? 2 : 0);
        p.tm = uint32_t(f.tm());
        p.tn = uint32_t(f.tn());
    }
}

bool direct_contract(aq_ctx* ctx, DirectArgs a) {
    const Pick p = pick_shape(a);
    if (p.cfg < 0) return false;
    const DirCfg& f = kDirCfg[p.cfg];
    a.tilesM = (a.M + f.tm() - 1) / f.tm();
    a.tilesN = (a.N + f.tn() - 1) / f.tn();
    const uint32_t chunks = (a.K + 15) / 16;
    a.kchunk = (chunks + p.nsplit - 1) / p.nsplit * 16;
    a.nsplit = (a.K + a.kchunk - 1) / a.kchunk;
    const uint64_t tiles = uint64_t(a.tilesM) * a.tilesN * a.batch;
    if (tiles * a.nsplit >= kDirBlocks) return false;
    Scratch part(ctx, a.nsplit > 1 ? size_t(tiles) * a.nsplit * f.tm() * f.tn() * 8 : 0);
    for (DirDigits* d : {&a.m, &a.n, &a.k}) set_dividers(*d);
    a.P = part.as<double>();
    const int config = p.cfg * 4 + (k_layout(f, a.k, a.k.s0) ? 1 : 0) + (k_layout(f, a.k, a.k.s1) ? 2 : 0);
    char name[64];
    snprintf(name, sizeof(name), "direct_f64_%dx%d", f.tm(), f.tn());
    const double mn = double(a.M) * a.N * a.batch;
    // a server's slots merge same-kernel problems of different jobs; the thin
    // ones launch alone, as thin GEMMs do
    const bool grouped = ctx->batcher && !ctx->capture && a.M > 16 && a.N > 16 &&
                         tiles * a.nsplit < kDirBlocks / kDirGroup &&
                         batcher_offer_direct(ctx, config, a, int64_t(tiles) * a.nsplit);
    if (!grouped) {
        TimedLaunch tl(ctx, name, 2.0 * mn * a.K,
                       8.0 * ((double(a.M) + a.N) * a.K * a.batch + mn * (a.beta != 0.0 ? 2 : 1)));
        dispatch_direct(config, dim3(unsigned(tiles * a.nsplit)), ctx->stream, &a, nullptr);
    }
    if (a.nsplit > 1) {
        const uint32_t te = uint32_t(f.tm() * f.tn());
        TimedLaunch tl(ctx, "direct_reduce", mn * a.nsplit, 8.0 * double(tiles) * te * (a.nsplit + 1));
        hipLaunchKernelGGL(k_direct_reduce, dim3(unsigned(tiles * (te / 256))), dim3(256), 0, ctx->stream, a,
                           uint32_t(f.tm()), te);
        AQ_HIP(hipGetLastError());
    }
    return true;
}

}  // namespace aqamd
