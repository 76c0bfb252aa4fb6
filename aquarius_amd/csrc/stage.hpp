// The contraction stage of a small closed-shell iteration as a program of
// batched launches (stage.cpp).  Not part of the C ABI.
#pragma once

#include "direct.hpp"

#include "../../include/aqamd.hpp"

#include <string>
#include <vector>

namespace aqamd {

// Levels of independent contractions, each followed by an assembly that forms
// tensors from their tiles and from other tensors.  Built once on a solver's
// tensors (whose addresses it keeps: a solver drops its program whenever it
// replaces a tensor) and run every iteration.
class StageProgram {
  public:
    explicit StageProgram(aq_ctx* ctx) : ctx_(ctx) {}

    // A product for level `level`; its index names it in terms.
    int product(int level, const tensor::Tensor& A, const char* ia, const tensor::Tensor& B, const char* ib,
                const char* ic);
    // Begin output `out` (labels ic) of the assembly after `level`; sym: add the
    // value with labels (1,0,3,2).
    void output(int level, const tensor::Tensor& out, const char* ic, bool sym = false);
    // Terms of the output begun last.
    void add(double coef, const tensor::Tensor& X, const char* ix);
    void add(double coef, int product);
    void add_pairs(double coef, int product, bool antisymmetric);   // packed pairs (0,1) and (2,3)

    double largest_flops() const { return largest_; }
    // tiles, buffers, upload (allocates; synchronises); false if the products are
    // not of the stage's form or its buffers take more than `room` bytes
    bool finish(size_t room);
    void run();           // every launch on the context's stream

  private:
    struct Product {
        int level;
        DirectArgs a;
        std::string ic;
        uint32_t mulM[4], mulN[4];
    };
    struct Term {
        double coef;
        const tensor::Tensor* t;
        std::string ix;
        int product, kind;
    };
    struct Output {
        int level;
        const tensor::Tensor* t;
        std::string ic;
        bool sym;
        std::vector<Term> terms;
    };
    struct Level {
        StageLevel s;
        const AsmOut* outs = nullptr;
        const AsmTerm* terms = nullptr;
        int nout = 0;
        uint32_t blocks = 0;
        double flops = 0.0, bytes = 0.0;
    };
    aq_ctx* ctx_;
    bool ok_ = true;
    double largest_ = 0.0;
    std::vector<Product> products_;
    std::vector<Output> outputs_;
    std::vector<Level> levels_;
    std::vector<const tensor::Tensor*> written_;
    tensor::Tensor tiles_, desc_;
};

// What a program's buffers take, from the labels alone: a-h virtual, i-o occupied,
// p, q / r, s symmetric / antisymmetric virtual pairs, x / y occupied ones.
class StageSizes {
  public:
    StageSizes(int o, int v) : o_(o), v_(v) {}
    int product(int level, const tensor::Tensor&, const char* ia, const tensor::Tensor&, const char* ib, const char* ic);
    void output(int, const tensor::Tensor&, const char*, bool = false) {}
    void add(double, const tensor::Tensor&, const char*) {}
    void add(double, int) {}
    void add_pairs(double, int, bool) {}
    size_t bytes();       // 0: not of the stage's form

  private:
    double len(char c) const;
    double o_, v_;
    bool ok_ = true;
    std::vector<std::vector<DirectArgs>> levels_;
    int count_ = 0;
};

}  // namespace aqamd
