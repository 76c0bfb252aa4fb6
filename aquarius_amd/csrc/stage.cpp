// StageProgram: see stage.hpp; the kernels are in direct.hip.
#include "stage.hpp"

#include <algorithm>
#include <cstring>
#include <numeric>

namespace aqamd {

int StageProgram::product(int level, const tensor::Tensor& A, const char* ia, const tensor::Tensor& B, const char* ib,
                          const char* ic) {
    Product p;
    p.level = level;
    p.ic = ic;
    ok_ = ok_ && p.ic.size() <= 4 && plan_product(A.handle(), ia, B.handle(), ib, ic, p.a, p.mulM, p.mulN);
    largest_ = std::max(largest_, 2.0 * double(p.a.M) * double(p.a.N) * double(p.a.K));
    products_.push_back(p);
    return int(products_.size()) - 1;
}

void StageProgram::output(int level, const tensor::Tensor& out, const char* ic, bool sym) {
    if (sym) {
        const auto l = out.lengths();
        ok_ = ok_ && l.size() == 4 && l[0] == l[1] && l[2] == l[3];
    }
    outputs_.push_back({level, &out, ic, sym, {}});
}
void StageProgram::add(double coef, const tensor::Tensor& X, const char* ix) {
    outputs_.back().terms.push_back({coef, &X, ix, -1, 0});
}
void StageProgram::add(double coef, int product) { outputs_.back().terms.push_back({coef, nullptr, "", product, 1}); }
void StageProgram::add_pairs(double coef, int product, bool antisymmetric) {
    outputs_.back().terms.push_back({coef, nullptr, "", product, antisymmetric ? 3 : 2});
}

constexpr size_t kDescBytes = size_t(1) << 16;   // more than the descriptors take

static uint32_t log2_of(uint32_t x) {
    uint32_t l = 0;
    while ((1u << l) < x) ++l;
    return l;
}

// doubles of the tiles of a planned product
static int64_t tile_doubles(const DirectArgs& a) { return int64_t(a.tilesM) * a.tilesN * a.nsplit * a.tm * a.tn; }

double StageSizes::len(char c) const {
    switch (c) {
        case 'p': case 'q': return v_ * (v_ + 1) / 2;
        case 'r': case 's': return v_ * (v_ - 1) / 2;
        case 'x': return o_ * (o_ + 1) / 2;
        case 'y': return o_ * (o_ - 1) / 2;
        default: return c < 'i' ? v_ : o_;
    }
}

int StageSizes::product(int level, const tensor::Tensor&, const char* ia, const tensor::Tensor&, const char* ib,
                        const char* ic) {
    // as plan_product: the rows hold the first output label
    const std::string a(ia), b(ib);
    const std::string &X = b.find(ic[0]) != std::string::npos ? b : a, &Y = &X == &a ? b : a;
    double M = 1.0, N = 1.0, K = 1.0;
    for (char c : X) (Y.find(c) != std::string::npos ? K : M) *= len(c);
    for (char c : Y)
        if (X.find(c) == std::string::npos) N *= len(c);
    ok_ = ok_ && std::max({M * K, N * K, M * N}) < double(1 << 28);
    if (int(levels_.size()) <= level) levels_.resize(size_t(level) + 1);
    DirectArgs p{};
    p.batch = 1;
    if (ok_) {
        p.M = uint32_t(M);
        p.N = uint32_t(N);
        p.K = uint32_t(K);
    }
    levels_[size_t(level)].push_back(p);
    return count_++;
}

size_t StageSizes::bytes() {
    if (!ok_) return 0;
    int64_t total = 0;
    for (auto& l : levels_) {
        std::vector<DirectArgs*> a;
        for (auto& p : l) a.push_back(&p);
        plan_stage_level(a.data(), int(a.size()));
        for (const auto& p : l) total += tile_doubles(p);
    }
    return alloc_bytes(size_t(total) * 8) + kDescBytes;
}

bool StageProgram::finish(size_t room) {
    if (!ok_) return false;   // a contraction not of the batched stage's form
    int nlevels = 0;
    for (const auto& p : products_) nlevels = std::max(nlevels, p.level + 1);
    levels_.assign(size_t(nlevels), Level{});

    // tiles of every product, one buffer; a level's long blocks come first
    int64_t total = 0;
    std::vector<int64_t> at;
    for (int l = 0; l < nlevels; ++l) {
        std::vector<DirectArgs*> a;
        for (auto& p : products_)
            if (p.level == l) a.push_back(&p.a);
        plan_stage_level(a.data(), int(a.size()));
    }
    for (auto& p : products_) {
        at.push_back(total);
        total += tile_doubles(p.a);
    }
    if (alloc_bytes(size_t(total) * 8) + kDescBytes > room) return false;
    tiles_ = tensor::Tensor(ctx_, std::vector<int64_t>{std::max<int64_t>(total, 1)}, false);
    for (size_t k = 0; k < products_.size(); ++k) products_[k].a.P = tiles_.handle()->data + at[k];

    std::vector<char> host;
    auto place = [&](const void* src, size_t bytes) {
        const size_t off = (host.size() + 15) / 16 * 16;
        host.resize(off + bytes);
        std::memcpy(host.data() + off, src, bytes);
        return off;
    };
    struct Offsets { size_t prob, first, outs, terms; };
    std::vector<Offsets> offs(static_cast<size_t>(nlevels));
    for (int l = 0; l < nlevels; ++l) {
        Level& L = levels_[size_t(l)];
        std::vector<const Product*> ps;
        for (const auto& p : products_)
            if (p.level == l) ps.push_back(&p);
        std::stable_sort(ps.begin(), ps.end(), [](const Product* x, const Product* y) {
            auto block = [](const DirectArgs& a) { return double(a.kchunk) * a.tm * a.tn; };
            return block(x->a) > block(y->a);
        });
        std::vector<DirectArgs> args;
        std::vector<uint32_t> first{0};
        for (const auto* p : ps) {
            args.push_back(p->a);
            first.push_back(first.back() + p->a.tilesM * p->a.tilesN * p->a.nsplit);
            L.flops += 2.0 * double(p->a.M) * p->a.N * p->a.K;
            L.bytes += 8.0 * (double(p->a.M) + p->a.N) * p->a.K;
        }
        L.s.np = uint32_t(args.size());
        L.s.blocks = first.back();
        std::vector<AsmOut> outs;
        std::vector<AsmTerm> terms;
        for (const auto& o : outputs_) {
            if (o.level != l) continue;
            AsmOut q{};
            const aq_tensor* t = o.t->handle();
            q.out = t->data;
            q.n = uint32_t(t->size);
            for (int k = 0; k < 4; ++k) q.len[k] = k < t->ndim ? uint32_t(t->len[size_t(k)]) : 1u;
            q.first = L.blocks;
            q.term = uint32_t(terms.size());
            q.nterms = uint32_t(o.terms.size());
            q.sym = o.sym ? 1 : 0;
            const uint32_t nt = (q.len[0] + 15) / 16;
            L.blocks += o.sym ? nt * nt * (q.len[2] * (q.len[2] + 1) / 2) : (q.n + 255) / 256;
            outs.push_back(q);
            written_.push_back(o.t);
            for (const auto& tm : o.terms) {
                AsmTerm d{};
                d.coef = tm.coef;
                d.kind = uint32_t(tm.kind);
                if (tm.kind == 0) {
                    const aq_tensor* x = tm.t->handle();
                    d.p = x->data;
                    uint32_t s = 1;
                    for (size_t k = 0; k < tm.ix.size(); ++k) {
                        d.s0[o.ic.find(tm.ix[k])] = s;
                        s *= uint32_t(x->len[k]);
                    }
                } else {
                    const Product& p = products_[size_t(tm.product)];
                    d.p = p.a.P;
                    d.ltm = log2_of(p.a.tm);
                    d.ltn = log2_of(p.a.tn);
                    d.tilesM = p.a.tilesM;
                    d.nsplit = p.a.nsplit;
                    if (tm.kind == 1)
                        for (size_t k = 0; k < p.ic.size(); ++k) {
                            d.s0[o.ic.find(p.ic[k])] = p.mulM[k];
                            d.s1[o.ic.find(p.ic[k])] = p.mulN[k];
                        }
                }
                terms.push_back(d);
            }
        }
        AQ_CHECK(args.size() <= 64 && outs.size() <= 64, AQ_ERR_INVALID, "stage level size");
        if (L.s.blocks >= kDirBlocks / kDirGroup || L.blocks >= kDirBlocks) return false;
        L.nout = int(outs.size());
        Offsets& f = offs[size_t(l)];
        f.prob = place(args.data(), args.size() * sizeof(DirectArgs));
        f.first = place(first.data(), first.size() * sizeof(uint32_t));
        f.outs = place(outs.data(), outs.size() * sizeof(AsmOut));
        f.terms = place(terms.data(), terms.size() * sizeof(AsmTerm));
    }
    desc_ = tensor::Tensor(ctx_, std::vector<int64_t>{int64_t(host.size() + 7) / 8}, false);
    char* dev = reinterpret_cast<char*>(desc_.handle()->data);
    AQ_HIP(hipMemcpyAsync(dev, host.data(), host.size(), hipMemcpyHostToDevice, ctx_->stream));
    AQ_HIP(hipStreamSynchronize(ctx_->stream));
    for (int l = 0; l < nlevels; ++l) {
        Level& L = levels_[size_t(l)];
        const Offsets& f = offs[size_t(l)];
        L.s.prob = reinterpret_cast<const DirectArgs*>(dev + f.prob);
        L.s.first = reinterpret_cast<const uint32_t*>(dev + f.first);
        L.outs = reinterpret_cast<const AsmOut*>(dev + f.outs);
        L.terms = reinterpret_cast<const AsmTerm*>(dev + f.terms);
    }
    return true;
}

void StageProgram::run() {
    for (size_t l = 0; l < levels_.size(); ++l) {
        const Level& L = levels_[l];
        if (L.s.np && !(ctx_->batcher && !ctx_->capture && batcher_offer_stage(ctx_, int(l), L.s))) {
            TimedLaunch tl(ctx_, "stage_contract", L.flops, L.bytes);
            const StageLevel* one = &L.s;
            launch_stage(&one, 1, ctx_->stream);
        }
        if (L.nout) {
            TimedLaunch tl(ctx_, "stage_assemble", 0.0, 0.0);
            launch_assemble(ctx_->stream, L.outs, L.terms, L.nout, L.blocks);
        }
    }
    for (const auto* t : written_) t->handle()->version += 1;
}

}  // namespace aqamd
