// DIIS extrapolation (src/convergence/diis.hpp:16-227) over device-resident
// history, shared by the closed-shell and the spin-orbital CCSD drivers.
// Not part of the C ABI.
#pragma once

#include "internal.hpp"

#include "../../include/aqamd.hpp"

#include <algorithm>
#include <cmath>
#include <limits>
#include <memory>
#include <vector>

using aqamd::tensor::Tensor;

namespace aqamd {

inline void bump_t(const Tensor& t) { t.handle()->version += 1; }
inline double* dptr(const Tensor& t) { return t.handle()->data; }
inline int64_t tsize(const Tensor& t) { return t.handle()->size; }

// Solve the (n x n) symmetric system A x = b in place (row-major A), Gaussian
// elimination with partial pivoting.  Returns 0, or k > 0 when the k-th pivot
// is exactly zero (the dsysv 'info > 0' condition, diis.hpp:171-177).
inline int solve_small(int n, std::vector<double> A, std::vector<double>& b) {
    std::vector<int> perm(n);
    for (int i = 0; i < n; ++i) perm[i] = i;
    for (int k = 0; k < n; ++k) {
        int p = k;
        for (int i = k + 1; i < n; ++i)
            if (std::fabs(A[i * n + k]) > std::fabs(A[p * n + k])) p = i;
        if (A[p * n + k] == 0.0) return k + 1;
        if (p != k) {
            for (int j = 0; j < n; ++j) std::swap(A[k * n + j], A[p * n + j]);
            std::swap(b[k], b[p]);
        }
        for (int i = k + 1; i < n; ++i) {
            const double f = A[i * n + k] / A[k * n + k];
            if (f == 0.0) continue;
            for (int j = k; j < n; ++j) A[i * n + j] -= f * A[k * n + j];
            b[i] -= f * b[k];
        }
    }
    for (int k = n - 1; k >= 0; --k) {
        double s = b[k];
        for (int j = k + 1; j < n; ++j) s -= A[k * n + j] * b[j];
        b[k] = s / A[k * n + k];
    }
    return 0;
}

// Pulay DIIS over device-resident history (diis.hpp:36-227).
class DIIS {
  public:
    DIIS(aq_ctx* ctx, int order, int start, double damping, int nx, int ndx)
        : ctx_(ctx), nextrap_(order), start_(start), damping_(damping), nx_(nx), ndx_(ndx),
          e_((order + 1) * (order + 1), 0.0), c_(order + 1, 0.0), old_x_(order), old_dx_(order) {}

    bool used_eps_retry = false;

    void extrapolate(const std::vector<Tensor*>& x, const std::vector<Tensor*>& dx) {
        if (nextrap_ > 1) extrapolate(x, dx, [] {});
    }

    // `synced` is called once, after the first synchronisation of the stream
    // (results of reductions queued before this call are then on the host).
    template <class F>
    void extrapolate(const std::vector<Tensor*>& x, const std::vector<Tensor*>& dx, F&& synced) {
        const int n = nextrap_, n1 = n + 1;
        if (n <= 1) {
            AQ_HIP(hipStreamSynchronize(ctx_->stream));
            resolve_timing(ctx_);
            synced();
            return;
        }
        // slot k holds iteration n-k (diis.hpp:82-85)
        std::rotate(old_x_.begin(), old_x_.end() - 1, old_x_.end());
        std::rotate(old_dx_.begin(), old_dx_.end() - 1, old_dx_.end());
        {
            std::vector<double> r(e_.size());
            for (int i = 0; i < n1; ++i)
                for (int j = 0; j < n1; ++j) r[i * n1 + j] = e_[((i + n) % n1) * n1 + (j + n) % n1];
            e_.swap(r);
            std::rotate(c_.begin(), c_.end() - 1, c_.end());
        }
        // the newest slots (:92-120): the residuals are stored by the launch
        // that forms their products, x by the extrapolation (or `keep`)
        try {
            reserve(old_x_[0], x);
            reserve(old_dx_[0], dx);
        } catch (...) {   // the caller's results are there all the same
            if (hipStreamSynchronize(ctx_->stream) == hipSuccess) synced();
            throw;
        }

        // e[i][0] = <dx, old_dx[i]> for every stored slot (:122-135)
        int nreal = 1;
        while (nreal < n && !old_dx_[nreal].empty()) ++nreal;
        std::vector<double> p(nreal, 0.0);
        // up to kDiisDots history slots and kDiisSegs tensors per launch; each
        // inner product is reduced on its own, so the grouping does not
        // change any value
        bool told = false;
        for (int j0 = 0; j0 < ndx_; j0 += kDiisSegs) {
            const int nj = std::min(kDiisSegs, ndx_ - j0);
            for (int first = 0; first < nreal; first += kDiisDots) {
                const int kk = std::min(kDiisDots, nreal - first);
                DiisDot seg[kDiisSegs];
                for (int j = 0; j < nj; ++j) {
                    seg[j].x = dptr(*dx[j0 + j]);
                    seg[j].copy = first == 0 ? dptr(old_dx_[0][j0 + j]) : nullptr;
                    for (int i = 0; i < kk; ++i) seg[j].y[i] = dptr(old_dx_[first + i][j0 + j]);
                    seg[j].n = tsize(*dx[j0 + j]);
                }
                launch_diis_dot(ctx_, nj, seg, kk, kFirstSlot);
                AQ_HIP(hipStreamSynchronize(ctx_->stream));
                if (!told) synced();
                told = true;
                for (int j = 0; j < nj; ++j)
                    for (int i = 0; i < kk; ++i) p[first + i] += ctx_->h_result[kFirstSlot + j * kDiisDots + i];
            }
        }
        if (!told) {
            AQ_HIP(hipStreamSynchronize(ctx_->stream));
            synced();
        }
        resolve_timing(ctx_);
        for (auto& t : old_dx_[0]) bump_t(t);
        E(0, 0) = p[0];
        for (int i = 1; i < nreal; ++i) {
            E(i, 0) = p[i];
            E(0, i) = p[i];
        }
        for (int i = 0; i < nreal; ++i) {   // :141-149
            E(i, nreal) = -1.0;
            E(nreal, i) = -1.0;
            c_[i] = 0.0;
        }
        E(nreal, nreal) = 0.0;
        c_[nreal] = -1.0;

        if (nreal == 1) {         // :151
            keep(x);
            return;
        }

        if (--start_ > 1) {       // :153-164
            keep(x);
            if (damping_ > 0.0) {
                const double cf[2] = {damping_ - 1.0, damping_};
                for (int i = 0; i < nx_; ++i) {
                    double* a = dptr(old_x_[0][i]);
                    const DiisComb seg{a, nullptr, {a, dptr(old_x_[1][i])}, tsize(old_x_[0][i])};
                    launch_diis_combine(ctx_, 1, &seg, cf, 2);
                    bump_t(old_x_[0][i]);
                }
            }
            return;
        }

        const int m = nreal + 1;   // :166-188
        auto sub = [&]() {
            std::vector<double> A(m * m);
            for (int i = 0; i < m; ++i)
                for (int j = 0; j < m; ++j) A[i * m + j] = E(i, j);
            return A;
        };
        std::vector<double> b(c_.begin(), c_.begin() + m);
        std::vector<double> A = sub();
        int info = solve_small(m, A, b);
        used_eps_retry = false;
        if (info > 0) {
            const double eps = E(nreal - 1, nreal - 1) * std::numeric_limits<double>::epsilon();
            A = sub();
            for (int i = 0; i < nreal; ++i) A[i * m + i] += eps;
            b.assign(c_.begin(), c_.begin() + m);
            info = solve_small(m, A, b);
            used_eps_retry = true;
        }
        if (info != 0) keep(x);
        AQ_CHECK(info == 0, AQ_ERR_NUMERIC, "DIIS: Info in hesv: " + std::to_string(info));
        for (int i = 0; i < m; ++i) c_[i] = b[i];

        // x = sum_i c_i old_x[i], dx = sum_i c_i old_dx[i] (:205-226), the
        // newest term read from x (then stored into its slot) and dx itself
        std::vector<DiisComb> seg;
        const bool apart = distinct(x, dx);
        if (!apart) keep(x);      // a tensor listed twice is overwritten only from stored copies, in order
        for (int j = 0; j < ndx_; ++j) seg.push_back(terms(dx[j], apart, nullptr, old_dx_, j, nreal));
        for (int j = 0; j < nx_; ++j) seg.push_back(terms(x[j], apart, dptr(old_x_[0][j]), old_x_, j, nreal));
        const size_t per = apart ? kDiisSegs : 1;
        for (size_t q = 0; q < seg.size(); q += per)
            launch_diis_combine(ctx_, int(std::min(per, seg.size() - q)), &seg[q], c_.data(), nreal);
        for (int j = 0; j < ndx_; ++j) bump_t(*dx[j]);
        for (int j = 0; j < nx_; ++j) bump_t(*x[j]);
        for (auto& t : old_x_[0]) bump_t(t);
    }

    const std::vector<double>& coefficients() const { return c_; }

  private:
    double& E(int i, int j) { return e_[i * (nextrap_ + 1) + j]; }

    // first reduction slot of the inner products; a caller's results that are
    // read by `synced` sit below it
    static constexpr int kFirstSlot = kRedSlots - kDiisSegs * kDiisDots;

    void reserve(std::vector<Tensor>& slot, const std::vector<Tensor*>& src) {
        if (!slot.empty()) return;
        std::vector<Tensor> s;   // all of them or, when one does not fit, none
        for (auto* t : src) s.emplace_back(ctx_, t->lengths(), false);
        slot = std::move(s);
    }
    // x into its newest history slot
    void keep(const std::vector<Tensor*>& x) {
        for (size_t i = 0; i < x.size(); ++i) {
            AQ_HIP(hipMemcpyAsync(dptr(old_x_[0][i]), dptr(*x[i]), size_t(tsize(*x[i])) * 8,
                                  hipMemcpyDeviceToDevice, ctx_->stream));
            bump_t(old_x_[0][i]);
        }
    }
    static bool distinct(const std::vector<Tensor*>& x, const std::vector<Tensor*>& dx) {
        std::vector<const double*> p;
        for (auto* t : x) p.push_back(dptr(*t));
        for (auto* t : dx) p.push_back(dptr(*t));
        std::sort(p.begin(), p.end());
        return std::adjacent_find(p.begin(), p.end()) == p.end();
    }
    // the combination for tensor j; live: its newest term is `t` as it stands,
    // and goes to `copy`
    static DiisComb terms(Tensor* t, bool live, double* copy, std::vector<std::vector<Tensor>>& old, int j, int nreal) {
        DiisComb s{dptr(*t), live ? copy : nullptr, {live ? dptr(*t) : dptr(old[0][j])}, tsize(*t)};
        for (int i = 1; i < nreal; ++i) s.x.push_back(dptr(old[i][j]));
        return s;
    }

    aq_ctx* ctx_;
    int nextrap_, start_;
    double damping_;
    int nx_, ndx_;
    std::vector<double> e_, c_;
    std::vector<std::vector<Tensor>> old_x_, old_dx_;
};

}  // namespace aqamd
