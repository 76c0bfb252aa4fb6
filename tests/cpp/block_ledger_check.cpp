// The server's block bookkeeping (aqamd::BlockLedger, aqamd::SlotBlocks) under
// the server's own rules, without a device: jobs are admitted against a budget,
// allocate in blocks up to their reservations, free some on the way and all at
// their end, in random order.  After every step all that is held (in use, freed
// by running jobs, and kept) is within the budget; every block handed out fits
// its request, at most an eighth larger, is not in use, and comes from the same
// job or from one that has ended; nothing is in use at the end.  Prints the number
// of reused blocks per budget.  Exit status: violations found.
#include "../../aquarius_amd/csrc/blocks.hpp"

#include <cstdint>
#include <cstdio>
#include <map>
#include <random>
#include <vector>

using aqamd::BlockLedger;
using aqamd::KeptBlock;

struct Job {
    size_t reserved = 0, charged = 0;
    std::map<void*, size_t> mine;   // block -> charged bytes
    aqamd::SlotBlocks own;
    int id = 0;
    int steps = 0;
};

int main() {
    int bad = 0;
    std::mt19937_64 rng(11);
    auto uni = [&](double lo, double hi) { return lo + (hi - lo) * double(rng() >> 11) / 9007199254740992.0; };
    for (size_t budget : {size_t(1000000), size_t(64000000), size_t(3000000000)}) {
        BlockLedger led;
        led.limit = budget;
        size_t reserved = 0, device = 0;          // device: bytes allocated and not freed
        std::map<void*, size_t> size;             // every live block
        std::map<void*, int> used;
        std::vector<Job> run;
        uintptr_t next = 1;
        long reused = 0;
        const size_t shapes[6] = {budget / 97, budget / 61, budget / 60, budget / 23, budget / 11, budget / 10};
        std::map<void*, int> pending;             // freed by a running job -> its id
        int ids = 0;
        auto drop = [&](const KeptBlock& b) {
            device -= size[b.p];
            size.erase(b.p);
            pending.erase(b.p);
        };
        auto settle = [&] {
            while (led.over()) drop(led.pop_oldest());
        };
        auto give = [&](Job& j, void* p, bool drained) {
            const BlockLedger::Lent l = led.back(p);
            if (l.bytes != size[p] || l.asked != j.mine[p]) ++bad;
            used[p] -= 1;
            const KeptBlock b{p, l.bytes};
            if (drained && led.fits(l.bytes)) {
                led.keep(b);
                settle();
            } else if (!drained && j.charged - l.asked + j.own.bytes + l.bytes <= j.reserved) {
                j.own.keep(b);
                pending[p] = j.id;
            } else {
                drop(b);
            }
            j.charged -= j.mine[p];
            j.mine.erase(p);
        };
        auto end = [&](Job& j) {
            while (!j.own.blocks.empty()) {
                const KeptBlock b = j.own.pop_oldest();
                pending.erase(b.p);
                if (led.fits(b.bytes)) {
                    led.keep(b);
                    settle();
                } else {
                    drop(b);
                }
            }
            while (!j.mine.empty()) give(j, j.mine.begin()->first, true);
            reserved -= j.reserved;
            led.limit = budget - reserved;
        };
        auto check = [&] {
            if (device > budget) ++bad;
            if (led.kept() + reserved > budget) ++bad;
            if (led.kept() + led.slack() > led.limit && !led.empty()) ++bad;
        };
        for (int step = 0; step < 20000; ++step) {
            if (run.size() < 4 && uni(0, 1) < 0.3) {
                const size_t need = size_t(uni(0.02, 0.9) * double(budget));
                const size_t held = reserved ? reserved + led.slack() : 0;
                if (held + need <= budget) {
                    reserved += need;
                    led.limit = budget - reserved;
                    settle();
                    Job j;
                    j.reserved = need;
                    j.id = ++ids;
                    j.steps = int(uni(1, 60));
                    run.push_back(j);
                }
            } else if (!run.empty()) {
                const size_t k = size_t(uni(0, double(run.size()) - 1e-9));
                Job& j = run[k];
                if (--j.steps < 0) {
                    end(j);
                    run.erase(run.begin() + long(k));
                } else if (uni(0, 1) < 0.7 || j.mine.empty()) {
                    const size_t n = size_t(double(shapes[rng() % 6]) * uni(0.95, 1.0)) + 1;
                    if (j.charged + n <= j.reserved) {
                        KeptBlock b;
                        void* p = nullptr;
                        const size_t spare = led.limit > led.slack() ? led.limit - led.slack() : 0;
                        if (j.own.take(n, spare, b)) {
                            if (pending[b.p] != j.id) ++bad;
                            pending.erase(b.p);
                            led.lend(b.p, b.bytes, n);
                            settle();
                        } else if (led.take(n, b)) {
                            if (pending.count(b.p)) ++bad;
                        } else {
                            while (!j.own.blocks.empty() && j.charged + n + j.own.bytes > j.reserved) drop(j.own.pop_oldest());
                            b = KeptBlock{};
                        }
                        if (b.p) {
                            p = b.p;
                            ++reused;
                            if (b.bytes < n || b.bytes - n > n / 8 || size.count(p) == 0) ++bad;
                        } else {
                            p = reinterpret_cast<void*>(next++);
                            size[p] = n;
                            device += n;
                            led.lend(p, n, n);
                        }
                        if (++used[p] != 1) ++bad;
                        j.mine[p] = n;
                        j.charged += n;
                    }
                } else {
                    give(j, j.mine.begin()->first, false);
                }
            }
            check();
        }
        for (auto& j : run) end(j);
        if (led.slack() != 0 || led.kept() != device) ++bad;
        led.limit = 0;
        settle();
        if (device != 0 || !led.empty()) ++bad;
        std::printf("budget %zu: %ld blocks reused\n", budget, reused);
    }
    if (bad) std::printf("%d violations\n", bad);
    return bad != 0;
}
