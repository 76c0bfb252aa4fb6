// Bookkeeping of the device blocks that a server keeps between its jobs: no
// device calls, so that the bound can be checked on the host (context.cpp does
// the frees).
//
// Blocks go out at the size they were allocated with, so a reused block may be
// larger than what was asked for; a context is charged what it asked for, and
// the rest is `slack`.  The server sets `limit` to what its budget leaves beside
// the reservations of its running jobs.  A job holds at most its reservation (in
// use, and freed on its own stream: SlotBlocks) plus the slack, so while
// kept + slack <= limit, all that the server has from the device stays within
// its budget.
#pragma once

#include <algorithm>
#include <cstddef>
#include <list>
#include <unordered_map>

namespace aqamd {

struct KeptBlock {
    void* p = nullptr;
    size_t bytes = 0;
};

// The smallest of `blocks` for a request of n bytes, at most `waste` and an eighth larger.
inline std::list<KeptBlock>::iterator best_block(std::list<KeptBlock>& blocks, size_t n, size_t waste) {
    auto best = blocks.end();
    const size_t most = n + std::min(n / 8, waste);
    for (auto it = blocks.begin(); it != blocks.end(); ++it)
        if (it->bytes >= n && it->bytes <= most && (best == blocks.end() || it->bytes < best->bytes)) best = it;
    return best;
}

// Idle blocks, for any slot, and the sizes of those in use.
class BlockLedger {
  public:
    size_t limit = 0;
    size_t kept() const { return kept_; }
    size_t slack() const { return slack_; }
    bool empty() const { return blocks_.empty(); }
    bool over() const { return !blocks_.empty() && kept_ + slack_ > limit; }
    bool fits(size_t bytes) const { return bytes + slack_ <= limit; }

    // An idle block for n bytes; false: none.  kept + slack falls by n.
    bool take(size_t n, KeptBlock& b) {
        auto it = best_block(blocks_, n, n);
        if (it == blocks_.end()) return false;
        lend(it->p, it->bytes, n);
        b = *it;
        kept_ -= it->bytes;
        blocks_.erase(it);
        return true;
    }
    // A block of `bytes` is in use by a context that is charged `asked`.
    void lend(void* p, size_t bytes, size_t asked) {
        lent_[p] = {bytes, asked};
        slack_ += bytes - asked;
    }
    struct Lent {
        size_t bytes = 0, asked = 0;
    };
    // A block in use comes back; bytes = 0: not lent here.
    Lent back(void* p) {
        auto it = lent_.find(p);
        if (it == lent_.end()) return {};
        const Lent l = it->second;
        slack_ -= l.bytes - l.asked;
        lent_.erase(it);
        return l;
    }
    void keep(const KeptBlock& b) {
        blocks_.push_back(b);
        kept_ += b.bytes;
    }
    KeptBlock pop_oldest() {
        const KeptBlock b = blocks_.front();
        blocks_.pop_front();
        kept_ -= b.bytes;
        return b;
    }

  private:
    std::list<KeptBlock> blocks_;                // oldest first
    std::unordered_map<void*, Lent> lent_;
    size_t kept_ = 0, slack_ = 0;
};

// What a running job has freed and may still be read by work on its slot's stream:
// for that slot only, within the job's reservation.
struct SlotBlocks {
    std::list<KeptBlock> blocks;                 // oldest first
    size_t bytes = 0;

    bool take(size_t n, size_t waste, KeptBlock& b) {
        auto it = best_block(blocks, n, waste);
        if (it == blocks.end()) return false;
        b = *it;
        bytes -= it->bytes;
        blocks.erase(it);
        return true;
    }
    void keep(const KeptBlock& b) {
        blocks.push_back(b);
        bytes += b.bytes;
    }
    KeptBlock pop_oldest() {
        const KeptBlock b = blocks.front();
        blocks.pop_front();
        bytes -= b.bytes;
        return b;
    }
};

}  // namespace aqamd
