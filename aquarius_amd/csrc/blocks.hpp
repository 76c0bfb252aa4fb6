// Bookkeeping of the device blocks that a server keeps between its jobs: no
// device calls, so that the bound can be checked on the host (context.cpp does
// the waits and the frees).
//
// Blocks go out at the size they were allocated with, so a reused block may be
// larger than what was asked for; a context is charged what it asked for, and
// the rest is `slack`.  The server sets `limit` to what its budget leaves beside
// the reservations of its running jobs.  Jobs hold at most their reservations
// plus the slack, so while kept + slack <= limit, all that the server has from
// the device stays within its budget.
#pragma once

#include <algorithm>
#include <cstddef>
#include <list>
#include <unordered_map>

namespace aqamd {

class BlockLedger {
  public:
    struct Block {
        void* p = nullptr;
        size_t bytes = 0;
        void* stream = nullptr;   // of its last use
        void* freed = nullptr;    // event behind its last use
    };

    size_t limit = 0;
    size_t kept() const { return kept_; }
    size_t slack() const { return slack_; }
    bool empty() const { return blocks_.empty(); }
    bool over() const { return !blocks_.empty() && kept_ + slack_ > limit; }
    bool fits(size_t bytes) const { return bytes + slack_ <= limit; }

    // The smallest kept block for a request of n bytes, at most an eighth larger;
    // false: none.  kept + slack falls by n.
    bool take(size_t n, Block& b) {
        auto best = blocks_.end();
        for (auto it = blocks_.begin(); it != blocks_.end(); ++it)
            if (it->bytes >= n && it->bytes - n <= n / 8 && (best == blocks_.end() || it->bytes < best->bytes)) best = it;
        if (best == blocks_.end()) return false;
        lend(best->p, best->bytes, n);
        b = *best;
        kept_ -= best->bytes;
        blocks_.erase(best);
        return true;
    }
    // A block of `bytes` is in use by a context that is charged `asked`.
    void lend(void* p, size_t bytes, size_t asked) {
        lent_[p] = {bytes, asked};
        slack_ += bytes - asked;
    }
    // A block in use comes back (it is then kept or freed); its bytes, or 0: not lent here.
    size_t back(void* p) {
        auto it = lent_.find(p);
        if (it == lent_.end()) return 0;
        const size_t bytes = it->second.bytes;
        slack_ -= bytes - it->second.asked;
        lent_.erase(it);
        return bytes;
    }
    void keep(const Block& b) {
        blocks_.push_back(b);
        kept_ += b.bytes;
    }
    Block pop_oldest() {
        const Block b = blocks_.front();
        blocks_.pop_front();
        kept_ -= b.bytes;
        return b;
    }

  private:
    struct Lent {
        size_t bytes, asked;
    };
    std::list<Block> blocks_;                    // kept, oldest first
    std::unordered_map<void*, Lent> lent_;       // in use
    size_t kept_ = 0, slack_ = 0;
};

}  // namespace aqamd
