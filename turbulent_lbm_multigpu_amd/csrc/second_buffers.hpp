// second_buffers.hpp -- the second buffers of the solvers that took fused pairs
// (pair_kernel).  Plain C++: device memory comes in as SecondMemory, so the
// bookkeeping, which threads with a solver each share, is checked on the CPU.
#pragma once

#include <stddef.h>

#include <atomic>
#include <iterator>
#include <mutex>
#include <set>
#include <shared_mutex>
#include <vector>

namespace lbm {

// One device allocation holding the second buffers of one solver or of the
// members of a group.
struct SecondBlock {
    void *base = nullptr;
    size_t bytes = 0;
    int device = 0;
    int refs = 0;
};

// A solver's second buffer.  `at` is read by the solver's own thread; another
// thread may take it away between launches (give_all).
struct SecondBuffer {
    std::atomic<void *> at{nullptr};
    std::atomic<unsigned> *version = nullptr;  // bumped when `at` changes
    size_t bytes = 0;                          // what the solver needs
    int device = 0;
    size_t refused = 0;                        // > 0: there was no memory for so much,
    int wait = 0;                              // and as many sequences go by before it is asked for again
    SecondBlock *block = nullptr;
};

struct SecondMemory {
    virtual ~SecondMemory() = default;
    virtual void *allocate(int device, size_t bytes) = 0;  // null: not to be had
    virtual void release(void *base) = 0;
    virtual void drain(int device) = 0;  // waits for the launches that still use them
};

// They are a use of memory that nothing depends on: where an allocation of
// this library fails, they are given back and it is tried again.  Launches
// that use them hold in_use(), so none is enqueued while they are taken away;
// only that waits for them.  A sequence may be enqueued for as long as it runs
// (the queue is bounded), and nothing else of one thread waits for another's.
// The blocks of the last few destroyed solvers are kept for the next ones (an
// allocation costs a short run more than it gains): at most kSpares,
// kSpareBytes in all, until release_spares().
class SecondBuffers {
  public:
    static constexpr size_t kSpares = 8, kSpareBytes = (size_t)4 << 30;
    // Sequences that step in place after a refusal: asking takes the runtime a
    // good part of a short one, and the memory may be there later.
    static constexpr int kWait = 63;
    explicit SecondBuffers(SecondMemory &memory) : memory_(memory) {}

    // Gives these (of one device) their second buffers, those without one in a
    // block together; false if they have to do without.
    // Under in_use() they may have gone again.
    bool take(const std::vector<SecondBuffer *> &all) {
        std::vector<SecondBuffer *> without;
        size_t bytes = 0;
        for (SecondBuffer *s : all) {
            if (s->at) continue;
            without.push_back(s);
            bytes += aligned(s->bytes);
        }
        if (without.empty()) return true;
        bool wait = false;
        for (SecondBuffer *s : without) {
            if (s->wait == 0 || bytes < s->refused) continue;
            --s->wait;
            wait = true;
        }
        if (wait) return false;
        const std::lock_guard<std::mutex> lock(mutex_);
        const int device = without[0]->device;
        SecondBlock *b = nullptr;
        const auto spare = spare_for(device, bytes);
        if (spare != spares_.end()) {
            b = *spare;
            spare_bytes_ -= b->bytes;
            spares_.erase(spare);
        } else {
            void *const p = memory_.allocate(device, bytes);
            if (!p) {
                for (SecondBuffer *s : without) {
                    s->refused = bytes;
                    s->wait = kWait;
                }
                return false;
            }
            b = new SecondBlock{p, bytes, device, 0};
        }
        size_t off = 0;
        for (SecondBuffer *s : without) {
            s->block = b;
            b->refs++;
            s->wait = 0;
            s->at = (char *)b->base + off;
            off += aligned(s->bytes);
            held_.insert(s);
            (*s->version)++;
        }
        return true;
    }

    // Whether a block that is kept would do for these, so that none is allocated;
    // not, while another thread allocates or takes away: asking does not wait.
    bool has_spare(const std::vector<SecondBuffer *> &all) {
        size_t bytes = 0;
        for (SecondBuffer *s : all)
            if (!s->at) bytes += aligned(s->bytes);
        const std::unique_lock<std::mutex> lock(mutex_, std::try_to_lock);
        return lock.owns_lock() && !all.empty() && spare_for(all[0]->device, bytes) != spares_.end();
    }

    // A solver's last call.  The lock is taken before `at` is looked at: while
    // give_all is at work on this buffer, `at` may be null already with other
    // members still to be written, and the solver is freed when this returns.
    void give(SecondBuffer &s) {
        const std::lock_guard<std::mutex> lock(mutex_);
        drop(s);
    }

    // Takes away every second buffer and spare of the device; whether there were any.
    bool give_all(int device) {
        const std::lock_guard<std::mutex> gate(gate_);
        const std::unique_lock<std::shared_mutex> none_launching(launches_);
        const std::lock_guard<std::mutex> lock(mutex_);
        std::vector<SecondBuffer *> here;
        for (SecondBuffer *s : held_)
            if (s->device == device) here.push_back(s);
        if (here.empty() && spares_.empty()) return false;
        memory_.drain(device);
        for (SecondBuffer *s : here) drop(*s);
        free_spares(0, 0);
        return true;
    }

    // Frees the blocks that are kept for solvers to come.
    void release_spares() {
        const std::lock_guard<std::mutex> lock(mutex_);
        free_spares(0, 0);
    }

    std::shared_lock<std::shared_mutex> in_use() {
        const std::lock_guard<std::mutex> gate(gate_);  // behind a give_all that waits: its turn comes
        return std::shared_lock<std::shared_mutex>(launches_);
    }

  private:
    static size_t aligned(size_t bytes) { return (bytes + 255) & ~(size_t)255; }
    // The newest that is not more than twice as large.
    std::vector<SecondBlock *>::iterator spare_for(int device, size_t bytes) {
        for (auto it = spares_.end(); it != spares_.begin();) {
            --it;
            if ((*it)->device == device && (*it)->bytes >= bytes && (*it)->bytes <= 2 * bytes) return it;
        }
        return spares_.end();
    }
    void free_spares(size_t keep_bytes, size_t keep) {
        while (!spares_.empty() && (spare_bytes_ > keep_bytes || spares_.size() > keep)) {
            SecondBlock *b = spares_.front();
            memory_.release(b->base);
            spare_bytes_ -= b->bytes;
            spares_.erase(spares_.begin());
            delete b;
        }
    }
    void drop(SecondBuffer &s) {
        if (!s.at) return;
        s.at = nullptr;
        (*s.version)++;
        held_.erase(&s);
        SecondBlock *b = s.block;
        s.block = nullptr;
        if (--b->refs > 0) return;
        spares_.push_back(b);
        spare_bytes_ += b->bytes;
        free_spares(kSpareBytes, kSpares);
    }

    SecondMemory &memory_;
    std::mutex gate_;
    std::shared_mutex launches_;
    std::mutex mutex_;  // of what follows and of every buffer's block
    std::set<SecondBuffer *> held_;
    std::vector<SecondBlock *> spares_;  // oldest first
    size_t spare_bytes_ = 0;
};

}  // namespace lbm
