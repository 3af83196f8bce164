// Workspaces that grow on demand.  A larger workspace than a call needs only makes it faster, so
// memory that is short never refuses a call that its smallest form fits.  The memory calls are a
// parameter, so that the CPU tests can let them fail.
#pragma once
#include <stddef.h>

namespace fk20 {

// Mem: static bool alloc(void **p, size_t bytes), static void release(void *p), and
// static bool idle(), which waits for the work that may still use a buffer.
template <class Mem>
class Workspace {
  public:
    enum Fit { KEPT, MOVED, FAILED };
    void *ptr() const { return p_; }
    size_t bytes() const { return bytes_; }
    // whether fit(need, ..) has nothing to do
    bool holds(size_t need) const { return need <= need_; }

    // At least `need` bytes.  The buffer only moves (its old address dies) for a call that needs
    // more than every one before it, and then takes `want` bytes if they are there: a captured
    // graph stays valid through any smaller call, however much that one would want.
    Fit fit(size_t need, size_t want) {
        if (need <= need_) return KEPT;
        if (want < need) want = need;
        if (want <= bytes_) {
            need_ = need;
            return KEPT;
        }
        if (p_) {
            if (!Mem::idle()) return FAILED;
            drop();
        }
        if (!Mem::alloc(&p_, want)) {
            p_ = nullptr;
            want = need;
            if (!Mem::alloc(&p_, want)) {
                p_ = nullptr;
                return FAILED;
            }
        }
        bytes_ = want;
        need_ = need;
        return MOVED;
    }

    // As many of `bytes` as there are: the old buffer is kept where no larger one can be had.
    void try_grow(size_t bytes) {
        if (bytes <= bytes_) return;
        void *q = nullptr;
        if (!Mem::alloc(&q, bytes)) return;
        if (p_) {
            if (!Mem::idle()) {
                Mem::release(q);
                return;
            }
            drop();
        }
        p_ = q;
        bytes_ = bytes;
    }

    // Gives the buffer back; false if there is none or it may still be used.
    bool give_back() {
        if (!p_ || !Mem::idle()) return false;
        drop();
        return true;
    }

    void drop() {
        if (p_) Mem::release(p_);
        p_ = nullptr;
        bytes_ = need_ = 0;
    }

  private:
    void *p_ = nullptr;
    size_t bytes_ = 0, need_ = 0;
};

}  // namespace fk20
