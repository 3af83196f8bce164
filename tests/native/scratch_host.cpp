// Host build of the workspaces' growth rules (scratch.h) over a counted heap for CPU tests.
#include "../../fk20-cuda_amd/csrc/scratch.h"

#include <cstdlib>
#include <map>

static std::map<void *, size_t> g_blocks;
static size_t g_used, g_limit;
static unsigned g_allocs, g_idles;
static bool g_busy;

struct Heap {
    static bool alloc(void **p, size_t bytes) {
        g_allocs++;
        if (g_used + bytes > g_limit) return false;
        *p = malloc(1);
        g_blocks[*p] = bytes;
        g_used += bytes;
        return true;
    }
    static void release(void *p) {
        g_used -= g_blocks.at(p);
        g_blocks.erase(p);
        free(p);
    }
    static bool idle() {
        g_idles++;
        return !g_busy;
    }
};

static fk20::Workspace<Heap> g_ws[2];

extern "C" {
void scratch_host_reset(size_t limit) {
    for (auto &w : g_ws) w.drop();
    g_limit = limit;
    g_allocs = g_idles = 0;
    g_busy = false;
}
void scratch_host_set(size_t limit, int busy) {
    g_limit = limit;
    g_busy = busy != 0;
}
int scratch_host_fit(int k, size_t need, size_t want) { return (int)g_ws[k].fit(need, want); }
void scratch_host_try_grow(int k, size_t bytes) { g_ws[k].try_grow(bytes); }
int scratch_host_give_back(int k) { return g_ws[k].give_back(); }
size_t scratch_host_bytes(int k) { return g_ws[k].bytes(); }
const void *scratch_host_ptr(int k) { return g_ws[k].ptr(); }
size_t scratch_host_used(void) { return g_used; }
unsigned scratch_host_allocs(void) { return g_allocs; }
unsigned scratch_host_idles(void) { return g_idles; }
}
