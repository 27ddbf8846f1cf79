// The scratch arena of the mesh build on a device allocator whose allocations
// lie side by side: every piece stays inside one allocation, free pieces of one
// chunk are joined again, everything is given back.  Linked against the stand-ins
// below instead of the HIP runtime.
#include <cstdio>
#include <cstdlib>
#include <map>
#include <random>

#include "vsdmo_internal.h"

static char* const kBase = reinterpret_cast<char*>(size_t(1) << 40);   // never dereferenced
static size_t g_used = 0;
static std::map<char*, size_t> g_live;
static int g_mallocs = 0, g_syncs = 0;

extern "C" {
hipError_t hipMalloc(void** p, size_t n)
{
    *p = kBase + g_used;
    g_live[kBase + g_used] = n;
    g_used += n;   // the next allocation begins where this one ends
    ++g_mallocs;
    return hipSuccess;
}
hipError_t hipFree(void* p) { return g_live.erase(static_cast<char*>(p)) == 1 ? hipSuccess : hipErrorInvalidValue; }
hipError_t hipStreamSynchronize(hipStream_t) { ++g_syncs; return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}

static void check(bool ok, const char* what)
{
    if (ok) return;
    std::printf("FAILED: %s\n", what);
    std::exit(1);
}

// the whole of [p, p + n) in one live allocation
static bool inside_one(const char* p, size_t n)
{
    for (const auto& a : g_live)
        if (p >= a.first && p + n <= a.first + a.second) return true;
    return false;
}

int main()
{
    const size_t MB = size_t(1) << 20;
    {   // two chunks whose free ends touch: a piece larger than either end
        vsdmo::BuildArena ar(0, nullptr);
        char* a = static_cast<char*>(ar.get(MB / 2));
        char* b = static_cast<char*>(ar.get(MB * 3 / 4));   // a second chunk
        char* c = static_cast<char*>(ar.get(MB / 4));       // behind a: the first chunk's last quarter is left
        check(c == a + MB / 2 && g_mallocs == 2, "first fit");
        ar.put(b);
        char* d = static_cast<char*>(ar.get(MB + MB / 8));
        check(inside_one(d, MB + MB / 8), "a piece over two chunks");
        check(g_mallocs == 3, "a chunk of its own");
        ar.put(c);
        ar.put(a);
        check(ar.get(MB) == a && g_mallocs == 3, "the first chunk in one piece again");
    }
    check(g_live.empty() && g_syncs == 1, "all given back after a wait");
    for (unsigned seed = 0; seed < 200; ++seed) {   // the sizes of small builds' arrays, in any order
        std::mt19937 r(seed);
        vsdmo::BuildArena ar(0, nullptr);
        std::map<char*, size_t> held;
        for (int k = 0; k < 400; ++k) {
            if (!held.empty() && r() % 2) {
                auto it = std::next(held.begin(), r() % held.size());
                ar.put(it->first);
                held.erase(it);
                continue;
            }
            const size_t n = 4 * (1 + r() % (MB / 8));
            char* p = static_cast<char*>(ar.get(n));
            check(inside_one(p, n), "a piece over two chunks");
            auto next = held.lower_bound(p);
            check(next == held.end() || p + n <= next->first, "overlap with the next piece");
            check(next == held.begin() || std::prev(next)->first + std::prev(next)->second <= p, "overlap with the piece before");
            held[p] = n;
        }
    }
    check(g_live.empty(), "all given back");
    std::printf("ok\n");
    return 0;
}
