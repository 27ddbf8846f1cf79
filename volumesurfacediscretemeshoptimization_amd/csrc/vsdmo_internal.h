// vsdmo_internal.h -- internal types of libvsdmo (not part of the C ABI).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cstddef>
#include <string>
#include <vector>

#include "../../include/vsdmo.h"

namespace vsdmo {

// thread-local last error message (vsdmo_last_error)
void set_error(const std::string& msg);

struct HipError {
    hipError_t code;
    std::string where;
};

#define VSDMO_HIP(expr)                                                                     \
    do {                                                                                    \
        hipError_t _e = (expr);                                                             \
        if (_e != hipSuccess) throw ::vsdmo::HipError{ _e, std::string(#expr) + " at " +    \
                                                              __FILE__ + ":" + std::to_string(__LINE__) }; \
    } while (0)

struct StatusError {
    vsdmo_status status;
    std::string msg;
};

// Device scratch of one mesh build, on one stream: a few allocations handed
// out in pieces, first fit.  hipMalloc of 4 MB and more takes ~300 us, of 2 MB
// ~50 us, up to 1 MB ~0.5 us (hipFree alike), and a hipFree waits for the
// device; a build takes some 90 pieces.  So a build that needs more than 4 MB
// takes it at once, a smaller one as it goes, in chunks of 1 MB.  A piece that
// is put back is handed out again without a wait, as everything that uses it is
// on the one stream.  The destructor waits for the stream and frees all.
class BuildArena {
public:
    BuildArena(size_t bytes, hipStream_t s) : stream_(s)
    {
        if (bytes > (size_t(4) << 20)) grow(bytes);
    }
    BuildArena(const BuildArena&) = delete;
    BuildArena& operator=(const BuildArena&) = delete;
    ~BuildArena()
    {
        (void)hipStreamSynchronize(stream_);
        for (char* c : chunks_) (void)hipFree(c);
    }
    void* get(size_t bytes)
    {
        bytes = (bytes + 255) & ~size_t(255);
        for (;;) {
            for (size_t i = 0; i < pieces_.size(); ++i) {
                if (pieces_[i].used || pieces_[i].n < bytes) continue;
                const Piece rest{ pieces_[i].p + bytes, pieces_[i].n - bytes, pieces_[i].chunk, false };
                pieces_[i].n = bytes;
                pieces_[i].used = true;
                char* const p = pieces_[i].p;
                if (rest.n) pieces_.insert(pieces_.begin() + (std::ptrdiff_t)i + 1, rest);
                return p;
            }
            grow(bytes);
        }
    }
    void put(void* q) noexcept
    {
        for (size_t i = 0; i < pieces_.size(); ++i) {
            if (pieces_[i].p != q) continue;
            pieces_[i].used = false;
            join(i);
            if (i > 0) join(i - 1);
            return;
        }
    }

private:
    struct Piece { char* p; size_t n; size_t chunk; bool used; };
    void grow(size_t bytes)
    {
        bytes = std::max(bytes, size_t(1) << 20);
        void* c = nullptr;
        VSDMO_HIP(hipMalloc(&c, bytes));
        try {
            chunks_.push_back(static_cast<char*>(c));
        } catch (...) {
            (void)hipFree(c);
            throw;
        }
        pieces_.push_back({ static_cast<char*>(c), bytes, chunks_.size() - 1, false });
    }
    // piece i with its successor, if both are free and of one chunk.  (Two chunks
    // can lie side by side, but a copy or a fill has to stay within one allocation.)
    void join(size_t i) noexcept
    {
        if (i + 1 >= pieces_.size() || pieces_[i].used || pieces_[i + 1].used) return;
        if (pieces_[i].chunk != pieces_[i + 1].chunk) return;
        pieces_[i].n += pieces_[i + 1].n;
        pieces_.erase(pieces_.begin() + (std::ptrdiff_t)i + 1);
    }
    hipStream_t stream_;
    std::vector<char*> chunks_;
    std::vector<Piece> pieces_;   // each chunk's in address order
};

// device array, its own allocation or (arena) a piece of a build's scratch
template <class T>
struct DevBuf {
    T* p = nullptr;
    size_t n = 0;
    BuildArena* arena = nullptr;
    DevBuf() = default;
    explicit DevBuf(size_t count) { alloc(count); }
    explicit DevBuf(BuildArena& a, size_t count = 0) : arena(&a) { alloc(count); }
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    DevBuf(DevBuf&& o) noexcept : p(o.p), n(o.n), arena(o.arena) { o.p = nullptr; o.n = 0; }
    DevBuf& operator=(DevBuf&& o) noexcept
    {
        if (this != &o) { release(); p = o.p; n = o.n; arena = o.arena; o.p = nullptr; o.n = 0; }
        return *this;
    }
    ~DevBuf() { release(); }
    void alloc(size_t count)
    {
        release();
        n = count;
        if (!count) return;
        if (arena) p = static_cast<T*>(arena->get(count * sizeof(T)));
        else VSDMO_HIP(hipMalloc(&p, count * sizeof(T)));
    }
    void release()
    {
        if (p && arena) arena->put(p);
        else if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    void upload(const T* h, size_t count, hipStream_t s)
    {
        if (count) VSDMO_HIP(hipMemcpyAsync(p, h, count * sizeof(T), hipMemcpyHostToDevice, s));
    }
    void download(T* h, size_t count, hipStream_t s) const
    {
        if (count) VSDMO_HIP(hipMemcpyAsync(h, p, count * sizeof(T), hipMemcpyDeviceToHost, s));
    }
    std::vector<T> to_host(hipStream_t s) const
    {
        std::vector<T> v(n);
        download(v.data(), n, s);
        VSDMO_HIP(hipStreamSynchronize(s));
        return v;
    }
};

}  // namespace vsdmo

// Mesh: device-resident vertex positions (SoA), elements, colouring and the
// one-ring structures, all in the optimiser's vertex numbering:
//   [0, nFree) free surface | [nFree, nSurf) feature surface | [nSurf, nV) inner,
// each range sorted by colour.
struct vsdmo_mesh {
    int elem = 0, npe = 0, nV = 0, nE = 0;
    int flat = 0;
    int nSurf = 0, nFree = 0, nFeature = 0, nInner = 0;
    int nFaces = 0, fpe = 0;
    int maxRing = 0, maxHE = 0, nHE = 0;
    std::vector<int> colOffInner, colOffFree, colOffFeature;  // absolute ids
    std::vector<int> new_of_old;                               // host copy
    vsdmo::DevBuf<float> x, y, z;
    vsdmo::DevBuf<int> cells;        // npe * nE
    vsdmo::DevBuf<int> faces;        // fpe * nFaces
    vsdmo::DevBuf<int> ringRow;      // nV + 1
    vsdmo::DevBuf<int> ringVal;      // stride * nnz (3 tet, 7 hex)
    vsdmo::DevBuf<int> colorOf;      // nV
    vsdmo::DevBuf<int> newOfOld;     // nV
    vsdmo::DevBuf<int> heRow, heTarget, heOpp, heFace, heNext;
    vsdmo::DevBuf<uint8_t> isB1D, isFeature;
    vsdmo::DevBuf<int> nbr;          // canonical neighbour table (learned proposal), built on demand
    // position of every one-ring corner in its vertex's neighbour table
    // (kRingLocNone: not in it), kRingLocStride(elem) bytes per ring element;
    // built with nbr
    vsdmo::DevBuf<uint8_t> ringLoc;
    hipStream_t stream = nullptr;
    int n_opts = 0;   // live optimisers referencing this mesh
};
