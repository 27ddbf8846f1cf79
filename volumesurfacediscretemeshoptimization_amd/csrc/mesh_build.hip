// mesh_build.hip -- GPU construction of the DMO mesh structures.
//
// Steps (reference files under VSDMO/src/mesh):
//   boundary faces    MeshTetGPU.cu:178-200 / MeshHexGPU.cu:141-163,
//                     MeshGPUCommon.cu:25-94 (rotate smallest-first, sort,
//                     cancel opposite-orientation twins), :1376-1430
//   [surface|inner]   MeshTetGPU.cu:241-262 (stable partition)
//   colouring         MeshTetGPU.cu:298-392, VertexColoring.cu:76-125
//   colour sort       MeshTetGPU.cu:264-295 (stable sort of a range by colour)
//   one-ring CSR      MeshTetGPU.cu:113-142, MeshHexGPU.cu:116-139,
//                     MeshGPUCommon.cu:1313-1369
// Every step is deterministic: sorts are counting sorts followed by a per-row
// sort on the original index, so the output never depends on atomic order.
#include <algorithm>
#include <map>
#include <numeric>

#include "vsdmo_internal.h"
#include "vsdmo_numerics.h"

namespace vsdmo {

constexpr int TB = 256;
static inline int nblk(long long n, int tb = TB) { return (int)std::max<long long>(1, (n + tb - 1) / tb); }

// ------------------------------------------------------------------ scan
constexpr int SCAN_TB = 256;
constexpr int SCAN_PER = 4;
constexpr int SCAN_CHUNK = SCAN_TB * SCAN_PER;

__global__ void k_scan_chunk(const int* __restrict__ in, int* __restrict__ out, int* __restrict__ sums, int n)
{
    __shared__ int s[SCAN_TB];
    const int base = blockIdx.x * SCAN_CHUNK + threadIdx.x * SCAN_PER;
    int v[SCAN_PER];
    int t = 0;
#pragma unroll
    for (int i = 0; i < SCAN_PER; ++i) {
        v[i] = (base + i < n) ? in[base + i] : 0;
        t += v[i];
    }
    s[threadIdx.x] = t;
    __syncthreads();
    for (int off = 1; off < SCAN_TB; off <<= 1) {
        int a = (threadIdx.x >= off) ? s[threadIdx.x - off] : 0;
        __syncthreads();
        s[threadIdx.x] += a;
        __syncthreads();
    }
    int run = s[threadIdx.x] - t;  // exclusive prefix of this thread
#pragma unroll
    for (int i = 0; i < SCAN_PER; ++i) {
        if (base + i < n) out[base + i] = run;
        run += v[i];
    }
    if (threadIdx.x == SCAN_TB - 1 && sums) sums[blockIdx.x] = s[threadIdx.x];
}

__global__ void k_scan_add(int* __restrict__ out, const int* __restrict__ sums, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] += sums[i / SCAN_CHUNK];
}

// Read-back slots of the build steps, per host thread and device: a few
// device ints, the partial sums of the scans (grown on demand) and pinned
// host ints, so that a scalar comes back with one small DMA and one
// synchronisation.  Allocated on first use and kept for the life of the
// process (freeing them at thread exit could run after the HIP runtime has
// shut down).
struct BuildSlots {
    int* dev = nullptr;      // kSlots ints
    int* host = nullptr;     // kSlots pinned ints
    int* sums = nullptr;     // scan partial sums
    size_t sumsCap = 0;
};
constexpr int kSlots = 16;

static BuildSlots& build_slots(size_t sumsNeed = 0)
{
    thread_local std::map<int, BuildSlots> slots;
    int d = 0;
    VSDMO_HIP(hipGetDevice(&d));
    BuildSlots& b = slots[d];
    if (!b.dev) {
        VSDMO_HIP(hipMalloc(&b.dev, kSlots * sizeof(int)));
        VSDMO_HIP(hipHostMalloc(reinterpret_cast<void**>(&b.host), kSlots * sizeof(int), hipHostMallocDefault));
    }
    if (sumsNeed > b.sumsCap) {
        if (b.sums) VSDMO_HIP(hipFree(b.sums));
        b.sums = nullptr;
        const size_t cap = std::max<size_t>(sumsNeed, 4096);
        VSDMO_HIP(hipMalloc(&b.sums, cap * sizeof(int)));
        b.sumsCap = cap;
    }
    return b;
}

// n <= kSlots ints of device memory, read back through the pinned slots
const int* read_ints(const int* d, int n, hipStream_t s)
{
    BuildSlots& b = build_slots();
    VSDMO_HIP(hipMemcpyAsync(b.host, d, n * sizeof(int), hipMemcpyDeviceToHost, s));
    VSDMO_HIP(hipStreamSynchronize(s));
    return b.host;
}
int read_int(const int* d, hipStream_t s) { return read_ints(d, 1, s)[0]; }

__global__ void k_copy_int(const int* __restrict__ src, int* __restrict__ dst) { *dst = *src; }
__global__ void k_scan_total(const int* __restrict__ out, int n, const int* __restrict__ last, int* __restrict__ total)
{
    *total = out[n - 1] + *last;
}

// partial-sum ints the scan of n values needs over all its levels
static size_t scan_sums_need(int n)
{
    size_t need = 0;
    for (long long m = n; m > SCAN_CHUNK;) {
        m = (m + SCAN_CHUNK - 1) / SCAN_CHUNK;
        need += (size_t)m;
    }
    return need;
}

// exclusive scan on the device, partial sums of each level in sums
static void scan_levels(const int* in, int* out, int n, int* sums, hipStream_t s)
{
    const int nb = (n + SCAN_CHUNK - 1) / SCAN_CHUNK;
    if (nb == 1) {
        k_scan_chunk<<<1, SCAN_TB, 0, s>>>(in, out, nullptr, n);
        return;
    }
    k_scan_chunk<<<nb, SCAN_TB, 0, s>>>(in, out, sums, n);
    scan_levels(sums, sums, nb, sums + nb, s);
    k_scan_add<<<nblk(n), TB, 0, s>>>(out, sums, n);
}

// exclusive scan of n ints (out may alias in), the total left on the device
void exclusive_scan_nototal(const int* in, int* out, int n, hipStream_t s)
{
    if (n <= 0) return;
    scan_levels(in, out, n, build_slots(scan_sums_need(n)).sums, s);
    VSDMO_HIP(hipGetLastError());
}

// exclusive scan of n ints (out may alias in); returns the total
int exclusive_scan(const int* in, int* out, int n, hipStream_t s)
{
    if (n <= 0) return 0;
    BuildSlots& b = build_slots(scan_sums_need(n));
    k_copy_int<<<1, 1, 0, s>>>(in + (n - 1), b.dev);   // before an in-place scan overwrites it
    scan_levels(in, out, n, b.sums, s);
    k_scan_total<<<1, 1, 0, s>>>(out, n, b.dev, b.dev + 1);
    VSDMO_HIP(hipGetLastError());
    return read_int(b.dev + 1, s);
}

// ------------------------------------------------------ counting-sort CSR
// cnt[key]++, and the item's place among its key's (in any order): the counts'
// scan plus that place is a slot of its own, without a second round of atomics
__global__ void k_count_keys(const int* __restrict__ key, int n, int* __restrict__ cnt, int* __restrict__ place)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) place[i] = atomicAdd(&cnt[key[i]], 1);
}

__global__ void k_scatter_keys(const int* __restrict__ key, const int* __restrict__ place, int n,
                               const int* __restrict__ row, int* __restrict__ items)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) items[row[key[i]] + place[i]] = i;
}

__device__ __forceinline__ int lane_i(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }

// sort each row's item indices ascending (restores the stable order): a wave
// per row of up to 64 items, one on each lane, whose position is the number of
// smaller ones.  (A thread per row sorted by insertion in memory, one load
// after the other: 77 us for the 69k rows of 24 of a 40^3 tet cube, against
// 18.)  Longer rows are sorted by insertion.
__global__ __launch_bounds__(TB) void k_sort_rows(const int* __restrict__ row, int nrows, int* __restrict__ items)
{
    const int r = blockIdx.x * (TB / 64) + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (r >= nrows) return;
    const int s = uniform(row[r]), n = uniform(row[r + 1]) - s;
    if (n <= 64) {
        const int x = lane < n ? items[s + lane] : 0;
        int rank = 0;
        for (int j = 0; j < n; ++j) rank += lane_i(x, j) < x ? 1 : 0;
        if (lane < n) items[s + rank] = x;
    } else if (lane == 0) {
        for (int i = s + 1; i < s + n; ++i) {
            int x = items[i], j = i - 1;
            while (j >= s && items[j] > x) { items[j + 1] = items[j]; --j; }
            items[j + 1] = x;
        }
    }
}

// CSR of items 0..n-1 grouped by key in [0,nk): row[nk+1], items[n]; within a
// row ascending if sorted, else in any order
void group_csr(BuildArena& ar, const int* key, int n, int nk, DevBuf<int>& row, DevBuf<int>& items, bool sorted,
               hipStream_t s)
{
    row.alloc((size_t)nk + 1);
    items.alloc((size_t)std::max(n, 1));
    DevBuf<int> place(ar, (size_t)std::max(n, 1));
    VSDMO_HIP(hipMemsetAsync(row.p, 0, sizeof(int) * ((size_t)nk + 1), s));
    if (n > 0) k_count_keys<<<nblk(n), TB, 0, s>>>(key, n, row.p, place.p);
    exclusive_scan_nototal(row.p, row.p, nk + 1, s);
    if (n > 0) k_scatter_keys<<<nblk(n), TB, 0, s>>>(key, place.p, n, row.p, items.p);
    if (sorted && nk > 0) k_sort_rows<<<nblk((long long)nk * 64), TB, 0, s>>>(row.p, nk, items.p);
    VSDMO_HIP(hipGetLastError());
}
void stable_csr(BuildArena& ar, const int* key, int n, int nk, DevBuf<int>& row, DevBuf<int>& items, hipStream_t s)
{
    group_csr(ar, key, n, nk, row, items, true, s);
}

// ------------------------------------------------------------ boundary faces
__constant__ int c_tetFaces[4][3] = { { 2, 1, 0 }, { 0, 1, 3 }, { 1, 2, 3 }, { 0, 3, 2 } };
__constant__ int c_hexFaces[6][4] = { { 0, 1, 2, 3 }, { 1, 5, 6, 2 }, { 3, 2, 6, 7 },
                                      { 4, 0, 3, 7 }, { 1, 0, 4, 5 }, { 5, 4, 7, 6 } };

// all element faces, rotated smallest-first; fk: 4 ints per face (quad slot 3
// unused for tris), v0: first vertex
__global__ void k_emit_faces(const int* __restrict__ cells, int nE, int tet, int* __restrict__ fk, int* __restrict__ v0)
{
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nE) return;
    int nf = tet ? 4 : 6, k = tet ? 3 : 4, npe = tet ? 4 : 8;
    for (int f = 0; f < nf; ++f) {
        int a[4];
        for (int i = 0; i < k; ++i) a[i] = cells[(size_t)e * npe + (tet ? c_tetFaces[f][i] : c_hexFaces[f][i])];
        int m = 0;
        for (int i = 1; i < k; ++i) if (a[i] < a[m]) m = i;
        int id = e * nf + f;
        for (int i = 0; i < 4; ++i) fk[(size_t)id * 4 + i] = (i < k) ? a[(m + i) % k] : 0;
        v0[id] = a[m];
    }
}

// a face's order in its bucket (same first vertex): (v1, v2[, v3], emit index);
// v3 is 0 for triangles
struct FaceKey { int v1, v2, v3, idx; };
__device__ __forceinline__ FaceKey face_key(const int* fk, int item, int k)
{
    const int* a = fk + (size_t)item * 4;
    return { a[1], a[2], k == 4 ? a[3] : 0, item };
}
__device__ __forceinline__ bool face_less(FaceKey a, FaceKey b)
{
    if (a.v1 != b.v1) return a.v1 < b.v1;
    if (a.v2 != b.v2) return a.v2 < b.v2;
    if (a.v3 != b.v3) return a.v3 < b.v3;
    return a.idx < b.idx;
}
// b cancels a: (a,c,b) for (a,b,c) with b<c, (a,d,c,b) for (a,b,c,d) with b<d
__device__ __forceinline__ bool face_cancels(FaceKey a, FaceKey b, int k)
{
    return k == 3 ? a.v1 < a.v2 && b.v1 == a.v2 && b.v2 == a.v1
                  : a.v1 < a.v3 && b.v1 == a.v3 && b.v2 == a.v2 && b.v3 == a.v1;
}

// per bucket (same first vertex): sort by (v1, v2[, v3], emit index) into
// sorted, then cancel each face against the first of the opposite orientation
// after it (reference k_markDuplicateTris/Quads).  Those of the opposite
// orientation share one key beyond the emit index and sort after the face, so
// the first is the one of the smallest emit index.  A wave per bucket, a face
// on each lane: its position is the number of smaller ones, its match is found
// in the same pass.  (A thread per bucket sorted by insertion, every comparison
// a chain of loads: 323 us for the 69k buckets of 22 of a 40^3 tet cube,
// against 98.)  Buckets of more than 64 faces read the others' keys from
// memory, 64 faces at a time.
__global__ __launch_bounds__(TB) void k_bucket_faces(const int* __restrict__ row, int nb,
                                                     const int* __restrict__ items, const int* __restrict__ fk, int k,
                                                     int* __restrict__ sorted, uint8_t* __restrict__ dead)
{
    __shared__ int s_dead[TB];
    const int b = blockIdx.x * (TB / 64) + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (b >= nb) return;
    const int s = uniform(row[b]), n = uniform(row[b + 1]) - s;
    if (n <= 64) {
        int* const deadOf = s_dead + (threadIdx.x & ~63);
        deadOf[lane] = 0;
        const bool have = lane < n;
        const FaceKey x = have ? face_key(fk, items[s + lane], k) : FaceKey{ 0, 0, 0, 0 };
        int rank = 0, match = INT_MAX, at = 0;
        for (int j = 0; j < n; ++j) {
            const FaceKey y = { lane_i(x.v1, j), lane_i(x.v2, j), lane_i(x.v3, j), lane_i(x.idx, j) };
            rank += face_less(y, x) ? 1 : 0;
            if (face_cancels(x, y, k) && y.idx < match) { match = y.idx; at = j; }
        }
        wave_lds_fence();
        if (have && match != INT_MAX) { deadOf[lane] = 1; deadOf[at] = 1; }
        wave_lds_fence();
        if (have) { sorted[s + rank] = x.idx; dead[s + rank] = (uint8_t)deadOf[lane]; }
        return;
    }
    for (int i = lane; i < n; i += 64) {
        const FaceKey x = face_key(fk, items[s + i], k);
        int rank = 0;
        bool off = false;   // cancels a later face, or is the first to cancel an earlier one
        for (int j = 0; j < n; ++j) {
            const FaceKey y = face_key(fk, items[s + j], k);
            rank += face_less(y, x) ? 1 : 0;
            if (face_cancels(x, y, k)) off = true;
            if (!off && face_cancels(y, x, k)) {
                off = true;
                for (int l = 0; l < n && off; ++l) {
                    const FaceKey z = face_key(fk, items[s + l], k);
                    off = !(face_cancels(y, z, k) && z.idx < x.idx);
                }
            }
        }
        sorted[s + rank] = x.idx;
        dead[s + rank] = off ? 1 : 0;
    }
}

__global__ void k_alive(const uint8_t* __restrict__ dead, int n, int* __restrict__ flag)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) flag[i] = dead[i] ? 0 : 1;
}

__global__ void k_compact_faces(const int* __restrict__ items, const uint8_t* __restrict__ dead,
                                const int* __restrict__ pos, int n, const int* __restrict__ fk, int k,
                                int* __restrict__ out)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || dead[i]) return;
    const int* a = fk + (size_t)items[i] * 4;
    for (int j = 0; j < k; ++j) out[(size_t)pos[i] * k + j] = a[j];
}

__global__ void k_mark_vertices(const int* __restrict__ ids, int n, int* __restrict__ flag)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) flag[ids[i]] = 1;
}

// ------------------------------------------------------------ permutations
__global__ void k_partition_ids(const int* __restrict__ flag, const int* __restrict__ scan, int n, int nFirst,
                                int firstVal, int* __restrict__ newid)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    // scan counts flag==1 before v
    int ones = scan[v];
    int isOne = flag[v];
    bool first = (isOne == firstVal);
    int before = firstVal ? ones : (v - ones);
    newid[v] = first ? before : nFirst + (v - before);
}

// One renumbering in one launch: positions and the optional per-vertex arrays
// go to their spare copies, element and face ids are remapped in place, the
// composed renumbering and its inverse updated.  (Ten launches of 2-6 us, a
// gap before each.)
struct RenumberArgs {
    const int* newid;
    int nV, n8;                       // vertices; of them with u8 data (the first n8)
    long long nc, nf;
    const float* x; const float* y; const float* z;
    float* tx; float* ty; float* tz;
    int* cells; int* faces;
    int* newOfOld; int* oldOfCur;
    const uint8_t* a8[2]; uint8_t* t8[2];
    const int* a32; int* t32;
};
__global__ void k_renumber(RenumberArgs r)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < r.nc) r.cells[i] = r.newid[r.cells[i]];
    if (i < r.nf) r.faces[i] = r.newid[r.faces[i]];
    if (i >= r.nV) return;
    const int w = r.newid[i];
    r.tx[w] = r.x[i]; r.ty[w] = r.y[i]; r.tz[w] = r.z[i];
    if (r.a32) r.t32[w] = r.a32[i];
    if (i < r.n8) { r.t8[0][w] = r.a8[0][i]; r.t8[1][w] = r.a8[1][i]; }
    const int o = r.newid[r.newOfOld[i]];
    r.newOfOld[i] = o;
    r.oldOfCur[o] = (int)i;
}

// Applies newid (a permutation of all nV current ids) to positions, elements,
// faces, the composed renumbering and optional per-vertex arrays.
struct Renumber {
    vsdmo_mesh& m;
    BuildArena& ar;
    DevBuf<int> oldOfCur;   // current id -> input id
    // the arrays that the mesh's change places with
    DevBuf<float> tx, ty, tz;
    DevBuf<uint8_t> t8[2];
    DevBuf<int> t32;
    Renumber(vsdmo_mesh& mesh, BuildArena& arena) : m(mesh), ar(arena), oldOfCur(arena, mesh.nV)
    {
        tx.alloc(m.nV); ty.alloc(m.nV); tz.alloc(m.nV); t32.alloc(m.nV);
    }

    void apply(const int* newid, bool flags = false, bool colours = false)
    {
        RenumberArgs r{};
        r.newid = newid;
        r.nV = m.nV;
        r.nc = (long long)m.nE * m.npe;
        r.nf = (m.faces.p != m.cells.p) ? (long long)m.nFaces * m.fpe : 0;
        r.x = m.x.p; r.y = m.y.p; r.z = m.z.p;
        r.tx = tx.p; r.ty = ty.p; r.tz = tz.p;
        r.cells = m.cells.p; r.faces = m.faces.p;
        r.newOfOld = m.newOfOld.p; r.oldOfCur = oldOfCur.p;
        if (flags) {
            DevBuf<uint8_t>* a[2] = { &m.isB1D, &m.isFeature };
            r.n8 = (int)m.isB1D.n;
            for (int i = 0; i < 2; ++i) {
                if (t8[i].n != a[i]->n) t8[i].alloc(a[i]->n);
                r.a8[i] = a[i]->p; r.t8[i] = t8[i].p;
            }
        }
        if (colours) { r.a32 = m.colorOf.p; r.t32 = t32.p; }
        const long long n = std::max({ (long long)m.nV, r.nc, r.nf });
        k_renumber<<<nblk(n), TB, 0, m.stream>>>(r);
        VSDMO_HIP(hipGetLastError());
        std::swap(m.x, tx);
        std::swap(m.y, ty);
        std::swap(m.z, tz);
        if (flags) { std::swap(m.isB1D, t8[0]); std::swap(m.isFeature, t8[1]); }
        if (colours) std::swap(m.colorOf, t32);
    }
};

// ------------------------------------------------------------- colouring
// Neighbour walk of current vertex v: incident elements from the incidence
// CSR (input ids), other corners through the current element array.
struct Incidence {
    const int* row;   // nV+1 over input ids
    const int* val;   // element*8 + corner
    const int* oldOfCur;
    const int* cells;
    int npe;
};

// Greedy first-fit in index order by Jones-Plassmann rounds with priority n-i:
// a vertex is coloured once all its lower in-range neighbours are, with the
// smallest colour none of them uses.  The colour of a vertex depends only on
// the final colours of its lower neighbours, so the result equals the
// sequential greedy colouring whatever the round in which a vertex is reached.
__global__ void k_color_greedy_round(Incidence inc, int lo, int hi, int* __restrict__ col, int* __restrict__ left)
{
    const int v = lo + blockIdx.x * blockDim.x + threadIdx.x;
    volatile int* vc = col;
    bool wait = false;
    if (v < hi && vc[v - lo] < 0) {
        const int o = inc.oldOfCur[v];
        uint64_t mask = 0;
        bool big = false;
        for (int k = inc.row[o]; k < inc.row[o + 1] && !wait; ++k) {
            const int e = inc.val[k] >> 3, c = inc.val[k] & 7;
            for (int i = 0; i < inc.npe; ++i) {
                if (i == c) continue;
                const int u = inc.cells[(size_t)e * inc.npe + i];
                if (u < lo || u >= v) continue;
                const int cu = vc[u - lo];
                if (cu < 0) { wait = true; break; }
                if (cu < 64) mask |= (1ull << cu); else big = true;
            }
        }
        if (!wait) {
            int cc = __builtin_ctzll(~mask);
            if (big && cc == 64) {
                // more than 64 colours in use around v: linear mex search
                for (cc = 64;; ++cc) {
                    bool used = false;
                    for (int k = inc.row[o]; k < inc.row[o + 1] && !used; ++k) {
                        const int e = inc.val[k] >> 3, c = inc.val[k] & 7;
                        for (int i = 0; i < inc.npe; ++i) {
                            if (i == c) continue;
                            const int u = inc.cells[(size_t)e * inc.npe + i];
                            if (u >= lo && u < v && vc[u - lo] == cc) { used = true; break; }
                        }
                    }
                    if (!used) break;
                }
            }
            vc[v - lo] = cc;
        }
    }
    // one plain store per wave with a waiting vertex (no atomic per vertex)
    if (__ballot(wait) != 0 && (threadIdx.x & 63) == 0) *left = 1;
}

// Lower neighbours of each vertex v of [lo, hi): the in-range ids u < v of
// the corners of v's elements, as offsets from lo (an id appears once per
// element shared with v), for the single-pass colouring below
__global__ void k_lower_count(Incidence inc, int lo, int hi, int* __restrict__ cnt)
{
    const int v = lo + blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= hi) return;
    const int o = inc.oldOfCur[v];
    int c = 0;
    for (int k = inc.row[o]; k < inc.row[o + 1]; ++k) {
        const int e = inc.val[k] >> 3, cr = inc.val[k] & 7;
        for (int i = 0; i < inc.npe; ++i) {
            if (i == cr) continue;
            const int u = inc.cells[(size_t)e * inc.npe + i];
            c += (u >= lo && u < v) ? 1 : 0;
        }
    }
    cnt[v - lo] = c;
}

__global__ void k_lower_fill(Incidence inc, int lo, int hi, const int* __restrict__ row, int* __restrict__ val)
{
    const int v = lo + blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= hi) return;
    const int o = inc.oldOfCur[v];
    int w = row[v - lo];
    for (int k = inc.row[o]; k < inc.row[o + 1]; ++k) {
        const int e = inc.val[k] >> 3, cr = inc.val[k] & 7;
        for (int i = 0; i < inc.npe; ++i) {
            if (i == cr) continue;
            const int u = inc.cells[(size_t)e * inc.npe + i];
            if (u >= lo && u < v) val[w++] = u - lo;
        }
    }
}

// The greedy first-fit colouring of k_color_greedy_round in one launch: each
// vertex waits for the colours of its lower neighbours, then takes the
// smallest colour none of them uses.  A colour depends only on the final
// colours of the lower neighbours, so the result is the sequential greedy
// colouring.  A vertex waits only for lower vertices: those of its own wave
// (the wave loops until all its lanes are done, so the lowest waiting lane
// always finds its neighbours set), those of lower waves of its workgroup, and
// those of lower workgroups, which are dispatched before it.  The wait is
// bounded all the same: a vertex that has polled spinLimit times stops
// uncoloured and raises *gaveUp, and the round kernel completes the colouring
// with the same colours.
// The chains of waiting vertices bound it (a mesh numbered along its rows
// chains every vertex to the one before).  So a colour passes from lane to
// lane within a wave, through LDS within the workgroup (256 vertices), and
// only from workgroup to workgroup through memory, at device scope, ~2 us a
// step, where every step used to take that way: 59k inner vertices of a 40^3
// tet cube 884 us, 230 us now.
__global__ __launch_bounds__(256) void k_color_greedy_sweep(const int* __restrict__ row, const int* __restrict__ val,
                                                           int n, int* __restrict__ col, int spinLimit,
                                                           int* __restrict__ gaveUp)
{
    __shared__ int s_col[256];   // colours of the workgroup's vertices, -1 until set
    const int t = threadIdx.x, lane = t & 63, wave = uniform(t >> 6);
    const int b0 = blockIdx.x * 256, v = b0 + t;
    s_col[t] = -1;
    __syncthreads();
    const auto lds_colour = [&](int i) { return __hip_atomic_load(s_col + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
    const auto mem_colour = [&](int u) { return __hip_atomic_load(col + u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    bool todo = v < n;
    const int r0 = todo ? row[v] : 0, r1 = todo ? row[v + 1] : 0;
    constexpr int B = 8;    // list entries read together (their latencies overlap)
    constexpr int S = 12;   // lower neighbours in lower workgroups polled together
    int k = r0, id[S] = {}; // entries [r0, k) are read; id[]: those polled
    int pend = 0;           // the ids not yet coloured
    uint64_t mask = 0;      // colours of the lower neighbours seen so far
    bool big = false;       // one of them is 64 or more
    uint64_t own = 0, low[3] = { 0, 0, 0 };   // waiting for: lanes of this wave, of the workgroup's lower waves
    uint64_t passed = 0;                      // lanes of this wave whose colour has been passed on
    int polls = 0;
    const auto seen = [&](int c) { if (c < 64) mask |= 1ull << c; else big = true; };
    while (__ballot(todo) != 0) {
        // lower workgroups: up to S distinct ids, read ahead of the wait (the
        // list, which names a neighbour once per shared element, takes several
        // loads one after the other) and polled together
        while (todo && (pend != 0 || k < r1)) {
            if (pend == 0) {
                int cnt = 0;
                while (k < r1 && cnt < S) {
                    int e[B], used = 0;
                    // entries past the list re-read its last one (k < r1), so every
                    // load is unconditional and in bounds; their values are ignored
#pragma unroll
                    for (int j = 0; j < B; ++j) e[j] = val[min(k + j, r1 - 1)];
#pragma unroll
                    for (int j = 0; j < B; ++j) {
                        if (k + j >= r1 || cnt == S) continue;
                        ++used;
                        const int i = e[j] - b0;
                        if (i < 0) {
                            bool known = false;
#pragma unroll
                            for (int q = 0; q < S; ++q) known = known || (q < cnt && id[q] == e[j]);
                            if (known) continue;
#pragma unroll
                            for (int q = 0; q < S; ++q) id[q] = q == cnt ? e[j] : id[q];
                            ++cnt;
                            continue;
                        }
                        const uint64_t bit = 1ull << (i & 63);
                        if ((i >> 6) == wave) own |= bit;
                        else if ((i >> 6) == 0) low[0] |= bit;
                        else if ((i >> 6) == 1) low[1] |= bit;
                        else low[2] |= bit;
                    }
                    k += used;
                }
                pend = (1 << cnt) - 1;
#pragma unroll
                for (int q = 0; q < S; ++q) id[q] = q < cnt ? id[q] : v;   // loads stay in bounds
            }
            if (pend != 0) {
                int cu[S];
#pragma unroll
                for (int q = 0; q < S; ++q) cu[q] = mem_colour(id[q]);
#pragma unroll
                for (int q = 0; q < S; ++q)
                    if ((pend >> q & 1) && cu[q] >= 0) { seen(cu[q]); pend &= ~(1 << q); }
                if (pend != 0) break;
            }
        }
        // the workgroup's lower waves
#pragma unroll
        for (int w = 0; w < 3; ++w) {
            uint64_t rest = todo ? low[w] : 0;
            while (rest) {
                const int i = __builtin_ctzll(rest);
                rest &= rest - 1;
                const int c = lds_colour(w * 64 + i);
                if (c < 0) break;
                seen(c);
                low[w] &= ~(1ull << i);
            }
        }
        // lanes of this wave that passed their colour on before this lane read
        // its list that far
        for (uint64_t rest = todo ? own & passed : 0; rest; rest &= rest - 1) seen(lds_colour(wave * 64 + __builtin_ctzll(rest)));
        own &= ~passed;
        // this wave: lanes that are ready take their colour and pass it on, until none is
        for (;;) {
            const bool ready = todo && pend == 0 && k == r1 && (low[0] | low[1] | low[2] | own) == 0;
            uint64_t done = __ballot(ready);
            if (done == 0) break;
            passed |= done;
            int cc = 0;
            if (ready) {
                cc = (~mask == 0ull) ? 64 : __builtin_ctzll(~mask);
                if (big && cc == 64) {
                    // more than 64 colours around v: linear mex search
                    for (;; ++cc) {
                        bool used = false;
                        for (int j = r0; j < r1 && !used; ++j)
                            used = (val[j] >= b0 ? lds_colour(val[j] - b0) : mem_colour(val[j])) == cc;
                        if (!used) break;
                    }
                }
                __hip_atomic_store(s_col + t, cc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_store(col + v, cc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                todo = false;
            }
            while (done) {
                const int l = __builtin_ctzll(done);
                done &= done - 1;
                const int c = lane_i(cc, l);
                if (own >> l & 1) { seen(c); own &= ~(1ull << l); }
            }
        }
        // a poll of memory counts as 16 of LDS, which are that much shorter
        polls += pend != 0 ? 16 : 1;
        if (todo && (polls >> 4) >= spinLimit) {
            __hip_atomic_store(gaveUp, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            todo = false;
        }
        __builtin_amdgcn_s_sleep(1);
    }
}

// Reference color_jpl round c (VertexColoring.cu:76-105): v takes colour c iff
// every in-range neighbour that is uncoloured or coloured c in this round has
// a lower priority n-u, i.e. a larger index.
__global__ void k_color_jpl_round(Incidence inc, int lo, int hi, int c, int* __restrict__ col, int* __restrict__ left)
{
    const int v = lo + blockIdx.x * blockDim.x + threadIdx.x;
    volatile int* vc = col;
    bool wait = false;
    if (v < hi && vc[v - lo] == -1) {
        const int o = inc.oldOfCur[v];
        bool ok = true;
        for (int k = inc.row[o]; k < inc.row[o + 1] && ok; ++k) {
            const int e = inc.val[k] >> 3, cr = inc.val[k] & 7;
            for (int i = 0; i < inc.npe; ++i) {
                if (i == cr) continue;
                const int u = inc.cells[(size_t)e * inc.npe + i];
                if (u < lo || u >= hi || u == v) continue;
                const int cu = vc[u - lo];
                if ((cu != -1) && (cu != c)) continue;
                if (!(v < u)) { ok = false; break; }
            }
        }
        if (ok) vc[v - lo] = c; else wait = true;
    }
    if (__ballot(wait) != 0 && (threadIdx.x & 63) == 0) *left = 1;
}

__global__ void k_max_reduce(const int* __restrict__ a, int n, int* __restrict__ out)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) atomicMax(out, a[i]);
}

// colours of one sort at most (the per-block counts live in LDS)
constexpr int kMaxSortColours = 16384;

// per block of TB vertices of [0, n): the count of each colour, stored
// colour-major (hist[c * nb + b]) so that one exclusive scan gives every
// (colour, block) its first position in the colour-sorted order
__global__ void k_colour_hist(const int* __restrict__ col, int n, int nc, int nb, int* __restrict__ hist)
{
    extern __shared__ int sh[];
    for (int c = threadIdx.x; c < nc; c += blockDim.x) sh[c] = 0;
    __syncthreads();
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) atomicAdd(&sh[col[i]], 1);
    __syncthreads();
    for (int c = threadIdx.x; c < nc; c += blockDim.x) hist[(size_t)c * nb + blockIdx.x] = sh[c];
}

// new id of vertex lo + i: lo + the scanned first position of (its colour,
// its block) + the vertices of its colour before it in the block
__global__ __launch_bounds__(TB) void k_colour_place(const int* __restrict__ col, int n, int nb,
                                                     const int* __restrict__ pos, int lo, int* __restrict__ newid)
{
    __shared__ int sc[TB];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int c = (i < n) ? col[i] : -1;
    sc[threadIdx.x] = c;
    __syncthreads();
    if (i >= n) return;
    int r = 0;
    for (int j = 0; j < (int)threadIdx.x; ++j) r += (sc[j] == c) ? 1 : 0;
    newid[lo + i] = lo + pos[(size_t)c * nb + blockIdx.x] + r;
}

// first vertex of each colour, off[c] = lo + pos[c * nb], and the end of the last
__global__ void k_colour_offsets(const int* __restrict__ pos, int nb, int nc, int lo, int n, int* __restrict__ off)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c <= nc) off[c] = lo + (c < nc ? pos[(size_t)c * nb] : n);
}

__global__ void k_fill_int(int* p, int v) { *p = v; }

__global__ void k_iota(int* __restrict__ a, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = i;
}

__global__ void k_fill_range(int* __restrict__ a, int lo, int n, const int* __restrict__ col)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[lo + i] = col[i];
}

// Class partition check (the rule of k_checkColoring, MeshGPUCommon.cu:
// 1470-1680): the vertices [off[0], off[nc]) are split into the classes
// [off[c], off[c+1]); no element may hold two vertices of one class, or
// their searches in one launch would read each other's positions.  One
// thread per element; a corner's class by binary search of the offsets.
__global__ void k_check_classes(const int* __restrict__ cells, int nE, int npe, const int* __restrict__ off, int nc,
                                int* __restrict__ bad)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nE) return;
    const int lo = off[0], hi = off[nc];
    int cls[8];
    for (int i = 0; i < npe; ++i) {
        const int v = cells[(size_t)e * npe + i];
        int c = -1;
        if (v >= lo && v < hi) {
            int a = 0, b = nc - 1;          // largest c with off[c] <= v
            while (a < b) {
                const int mid = (a + b + 1) >> 1;
                if (off[mid] <= v) a = mid; else b = mid - 1;
            }
            c = a;
        }
        cls[i] = c;
        for (int j = 0; j < i; ++j)
            if (c >= 0 && cls[j] == c) atomicMin(bad, c);
    }
}

// the partitions' verdicts, read together with the last of the build's values
struct ClassChecks {
    DevBuf<int> bad;   // per partition: the lowest class with two vertices of one element, INT_MAX if none
    std::vector<std::vector<int>> off;
    explicit ClassChecks(BuildArena& ar) : bad(ar, kMax) {}
    static constexpr int kMax = 3;
    void add(const vsdmo_mesh& m, const int* doff, const std::vector<int>& o)
    {
        const int i = (int)off.size(), nc = (int)o.size() - 1;
        off.push_back(o);
        k_fill_int<<<1, 1, 0, m.stream>>>(bad.p + i, INT_MAX);
        if (nc > 0 && m.nE > 0) k_check_classes<<<nblk(m.nE), TB, 0, m.stream>>>(m.cells.p, m.nE, m.npe, doff, nc, bad.p + i);
        VSDMO_HIP(hipGetLastError());
    }
    void verify(hipStream_t s) const
    {
        if (off.empty()) return;
        const int* h = read_ints(bad.p, (int)off.size(), s);
        for (size_t i = 0; i < off.size(); ++i)
            if (h[i] != INT_MAX)
                throw StatusError{ VSDMO_TOPOLOGY, "colour class " + std::to_string(h[i]) + " (vertices " +
                                                       std::to_string(off[i][h[i]]) + ".." +
                                                       std::to_string(off[i][h[i] + 1] - 1) +
                                                       ") holds two vertices of one element" };
    }
};

// a partition given by the caller
void check_classes(const vsdmo_mesh& m, const std::vector<int>& off)
{
    BuildArena ar(0, m.stream);
    DevBuf<int> doff(ar, off.size());
    ClassChecks checks(ar);
    doff.upload(off.data(), off.size(), m.stream);
    checks.add(m, doff.p, off);
    checks.verify(m.stream);
}

// colour [lo,hi) of the current numbering and sort it stably by colour.
// Returns absolute colour offsets, checked to be independent sets.
// default polls of a vertex in the single-pass greedy colouring before it
// leaves its colour to the rounds (a wait of ~0.1 s at most; the chains of
// the meshes here need a few hundred)
constexpr int kSweepPolls = 1 << 16;

std::vector<int> colour_and_sort(vsdmo_mesh& m, Renumber& rn, ClassChecks& checks, const int* incRow,
                                 const int* incVal, int lo, int hi, const vsdmo_mesh_params& prm, bool flags)
{
    BuildArena& ar = rn.ar;
    hipStream_t s = m.stream;
    int n = hi - lo;
    if (n <= 0) return { lo };
    const int mode = prm.coloring;
    const int polls = prm.coloring_polls > 0 ? prm.coloring_polls : kSweepPolls;
    Incidence inc{ incRow, incVal, rn.oldOfCur.p, m.cells.p, m.npe };
    // rounds go out in batches of kRoundsPerCheck, each round raising its own
    // flag when a vertex still waits, and the host reads the flag of the
    // batch's last round: a round after the colouring is complete finds every
    // vertex coloured and changes nothing, so the colours are those of one
    // check per round, with 1/kRoundsPerCheck of the syncs
    constexpr int kRoundsPerCheck = 16;
    DevBuf<int> col(ar, n), left(ar, kRoundsPerCheck), flag(ar, 2);   // flag: polls ran out, largest colour
    VSDMO_HIP(hipMemsetAsync(col.p, 0xff, sizeof(int) * n, s));
    VSDMO_HIP(hipMemsetAsync(flag.p, 0, 2 * sizeof(int), s));
    int h_left = 1, nc = 0;
    const auto colours = [&]() {
        k_max_reduce<<<nblk(n), TB, 0, s>>>(col.p, n, flag.p + 1);
        VSDMO_HIP(hipGetLastError());
        const int* h = read_ints(flag.p, 2, s);
        h_left = h[0];
        nc = h[1] + 1;
    };
    if (mode != VSDMO_COLOR_JPL) {
        // greedy: one sweep over lower-neighbour lists; the rounds below only
        // run if a vertex ran out of polls
        DevBuf<int> lrow(ar, (size_t)n + 1);
        k_lower_count<<<nblk(n), TB, 0, s>>>(inc, lo, hi, lrow.p);
        VSDMO_HIP(hipMemsetAsync(lrow.p + n, 0, sizeof(int), s));
        const int tot = exclusive_scan(lrow.p, lrow.p, n + 1, s);
        DevBuf<int> lval(ar, (size_t)std::max(tot, 1));
        k_lower_fill<<<nblk(n), TB, 0, s>>>(inc, lo, hi, lrow.p, lval.p);
        k_color_greedy_sweep<<<nblk(n), TB, 0, s>>>(lrow.p, lval.p, n, col.p, std::min(polls, 1 << 26), flag.p);
        VSDMO_HIP(hipGetLastError());
        colours();
    }
    const bool rounds = h_left != 0;
    for (int round = 0; h_left != 0;) {
        if (round > n + 1) throw StatusError{ VSDMO_TOPOLOGY, "colouring did not converge" };
        VSDMO_HIP(hipMemsetAsync(left.p, 0, sizeof(int) * kRoundsPerCheck, s));
        for (int k = 0; k < kRoundsPerCheck; ++k, ++round) {
            if (mode == VSDMO_COLOR_JPL)
                k_color_jpl_round<<<nblk(n), TB, 0, s>>>(inc, lo, hi, round, col.p, left.p + k);
            else
                k_color_greedy_round<<<nblk(n), TB, 0, s>>>(inc, lo, hi, col.p, left.p + k);
        }
        VSDMO_HIP(hipGetLastError());
        h_left = read_int(left.p + kRoundsPerCheck - 1, s);
    }
    if (rounds) colours();
    if (nc > kMaxSortColours) throw StatusError{ VSDMO_NOT_SUPPORTED, "more than 16384 colours" };
    // stable counting sort by colour: per block of TB vertices the count of
    // each colour, scanned colour-major, gives each (colour, block) its first
    // position; a vertex adds the same-coloured vertices before it in its block
    const int nb = nblk(n);
    DevBuf<int> newid(ar, m.nV), pos(ar, (size_t)nc * nb), doff(ar, (size_t)nc + 1);
    k_iota<<<nblk(m.nV), TB, 0, s>>>(newid.p, m.nV);
    k_colour_hist<<<nb, TB, sizeof(int) * nc, s>>>(col.p, n, nc, nb, pos.p);
    exclusive_scan_nototal(pos.p, pos.p, nc * nb, s);
    k_colour_place<<<nb, TB, 0, s>>>(col.p, n, nb, pos.p, lo, newid.p);
    k_colour_offsets<<<nblk(nc + 1), TB, 0, s>>>(pos.p, nb, nc, lo, n, doff.p);
    std::vector<int> off(nc + 1, 0);
    doff.download(off.data(), nc + 1, s);
    k_fill_range<<<nblk(n), TB, 0, s>>>(m.colorOf.p, lo, n, col.p);
    rn.apply(newid.p, flags, true);
    VSDMO_HIP(hipStreamSynchronize(s));
    checks.add(m, doff.p, off);
    return off;
}

// ------------------------------------------------------------ one-ring CSR
__constant__ int c_halfface[4][3] = { { 1, 2, 3 }, { 0, 3, 2 }, { 0, 1, 3 }, { 0, 2, 1 } };
__constant__ int c_halfhex[8][7] = { { 1, 2, 3, 4, 5, 6, 7 }, { 5, 6, 2, 0, 4, 7, 3 }, { 6, 7, 3, 1, 5, 4, 0 },
                                     { 7, 4, 0, 2, 6, 5, 1 }, { 0, 3, 7, 5, 1, 2, 6 }, { 4, 7, 6, 1, 0, 3, 2 },
                                     { 5, 4, 7, 2, 1, 0, 3 }, { 6, 5, 4, 3, 2, 1, 0 } };

// ring sizes, in cnt[n] and (with a zero at its end, for the scan) in row[n + 1]
__global__ void k_ring_counts(const int* __restrict__ incRow, const int* __restrict__ oldOfCur, int n,
                              int* __restrict__ cnt, int* __restrict__ row)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v < n) { int o = oldOfCur[v]; cnt[v] = row[v] = incRow[o + 1] - incRow[o]; }
    if (v == n) row[v] = 0;
}

__global__ void k_ring_fill(const int* __restrict__ incRow, const int* __restrict__ incVal, const int* __restrict__ oldOfCur,
                            const int* __restrict__ ringRow, const int* __restrict__ cells, int n, int tet,
                            int* __restrict__ ringVal)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    int o = oldOfCur[v];
    int st = tet ? 3 : 7, npe = tet ? 4 : 8;
    int w = ringRow[v];
    for (int k = incRow[o]; k < incRow[o + 1]; ++k, ++w) {
        int e = incVal[k] >> 3, c = incVal[k] & 7;
        for (int j = 0; j < st; ++j)
            ringVal[(size_t)w * st + j] = cells[(size_t)e * npe + (tet ? c_halfface[c][j] : c_halfhex[c][j])];
    }
}

__global__ void k_incidence_keys(const int* __restrict__ cells, long long n, int* __restrict__ key)
{
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) key[i] = cells[i];
}

__global__ void k_incidence_vals(const int* __restrict__ items, long long n, int npe, int* __restrict__ val)
{
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) { int it = items[i]; val[i] = (it / npe) * 8 + (it % npe); }
}

struct SurfaceInputs {
    const int* incRow;   // incidence over input ids (colouring adjacency)
    const int* incVal;
};
void build_surface(vsdmo_mesh& m, Renumber& rn, ClassChecks& checks, const SurfaceInputs& si,
                   const vsdmo_mesh_params& prm);

// ------------------------------------------------------------------ build
__global__ void k_mesh_init(const float* __restrict__ xyz, int nV, float* __restrict__ x, float* __restrict__ y,
                            float* __restrict__ z, int* __restrict__ colorOf, int* __restrict__ newOfOld,
                            int* __restrict__ notFlat)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nV) return;
    x[v] = xyz[3 * (size_t)v];
    y[v] = xyz[3 * (size_t)v + 1];
    const float pz = xyz[3 * (size_t)v + 2];
    z[v] = pz;
    if (pz != 0.0f) *notFlat = 1;
    colorOf[v] = 0;
    newOfOld[v] = v;
}

bool init_mesh(vsdmo_mesh& m, const float* xyz)
{
    hipStream_t s = m.stream;
    DevBuf<float> in((size_t)m.nV * 3);
    DevBuf<int> notFlat(1);
    in.upload(xyz, (size_t)m.nV * 3, s);
    VSDMO_HIP(hipMemsetAsync(notFlat.p, 0, sizeof(int), s));
    k_mesh_init<<<nblk(m.nV), TB, 0, s>>>(in.p, m.nV, m.x.p, m.y.p, m.z.p, m.colorOf.p, m.newOfOld.p, notFlat.p);
    VSDMO_HIP(hipGetLastError());
    return read_int(notFlat.p, s) == 0;
}

void build_volume(vsdmo_mesh& m, const vsdmo_mesh_params& prm)
{
    hipStream_t s = m.stream;
    const bool tet = (m.elem == VSDMO_TET);
    const int npe = m.npe, nV = m.nV, nE = m.nE;
    const long long nci = (long long)nE * npe;

    const int nf = tet ? 4 : 6, k = tet ? 3 : 4, n = nE * nf;
    // the largest at one time: the incidence, and the faces' arrays (8 ints a face)
    BuildArena ar(sizeof(int) * ((size_t)nci + 9 * (size_t)n + 8 * (size_t)nV), s);

    // incidence in input ids: vertex -> (element, corner), ordered by element
    DevBuf<int> incRow(ar), incVal(ar, nci);
    {
        DevBuf<int> key(ar, nci), items(ar);
        k_incidence_keys<<<nblk(nci), TB, 0, s>>>(m.cells.p, nci, key.p);
        stable_csr(ar, key.p, (int)nci, nV, incRow, items, s);
        k_incidence_vals<<<nblk(nci), TB, 0, s>>>(items.p, nci, npe, incVal.p);
    }

    // boundary faces
    {
        DevBuf<int> fk(ar, (size_t)n * 4), v0(ar, n), row(ar), any(ar);
        DevBuf<uint8_t> dead(ar, n);
        k_emit_faces<<<nblk(nE), TB, 0, s>>>(m.cells.p, nE, tet, fk.p, v0.p);
        group_csr(ar, v0.p, n, nV, row, any, false, s);
        DevBuf<int> items(ar, n);
        k_bucket_faces<<<nblk((long long)nV * 64), TB, 0, s>>>(row.p, nV, any.p, fk.p, k, items.p, dead.p);
        // the keys and the unsorted order are no longer needed
        int* const alive = v0.p;
        int* const pos = any.p;
        k_alive<<<nblk(n), TB, 0, s>>>(dead.p, n, alive);
        int nb = exclusive_scan(alive, pos, n, s);
        m.fpe = k;
        m.nFaces = nb;
        m.faces.alloc((size_t)std::max(nb, 1) * k);
        k_compact_faces<<<nblk(n), TB, 0, s>>>(items.p, dead.p, pos, n, fk.p, k, m.faces.p);
        VSDMO_HIP(hipGetLastError());
    }

    Renumber rn(m, ar);
    ClassChecks checks(ar);
    // [surface | inner], stable
    {
        DevBuf<int> flag(ar, nV), scan(ar, nV), newid(ar, nV);
        VSDMO_HIP(hipMemsetAsync(flag.p, 0, sizeof(int) * nV, s));
        long long nfi = (long long)m.nFaces * m.fpe;
        if (nfi > 0) k_mark_vertices<<<nblk(nfi), TB, 0, s>>>(m.faces.p, (int)nfi, flag.p);
        int nS = exclusive_scan(flag.p, scan.p, nV, s);
        k_partition_ids<<<nblk(nV), TB, 0, s>>>(flag.p, scan.p, nV, nS, 1, newid.p);
        rn.apply(newid.p);
        m.nSurf = nS;
        m.nInner = nV - nS;
    }
    // inner colouring and colour sort
    m.colOffInner = colour_and_sort(m, rn, checks, incRow.p, incVal.p, m.nSurf, nV, prm, false);

    // surface: features, [free | feature], colouring, halfedges
    SurfaceInputs si{ incRow.p, incVal.p };
    build_surface(m, rn, checks, si, prm);

    // one-ring CSR in the final numbering
    {
        DevBuf<int> cnt(ar, nV);
        m.ringRow.alloc((size_t)nV + 1);
        k_ring_counts<<<nblk((long long)nV + 1), TB, 0, s>>>(incRow.p, rn.oldOfCur.p, nV, cnt.p, m.ringRow.p);
        exclusive_scan_nototal(m.ringRow.p, m.ringRow.p, nV + 1, s);
        int st = tet ? 3 : 7;
        m.ringVal.alloc((size_t)nci * st);   // an entry per element and corner
        k_ring_fill<<<nblk(nV), TB, 0, s>>>(incRow.p, incVal.p, rn.oldOfCur.p, m.ringRow.p, m.cells.p, nV, tet, m.ringVal.p);
        DevBuf<int> mx(ar, 1);
        VSDMO_HIP(hipMemsetAsync(mx.p, 0, sizeof(int), s));
        k_max_reduce<<<nblk(nV), TB, 0, s>>>(cnt.p, nV, mx.p);
        VSDMO_HIP(hipGetLastError());
        m.maxRing = read_int(mx.p, s);
        checks.verify(s);
    }
}

// surface meshes (tri): all vertices are surface vertices
void build_surface_mesh(vsdmo_mesh& m, const vsdmo_mesh_params& prm)
{
    hipStream_t s = m.stream;
    const int npe = m.npe, nV = m.nV, nE = m.nE;
    const long long nci = (long long)nE * npe;
    // the largest at one time: the incidence and the halfedges' arrays
    BuildArena ar(sizeof(int) * (18 * (size_t)nci + 8 * (size_t)nV), s);
    DevBuf<int> incRow(ar), incVal(ar, nci);
    {
        DevBuf<int> key(ar, nci), items(ar);
        k_incidence_keys<<<nblk(nci), TB, 0, s>>>(m.cells.p, nci, key.p);
        stable_csr(ar, key.p, (int)nci, nV, incRow, items, s);
        k_incidence_vals<<<nblk(nci), TB, 0, s>>>(items.p, nci, npe, incVal.p);
    }
    m.nSurf = nV;
    m.nInner = 0;
    m.colOffInner = { nV };
    m.fpe = npe;
    m.nFaces = nE;
    m.faces.alloc((size_t)nE * npe);
    VSDMO_HIP(hipMemcpyAsync(m.faces.p, m.cells.p, sizeof(int) * nci, hipMemcpyDeviceToDevice, s));
    Renumber rn(m, ar);
    ClassChecks checks(ar);
    {
        DevBuf<int> id(ar, nV);
        k_iota<<<nblk(nV), TB, 0, s>>>(id.p, nV);
        rn.apply(id.p);
    }
    SurfaceInputs si{ incRow.p, incVal.p };
    build_surface(m, rn, checks, si, prm);
    m.ringRow.alloc((size_t)nV + 1);
    VSDMO_HIP(hipMemsetAsync(m.ringRow.p, 0, sizeof(int) * ((size_t)nV + 1), s));
    checks.verify(s);
}

}  // namespace vsdmo

// =====================================================================
// Surface structures (reference VSDMO/src/mesh/MeshTriGPU.cu:37-52,128-214,
// 463-510,646-784; MeshQuadGPU.cu:37-45,156-243,342-390,481-536;
// MeshGPUCommon.cu:96-135,139-161,211-361,363-411,466-495,565-621,1227-1239)
// =====================================================================
namespace vsdmo {

// canonical face normal: quads use v0, v1, v3 (k_calcFaceNormals)
__global__ void k_face_normals(const float* __restrict__ x, const float* __restrict__ y, const float* __restrict__ z,
                               const int* __restrict__ faces, int nF, int k, float* __restrict__ fn)
{
    int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nF) return;
    int a = faces[(size_t)f * k], b = faces[(size_t)f * k + 1], c = faces[(size_t)f * k + (k == 3 ? 2 : 3)];
    float e0x = x[b] - x[a], e0y = y[b] - y[a], e0z = z[b] - z[a];
    float e1x = x[c] - x[a], e1y = y[c] - y[a], e1z = z[c] - z[a];
    float cx = e0y * e1z - e0z * e1y, cy = e0z * e1x - e0x * e1z, cz = e0x * e1y - e0y * e1x;
    float l = sqrtf(fmaf(cx, cx, fmaf(cy, cy, cz * cz)));
    fn[3 * f] = cx / l;
    fn[3 * f + 1] = cy / l;
    fn[3 * f + 2] = cz / l;
}

__device__ __forceinline__ int he_src(const int* faces, int k, int h) { return faces[h]; }
__device__ __forceinline__ int he_dst(const int* faces, int k, int h)
{
    int f = h / k, i = h - f * k;
    return faces[(size_t)f * k + (i + 1 == k ? 0 : i + 1)];
}

__global__ void k_he_src(const int* __restrict__ faces, int n, int* __restrict__ key)
{
    int h = blockIdx.x * blockDim.x + threadIdx.x;
    if (h < n) key[h] = faces[h];
}

// opposite of every sorted raw halfedge: last match in the target's row
// (k_setOppositeHalfedgeHelper)
__global__ void k_he_opp_raw(const int* __restrict__ row, const int* __restrict__ items, int nS,
                             const int* __restrict__ faces, int k, int* __restrict__ opp)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nS) return;
    for (int p = row[v]; p < row[v + 1]; ++p) {
        int d = he_dst(faces, k, items[p]);
        int o = -1;
        for (int q = row[d]; q < row[d + 1]; ++q)
            if (he_dst(faces, k, items[q]) == v) o = q;
        opp[p] = o;
    }
}

// boundary-1D flags and features (k_initBoundary1DRowPtr, k_initFeaturesRowPtr
// with the angle test written as cos < cos(threshold))
__global__ void k_features(const int* __restrict__ row, const int* __restrict__ items, const int* __restrict__ opp,
                           int nS, const int* __restrict__ faces, int k, const float* __restrict__ fn, int flat,
                           float cthr, uint8_t* __restrict__ b1d, uint8_t* __restrict__ feat)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nS) return;
    bool isb = false;
    for (int p = row[v]; p < row[v + 1]; ++p) if (opp[p] == -1) { isb = true; break; }
    if (isb) b1d[v] = 1;
    if (flat) {
        if (isb) feat[v] = 1;
        return;
    }
    for (int p = row[v]; p < row[v + 1]; ++p) {
        int h = items[p];
        int d = he_dst(faces, k, h);
        if (opp[p] == -1) { feat[v] = 1; feat[d] = 1; continue; }
        const float* a = fn + 3 * (h / k);
        const float* b = fn + 3 * (items[opp[p]] / k);
        float dot = fmaf(a[0], b[0], fmaf(a[1], b[1], a[2] * b[2]));
        float la = fmaf(a[0], a[0], fmaf(a[1], a[1], a[2] * a[2]));
        float lb = fmaf(b[0], b[0], fmaf(b[1], b[1], b[2] * b[2]));
        float c = dot / sqrtf(la * lb);
        if (c < cthr) { feat[v] = 1; feat[d] = 1; }
    }
}

__global__ void k_u8_to_int(const uint8_t* __restrict__ a, int n, int* __restrict__ b)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = a[i] ? 1 : 0;
}

// stable partition of [0,nS): flag==0 first; identity on [nS,nV)
__global__ void k_partition_surface(const int* __restrict__ flag, const int* __restrict__ scan, int nS, int nV,
                                    int nZero, int* __restrict__ newid)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nV) return;
    if (v >= nS) { newid[v] = v; return; }
    int ones = scan[v];
    newid[v] = flag[v] ? nZero + ones : (v - ones);
}

// merged raw + dummy halfedges: raw sorted position p keeps (src, dst, face);
// every raw halfedge without opposite adds (dst -> src, face -1), appended in
// sorted-position order (k_addBoundaryHalfedges + stable compaction)
__global__ void k_he_merge(const int* __restrict__ row, const int* __restrict__ items, const int* __restrict__ opp,
                           const int* __restrict__ dpos, int nS, int nRaw, const int* __restrict__ faces, int k,
                           int* __restrict__ mKey, int* __restrict__ mTgt, int* __restrict__ mFace)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nS) return;
    for (int p = row[v]; p < row[v + 1]; ++p) {
        int h = items[p];
        int d = he_dst(faces, k, h);
        mKey[p] = v; mTgt[p] = d; mFace[p] = h / k;
        if (opp[p] == -1) {
            int q = nRaw + dpos[p];
            mKey[q] = d; mTgt[q] = v; mFace[q] = -1;
        }
    }
}

__global__ void k_noopp(const int* __restrict__ opp, int n, int* __restrict__ flag)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) flag[i] = (opp[i] == -1) ? 1 : 0;
}

__global__ void k_gather2(const int* __restrict__ items, int n, const int* __restrict__ a, const int* __restrict__ b,
                          int* __restrict__ oa, int* __restrict__ ob)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) { oa[i] = a[items[i]]; ob[i] = b[items[i]]; }
}

__global__ void k_opp_sorted(const int* __restrict__ row, int nS, const int* __restrict__ tgt, int* __restrict__ opp)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nS) return;
    for (int p = row[v]; p < row[v + 1]; ++p) {
        int d = tgt[p], o = -1;
        for (int q = row[d]; q < row[d + 1]; ++q) if (tgt[q] == v) o = q;
        opp[p] = o;
    }
}

__device__ __forceinline__ int third_vertex(const int* f, int k, int src, int dst)
{
    if (k == 3) {
        if (f[0] != src && f[0] != dst) return f[0];
        if (f[1] != src && f[1] != dst) return f[1];
        return f[2];
    }
    if (dst == f[1]) return f[3];
    if (dst == f[2]) return f[0];
    if (dst == f[3]) return f[1];
    return f[2];
}

// counter-clockwise fan order per vertex (k_sortCCWDummyOpposite): start at
// the boundary halfedge whose twin is a dummy, else at the smallest feature
// neighbour (feature vertices), else at the smallest neighbour; then walk to
// the halfedge pointing at the third vertex of the current face.
__global__ void k_ccw(const int* __restrict__ row, int nS, const int* __restrict__ tgt, const int* __restrict__ face,
                      const int* __restrict__ opp, const uint8_t* __restrict__ b1d, const uint8_t* __restrict__ feat,
                      const int* __restrict__ faces, int k, int* __restrict__ order, int* __restrict__ err)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nS) return;
    int st = row[v], cnt = row[v + 1] - st;
    if (cnt == 0) { atomicOr(err, 1); return; }
    int cur = st;
    if (b1d[v]) {
        int j = 0;
        while (opp[cur] < 0 || face[opp[cur]] != -1) {
            ++j;
            if (j >= cnt) { atomicOr(err, 2); return; }
            cur = st + j;
        }
    } else if (feat[v]) {
        int best = -1, bt = 0x7fffffff;
        for (int j = 0; j < cnt; ++j) {
            int t = tgt[st + j];
            if (feat[t] && t < bt) { bt = t; best = j; }
        }
        if (best < 0) { atomicOr(err, 4); return; }
        cur = st + best;
    } else {
        for (int j = 1; j < cnt; ++j) if (tgt[st + j] < tgt[cur]) cur = st + j;
    }
    int pos = 0;
    order[st + pos++] = cur;
    bool found;
    do {
        int f = face[cur];
        if (f < 0) { atomicOr(err, 8); return; }
        int nxt = third_vertex(faces + (size_t)f * k, k, v, tgt[cur]);
        found = false;
        for (int j = 0; j < cnt; ++j)
            if (tgt[st + j] == nxt) {
                found = true;
                cur = st + j;
                if (pos < cnt) order[st + pos] = cur;
                ++pos;
            }
    } while (found && pos < cnt);
    if (pos != cnt) atomicOr(err, 16);
}

// final opposite and next (last match), k_setOppositeHalfedgeHelper /
// k_setNextHalfedgeHelper
__global__ void k_opp_next(const int* __restrict__ row, int nS, const int* __restrict__ tgt, const int* __restrict__ face,
                           int* __restrict__ opp, int* __restrict__ next)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nS) return;
    for (int p = row[v]; p < row[v + 1]; ++p) {
        int d = tgt[p], o = -1, nx = -1, f = face[p];
        for (int q = row[d]; q < row[d + 1]; ++q) {
            if (tgt[q] == v) o = q;
            if (face[q] == f) nx = q;
        }
        opp[p] = o;
        next[p] = nx;
    }
}

__global__ void k_row_sizes(const int* __restrict__ row, int n, int* __restrict__ mx)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v < n) atomicMax(mx, row[v + 1] - row[v]);
}

void build_surface(vsdmo_mesh& m, Renumber& rn, ClassChecks& checks, const SurfaceInputs& si,
                   const vsdmo_mesh_params& prm)
{
    hipStream_t s = m.stream;
    BuildArena& ar = rn.ar;
    const int nS = m.nSurf, nF = m.nFaces, k = m.fpe;
    const int nV = m.nV;
    m.isB1D.alloc(std::max(nS, 1));
    m.isFeature.alloc(std::max(nS, 1));
    VSDMO_HIP(hipMemsetAsync(m.isB1D.p, 0, std::max(nS, 1), s));
    VSDMO_HIP(hipMemsetAsync(m.isFeature.p, 0, std::max(nS, 1), s));
    if (nS == 0 || nF == 0) {
        m.nFree = 0; m.nFeature = 0;
        m.colOffFree = { 0 };
        m.colOffFeature = { 0 };
        m.heRow.alloc(1);
        VSDMO_HIP(hipMemsetAsync(m.heRow.p, 0, sizeof(int), s));
        return;
    }
    const int nRaw = nF * k;
    float ang = prm.feature_angle_deg > 0.0f ? prm.feature_angle_deg : 20.0f;
    const float cthr = (float)std::cos((double)ang * 3.14159265358979323846 / 180.0);
    // features on the current numbering
    {
        DevBuf<float> fn(ar, (size_t)nF * 3);
        k_face_normals<<<nblk(nF), TB, 0, s>>>(m.x.p, m.y.p, m.z.p, m.faces.p, nF, k, fn.p);
        DevBuf<int> key(ar, nRaw), row(ar), items(ar), opp(ar, nRaw);
        k_he_src<<<nblk(nRaw), TB, 0, s>>>(m.faces.p, nRaw, key.p);
        stable_csr(ar, key.p, nRaw, nS, row, items, s);
        k_he_opp_raw<<<nblk(nS), TB, 0, s>>>(row.p, items.p, nS, m.faces.p, k, opp.p);
        k_features<<<nblk(nS), TB, 0, s>>>(row.p, items.p, opp.p, nS, m.faces.p, k, fn.p, m.flat, cthr,
                                           m.isB1D.p, m.isFeature.p);
        VSDMO_HIP(hipGetLastError());
    }
    // [free | feature], stable
    {
        DevBuf<int> flag(ar, nS), scan(ar, nS), newid(ar, nV);
        k_u8_to_int<<<nblk(nS), TB, 0, s>>>(m.isFeature.p, nS, flag.p);
        int nFeat = exclusive_scan(flag.p, scan.p, nS, s);
        int nFree = nS - nFeat;
        k_partition_surface<<<nblk(nV), TB, 0, s>>>(flag.p, scan.p, nS, nV, nFree, newid.p);
        rn.apply(newid.p, true);
        m.nFree = nFree;
        m.nFeature = nFeat;
    }
    m.colOffFree = colour_and_sort(m, rn, checks, si.incRow, si.incVal, 0, m.nFree, prm, true);
    m.colOffFeature = colour_and_sort(m, rn, checks, si.incRow, si.incVal, m.nFree, nS, prm, true);
    // halfedges on the final numbering
    {
        DevBuf<int> key(ar, nRaw), row(ar), items(ar), opp(ar, nRaw), noopp(ar, nRaw), dpos(ar, nRaw);
        k_he_src<<<nblk(nRaw), TB, 0, s>>>(m.faces.p, nRaw, key.p);
        stable_csr(ar, key.p, nRaw, nS, row, items, s);
        k_he_opp_raw<<<nblk(nS), TB, 0, s>>>(row.p, items.p, nS, m.faces.p, k, opp.p);
        k_noopp<<<nblk(nRaw), TB, 0, s>>>(opp.p, nRaw, noopp.p);
        int nd = exclusive_scan(noopp.p, dpos.p, nRaw, s);
        int tot = nRaw + nd;
        DevBuf<int> mKey(ar, tot), mTgt(ar, tot), mFace(ar, tot);
        k_he_merge<<<nblk(nS), TB, 0, s>>>(row.p, items.p, opp.p, dpos.p, nS, nRaw, m.faces.p, k, mKey.p, mTgt.p, mFace.p);
        DevBuf<int> items2(ar);
        stable_csr(ar, mKey.p, tot, nS, m.heRow, items2, s);
        DevBuf<int> sTgt(ar, tot), sFace(ar, tot), sOpp(ar, tot), order(ar, tot), err(ar, 2);   // err: fan walk, longest row
        k_gather2<<<nblk(tot), TB, 0, s>>>(items2.p, tot, mTgt.p, mFace.p, sTgt.p, sFace.p);
        k_opp_sorted<<<nblk(nS), TB, 0, s>>>(m.heRow.p, nS, sTgt.p, sOpp.p);
        VSDMO_HIP(hipMemsetAsync(err.p, 0, 2 * sizeof(int), s));
        VSDMO_HIP(hipMemsetAsync(order.p, 0, sizeof(int) * tot, s));
        k_ccw<<<nblk(nS), TB, 0, s>>>(m.heRow.p, nS, sTgt.p, sFace.p, sOpp.p, m.isB1D.p, m.isFeature.p, m.faces.p, k,
                                      order.p, err.p);
        k_row_sizes<<<nblk(nS), TB, 0, s>>>(m.heRow.p, nS, err.p + 1);
        {
            const int* h = read_ints(err.p, 2, s);
            const int herr = h[0];
            m.maxHE = h[1];
            if (herr)
                throw StatusError{ VSDMO_TOPOLOGY, "surface halfedge fan walk failed (non-manifold surface?) code " +
                                                       std::to_string(herr) };
        }
        m.heTarget.alloc(tot); m.heFace.alloc(tot); m.heOpp.alloc(tot); m.heNext.alloc(tot);
        k_gather2<<<nblk(tot), TB, 0, s>>>(order.p, tot, sTgt.p, sFace.p, m.heTarget.p, m.heFace.p);
        k_opp_next<<<nblk(nS), TB, 0, s>>>(m.heRow.p, nS, m.heTarget.p, m.heFace.p, m.heOpp.p, m.heNext.p);
        VSDMO_HIP(hipGetLastError());
        m.nHE = tot;
    }
}

}  // namespace vsdmo
