// dmo_kernels.hip -- DMO vertex-search and quality kernels for gfx950.
//
// One wave64 per vertex; 4 of them where a launch or a list is short (*_vertex_wide),
// a quarter of one for flat triangles of large classes (flat_group8).  The one-ring is staged in LDS as per-element
// constants in a vertex-local frame.  A level of the 3D searches has nq^3
// candidates, index i + nq (j + nq k), the lowest index winning ties; bounds
// leave out what cannot decide it (tet_vertex: candidates no better than the
// current score; hex_vertex: sub-tets no candidate's minimum can be), and what
// is left is scored in the canonical order, so every result is the full
// search's, bit for bit.
//
// Reference kernels: k_optimizeHierarchicalInnerTet / Hex
// (VSDMO/src/dmo/DMOTetImplCub.h:20-137, DMOHexImplCub.h:20-137) and
// k_optimizeHierarchical2DFlat (DMOTriFlatImplCub.h:23-152).
#include <float.h>
#include <type_traits>

#include "vsdmo_internal.h"
#include "vsdmo_numerics.h"
#include "dmo_kernels.h"
#include "mlp_internal.h"

namespace vsdmo {

// a = fminf(a, ..) without the canonicalising v_max per operand that fminf costs
// here (no operand comes straight from a transcendental instruction)
__device__ __forceinline__ void min_into(float& a, float b) { asm("v_min_f32 %0, %0, %1" : "+v"(a) : "v"(b)); }
__device__ __forceinline__ void min_into(float& a, float b, float c)
{
    asm("v_min3_f32 %0, %0, %1, %2" : "+v"(a) : "v"(b), "v"(c));
}

// ------------------------------------------------------------------ tets
// LDS of a tet vertex search: the ring's constants, the level's plane of each
// element (4 floats: gradient, offset for cells; the offset for candidates in
// an array of its own; both padded to tiles of 16), the cells a level keeps and
// the candidates to score
constexpr int kTetCells = 64, kTetBuf = 128, kTetFew = 3;
__host__ __device__ constexpr int tet_rows(int ringCap) { return (ringCap + 15) / 16 * 16; }
__host__ __device__ constexpr size_t tet_wave_lds(int ringCap)
{
    return sizeof(TetC) * (size_t)ringCap + 5 * sizeof(float) * (size_t)tet_rows(ringCap) +
           (kTetCells + kTetBuf) * sizeof(int);
}

// the staged state of one vertex search
struct TetFrame {
    float x0x, x0y, x0z, ex, ey, ez, sg, is3;
    int n;
};

typedef float v4f __attribute__((ext_vector_type(4)));
// or of the bits of 4 products: its sign bit says whether one is negative (a
// fminf of a product costs a canonicalising v_max per operand besides)
__device__ __forceinline__ int sign4(v4f v)
{
    const float a = v[0], b = v[1], c = v[2], d = v[3];
    return __builtin_bit_cast(int, a) | __builtin_bit_cast(int, b) | __builtin_bit_cast(int, c) | __builtin_bit_cast(int, d);
}
// m[t]: per lane the or over 4 of 16 rows of column 16 t + lane % 16 (the lane's
// group lane / 16 holds rows 4 (lane / 16) + 0..3).  Returns the or over all
// rows of column `lane`: the swaps exchange halves, then odd and even groups,
// so that group t collects column tile t.  Every lane must call it.
__device__ __forceinline__ int or_columns(const int (&m)[4])
{
    auto swap32 = [](int a, int b) {
        const auto r = __builtin_amdgcn_permlane32_swap((unsigned)a, (unsigned)b, false, false);
        return (int)(r[0] | r[1]);
    };
    auto swap16 = [](int a, int b) {
        const auto r = __builtin_amdgcn_permlane16_swap((unsigned)a, (unsigned)b, false, false);
        return (int)(r[0] | r[1]);
    };
    return swap16(swap32(m[0], m[2]), swap32(m[1], m[3]));
}

// The nested grid search of a tet vertex, one wave.
//
// A candidate beats the current score q only if det > y L^1.5 for every ring
// element, y = (q / kCTet)^1.5.  With L = 3 F, F = |p - g|^2 + K, the function f =
// det - s F^1.5, s = 3^1.5 y, is concave (det is affine, F^1.5 convex), so it
// stays below its tangent plane at the window's centre: a candidate below 0 on
// some element's plane is no better.  One lane per element makes the level's
// planes.  The 64 cells of 2 x 2 x 2 candidates (nq 8) are tried against them in
// one small matrix product on the FP32 MFMA, (plane) x (cell centre, 1); a
// plane's maximum over a cell is its value at the centre plus sum h |gradient|.
// The kept cells' candidates are tried the same way, 8 cells at a time, and
// what is left is scored in the canonical order, one candidate per lane over
// the whole ring, or, up to kTetFew of them, one after the other with one
// element per lane.  The best score (the lowest index on a tie) is the level's:
// the full search's bits.  Scoring 512 candidates takes ~98 VALU operations per
// element.  On 40^3 cubes 0 / 0-1 / 5-30 candidates of the three levels are
// scored once the mesh has settled, 50-90 at the start.
//
// Margins: s carries -2^-9, the planes 2^-18 of the sum of their terms'
// magnitudes over the search's reach P (a.reach in window units), K is lowered
// by 2^-18 of L's terms, and a candidate's coordinates may be off by delta (1e-3
// of the spacing and 2^-20 of the world coordinate); the canonical evaluation
// rounds by a few 2^-24, its selection by ~2^-22 per comparison.  Vertices at q
// < 0 (an inverted ring) look at the cells with positive planes first and at the
// others only if no candidate there reaches 0.  Frames outside the planes'
// range score every candidate.
//
// Bound by VALU issue (and the matrix unit, ~15 % of the time).  Scoring every
// candidate, with 8 candidates per lane, took 9,200 VALU operations per vertex
// and 81 us per class of the 40^3 cube (7,400 vertices); here 3,950 and 80 us
// in the first iteration, 1,270 and 25 us in the 20th.  A gradient bound at
// every cell's centre instead of the planes (23 operations per element and 64
// cells) took 3,430 on average against 1,920; the planes as fused multiply-adds
// over LDS broadcasts 2,240; ranking the kept candidates by det F^-1.5 on the
// MFMA before scoring was slower than scoring them (8.9 against 6.9 ms per 20
// iterations).
template <int NQ>
__device__ void tet_vertex(const SearchArgs& a, int vid, bool emin, unsigned char* lds, int ringCap)
{
    const int lane = (int)(threadIdx.x & 63);
    TetC* s_tc = reinterpret_cast<TetC*>(lds);
    float* s_pl = reinterpret_cast<float*>(s_tc + ringCap);
    float* s_pw = s_pl + 4 * tet_rows(ringCap);
    int* s_cell = reinterpret_cast<int*>(s_pw + tet_rows(ringCap));
    int* s_buf = s_cell + kTetCells;
    TetFrame f;
    const int r0 = uniform(a.ringRow[vid]);
    f.n = uniform(a.ringRow[vid + 1]) - r0;
    if (f.n <= 0) return;   // no element: nothing scores below the start
    f.x0x = a.x[vid]; f.x0y = a.y[vid]; f.x0z = a.z[vid];
    float ex = emin ? FLT_MAX : -FLT_MAX, ey = ex, ez = ex, mabs = 0.0f;
    auto extent = [&](float dxs, float dys, float dzs) {
        const float dx = fabsf(dxs), dy = fabsf(dys), dz = fabsf(dzs);
        ex = emin ? fminf(ex, dx) : fmaxf(ex, dx);
        ey = emin ? fminf(ey, dy) : fmaxf(ey, dy);
        ez = emin ? fminf(ez, dz) : fmaxf(ez, dz);
        mabs = fmaxf(mabs, fmaxf(dx, fmaxf(dy, dz)));
    };
    // the lane's first element keeps its corner offsets in registers for the
    // constants, so the positions are read from memory once
    const bool own0 = lane < f.n;
    float d0[3][3];
    if (own0) {
        const int* h = a.ringVal + (size_t)(r0 + lane) * 3;
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const int v = h[t];
            d0[t][0] = a.x[v] - f.x0x; d0[t][1] = a.y[v] - f.x0y; d0[t][2] = a.z[v] - f.x0z;
            extent(d0[t][0], d0[t][1], d0[t][2]);
        }
    }
    for (int e = lane + 64; e < f.n; e += 64) {
        const int* h = a.ringVal + (size_t)(r0 + e) * 3;
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const int v = h[t];
            extent(a.x[v] - f.x0x, a.y[v] - f.x0y, a.z[v] - f.x0z);
        }
    }
    if (emin) { f.ex = wave_min_u(ex); f.ey = wave_min_u(ey); f.ez = wave_min_u(ez); }
    else { f.ex = wave_max_u(ex); f.ey = wave_max_u(ey); f.ez = wave_max_u(ez); }
    f.sg = pow2_scale(wave_max_u(mabs));
    const float isg = 1.0f / f.sg;
    f.is3 = ((1.0f * isg) * isg) * isg;
    TetC c0{ 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f };
    if (own0) {
        f3 p[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) p[t] = { d0[t][0] * f.sg, d0[t][1] * f.sg, d0[t][2] * f.sg };
        c0 = tet_consts(p[0], p[1], p[2]);
        s_tc[lane] = c0;
    }
    for (int e = lane + 64; e < f.n; e += 64) {
        const int* h = a.ringVal + (size_t)(r0 + e) * 3;
        f3 p[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            int v = h[t];
            p[t] = { (a.x[v] - f.x0x) * f.sg, (a.y[v] - f.x0y) * f.sg, (a.z[v] - f.x0z) * f.sg };
        }
        s_tc[e] = tet_consts(p[0], p[1], p[2]);
    }
    wave_lds_fence();

    auto lanes_score = [&](float det, float L, float& q) { return tet_lanes_score(own0, det, L, f.is3, q); };
    // start score (p = 0: det = D, L = K exactly)
    float qcur = 0.0f;
    if (f.n > 64 || !lanes_score(c0.D, c0.K, qcur)) {
        TetAcc acc = tet_acc0();
        for (int e = 0; e < f.n; ++e) tet_acc_add(acc, s_tc[e].D, s_tc[e].K);
        qcur = tet_acc_score(acc, f.is3);
    }

    constexpr int NB = NQ / 2, NC = NB * NB * NB;   // cells per axis, cells
    constexpr unsigned long long kAllCells = NC == 64 ? ~0ull : (1ull << NC) - 1ull;
    constexpr float kR = 0x1p-18f, kStep = 1.0f / (float)(NQ - 1);
    // P bounds every candidate's frame coordinates
    const float P = 2.03f * a.reach + 0x1p-17f * (fmaxf(fabsf(f.x0x), fmaxf(fabsf(f.x0y), fabsf(f.x0z))) * f.sg);
    // the element's g and lowered K (F = |p - g|^2 + K)
    struct Quad { float gx, gy, gz, K; };
    auto quad = [&](const TetC& c) {
        Quad q;
        q.gx = c.m2sx * (-1.0f / 6.0f); q.gy = c.m2sy * (-1.0f / 6.0f); q.gz = c.m2sz * (-1.0f / 6.0f);
        q.K = (c.K * (1.0f / 3.0f) - fmaf(q.gx, q.gx, fmaf(q.gy, q.gy, q.gz * q.gz))) -
              kR * (c.K + P * (fabsf(c.m2sx) + fabsf(c.m2sy) + fabsf(c.m2sz) + 9.0f * P));
        return q;
    };
    const Quad q0 = quad(c0);
    const int comp = lane >> 4, col = lane & 15;   // the lane's row (x, y, z, 1) and column of the products' operands
    const int nt = (f.n + 15) >> 4;
    bool fast = false;
    // cell `lane`, packed indices along x, y, z; column 16 t + col's place along
    // the lane's axis in window half-widths (candidate i lies at 1 - 2 i / (nq -
    // 1), a cell between candidates 2 b and 2 b + 1)
    const int myCell = (lane % NB) | ((lane / NB) % NB) << 8 | (lane / (NB * NB)) << 16;
    float cellU[4] = { 0.0f, 0.0f, 0.0f, 0.0f };
    if constexpr (NC > 8) {
        bool ok = P <= 32.0f;
        ok = ok && (!own0 || (q0.K >= kSelF && c0.K <= 4096.0f));
        for (int e = lane + 64; e < f.n; e += 64) ok = ok && quad(s_tc[e]).K >= kSelF && s_tc[e].K <= 4096.0f;
        fast = __ballot(!ok) == 0ull;
        // rows past the ring bound nothing
        if (lane < 16 * nt - f.n) {
            const int e = f.n + lane;
            *reinterpret_cast<float4*>(s_pl + 4 * e) = make_float4(0.0f, 0.0f, 0.0f, 1e30f);
            s_pw[e] = 1e30f;
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int cell = 16 * t + col;
            const int b = comp == 0 ? cell % NB : comp == 1 ? (cell / NB) % NB : cell / (NB * NB);
            cellU[t] = 1.0f - kStep * (float)(4 * b + 1);
        }
    }
    // the lane's plane operand of tile et, for cells and for candidates
    const float* const opCell = s_pl + 4 * col + comp;
    const float* const opCand = comp < 3 ? opCell : s_pw + col;
    const int opStep = comp < 3 ? 64 : 16;

    float cx = f.x0x, cy = f.x0y, cz = f.x0z, ds = a.gridScale;
    bool moved = false;
    for (int d = 0; d < a.depth; ++d, ds = ds * a.shrink) {
        const float gxM = cx + ds * f.ex, gxm = cx - ds * f.ex;
        const float gyM = cy + ds * f.ey, gym = cy - ds * f.ey;
        const float gzM = cz + ds * f.ez, gzm = cz - ds * f.ez;
        // det / L^1.5 of the current score, less the margin; 0: only the signs decide
        float yq = 0.0f;
        if (fast && qcur > 0.0f) {
            const float t = qcur * (1.0f / kCTet);
            yq = (t * __builtin_amdgcn_sqrtf(t)) * (1.0f - 0x1p-9f);
            if (!(yq >= kSelY)) yq = 0.0f;
        }
        const float s = yq * 5.1961524f;   // 3^1.5: against det / F^1.5
        unsigned long long mask = kAllCells, rest = 0ull;
        float o = 0.0f, D = 0.0f;   // the window's centre and half-width along the lane's axis
        // the window's half-widths in frame coordinates.  Below kTiny the planes'
        // margins keep it whole: every candidate is scored without them (6 iterations
        // at depth 8: 32^3 5.3 -> 5.1 ms at any line from 2^-9 to 2^-7, 20^3 at nq 6 2.57 ms
        // at 2^-8, 2.42 at 2^-7)
        constexpr float kTiny = 0x1p-7f;
        const float Dx = (ds * f.ex) * f.sg, Dy = (ds * f.ey) * f.sg, Dz = (ds * f.ez) * f.sg;
        const bool planes = NC > 8 && fast && fmaxf(Dx, fmaxf(Dy, Dz)) > kTiny;
        if constexpr (NC > 8) if (planes) {
            const float ox = (cx - f.x0x) * f.sg, oy = (cy - f.x0y) * f.sg, oz = (cz - f.x0z) * f.sg;   // its centre
            const float dx = 1e-3f * kStep * Dx + 0x1p-20f * ((fabsf(cx) + ds * f.ex) * f.sg);
            const float dy = 1e-3f * kStep * Dy + 0x1p-20f * ((fabsf(cy) + ds * f.ey) * f.sg);
            const float dz = 1e-3f * kStep * Dz + 0x1p-20f * ((fabsf(cz) + ds * f.ez) * f.sg);
            auto plane = [&](int e, const TetC& c, const Quad& q) {
                const float wx = ox - q.gx, wy = oy - q.gy, wz = oz - q.gz;
                const float F = fmaf(wx, wx, fmaf(wy, wy, fmaf(wz, wz, q.K)));
                const float sr = s * __builtin_amdgcn_sqrtf(F), g = 3.0f * sr;
                const float px = fmaf(-g, wx, c.nnx), py = fmaf(-g, wy, c.nny), pz = fmaf(-g, wz, c.nnz);
                const float det = fmaf(c.nnx, ox, fmaf(c.nny, oy, fmaf(c.nnz, oz, c.D)));
                const float ax = fabsf(px), ay = fabsf(py), az = fabsf(pz);
                const float m = kR * (fabsf(c.D) + sr * F +
                                      P * ((ax + ay + az) + (fabsf(c.nnx) + fabsf(c.nny) + fabsf(c.nnz))));
                const float w = (fmaf(-sr, F, det) - fmaf(px, ox, fmaf(py, oy, pz * oz))) +
                                (m + fmaf(ax, dx, fmaf(ay, dy, az * dz)));
                *reinterpret_cast<float4*>(s_pl + 4 * e) =
                    make_float4(px, py, pz, fmaf(ax, kStep * Dx, fmaf(ay, kStep * Dy, fmaf(az, kStep * Dz, w))));
                s_pw[e] = w;
            };
            if (own0) plane(lane, s_tc[lane], q0);
            for (int e = lane + 64; e < f.n; e += 64) plane(e, s_tc[e], quad(s_tc[e]));
            wave_lds_fence();
            o = comp == 0 ? ox : comp == 1 ? oy : comp == 2 ? oz : 1.0f;
            D = comp == 0 ? Dx : comp == 1 ? Dy : comp == 2 ? Dz : 0.0f;
            int neg[4] = { 0, 0, 0, 0 };
            for (int et = 0; et < nt; ++et) {
                const float A = opCell[64 * et];
#pragma unroll
                for (int t = 0; t < (NC + 15) / 16; ++t) {
                    neg[t] |= sign4(__builtin_amdgcn_mfma_f32_16x16x4f32(A, fmaf(D, cellU[t], o), v4f{ 0.0f, 0.0f, 0.0f, 0.0f }, 0, 0, 0));
                }
            }
            mask = __ballot(or_columns(neg) >= 0) & kAllCells;
            if (qcur < 0.0f) {
                rest = kAllCells & ~mask;
                if (mask == 0ull) { mask = rest; rest = 0ull; }
            }
        }
        float best = -FLT_MAX;
        int cand = 0;
        auto better = [&](float q, int code) {   // uniform
            if (q > best || (q == best && code < cand)) { best = q; cand = code; }
        };
        // every candidate, index i + nq (j + nq k): a line along x per lane, half of
        // it at a time (the whole line's accumulators would spill)
        constexpr int H = NQ / 2;
        auto score_all = [&]() {
            const int j = lane % NQ, k = lane / NQ;
            const float py = (grid_coord(a.aff, j, NQ, gym, gyM) - f.x0y) * f.sg;
            const float pz = (grid_coord(a.aff, k, NQ, gzm, gzM) - f.x0z) * f.sg;
            const float Qyz = 3.0f * fmaf(pz, pz, py * py);
            float own = -FLT_MAX;
            int bi = 0;
#pragma unroll 1
            for (int i0 = 0; i0 < NQ; i0 += H) {
                float px[H], t3[H];
                TetAcc acc[H];
#pragma unroll
                for (int i = 0; i < H; ++i) {
                    px[i] = (grid_coord(a.aff, i0 + i, NQ, gxm, gxM) - f.x0x) * f.sg;
                    t3[i] = 3.0f * px[i];
                    acc[i] = tet_acc0();
                }
#pragma unroll 1
                for (int e = 0; e < f.n; ++e) {
                    const TetC t = s_tc[e];
                    const float Tyz = fmaf(t.nny, py, fmaf(t.nnz, pz, t.D));
                    const float Ryz = fmaf(t.m2sy, py, fmaf(t.m2sz, pz, t.K + Qyz));
#pragma unroll
                    for (int i = 0; i < H; ++i) {   // tet_acc_add
                        const float det = fmaf(t.nnx, px[i], Tyz), L = fmaf(px[i], t3[i] + t.m2sx, Ryz);
                        const float d2 = det * det, L3 = (L * L) * L;
                        const bool take = d2 * acc[i].bL3 < acc[i].bd2 * L3;
                        acc[i].bd2 = take ? d2 : acc[i].bd2;
                        acc[i].bL3 = take ? L3 : acc[i].bL3;
                        min_into(acc[i].dmin, det);
                    }
                }
#pragma unroll
                for (int i = 0; i < H; ++i) {
                    const float q = tet_acc_score(acc[i], f.is3);
                    if (lane < NQ * NQ && q > own) { own = q; bi = i0 + i; }
                }
            }
            const float m = wave_max_u(own);
            const int l = __builtin_ctzll(__ballot(own == m));
            better(m, __builtin_amdgcn_readlane(bi, l) + NQ * l);
        };
        // the canonical scores of the first n (at most 64) buffered candidates; with
        // no more than 64 in all, of candidate `lane`
        auto score = [&](int n) {
            const int code = NC > 8 ? s_buf[min(lane, n - 1)] : min(lane, n - 1);   // lanes past n repeat the last one
            if (n <= kTetFew && f.n <= 64) {
                const TetC c0 = s_tc[own0 ? lane : 0];
                bool told = true;
                for (int c = 0; c < n && told; ++c) {
                    const int at = __builtin_amdgcn_readlane(code, c);
                    const float px = (grid_coord(a.aff, at % NQ, NQ, gxm, gxM) - f.x0x) * f.sg;
                    const float py = (grid_coord(a.aff, (at / NQ) % NQ, NQ, gym, gyM) - f.x0y) * f.sg;
                    const float pz = (grid_coord(a.aff, at / (NQ * NQ), NQ, gzm, gzM) - f.x0z) * f.sg;
                    const float Qyz = 3.0f * fmaf(pz, pz, py * py), t3 = 3.0f * px;
                    const float Tyz = fmaf(c0.nny, py, fmaf(c0.nnz, pz, c0.D));
                    const float Ryz = fmaf(c0.m2sy, py, fmaf(c0.m2sz, pz, c0.K + Qyz));
                    float q = 0.0f;
                    told = lanes_score(fmaf(c0.nnx, px, Tyz), fmaf(px, t3 + c0.m2sx, Ryz), q);
                    if (told) better(q, at);
                }
                if (told) return;
            }
            // up to 16 (32) candidates: the four (two) lanes of a candidate take a
            // quarter (half) of the ring each
            const int split = !fast ? 1 : n <= 16 ? 4 : n <= 32 ? 2 : 1;
            const int mine = split == 1 ? code : s_buf[min(lane & (split == 4 ? 15 : 31), n - 1)];
            const int part = split == 1 ? 0 : split == 4 ? lane >> 4 : lane >> 5;
            const float px = (grid_coord(a.aff, mine % NQ, NQ, gxm, gxM) - f.x0x) * f.sg;
            const float py = (grid_coord(a.aff, (mine / NQ) % NQ, NQ, gym, gyM) - f.x0y) * f.sg;
            const float pz = (grid_coord(a.aff, mine / (NQ * NQ), NQ, gzm, gzM) - f.x0z) * f.sg;
            const float Qyz = 3.0f * fmaf(pz, pz, py * py), t3 = 3.0f * px;
            TetAcc acc = tet_acc0();
            auto ring = [&](int first, int len) {   // a part's last element may repeat: it changes nothing
#pragma unroll 4
                for (int e = 0; e < len; ++e) {
                    const TetC t = s_tc[min(first + e, f.n - 1)];
                    const float Tyz = fmaf(t.nny, py, fmaf(t.nnz, pz, t.D));
                    const float Ryz = fmaf(t.m2sy, py, fmaf(t.m2sz, pz, t.K + Qyz));
                    tet_acc_add(acc, fmaf(t.nnx, px, Tyz), fmaf(px, t3 + t.m2sx, Ryz));
                }
            };
            const int len = (f.n + split - 1) / split;
            ring(part * len, len);
            if (split > 1) {
                // the parts in ring order: the later one's pair where its ratio is
                // clearly smaller, the earlier one's where it is clearly larger;
                // where neither, or the determinants leave the selection's range,
                // the wave scores the ring in one piece.  Clearly: by more than
                // kJoin, which exceeds what a chain of near ties can shift: a comparison
                // of two rounded products takes or leaves a pair wrongly only within
                // 2^-23 of the selected one, so over the at most 512 elements of a part a
                // selection that starts elsewhere ends with the same pair, or within 514 x
                // 2^-23 < 2^-13 of where it started.  (At 2^-8 two parts' minima often came
                // too close and the ring was gone through again: 40^3 cube, 20
                // iterations, 6.56 against 6.22 ms.)
                constexpr float kJoin = 0x1p-12f;
                static_assert(kJoin >= 2.0f * (kMaxRingTet / 2 + 2) * 0x1p-23f, "twice the shift of the largest part");
                bool told = true;
                auto join = [&](int far) {
                    const float od2 = __shfl_xor(acc.bd2, far), oL3 = __shfl_xor(acc.bL3, far), od = __shfl_xor(acc.dmin, far);
                    const float u = od2 * acc.bL3, v = acc.bd2 * oL3;
                    told = told && !(fabsf(u - v) <= kJoin * fmaxf(u, v));
                    acc.bd2 = u < v ? od2 : acc.bd2;
                    acc.bL3 = u < v ? oL3 : acc.bL3;
                    acc.dmin = fminf(acc.dmin, od);
                };
                if (split == 4) join(16);
                join(32);
                if (__ballot(!(told && acc.dmin >= kSelD) && !(acc.dmin < 0.0f)) != 0ull) {
                    acc = tet_acc0();
                    ring(0, f.n);
                }
            }
            // no cube roots where no ratio reaches the current score's
            if (yq > 0.0f &&
                __ballot(acc.dmin > 0.0f && acc.bd2 * __builtin_amdgcn_rcpf(acc.bL3) >= yq * yq) == 0ull)
                return;
            const float q = tet_acc_score(acc, f.is3);
            const float m = wave_max_u(q);
            unsigned long long bal = __ballot(q == m);
            int lo = 0x7fffffff;
            if (NC <= 8 && bal) { lo = __builtin_amdgcn_readlane(mine, __builtin_ctzll(bal)); bal = 0ull; }
            while (bal) {
                lo = min(lo, __builtin_amdgcn_readlane(mine, __builtin_ctzll(bal)));
                bal &= bal - 1;
            }
            better(m, lo);
        };
        if constexpr (NC <= 8) {
            score(NQ * NQ * NQ);
            mask = 0ull;
        }
        while (mask != 0ull) {
            const int cnt = __popcll(mask);
            // eight cells are a pass of one candidate per lane over the ring, all of
            // them two passes of H: with more cells than the latter costs (windows so
            // small that no plane tells their candidates apart, inverted rings) every
            // candidate is scored.  (6 iterations, through the lists / so: 32^3 at depth
            // 8 8.8 / 5.3 ms, 36^3 moved by 1,000 4.0 / 2.9 ms, 28^3 with jitter 0.9 2.4 /
            // 1.8 ms.  With the line at a third of the cells the 40^3 cube takes 6.1 ms
            // for 20 iterations, at a half 5.8.)  The coarser cells of nq 6 say less of their
            // candidates: there the lists are only left out with the planes (28^3 at nq 6,
            // 12 iterations 2.66 ms, with the line at 24 of 27 cells 2.69).
            if (NQ == 8 ? cnt > 8 * H : !planes) {
                score_all();
                break;
            }
            if ((mask >> lane) & 1ull) s_cell[__popcll(mask & ((1ull << lane) - 1ull))] = myCell;
            wave_lds_fence();
            int nbuf = 0;
            for (int c = 0; c < cnt; c += 8) {
                // candidate `lane` of the chunk: cell lane / 8, corner lane % 8
                const int cell = s_cell[min(c + (lane >> 3), cnt - 1)];
                const int code = (2 * (cell & 255) + (lane & 1)) +
                                 NQ * ((2 * ((cell >> 8) & 255) + ((lane >> 1) & 1)) +
                                       NQ * (2 * (cell >> 16) + ((lane >> 2) & 1)));
                bool keep = c + (lane >> 3) < cnt;
                if constexpr (NC > 8) if (fast && qcur >= 0.0f) {
                    // column 16 t + col: its coordinate along the lane's axis
                    float B[4];
                    int neg[4] = { 0, 0, 0, 0 };
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const int cl = s_cell[min(c + 2 * t + (col >> 3), cnt - 1)];
                        const int i = 2 * ((cl >> (8 * comp)) & 255) + ((lane >> comp) & 1);
                        B[t] = fmaf(D, 1.0f - 2.0f * kStep * (float)i, o);
                    }
                    for (int et = 0; et < nt; ++et) {
                        const float A = opCand[opStep * et];
#pragma unroll
                        for (int t = 0; t < 4; ++t)
                            neg[t] |= sign4(__builtin_amdgcn_mfma_f32_16x16x4f32(A, B[t], v4f{ 0.0f, 0.0f, 0.0f, 0.0f }, 0, 0, 0));
                    }
                    const int v = or_columns(neg);   // every lane takes part
                    keep = keep && v >= 0;
                }
                const unsigned long long bal = __ballot(keep);
                if (keep) s_buf[nbuf + __popcll(bal & ((1ull << lane) - 1ull))] = code;
                nbuf += __popcll(bal);
                wave_lds_fence();
                if (nbuf >= 64) {
                    score(64);
                    nbuf -= 64;
                    const int mv = s_buf[64 + lane];
                    wave_lds_fence();
                    if (lane < nbuf) s_buf[lane] = mv;
                    wave_lds_fence();
                }
            }
            if (nbuf > 0) score(nbuf);
            wave_lds_fence();   // the lists are rewritten
            mask = 0ull;
            if (!(best >= 0.0f)) { mask = rest; rest = 0ull; }
        }
        if (qcur < best) {
            const int wi = cand % NQ, wj = (cand / NQ) % NQ, wk = cand / (NQ * NQ);
            cx = grid_coord(a.aff, wi, NQ, gxm, gxM);
            cy = grid_coord(a.aff, wj, NQ, gym, gyM);
            cz = grid_coord(a.aff, wk, NQ, gzm, gzM);
            qcur = best;
            moved = true;
        }
    }
    if (moved && lane == 0) { a.xw[vid] = cx; a.yw[vid] = cy; a.zw[vid] = cz; }
}

// The same search on the 4 waves of a block, every candidate scored: lane l = j
// + nq k of wave w owns the candidates (i, j, k), i = w nq / 4 and on.  It takes
// twice the operations of tet_vertex, four times as many lanes at once, and
// none of tet_vertex's chain of filters and lists: for launches that leave most
// of the chip idle, where a vertex's chain sets the time (kTetWideMax).
// lds: tet_wide_lds bytes.
struct TetBest { float q; int cand; };
__host__ __device__ constexpr size_t tet_wide_lds(int ringCap)
{
    return sizeof(TetC) * (size_t)ringCap + 8 * sizeof(TetBest);
}
template <int NQ>
__device__ void tet_vertex_wide(const SearchArgs& a, int vid, unsigned char* lds, int ringCap)
{
    constexpr int W = 4, CPL = NQ / W;
    static_assert(NQ % W == 0 && NQ * NQ <= 64, "nq 4 or 8");
    const int lane = (int)(threadIdx.x & 63), wave = uniform((int)(threadIdx.x >> 6));
    const bool emin = a.extentMin != 0;
    TetC* s_tc = reinterpret_cast<TetC*>(lds);
    TetBest* s_best = reinterpret_cast<TetBest*>(s_tc + ringCap);   // [level parity][wave]
    TetFrame f;
    const int r0 = uniform(a.ringRow[vid]);
    f.n = uniform(a.ringRow[vid + 1]) - r0;
    if (f.n <= 0) return;
    f.x0x = a.x[vid]; f.x0y = a.y[vid]; f.x0z = a.z[vid];
    // every wave reads the whole ring (its frame needs no barrier), the first
    // one writes the constants
    float ex = emin ? FLT_MAX : -FLT_MAX, ey = ex, ez = ex, mabs = 0.0f;
    const bool own0 = lane < f.n;
    f3 d0[3];
    for (int e = lane; e < f.n; e += 64) {
        const int* h = a.ringVal + (size_t)(r0 + e) * 3;
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const int v = h[t];
            const f3 o = { a.x[v] - f.x0x, a.y[v] - f.x0y, a.z[v] - f.x0z };
            if (e == lane) d0[t] = o;
            const float dx = fabsf(o.x), dy = fabsf(o.y), dz = fabsf(o.z);
            ex = emin ? fminf(ex, dx) : fmaxf(ex, dx);
            ey = emin ? fminf(ey, dy) : fmaxf(ey, dy);
            ez = emin ? fminf(ez, dz) : fmaxf(ez, dz);
            mabs = fmaxf(mabs, fmaxf(dx, fmaxf(dy, dz)));
        }
    }
    if (emin) { f.ex = wave_min_u(ex); f.ey = wave_min_u(ey); f.ez = wave_min_u(ez); }
    else { f.ex = wave_max_u(ex); f.ey = wave_max_u(ey); f.ez = wave_max_u(ez); }
    f.sg = pow2_scale(wave_max_u(mabs));
    const float isg = 1.0f / f.sg;
    f.is3 = ((1.0f * isg) * isg) * isg;
    TetC c0{ 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f };
    if (own0) {
        c0 = tet_consts(scl3(d0[0], f.sg), scl3(d0[1], f.sg), scl3(d0[2], f.sg));
        if (wave == 0) s_tc[lane] = c0;
    }
    if (wave == 0)
        for (int e = lane + 64; e < f.n; e += 64) {
            const int* h = a.ringVal + (size_t)(r0 + e) * 3;
            f3 p[3];
            for (int t = 0; t < 3; ++t) {
                const int v = h[t];
                p[t] = { (a.x[v] - f.x0x) * f.sg, (a.y[v] - f.x0y) * f.sg, (a.z[v] - f.x0z) * f.sg };
            }
            s_tc[e] = tet_consts(p[0], p[1], p[2]);
        }
    __syncthreads();
    float qcur = 0.0f;
    if (f.n > 64 || !tet_lanes_score(own0, c0.D, c0.K, f.is3, qcur)) {
        TetAcc acc = tet_acc0();
        for (int e = 0; e < f.n; ++e) tet_acc_add(acc, s_tc[e].D, s_tc[e].K);
        qcur = tet_acc_score(acc, f.is3);
    }
    float cx = f.x0x, cy = f.x0y, cz = f.x0z, ds = a.gridScale;
    const int j = lane % NQ, k = lane / NQ;
    const bool active = lane < NQ * NQ;
    bool moved = false;
    for (int d = 0; d < a.depth; ++d, ds = ds * a.shrink) {
        const float gxM = cx + ds * f.ex, gxm = cx - ds * f.ex;
        const float gyM = cy + ds * f.ey, gym = cy - ds * f.ey;
        const float gzM = cz + ds * f.ez, gzm = cz - ds * f.ez;
        const float py = (grid_coord(a.aff, j, NQ, gym, gyM) - f.x0y) * f.sg;
        const float pz = (grid_coord(a.aff, k, NQ, gzm, gzM) - f.x0z) * f.sg;
        const float Qyz = 3.0f * fmaf(pz, pz, py * py);
        float px[CPL], t3[CPL];
        TetAcc acc[CPL];
#pragma unroll
        for (int i = 0; i < CPL; ++i) {
            px[i] = (grid_coord(a.aff, wave * CPL + i, NQ, gxm, gxM) - f.x0x) * f.sg;
            t3[i] = 3.0f * px[i];
            acc[i] = tet_acc0();
        }
#pragma unroll 4
        for (int e = 0; e < f.n; ++e) {
            const TetC c = s_tc[e];
            const float Tyz = fmaf(c.nny, py, fmaf(c.nnz, pz, c.D));
            const float Ryz = fmaf(c.m2sy, py, fmaf(c.m2sz, pz, c.K + Qyz));
#pragma unroll
            for (int i = 0; i < CPL; ++i)
                tet_acc_add(acc[i], fmaf(c.nnx, px[i], Tyz), fmaf(px[i], t3[i] + c.m2sx, Ryz));
        }
        float own = -FLT_MAX;
        int bi = 0;
#pragma unroll
        for (int i = 0; i < CPL; ++i) {
            const float q = tet_acc_score(acc[i], f.is3);
            if (active && q > own) { own = q; bi = i; }
        }
        const float m = wave_max_u(own);
        const int l = __builtin_ctzll(__ballot(own == m));
        if (lane == l) s_best[(d & 1) * W + wave] = { m, wave * CPL + bi + NQ * l };
        __syncthreads();   // one a level: the next one's values go to the other half
        float best = -FLT_MAX;
        int cand = 0;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const TetBest b = s_best[(d & 1) * W + w];
            if (b.q > best || (b.q == best && b.cand < cand)) { best = b.q; cand = b.cand; }
        }
        if (qcur < best) {
            cx = grid_coord(a.aff, cand % NQ, NQ, gxm, gxM);
            cy = grid_coord(a.aff, (cand / NQ) % NQ, NQ, gym, gyM);
            cz = grid_coord(a.aff, cand / (NQ * NQ), NQ, gzm, gzM);
            qcur = best;
            moved = true;
        }
    }
    if (moved && threadIdx.x == 0) { a.xw[vid] = cx; a.yw[vid] = cy; a.zw[vid] = cz; }
    __syncthreads();   // the next vertex restages the ring
}
// vertices up to which a launch takes tet_vertex_wide: by themselves, 4 waves
// per SIMD (plain tet cubes, 6 iterations, one wave per vertex against wide: 13^3
// with classes of ~170 vertices 1.24 / 0.92 ms, 20^3 with 500-900 1.45 / 1.30,
// 24^3 with up to 1,600 1.65 / 1.61; with the line at 2,048 24^3 takes 1.74), and
// beside a class's windows (40^3, mode 1: at 256 1.75 ms, at 512 1.77, at 1,024
// 1.84, never 1.87).  Beside the windows of a class of more than 4,096 vertices a
// short list is over before they are, in one wave per vertex and without the raised
// priority: four waves and the priority only hold the windows up (40^3, mode 3,
// ~100 vertices deferred of classes of ~7,400, one-mesh batch: 0.206 ms an iteration
// wide, 0.203 in one wave at raised priority, 0.201 in one wave without; 16^3 to
// 40^3 in mode 1 are the same within 2 %)
constexpr int kTetWideMax = 1024, kTetWideDef = 256, kTetWideClass = 4096;

// ------------------------------------------------------------------ hexes
struct HexLds { float cd[4], cF[4]; HexP hp[5]; };

// LDS of a hex vertex search per ring element: the constants and the codes of
// the element's sub-tets in the list of those a level scores
constexpr size_t kHexLdsPer = sizeof(HexLds) + 5 * sizeof(int);
// rounded up for a wave's slice of a block's LDS
__host__ __device__ constexpr size_t hex_wave_lds(int ringCap) { return (kHexLdsPer * (size_t)ringCap + 15) / 16 * 16; }
static_assert(tet_wave_lds(kMaxRingTet) <= 64 * 1024 && hex_wave_lds(kMaxRingHex) <= 64 * 1024, "a ring fits a block");
__device__ __forceinline__ int* hex_act(unsigned char* lds, int ringCap)
{
    return reinterpret_cast<int*>(lds + sizeof(HexLds) * (size_t)ringCap);
}

// staged state of a hex vertex search (as TetFrame), plus the accumulator of
// the 4 sub-tets per ring element that do not contain the moving vertex
struct HexFrame {
    float x0x, x0y, x0z, ex, ey, ez, sg, epsD, epsF;
    int n;
    bool corner8;   // the principal-axes sub-tet (slot 4 of HexP) left out
    bool inRange;   // hex_free_lanes: every p-free pair is in sel_range
    HexAcc acc0;
};

// One-wave staging of vid's ring: constants in LDS, the p-free accumulator.
__device__ HexFrame hex_stage(const SearchArgs& a, int vid, bool emin, HexLds* s_hx)
{
    const int lane = (int)(threadIdx.x & 63);
    HexFrame f;
    const int r0 = uniform(a.ringRow[vid]);
    f.n = uniform(a.ringRow[vid + 1]) - r0;
    f.x0x = a.x[vid]; f.x0y = a.y[vid]; f.x0z = a.z[vid];
    f.corner8 = a.hexCorner8 != 0;
    float ex = emin ? FLT_MAX : -FLT_MAX, ey = ex, ez = ex, mabs = 0.0f;
    auto extent = [&](float dxs, float dys, float dzs) {
        const float dx = fabsf(dxs), dy = fabsf(dys), dz = fabsf(dzs);
        ex = emin ? fminf(ex, dx) : fmaxf(ex, dx);
        ey = emin ? fminf(ey, dy) : fmaxf(ey, dy);
        ez = emin ? fminf(ez, dz) : fmaxf(ez, dz);
        mabs = fmaxf(mabs, fmaxf(dx, fmaxf(dy, dz)));
    };
    // the lane's first element keeps its corner offsets in registers for
    // the constants (the positions are read once)
    const bool own0 = lane < f.n;
    float d0[7][3];
    if (own0) {
        const int* h = a.ringVal + (size_t)(r0 + lane) * 7;
#pragma unroll
        for (int t = 0; t < 7; ++t) {
            const int v = h[t];
            d0[t][0] = a.x[v] - f.x0x; d0[t][1] = a.y[v] - f.x0y; d0[t][2] = a.z[v] - f.x0z;
            extent(d0[t][0], d0[t][1], d0[t][2]);
        }
    }
    for (int e = lane + 64; e < f.n; e += 64) {
        const int* h = a.ringVal + (size_t)(r0 + e) * 7;
        for (int t = 0; t < 7; ++t) {
            const int v = h[t];
            extent(a.x[v] - f.x0x, a.y[v] - f.x0y, a.z[v] - f.x0z);
        }
    }
    if (emin) { f.ex = wave_min_u(ex); f.ey = wave_min_u(ey); f.ez = wave_min_u(ez); }
    else { f.ex = wave_max_u(ex); f.ey = wave_max_u(ey); f.ez = wave_max_u(ez); }
    f.sg = pow2_scale(wave_max_u(mabs));
    const float s2 = f.sg * f.sg, s3 = s2 * f.sg;
    f.epsD = kHexEps * s3; f.epsF = kHexEps * s2;
    if (own0) {
        f3 r[8];
        r[0] = { 0.0f, 0.0f, 0.0f };
#pragma unroll
        for (int t = 0; t < 7; ++t) r[t + 1] = { d0[t][0] * f.sg, d0[t][1] * f.sg, d0[t][2] * f.sg };
        HexLds L;
        hex_consts(r, L.cd, L.cF, L.hp);
        s_hx[lane] = L;
    }
    for (int e = lane + 64; e < f.n; e += 64) {
        const int* h = a.ringVal + (size_t)(r0 + e) * 7;
        f3 r[8];
        r[0] = { 0.0f, 0.0f, 0.0f };
        for (int t = 0; t < 7; ++t) {
            int v = h[t];
            r[t + 1] = { (a.x[v] - f.x0x) * f.sg, (a.y[v] - f.x0y) * f.sg, (a.z[v] - f.x0z) * f.sg };
        }
        HexLds L;
        hex_consts(r, L.cd, L.cF, L.hp);
        s_hx[e] = L;
    }
    wave_lds_fence();
    f.acc0 = hex_acc0();
    f.inRange = hex_free_lanes(s_hx, f.n, f.acc0);
    return f;
}

// Whether the vertex cannot move: when the sub-tets it is not part of
// already score 0 (a determinant below epsD or a Frobenius term below epsF),
// every candidate's accumulator starts from acc0 and takes fminf of those
// minima, so every candidate -- the start included -- scores exactly 0 and
// none is strictly better than the start.  The search is skipped; the result
// is the full search's.
__device__ __forceinline__ bool hex_pinned(const HexFrame& f)
{
    return f.acc0.dmin < f.epsD || f.acc0.fmin < f.epsF;
}

// What a level can say about one p-dependent sub-tet over its whole window (a
// box of half-widths H around c, frame coordinates): with |J|^2 = alpha (|p -
// g|^2 + kn), bounds of det / F^1.5 from above (ub) and below (lb) for every
// candidate, and whether det and F of every candidate stay clear of the
// metric's thresholds (clear) and of the selection's (sel).  The margins cover
// the rounding of the candidates' canonical evaluation: md, mf bound its
// absolute error (2^-18 of the sum of the terms' magnitudes, against a few
// 2^-24).
struct HexBound { float ub, lb; bool clear, sel; };
__device__ __forceinline__ HexBound hex_bound(const HexP& h, bool a3, float cx, float cy, float cz, float Hx, float Hy,
                                              float Hz, float epsD, float epsF)
{
    constexpr float kR = 0x1p-18f;
    const float ia = a3 ? 1.0f / 3.0f : 1.0f, al = a3 ? 3.0f : 1.0f;
    const float iy = a3 ? 0.19245009f : 1.0f;   // alpha^-1.5
    const float gx = -0.5f * ia * h.sx, gy = -0.5f * ia * h.sy, gz = -0.5f * ia * h.sz;
    const float Px = fabsf(cx) + Hx, Py = fabsf(cy) + Hy, Pz = fabsf(cz) + Hz;
    const float kn = ia * h.K - fmaf(gx, gx, fmaf(gy, gy, gz * gz));
    const float mf = kR * (ia * h.K + fmaf(Px, Px + 2.0f * fabsf(gx), fmaf(Py, Py + 2.0f * fabsf(gy), Pz * (Pz + 2.0f * fabsf(gz)))));
    const float wx = fabsf(cx - gx), wy = fabsf(cy - gy), wz = fabsf(cz - gz);
    const float lx = fmaxf(wx - Hx, 0.0f), ly = fmaxf(wy - Hy, 0.0f), lz = fmaxf(wz - Hz, 0.0f);
    const float ux = wx + Hx, uy = wy + Hy, uz = wz + Hz;
    const float Fl = (kn - mf) + fmaf(lx, lx, fmaf(ly, ly, lz * lz));
    const float Fu = (kn + mf) + fmaf(ux, ux, fmaf(uy, uy, uz * uz));
    const float nx = fabsf(h.gx), ny = fabsf(h.gy), nz = fabsf(h.gz);
    const float dc = fmaf(h.gx, cx, fmaf(h.gy, cy, fmaf(h.gz, cz, h.D)));
    const float A = fmaf(nx, Hx, fmaf(ny, Hy, nz * Hz));
    const float md = kR * (fabsf(h.D) + fmaf(nx, Px, fmaf(ny, Py, nz * Pz)));
    const float dhi = (dc + A) + md, dlo = (dc - A) - md;
    const float ru = __builtin_amdgcn_rsqf(Fl), rl = __builtin_amdgcn_rsqf(Fu);
    HexBound b;
    b.ub = ((dhi * ru) * (ru * ru)) * iy;   // NaN where Fl <= 0: no bound
    b.lb = ((dlo * rl) * (rl * rl)) * iy;
    b.sel = al * Fl >= kSelF;
    b.clear = dlo >= 1.001f * epsD && al * Fl >= 1.001f * epsF;
    return b;
}

// the selection of hex_acc_add
__device__ __forceinline__ void hex_select(HexAcc& a, float det, float F)
{
    const float d2 = det * det, F3 = (F * F) * F;
    const bool take = d2 * a.bF3 < a.bd2 * F3;
    a.bd2 = take ? d2 : a.bd2;
    a.bF3 = take ? F3 : a.bF3;
}

// A p-dependent sub-tet on a line of candidates along x (y, z fixed): det and F
// of candidate px.  Al: alpha, 1 or 3, as a type (known to the compiler) or a float;
// alpha * x is exact for 1 and rounds as 3 x for 3.
template <class Al>
struct HexLine {
    const HexP& h;
    Al al;
    float T, R;
    __device__ __forceinline__ HexLine(const HexP& hp, Al alpha, float py, float pz, float Q1) : h(hp), al(alpha)
    {
        T = fmaf(h.gy, py, fmaf(h.gz, pz, h.D));
        R = fmaf(h.sy, py, fmaf(h.sz, pz, h.K + al * Q1));
    }
    __device__ __forceinline__ float det(float px) const { return fmaf(h.gx, px, T); }
    __device__ __forceinline__ float F(float px) const { return fmaf(px, al * px + h.sx, R); }
};
struct Alpha1 { __device__ __forceinline__ float operator*(float x) const { return x; } };
struct Alpha3 { __device__ __forceinline__ float operator*(float x) const { return 3.0f * x; } };

// one sub-tet, or two in their order, added to the accumulators of the CPL
// candidates px[i] of a lane
template <int CPL, class Al>
__device__ __forceinline__ void hex_add(HexAcc* acc, const HexP& h, Al al, const float* px, float py, float pz, float Q1)
{
    const HexLine<Al> l(h, al, py, pz, Q1);
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
        const float det = l.det(px[i]), F = l.F(px[i]);
        hex_select(acc[i], det, F);
        min_into(acc[i].dmin, det);
        min_into(acc[i].fmin, F);
    }
}
template <int CPL, class Aa, class Ab>
__device__ __forceinline__ void hex_add2(HexAcc* acc, const HexP& ha, Aa aa, const HexP& hb, Ab ab, const float* px,
                                         float py, float pz, float Q1)
{
    const HexLine<Aa> la(ha, aa, py, pz, Q1);
    const HexLine<Ab> lb(hb, ab, py, pz, Q1);
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
        const float da = la.det(px[i]), Fa = la.F(px[i]), db = lb.det(px[i]), Fb = lb.F(px[i]);
        hex_select(acc[i], da, Fa);
        hex_select(acc[i], db, Fb);
        min_into(acc[i].dmin, da, db);
        min_into(acc[i].fmin, Fa, Fb);
    }
}

// all sub-tets of the ring, in its order
template <int CPL>
__device__ __forceinline__ void hex_add_ring(HexAcc* acc, const HexLds* hx, int n, bool corner8, const float* px, float py,
                                             float pz, float Q1)
{
#pragma unroll 1
    for (int e = 0; e < n; ++e) {
        const HexP* hp = hx[e].hp;
        hex_add2<CPL>(acc, hp[0], Alpha1{}, hp[1], Alpha3{}, px, py, pz, Q1);
        hex_add2<CPL>(acc, hp[2], Alpha1{}, hp[3], Alpha1{}, px, py, pz, Q1);
        if (!corner8) hex_add<CPL>(acc, hp[4], Alpha3{}, px, py, pz, Q1);
    }
}

// The nested grid search of a hex vertex, one wave: lane l = j + nq*k owns the
// candidates (i, j, k), i = 0..nq-1 (index i + nq*l; the lowest index wins).
//
// Every level first bounds each sub-tet over its whole window, one sub-tet
// per lane.  U, the smallest upper bound (the p-free sub-tets' minimum
// included), bounds every candidate's minimum; a sub-tet whose lower bound is
// clearly above U, and whose det and F are clear of the thresholds, is never
// the one a candidate's selection ends with, so the candidates are scored over
// the others alone, in ring order: the same bits.  On 48^3 cubes 0.5-3 of the
// 40 sub-tets are left (the windows are scaled by the smallest one-ring offset
// and the p-free sub-tets cap the minimum).  With none left every candidate
// scores exactly the cap, and with U clearly below the current score none is
// better: the level is decided without scoring.  Where the bounds as a whole
// are out of range (a sub-tet may be inverted or flat in the window), the p-free
// minimum alone still rules out the sub-tets that are clearly above it: every
// candidate's selection starts from it.  Rings whose p-free sub-tets are out of
// range score every sub-tet.
//
// Bound by VALU issue: 15,000 -> 2,300 VALU operations per vertex, 214 -> 50 us
// per class of the 48^3 cube (13.8k vertices); about half of it is the staging
// of the ring, 8 of 64 lanes wide.
template <int NQ>
__device__ void hex_vertex(const SearchArgs& a, int vid, bool emin, HexLds* s_hx, int* s_act)
{
    const int lane = (int)(threadIdx.x & 63);
    const HexFrame f = hex_stage(a, vid, emin, s_hx);
    if (hex_pinned(f)) return;   // uniform: every lane holds the same frame
    const int ns = f.corner8 ? 4 : 5, nSub = ns * f.n;
    float qcur = hex_start_lanes(s_hx, f.n, f.corner8, f.acc0, f.inRange, f.epsD, f.epsF);
    const float S0 = hex_acc_score(f.acc0, f.epsD, f.epsF);   // the score of a candidate that selects none
    // the cap's det / F^1.5
    const float capY = f.inRange ? __builtin_amdgcn_sqrtf(f.acc0.bd2 * __builtin_amdgcn_rcpf(f.acc0.bF3)) : FLT_MAX;
    float cx = f.x0x, cy = f.x0y, cz = f.x0z, ds = a.gridScale;
    const int j = lane % NQ, k = lane / NQ;
    const bool active = lane < NQ * NQ;
    bool moved = false;
    for (int d = 0; d < a.depth; ++d, ds = ds * a.shrink) {
        const float gxM = cx + ds * f.ex, gxm = cx - ds * f.ex;
        const float gyM = cy + ds * f.ey, gym = cy - ds * f.ey;
        const float gzM = cz + ds * f.ez, gzm = cz - ds * f.ez;
        // window box in frame coordinates, widened by the rounding of the
        // candidates' world coordinates
        const float wx = (cx - f.x0x) * f.sg, wy = (cy - f.x0y) * f.sg, wz = (cz - f.x0z) * f.sg;
        const float Hx = 1.001f * (ds * f.ex) * f.sg + 0x1p-20f * (fabsf(cx) + ds * f.ex) * f.sg;
        const float Hy = 1.001f * (ds * f.ey) * f.sg + 0x1p-20f * (fabsf(cy) + ds * f.ey) * f.sg;
        const float Hz = 1.001f * (ds * f.ez) * f.sg + 0x1p-20f * (fabsf(cz) + ds * f.ez) * f.sg;
        auto bound = [&](int t) {
            const int e = sub_elem(t, f.corner8), s = t - e * ns;
            return hex_bound(s_hx[e].hp[s], s == 1 || s == 4, wx, wy, wz, Hx, Hy, Hz, f.epsD, f.epsF);
        };
        float u = FLT_MAX;
        bool sel = true;
        HexBound b0{ FLT_MAX, FLT_MAX, true, true };
        for (int t = lane; t < nSub; t += 64) {
            const HexBound b = bound(t);
            if (t == lane) b0 = b;
            u = fminf(u, b.ub);
            sel = sel && b.sel;
        }
        const float U = fminf(wave_min_u(u), capY);
        if (U < 0.0f) continue;   // a determinant below 0 all over the window: every candidate scores 0
        const bool fast = f.inRange && __ballot(!sel) == 0ull && U >= kSelY;
        const float tq = qcur * (1.0f / 3.0f), yq = tq * __builtin_amdgcn_sqrtf(tq);   // qcur's det / F^1.5
        if (fast && U * (1.0f + kSel) < yq * (1.0f - kSel)) continue;   // no candidate reaches qcur
        const float lim0 = (fast ? U : capY) * (1.0f + 2.0f * kSel);
        const bool drops = fast || (f.inRange && capY >= kSelY);
        int nAct = 0;
        for (int t0 = 0; t0 < nSub; t0 += 64) {
            const int t = t0 + lane;
            const int e = sub_elem(t, f.corner8), s = t - e * ns;
            bool keep = t < nSub;
            if (keep && drops) {
                const HexBound b = t0 == 0 ? b0 : bound(t);
                keep = !(b.clear && b.sel && b.lb * (1.0f - kSel) > lim0);
            }
            const unsigned long long bal = __ballot(keep);
            if (keep)
                s_act[nAct + __popcll(bal & ((1ull << lane) - 1ull))] = (e << 4) | (s << 1) | (s == 1 || s == 4 ? 1 : 0);
            nAct += __popcll(bal);
        }
        if (nAct == 0) {   // every candidate scores S0: the first one, if that is better
            if (qcur < S0) {
                cx = grid_coord(a.aff, 0, NQ, gxm, gxM);
                cy = grid_coord(a.aff, 0, NQ, gym, gyM);
                cz = grid_coord(a.aff, 0, NQ, gzm, gzM);
                qcur = S0;
                moved = true;
            }
            continue;
        }
        wave_lds_fence();
        const float py = (grid_coord(a.aff, j, NQ, gym, gyM) - f.x0y) * f.sg;
        const float pz = (grid_coord(a.aff, k, NQ, gzm, gzM) - f.x0z) * f.sg;
        float px[NQ];
#pragma unroll
        for (int i = 0; i < NQ; ++i) px[i] = (grid_coord(a.aff, i, NQ, gxm, gxM) - f.x0x) * f.sg;
        const float Q1 = fmaf(pz, pz, py * py);
        HexAcc acc[NQ];
#pragma unroll
        for (int i = 0; i < NQ; ++i) acc[i] = f.acc0;
        // Most are left (windows much wider than the ring's smallest offset, regular
        // rings): all of them, straight through the ring, 101 operations per sub-tet for
        // the line's 8 candidates.  Through the list, two at a time, 113.  (One at a time
        // with the code read from LDS it took 153: 40^3 hexes with the largest offset as
        // extent 7.1 ms for 6 iterations, 5.7 so; without jitter 9.4 ms, 6.8 so.  The
        // line at a half makes the former 5.9 ms, at 30 % 6.2.)
        if (4 * nAct > 3 * nSub) {
            hex_add_ring<NQ>(acc, s_hx, f.n, f.corner8, px, py, pz, Q1);
        } else {
            const auto sub = [&](int code) { return s_hx[code >> 4].hp[(code >> 1) & 7]; };
            const auto alpha = [](int code) { return (code & 1) ? 3.0f : 1.0f; };
            for (int q0 = 0; q0 < nAct; q0 += 64) {   // 64 codes at a time on the lanes
                const int m = min(nAct - q0, 64), codes = s_act[q0 + min(lane, m - 1)];
                for (int q = 0; q + 1 < m; q += 2) {
                    const int ca = __builtin_amdgcn_readlane(codes, q), cb = __builtin_amdgcn_readlane(codes, q + 1);
                    const HexP ha = sub(ca), hb = sub(cb);
                    hex_add2<NQ>(acc, ha, alpha(ca), hb, alpha(cb), px, py, pz, Q1);
                }
                if (m & 1) {
                    const int c = __builtin_amdgcn_readlane(codes, m - 1);
                    const HexP h = sub(c);
                    hex_add<NQ>(acc, h, alpha(c), px, py, pz, Q1);
                }
            }
        }
        wave_lds_fence();   // the next level rewrites the list
        // scores: only of candidates whose ratio is within rounding of the
        // best one's (a clearly smaller ratio has a smaller score), and none
        // where the accumulator is still the cap's
        float y[NQ], ym = 0.0f;
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            y[i] = (acc[i].dmin < f.epsD || acc[i].fmin < f.epsF) ? 0.0f : acc[i].bd2 * __builtin_amdgcn_rcpf(acc[i].bF3);
            ym = fmaxf(ym, y[i]);
        }
        const float Y = wave_max_u(active ? ym : 0.0f);
        const bool quick = fast && Y > 1e-30f;   // below, the ratios are not exact enough to rank by
        if (quick && Y < (yq * yq) * (1.0f - 4.0f * kSel)) continue;
        const float lim = Y * (1.0f - kSel);
        float best = -FLT_MAX;
        int bi = 0;
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            const bool in = active && (!quick || y[i] >= lim);
            const bool cap = quick && acc[i].bd2 == f.acc0.bd2 && acc[i].bF3 == f.acc0.bF3;
            float q = S0;
            if (__ballot(in && !cap) != 0ull) {
                const float qe = hex_acc_score(acc[i], f.epsD, f.epsF);
                q = cap ? S0 : qe;
            }
            if (in && q > best) { best = q; bi = i; }
        }
        const float bm = wave_max_u(best);
        if (qcur < bm) {
            const int l = __builtin_ctzll(__ballot(best == bm));
            const int wi = __builtin_amdgcn_readlane(bi, l), wj = l % NQ, wk = l / NQ;
            cx = grid_coord(a.aff, wi, NQ, gxm, gxM);
            cy = grid_coord(a.aff, wj, NQ, gym, gyM);
            cz = grid_coord(a.aff, wk, NQ, gzm, gzM);
            qcur = bm;
            moved = true;
        }
    }
    if (moved && lane == 0) { a.xw[vid] = cx; a.yw[vid] = cy; a.zw[vid] = cz; }
}

// The same search on the 4 waves of a block, every sub-tet scored, for fallback
// lists with the largest offset as extent: lane l = j + nq k of wave w owns the
// candidates (i, j, k), i = w nq / 4 and on.  Those windows leave the bounds little
// to drop, and a short list waits for its slowest wave (24^3 cube, immediate
// fallback, mode 1, 8 iterations: 9.7 ms with a wave per vertex, 5.9 so).  lds:
// hex_wide_lds bytes.
__host__ __device__ constexpr size_t hex_wide_lds(int ringCap)
{
    return sizeof(HexLds) * (size_t)ringCap + 8 * sizeof(TetBest) + sizeof(HexFrame);
}
static_assert(hex_wide_lds(1) <= 4 * hex_wave_lds(1) && hex_wide_lds(kMaxRingHex) <= 64 * 1024,
              "fits the four waves' slices of a block, and a block of its own");
template <int NQ>
__device__ void hex_vertex_wide(const SearchArgs& a, int vid, unsigned char* lds, int ringCap)
{
    constexpr int W = 4, CPL = NQ / W;
    static_assert(NQ % W == 0 && NQ * NQ <= 64, "nq 4 or 8");
    const int lane = (int)(threadIdx.x & 63), wave = uniform((int)(threadIdx.x >> 6));
    HexLds* s_hx = reinterpret_cast<HexLds*>(lds);
    TetBest* s_best = reinterpret_cast<TetBest*>(s_hx + ringCap);   // [level parity][wave]
    HexFrame* s_f = reinterpret_cast<HexFrame*>(s_best + 2 * W);
    if (wave == 0) {
        const HexFrame own = hex_stage(a, vid, a.extentMin != 0, s_hx);
        if (lane == 0) *s_f = own;
    }
    __syncthreads();
    const HexFrame f = *s_f;
    float cx = f.x0x, cy = f.x0y, cz = f.x0z, ds = a.gridScale;
    bool moved = false;
    if (!hex_pinned(f)) {   // uniform over the block
        float qcur = hex_start_lanes(s_hx, f.n, f.corner8, f.acc0, f.inRange, f.epsD, f.epsF);
        const int j = lane % NQ, k = lane / NQ;
        for (int d = 0; d < a.depth; ++d, ds = ds * a.shrink) {
            const float gxM = cx + ds * f.ex, gxm = cx - ds * f.ex;
            const float gyM = cy + ds * f.ey, gym = cy - ds * f.ey;
            const float gzM = cz + ds * f.ez, gzm = cz - ds * f.ez;
            const float py = (grid_coord(a.aff, j, NQ, gym, gyM) - f.x0y) * f.sg;
            const float pz = (grid_coord(a.aff, k, NQ, gzm, gzM) - f.x0z) * f.sg;
            const float Q1 = fmaf(pz, pz, py * py);
            float px[CPL];
            HexAcc acc[CPL];
#pragma unroll
            for (int i = 0; i < CPL; ++i) {
                px[i] = (grid_coord(a.aff, wave * CPL + i, NQ, gxm, gxM) - f.x0x) * f.sg;
                acc[i] = f.acc0;
            }
            hex_add_ring<CPL>(acc, s_hx, f.n, f.corner8, px, py, pz, Q1);
            float own = -FLT_MAX;
            int bi = 0;
#pragma unroll
            for (int i = 0; i < CPL; ++i) {
                const float q = hex_acc_score(acc[i], f.epsD, f.epsF);
                if (lane < NQ * NQ && q > own) { own = q; bi = i; }
            }
            const float m = wave_max_u(own);
            const int l = __builtin_ctzll(__ballot(own == m));
            if (lane == l) s_best[(d & 1) * W + wave] = { m, wave * CPL + bi + NQ * l };
            __syncthreads();   // one a level: the next one's values go to the other half
            float best = -FLT_MAX;
            int cand = 0;
#pragma unroll
            for (int w = 0; w < W; ++w) {
                const TetBest b = s_best[(d & 1) * W + w];
                if (b.q > best || (b.q == best && b.cand < cand)) { best = b.q; cand = b.cand; }
            }
            if (qcur < best) {
                cx = grid_coord(a.aff, cand % NQ, NQ, gxm, gxM);
                cy = grid_coord(a.aff, (cand / NQ) % NQ, NQ, gym, gyM);
                cz = grid_coord(a.aff, cand / (NQ * NQ), NQ, gzm, gzM);
                qcur = best;
                moved = true;
            }
        }
    }
    if (moved && threadIdx.x == 0) { a.xw[vid] = cx; a.yw[vid] = cy; a.zw[vid] = cz; }
    __syncthreads();   // the next vertex restages the ring
}

// ------------------------------------------------------------- flat tris
// Lane l of wave 0 holds the reference thread t = l/2's candidate B (l even)
// or A (l odd): A = (t/nq, t%nq), B = (t/nq + nq/2, t%nq).  The lowest lane
// among the maxima is the reference's winner (lowest thread; B on an exact
// tie).
template <int NQ>
__device__ void flat_vertex(const SearchArgs& a, int vid, TriC* s_tr)
{
    const int tid = (int)(threadIdx.x & 63);
    const int h0 = uniform(a.heRow[vid]);
    const int n = uniform(a.heRow[vid + 1]) - h0;
    const float x0x = a.x[vid], x0y = a.y[vid];

    float ex = -FLT_MAX, ey = -FLT_MAX, mabs = 0.0f;
    for (int e = tid; e < n; e += 64) {
        int v = a.heTarget[h0 + e];
        float dx = fabsf(a.x[v] - x0x), dy = fabsf(a.y[v] - x0y);
        ex = fmaxf(ex, dx);
        ey = fmaxf(ey, dy);
        mabs = fmaxf(mabs, fmaxf(dx, dy));
    }
    ex = wave_max_u(ex);
    ey = wave_max_u(ey);
    const float sg = pow2_scale(wave_max_u(mabs));
    const float isg = 1.0f / sg;
    const float is2 = (1.0f * isg) * isg;
    for (int e = tid; e < n; e += 64) {
        int va = a.heTarget[h0 + e];
        int vb = a.heTarget[h0 + (e + 1 == n ? 0 : e + 1)];
        s_tr[e] = tri_consts((a.x[va] - x0x) * sg, (a.y[va] - x0y) * sg, (a.x[vb] - x0x) * sg, (a.y[vb] - x0y) * sg);
    }
    wave_lds_fence();

    auto score = [&](float px, float py) {
        const float Q2 = 2.0f * (py * py);
        const float t2 = 2.0f * px;
        TriAcc acc = tri_acc0();
        for (int e = 0; e < n; ++e) {
            const TriC c = s_tr[e];
            float Ty = fmaf(c.gy, py, c.C);
            float Ry = fmaf(c.sy, py, c.K + Q2);
            tri_acc_add(acc, fmaf(c.gx, px, Ty), fmaf(px, t2 + c.sx, Ry));
        }
        return tri_acc_score(acc, is2);
    };

    float qcur = score(0.0f, 0.0f);
    const float qold = qcur;
    const int t = tid >> 1;
    const bool isA = (tid & 1) != 0;
    const int ci = t / NQ + (isA ? 0 : NQ / 2), cj = t % NQ;
    const bool active = t < NQ * NQ / 2;
    float cx = x0x, cy = x0y;
    float ds = a.gridScale;
    float qlast = -FLT_MAX;
    for (int d = 0; d < a.depth; ++d) {
        const float gxM = cx + ds * ex, gxm = cx - ds * ex;
        const float gyM = cy + ds * ey, gym = cy - ds * ey;
        const float q = active ? score((grid_coord(a.aff, ci, NQ, gxm, gxM) - x0x) * sg,
                                       (grid_coord(a.aff, cj, NQ, gym, gyM) - x0y) * sg)
                               : -FLT_MAX;
        const float best = wave_max_u(q);
        if (qcur < best) {
            const int wl = __builtin_ctzll(__ballot(q == best));
            const int wt = wl >> 1;
            const int wi = wt / NQ + ((wl & 1) ? 0 : NQ / 2), wj = wt % NQ;
            cx = grid_coord(a.aff, wi, NQ, gxm, gxM);
            cy = grid_coord(a.aff, wj, NQ, gym, gyM);
            qcur = best;
        }
        qlast = best;
        ds = ds * a.shrink;
    }
    if (qold < qlast && tid == 0) { a.xw[vid] = cx; a.yw[vid] = cy; }
}

// one vertex per wave and block, vertices [cStart, cEnd) of one colour class.
// The tet search asks for 6 waves per SIMD (80 VGPRs, 2 of them spilled outside the
// loops): 40^3 cube, 20 iterations, 6.15 ms; reading the spilled quadric back from
// LDS instead 6.28.  Before the levels that score every candidate 6.53 ms (no
// spill) against 6.64 at 5, 6.66 at 7 and 6.84 at 8 waves
#ifndef VSDMO_TET_MIN_WAVES
#define VSDMO_TET_MIN_WAVES 6
#endif
template <int NQ>
__global__ __launch_bounds__(64, VSDMO_TET_MIN_WAVES) void k_search_tet(SearchArgs a, int ringCap)
{
    extern __shared__ __align__(16) unsigned char s_tcv[];
    tet_vertex<NQ>(a, a.cStart + blockIdx.x, a.extentMin != 0, s_tcv, ringCap);
}
template <int NQ>
__global__ __launch_bounds__(256) void k_search_tet_wide(SearchArgs a, int ringCap)
{
    extern __shared__ __align__(16) unsigned char s_twv[];
    tet_vertex_wide<NQ>(a, a.cStart + blockIdx.x, s_twv, ringCap);
}
// the hex search asks for 4 waves per SIMD (128 VGPRs, no spill): 48^3 cube,
// 10 iterations, 5.1 ms against 5.5 ms at 3 (129 VGPRs) and 5.1-5.2 ms at 5
// and 6 (spills); 31^3 with the surface free 4.9, 4.8, 5.3 and 5.3 ms
#ifndef VSDMO_HEX_MIN_WAVES
#define VSDMO_HEX_MIN_WAVES 4
#endif
template <int NQ>
__global__ __launch_bounds__(64, VSDMO_HEX_MIN_WAVES) void k_search_hex(SearchArgs a, int ringCap)
{
    extern __shared__ __align__(16) unsigned char s_hxv[];
    hex_vertex<NQ>(a, a.cStart + blockIdx.x, a.extentMin != 0, reinterpret_cast<HexLds*>(s_hxv),
                   hex_act(s_hxv, ringCap));
}
template <int NQ>
__global__ __launch_bounds__(64) void k_search_flat(SearchArgs a)
{
    extern __shared__ TriC s_tr[];
    flat_vertex<NQ>(a, a.cStart + blockIdx.x, s_tr);
}

KernelEvents*& kernel_events()
{
    static thread_local KernelEvents* slot = nullptr;
    return slot;
}

__global__ void k_fill_int(int* __restrict__ p, int n, int v)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// ------------------------------------------------------ learned proposal
// Vertex i of the colour class gets the proposal c = v + L_i * Y_i (network
// output in units of its mean edge length L_i; mode 2: c = v).  A 4x4x4 grid
// (candidate index i + 4j + 16k, lowest wins ties) is searched around c on a
// window `frac` times the plain first-level window, for `depthL` levels with
// the window shrunk by 2/3 per level; the centre moves to a level's best
// candidate when it is strictly better than the best quality so far, which
// starts at q(v).  Fallback rule: when the window's best candidate is lower
// than q(v), the vertex goes on the class's fallback list.  Its plain full
// search runs in a second launch before the next class (immediate policy:
// the update is the plain path's, bit for bit) or in the class's next pass,
// beside that pass's windows (deferred policy: the vertex keeps its position
// until then).  A tie at a positive quality (a level's best equals q(v) > 0) leaves
// the vertex where it is: it is the mark of a ring whose minimum is held by
// sub-tets the vertex is not part of (hexes), which no position raises.  At
// quality 0 a tie can also be the vertex's own inverted sub-tet, which the
// full window may still repair: such vertices fall back, unless hex_pinned.
struct LearnArgs {
    const float* Y;
    const float* L;
    int mode;
    int depthL;
    float frac;
    int* fallbacks;   // running total (the list launch adds the class's count)
    int* list;        // this class's fallback vertices (appended)
    int* cnt;         // their number (zero before the class)
    // network run inside the window kernel (mode 1, one 16-vertex tile per
    // block): bf16 / fp32 packed parameters and the neighbour table
    const uint16_t* wb;
    const float* w;
    const int* nbr;
    // deferred fallback (epoch non-null): the vertices appended to list in
    // iteration `it` take the full search in the class's next pass, from
    // listIn / cntIn (the previous iteration's list); epoch[vid] = the
    // iteration that deferred vid, whose window the next pass skips
    const int* listIn;
    const int* cntIn;
    int* epoch;
    int it;
    // class positions -> vertex ids through a work-item list (a batch round:
    // id in the low 30 bits); null: the class is the range a.cStart + position
    const int* items;
    // deferred fallback with the iteration in device memory (a replayed
    // graph): it = *itDev; list / cnt are the parity-0 buffers of the class,
    // parity p at + p * listStride / cntStride; this iteration appends to
    // parity it & 1 and reads the previous iteration's from the other
    const int* itDev;
    int listStride, cntStride;
    // FUSED: the ring corners' positions in the neighbour table (LearnNet.loc)
    const uint8_t* loc;
};

// the concrete iteration and list buffers of a deferred pass
__device__ __forceinline__ LearnArgs learn_resolve(const LearnArgs& la)
{
    if (!la.itDev) return la;
    LearnArgs r = la;
    const int it = *la.itDev;
    const size_t p = (size_t)(it & 1), q = p ^ 1;
    r.it = it;
    r.list = la.list + p * la.listStride;
    r.cnt = la.cnt + p * la.cntStride;
    r.listIn = la.list + q * la.listStride;
    r.cntIn = la.cnt + q * la.cntStride;
    return r;
}

// vertex id of class position ci
__device__ __forceinline__ int learned_vertex(const SearchArgs& a, const LearnArgs& la, int ci)
{
    return la.items ? (la.items[a.cStart + ci] & 0x3fffffff) : a.cStart + ci;
}

// The proposal window runs 4 vertices per wave, 16 lanes each: lane s =
// j + 4k of a group owns the candidates (i, j, k), i = 0..3, which share the
// (y, z) part of every ring element, so one LDS read of an element's
// constants serves 4 candidates (one candidate per lane would spend a third
// of the wave's cycles waiting on LDS).
// vertices per wave in the proposal window (1, 2 and 4 measured on 40^3 tet
// and 48^3 hex cubes: 4 is fastest for hexes and within noise of 2 for tets)
constexpr int kLV = 4;
// mode 3's second window, around the vertex itself, is this fraction of the
// first (the vertices whose proposal window fails are close to a converged
// position: on the seed-7 and seed-8 40^3 tet cubes 1/4 cut the fallbacks
// ~9x against a second window of the first's size, 1/6.7 and 1/5 measured
// the same, 1/2 and 1/1 slower; a power of two keeps the scaling exact)
constexpr float kMode3Window = 0.25f;

// over the 16 lanes of the DPP row, in all of them.  The rows of a wave may be
// in different branches, the lanes of one may not.  (Shuffles, an LDS round trip
// for each of 4 steps and each value, made the learned 40^3 tet iterations 2 %
// longer.)
#define VSDMO_ROW_REDUCE(OP)                                       \
    asm("s_nop 1\n\t" OP " %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n\t" \
        "s_nop 1\n\t" OP " %0, %0, %0 row_ror:4 row_mask:0xf bank_mask:0xf\n\t" \
        "s_nop 1\n\t" OP " %0, %0, %0 row_ror:2 row_mask:0xf bank_mask:0xf\n\t" \
        "s_nop 1\n\t" OP " %0, %0, %0 row_ror:1 row_mask:0xf bank_mask:0xf"      \
        : "+v"(v))
__device__ __forceinline__ float row_max(float v)
{
    VSDMO_ROW_REDUCE("v_max_f32_dpp");
    return v;
}
__device__ __forceinline__ float row_min(float v)
{
    VSDMO_ROW_REDUCE("v_min_f32_dpp");
    return v;
}
#undef VSDMO_ROW_REDUCE

// the place in its row of 16 of the first lane that b holds for (some lane's)
__device__ __forceinline__ int row_first(bool b)
{
    const unsigned m = (unsigned)(__ballot(b) >> ((int)(threadIdx.x & 63) & ~15)) & 0xffffu;
    return __builtin_ctz(m | 0x10000u) & 15;
}
// a lane's value of the row, the same lane in all of them
__device__ __forceinline__ int row_lane(int v, int l) { return __shfl(v, l, 16); }

// The flat search of flat_vertex at nq = 8 for 4 vertices per wave.  The 64
// candidate slots of a vertex are the lanes of the one-wave layout (thread
// t = slot / 2 holds B = (t / 8 + 4, t % 8) at even and A = (t / 8, t % 8) at
// odd slots); here they are spread 4 per lane over a group of 16 lanes.  Each
// lane keeps its first best slot and the group argmax takes the larger
// score, then the lower slot: the wave argmax of the one-wave layout, so
// every decision and every result is the same.  The two slots of a thread
// share the (y) part of each element.  vid < 0: an idle group (no writes);
// s_tr: the group's cap TriC entries of LDS.
constexpr int kFlatGroups = 16;   // vertices per 256-thread block

__device__ void flat_group8(const SearchArgs& a, int vid, TriC* s_tr)
{
    constexpr int NQ = 8, G = 16;
    const int s = (int)(threadIdx.x & (G - 1));
    const bool live = vid >= 0;
    const int h0 = live ? a.heRow[vid] : 0;
    const int n = live ? a.heRow[vid + 1] - h0 : 0;
    const float x0x = live ? a.x[vid] : 0.0f, x0y = live ? a.y[vid] : 0.0f;
    float ex = -FLT_MAX, ey = -FLT_MAX, mabs = 0.0f;
    for (int e = s; e < n; e += G) {
        const int v = a.heTarget[h0 + e];
        const float dx = fabsf(a.x[v] - x0x), dy = fabsf(a.y[v] - x0y);
        ex = fmaxf(ex, dx);
        ey = fmaxf(ey, dy);
        mabs = fmaxf(mabs, fmaxf(dx, dy));
    }
    ex = row_max(ex);
    ey = row_max(ey);
    mabs = row_max(mabs);
    const float sg = pow2_scale(mabs);
    const float isg = 1.0f / sg;
    const float is2 = (1.0f * isg) * isg;
    for (int e = s; e < n; e += G) {
        const int va = a.heTarget[h0 + e];
        const int vb = a.heTarget[h0 + (e + 1 == n ? 0 : e + 1)];
        s_tr[e] = tri_consts((a.x[va] - x0x) * sg, (a.y[va] - x0y) * sg, (a.x[vb] - x0x) * sg, (a.y[vb] - x0y) * sg);
    }
    __syncthreads();

    float qcur;
    {
        TriAcc acc = tri_acc0();
        const float px = 0.0f, py = 0.0f, Q2 = 2.0f * (py * py), t2 = 2.0f * px;
        for (int e = 0; e < n; ++e) {
            const TriC c = s_tr[e];
            const float Ty = fmaf(c.gy, py, c.C);
            const float Ry = fmaf(c.sy, py, c.K + Q2);
            tri_acc_add(acc, fmaf(c.gx, px, Ty), fmaf(px, t2 + c.sx, Ry));
        }
        qcur = tri_acc_score(acc, is2);
    }
    const float qold = qcur;
    // slots 4s + i: threads t0 = 2s (i = 0 B, 1 A) and t1 = 2s + 1 (i = 2 B, 3 A)
    const int t0 = 2 * s, t1 = 2 * s + 1;
    const int cj[2] = { t0 % NQ, t1 % NQ };
    const int ci[4] = { t0 / NQ + NQ / 2, t0 / NQ, t1 / NQ + NQ / 2, t1 / NQ };
    float cx = x0x, cy = x0y;
    float ds = a.gridScale;
    float qlast = -FLT_MAX;
    for (int d = 0; d < a.depth; ++d) {
        const float gxM = cx + ds * ex, gxm = cx - ds * ex;
        const float gyM = cy + ds * ey, gym = cy - ds * ey;
        float py[2], Q2[2], px[4], t2[4];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            py[j] = (grid_coord(a.aff, cj[j], NQ, gym, gyM) - x0y) * sg;
            Q2[j] = 2.0f * (py[j] * py[j]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            px[i] = (grid_coord(a.aff, ci[i], NQ, gxm, gxM) - x0x) * sg;
            t2[i] = 2.0f * px[i];
        }
        TriAcc acc[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = tri_acc0();
        for (int e = 0; e < n; ++e) {
            const TriC c = s_tr[e];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float Ty = fmaf(c.gy, py[j], c.C);
                const float Ry = fmaf(c.sy, py[j], c.K + Q2[j]);
#pragma unroll
                for (int i = 2 * j; i < 2 * j + 2; ++i)
                    tri_acc_add(acc[i], fmaf(c.gx, px[i], Ty), fmaf(px[i], t2[i] + c.sx, Ry));
            }
        }
        float best = -FLT_MAX;
        int bi = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float q = tri_acc_score(acc[i], is2);
            if (q > best) { best = q; bi = i; }
        }
        const float own = best;
        best = row_max(own);
        const int l = row_first(own == best), wl = 4 * l + row_lane(bi, l);
        if (qcur < best) {
            const int wt = wl >> 1;
            const int wi = wt / NQ + ((wl & 1) ? 0 : NQ / 2), wj = wt % NQ;
            cx = grid_coord(a.aff, wi, NQ, gxm, gxM);
            cy = grid_coord(a.aff, wj, NQ, gym, gyM);
            qcur = best;
        }
        qlast = best;
        ds = ds * a.shrink;
    }
    if (live && qold < qlast && s == 0) { a.xw[vid] = cx; a.yw[vid] = cy; }
}

// 16 vertices of the class per 256-thread block; cap TriC per group
__global__ __launch_bounds__(256) void k_search_flat8x4(SearchArgs a, int cap)
{
    extern __shared__ TriC s_trg[];
    const int g = (int)(threadIdx.x >> 4);
    const int i = (int)blockIdx.x * kFlatGroups + g;
    const int vid = (a.cStart + i < a.cEnd) ? a.cStart + i : -1;
    flat_group8(a, vid, s_trg + (size_t)g * cap);
}

// the flat triangle items [lo, hi) of a batch round, 16 per block
__global__ __launch_bounds__(256) void k_batch_flat8x4(SearchArgs a, const int* __restrict__ items, int lo, int hi,
                                                      int cap)
{
    extern __shared__ TriC s_trb[];
    const int g = (int)(threadIdx.x >> 4);
    const int i = lo + (int)blockIdx.x * kFlatGroups + g;
    const int vid = (i < hi) ? (items[i] & 0x3fffffff) : -1;
    flat_group8(a, vid, s_trb + (size_t)g * cap);
}

// whether the 4-per-wave flat search runs: nq 8, the block's fans fit 64 KB
// of LDS, and at least kFlat4MinVertices vertices (256 blocks: a smaller
// launch spreads over more CUs with one vertex per wave; measured on the 64^2
// grid's ~960-vertex classes, 0.112 against 0.123 ms per iteration)
constexpr int kFlat4MinVertices = 256 * kFlatGroups;
static bool flat8x4_ok(int nq, int ringCap, int nVertices)
{
    return nq == 8 && kFlatGroups * sizeof(TriC) * (size_t)ringCap <= 65536 && nVertices >= kFlat4MinVertices;
}


// proposal displacement of the group's vertex (class position ci, at (vx,
// vy, vz)): c = v + l * y.  FUSED: the block's 16 vertices (class positions
// ci0 + 0..15, group gb = threadIdx.x / 16) are one tile of the network, run
// here in the LDS lds (free again on return) from the inputs the caller
// gathered (ng: the row's table neighbours, nw: the wave's weights);
// otherwise l, y come from the separate inference launch's L, Y (mode 1) or
// are zero (mode 2).
template <bool FUSED>
__device__ __forceinline__ void learned_offset(const SearchArgs& a, const LearnArgs& la, int ci0, int gb, int ci,
                                               float vx, float vy, float vz, const MlpGather& ng, const MlpW& nw,
                                               unsigned char* lds, float* relOut, float& l, float& y0, float& y1,
                                               float& y2)
{
    l = 0.0f; y0 = 0.0f; y1 = 0.0f; y2 = 0.0f;
    if constexpr (FUSED) {
        MlpLds& sm = *reinterpret_cast<MlpLds*>(lds);
        const bool live = ci0 + gb < a.cEnd - a.cStart;
        mlp_features16_from(ng, vx, vy, vz, live, sm, relOut);
        mlp_layers16_w(nw, la.wb, la.w, sm);
        l = sm.L[gb]; y0 = sm.Y[gb][0]; y1 = sm.Y[gb][1]; y2 = sm.Y[gb][2];
        __syncthreads();   // the ring staging reuses the LDS
    } else if (learn_uses_net(la.mode)) {
        l = la.L[ci]; y0 = la.Y[3 * ci]; y1 = la.Y[3 * ci + 1]; y2 = la.Y[3 * ci + 2];
    }
    (void)ci; (void)vx; (void)vy; (void)vz; (void)ng; (void)nw; (void)relOut;
}

// LDS of a FUSED window block: the network's LDS, reused for the 16 rings,
// then (at learned_rel_offset) the 16 rows of table-neighbour positions
// relative to their vertex, which the ring staging reads
__host__ __device__ constexpr size_t learned_rel_offset(size_t per, int ringCap)
{
    return ((sizeof(MlpLds) > (size_t)kMlpRows * ringCap * per ? sizeof(MlpLds) : (size_t)kMlpRows * ringCap * per)
            + 15) / 16 * 16;
}
constexpr size_t kLearnedRelBytes = sizeof(float) * kMlpRows * kNbr * 3;

// append vid to the class's fallback list where need (one lane per group):
// one atomic per wave for the wave's fallbacks (the list order does not
// matter: the class's vertices are independent).  Every lane calls it.  A
// class appends at most its cap = class size vertices (its count starts at
// zero); the bound only guards the list.
__device__ __forceinline__ void fallback_append(const LearnArgs& la, bool need, int vid, int cap)
{
    const unsigned long long bal = __ballot(need);
    if (bal == 0ull) return;
    const int lane = threadIdx.x & 63;
    int base = 0;
    if (lane == 0) base = atomicAdd(la.cnt, __popcll(bal));
    base = __shfl(base, 0);
    const int idx = base + __popcll(bal & ((1ull << lane) - 1ull));
    if (need && idx >= 0 && idx < cap) la.list[idx] = vid;
}

// The window search of the WPB * LV class vertices of block blk: LV
// vertices per wave on WPB waves; with FUSED (WPB = 4, LV = 4) the block
// first runs their 16-vertex network tile.  lds: WPB * LV rings (after the
// network's LDS).
template <int NQ, int LV, int WPB, bool FUSED>
__device__ void tet_window(const SearchArgs& a, const LearnArgs& la, int ringCap, int blk, unsigned char* s_tcl)
{
    constexpr int NL = 4, G = 64 / LV, CPL = NL * NL * NL / G;   // lanes per vertex, candidates per lane
    constexpr int VPB = WPB * LV;
    static_assert(G == 16 && CPL == NL, "a lane group is a DPP row, a lane a line of candidates along x");
    static_assert(!FUSED || VPB == kMlpRows, "one network tile per block");
    const int s = threadIdx.x % G, gb = threadIdx.x / G;
    const int nc = a.cEnd - a.cStart, ci0 = VPB * blk;
    // a group past the end of the class mirrors the class's last vertex and writes nothing
    const int ci = min(ci0 + gb, nc - 1);
    const int vid = learned_vertex(a, la, ci);
    // a vertex deferred by the previous iteration takes the full search in this launch instead
    const bool own = ci0 + gb < nc && !(la.epoch && la.epoch[vid] == la.it - 1);
    TetFrame f;
    const int r0 = a.ringRow[vid];
    f.n = a.ringRow[vid + 1] - r0;
    f.x0x = a.x[vid]; f.x0y = a.y[vid]; f.x0z = a.z[vid];
    // the network's neighbours, the lane's first PRE ring elements and the
    // network's weights are loaded into registers before the network runs
    // (their latencies overlap; no other vertex of this launch moves these
    // positions: ring and table neighbours belong to other colour classes).
    // FUSED: a ring element is its corners' positions in the neighbour table
    // (one 4-byte word), whose positions relative to v the features leave in
    // LDS; otherwise its corner positions.
    MlpGather ng{};
    if constexpr (FUSED) ng = mlp_gather16(a.x, a.y, a.z, la.nbr, vid, ci0 + gb < nc);
    constexpr int PRE = 2;
    uint32_t lw[PRE];
    float rx[PRE][3], ry[PRE][3], rz[PRE][3];
#pragma unroll
    for (int k = 0; k < PRE; ++k) {
        const int e = s + k * G;
        lw[k] = 0xffffffffu;
#pragma unroll
        for (int t = 0; t < 3; ++t) { rx[k][t] = f.x0x; ry[k][t] = f.x0y; rz[k][t] = f.x0z; }
        if (e < f.n) {
            if constexpr (FUSED) {
                lw[k] = *reinterpret_cast<const uint32_t*>(la.loc + (size_t)(r0 + e) * kRingLocStrideTet);
            } else {
#pragma unroll
                for (int t = 0; t < 3; ++t) {
                    const int v = a.ringVal[(size_t)(r0 + e) * 3 + t];
                    rx[k][t] = a.x[v]; ry[k][t] = a.y[v]; rz[k][t] = a.z[v];
                }
            }
        }
    }
    MlpW nw{};
    if constexpr (FUSED) nw = mlp_load_w16(la.wb, la.w);
    float* rel = FUSED ? reinterpret_cast<float*>(s_tcl + learned_rel_offset(sizeof(TetC), ringCap)) : nullptr;
    float pl, py0, py1, py2;
    learned_offset<FUSED>(a, la, ci0, gb, ci, f.x0x, f.x0y, f.x0z, ng, nw, s_tcl, rel, pl, py0, py1, py2);
    const float* relRow = FUSED ? rel + (size_t)gb * kNbr * 3 : nullptr;
    TetC* tc = reinterpret_cast<TetC*>(s_tcl) + (size_t)gb * ringCap;
    // corner t of ring element e relative to v: from the table (w: the
    // element's packed table positions) or, for a corner the table does not
    // hold (or without a table), from the positions
    auto corner = [&](int e, int t, uint32_t w, float& dx, float& dy, float& dz) {
        const uint32_t li = (w >> (8 * t)) & 0xffu;
        if (FUSED && li != kRingLocNone) {
            dx = relRow[3 * li]; dy = relRow[3 * li + 1]; dz = relRow[3 * li + 2];
        } else {
            const int v = a.ringVal[(size_t)(r0 + e) * 3 + t];
            dx = a.x[v] - f.x0x; dy = a.y[v] - f.x0y; dz = a.z[v] - f.x0z;
        }
    };
    auto word = [&](int e) -> uint32_t {
        if constexpr (FUSED) return *reinterpret_cast<const uint32_t*>(la.loc + (size_t)(r0 + e) * kRingLocStrideTet);
        else return 0xffffffffu;
    };
    // window half-extents and frame scale (max / min: the order of the
    // elements does not matter), then the ring constants into LDS
    const bool emin = a.extentMin != 0;
    float ex = emin ? FLT_MAX : -FLT_MAX, ey = ex, ez = ex, mabs = 0.0f;
    auto extent = [&](float dxs, float dys, float dzs) {   // signed offsets from v
        const float dx = fabsf(dxs), dy = fabsf(dys), dz = fabsf(dzs);
        ex = emin ? fminf(ex, dx) : fmaxf(ex, dx);
        ey = emin ? fminf(ey, dy) : fmaxf(ey, dy);
        ez = emin ? fminf(ez, dz) : fmaxf(ez, dz);
        mabs = fmaxf(mabs, fmaxf(dx, fmaxf(dy, dz)));
    };
#pragma unroll
    for (int k = 0; k < PRE; ++k) {
        const int e = s + k * G;
        if (e < f.n) {
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                float dx, dy, dz;
                if constexpr (FUSED) corner(e, t, lw[k], dx, dy, dz);
                else { dx = rx[k][t] - f.x0x; dy = ry[k][t] - f.x0y; dz = rz[k][t] - f.x0z; }
                extent(dx, dy, dz);
            }
        }
    }
    for (int e = s + PRE * G; e < f.n; e += G) {
        const uint32_t w = word(e);
        for (int t = 0; t < 3; ++t) {
            float dx, dy, dz;
            corner(e, t, w, dx, dy, dz);
            extent(dx, dy, dz);
        }
    }
    if (emin) { ex = row_min(ex); ey = row_min(ey); ez = row_min(ez); }
    else { ex = row_max(ex); ey = row_max(ey); ez = row_max(ez); }
    mabs = row_max(mabs);
    f.ex = ex; f.ey = ey; f.ez = ez;
    f.sg = pow2_scale(mabs);
    const float isg = 1.0f / f.sg;
    f.is3 = ((1.0f * isg) * isg) * isg;
#pragma unroll
    for (int k = 0; k < PRE; ++k) {
        const int e = s + k * G;
        if (e < f.n) {
            f3 p[3];
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                float dx, dy, dz;
                if constexpr (FUSED) corner(e, t, lw[k], dx, dy, dz);
                else { dx = rx[k][t] - f.x0x; dy = ry[k][t] - f.x0y; dz = rz[k][t] - f.x0z; }
                p[t] = { dx * f.sg, dy * f.sg, dz * f.sg };
            }
            tc[e] = tet_consts(p[0], p[1], p[2]);
        }
    }
    for (int e = s + PRE * G; e < f.n; e += G) {
        const uint32_t w = word(e);
        f3 p[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            float dx, dy, dz;
            corner(e, t, w, dx, dy, dz);
            p[t] = { dx * f.sg, dy * f.sg, dz * f.sg };
        }
        tc[e] = tet_consts(p[0], p[1], p[2]);
    }
    __syncthreads();

    float cx = f.x0x, cy = f.x0y, cz = f.x0z;
    if (learn_uses_net(la.mode)) { cx = f.x0x + pl * py0; cy = f.x0y + pl * py1; cz = f.x0z + pl * py2; }
    // q0, the start position's score, is accumulated beside the candidates
    // of the first level (at p = 0: det = D, L = K exactly, the terms
    // tet_score adds, in the same ring order)
    float q0 = 0.0f, qbest = 0.0f;
    bool haveQ0 = false;
    bool moved = false, tie = false;
    const float affL = 1.0f / (float)(NL - 1);
    const int lj = s % NL, lk = s / NL;
    // depthL levels of the 4x4x4 window around (cx, cy, cz); the branch
    // conditions are uniform over the vertex's lane group
    auto levels = [&](float scale) {
        float ds = (la.frac * scale) * a.gridScale;
        for (int d = 0; d < la.depthL; ++d) {
            const float gxM = cx + ds * f.ex, gxm = cx - ds * f.ex;
            const float gyM = cy + ds * f.ey, gym = cy - ds * f.ey;
            const float gzM = cz + ds * f.ez, gzm = cz - ds * f.ez;
            const float py = (grid_coord(affL, lj, NL, gym, gyM) - f.x0y) * f.sg;
            const float pz = (grid_coord(affL, lk, NL, gzm, gzM) - f.x0z) * f.sg;
            float px[CPL], t3[CPL];
    #pragma unroll
            for (int i = 0; i < CPL; ++i) {
                px[i] = (grid_coord(affL, i, NL, gxm, gxM) - f.x0x) * f.sg;
                t3[i] = 3.0f * px[i];
            }
            const float Qyz = 3.0f * fmaf(pz, pz, py * py);
            TetAcc acc[CPL];
    #pragma unroll
            for (int i = 0; i < CPL; ++i) acc[i] = tet_acc0();
            // one pass over the ring; the first level run also accumulates q0
            // (later levels and mode 3's window skip it)
            auto ring = [&](auto withQ0) {
                constexpr bool WQ = decltype(withQ0)::value;
                TetAcc acc0 = tet_acc0();
                // two elements per iteration (the minima fold into v_min3)
    #pragma unroll 2
                for (int e = 0; e < f.n; ++e) {
                    const TetC c = tc[e];
                    const float Tyz = fmaf(c.nny, py, fmaf(c.nnz, pz, c.D));
                    const float Ryz = fmaf(c.m2sy, py, fmaf(c.m2sz, pz, c.K + Qyz));
    #pragma unroll
                    for (int i = 0; i < CPL; ++i)
                        tet_acc_add(acc[i], fmaf(c.nnx, px[i], Tyz), fmaf(px[i], t3[i] + c.m2sx, Ryz));
                    if constexpr (WQ) tet_acc_add(acc0, c.D, c.K);
                }
                if constexpr (WQ) { q0 = tet_acc_score(acc0, f.is3); qbest = q0; haveQ0 = true; }
            };
            if (!haveQ0) ring(std::true_type{});
            else ring(std::false_type{});
            float best = -FLT_MAX;
            int bi = 0;
    #pragma unroll
            for (int i = 0; i < CPL; ++i) {
                float q = tet_acc_score(acc[i], f.is3);
                if (q > best) { best = q; bi = i; }
            }
            const float own = best;
            best = row_max(own);
            const int l = row_first(own == best), cand = row_lane(bi, l) + NL * l;
            tie = tie || (best == q0 && q0 > 0.0f);
            if (qbest < best) {
                cx = grid_coord(affL, cand % NL, NL, gxm, gxM);
                cy = grid_coord(affL, (cand / NL) % NL, NL, gym, gyM);
                cz = grid_coord(affL, cand / (NL * NL), NL, gzm, gzM);
                qbest = best;
                moved = true;
            }
            ds = ds * (2.0f / (float)(NL - 1));
        }
    };
    levels(1.0f);
    // mode 3: where the network's window finds nothing better, a window a
    // quarter of its size around the vertex itself before the full search
    if (la.mode == 3 && !moved && !tie) {
        cx = f.x0x; cy = f.x0y; cz = f.x0z;
        levels(kMode3Window);
    }
    if (moved && own && s == 0) { a.xw[vid] = cx; a.yw[vid] = cy; a.zw[vid] = cz; }
    const bool need = !moved && !tie && own && s == 0;
    fallback_append(la, need, vid, nc);
    if (need && la.epoch) la.epoch[vid] = la.it;
}

// As tet_window for hexes, with hex_vertex's bounds in front of every level.
// Every level scored the 40 sub-tets of a regular ring for all 64 candidates;
// with the bounds a few are left (15.2 -> 9.5 M VALU operations per 48^3 class,
// 35.8 -> 29.0 us).  A branch per lane (the sub-tet's alpha, a short circuit)
// costs more here than what it skips: selects as arithmetic, 44 -> 37 us; the
// last waves set the time, hence the early ends for pinned and inverted rings.
// C8: the eight-corner hex metric (a.hexCorner8) as a template argument.
template <int NQ, int LV, int WPB, bool FUSED, bool C8>
__device__ void hex_window(const SearchArgs& a, const LearnArgs& la, int ringCap, int blk, unsigned char* s_hxl)
{
    constexpr int NL = 4, G = 64 / LV, CPL = NL * NL * NL / G;
    constexpr int VPB = WPB * LV;
    static_assert(G == 16 && CPL == NL, "a lane group is a DPP row, a lane a line of candidates along x");
    static_assert(!FUSED || VPB == kMlpRows, "one network tile per block");
    const int s = threadIdx.x % G, gb = threadIdx.x / G;
    const int nc = a.cEnd - a.cStart, ci0 = VPB * blk;
    const int ci = min(ci0 + gb, nc - 1);
    const int vid = learned_vertex(a, la, ci);
    const bool own = ci0 + gb < nc && !(la.epoch && la.epoch[vid] == la.it - 1);
    HexFrame f;
    const int r0 = a.ringRow[vid];
    f.n = a.ringRow[vid + 1] - r0;
    f.x0x = a.x[vid]; f.x0y = a.y[vid]; f.x0z = a.z[vid];
    // the network's inputs (table neighbours, weights) and the packed table
    // positions of the lane's first ring element are loaded before it runs
    MlpGather ng{};
    MlpW nw{};
    uint2 lw0 = make_uint2(0xffffffffu, 0xffffffffu);
    if constexpr (FUSED) {
        ng = mlp_gather16(a.x, a.y, a.z, la.nbr, vid, ci0 + gb < nc);
        if (s < f.n) lw0 = *reinterpret_cast<const uint2*>(la.loc + (size_t)(r0 + s) * kRingLocStrideHex);
        nw = mlp_load_w16(la.wb, la.w);
    }
    float* rel = FUSED ? reinterpret_cast<float*>(s_hxl + learned_rel_offset(sizeof(HexLds), ringCap)) : nullptr;
    float pl, py0, py1, py2;
    learned_offset<FUSED>(a, la, ci0, gb, ci, f.x0x, f.x0y, f.x0z, ng, nw, s_hxl, rel, pl, py0, py1, py2);
    const float* relRow = FUSED ? rel + (size_t)gb * kNbr * 3 : nullptr;
    HexLds* hx = reinterpret_cast<HexLds*>(s_hxl) + (size_t)gb * ringCap;
    // corner t of ring element e relative to v: from the table (w: the
    // element's packed table positions) or, for a corner the table does not
    // hold (or without a table), from the positions
    auto word = [&](int e) -> uint2 {
        if constexpr (FUSED)
            return e == s ? lw0 : *reinterpret_cast<const uint2*>(la.loc + (size_t)(r0 + e) * kRingLocStrideHex);
        else return make_uint2(0xffffffffu, 0xffffffffu);
    };
    auto corner = [&](int e, int t, uint2 w, float& dx, float& dy, float& dz) {
        const uint32_t li = ((t < 4 ? w.x : w.y) >> (8 * (t & 3))) & 0xffu;
        if (FUSED && li != kRingLocNone) {
            dx = relRow[3 * li]; dy = relRow[3 * li + 1]; dz = relRow[3 * li + 2];
        } else {
            const int v = a.ringVal[(size_t)(r0 + e) * 7 + t];
            dx = a.x[v] - f.x0x; dy = a.y[v] - f.x0y; dz = a.z[v] - f.x0z;
        }
    };
    // window half-extents (group_extents's rule) and frame scale
    {
        const bool emin = a.extentMin != 0;
        float ex = emin ? FLT_MAX : -FLT_MAX, ey = ex, ez = ex, mabs = 0.0f;
        for (int e = s; e < f.n; e += G) {
            const uint2 w = word(e);
            for (int t = 0; t < 7; ++t) {
                float dx, dy, dz;
                corner(e, t, w, dx, dy, dz);
                dx = fabsf(dx); dy = fabsf(dy); dz = fabsf(dz);
                ex = emin ? fminf(ex, dx) : fmaxf(ex, dx);
                ey = emin ? fminf(ey, dy) : fmaxf(ey, dy);
                ez = emin ? fminf(ez, dz) : fmaxf(ez, dz);
                mabs = fmaxf(mabs, fmaxf(dx, fmaxf(dy, dz)));
            }
        }
        if (emin) { ex = row_min(ex); ey = row_min(ey); ez = row_min(ez); }
        else { ex = row_max(ex); ey = row_max(ey); ez = row_max(ez); }
        f.ex = ex; f.ey = ey; f.ez = ez;
        f.sg = pow2_scale(row_max(mabs));
    }
    const float s2 = f.sg * f.sg, s3 = s2 * f.sg;
    f.epsD = kHexEps * s3; f.epsF = kHexEps * s2;
    for (int e = s; e < f.n; e += G) {
        const uint2 w = word(e);
        f3 r[8];
        r[0] = { 0.0f, 0.0f, 0.0f };
        for (int t = 0; t < 7; ++t) {
            float dx, dy, dz;
            corner(e, t, w, dx, dy, dz);
            r[t + 1] = { dx * f.sg, dy * f.sg, dz * f.sg };
        }
        HexLds L;
        hex_consts(r, L.cd, L.cF, L.hp);
        hx[e] = L;
    }
    __syncthreads();
    // the selection over the group's pairs pair(0..n-1), continued from acc (as
    // select_lanes, whose conditions are checked here: else in order)
    const int gbase = (int)(threadIdx.x & 63) & ~(G - 1);
    const auto group_bits = [&](bool b) { return (unsigned)(__ballot(b) >> gbase) & 0xffffu; };
    const auto select = [&](HexAcc& acc, bool hasAcc, bool accInRange, int n, auto pair) {
        bool ok = accInRange && n > 0 && n <= 4 * G;
        float y[4], d2[4], F3[4], dm = FLT_MAX, fm = FLT_MAX, ym = FLT_MAX;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            y[q] = FLT_MAX;
            d2[q] = 1.0f;
            F3[q] = 0.0f;   // a place without a pair replaces none
            if (s + q * G < n) {
                const float2 v = pair(s + q * G);
                ok = ok & sel_range(v.x, v.y);
                dm = fminf(dm, v.x);
                fm = fminf(fm, v.y);
                d2[q] = v.x * v.x;
                F3[q] = (v.y * v.y) * v.y;
                y[q] = d2[q] * __builtin_amdgcn_rcpf(F3[q]);
                ym = fminf(ym, y[q]);
            }
        }
        ok = group_bits(!ok) == 0;
        if (n <= 4 * G) {
            acc.dmin = fminf(acc.dmin, row_min(dm));
            acc.fmin = fminf(acc.fmin, row_min(fm));
            if (acc.dmin < f.epsD || acc.fmin < f.epsF) return false;   // scores 0, whatever is selected
        }
        if (!ok) {
            for (int t = 0; t < n; ++t) { const float2 v = pair(t); hex_acc_add(acc, v.x, v.y); }
            return false;
        }
        const float ya = hasAcc ? acc.bd2 * __builtin_amdgcn_rcpf(acc.bF3) : FLT_MAX;
        const float lim = fminf(row_min(ym), ya) * (1.0f + 2.0f * kSel);
        unsigned long long band = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) band |= (unsigned long long)group_bits(y[q] <= lim) << (16 * q);
        if (!(ya <= lim)) { acc.bd2 = 1.0f; acc.bF3 = 0.0f; }   // replaced by the band's first
        if (__popcll(band) <= 4) {   // a few: one after the other
            for (; band; band &= band - 1) {
                const float2 v = pair(__builtin_ctzll(band));
                const float b2 = v.x * v.x, b3 = (v.y * v.y) * v.y;
                const bool take = b2 * acc.bF3 < acc.bd2 * b3;
                acc.bd2 = take ? b2 : acc.bd2;
                acc.bF3 = take ? b3 : acc.bF3;
            }
            return true;
        }
        for (;;) {   // more: on to the first that replaces the selected one, as select_lanes
            unsigned long long m = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) m |= (unsigned long long)group_bits(d2[q] * acc.bF3 < acc.bd2 * F3[q]) << (16 * q);
            m &= band;
            if (m == 0) break;
            const int t = __builtin_ctzll(m);
            const float2 v = pair(t);
            acc.bd2 = v.x * v.x;
            acc.bF3 = (v.y * v.y) * v.y;
            band &= ~((2ull << t) - 1ull);
        }
        return true;
    };
    constexpr int ns = C8 ? 4 : 5;
    const int nSub = ns * f.n;
    const auto sub = [&](int t) -> const HexP& {
        const int e = sub_elem(t, C8);
        return hx[e].hp[t - e * ns];
    };
    const auto alpha3 = [&](int t) { return (0x12 >> (t - sub_elem(t, C8) * ns) & 1) != 0; };   // slots 1 and 4
    f.acc0 = hex_acc0();
    f.inRange = select(f.acc0, false, true, 4 * f.n, [&](int t) { return make_float2(hx[t >> 2].cd[t & 3], hx[t >> 2].cF[t & 3]); });
    // q0: the start position's score (at p = 0: det = D, |J|^2 = K exactly)
    float q0;
    {
        HexAcc acc = f.acc0;
        select(acc, true, f.inRange, nSub, [&](int t) { const HexP& h = sub(t); return make_float2(h.D, h.K); });
        q0 = hex_acc_score(acc, f.epsD, f.epsF);
    }
    const float S0 = hex_acc_score(f.acc0, f.epsD, f.epsF);   // the score of a candidate that selects none
    const float capY = f.inRange ? __builtin_amdgcn_sqrtf(f.acc0.bd2 * __builtin_amdgcn_rcpf(f.acc0.bF3)) : FLT_MAX;
    const bool bounded = f.inRange && nSub <= 4 * G;
    const bool pinned = hex_pinned(f);   // every candidate scores 0

    float cx = f.x0x, cy = f.x0y, cz = f.x0z;
    if (learn_uses_net(la.mode)) { cx = f.x0x + pl * py0; cy = f.x0y + pl * py1; cz = f.x0z + pl * py2; }
    float qbest = q0;
    bool moved = false, tie = false;
    const float affL = 1.0f / (float)(NL - 1);
    const int lj = s % NL, lk = s / NL;
    // depthL levels of the 4x4x4 window around (cx, cy, cz), by the bounds of
    // hex_vertex: up to 4 sub-tets on each lane of the group, and only those
    // that can decide a candidate are scored (per candidate in ring order, the
    // same bits).  The branches are uniform over the vertex's lane group.
    auto levels = [&](float scale) {
        float ds = (la.frac * scale) * a.gridScale;
        for (int d = 0; d < la.depthL && !pinned; ++d, ds = ds * (2.0f / (float)(NL - 1))) {
            const float gxM = cx + ds * f.ex, gxm = cx - ds * f.ex;
            const float gyM = cy + ds * f.ey, gym = cy - ds * f.ey;
            const float gzM = cz + ds * f.ez, gzm = cz - ds * f.ez;
            const float tq = qbest * (1.0f / 3.0f), yq = tq * __builtin_amdgcn_sqrtf(tq);   // qbest's det / F^1.5
            bool fast = false;
            unsigned long long act = ~0ull;
            if (bounded) {
                const float wx = (cx - f.x0x) * f.sg, wy = (cy - f.x0y) * f.sg, wz = (cz - f.x0z) * f.sg;
                const float Hx = 1.001f * (ds * f.ex) * f.sg + 0x1p-20f * (fabsf(cx) + ds * f.ex) * f.sg;
                const float Hy = 1.001f * (ds * f.ey) * f.sg + 0x1p-20f * (fabsf(cy) + ds * f.ey) * f.sg;
                const float Hz = 1.001f * (ds * f.ez) * f.sg + 0x1p-20f * (fabsf(cz) + ds * f.ez) * f.sg;
                float u = FLT_MAX, lb[4];   // lb: -FLT_MAX where the sub-tet has to be scored
                bool sel = true;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    lb[q] = -FLT_MAX;
                    const int t = s + q * G;
                    if (t < nSub) {
                        const HexBound b = hex_bound(sub(t), alpha3(t), wx, wy, wz, Hx, Hy, Hz, f.epsD, f.epsF);
                        u = fminf(u, b.ub);
                        sel = sel & b.sel;
                        lb[q] = b.clear && b.sel ? b.lb : -FLT_MAX;
                    }
                }
                const float U = fminf(row_min(u), capY);
                if (U < 0.0f) continue;   // every candidate scores 0
                fast = group_bits(!sel) == 0 && U >= kSelY;
                if (fast && U * (1.0f + kSel) < yq * (1.0f - kSel)) continue;   // no candidate reaches qbest
                const float lim0 = (fast ? U : capY >= kSelY ? capY : FLT_MAX) * (1.0f + 2.0f * kSel);
                act = 0;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const bool drop = lb[q] * (1.0f - kSel) > lim0;
                    act |= (unsigned long long)group_bits(s + q * G < nSub && !drop) << (16 * q);
                }
            }
            float best = S0;   // with nothing to score every candidate scores S0: the first
            int cand = 0;
            if (act != 0) {
                const float py = (grid_coord(affL, lj, NL, gym, gyM) - f.x0y) * f.sg;
                const float pz = (grid_coord(affL, lk, NL, gzm, gzM) - f.x0z) * f.sg;
                float px[CPL];
#pragma unroll
                for (int i = 0; i < CPL; ++i) px[i] = (grid_coord(affL, i, NL, gxm, gxM) - f.x0x) * f.sg;
                const float Q1 = fmaf(pz, pz, py * py);
                HexAcc acc[CPL];
#pragma unroll
                for (int i = 0; i < CPL; ++i) acc[i] = f.acc0;
                const auto alpha = [&](int t) { return alpha3(t) ? 3.0f : 1.0f; };   // 1 * x is x, to the bit
                const auto add = [&](const HexP h, float al) { hex_add<CPL>(acc, h, al, px, py, pz, Q1); };
                // where most are left to one of the wave's groups, all of them for all (as
                // in hex_vertex; the groups' branches would run one after the other)
                if (__ballot(!bounded || 4 * __popcll(act) > 3 * nSub) != 0ull) {
                    hex_add_ring<CPL>(acc, hx, f.n, C8, px, py, pz, Q1);
                } else {
                    HexP h = sub(__builtin_ctzll(act));
                    float al = alpha(__builtin_ctzll(act));
                    for (unsigned long long m = act & (act - 1);; m &= m - 1) {   // the next one's loads ahead
                        const int t = __builtin_ctzll(m | 1ull << 63);
                        const HexP hn = sub(m ? t : 0);
                        const float an = alpha(m ? t : 0);
                        add(h, al);
                        if (!m) break;
                        h = hn;
                        al = an;
                    }
                }
                // scores: only of candidates whose ratio is within rounding of the best one's
                float y[CPL], ym = 0.0f;
#pragma unroll
                for (int i = 0; i < CPL; ++i) {
                    y[i] = (acc[i].dmin < f.epsD || acc[i].fmin < f.epsF) ? 0.0f : acc[i].bd2 * __builtin_amdgcn_rcpf(acc[i].bF3);
                    ym = fmaxf(ym, y[i]);
                }
                const float Y = row_max(ym);
                const bool quick = fast && Y > 1e-30f;   // below, the ratios are not exact enough to rank by
                if (quick && Y < (yq * yq) * (1.0f - 4.0f * kSel)) continue;
                const float lim = Y * (1.0f - kSel);
                best = -FLT_MAX;
                int bi = 0;
#pragma unroll
                for (int i = 0; i < CPL; ++i) {
                    const bool in = !quick || y[i] >= lim;
                    float q = S0;
                    if (in && !(quick && acc[i].bd2 == f.acc0.bd2 && acc[i].bF3 == f.acc0.bF3))
                        q = hex_acc_score(acc[i], f.epsD, f.epsF);
                    if (in && q > best) { best = q; bi = i; }
                }
                const float own = best;
                best = row_max(own);
                const int l = row_first(own == best);
                cand = row_lane(bi, l) + NL * l;
            }
            tie = tie || (best == q0 && q0 > 0.0f);
            if (qbest < best) {
                cx = grid_coord(affL, cand % NL, NL, gxm, gxM);
                cy = grid_coord(affL, (cand / NL) % NL, NL, gym, gyM);
                cz = grid_coord(affL, cand / (NL * NL), NL, gzm, gzM);
                qbest = best;
                moved = true;
            }
        }
    };
    levels(1.0f);
    if (la.mode == 3 && !moved && !tie && !hex_pinned(f)) {
        cx = f.x0x; cy = f.x0y; cz = f.x0z;
        levels(kMode3Window);
    }
    if (moved && own && s == 0) { a.xw[vid] = cx; a.yw[vid] = cy; a.zw[vid] = cz; }
    const bool need = !moved && !tie && !hex_pinned(f) && own && s == 0;
    fallback_append(la, need, vid, nc);
    if (need && la.epoch) la.epoch[vid] = la.it;
}

// immediate fallback: one block = LV vertices on one wave, or (FUSED) 4 waves
// of LV = 4 vertices that first run their network tile; the fallbacks go to a
// second launch (k_search_list_*)
template <int NQ, int LV, bool FUSED>
__global__ __launch_bounds__(FUSED ? 256 : 64) void k_search_tet_learned(SearchArgs a, LearnArgs la, int ringCap)
{
    extern __shared__ __align__(16) unsigned char s_tcl[];
    tet_window<NQ, LV, FUSED ? 4 : 1, FUSED>(a, la, ringCap, blockIdx.x, s_tcl);
}
template <int NQ, int LV, bool FUSED, bool C8>
__global__ __launch_bounds__(FUSED ? 256 : 64) void k_search_hex_learned(SearchArgs a, LearnArgs la, int ringCap)
{
    extern __shared__ __align__(16) unsigned char s_hxl[];
    hex_window<NQ, LV, FUSED ? 4 : 1, FUSED, C8>(a, la, ringCap, blockIdx.x, s_hxl);
}

// deferred fallback: the first gridDim.x - nbList blocks take the windows of
// 16 class vertices each (the vertices deferred last iteration excepted),
// the last nbList blocks the full searches (a wave per vertex; 4 for short tet
// lists and for hexes with the largest offset as extent) of the
// vertices the previous iteration deferred; both are vertices of one colour
// class, so the two kinds run side by side.  The windows come first so that
// the dispatcher starts them before the list blocks, most of which find no
// vertex (list blocks first: 0.27 against 0.226 ms per learned 40^3 tet
// iteration).
template <int NQ, bool FUSED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
void k_search_tet_learned_def(SearchArgs a, LearnArgs la0, int ringCap, int nbList)
{
    extern __shared__ __align__(16) unsigned char s_tcd[];
    const LearnArgs la = learn_resolve(la0);
    const int nbWin = (int)gridDim.x - nbList;
    if ((int)blockIdx.x >= nbWin) {
        const int lb = (int)blockIdx.x - nbWin;
        const int n = min(*la.cntIn, a.cEnd - a.cStart);
        if (lb == 0 && threadIdx.x == 0) atomicAdd(la.fallbacks, n);
        const bool small = a.cEnd - a.cStart <= kTetWideClass;
        if (small || n > kTetWideDef) __builtin_amdgcn_s_setprio(3);   // as in the hex kernel below
        if (small && n <= kTetWideDef) {
            for (int i = lb; i < n; i += nbList) tet_vertex_wide<NQ>(a, uniform(la.listIn[i]), s_tcd, ringCap);
            return;
        }
        const int w = uniform((int)(threadIdx.x >> 6));   // one vertex per wave, in the wave's own LDS
        unsigned char* lds = s_tcd + (size_t)w * tet_wave_lds(ringCap);
        for (int i = lb + w * nbList; i < n; i += 4 * nbList) {
            tet_vertex<NQ>(a, uniform(la.listIn[i]), a.extentMin != 0, lds, ringCap);
            wave_lds_fence();   // the next vertex restages the ring
        }
        return;
    }
    tet_window<NQ, 4, 4, FUSED>(a, la, ringCap, (int)blockIdx.x, s_tcd);
}
// 4 waves per SIMD (<= 128 registers): a 48^3 class (~13k vertices, 3.3k
// waves) then fits the chip's wave slots in one round
template <int NQ, bool FUSED, bool C8>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
void k_search_hex_learned_def(SearchArgs a, LearnArgs la0, int ringCap, int nbList)
{
    extern __shared__ __align__(16) unsigned char s_hxd[];
    const LearnArgs la = learn_resolve(la0);
    const int nbWin = (int)gridDim.x - nbList;
    if ((int)blockIdx.x >= nbWin) {
        const int lb = (int)blockIdx.x - nbWin;
        const int n = min(*la.cntIn, a.cEnd - a.cStart);
        if (lb == 0 && threadIdx.x == 0) atomicAdd(la.fallbacks, n);
        // a full search alone takes as long as the windows' four rounds beside it:
        // it goes first (last wave of a class at 23 us instead of 31)
        __builtin_amdgcn_s_setprio(3);
        if (!a.extentMin) {
            for (int i = lb; i < n; i += nbList) hex_vertex_wide<NQ>(a, uniform(la.listIn[i]), s_hxd, ringCap);
            return;
        }
        const int w = uniform((int)(threadIdx.x >> 6));   // one vertex per wave, in the wave's own LDS
        unsigned char* lds = s_hxd + (size_t)w * hex_wave_lds(ringCap);
        for (int i = lb + w * nbList; i < n; i += 4 * nbList) {
            hex_vertex<NQ>(a, uniform(la.listIn[i]), a.extentMin != 0, reinterpret_cast<HexLds*>(lds),
                           hex_act(lds, ringCap));
            wave_lds_fence();   // the next vertex restages the ring
        }
        return;
    }
    hex_window<NQ, 4, 4, FUSED, C8>(a, la, ringCap, (int)blockIdx.x, s_hxd);
}

// plain search of the vertices list[0 .. *cnt) (the fallbacks of a class),
// one vertex per wave at a time, waves striding over the list
// (the grid is sized for a typical fallback share, the length is only known
// on the device)
// WIDE: blocks of 4 waves, which take a vertex together while the list is
// short, a vertex each otherwise
template <int NQ, bool WIDE>
__global__ __launch_bounds__(WIDE ? 256 : 64) void k_search_list_tet(SearchArgs a, const int* __restrict__ list,
                                                                    const int* __restrict__ cnt, int* fallbacks,
                                                                    int ringCap)
{
    extern __shared__ __align__(16) unsigned char s_tcf[];
    const int n = min(*cnt, a.cEnd - a.cStart);
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(fallbacks, n);
    if constexpr (WIDE) {
        if (n <= kTetWideMax) {
            for (int i = blockIdx.x; i < n; i += gridDim.x) tet_vertex_wide<NQ>(a, uniform(list[i]), s_tcf, ringCap);
            return;
        }
    }
    const int w = uniform((int)(threadIdx.x >> 6));
    for (int i = blockIdx.x + w * gridDim.x; i < n; i += (WIDE ? 4 : 1) * gridDim.x) {
        tet_vertex<NQ>(a, uniform(list[i]), a.extentMin != 0, s_tcf + (size_t)w * tet_wave_lds(ringCap), ringCap);
        wave_lds_fence();   // the next vertex restages the ring
    }
}
template <int NQ>
__global__ __launch_bounds__(64) void k_search_list_hex(SearchArgs a, const int* __restrict__ list,
                                                       const int* __restrict__ cnt, int* fallbacks, int ringCap)
{
    extern __shared__ __align__(16) unsigned char s_hxf[];
    const int n = min(*cnt, a.cEnd - a.cStart);
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(fallbacks, n);
    for (int i = blockIdx.x; i < n; i += gridDim.x) {
        hex_vertex<NQ>(a, uniform(list[i]), a.extentMin != 0, reinterpret_cast<HexLds*>(s_hxf), hex_act(s_hxf, ringCap));
        wave_lds_fence();   // the next vertex restages the ring
    }
}
template <int NQ>
__global__ __launch_bounds__(256) void k_search_list_hex_wide(SearchArgs a, const int* __restrict__ list,
                                                             const int* __restrict__ cnt, int* fallbacks, int ringCap)
{
    extern __shared__ __align__(16) unsigned char s_hxw[];
    const int n = min(*cnt, a.cEnd - a.cStart);
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(fallbacks, n);
    for (int i = blockIdx.x; i < n; i += gridDim.x) hex_vertex_wide<NQ>(a, uniform(list[i]), s_hxw, ringCap);
}
template <int NQ>
static void list_nq(int kind, const SearchArgs& a, const int* list, const int* cnt, int* fallbacks, int grid,
                     int ringCap, hipStream_t s)
{
    const size_t lds = search_lds_bytes(kind, ringCap);
    if constexpr (NQ % 4 == 0) {
        if (kind == VSDMO_TET && 4 * lds <= 64 * 1024) {   // a vertex per wave fits a block's LDS
            launch_kernel(k_search_list_tet<NQ, true>, grid, 256, 4 * lds, s, a, list, cnt, fallbacks, ringCap);
            return;
        }
        if (kind == VSDMO_HEX && !a.extentMin) {
            launch_kernel(k_search_list_hex_wide<NQ>, grid, 256, hex_wide_lds(ringCap), s, a, list, cnt, fallbacks, ringCap);
            return;
        }
    }
    if (kind == VSDMO_TET) launch_kernel(k_search_list_tet<NQ, false>, grid, 64, lds, s, a, list, cnt, fallbacks, ringCap);
    else launch_kernel(k_search_list_hex<NQ>, grid, 64, lds, s, a, list, cnt, fallbacks, ringCap);
}

template <int NQ, int LV, bool FUSED>
static void learned_nq_lv(int kind, const SearchArgs& a, const LearnArgs& la, int ringCap, int nb, size_t lds, hipStream_t s)
{
    constexpr int T = FUSED ? 256 : 64;
    if (kind == VSDMO_TET) launch_kernel(k_search_tet_learned<NQ, LV, FUSED>, nb, T, lds, s, a, la, ringCap);
    else if (a.hexCorner8) launch_kernel(k_search_hex_learned<NQ, LV, FUSED, true>, nb, T, lds, s, a, la, ringCap);
    else launch_kernel(k_search_hex_learned<NQ, LV, FUSED, false>, nb, T, lds, s, a, la, ringCap);
}

static size_t learned_per(int kind) { return (kind == VSDMO_TET) ? sizeof(TetC) : sizeof(HexLds); }

// largest ring the window kernel's LDS (kLV rings per block, 64 KB) holds
int learned_ring_cap(int kind) { return (int)((64 * 1024) / (kLV * learned_per(kind))); }

// 16 rings per block in 64 KB of LDS
static bool rings16_fit(int kind, int ringCap)
{
    return (size_t)kMlpRows * std::max(ringCap, 1) * learned_per(kind) <= 64 * 1024;
}

// LDS of a FUSED window block: the network's (reused for the 16 rings) and
// the table-neighbour positions
static size_t fused_lds(int kind, int ringCap)
{
    return learned_rel_offset(learned_per(kind), std::max(ringCap, 1)) + kLearnedRelBytes;
}

// the fused kernel holds 16 rings and the table-neighbour positions per
// block in the same 64 KB
bool learned_fused_ok(int kind, int ringCap)
{
    return fused_lds(kind, ringCap) <= 64 * 1024;
}

// the deferred policy's kernels hold the 4-wave full searches, which split a line of
// candidates in four (nq 4 and 8), and 16 rings in LDS with or without the network
bool learned_deferred_ok(int kind, int nq, int ringCap)
{
    return (nq == 4 || nq == 8) && rings16_fit(kind, ringCap);
}


template <int NQ, bool FUSED>
static void learned_def_nq(int kind, const SearchArgs& a, const LearnArgs& la, int ringCap, int nbList, int nb,
                           size_t lds, hipStream_t s)
{
    if (kind == VSDMO_TET) launch_kernel(k_search_tet_learned_def<NQ, FUSED>, nbList + nb, 256, lds, s, a, la, ringCap, nbList);
    else if (a.hexCorner8)
        launch_kernel(k_search_hex_learned_def<NQ, FUSED, true>, nbList + nb, 256, lds, s, a, la, ringCap, nbList);
    else launch_kernel(k_search_hex_learned_def<NQ, FUSED, false>, nbList + nb, 256, lds, s, a, la, ringCap, nbList);
}

void launch_search_learned(int kind, int nq, const SearchArgs& a, const LearnNet& net, int mode, int depthL,
                           float frac, int* fallbacks, int* list, int* cnt, int ringCap, const LearnDefer* def,
                           hipStream_t s)
{
    const int nc = a.cEnd - a.cStart;
    if (nc <= 0) return;
    ringCap = std::max(ringCap, 1);
    const size_t per = learned_per(kind);
    const bool fused = learn_uses_net(mode) && net.wb && net.loc && learned_fused_ok(kind, ringCap);
    LearnArgs la{ net.Y, net.L, mode, depthL, frac, fallbacks, list, cnt, net.wb, net.w, net.nbr,
                  nullptr, nullptr, nullptr, 0, net.items };
    la.loc = net.loc;
    if (def) {
        // one launch: this iteration's windows, 16 vertices per block, beside
        // the previous iteration's fallbacks (list blocks sized for an eighth
        // of the class, they loop when more were deferred: a sixteenth
        // measured the same, a thirty-second slower on the 40^3 tet cube)
        la.listIn = def->listIn; la.cntIn = def->cntIn; la.epoch = def->epoch; la.it = def->it;
        la.itDev = def->itDev; la.listStride = def->listStride; la.cntStride = def->cntStride;
        const int nbList = std::max(1, std::min(nc, std::max(64, nc / 8)));
        const int nb = (nc + kMlpRows - 1) / kMlpRows;
        const size_t wave = kind == VSDMO_TET ? tet_wave_lds(ringCap) : hex_wave_lds(ringCap);
        const size_t lds = std::max(fused ? fused_lds(kind, ringCap) : (size_t)kMlpRows * ringCap * per, 4 * wave);
        switch (nq) {   // learned_deferred_ok
        case 4: fused ? learned_def_nq<4, true>(kind, a, la, ringCap, nbList, nb, lds, s)
                      : learned_def_nq<4, false>(kind, a, la, ringCap, nbList, nb, lds, s); break;
        case 8: fused ? learned_def_nq<8, true>(kind, a, la, ringCap, nbList, nb, lds, s)
                      : learned_def_nq<8, false>(kind, a, la, ringCap, nbList, nb, lds, s); break;
        default: break;
        }
        return;
    }
    const int vpb = fused ? kMlpRows : kLV;
    const int nb = (nc + vpb - 1) / vpb;
    const size_t lds = fused ? fused_lds(kind, ringCap) : (size_t)kLV * ringCap * per;
#define VSDMO_LEARN_CASE(Q)                                                                           \
    case Q:                                                                                          \
        if (fused) learned_nq_lv<Q, kLV, true>(kind, a, la, ringCap, nb, lds, s);                     \
        else learned_nq_lv<Q, kLV, false>(kind, a, la, ringCap, nb, lds, s);                          \
        break;
    switch (nq) {
        VSDMO_LEARN_CASE(2)
        VSDMO_LEARN_CASE(4)
        VSDMO_LEARN_CASE(6)
        VSDMO_LEARN_CASE(8)
    default: break;
    }
#undef VSDMO_LEARN_CASE
    // second launch: the plain search of the fallbacks, a wave per vertex, a
    // quarter of the class's vertices at a time (blocks loop when more fall back)
    const int g1 = std::max(1, std::min(nc, std::max(256, nc / 4)));
    switch (nq) {
    case 2: list_nq<2>(kind, a, list, cnt, fallbacks, g1, ringCap, s); break;
    case 4: list_nq<4>(kind, a, list, cnt, fallbacks, g1, ringCap, s); break;
    case 6: list_nq<6>(kind, a, list, cnt, fallbacks, g1, ringCap, s); break;
    case 8: list_nq<8>(kind, a, list, cnt, fallbacks, g1, ringCap, s); break;
    default: break;
    }
}

// ------------------------------------------------------- batched sweep
// Persistent kernel of one colour round of a batch of meshes: blocks take
// work items from a queue (one atomic counter per round) until it is empty.
// An item is a global vertex id with its element type in bits 30-31
// (0 tet, 1 hex, 2 flat tri).  Vertices of one round belong to one colour
// class of their mesh, so the order in which they are taken does not change
// any result.
// Items [lo, mid) are tet / hex searches, taken one at a time from the
// round's counter (their cost varies with the ring); items [mid, hi) are flat
// triangle searches, ~100x cheaper and uniform, statically strided over the
// blocks so that they cost no atomics.
template <int NQ>
__device__ __forceinline__ void batch_item(const SearchArgs& a, const int* rowHex, const int* valHex, int code,
                                           int tetCap, int hexCap, unsigned char* lds)
{
    const int vid = uniform(code & 0x3fffffff), type = uniform((code >> 30) & 3);
    if (type == 0) tet_vertex<NQ>(a, vid, false, lds, tetCap);
    else if (type == 1) {
        SearchArgs ah = a;
        ah.ringRow = rowHex;
        ah.ringVal = valHex;
        hex_vertex<NQ>(ah, vid, true, reinterpret_cast<HexLds*>(lds), hex_act(lds, hexCap));
    }
    else flat_vertex<NQ>(a, vid, reinterpret_cast<TriC*>(lds));
}

template <int NQ>
__global__ __launch_bounds__(64) void k_batch_round(SearchArgs a, const int* __restrict__ rowHex,
                                                   const int* __restrict__ valHex, const int* __restrict__ items,
                                                   int lo, int mid, int hi, int* __restrict__ ctr, int tetCap, int hexCap)
{
    extern __shared__ __align__(16) unsigned char s_dyn[];
    for (;;) {
        int at = 0;
        if (threadIdx.x == 0) at = atomicAdd(ctr, 1);
        const int it = lo + uniform(at);
        if (it >= mid) break;
        batch_item<NQ>(a, rowHex, valHex, items[it], tetCap, hexCap, s_dyn);
        wave_lds_fence();   // the next item restages the LDS
    }
    for (int it = mid + (int)blockIdx.x; it < hi; it += (int)gridDim.x) {
        batch_item<NQ>(a, rowHex, valHex, items[it], tetCap, hexCap, s_dyn);
        wave_lds_fence();
    }
}

// ------------------------------------------------------------ qualities
// element quality = ring score of the element seen from its vertex 0 at p'=0
__device__ float elem_quality(const float* __restrict__ X, const float* __restrict__ Y, const float* __restrict__ Z,
                              const int* c, int elem, bool corner8)
{
    const float x0x = X[c[0]], x0y = Y[c[0]], x0z = Z[c[0]];
    if (elem == VSDMO_TET) {
        float m = 0.0f;
        for (int i = 1; i < 4; ++i) {
            m = fmaxf(m, fabsf(X[c[i]] - x0x));
            m = fmaxf(m, fabsf(Y[c[i]] - x0y));
            m = fmaxf(m, fabsf(Z[c[i]] - x0z));
        }
        const float sg = pow2_scale(m);
        const float isg = 1.0f / sg;
        f3 p[3];
        for (int i = 0; i < 3; ++i) {
            int v = c[i + 1];
            p[i] = { (X[v] - x0x) * sg, (Y[v] - x0y) * sg, (Z[v] - x0z) * sg };
        }
        TetC tc = tet_consts(p[0], p[1], p[2]);
        const float px = 0.0f, py = 0.0f, pz = 0.0f;
        const float Qyz = 3.0f * fmaf(pz, pz, py * py), t3 = 3.0f * px;
        TetAcc acc = tet_acc0();
        float Tyz = fmaf(tc.nny, py, fmaf(tc.nnz, pz, tc.D));
        float Ryz = fmaf(tc.m2sy, py, fmaf(tc.m2sz, pz, tc.K + Qyz));
        tet_acc_add(acc, fmaf(tc.nnx, px, Tyz), fmaf(px, t3 + tc.m2sx, Ryz));
        return tet_acc_score(acc, ((1.0f * isg) * isg) * isg);
    }
    if (elem == VSDMO_HEX) {
        float m = 0.0f;
        for (int i = 1; i < 8; ++i) {
            m = fmaxf(m, fabsf(X[c[i]] - x0x));
            m = fmaxf(m, fabsf(Y[c[i]] - x0y));
            m = fmaxf(m, fabsf(Z[c[i]] - x0z));
        }
        const float sg = pow2_scale(m);
        const float s2 = sg * sg, s3 = s2 * sg;
        f3 r[8];
        r[0] = { 0.0f, 0.0f, 0.0f };
        for (int i = 1; i < 8; ++i) {
            int v = c[i];
            r[i] = { (X[v] - x0x) * sg, (Y[v] - x0y) * sg, (Z[v] - x0z) * sg };
        }
        float cd[4], cF[4];
        HexP hp[5];
        hex_consts(r, cd, cF, hp);
        HexAcc acc = hex_acc0();
        for (int sIdx = 0; sIdx < 4; ++sIdx) hex_acc_add(acc, cd[sIdx], cF[sIdx]);
        const float px = 0.0f, py = 0.0f, pz = 0.0f;
        const float Q1 = fmaf(pz, pz, py * py), Q3 = 3.0f * Q1, t3 = 3.0f * px;
#pragma unroll
        for (int sIdx = 0; sIdx < 5; ++sIdx) {   // unrolled: hp[] stays in registers
            if (sIdx == 4 && corner8) break;
            const bool a3 = (sIdx == 1 || sIdx == 4);
            float Tyz = fmaf(hp[sIdx].gy, py, fmaf(hp[sIdx].gz, pz, hp[sIdx].D));
            float Ryz = fmaf(hp[sIdx].sy, py, fmaf(hp[sIdx].sz, pz, hp[sIdx].K + (a3 ? Q3 : Q1)));
            hex_acc_add(acc, fmaf(hp[sIdx].gx, px, Tyz), fmaf(px, (a3 ? t3 : px) + hp[sIdx].sx, Ryz));
        }
        return hex_acc_score(acc, kHexEps * s3, kHexEps * s2);
    }
    if (elem == VSDMO_QUAD)
        return mr_quad3(f3{ x0x, x0y, x0z }, f3{ X[c[1]], Y[c[1]], Z[c[1]] }, f3{ X[c[2]], Y[c[2]], Z[c[2]] },
                        f3{ X[c[3]], Y[c[3]], Z[c[3]] }, nullptr);
    if (elem == kElemTri3)
        return mr_tri3(f3{ x0x, x0y, x0z }, f3{ X[c[1]], Y[c[1]], Z[c[1]] }, f3{ X[c[2]], Y[c[2]], Z[c[2]] }, nullptr);
    float m = 0.0f;
    for (int i = 1; i < 3; ++i) {
        m = fmaxf(m, fabsf(X[c[i]] - x0x));
        m = fmaxf(m, fabsf(Y[c[i]] - x0y));
    }
    const float sg = pow2_scale(m);
    const float isg = 1.0f / sg;
    TriC tc = tri_consts((X[c[1]] - x0x) * sg, (Y[c[1]] - x0y) * sg, (X[c[2]] - x0x) * sg, (Y[c[2]] - x0y) * sg);
    const float px = 0.0f, py = 0.0f;
    const float Q2 = 2.0f * (py * py), t2 = 2.0f * px;
    TriAcc acc = tri_acc0();
    float Ty = fmaf(tc.gy, py, tc.C);
    float Ry = fmaf(tc.sy, py, tc.K + Q2);
    tri_acc_add(acc, fmaf(tc.gx, px, Ty), fmaf(px, t2 + tc.sx, Ry));
    return tri_acc_score(acc, (1.0f * isg) * isg);
}

// elements per thread of the quality kernels: up to 4 (strided by 256), as
// long as the launch keeps at least 512 blocks (two per CU)
int quality_per_thread(long long nElements)
{
    int per = 4;
    while (per > 1 && nElements < (long long)per * 256 * 512) per >>= 1;
    return per;
}

// min and FP64 sum over the 256 threads of a block: a butterfly within each
// wave (lane 0's value: the order of its additions is fixed), then the 4 waves
// in order; the result is every thread's.  One call per kernel (static LDS).
__device__ __forceinline__ void block_minsum256(float& m, double& s)
{
    __shared__ float wm[4];
    __shared__ double ws[4];
#pragma unroll
    for (int k = 32; k >= 1; k >>= 1) {
        m = fminf(m, __shfl_xor(m, k));
        s = s + __shfl_xor(s, k);
    }
    const int w = (int)(threadIdx.x >> 6);
    if ((threadIdx.x & 63) == 0) { wm[w] = m; ws[w] = s; }
    __syncthreads();
    m = fminf(fminf(wm[0], wm[1]), fminf(wm[2], wm[3]));
    s = (ws[0] + ws[1]) + (ws[2] + ws[3]);
}

// true in the one thread that arrives last of all blocks, each of which has
// one thread call it after its agent-scope stores.  Those are complete at the
// point of coherence once they have left the wave's memory counter, so no
// release of the whole L2 is needed.
__device__ __forceinline__ bool last_block(int* ticket, int b, int nb)
{
    // the wait and the compiler's fence in one: the builtin alone does not touch
    // memory, so a relaxed store could be moved past it
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const int g = b % kTicketGroups, ng = nb < kTicketGroups ? nb : kTicketGroups;
    const int members = nb / kTicketGroups + (g < nb % kTicketGroups);
    if (__hip_atomic_fetch_add(ticket + (g + 1) * kTicketStride, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
        != members - 1) return false;
    return __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == ng - 1;
}

// the qualities of the block's 256 * per elements (per per thread, strided by
// 256), written to q, and their min and FP64 sum in a fixed order.  The block
// that takes the last ticket reduces the blocks' partials (strided, then a
// fixed tree: the order of the additions depends only on the block count) and
// writes {min, surface error bits, sum} straight into pinned host memory: one
// launch, where a second reduction kernel (3-5 us with its gap) and a 16-byte
// copy (2-5 us) followed.  Partials and tickets go through the device's point of
// coherence (agent-scope stores and loads), as the blocks run on all XCDs.
// The tickets are counted in groups, then over the groups: with one counter
// and a release of the L2 by every block, 750 blocks (384k elements) took
// 9 us more per iteration than the two launches; in groups they take 1-2 us less.
__global__ __launch_bounds__(256) void k_elem_quality(QualityArgs a, float* pmin, double* psum, int* ticket,
                                                      const int* err, QualityOut* out, int per)
{
    __shared__ float smin[256];
    __shared__ double ssum[256];
    __shared__ int s_last;
    float v = FLT_MAX;
    double sv = 0.0;
    for (int k = 0; k < per; ++k) {
        const int e = blockIdx.x * 256 * per + k * 256 + (int)threadIdx.x;
        if (e < a.nE) {
            const float q = elem_quality(a.x, a.y, a.z, a.cells + (size_t)e * a.npe, a.elem, a.hexCorner8 != 0);
            a.q[e] = q;
            v = fminf(v, q);
            sv = sv + (double)q;
        }
    }
    block_minsum256(v, sv);
    if (threadIdx.x == 0) {
        __hip_atomic_store(pmin + blockIdx.x, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(psum + blockIdx.x, sv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = last_block(ticket, (int)blockIdx.x, (int)gridDim.x);
    }
    __syncthreads();
    if (!s_last) return;
    float m = FLT_MAX;
    double s = 0.0;
    for (int i = threadIdx.x; i < (int)gridDim.x; i += 256) {
        m = fminf(m, __hip_atomic_load(pmin + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        s = s + __hip_atomic_load(psum + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    smin[threadIdx.x] = m;
    ssum[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) {
            smin[threadIdx.x] = fminf(smin[threadIdx.x], smin[threadIdx.x + k]);
            ssum[threadIdx.x] = ssum[threadIdx.x] + ssum[threadIdx.x + k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out->min = smin[0];
        out->err = *err;
        out->sum = ssum[0];
    }
    // for the next launch
    if (threadIdx.x <= kTicketGroups) ticket[threadIdx.x * kTicketStride] = 0;
}

// batch qualities: one block of 256 per chunk of at most 256 * a.per
// elements of one mesh; per-chunk min and FP64 sum in a fixed order
__global__ __launch_bounds__(256) void k_batch_quality(BatchQArgs a)
{
    const int c = blockIdx.x;
    const int e0 = a.chunkElem0[c], ne = a.chunkElem0[c + 1] - e0;
    const int elem = a.chunkType[c];
    const int npe = elem == VSDMO_TET ? 4 : elem == VSDMO_HEX ? 8 : 3;
    float m = FLT_MAX;
    double s = 0.0;
    for (int k = 0; k < a.per; ++k) {
        const int t = k * 256 + (int)threadIdx.x;
        if (t < ne) {
            const float q = elem_quality(a.x, a.y, a.z, a.cells + a.chunkCell0[c] + (size_t)t * npe, elem,
                                         a.hexCorner8 != 0);
            m = fminf(m, q);
            s = s + (double)q;
        }
    }
    block_minsum256(m, s);
    if (threadIdx.x == 0) { a.cmin[c] = m; a.csum[c] = s; }
}

// per-mesh min / FP64 sum over the mesh's chunks: one block per mesh,
// strided partials then a fixed tree (the order depends only on the chunk
// count); the minimum is also written to history row *hctr
__global__ void k_batch_mesh_reduce(BatchQArgs a)
{
    __shared__ float smin[256];
    __shared__ double ssum[256];
    const int b = blockIdx.x;
    float m = FLT_MAX;
    double s = 0.0;
    for (int c = a.meshChunk0[b] + (int)threadIdx.x; c < a.meshChunk0[b + 1]; c += 256) {
        m = fminf(m, a.cmin[c]);
        s = s + a.csum[c];
    }
    smin[threadIdx.x] = m;
    ssum[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) {
            smin[threadIdx.x] = fminf(smin[threadIdx.x], smin[threadIdx.x + k]);
            ssum[threadIdx.x] = ssum[threadIdx.x] + ssum[threadIdx.x + k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        a.mmin[b] = smin[0];
        a.msum[b] = ssum[0];
        const int row = *a.hctr;
        if (row < a.hcap) a.hist[(size_t)row * a.nMeshes + b] = smin[0];
    }
}

// advances the history row after every mesh of the iteration wrote it
__global__ void k_batch_history_next(int* hctr)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *hctr = *hctr + 1;
}

__global__ void k_histogram(const float* __restrict__ q, int n, int ncols, int* __restrict__ bins)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float v = fminf(0.9999f, q[i]);
    long idx = (long)(v * (float)ncols);
    if (idx < 0) idx = 0;
    atomicAdd(&bins[idx], 1);
}

// ------------------------------------------------------------- launchers
template <int NQ>
static void launch_nq(int kind, const SearchArgs& a, int nBlocks, int ringCap, hipStream_t s)
{
    const size_t lds = search_lds_bytes(kind, ringCap);
    if constexpr (NQ % 4 == 0) {
        if (kind == VSDMO_TET && nBlocks <= kTetWideMax) {
            launch_kernel(k_search_tet_wide<NQ>, nBlocks, 256, tet_wide_lds(ringCap), s, a, ringCap);
            return;
        }
    }
    if (kind == VSDMO_TET) launch_kernel(k_search_tet<NQ>, nBlocks, 64, lds, s, a, ringCap);
    else if (kind == VSDMO_HEX) launch_kernel(k_search_hex<NQ>, nBlocks, 64, lds, s, a, ringCap);
    else launch_kernel(k_search_flat<NQ>, nBlocks, 64, lds, s, a);
}
// Non-persistent variant of a round: one block per item, scheduled by the
// hardware dispatcher (no queue, no atomics), one launch per element type
// (0 tet, 1 hex, 2 flat tri) with the search body of that type alone, so
// that each keeps the registers and LDS of its own body.  The tet body asks
// for the plain tet search's occupancy (VSDMO_TET_MIN_WAVES waves per SIMD).
template <int NQ, int TYPE>
__global__ __launch_bounds__(64, TYPE == 0 ? VSDMO_TET_MIN_WAVES : TYPE == 1 ? VSDMO_HEX_MIN_WAVES : 1)
void k_batch_typed(SearchArgs a, const int* __restrict__ rowHex, const int* __restrict__ valHex,
                   const int* __restrict__ items, int lo, int ringCap)
{
    extern __shared__ __align__(16) unsigned char s_typ[];
    const int vid = items[lo + blockIdx.x] & 0x3fffffff;
    if constexpr (TYPE == 0) {
        tet_vertex<NQ>(a, vid, false, s_typ, ringCap);
    } else if constexpr (TYPE == 1) {
        SearchArgs ah = a;
        ah.ringRow = rowHex;
        ah.ringVal = valHex;
        hex_vertex<NQ>(ah, vid, true, reinterpret_cast<HexLds*>(s_typ), hex_act(s_typ, ringCap));
    } else {
        flat_vertex<NQ>(a, vid, reinterpret_cast<TriC*>(s_typ));
    }
}

template <int NQ>
static void batch_typed_nq(const SearchArgs& a, const int* rowHex, const int* valHex, const int* items, int lo, int hi,
                           int type, int ringCap, hipStream_t s)
{
    const unsigned n = (unsigned)(hi - lo);
    const size_t lds = search_lds_bytes(type == 0 ? VSDMO_TET : type == 1 ? VSDMO_HEX : VSDMO_TRI, ringCap);
    if (type == 0) k_batch_typed<NQ, 0><<<n, 64, lds, s>>>(a, rowHex, valHex, items, lo, ringCap);
    else if (type == 1) k_batch_typed<NQ, 1><<<n, 64, lds, s>>>(a, rowHex, valHex, items, lo, ringCap);
    else k_batch_typed<NQ, 2><<<n, 64, lds, s>>>(a, rowHex, valHex, items, lo, ringCap);
}

template <int NQ>
static int batch_occ_nq(size_t lds)
{
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_batch_round<NQ>, 64, lds) != hipSuccess) nb = 1;
    return nb;
}

bool waves_supported(int nq, int w)
{
    return w == 0 || w == 1 || (w == 2 && nq % 2 == 0) || (w == 4 && nq % 4 == 0);
}

int batch_round_blocks_per_cu(int nq, size_t lds)
{
    switch (nq) {
    case 2: return batch_occ_nq<2>(lds);
    case 4: return batch_occ_nq<4>(lds);
    case 6: return batch_occ_nq<6>(lds);
    default: return batch_occ_nq<8>(lds);
    }
}

void launch_batch_round(int nq, const SearchArgs& a, const int* rowHex, const int* valHex, const int* items, int lo,
                        int mid, int hi, int* ctr, int grid, size_t lds, int tetCap, int hexCap, hipStream_t s)
{
    if (hi <= lo || grid <= 0) return;
#define VSDMO_ROUND_CASE(Q)                                                                                        \
    case Q: k_batch_round<Q><<<grid, 64, lds, s>>>(a, rowHex, valHex, items, lo, mid, hi, ctr, tetCap, hexCap); break;
    switch (nq) {
        VSDMO_ROUND_CASE(2)
        VSDMO_ROUND_CASE(4)
        VSDMO_ROUND_CASE(6)
        VSDMO_ROUND_CASE(8)
    default: break;
    }
#undef VSDMO_ROUND_CASE
}

void launch_batch_typed(int nq, const SearchArgs& a, const int* rowHex, const int* valHex, const int* items, int lo,
                        int hi, int type, int ringCap, hipStream_t s)
{
    if (hi <= lo) return;
    ringCap = std::max(ringCap, 1);
    if (type == 2 && flat8x4_ok(nq, ringCap, hi - lo)) {
        const int groups = (hi - lo + kFlatGroups - 1) / kFlatGroups;
        k_batch_flat8x4<<<groups, 256, kFlatGroups * sizeof(TriC) * (size_t)ringCap, s>>>(a, items, lo, hi, ringCap);
        return;
    }
    switch (nq) {
    case 2: batch_typed_nq<2>(a, rowHex, valHex, items, lo, hi, type, ringCap, s); break;
    case 4: batch_typed_nq<4>(a, rowHex, valHex, items, lo, hi, type, ringCap, s); break;
    case 6: batch_typed_nq<6>(a, rowHex, valHex, items, lo, hi, type, ringCap, s); break;
    case 8: batch_typed_nq<8>(a, rowHex, valHex, items, lo, hi, type, ringCap, s); break;
    default: break;
    }
}

void launch_fill_int(int* p, int n, int v, hipStream_t s)
{
    if (n > 0) k_fill_int<<<(n + 255) / 256, 256, 0, s>>>(p, n, v);
}

// zero the n counters of parity (*itDev & 1): cnt + parity * n
__global__ void k_parity_zero(int* __restrict__ cnt, int n, const int* __restrict__ itDev)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) cnt[(size_t)(*itDev & 1) * n + i] = 0;
}

__global__ void k_add_int(int* __restrict__ p, int v)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) *p += v;
}

void launch_parity_zero(int* cnt, int n, const int* itDev, hipStream_t s)
{
    if (n > 0) k_parity_zero<<<(n + 255) / 256, 256, 0, s>>>(cnt, n, itDev);
}

void launch_add_int(int* p, int v, hipStream_t s) { k_add_int<<<1, 64, 0, s>>>(p, v); }

void launch_batch_quality(const BatchQArgs& a, hipStream_t s)
{
    if (a.nChunks > 0) k_batch_quality<<<a.nChunks, 256, 0, s>>>(a);
    if (a.nMeshes > 0) k_batch_mesh_reduce<<<a.nMeshes, 256, 0, s>>>(a);
    k_batch_history_next<<<1, 64, 0, s>>>(a.hctr);
}

size_t search_lds_bytes(int kind, int ringCap)
{
    ringCap = std::max(ringCap, 1);
    if (kind == VSDMO_TET) return tet_wave_lds(ringCap);
    return (kind == VSDMO_HEX ? kHexLdsPer : sizeof(TriC)) * (size_t)ringCap;
}

size_t batch_lds_bytes(int maxRingTet, int maxRingHex, int maxHETri)
{
    return std::max(search_lds_bytes(VSDMO_TET, maxRingTet),
                    std::max(search_lds_bytes(VSDMO_HEX, maxRingHex), search_lds_bytes(VSDMO_TRI, maxHETri)));
}

void launch_search(int kind, int nq, const SearchArgs& a, int ringCap, hipStream_t s)
{
    int nBlocks = a.cEnd - a.cStart;
    if (nBlocks <= 0) return;
    ringCap = std::max(ringCap, 1);
    if (kind == VSDMO_TRI && flat8x4_ok(nq, ringCap, nBlocks)) {
        const int groups = (nBlocks + kFlatGroups - 1) / kFlatGroups;
        launch_kernel(k_search_flat8x4, groups, 256, kFlatGroups * sizeof(TriC) * (size_t)ringCap, s, a, ringCap);
        return;
    }
    switch (nq) {
    case 2: launch_nq<2>(kind, a, nBlocks, ringCap, s); break;
    case 4: launch_nq<4>(kind, a, nBlocks, ringCap, s); break;
    case 6: launch_nq<6>(kind, a, nBlocks, ringCap, s); break;
    case 8: launch_nq<8>(kind, a, nBlocks, ringCap, s); break;
    default: break;
    }
}

void launch_quality(const QualityArgs& a, float* pmin, double* psum, int* ticket, const int* err, QualityOut* out,
                    hipStream_t s)
{
    const int per = quality_per_thread(a.nE);
    const int nb = (a.nE + 256 * per - 1) / (256 * per);
    k_elem_quality<<<nb, 256, 0, s>>>(a, pmin, psum, ticket, err, out, per);
}

void launch_histogram(const float* q, int n, int ncols, int* bins, hipStream_t s)
{
    k_histogram<<<(n + 255) / 256, 256, 0, s>>>(q, n, ncols, bins);
}

}  // namespace vsdmo
