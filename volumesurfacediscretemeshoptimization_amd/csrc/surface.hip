// surface.hip -- surface-vertex DMO on the GPU: local quadric fits (own 3x3
// LU), feature-sector fits, 1D feature-curve fits, nearest-neighbour walk,
// and the 2D surface / 1D feature-curve searches with projection onto the
// blended local surfaces.
//
// Reference (VSDMO/src/dmo/...): surfaceP/Surface.h:18-169, Surface.cu:11-121,
// surfaceP/SurfaceFeature.h:79-106, SurfaceFeature.cu:12-223,
// Surface1D.h:13-114, Surface1D.cu:7-103, SurfaceEstimation.h:122-197,
// DMOCommon.cu:11-43, DMOCommon.h:130-165, DMOHexImplCub.h:141-489,
// DMOTetImplCub.h:141-494; surface meshes DMOTriImplCub.h:25-380,
// DMOQuadImplCub.h:23-404, DMOQualityTri.h:257-275, DMOQualityQuad.h:30-50,
// MeshGPUCommon.cu:413-434 (vertex normals), Laplace.cu:8-41.  Expressions follow the reference literally
// (dot = (x*x' + y*y') + z*z', normalize divides by sqrtf(dot)) with
// contraction off, so a host restatement of the same expressions reproduces
// every value.
#include <float.h>

#include "dmo_kernels.h"
#include "vsdmo_internal.h"
#include "vsdmo_numerics.h"

namespace vsdmo {

constexpr int kMaxNeigh = 40;
constexpr int kTableSize = 20;
constexpr float kSEps = 1.19209e-07f;

struct w3 { float x, y, z; };
__device__ __forceinline__ w3 W(const float* p) { return { p[0], p[1], p[2] }; }
__device__ __forceinline__ w3 WP(const float* x, const float* y, const float* z, int v) { return { x[v], y[v], z[v] }; }
__device__ __forceinline__ w3 wsub(w3 a, w3 b) { return { a.x - b.x, a.y - b.y, a.z - b.z }; }
__device__ __forceinline__ w3 wadd(w3 a, w3 b) { return { a.x + b.x, a.y + b.y, a.z + b.z }; }
__device__ __forceinline__ w3 wmul(float s, w3 a) { return { s * a.x, s * a.y, s * a.z }; }
__device__ __forceinline__ float wdot(w3 a, w3 b) { return (a.x * b.x + a.y * b.y) + a.z * b.z; }
__device__ __forceinline__ w3 wcross(w3 a, w3 b)
{
    return { a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x };
}
__device__ __forceinline__ float wnorm(w3 a) { return sqrtf((a.x * a.x + a.y * a.y) + a.z * a.z); }
__device__ __forceinline__ w3 wnormalize(w3 a)
{
    float l = wnorm(a);
    return { a.x / l, a.y / l, a.z / l };
}

// local surface record: p0 (3), e0 e1 e2 (9), a b c (3), numPoints (1)
struct LSurf { w3 p0, e[3]; float a, b, c, np; };
struct LSurf1 { w3 p0, e[2]; float a; };
static_assert(sizeof(LSurf) == 16 * sizeof(float), "LSurf layout");
static_assert(sizeof(LSurf1) == 10 * sizeof(float), "LSurf1 layout");

__device__ __forceinline__ float poly(const LSurf& s, float u, float v) { return (s.a * u * u + s.b * u * v) + s.c * v * v; }
__device__ __forceinline__ w3 l2w(const LSurf& s, float u, float v, float w)
{
    return wadd(wadd(wadd(s.p0, wmul(u, s.e[0])), wmul(v, s.e[1])), wmul(w, s.e[2]));
}

// 3x3 LU with partial pivoting (first maximal |pivot|) and solve; column-major A
__device__ void lu_solve3(const float* Acm, const float* rhs, float* x)
{
    float A[3][3], b[3];
    for (int i = 0; i < 3; ++i) {
        for (int j = 0; j < 3; ++j) A[i][j] = Acm[i + 3 * j];
        b[i] = rhs[i];
    }
    int piv[3] = { 0, 1, 2 };
    for (int j = 0; j < 3; ++j) {
        int p = j;
        float mx = fabsf(A[j][j]);
        for (int i = j + 1; i < 3; ++i)
            if (fabsf(A[i][j]) > mx) { mx = fabsf(A[i][j]); p = i; }
        if (p != j) {
            for (int k = 0; k < 3; ++k) { float t = A[j][k]; A[j][k] = A[p][k]; A[p][k] = t; }
            int t = piv[j]; piv[j] = piv[p]; piv[p] = t;
        }
        for (int i = j + 1; i < 3; ++i) {
            A[i][j] = A[i][j] / A[j][j];
            for (int k = j + 1; k < 3; ++k) A[i][k] = A[i][k] - A[i][j] * A[j][k];
        }
    }
    float y[3];
    for (int i = 0; i < 3; ++i) y[i] = b[piv[i]];
    for (int i = 1; i < 3; ++i)
        for (int k = 0; k < i; ++k) y[i] = y[i] - A[i][k] * y[k];
    for (int i = 2; i >= 0; --i) {
        for (int k = i + 1; k < 3; ++k) y[i] = y[i] - A[i][k] * y[k];
        y[i] = y[i] / A[i][i];
    }
    x[0] = y[0]; x[1] = y[1]; x[2] = y[2];
}

__device__ void frame3(w3 n, w3 r, w3* e0, w3* e1, w3* e2)
{
    if (wnorm(wcross(n, r)) < 10.0f * kSEps) r = { n.x, n.z, -n.y };
    w3 t1 = wcross(n, r);
    w3 t2 = wcross(n, t1);
    *e2 = wnormalize(n);
    *e0 = wnormalize(t1);
    *e1 = wnormalize(t2);
}

__device__ void fit_quadric(LSurf& s, const w3* pts, int np)
{
    float M[9] = { 0, 0, 0, 0, 0, 0, 0, 0, 0 }, R[3] = { 0, 0, 0 };
    for (int i = 0; i < np; ++i) {
        w3 p = wsub(pts[i], s.p0);
        float u = wdot(s.e[0], p), v = wdot(s.e[1], p), w = wdot(s.e[2], p);
        R[0] += u * u * w; R[1] += u * v * w; R[2] += v * v * w;
        M[0] += u * u * u * u; M[1] += u * u * u * v; M[4] += u * u * v * v;
        M[2] += u * u * v * v; M[5] += u * v * v * v; M[8] += v * v * v * v;
    }
    M[3] = M[1]; M[6] = M[2]; M[7] = M[5];
    float abc[3];
    lu_solve3(M, R, abc);
    s.a = abc[0]; s.b = abc[1]; s.c = abc[2];
    s.np = (float)np;
    if (np <= 4) { s.a = 0.0f; s.b = 0.0f; s.c = 0.0f; }
    if (s.a != s.a) s.a = 0.0f;
    if (s.b != s.b) s.b = 0.0f;
    if (s.c != s.c) s.c = 0.0f;
}

// ------------------------------------------------------------- init kernels
__device__ __forceinline__ void face_normal(const SurfArgs& a, int f)
{
    const int* F = a.faces + (size_t)f * a.fpe;
    w3 p0 = WP(a.x, a.y, a.z, F[0]), p1 = WP(a.x, a.y, a.z, F[1]), p2 = WP(a.x, a.y, a.z, F[a.fpe == 3 ? 2 : 3]);
    w3 n = wnormalize(wcross(wsub(p1, p0), wsub(p2, p0)));
    a.fnorm[3 * f] = n.x; a.fnorm[3 * f + 1] = n.y; a.fnorm[3 * f + 2] = n.z;
}
__global__ void k_surf_face_normals(SurfArgs a)
{
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f < a.nFaces) face_normal(a, f);
}

__global__ void k_surf_vertex_init(SurfArgs a)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= a.nS) return;
    // vertex normal: normalized sum of incident face normals (CCW order)
    w3 n = { 0.0f, 0.0f, 0.0f };
    for (int h = a.heRow[v]; h < a.heRow[v + 1]; ++h)
        if (a.heFace[h] != -1) n = wadd(n, W(a.fnorm + 3 * a.heFace[h]));
    n = wnormalize(n);
    a.vnorm[3 * v] = n.x; a.vnorm[3 * v + 1] = n.y; a.vnorm[3 * v + 2] = n.z;
    a.pinit[3 * v] = a.x[v]; a.pinit[3 * v + 1] = a.y[v]; a.pinit[3 * v + 2] = a.z[v];
    a.nn[v] = v;
    w3 pv = WP(a.x, a.y, a.z, v);
    const bool feat = a.isFeature[v] != 0;
    // 1D curve fit of feature vertices (Surface1D.cu:48-91)
    if (feat) {
        int nb[kMaxNeigh + 1], np = 0, vf = -1;
        nb[np++] = v;
        for (int h = a.heRow[v]; h < a.heRow[v + 1]; ++h) {
            int d = a.heTarget[h];
            if (a.isFeature[d] && np < kMaxNeigh) { nb[np++] = d; vf = d; }
        }
        if (vf >= 0) {
            w3 nrm = a.flat ? w3{ 0.0f, 0.0f, 1.0f } : n;
            w3 r = wsub(WP(a.x, a.y, a.z, vf), pv);
            if (wnorm(wcross(nrm, r)) < 10.0f * kSEps) r = { nrm.x, nrm.z, -nrm.y };
            w3 t1 = wcross(nrm, r), t2 = wcross(nrm, t1);
            nrm = wnormalize(nrm);
            t2 = wnormalize(t2);
            LSurf1 q;
            q.p0 = pv; q.e[0] = t2; q.e[1] = nrm;
            float ATA = 0.0f, ATb = 0.0f;
            for (int i = 0; i < np; ++i) {
                w3 p = wsub(WP(a.x, a.y, a.z, nb[i]), q.p0);
                float u = wdot(q.e[0], p), vv = wdot(q.e[1], p);
                ATb += u * u * vv;
                ATA += u * u * u * u;
            }
            q.a = ATb / ATA;
            reinterpret_cast<LSurf1*>(a.ls1)[v] = q;
        }
        // 1D eligibility: two feature neighbours, cos <= cos(160 deg)
        int nf = 0;
        w3 pp[2] = { { 0, 0, 0 }, { 0, 0, 0 } };
        for (int h = a.heRow[v]; h < a.heRow[v + 1]; ++h) {
            int d = a.heTarget[h];
            if (a.isFeature[d]) { if (nf < 2) pp[nf] = WP(a.x, a.y, a.z, d); ++nf; }
        }
        uint8_t ok = 0;
        if (nf == 2) {
            w3 ea = wsub(pp[0], pv), eb = wsub(pp[1], pv);
            float c = wdot(ea, eb) / sqrtf(wdot(ea, ea) * wdot(eb, eb));
            if (c <= a.cos160) ok = 1;
        }
        a.opt1d[v] = ok;
    } else {
        a.opt1d[v] = 0;
    }
    // quadric fit over {v} and its one-ring (Surface.cu:11-105); ring 2 adds
    // the one-ring's CCW targets not yet taken, neighbour by neighbour
    w3 pts[kMaxFitPoints + 1];
    int np = 0;
    pts[np++] = pv;
    for (int h = a.heRow[v]; h < a.heRow[v + 1] && np < kMaxNeigh; ++h) pts[np++] = WP(a.x, a.y, a.z, a.heTarget[h]);
    if (a.ring2) {
        int ids[kMaxFitPoints];
        int ni = 0;
        ids[ni++] = v;
        for (int h = a.heRow[v]; h < a.heRow[v + 1] && ni < np; ++h) ids[ni++] = a.heTarget[h];
        const int n1 = ni;
        bool over = false;
        for (int k = 1; k < n1 && !over; ++k) {
            const int d = ids[k];
            for (int h = a.heRow[d]; h < a.heRow[d + 1]; ++h) {
                const int t = a.heTarget[h];
                bool seen = false;
                for (int q = 0; q < ni && !seen; ++q) seen = ids[q] == t;
                if (seen) continue;
                if (ni == kMaxFitPoints) { over = true; break; }
                ids[ni++] = t;
                pts[np++] = WP(a.x, a.y, a.z, t);
            }
        }
        if (over) atomicOr(a.err, kSurfErrFitPoints);
    }
    if (np == 5) { pts[np] = wmul(0.5f, wadd(pts[2], pts[3])); ++np; }
    LSurf q;
    q.p0 = pts[0];
    int first = a.heTarget[a.heRow[v]];
    frame3(n, wsub(WP(a.x, a.y, a.z, first), pv), &q.e[0], &q.e[1], &q.e[2]);
    fit_quadric(q, pts, np);
    reinterpret_cast<LSurf*>(a.ls)[v] = q;
}

// number of sector surfaces of each feature vertex (k_countLocalSurfacesFeature)
__global__ void k_sector_count(SurfArgs a, int* cnt)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.nFeature) return;
    int v = a.nFree + i, c = 0;
    for (int h = a.heRow[v] + 1; h < a.heRow[v + 1]; ++h) if (a.isFeature[a.heTarget[h]]) ++c;
    if (!a.isB1D[v]) ++c;
    cnt[i] = c;
}

// Feature sectors of feature vertex v (the local surfaces of its smooth
// pieces between feature edges; reference SurfaceFeature.cu:134-223).  The
// CCW fan t_0 .. t_{n-1} of v is cut at every target t_k, k >= 1, that is a
// feature vertex.  Sector s holds v, its opening target (t_0 for sector 0,
// the previous cut target after that), the targets after it and its closing
// cut target.  On a closed fan (v not on a surface boundary) one more sector
// wraps from the last cut target round to t_0.  The table maps fan position
// k (< kTableSize) to the sector holding t_k after its opening target;
// position 0 maps to sector 0.  Targets after the last cut of an open fan
// belong to no sector: reported as an error.  Lists hold at most kMaxNeigh
// vertices.
__global__ void k_sector_lists(SurfArgs a, int* secN, int* secCnt)
{
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= a.nFeature) return;
    const int v = a.nFree + f;
    const int* fan = a.heTarget + a.heRow[v];
    const int n = a.heRow[v + 1] - a.heRow[v];
    const int first = a.frow[f], count = a.frow[f + 1] - first;
    int* tab = a.table + (size_t)kTableSize * f;
    for (int k = 0; k < kTableSize; ++k) tab[k] = -1;
    tab[0] = 0;
    // emit sector sec: v, fan[open], fan[open + 1 .. close) and closing target c
    auto emit = [&](int sec, int open, int close, int c) {
        int* list = secN + (size_t)kMaxNeigh * (first + sec);
        int len = 0;
        list[len++] = v;
        list[len++] = fan[open];
        for (int k = open + 1; k < close && len < kMaxNeigh; ++k) list[len++] = fan[k];
        if (len < kMaxNeigh) list[len++] = c;
        secCnt[first + sec] = len;
    };
    int sec = 0, open = 0;
    for (int k = 1; k < n; ++k) {
        if (sec >= count) {                       // past the last cut of an open fan
            atomicOr(a.err, kSurfErrUnsectored);
            break;
        }
        if (k < kTableSize) tab[k] = sec;
        if (a.isFeature[fan[k]]) {
            emit(sec, open, k, fan[k]);
            ++sec;
            open = k;
        }
    }
    if (!a.isB1D[v] && sec < count) emit(sec, open, n, fan[0]);
}

__global__ void k_sector_fit(SurfArgs a, const int* secN, const int* secCnt, int nSec)
{
    int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nSec) return;
    const int* L = secN + (size_t)kMaxNeigh * q;
    int np = secCnt[q];
    if (np < 2) return;   // not reached for closed surfaces
    int v = L[0];
    w3 pts[kMaxNeigh + 1];
    for (int i = 0; i < np; ++i) pts[i] = WP(a.x, a.y, a.z, L[i]);
    if (np == 5) { pts[np] = wmul(0.5f, wadd(pts[2], pts[3])); ++np; }
    w3 n = { 0.0f, 0.0f, 0.0f };
    for (int h = a.heRow[v]; h < a.heRow[v + 1]; ++h)
        if (a.heTarget[h] == L[1] && a.heFace[h] >= 0) n = W(a.fnorm + 3 * a.heFace[h]);
    LSurf s;
    s.p0 = pts[0];
    frame3(n, wsub(WP(a.x, a.y, a.z, L[1]), WP(a.x, a.y, a.z, v)), &s.e[0], &s.e[1], &s.e[2]);
    fit_quadric(s, pts, np);
    reinterpret_cast<LSurf*>(a.fs)[q] = s;
}

// nearest-neighbour walk over the initial surface positions within the
// vertex's feature class (k_updateNearestNeighbor)
__device__ void update_nn(const SurfArgs& a, int v)
{
    w3 p = WP(a.x, a.y, a.z, v);
    int vh = a.nn[v];
    w3 d0 = wsub(p, W(a.pinit + 3 * vh));
    float sq = wdot(d0, d0);
    const uint8_t fv = a.isFeature[v];
    int vnew;
    do {
        vnew = vh;
        int c = vh;
        for (int h = a.heRow[c]; h < a.heRow[c + 1]; ++h) {
            int dst = a.heTarget[h];
            if ((fv != 0) != (a.isFeature[dst] != 0)) continue;
            w3 dd = wsub(p, W(a.pinit + 3 * dst));
            float sd = wdot(dd, dd);
            if (sd < sq) { sq = sd; vh = dst; }
        }
    } while (vnew != vh);
    a.nn[v] = vnew;
}
__global__ void k_update_nn(SurfArgs a)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v < a.nS) update_nn(a, v);
}

// ------------------------------------------------------------- projection
// localSurfaceEstimationWithFeature: evaluate the nearest neighbour's quadric
// at (u,v), then blend with its projections onto each one-ring neighbour's
// surface (sector surfaces for feature neighbours), weights 1/(d^2 + eps).
// Two passes over the neighbours (weights, then the weighted sum); the
// arithmetic is the single-pass one.  Everything but (u,v) -- the fits, the
// nearest neighbours' initial positions and the sector choice -- is the same
// for all candidates of a search, so the searches stage it once in LDS
// (Proj2 / Proj1) and blend from there.

// position of surface vertex t at the start of the running colour pass
__device__ __forceinline__ w3 pass_start(const SurfArgs& a, int t)
{
    const bool own = t >= a.cLo && t < a.cHi;   // its class is being searched
    return WP(own ? a.sx : a.x, own ? a.sy : a.y, own ? a.sz : a.z, t);
}

// the surface a one-ring neighbour projects onto: the fit of its nearest
// neighbour nn, or for a feature nn the sector fit of the halfedge of nn whose
// target (snapshot position) is closest to vidPos
__device__ LSurf neighbour_fit(const SurfArgs& a, int nn, w3 vidPos)
{
    const LSurf* ls = reinterpret_cast<const LSurf*>(a.ls);
    if (!a.isFeature[nn]) return ls[nn];
    const int off = nn - a.nFree;
    float md = 3.40282347e+38f;
    int arg = 0, idx = 0;
    for (int h = a.heRow[nn]; h < a.heRow[nn + 1]; ++h, ++idx) {
        w3 t = wsub(pass_start(a, a.heTarget[h]), vidPos);
        float dd = wdot(t, t);
        if (dd < md) { md = dd; arg = idx; }
    }
    int sid = (arg < kTableSize) ? a.table[kTableSize * off + arg] : -1;
    const int nsec = a.frow[off + 1] - a.frow[off];
    if (sid < 0 || sid >= nsec) {
        // the reference asserts sid != -1 (SurfaceEstimation.h:172); here the
        // optimiser reports VSDMO_TOPOLOGY after the pass
        atomicOr(a.err, kSurfErrNoSector);
        sid = 0;
    }
    return nsec > 0 ? reinterpret_cast<const LSurf*>(a.fs)[a.frow[off] + sid] : ls[nn];
}

// the blend of the 2D projection over a source of L (the NN's fit), q0 (its
// initial position), nh, qn(i) (initial position of neighbour i's NN) and
// LN(i) (the surface neighbour i projects onto)
template <class Src>
__device__ w3 blend2(const Src& s, float u, float v)
{
    const LSurf L = s.L();
    const float w = poly(L, u, v);
    const w3 pw = l2w(L, u, v, w);
    const int nh = s.nh();
    float isum = 0.0f;
    {
        w3 d = wsub(s.q0(), pw);
        isum += 1.0f / (wdot(d, d) + kSEps);
    }
    for (int i = 0; i < nh; ++i) {
        w3 d = wsub(s.qn(i), pw);
        isum += 1.0f / (wdot(d, d) + kSEps);
    }
    const float ii = 1.0f / isum;
    w3 sum = { 0.0f, 0.0f, 0.0f };
    {
        w3 d = wsub(s.q0(), pw);
        float inv = 1.0f / (wdot(d, d) + kSEps);
        sum = wadd(sum, wmul(ii, wmul(inv, pw)));
    }
    for (int i = 0; i < nh; ++i) {
        w3 d = wsub(s.qn(i), pw);
        float inv = 1.0f / (wdot(d, d) + kSEps);
        const LSurf LN = s.LN(i);
        w3 q = wsub(pw, LN.p0);
        float lu = wdot(q, LN.e[0]), lv = wdot(q, LN.e[1]);
        float lw = poly(LN, lu, lv);
        sum = wadd(sum, wmul(ii, wmul(inv, l2w(LN, lu, lv, lw))));
    }
    return sum;
}

// 1D: the curve v = a u^2 of the NN's 1D fit, blended with the projections
// onto the curves of the listed feature neighbours' NNs
template <class Src>
__device__ w3 blend1(const Src& s, float u)
{
    const LSurf1 L = s.L();
    const float v = L.a * u * u;
    const w3 pw = wadd(wadd(L.p0, wmul(u, L.e[0])), wmul(v, L.e[1]));
    const int n = s.nh();
    float isum = 0.0f;
    {
        w3 d = wsub(s.q0(), pw);
        isum += 1.0f / (wdot(d, d) + kSEps);
    }
    for (int i = 0; i < n; ++i) {
        w3 d = wsub(s.qn(i), pw);
        isum += 1.0f / (wdot(d, d) + kSEps);
    }
    const float ii = 1.0f / isum;
    w3 sum = { 0.0f, 0.0f, 0.0f };
    {
        w3 d = wsub(s.q0(), pw);
        float inv = 1.0f / (wdot(d, d) + kSEps);
        sum = wadd(sum, wmul(ii, wmul(inv, pw)));
    }
    for (int i = 0; i < n; ++i) {
        w3 d = wsub(s.qn(i), pw);
        float inv = 1.0f / (wdot(d, d) + kSEps);
        const LSurf1 LN = s.LN(i);
        w3 q = wsub(pw, LN.p0);
        float lu = wdot(q, LN.e[0]);
        float lv = LN.a * lu * lu;
        sum = wadd(sum, wmul(ii, wmul(inv, wadd(wadd(LN.p0, wmul(lu, LN.e[0])), wmul(lv, LN.e[1])))));
    }
    return sum;
}

// staged (LDS) sources
struct alignas(16) Proj2 {
    LSurf L;
    LSurf LN[kMaxNeigh];
    float4 q[kMaxNeigh + 1];   // q0, then qn; w unused
    int n;
};
struct Proj2Src {
    const Proj2* c;
    __device__ w3 q(int i) const { const float4 t = c->q[i]; return { t.x, t.y, t.z }; }
    __device__ LSurf L() const { return c->L; }
    __device__ w3 q0() const { return q(0); }
    __device__ int nh() const { return c->n; }
    __device__ w3 qn(int i) const { return q(i + 1); }
    __device__ LSurf LN(int i) const { return c->LN[i]; }
};
struct Proj1 {
    LSurf1 L;
    w3 q0;
    int n;
    int nb[kMaxNeigh];
    w3 qn[kMaxNeigh];
    LSurf1 LN[kMaxNeigh];
};
struct Proj1Src {
    const Proj1* c;
    __device__ LSurf1 L() const { return c->L; }
    __device__ w3 q0() const { return c->q0; }
    __device__ int nh() const { return c->n; }
    __device__ w3 qn(int i) const { return c->qn[i]; }
    __device__ LSurf1 LN(int i) const { return c->LN[i]; }
};

// stage vid's 2D projection data: lane i < nh resolves one-ring neighbour i
// (its NN, that NN's initial position and fit / sector fit); all lanes call
// it, it ends with a barrier
__device__ void stage_proj2(const SurfArgs& a, int vid, w3 vidPos, Proj2* c)
{
    const int lane = threadIdx.x;
    const int h0 = a.heRow[vid];
    int nh = a.heRow[vid + 1] - h0;
    if (nh > kMaxNeigh) nh = kMaxNeigh;
    if (lane == 0) {
        const int n0 = a.nn[vid];
        c->L = reinterpret_cast<const LSurf*>(a.ls)[n0];
        const w3 q = W(a.pinit + 3 * n0);
        c->q[0] = { q.x, q.y, q.z, 0.0f };
        c->n = nh;
    }
    if (lane < nh) {
        const int nn = a.nn[a.heTarget[h0 + lane]];
        const w3 q = W(a.pinit + 3 * nn);
        c->q[lane + 1] = { q.x, q.y, q.z, 0.0f };
        c->LN[lane] = neighbour_fit(a, nn, vidPos);
    }
    __syncthreads();
}

// blend2 of the staged data, the same operations on the same values with two
// savings: 1 / x by recip_rn, and each of the first kBlendRegs weights computed
// once and kept for the second loop.  A position whose weights leave
// recip_rn's range (or NaN) takes blend2 itself.  The searches are bound by
// the issue of vector instructions: a triangle fan's vertex took 4,420, it
// takes 2,630 with this and FanScore's ratios (sphere of 55k vertices, one
// colour: 65.6 -> 41.0 us; quads of a 181^2 field 48.1 -> 35.3; the 2D passes
// of a 13^3 tet cube 16.2 -> 13.9).  The empty asm keeps the compiler from
// loading all neighbours' fits ahead of the levels (215 registers, and spills
// under any bound: 113 us); as it is it takes 52.
constexpr int kBlendRegs = 8;
__device__ __forceinline__ w3 blend2_staged(const Proj2* c, float u, float v)
{
    const Proj2Src s{ c };
    const int nh = uniform(c->n);
    asm volatile("" ::: "memory");
    const LSurf L = c->L;
    const w3 pw = l2w(L, u, v, poly(L, u, v));
    const auto weight = [&](int i) {
        const w3 d = wsub(s.q(i), pw);
        return recip_rn(wdot(d, d) + kSEps);
    };
    asm volatile("" ::: "memory");
    const float w0 = weight(0);
    float isum = w0, wmin = w0, w[kBlendRegs];
#pragma unroll
    for (int i = 0; i < kBlendRegs; ++i) {
        if (i >= nh) break;
        w[i] = weight(i + 1);
        isum += w[i];
        wmin = fminf(wmin, w[i]);
    }
    for (int i = kBlendRegs; i < nh; ++i) {
        const float t = weight(i + 1);
        isum += t;
        wmin = fminf(wmin, t);
    }
    // every x below 2^100 (a NaN or an infinity among them makes isum NaN)
    if (!(wmin > 0x1p-100f && isum < 0x1p100f)) return blend2(s, u, v);
    const float ii = recip_rn(isum);
    w3 sum = wadd(w3{ 0.0f, 0.0f, 0.0f }, wmul(ii, wmul(w0, pw)));
    const auto term = [&](int i, float wi) {
        const LSurf LN = c->LN[i];
        const w3 q = wsub(pw, LN.p0);
        const float lu = wdot(q, LN.e[0]), lv = wdot(q, LN.e[1]);
        return wmul(ii, wmul(wi, l2w(LN, lu, lv, poly(LN, lu, lv))));
    };
#pragma unroll
    for (int i = 0; i < kBlendRegs; ++i) {
        if (i >= nh) break;
        if (i % 2 == 0) asm volatile("" ::: "memory");
        sum = wadd(sum, term(i, w[i]));
    }
    for (int i = kBlendRegs; i < nh; ++i) sum = wadd(sum, term(i, weight(i + 1)));
    return sum;
}

// stage vid's 1D projection data: the curve neighbours -- feature neighbours
// that have exactly two feature neighbours themselves, in halfedge order -- are
// listed by the lanes, a halfedge of vid each, then lane i < n resolves
// neighbour i; all lanes call it, it ends with a barrier.  (One lane listed
// them, some 30 loads one after the other: 1.1-1.9 us of a colour's 9-13.)
__device__ void stage_proj1(const SurfArgs& a, int vid, Proj1* c)
{
    const LSurf1* ls1 = reinterpret_cast<const LSurf1*>(a.ls1);
    const int lane = threadIdx.x;
    const int h0 = a.heRow[vid], h1 = a.heRow[vid + 1];
    int cnt = 0;
    for (int b = h0; b < h1; b += 64) {
        bool take = false;
        int d = 0;
        if (b + lane < h1) {
            d = a.heTarget[b + lane];
            if (a.isFeature[d]) {
                const int e0 = a.heRow[d], e1 = a.heRow[d + 1];
                int k = 0;
                for (int e = e0; e < e1; e += 8) {   // loads together, the last one repeated past the row
                    int t[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) t[j] = a.heTarget[min(e + j, e1 - 1)];
#pragma unroll
                    for (int j = 0; j < 8; ++j) k += (a.isFeature[t[j]] && e + j < e1) ? 1 : 0;
                }
                take = k == 2;
            }
        }
        const unsigned long long bal = __ballot(take);
        const int at = cnt + __popcll(bal & ((1ull << lane) - 1ull));
        if (take && at < kMaxNeigh) c->nb[at] = d;
        cnt += __popcll(bal);
    }
    if (lane == 0) {
        c->n = min(cnt, kMaxNeigh);
        const int n0 = a.nn[vid];
        c->L = ls1[n0];
        c->q0 = W(a.pinit + 3 * n0);
    }
    __syncthreads();
    if (lane < c->n) {
        const int nn = a.nn[c->nb[lane]];
        c->qn[lane] = W(a.pinit + 3 * nn);
        c->LN[lane] = ls1[nn];
    }
    __syncthreads();
}

// unstaged source for single evaluations (surface sampling)
struct Proj2Global {
    const SurfArgs* a;
    int vid, h0, n;
    w3 vidPos;
    __device__ LSurf L() const { return reinterpret_cast<const LSurf*>(a->ls)[a->nn[vid]]; }
    __device__ w3 q0() const { return W(a->pinit + 3 * a->nn[vid]); }
    __device__ int nh() const { return n; }
    __device__ w3 qn(int i) const { return W(a->pinit + 3 * a->nn[a->heTarget[h0 + i]]); }
    __device__ LSurf LN(int i) const { return neighbour_fit(*a, a->nn[a->heTarget[h0 + i]], vidPos); }
};

__device__ w3 project2d(const SurfArgs& a, int vid, w3 vidPos, float u, float v)
{
    const int h0 = a.heRow[vid];
    int nh = a.heRow[vid + 1] - h0;
    if (nh > kMaxNeigh) nh = kMaxNeigh;
    return blend2(Proj2Global{ &a, vid, h0, nh, vidPos }, u, v);
}


// ------------------------------------------------------------- ring scores
struct HexRingLds { float cd[4], cF[4]; HexP hp[5]; };

struct RingFrame {
    float x0x, x0y, x0z, sg, is3, epsD, epsF, minDist, maxDist;
    int n;
    int nsub;   // p-dependent hex sub-tets scored: 5, or 4 without the principal-axes tet
    bool inRange;   // as hex_free_lanes returned it
};

// stage the volume one-ring of vid in LDS (same constants as the inner
// search) and return frame data; all lanes call it
__device__ RingFrame stage_ring(const SurfArgs& a, int vid, bool tet, void* lds, HexAcc* hacc)
{
    const int lane = threadIdx.x;
    RingFrame f;
    const int r0 = a.ringRow[vid];
    f.n = a.ringRow[vid + 1] - r0;
    f.x0x = a.x[vid]; f.x0y = a.y[vid]; f.x0z = a.z[vid];
    f.nsub = a.hexCorner8 ? 4 : 5;
    const int st = tet ? 3 : 7;
    float mabs = 0.0f, mn = FLT_MAX, mx = -FLT_MAX;
    for (int e = lane; e < f.n; e += 64) {
        const int* h = a.ringVal + (size_t)(r0 + e) * st;
        for (int t = 0; t < st; ++t) {
            int v = h[t];
            w3 d = { a.x[v] - f.x0x, a.y[v] - f.x0y, a.z[v] - f.x0z };
            mabs = fmaxf(mabs, fmaxf(fabsf(d.x), fmaxf(fabsf(d.y), fabsf(d.z))));
            float dist = wnorm(d);
            mn = fminf(mn, dist);
            mx = fmaxf(mx, dist);
        }
    }
    f.minDist = wave_min_u(mn); f.maxDist = wave_max_u(mx);
    f.sg = pow2_scale(wave_max_u(mabs));
    const float isg = 1.0f / f.sg;
    f.is3 = ((1.0f * isg) * isg) * isg;
    const float s2 = f.sg * f.sg, s3 = s2 * f.sg;
    f.epsD = kHexEps * s3; f.epsF = kHexEps * s2;
    for (int e = lane; e < f.n; e += 64) {
        const int* h = a.ringVal + (size_t)(r0 + e) * st;
        if (tet) {
            f3 p[3];
            for (int t = 0; t < 3; ++t) {
                int v = h[t];
                p[t] = { (a.x[v] - f.x0x) * f.sg, (a.y[v] - f.x0y) * f.sg, (a.z[v] - f.x0z) * f.sg };
            }
            reinterpret_cast<TetC*>(lds)[e] = tet_consts(p[0], p[1], p[2]);
        } else {
            f3 r[8];
            r[0] = { 0.0f, 0.0f, 0.0f };
            for (int t = 0; t < 7; ++t) {
                int v = h[t];
                r[t + 1] = { (a.x[v] - f.x0x) * f.sg, (a.y[v] - f.x0y) * f.sg, (a.z[v] - f.x0z) * f.sg };
            }
            HexRingLds L;
            hex_consts(r, L.cd, L.cF, L.hp);
            reinterpret_cast<HexRingLds*>(lds)[e] = L;
        }
    }
    __syncthreads();
    f.inRange = false;
    if (!tet) {
        HexAcc acc = hex_acc0();
        f.inRange = hex_free_lanes(reinterpret_cast<const HexRingLds*>(lds), f.n, acc);
        *hacc = acc;
    }
    return f;
}

// the p-dependent hex sub-tets of the ring at one point, NS per element (5:
// the nine-tet metric, 4: eight corners; a compile-time count keeps the
// element loop free of the metric branch)
template <int NS>
__device__ __forceinline__ void ring_hex_add(HexAcc& acc, const HexRingLds* L, int n, float px, float py, float pz)
{
    const float Q1 = fmaf(pz, pz, py * py), Q3 = 3.0f * Q1, t3 = 3.0f * px;
    for (int e = 0; e < n; ++e)
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const HexP h = L[e].hp[s];
            const bool a3 = (s == 1 || s == 4);
            float Tyz = fmaf(h.gy, py, fmaf(h.gz, pz, h.D));
            float Ryz = fmaf(h.sy, py, fmaf(h.sz, pz, h.K + (a3 ? Q3 : Q1)));
            hex_acc_add(acc, fmaf(h.gx, px, Tyz), fmaf(px, (a3 ? t3 : px) + h.sx, Ryz));
        }
}

__device__ float ring_score(const RingFrame& f, bool tet, const void* lds, const HexAcc& hacc, w3 p)
{
    const float px = (p.x - f.x0x) * f.sg, py = (p.y - f.x0y) * f.sg, pz = (p.z - f.x0z) * f.sg;
    if (tet) {
        const TetC* tc = reinterpret_cast<const TetC*>(lds);
        const float Qyz = 3.0f * fmaf(pz, pz, py * py);
        const float t3 = 3.0f * px;
        TetAcc acc = tet_acc0();
        for (int e = 0; e < f.n; ++e) {
            const TetC c = tc[e];
            float Tyz = fmaf(c.nny, py, fmaf(c.nnz, pz, c.D));
            float Ryz = fmaf(c.m2sy, py, fmaf(c.m2sz, pz, c.K + Qyz));
            tet_acc_add(acc, fmaf(c.nnx, px, Tyz), fmaf(px, t3 + c.m2sx, Ryz));
        }
        return tet_acc_score(acc, f.is3);
    }
    const HexRingLds* L = reinterpret_cast<const HexRingLds*>(lds);
    HexAcc acc = hacc;
    if (f.nsub == 4) ring_hex_add<4>(acc, L, f.n, px, py, pz);
    else ring_hex_add<5>(acc, L, f.n, px, py, pz);
    return hex_acc_score(acc, f.epsD, f.epsF);
}

// ------------------------------------------------------------- search bodies
// Scorers: score(p) is what the search maximises (one candidate per lane);
// start(p0, qs, qref) gives the start position's score and the reference the
// last level's maximum must beat for the write (all lanes call it).

// volume one-ring of a tet / hex surface vertex
struct VolScore {
    RingFrame f;
    bool tet;
    const void* lds;
    HexAcc hacc;
    __device__ float score(w3 p) const { return ring_score(f, tet, lds, hacc, p); }
    static constexpr int kLanes = 1;
    __device__ float score_lanes(w3 p) const { return score(p); }
    // start score (maximised from) and the reference the last level must beat
    // (p is the frame's origin): the ring's pairs on the wave's lanes, where
    // every lane went through the whole ring (one colour's 2D pass of a 31^3 hex
    // cube 18.0 -> 16.9 us, with the DPP reductions)
    __device__ void start(w3 p, float& qs, float& qref) const
    {
        if (!tet) {
            qs = hex_start_lanes(reinterpret_cast<const HexRingLds*>(lds), f.n, f.nsub == 4, hacc, f.inRange, f.epsD, f.epsF);
        } else {
            const bool have = (int)threadIdx.x < f.n;
            const TetC& c = reinterpret_cast<const TetC*>(lds)[have ? threadIdx.x : 0];
            if (f.n > 64 || !tet_lanes_score(have, c.D, c.K, f.is3, qs)) qs = score(p);
        }
        qref = qs;
    }
};

// fan of a surface-mesh vertex (DMOQualityTri.h:257-275, DMOQualityQuad.h:
// 30-50): triangles (p, r_k, r_k+1), quads (p, r_k, d_k, r_k+1); score()
// signs each element by the nearest neighbour's vertex normal n, final_ref()
// uses the unsigned metric
template <int CTRL>
__device__ __forceinline__ float lane_swap(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
template <bool QUAD>
struct FanScore {
    const w3* pts;
    // per element, what no candidate changes: triangles (r_k+1, |e2|^2);
    // quads (e1, |e1|^2), (e2, |e2|^2), (r_k+1, -)
    const float4* cst;
    int ne;
    w3 n;
    bool unitN;   // |n| within 1 %, or 0
    __device__ float elem(w3 p, int k, bool oriented) const
    {
        const f3 nn = { n.x, n.y, n.z };
        const f3* no = oriented ? &nn : nullptr;
        const f3 q = { p.x, p.y, p.z };
        if (QUAD) {
            const w3 a = pts[2 * k], b = pts[2 * k + 1], c = pts[2 * k + 2];
            return mr_quad3(q, f3{ a.x, a.y, a.z }, f3{ b.x, b.y, b.z }, f3{ c.x, c.y, c.z }, no);
        }
        const w3 a = pts[k], b = pts[k + 1];
        return mr_tri3(q, f3{ a.x, a.y, a.z }, f3{ b.x, b.y, b.z }, no);
    }
    __device__ void elem2(w3 p, int k, float& qs, float& qu) const
    {
        const f3 nn = { n.x, n.y, n.z };
        const f3 q = { p.x, p.y, p.z };
        if (QUAD) {
            const w3 a = pts[2 * k], b = pts[2 * k + 1], c = pts[2 * k + 2];
            mr_quad3_both(q, f3{ a.x, a.y, a.z }, f3{ b.x, b.y, b.z }, f3{ c.x, c.y, c.z }, nn, qs, qu);
        } else {
            const w3 a = pts[k], b = pts[k + 1];
            mr_tri3_both(q, f3{ a.x, a.y, a.z }, f3{ b.x, b.y, b.z }, nn, qs, qu);
        }
    }
    // the minimum over the fan.  The elements' qualities are first compared by
    // ratios that need no square root, unit normal or division of their own
    // (of exactly the values that the metric would use), and the metric's last
    // steps are done once, for the smallest: rounding is monotonic, so its
    // value is the minimum of the rounded ones.  Where an element's sign, the
    // smallest element or the range of a value is not certain, the lane
    // evaluates every element instead.  The metric spent 110 instructions on a
    // triangle, 36 of them in the unit normal's divisions and 25 in the root
    // and the quotient; this takes 42.
    __device__ float score(w3 p) const
    {
        float r1 = 0x1p126f, r2 = 0x1p126f, sA = 0.0f, sB = 0.0f, sl = 1.0f;
        bool unsure = !unitN, fail = false;
        const w3 f = pts[0];
        w3 e0 = wsub(f, p);
        float d0 = wdot(e0, e0);
        for (int k = 0; k < ne; ++k) {
            float key, l, A, Bq = 0.0f;
            if (QUAD) {
                const float4 c1 = cst[3 * k], c2 = cst[3 * k + 1], c3 = cst[3 * k + 2];
                const w3 e1 = { c1.x, c1.y, c1.z }, e2 = { c2.x, c2.y, c2.z };
                const w3 g = wsub(w3{ c3.x, c3.y, c3.z }, p);   // -e3
                const float d3 = wdot(g, g);
                l = ((d0 + c1.w) + c2.w) + d3;
                // e1 x -e0 and e3 x -e2
                const w3 N1 = wcross(e0, e1), N2 = wcross(g, e2);
                A = wdot(N1, N1);
                Bq = wdot(N2, N2);
                const float t1 = fdot(N1), t2 = fdot(N2);
                // n . unit(N) against 0.7, both sides squared
                const float lo = 0.49f * (1.0f - 0x1p-16f), hi = 0.49f * (1.0f + 0x1p-16f);
                const bool f1 = t1 < 0.0f || t1 * t1 < lo * A, f2 = t2 < 0.0f || t2 * t2 < lo * Bq;
                const bool ok1 = t1 > 0.0f && t1 * t1 > hi * A, ok2 = t2 > 0.0f && t2 * t2 > hi * Bq;
                const bool inA = A > 0x1p-96f && A < 0x1p100f, inB = Bq > 0x1p-96f && Bq < 0x1p100f;
                fail = fail || (inA && f1) || (inB && f2);
                unsure = unsure || !(inA && inB && ok1 && ok2);
                key = (__builtin_amdgcn_sqrtf(A) + __builtin_amdgcn_sqrtf(Bq)) * __builtin_amdgcn_rcpf(l);
                unsure = unsure || !(key > 0x1p-60f);
                e0 = g;
                d0 = d3;
            } else {
                const float4 c = cst[k];
                const w3 e1 = wsub(w3{ c.x, c.y, c.z }, p);
                const float d1 = wdot(e1, e1);
                l = (d0 + d1) + c.w;
                const w3 N = wcross(e0, e1);
                A = wdot(N, N);
                const float t = fdot(N);
                // both signs of n . unit(N) and of the rounded t agree beyond
                // 8 ulp of |N| |n|
                unsure = unsure || !(t * t > 0x1p-36f * A && A > 0x1p-96f);
                key = A * __builtin_amdgcn_rcpf(l * l);
                unsure = unsure || !(key > 0x1p-60f);
                key = __builtin_copysignf(key, t);
                e0 = e1;
                d0 = d1;
            }
            r2 = __builtin_amdgcn_fmed3f(r1, r2, key);
            const bool take = key < r1;
            r1 = take ? key : r1;
            sA = take ? A : sA;
            if (QUAD) sB = take ? Bq : sB;
            sl = take ? l : sl;
        }
        if (QUAD && unitN && fail) return -1.0f;
        // the metric's roundings and the ratios' own stay below 2^-20 of the key
        unsure = unsure || !(r2 - r1 > 0x1p-18f * (fabsf(r1) + fabsf(r2)));
        if (!unsure) {
            if (QUAD) return (2.0f * (sqrt_rn(sA) + sqrt_rn(sB))) / sl;
            return (kTwoSqrt3 * __builtin_copysignf(sqrt_rn(sA), r1)) / sl;
        }
        float q = FLT_MAX;
        for (int k = 0; k < ne; ++k) q = fminf(q, elem(p, k, true));
        return q;
    }
    __device__ __forceinline__ float fdot(w3 N) const { return fmaf(N.z, n.z, fmaf(N.y, n.y, N.x * n.x)); }
    // the same minimum for a position that eight lanes hold, an element per
    // lane: a 1D search has 8 candidates and left 56 lanes idle (sphere of 55k
    // vertices, one colour: 16.6 -> 10.4 us)
    static constexpr int kLanes = 8;
    __device__ float score_lanes(w3 p) const
    {
        float q = FLT_MAX;
        for (int k = threadIdx.x % kLanes; k < ne; k += kLanes) q = fminf(q, elem(p, k, true));
        q = fminf(q, lane_swap<0xB1>(q));    // lane ^ 1
        q = fminf(q, lane_swap<0x4E>(q));    // lane ^ 2
        return fminf(q, lane_swap<0x141>(q));   // 7 - lane within each eight
    }
    // lane k < ne evaluates fan element k signed and unsigned; two wave
    // min-reductions (fminf is exact, so the order does not matter)
    __device__ void start(w3 p, float& qs, float& qref) const
    {
        const int k = threadIdx.x;
        float s = FLT_MAX, u = FLT_MAX;
        if (k < ne) elem2(p, k, s, u);
        qs = wave_min_u(s);
        qref = wave_min_u(u);
    }
};

// fan of a flat triangle mesh's boundary vertex in the canonical 2D
// evaluation (frame of the start position x0, scale sg)
struct FlatScore {
    const TriC* tc;
    int ne;
    w3 x0;
    float sg, is2;
    __device__ float score(w3 q) const
    {
        const float px = (q.x - x0.x) * sg, py = (q.y - x0.y) * sg;
        const float Q2 = 2.0f * (py * py);
        const float t2 = 2.0f * px;
        TriAcc acc = tri_acc0();
        for (int e = 0; e < ne; ++e) {
            const TriC c = tc[e];
            float Ty = fmaf(c.gy, py, c.C);
            float Ry = fmaf(c.sy, py, c.K + Q2);
            tri_acc_add(acc, fmaf(c.gx, px, Ty), fmaf(px, t2 + c.sx, Ry));
        }
        return tri_acc_score(acc, is2);
    }
    static constexpr int kLanes = 1;
    __device__ float score_lanes(w3 p) const { return score(p); }
    __device__ void start(w3 p, float& qs, float& qref) const { qs = score(p); qref = qs; }
};

// 2D search on the blended local surfaces.  Lane l holds reference thread
// t = l/2's candidate A (l even) or B (l odd): A = (t/nq, t%nq), B = (t/nq +
// nq/2, t%nq); the surface kernels keep A on an exact tie, so A ranks first.
// Window half-width s_d * dist in the nearest neighbour's (u,v).
template <class S>
__device__ void surf2d_search(const SurfArgs& a, int vid, w3 vidPos, float dist, int nq, const S& sc)
{
    const int lane = threadIdx.x;
    __shared__ Proj2 s_proj;
    stage_proj2(a, vid, vidPos, &s_proj);
    const LSurf L = s_proj.L;
    w3 cur = vidPos;
    const w3 cvec = wsub(cur, L.p0);
    float cu = wdot(L.e[0], cvec), cv = wdot(L.e[1], cvec);
    float qcur, qold;
    sc.start(cur, qcur, qold);
    float qlast = -FLT_MAX;
    const int t = lane >> 1;
    const bool isB = (lane & 1) != 0;
    const bool active = t < nq * nq / 2;
    const int ci = t / nq + (isB ? nq / 2 : 0), cj = t % nq;
    float ds = a.gridScale;
    for (int d = 0; d < a.depth; ++d) {
        const float uMax = ds * dist, uMin = -(ds * dist);
        float best = -FLT_MAX;
        float u = 0.0f, v = 0.0f;
        w3 pc = { 0.0f, 0.0f, 0.0f };
        if (active) {
            u = cu + a.aff * ((float)ci * uMin + (float)(nq - 1 - ci) * uMax);
            v = cv + a.aff * ((float)cj * uMin + (float)(nq - 1 - cj) * uMax);
            pc = blend2_staged(&s_proj, u, v);
            best = sc.score(pc);
        }
        const float own = best;
        best = wave_max_u(own);
        if (qcur < best) {
            // the winner's projected point (the projection of (bu, bv))
            const int wl = __builtin_ctzll(__ballot(own == best));
            cu = lane_f(u, wl); cv = lane_f(v, wl);
            cur = { lane_f(pc.x, wl), lane_f(pc.y, wl), lane_f(pc.z, wl) };
            qcur = best;
        }
        qlast = best;
        ds = ds * a.shrink;
    }
    if (qold < qlast && lane == 0) { a.xw[vid] = cur.x; a.yw[vid] = cur.y; a.zw[vid] = cur.z; }
}

// 1D search along the feature curve: lanes S::kLanes * i and on hold candidate
// i < nq; the curve projection blends the fits of the curve neighbours
template <class S>
__device__ void surf1d_search(const SurfArgs& a, int vid, w3 vidPos, float dist, int nq, const S& sc)
{
    const int lane = threadIdx.x;
    __shared__ Proj1 s_proj;
    stage_proj1(a, vid, &s_proj);
    const Proj1Src ps{ &s_proj };
    const LSurf1 L = s_proj.L;
    w3 cur = vidPos;
    const w3 cvec = wsub(cur, L.p0);
    float cu = wdot(L.e[0], cvec);
    float qcur, qold;
    sc.start(cur, qcur, qold);
    float qlast = -FLT_MAX;
    const int ci = lane / S::kLanes;
    const bool active = ci < nq;
    float ds = a.gridScale;
    for (int d = 0; d < a.depth; ++d) {
        const float uMax = ds * dist, uMin = -(ds * dist);
        float best = -FLT_MAX, u = 0.0f;
        w3 pc = { 0.0f, 0.0f, 0.0f };
        if (active) {
            u = cu + a.aff * ((float)ci * uMin + (float)(nq - 1 - ci) * uMax);
            pc = blend1(ps, u);
            best = sc.score_lanes(pc);
        }
        const float own = best;
        best = wave_max_u(own);
        if (qcur < best) {
            const int wl = __builtin_ctzll(__ballot(own == best));
            cu = lane_f(u, wl);
            cur = { lane_f(pc.x, wl), lane_f(pc.y, wl), lane_f(pc.z, wl) };
            qcur = best;
        }
        qlast = best;
        ds = ds * a.shrink;
    }
    if (qold < qlast && lane == 0) { a.xw[vid] = cur.x; a.yw[vid] = cur.y; a.zw[vid] = cur.z; }
}

// ------------------------------------------------- tet / hex surface searches
// Window half-width: s_d * (min distance to the ring points for hexes, max
// for tets).  (k_optimizeHierarchical2DTet/Hex, 1DTet/Hex)
__global__ __launch_bounds__(64) void k_search_surf2d(SurfArgs a, int cStart, int nq, int tet)
{
    extern __shared__ float s_lds[];
    const int vid = cStart + blockIdx.x;
    VolScore sc;
    sc.hacc = hex_acc0();
    sc.f = stage_ring(a, vid, tet != 0, s_lds, &sc.hacc);
    if (sc.f.n <= 0) return;
    sc.tet = tet != 0;
    sc.lds = s_lds;
    surf2d_search(a, vid, w3{ sc.f.x0x, sc.f.x0y, sc.f.x0z }, tet ? sc.f.maxDist : sc.f.minDist, nq, sc);
}

__global__ __launch_bounds__(64) void k_search_feat1d(SurfArgs a, int cStart, int nq, int tet)
{
    extern __shared__ float s_lds[];
    const int vid = cStart + blockIdx.x;
    if (!a.opt1d[vid]) return;   // uniform over the block
    VolScore sc;
    sc.hacc = hex_acc0();
    sc.f = stage_ring(a, vid, tet != 0, s_lds, &sc.hacc);
    if (sc.f.n <= 0) return;
    sc.tet = tet != 0;
    sc.lds = s_lds;
    surf1d_search(a, vid, w3{ sc.f.x0x, sc.f.x0y, sc.f.x0z }, tet ? sc.f.maxDist : sc.f.minDist, nq, sc);
}

// ------------------------------------------------ surface-mesh (tri / quad)
// Stage the fan of vid in LDS: lane i < n loads the halfedge target r_i (and
// for quads the diagonal d_i, the target of the halfedge after vid -> r_i in
// its face); closed (r_n = r_0) unless open.  Returns false (uniformly) when
// the vertex has no fan element.  dist: the largest distance from vid to the
// r_i (and d_i).  The d_i are start-of-pass positions: on a surface boundary
// the "diagonal" of the boundary halfedge is the boundary neighbour of the
// next boundary vertex, which can be in the colour class being updated;
// every other fan vertex shares an element with vid, so it does not move.
template <bool QUAD>
struct FanLds {
    float4 cst[(QUAD ? 3 : 1) * kMaxNeigh];
    w3 pts[(QUAD ? 2 : 1) * kMaxNeigh + 1];
};
template <bool QUAD>
__device__ bool stage_fan(const SurfArgs& a, int vid, bool open, FanLds<QUAD>& lds, FanScore<QUAD>& sc, float& dist)
{
    const int lane = threadIdx.x;
    const int h0 = a.heRow[vid], n = a.heRow[vid + 1] - h0;
    if (n <= 0 || n > kMaxNeigh) return false;
    const w3 x0 = WP(a.x, a.y, a.z, vid);
    const int K = QUAD ? 2 : 1;
    w3* pts = lds.pts;
    float mx = -FLT_MAX;
    if (lane < n) {
        const int h = h0 + lane;
        const w3 r = WP(a.x, a.y, a.z, a.heTarget[h]);
        pts[K * lane] = r;
        mx = wnorm(wsub(r, x0));
        if (QUAD) {
            const int nx = a.heNext[h];
            const w3 dg = pass_start(a, a.heTarget[nx >= 0 ? nx : h]);
            pts[K * lane + 1] = dg;
            mx = fmaxf(mx, wnorm(wsub(dg, x0)));
        }
    }
    if (lane == 0 && !open) pts[K * n] = WP(a.x, a.y, a.z, a.heTarget[h0]);
    __syncthreads();
    sc.pts = pts;
    sc.cst = lds.cst;
    sc.ne = open ? n - 1 : n;
    sc.n = W(a.vnorm + 3 * a.nn[vid]);
    const float nn = wdot(sc.n, sc.n);
    sc.unitN = nn < 1.02f && (nn > 0.98f || nn == 0.0f);
    dist = wave_max_u(mx);
    if (lane < sc.ne) {
        const w3 r = pts[K * (lane + 1)], a0 = pts[K * lane];
        if (QUAD) {
            const w3 dg = pts[2 * lane + 1];
            const w3 e1 = wsub(dg, a0), e2 = wsub(r, dg);
            lds.cst[3 * lane] = { e1.x, e1.y, e1.z, wdot(e1, e1) };
            lds.cst[3 * lane + 1] = { e2.x, e2.y, e2.z, wdot(e2, e2) };
            lds.cst[3 * lane + 2] = { r.x, r.y, r.z, 0.0f };
        } else {
            const w3 e2 = wsub(r, a0);
            lds.cst[lane] = { r.x, r.y, r.z, wdot(e2, e2) };
        }
    }
    __syncthreads();
    return sc.ne > 0;
}

// free vertices: 2D search, fan always closed (k_optimizeHierarchical2D,
// DMOTriImplCub.h:25-200, DMOQuadImplCub.h:23-212)
template <bool QUAD>
__global__ __launch_bounds__(64) void k_search_fan2d(SurfArgs a, int cStart, int nq)
{
    __shared__ FanLds<QUAD> s_fan;
    const int vid = cStart + blockIdx.x;
    FanScore<QUAD> sc;
    float dist;
    if (!stage_fan<QUAD>(a, vid, false, s_fan, sc, dist)) return;
    surf2d_search(a, vid, WP(a.x, a.y, a.z, vid), dist, nq, sc);
}

// feature vertices: 1D search, fan open on a surface boundary
// (k_optimizeHierarchical1D, DMOTriImplCub.h:205-378, DMOQuadImplCub.h:216-402)
template <bool QUAD>
__global__ __launch_bounds__(64) void k_search_fan1d(SurfArgs a, int cStart, int nq)
{
    __shared__ FanLds<QUAD> s_fan;
    const int vid = cStart + blockIdx.x;
    if (!a.opt1d[vid]) return;   // uniform over the block
    FanScore<QUAD> sc;
    float dist;
    if (!stage_fan<QUAD>(a, vid, a.isB1D[vid] != 0, s_fan, sc, dist)) return;
    surf1d_search(a, vid, WP(a.x, a.y, a.z, vid), dist, nq, sc);
}

// after a surface mesh's passes: the nearest-neighbour walk (the first nbS
// blocks) and the face normals, both from the final positions
__global__ __launch_bounds__(256) void k_nn_face_normals(SurfArgs a, int nbS)
{
    const int b = (int)blockIdx.x, t = (int)threadIdx.x;
    if (b < nbS) {
        const int v = b * 256 + t;
        if (v < a.nS) update_nn(a, v);
    } else {
        const int f = (b - nbS) * 256 + t;
        if (f < a.nFaces) face_normal(a, f);
    }
}

// vertex normals from the current face normals (k_calcVertexNormals)
__global__ void k_surf_vertex_normals(SurfArgs a)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= a.nS) return;
    w3 n = { 0.0f, 0.0f, 0.0f };
    for (int h = a.heRow[v]; h < a.heRow[v + 1]; ++h)
        if (a.heFace[h] != -1) n = wadd(n, W(a.fnorm + 3 * a.heFace[h]));
    n = wnormalize(n);
    a.vnorm[3 * v] = n.x; a.vnorm[3 * v + 1] = n.y; a.vnorm[3 * v + 2] = n.z;
}

// positions snapshot before the surface passes (one launch for x, y, z)
__global__ void k_snapshot(const float* x, const float* y, const float* z, float* sx, float* sy, float* sz, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    sx[i] = x[i]; sy[i] = y[i]; sz[i] = z[i];
}

// Laplace smoothing of one colour class of free surface vertices
// (k_laplaceSmoothing, Laplace.cu:8-28): p <- (p + sum of the halfedge
// targets) * (1 / (1 + n))
__global__ void k_laplace(float* x, float* y, float* z, const int* heRow, const int* heTarget, int lo, int hi)
{
    int v = lo + blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= hi) return;
    const int h0 = heRow[v], n = heRow[v + 1] - h0;
    w3 q = WP(x, y, z, v);
    for (int h = h0; h < h0 + n; ++h) q = wadd(q, WP(x, y, z, heTarget[h]));
    q = wmul(1.0f / (float)(1 + n), q);
    x[v] = q.x; y[v] = q.y; z[v] = q.z;
}

// ------------------------------------------------------ 1D flat boundary search
// Boundary vertices of a flat triangle mesh follow their boundary curve
// (k_optimizeHierarchical1DFlat): the ring is the halfedge fan (closed only
// off a surface boundary), the window half-width is s_d times the largest
// Euclidean distance to the fan, and candidates are scored by the 2D mean
// ratio of the fan triangles in the frame of the start position.
__global__ __launch_bounds__(64) void k_search_flat1d(SurfArgs a, int cStart, int nq)
{
    __shared__ TriC s_tr[kMaxNeigh];
    const int lane = threadIdx.x;
    const int vid = cStart + blockIdx.x;
    if (!a.opt1d[vid]) return;   // uniform over the block
    const int h0 = a.heRow[vid], n = a.heRow[vid + 1] - h0;
    const int nOne = n + (a.isB1D[vid] ? 0 : 1);
    if (n <= 0 || nOne < 2 || n > kMaxNeigh) return;
    const w3 x0 = WP(a.x, a.y, a.z, vid);
    float mabs = 0.0f, mx = -FLT_MAX;
    if (lane < n) {
        w3 d = wsub(WP(a.x, a.y, a.z, a.heTarget[h0 + lane]), x0);
        mabs = fmaxf(fabsf(d.x), fabsf(d.y));
        mx = wnorm(d);
    }
    mabs = wave_max_u(mabs);
    mx = wave_max_u(mx);
    const float sg = pow2_scale(mabs);
    const float isg = 1.0f / sg;
    const float is2 = (1.0f * isg) * isg;
    const int ne = nOne - 1;
    if (lane < ne) {
        const int va = a.heTarget[h0 + lane], vb = a.heTarget[h0 + (lane + 1 == n ? 0 : lane + 1)];
        s_tr[lane] = tri_consts((a.x[va] - x0.x) * sg, (a.y[va] - x0.y) * sg, (a.x[vb] - x0.x) * sg, (a.y[vb] - x0.y) * sg);
    }
    __syncthreads();
    surf1d_search(a, vid, x0, mx, nq, FlatScore{ s_tr, ne, x0, sg, is2 });
}

// ------------------------------------------------------- surface sampling
// Points of vid's local surfaces on an nu x nv grid (k_fillEstimateLocalSurfacePoints
// with USE_SURF_OF_NN = false, DMOCommon.h:197-276; k_fillLocalSurfacePoints,
// DMOCommon.cu:73-150): idx = i*nu + j.  mode 0 blends the projections
// (window s * maxDist), mode 1 evaluates the NN's fit or its sector fit sid
// (window 2 s * maxDist).  One thread per point.
__global__ void k_surface_points(SurfArgs a, int vid, int nu, int nv, int mode, int sid, float* out)
{
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nu * nv) return;
    const w3 pv = WP(a.x, a.y, a.z, vid);
    float mx = -FLT_MAX;
    for (int h = a.heRow[vid]; h < a.heRow[vid + 1]; ++h) mx = fmaxf(mx, wnorm(wsub(WP(a.x, a.y, a.z, a.heTarget[h]), pv)));
    const int nn = a.nn[vid];
    LSurf L = reinterpret_cast<const LSurf*>(a.ls)[nn];
    if (mode == 1 && nn >= a.nFree) {
        int off = nn - a.nFree, nsec = a.frow[off + 1] - a.frow[off];
        if (sid >= nsec) sid = nsec - 1;
        if (nsec > 0 && sid >= 0) L = reinterpret_cast<const LSurf*>(a.fs)[a.frow[off] + sid];
    }
    const w3 c = wsub(pv, L.p0);
    const float cu = wdot(L.e[0], c), cv = wdot(L.e[1], c);
    float uMax = a.gridScale * mx, uMin = -(a.gridScale * mx);
    if (mode == 1) { uMax *= 2.0f; uMin *= 2.0f; }
    const float au = 1.0f / (float)(nu - 1), av = 1.0f / (float)(nv - 1);
    const int j = idx % nu, i = idx / nu;
    const float u = cu + au * ((float)i * uMin + (float)(nu - 1 - i) * uMax);
    const float v = cv + av * ((float)j * uMin + (float)(nv - 1 - j) * uMax);
    const w3 q = (mode == 0) ? project2d(a, vid, pv, u, v) : l2w(L, u, v, poly(L, u, v));
    out[3 * idx] = q.x; out[3 * idx + 1] = q.y; out[3 * idx + 2] = q.z;
}

// ------------------------------------------------------------- launchers
static inline int nb256(long long n) { return (int)((n + 255) / 256 > 0 ? (n + 255) / 256 : 1); }

size_t surf_lds_bytes(int elem, int maxRing)
{
    size_t per = (elem == VSDMO_TET) ? sizeof(TetC) : sizeof(HexRingLds);
    return per * (size_t)(maxRing > 0 ? maxRing : 1);
}

void surf_init_launch(const SurfArgs& a, hipStream_t s)
{
    k_surf_face_normals<<<nb256(a.nFaces), 256, 0, s>>>(a);
    k_surf_vertex_init<<<nb256(a.nS), 256, 0, s>>>(a);
}
void surf_sector_count_launch(const SurfArgs& a, int* cnt, hipStream_t s)
{
    k_sector_count<<<nb256(a.nFeature), 256, 0, s>>>(a, cnt);
}
void surf_sector_launch(const SurfArgs& a, int* secN, int* secCnt, int nSec, hipStream_t s)
{
    k_sector_lists<<<nb256(a.nFeature), 256, 0, s>>>(a, secN, secCnt);
    if (nSec > 0) k_sector_fit<<<nb256(nSec), 256, 0, s>>>(a, secN, secCnt, nSec);
}
void surf_nn_launch(const SurfArgs& a, hipStream_t s)
{
    k_update_nn<<<nb256(a.nS), 256, 0, s>>>(a);
}
static SurfArgs of_class(const SurfArgs& a, int cStart, int cEnd)
{
    SurfArgs c = a;
    c.cLo = cStart; c.cHi = cEnd;
    return c;
}
void surf_search2d_launch(const SurfArgs& a, int cStart, int cEnd, int nq, int tet, size_t lds, hipStream_t s)
{
    if (cEnd > cStart) k_search_surf2d<<<cEnd - cStart, 64, lds, s>>>(of_class(a, cStart, cEnd), cStart, nq, tet);
}
void surf_search1d_launch(const SurfArgs& a, int cStart, int cEnd, int nq, int tet, size_t lds, hipStream_t s)
{
    if (cEnd > cStart) k_search_feat1d<<<cEnd - cStart, 64, lds, s>>>(a, cStart, nq, tet);
}
void surf_points_launch(const SurfArgs& a, int vid, int nu, int nv, int mode, int sid, float* out, hipStream_t s)
{
    const int n = nu * nv;
    if (n > 0) k_surface_points<<<(n + 63) / 64, 64, 0, s>>>(a, vid, nu, nv, mode, sid, out);
}
void surf_flat1d_launch(const SurfArgs& a, int cStart, int cEnd, int nq, hipStream_t s)
{
    if (cEnd > cStart) k_search_flat1d<<<cEnd - cStart, 64, 0, s>>>(a, cStart, nq);
}
void surf_fan2d_launch(const SurfArgs& a, int cStart, int cEnd, int nq, hipStream_t s)
{
    if (cEnd <= cStart) return;
    const SurfArgs c = of_class(a, cStart, cEnd);
    if (a.fpe == 4) launch_kernel(k_search_fan2d<true>, cEnd - cStart, 64, 0, s, c, cStart, nq);
    else launch_kernel(k_search_fan2d<false>, cEnd - cStart, 64, 0, s, c, cStart, nq);
}
void surf_fan1d_launch(const SurfArgs& a, int cStart, int cEnd, int nq, hipStream_t s)
{
    if (cEnd <= cStart) return;
    const SurfArgs c = of_class(a, cStart, cEnd);
    if (a.fpe == 4) launch_kernel(k_search_fan1d<true>, cEnd - cStart, 64, 0, s, c, cStart, nq);
    else launch_kernel(k_search_fan1d<false>, cEnd - cStart, 64, 0, s, c, cStart, nq);
}
void surf_nn_normals_launch(const SurfArgs& a, hipStream_t s)
{
    const int nbS = nb256(a.nS);
    k_nn_face_normals<<<nbS + nb256(a.nFaces), 256, 0, s>>>(a, nbS);
    k_surf_vertex_normals<<<nb256(a.nS), 256, 0, s>>>(a);
}
void snapshot_launch(const SurfArgs& a, hipStream_t s)
{
    if (a.nS > 0) k_snapshot<<<nb256(a.nS), 256, 0, s>>>(a.x, a.y, a.z, const_cast<float*>(a.sx), const_cast<float*>(a.sy),
                                                         const_cast<float*>(a.sz), a.nS);
}
void laplace_launch(float* x, float* y, float* z, const int* heRow, const int* heTarget, int lo, int hi, hipStream_t s)
{
    if (hi > lo) k_laplace<<<nb256(hi - lo), 256, 0, s>>>(x, y, z, heRow, heTarget, lo, hi);
}

}  // namespace vsdmo
