// ud_sample.hip -- the sampling module on gfx950: LBVH build, Hermite FGT,
// the per-pixel sequential-Poisson sampler (sampling.sample; reference:
// samplingCuda.cu:197-290, buildDynamicRadixTree.cuh,
// evaluateDynamicRadixTree.cuh, sequentialPoissonDynamicTree.cuh), the
// fixed-order densities (approximateFMMWeights; transformRadixTree.cuh) and
// Poisson-rate sampling with inclusion probabilities (no reference kernel).
//
// Every stage runs on the device with sizes kept in device memory, so a view
// costs no host synchronisation:
//   1 k_bandwidth     per-splat isotropic h_k -> fixed-point sum (2^-40 units)
//   2 k_view_params   h, query radius, screen bounds
//   3 k_cull_*        order-preserving compaction of visible splats + Morton
//   4 k_sort_*        3-pass LSD radix sort of 20-bit Morton keys (stable,
//                     wavefront ballot ranking)
//   5 k_hierarchy     Karras 2012 split on 64-bit keys (morton << 32 | pos)
//   6 k_bottom_up     atomic fan-in: boxes, counts, centres, Hermite degree
//   7 k_coef_blocks   coefficient slots (deg+1)^2 of the reachable expanded
//                     nodes, one reservation per workgroup
//   8 k_moments       Hermite moments per node over its contiguous leaf range,
//                     accumulated in FP64 in leaf order
//   9 k_sample_walk   per pixel tile: union FGT walk (k_sample_descend: the capacity
//                     descents)
//  10 k_sample_draw   wavefront per pixel: sequential Poisson keys u/p from
//                     Philox4x32-10, the k smallest in order (k_sample_replay:
//                     pixels with equal keys)
// Views of at most 4096 splats take stages 1-4 in one workgroup (k_front_small).
// The fixed-order and Poisson-rate paths share stages 1-6 and add expansion
// selection and moments per band (k_fixed_*), walk records (k_fmm_records,
// k_walk_records), the density walk (k_fmm_eval) and the thinning pass
// (k_poisson).  Batches of views run each stage as one launch (views on
// blockIdx.y) where the workspace holds them all.
// All FP32 arithmetic on the tree and in the samplers follows a fixed operation
// order (no contraction) so that index sets are reproducible bit for bit.
#include "ud_device.h"
#include "../../include/udsplat.h"

#include <type_traits>
#include <utility>
#include <vector>

using namespace ud;

namespace {

constexpr int kMaxDegree = 16;
constexpr int kMaxDepth = 64;        // descent trace bound (reference STACKSIZE)
// runs of consecutive 8x8 tiles dealt to each XCD in turn by the sampler's
// passes (k_sample_walk / draw / replay): their cost follows the splat density,
// so each XCD takes runs from the whole image (4 tiles: walk + draw 2.73 -> 2.59 ms
// at 1M splats, 512x512, against one contiguous block of tiles per XCD)
constexpr uint32_t kSampTileRun = 4;
constexpr int kTrieFields = 5;       // 4-byte fields per descent-trie entry (TrieRef)
constexpr int kWalkEntries = 384;    // trie entries the walk may create
// per tile, for the descents: entries of the walk, error flag; the pixels' totals from 64
// on; the entries' info and node from 128 on
constexpr int kTileInfo = 128 + 2 * kWalkEntries;
// entries the descents may add: 32 per launch, and at least 96, since the walk keeps
// its up to 5 x 96 rows of values there
__host__ __device__ constexpr int walk_extra(int L) { return 32 * (L > 3 ? L : 3); }
constexpr int kCullTile = 1024;      // elements per workgroup in the cull pass
// elements per workgroup in a sort pass: up to 128 workgroups of the smaller tile each add up
// the others' histograms themselves, one launch less per pass and fewer rounds in each
// (20 011 splats of two views: 12 sort launches of 55 us, here 6 of 34); beyond, the
// histograms are scanned in a launch of their own
constexpr int kSortTile = 2048, kSortTileSmall = 1024, kSortSelf = 128;
inline int sort_tile(long n) { return n <= (long)kSortTileSmall * kSortSelf ? kSortTileSmall : kSortTile; }
constexpr int kFixedDegree = 6;      // default expansion order of the fixed-order densities (hermitefmm.cuh:11)
constexpr int kFixedPMin = 4, kFixedPMax = 8;              // orders ude_set_fixed_degree accepts
constexpr int kFixedCoefsMax = (kFixedPMax + 1) * (kFixedPMax + 1);

// Gaussian bandwidth of a fixed-order density: h, 1 / sqrt(2 h^2), the leaf
// coefficient 1 / (2 pi sqrt(h)) and the query radius
struct Band {
    float h, is2h, c, radius;
};

struct ViewState {
    unsigned long long hsum;
    unsigned int hcnt;
    int nc;
    float h, radius, lo, hix, hiy, s2h, prec, is2h;
    unsigned long long blocks;   // internal nodes with a Hermite expansion, and above bit 32 their coefficients
    int nseeds;       // block-spanning fan-in starts (bottom-up, second level)
    int pad;
    Band band[2];     // fixed-order densities: tree bandwidth, wide proposal bandwidth
    unsigned long long nfix;     // accepted internal nodes of band 0, and of band 1 above bit 32
    int hhist[256];   // visible splats' proposal bandwidths, 1/16 px bins over [0, 16)
};

struct NodeGeo {      // traversal record
    float lox, loy, hix, hiy;
    float cx, cy, r2;
    int deg;
};
struct NodeLnk {
    int left, right, parent, count;
};
struct NodeAux {
    int off, first, last, pad;   // pad: a leaf's splat id
};
// per internal node: its two children as the sampler's walk reads them (one
// record per descent; a node's own fields arrive with its parent's record)
struct SampChild {
    float lox, loy, hix, hiy;    // box
    float cx, cy, r2;            // expansion centre, squared truncation radius
    int deg;                     // Hermite degree, -1 when the walk goes below
    int off, count, id, first;   // coefficient offset, leaves under it, node index, its first leaf
};
struct SampRec {
    SampChild l, r;
};
// per node: what the per-pixel Poisson walk reads of it in one load
struct PNode {
    float lox, loy, hix, hiy;    // box
    int left;                    // left child, -1 for leaves
    int esc;                     // next node in preorder after the subtree, -1 after the last
    int first, last;             // sorted leaf range
};
// per sorted leaf: the footprint proposal's record (foot_f32)
struct FootLeaf {
    float x, y;                  // screen position (the tree's)
    float t00, t01, t11, amp;    // whitening and peak of the EWA weight
    float pad[2];
};
// the footprint term is capped by one envelope for every splat, E(d) =
// exp(-max(0, d - kFootRcap)^2 a1) with a1 = 1 / 2h_1^2, the wide band's decay:
// min(1, w) equals w where w is below E, which holds beyond kFootRcap pixels
// for every splat whose largest axis is within h_1 and whose core min(1, w) = 1
// reaches at most kFootRcap; for the others (edge-on needles, the widest 0.1 %)
// the cap trims the footprint term and the wide band's half still covers them.
// A node's bound is then E at its box distance, with no per-node data.
constexpr float kFootRcap = 2.0f;

// per internal node: what the fixed-order density walk needs of its two
// children, so that one wave-uniform load serves a descent
struct FmmRec {
    float lbox[4], rbox[4];      // children's boxes (lo.x, lo.y, hi.x, hi.y)
    float lc[2], rc[2];          // children's centres
    int left, right;
    int lfix[2], rfix[2];        // children's expansion offsets per band, -1 for none / leaves
    int pad[2];
};

struct TreeWs {
    ViewState* vs;
    uint32_t *keysA, *keysB;
    int32_t *idsA, *idsB;
    int *cullCounts, *sortHist, *scanBlocks;
    NodeGeo* geo;
    NodeLnk* lnk;
    NodeAux* aux;
    int* flags;
    int* seeds;
    int* momList;
    float* trie;
    SampRec* srec;        // per internal node: children records of the sampler's walk
    int2* reach;          // per launch and pixel lane: leaf range the capacity descent reached
    int* tileInfo;        // per sampler tile: what the descents need of its walk (kTileInfo words)
    int* walkQueue;       // [0]: count, then the tiles k_sample_walk left to its passes
    int* tieQueue;                    // [0]: count, then (sampler lane, final key bits) per lane that met equal keys
    float2* leafXY;       // sorted position -> screen position of the leaf
    float* coef;
    // fixed-order densities (approximateFMMWeights, Poisson-rate sampling)
    int* fixOff[2];       // per internal node and band: coefficient offset, -1 = no expansion
    int* fixList[2];      // per band: accepted internal nodes
    float* fixCoef[2];    // per band: 49 coefficients per accepted node
    float* hraw;          // per splat id: proposal bandwidth sqrt(lambda_max(V))
    PNode* pnode;         // per node: Poisson walk record
    FootLeaf* footLeaf;   // per sorted leaf: footprint proposal record
    double* footSum;      // sum of the visible splats' footprint masses
    FmmRec* frec;         // per internal node: children for the density walk
    float* dens[2];       // per pixel and band: density D_b(q)
};

enum WsMode { kModeSample = 0, kModeFixed = 1, kModePoisson = 2 };

inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

int trie_entries(int k);

// carve the workspace; returns total bytes (ws may be null to only measure)
// mode kModeSample: dynamic degrees + descent trie; kModeFixed: degree-6 moments of
// the accepted internal nodes only; kModePoisson: fixed tree + proposal bandwidths
// + density image
size_t carve(void* ws, int N, int W, int H, int k, int mode, TreeWs* t)
{
    long n = N > 0 ? N : 1;
    long nn = 2 * n;
    long nCull = (n + kCullTile - 1) / kCullTile;
    long nSort = (n + sort_tile(n) - 1) / sort_tile(n);
    const bool fixedOrder = mode != kModeSample;
    long coefCap = (long)(kMaxDegree + 1) * (kMaxDegree + 1) * (n - 1 > 0 ? n - 1 : 1) + n;
    size_t off = 0;
    char* base = (char*)ws;
    auto take = [&](size_t bytes) { size_t o = off; off = align256(off + bytes); return base ? (void*)(base + o) : nullptr; };
    TreeWs w;
    w.vs = (ViewState*)take(sizeof(ViewState));
    w.keysA = (uint32_t*)take(4 * n);
    w.keysB = (uint32_t*)take(4 * n);
    w.idsA = (int32_t*)take(4 * n);
    w.idsB = (int32_t*)take(4 * n);
    w.cullCounts = (int*)take(4 * (nCull + 1));
    w.sortHist = (int*)take(4 * 256 * (nSort + 1));
    w.scanBlocks = (int*)take(4 * 256 * (nSort + 1));
    w.geo = (NodeGeo*)take(sizeof(NodeGeo) * nn);
    w.lnk = (NodeLnk*)take(sizeof(NodeLnk) * nn);
    w.aux = (NodeAux*)take(sizeof(NodeAux) * nn);
    w.flags = (int*)take(4 * n);
    w.seeds = (int*)take(4 * n);
    w.momList = (int*)take(4 * n);
    long lanes = (long)((W + 7) / 8) * ((H + 7) / 8) * 64;
    w.trie = fixedOrder ? nullptr : (float*)take(4L * kTrieFields * trie_entries(k) * lanes);
    w.srec = fixedOrder ? nullptr : (SampRec*)take(sizeof(SampRec) * n);
    w.reach = fixedOrder ? nullptr : (int2*)take(8L * 16 * lanes);
    w.tileInfo = fixedOrder ? nullptr : (int*)take(4L * kTileInfo * (lanes / 64));
    w.walkQueue = fixedOrder ? nullptr : (int*)take(4 * (lanes / 64 + 1));
    w.tieQueue = fixedOrder ? nullptr : (int*)take(4 * (2 * lanes + 1));
    w.leafXY = (float2*)take(8 * n);
    w.coef = fixedOrder ? nullptr : (float*)take(4 * coefCap);
    w.hraw = nullptr;
    w.pnode = nullptr;
    w.footLeaf = nullptr;
    w.footSum = nullptr;
    w.frec = nullptr;
    for (int b = 0; b < 2; b++) { w.fixOff[b] = w.fixList[b] = nullptr; w.fixCoef[b] = w.dens[b] = nullptr; }
    const int nb = mode == kModePoisson ? 2 : mode == kModeFixed ? 1 : 0;
    for (int b = 0; b < nb; b++) {
        w.fixOff[b] = (int*)take(4 * n);
        w.fixList[b] = (int*)take(4 * n);
        w.fixCoef[b] = (float*)take(4L * kFixedCoefsMax * (n - 1 > 0 ? n - 1 : 1));
    }
    if (nb > 0) w.frec = (FmmRec*)take(sizeof(FmmRec) * n);
    if (mode == kModePoisson) {
        w.hraw = (float*)take(4 * n);
        w.pnode = (PNode*)take(sizeof(PNode) * nn);
        w.footLeaf = (FootLeaf*)take(sizeof(FootLeaf) * n);
        w.footSum = (double*)take(8);
        w.dens[0] = (float*)take(4L * W * H);
        w.dens[1] = (float*)take(4L * W * H);
    }
    if (t) *t = w;
    return off;
}

// ---------------------------------------------------------------------------
// Screen-space covariance V (row-major) of one splat in FP32, the operation
// order of samplingCuda.cu:106-150.
__device__ void cov_f32(float Wf, float Hf, float ff, const float* p, const float* n, const float* sd,
                        float smoothing, float V[4], float* detAOut = nullptr)
{
    float sx, sy;
    screen_f32(Wf, Hf, ff, p, sx, sy);
    float y0x = sx + 1.0f, y0y = sy, y1x = sx, y1y = sy + 1.0f;
    float tf = 2.0f * ff;
    float x0[3] = { (Wf - 2.0f * y0x) / tf, -((Hf - 2.0f * y0y) / tf), 1.0f };
    float x1[3] = { (Wf - 2.0f * y1x) / tf, -((Hf - 2.0f * y1y) / tf), 1.0f };
    float a = dot3(p, n);
    float xt0 = a / dot3(x0, n), xt1 = a / dot3(x1, n);
    float t0[3], t1[3];
    for (int c = 0; c < 3; c++) { t0[c] = x0[c] * xt0 - p[c]; t1[c] = x1[c] * xt1 - p[c]; }
    float nt0 = sqrtf(dot3(t0, t0));
    float inv0 = 1.0f / nt0;
    float u0[3] = { t0[0] * inv0, t0[1] * inv0, t0[2] * inv0 };
    float u1[3] = { u0[1] * n[2] - u0[2] * n[1], u0[2] * n[0] - u0[0] * n[2], u0[0] * n[1] - u0[1] * n[0] };
    float A00 = nt0, A01 = dot3(t1, u0), A10 = 0.0f, A11 = dot3(t1, u1);
    float detA = A00 * A11 - A01 * A10;
    if (detAOut) *detAOut = detA;
    float idA = 1.0f / detA;
    float J00 = A11 * idA, J01 = -A01 * idA, J10 = -A10 * idA, J11 = A00 * idA;
    float d0 = sd[0] * sd[0], d1 = sd[1] * sd[1];
    float M00 = J00 * d0 + J01 * 0.0f, M01 = J00 * 0.0f + J01 * d1;
    float M10 = J10 * d0 + J11 * 0.0f, M11 = J10 * 0.0f + J11 * d1;
    float V00 = M00 * J00 + M01 * J01, V01 = M00 * J10 + M01 * J11;
    float V10 = M10 * J00 + M11 * J01, V11 = M10 * J10 + M11 * J11;
    V[0] = V00 + smoothing; V[1] = V01 + 0.0f; V[2] = V10 + 0.0f; V[3] = V11 + smoothing;
}

// Per-splat bandwidth before the one-pixel cap, 1 / sqrt(lambda_min(V^-1))
// (samplingCuda.cu:106-163) in FP32, fixed operation order.
__device__ float iso_hraw(float Wf, float Hf, float ff, const float* p, const float* n, const float* sd, float smoothing)
{
    float V[4];
    cov_f32(Wf, Hf, ff, p, n, sd, smoothing, V);
    float V00 = V[0], V01 = V[1], V10 = V[2], V11 = V[3];
    float dV = V00 * V11 - V01 * V10;
    float idV = 1.0f / dV;
    float I00 = V11 * idV, I01 = -V01 * idV, I10 = -V10 * idV, I11 = V00 * idV;
    float tr = I00 + I11;
    float det = I00 * I11 - I01 * I10;
    float disc = 0.25f * (tr * tr) - det;
    float sq = sqrtf(disc);
    float l1 = 0.5f * tr + sq, l2 = 0.5f * tr - sq;
    float lk = fminf(l1, l2);
    return 1.0f / sqrtf(lk);
}

// Splat bandwidth for the Poisson-rate proposal: sqrt(lambda_max(V)) from V
// itself (well conditioned, unlike the smallest eigenvalue of V^-1 for splats
// seen at grazing angles); NaN for degenerate geometry.
__device__ float prop_h(float Wf, float Hf, float ff, const float* p, const float* n, const float* sd, float smoothing)
{
    float V[4];
    cov_f32(Wf, Hf, ff, p, n, sd, smoothing, V);
    float tr = V[0] + V[3];
    float det = V[0] * V[3] - V[1] * V[2];
    float disc = 0.25f * (tr * tr) - det;
    float lmax = 0.5f * tr + sqrtf(fmaxf(disc, 0.0f));
    return sqrtf(lmax);
}

// Footprint proposal of Poisson-rate sampling (no reference counterpart): the
// splat's own EWA weight w(q) = amp exp(-(u^2 + v^2) / 2), (u, v) = T (q - s),
// T^T T = V^-1 (upper triangular), amp = 1 / (2 pi sqrt(det V) |det A|), with V
// and A the FP32 screen covariance and Jacobian of cov_f32, and its isotropic
// envelope amp exp(-|q - s|^2 m), m = 1 / (2 lambda_max(V)) >= the envelope's
// exponent along any direction.  Degenerate geometry gives amp = 0 (the splat is
// then drawn through the wide-band half of the mixture alone).
__device__ void foot_f32(float Wf, float Hf, float ff, const float* p, const float* n, const float* sd,
                         float smoothing, float& t00, float& t01, float& t11, float& amp, float& m, float& mass)
{
    float V[4], detA;
    cov_f32(Wf, Hf, ff, p, n, sd, smoothing, V, &detA);
    float tr = V[0] + V[3];
    float det = V[0] * V[3] - V[1] * V[2];
    float disc = 0.25f * (tr * tr) - det;
    float lmax = 0.5f * tr + sqrtf(fmaxf(disc, 0.0f));
    t00 = sqrtf(V[3] / det);
    t01 = -V[1] / sqrtf(V[3] * det);
    t11 = 1.0f / sqrtf(V[3]);
    const float area = (2.0f * 3.14159265358979f) * sqrtf(det);     // 2 pi sqrt(det V)
    amp = 1.0f / (area * fabsf(detA));
    m = 0.5f / lmax;
    // integral of min(w, 1) over the plane
    mass = area * (amp <= 1.0f ? amp : 1.0f + plogf(amp));
    const bool ok = det > 0.0f && lmax > 0.0f && V[3] > 0.0f && isfinite(t00) && isfinite(t01) && isfinite(t11) &&
                    isfinite(amp) && isfinite(m) && isfinite(mass);
    if (!ok) { t00 = t01 = t11 = 0.0f; amp = 0.0f; m = 0.0f; mass = 0.0f; }
}

// the footprint cap E(d) at distance d (see kFootRcap)
__device__ __forceinline__ float foot_env(float a1, float d)
{
    const float e = fmaxf(0.0f, d - kFootRcap);
    return pexpf(-((e * e) * a1));
}

// the footprint term of one leaf at q: min(1, w(q), E(|q - s|))
__device__ __forceinline__ float foot_leaf(const FootLeaf& L, float a1, float qx, float qy, float d2)
{
    const float dx = qx - L.x, dy = qy - L.y;
    float u = L.t00 * dx;
    u = u + L.t01 * dy;
    const float v = L.t11 * dy;
    float e = u * u;
    e = e + v * v;
    const float w = L.amp * pexpf(-(0.5f * e));
    return fminf(1.0f, fminf(w, foot_env(a1, sqrtf(d2))));
}

// node bound of the footprint term at squared box distance d2: E, inflated by
// 2^-20 so that a one-ulp step of the exponential cannot put a leaf above it
__device__ __forceinline__ float foot_bound(float a1, float d2)
{
    return fminf(1.0f, foot_env(a1, sqrtf(d2)) * 1.00000095367431640625f);
}

// isotropic bandwidth capped at one pixel (samplingCuda.cu:160)
__device__ float iso_h(float Wf, float Hf, float ff, const float* p, const float* n, const float* sd, float smoothing)
{
    return fminf(1.0f, iso_hraw(Wf, Hf, ff, p, n, sd, smoothing));
}

// Tree-build kernels run over a batch of views at once, view = blockIdx.y: the
// views' workspaces lie ws bytes apart, their points / normals pts bytes apart
// and their std-devs sd bytes apart (0 when shared).  A single view passes {}.
struct VStride {
    size_t ws, pts, sd;
};

template <class T>
__device__ __forceinline__ T* vw(T* p, size_t stride)
{
    return p ? (T*)((char*)p + (size_t)blockIdx.y * stride) : p;
}

__device__ __forceinline__ void zero_state(ViewState* vs)
{
    if (threadIdx.x == 0) {
        vs->hsum = 0; vs->hcnt = 0; vs->nc = 0; vs->blocks = 0; vs->nseeds = 0;
        vs->nfix = 0;
    }
    for (int b = threadIdx.x; b < 256; b += blockDim.x) vs->hhist[b] = 0;
}

__global__ void k_zero_state(ViewState* vs, VStride vsd) { zero_state(vw(vs, vsd.ws)); }

__global__ __launch_bounds__(1024) void k_bandwidth(int N, float Wf, float Hf, float ff, float smoothing,
                                                   const float* __restrict__ pts, const float* __restrict__ nrm,
                                                   const float* __restrict__ sd, ViewState* vs, float* hraw, VStride vsd)
{
    pts = vw(pts, vsd.pts);
    nrm = vw(nrm, vsd.pts);
    sd = vw(sd, vsd.sd);
    vs = vw(vs, vsd.ws);
    hraw = vw(hraw, vsd.ws);
    __shared__ unsigned long long ssum[16];
    __shared__ unsigned int scnt[16];
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    unsigned long long q = 0;
    unsigned int c = 0;
    // grid-stride over the splats (a capped grid keeps the two device-wide atomics
    // per workgroup few; the fixed-point sum does not depend on the grouping)
    for (; t < N; t += gridDim.x * blockDim.x) {
        float hk = iso_h(Wf, Hf, ff, pts + 3L * t, nrm + 3L * t, sd + 2L * t, smoothing);
        if (hraw) hraw[t] = prop_h(Wf, Hf, ff, pts + 3L * t, nrm + 3L * t, sd + 2L * t, smoothing);
        if (isfinite(hk)) { q += (unsigned long long)((double)hk * 1099511627776.0); c += 1; }
    }
    for (int o = 32; o > 0; o >>= 1) {
        q += __shfl_xor(q, o, 64);
        c += __shfl_xor(c, o, 64);
    }
    int wv = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { ssum[wv] = q; scnt[wv] = c; }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long s = 0;
        unsigned int cc = 0;
        for (int q = 0; q < (int)(blockDim.x >> 6); q++) { s += ssum[q]; cc += scnt[q]; }
        if (cc) { atomicAdd(&vs->hsum, s); atomicAdd(&vs->hcnt, cc); }
    }
}

// query radius r with exp(-r^2 / 2h^2) / (2 pi sqrt(h)) = precision (samplingCuda.cu:251-252)
__device__ float band_radius(float h, double prec)
{
    float normalization = (float)(2.0 * UD_PI * (double)sqrtf(h));
    return (float)(sqrt(2.0) * (double)h * sqrt(-log(prec) - log((double)normalization)));
}

__device__ Band make_band(float h, double prec)
{
    Band b;
    b.h = h;
    b.is2h = 1.0f / sqrtf((2.0f * h) * h);
    b.c = (float)(1.0 / (2.0 * UD_PI * (double)sqrtf(h)));    // buildRadixTree.cuh:580
    b.radius = band_radius(h, prec);
    return b;
}

__device__ __forceinline__ void view_params(ViewState* vs, float Wf, float Hf, double prec)
{
    double hd = ((double)vs->hsum * (1.0 / 1099511627776.0)) / (double)vs->hcnt;
    float h = (float)hd;
    float radius = band_radius(h, prec);
    vs->h = h;
    vs->radius = radius;
    vs->lo = -radius;
    vs->hix = Wf + radius;
    vs->hiy = Hf + radius;
    vs->s2h = sqrtf((2.0f * h) * h);
    vs->is2h = 1.0f / vs->s2h;
    vs->prec = (float)prec;
    vs->nc = 0;
    vs->band[0] = make_band(h, prec);
}

__global__ void k_view_params(ViewState* vs, float Wf, float Hf, double prec, VStride vsd)
{
    if (threadIdx.x == 0) view_params(vw(vs, vsd.ws), Wf, Hf, prec);
}

__device__ __forceinline__ bool visible(const ViewState& v, float Wf, float Hf, float ff, const float* p, float& sx, float& sy)
{
    screen_f32(Wf, Hf, ff, p, sx, sy);
    bool vis = (p[2] <= 0.0f);
    vis &= (v.lo <= sx); vis &= (v.hix >= sx);
    vis &= (v.lo <= sy); vis &= (v.hiy >= sy);
    return vis;
}

// 10-bit cell coordinates interleaved into a 20-bit key (x bits above y bits).
// The reference spreads the bits three apart (a 3D code with z = 0,
// buildRadixTree.cuh:18-54); the compact code orders the splats identically and
// its highest differing bit is a monotone function of the spread one, so the
// Karras hierarchy on it is the same tree, and the sort needs three 8-bit
// passes instead of four.
__device__ __forceinline__ uint32_t expand_bits2(uint32_t v)
{
    v = (v | (v << 8)) & 0x00FF00FFu;
    v = (v | (v << 4)) & 0x0F0F0F0Fu;
    v = (v | (v << 2)) & 0x33333333u;
    v = (v | (v << 1)) & 0x55555555u;
    return v;
}

__device__ __forceinline__ uint32_t morton2(float ux, float uy)
{
    float cx = fminf(fmaxf(ux * 1024.0f, 0.0f), 1023.0f);
    float cy = fminf(fmaxf(uy * 1024.0f, 0.0f), 1023.0f);
    return 2u * expand_bits2((uint32_t)cx) + expand_bits2((uint32_t)cy);
}

// orders the wavefront's LDS accesses (its LDS operations execute in order)
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// exclusive scan of one int per thread over a 256-thread workgroup
__device__ __forceinline__ int block_excl_scan(int v, int* sh /*[4]*/, int& total)
{
    int incl = wave_incl_scan(v);
    int wv = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 63) sh[wv] = incl;
    __syncthreads();
    int off = 0;
    for (int q = 0; q < wv; q++) off += sh[q];
    total = sh[0] + sh[1] + sh[2] + sh[3];
    __syncthreads();
    return off + incl - v;
}

__global__ __launch_bounds__(256) void k_cull_count(int N, float Wf, float Hf, float ff,
                                                    const float* __restrict__ pts, const ViewState* __restrict__ vs,
                                                    int* __restrict__ counts, VStride vsd)
{
    pts = vw(pts, vsd.pts);
    vs = vw(vs, vsd.ws);
    counts = vw(counts, vsd.ws);
    __shared__ int sh[4];
    ViewState v = *vs;
    int base = blockIdx.x * kCullTile;
    int c = 0;
    for (int r = 0; r < kCullTile / 256; r++) {
        int e = base + r * 256 + threadIdx.x;
        float sx, sy;
        if (e < N && visible(v, Wf, Hf, ff, pts + 3L * e, sx, sy)) c++;
    }
    int total;
    block_excl_scan(c, sh, total);
    if (threadIdx.x == 0) counts[blockIdx.x] = total;
}

// single-workgroup exclusive scan of n ints in place; total to *totalOut
__global__ __launch_bounds__(1024) void k_scan_small(int* data, int n, int* totalOut, VStride vsd)
{
    data = vw(data, vsd.ws);
    totalOut = vw(totalOut, vsd.ws);
    __shared__ int sh[16];
    __shared__ int carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (int base = 0; base < n; base += 1024) {
        int e = base + threadIdx.x;
        int v = e < n ? data[e] : 0;
        int incl = wave_incl_scan(v);
        int wv = threadIdx.x >> 6;
        if ((threadIdx.x & 63) == 63) sh[wv] = incl;
        __syncthreads();
        int off = 0;
        for (int q = 0; q < wv; q++) off += sh[q];
        int tot = 0;
        for (int q = 0; q < 16; q++) tot += sh[q];
        int c = carry;
        if (e < n) data[e] = c + off + incl - v;
        __syncthreads();
        if (threadIdx.x == 0) carry = c + tot;
        __syncthreads();
    }
    if (threadIdx.x == 0) *totalOut = carry;
}

__global__ __launch_bounds__(256) void k_cull_scatter(int N, float Wf, float Hf, float ff,
                                                      const float* __restrict__ pts, ViewState* vs,
                                                      const int* __restrict__ offs, uint32_t* __restrict__ keys,
                                                      int32_t* __restrict__ ids, VStride vsd)
{
    pts = vw(pts, vsd.pts);
    vs = vw(vs, vsd.ws);
    offs = vw(offs, vsd.ws);
    keys = vw(keys, vsd.ws);
    ids = vw(ids, vsd.ws);
    __shared__ int sh[4];
    ViewState v = *vs;
    int base = blockIdx.x * kCullTile;
    int run;
    if (gridDim.x <= 256) {                                 // counts, not yet scanned: add those before
        block_excl_scan((int)threadIdx.x < (int)blockIdx.x ? offs[threadIdx.x] : 0, sh, run);
        if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) vs->nc = run + offs[blockIdx.x];
    } else {
        run = offs[blockIdx.x];
    }
    for (int r = 0; r < kCullTile / 256; r++) {
        int e = base + r * 256 + threadIdx.x;
        float sx = 0.0f, sy = 0.0f;
        bool vis = e < N && visible(v, Wf, Hf, ff, pts + 3L * e, sx, sy);
        int total;
        int pos = run + block_excl_scan(vis ? 1 : 0, sh, total);
        if (vis) {
            float ux = (sx - v.lo) / (v.hix - v.lo);
            float uy = (sy - v.lo) / (v.hiy - v.lo);
            keys[pos] = morton2(ux, uy);
            ids[pos] = e;
        }
        run += total;
    }
}

// ---------------------------------------------------------------------------
// LSD radix sort, 8-bit digits.  Histogram -> digit-major scan -> stable scatter.
// ---------------------------------------------------------------------------
template <int TILE>
__global__ __launch_bounds__(256) void k_sort_hist(const ViewState* __restrict__ vs, const uint32_t* __restrict__ keys,
                                                   int shift, int nblk, int* __restrict__ hist, VStride vsd)
{
    vs = vw(vs, vsd.ws);
    keys = vw(keys, vsd.ws);
    hist = vw(hist, vsd.ws);
    __shared__ int h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    int n = vs->nc;
    int base = blockIdx.x * TILE;
    for (int r = 0; r < TILE / 256; r++) {
        int e = base + r * 256 + threadIdx.x;
        if (e < n) atomicAdd(&h[(keys[e] >> shift) & 255u], 1);
    }
    __syncthreads();
    // the smaller tile's histograms by workgroup, the larger's by digit for the scan
    if (TILE == kSortTileSmall) hist[blockIdx.x * 256 + threadIdx.x] = h[threadIdx.x];
    else hist[threadIdx.x * nblk + blockIdx.x] = h[threadIdx.x];
}

// exclusive scan of hist[d][0..nblk) for each digit d (one workgroup per digit);
// digit totals to tot[d]
__global__ __launch_bounds__(256) void k_sort_scan_digits(int* hist, int nblk, int* tot, VStride vsd)
{
    hist = vw(hist, vsd.ws);
    tot = vw(tot, vsd.ws);
    __shared__ int sh[4];
    __shared__ int carry;
    int* h = hist + (long)blockIdx.x * nblk;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (int base = 0; base < nblk; base += 256) {
        int e = base + threadIdx.x;
        int v = e < nblk ? h[e] : 0;
        int total;
        int ex = block_excl_scan(v, sh, total);
        int c = carry;
        if (e < nblk) h[e] = c + ex;
        __syncthreads();
        if (threadIdx.x == 0) carry = c + total;
        __syncthreads();
    }
    if (threadIdx.x == 0) tot[blockIdx.x] = carry;
}

template <int TILE>
__global__ __launch_bounds__(256) void k_sort_scatter(const ViewState* __restrict__ vs, const uint32_t* __restrict__ kin,
                                                      const int32_t* __restrict__ iin, int shift, int nblk,
                                                      const int* __restrict__ hist, const int* __restrict__ digitTot,
                                                      uint32_t* __restrict__ kout, int32_t* __restrict__ iout, VStride vsd)
{
    vs = vw(vs, vsd.ws);
    kin = vw(kin, vsd.ws);
    iin = vw(iin, vsd.ws);
    hist = vw(hist, vsd.ws);
    digitTot = vw(digitTot, vsd.ws);
    kout = vw(kout, vsd.ws);
    iout = vw(iout, vsd.ws);
    __shared__ int run[256];
    __shared__ int wc[4][256];
    int n = vs->nc;
    __shared__ int sh[4];
    int base = blockIdx.x * TILE;
    // this workgroup's place in each digit: those of the digits before, and of the same
    // digit in the workgroups before
    int tot = 0, pre = 0, all;
    if (TILE == kSortTileSmall) {
#pragma unroll 8
        for (int q = 0; q < nblk; q++) {
            const int v = hist[q * 256 + threadIdx.x];
            tot += v;
            pre += q < (int)blockIdx.x ? v : 0;
        }
    } else {
        tot = digitTot[threadIdx.x];
        pre = hist[threadIdx.x * nblk + blockIdx.x];
    }
    run[threadIdx.x] = block_excl_scan(tot, sh, all) + pre;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int r = 0; r < TILE / 256; r++) {
        for (int q = 0; q < 4; q++) wc[q][threadIdx.x] = 0;
        __syncthreads();
        int e = base + r * 256 + threadIdx.x;
        bool act = e < n;
        uint32_t key = act ? kin[e] : 0u;
        int32_t id = act ? iin[e] : 0;
        uint32_t dg = (key >> shift) & 255u;
        // lanes of this wave with the same digit
        unsigned long long m = __ballot(act);
        for (int b = 0; b < 8; b++) {
            unsigned long long bb = __ballot((dg >> b) & 1u);
            m &= ((dg >> b) & 1u) ? bb : ~bb;
        }
        int rk = __popcll(m & lt);
        if (act && rk == 0) wc[wv][dg] = __popcll(m);
        __syncthreads();
        if (act) {
            int off = run[dg];
            for (int q = 0; q < wv; q++) off += wc[q][dg];
            int pos = off + rk;
            kout[pos] = key;
            iout[pos] = id;
        }
        __syncthreads();
        run[threadIdx.x] += wc[0][threadIdx.x] + wc[1][threadIdx.x] + wc[2][threadIdx.x] + wc[3][threadIdx.x];
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// State, bandwidth, cull and sort of up to kFrontSplats splats in one workgroup and one
// launch: at these sizes the 11 kernels above are mostly their own starts and ends, while
// the network's steps grow with the splats.  sampling.sample of one 64x64 view, k = 8, on the
// device / until the call has ended, those kernels -> this one: 64 splats 71 -> 54 / 129 ->
// 95 us, 1024 146 -> 132 / 187 -> 161, 3072 218 -> 220 / 257 -> 249, 4096 248 -> 253 / 287 ->
// 283; 16 views of 4096 306 both / 362 -> 358.  The line lies where the device's time is even,
// and where a 20-bit key and a position fill a 32-bit word, which a bitonic network in LDS
// sorts; the order is the stable radix sort's.
// ---------------------------------------------------------------------------
constexpr int kFrontSplats = 4096;

__global__ __launch_bounds__(1024) void k_front_small(int N, float Wf, float Hf, float ff, float smoothing, double prec,
                                                      const float* __restrict__ pts, const float* __restrict__ nrm,
                                                      const float* __restrict__ sd, ViewState* vs, float* hraw,
                                                      uint32_t* __restrict__ keys, int32_t* __restrict__ ids,
                                                      VStride vsd)
{
    pts = vw(pts, vsd.pts);
    nrm = vw(nrm, vsd.pts);
    sd = vw(sd, vsd.sd);
    vs = vw(vs, vsd.ws);
    hraw = vw(hraw, vsd.ws);
    keys = vw(keys, vsd.ws);
    ids = vw(ids, vsd.ws);
    __shared__ uint32_t word[kFrontSplats];
    __shared__ int32_t idAt[kFrontSplats];
    __shared__ ViewState v;
    __shared__ unsigned long long ssum[16];
    __shared__ unsigned int scnt[16];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    zero_state(vs);
    unsigned long long q = 0;
    unsigned int c = 0;
    for (int t = tid; t < N; t += 1024) {
        const float hk = iso_h(Wf, Hf, ff, pts + 3L * t, nrm + 3L * t, sd + 2L * t, smoothing);
        if (hraw) hraw[t] = prop_h(Wf, Hf, ff, pts + 3L * t, nrm + 3L * t, sd + 2L * t, smoothing);
        if (isfinite(hk)) { q += (unsigned long long)((double)hk * 1099511627776.0); c += 1; }
    }
    for (int o = 32; o > 0; o >>= 1) {
        q += __shfl_xor(q, o, 64);
        c += __shfl_xor(c, o, 64);
    }
    if (lane == 0) { ssum[wid] = q; scnt[wid] = c; }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < 16; w++) { ssum[0] += ssum[w]; scnt[0] += scnt[w]; }
        vs->hsum = v.hsum = ssum[0];
        vs->hcnt = v.hcnt = scnt[0];
        view_params(vs, Wf, Hf, prec);
        view_params(&v, Wf, Hf, prec);
    }
    __syncthreads();
    // the visible splats in order: key, and the position in that order
    int n = 0;
    for (int r = 0; r < N; r += 1024) {
        const int e = r + tid;
        float sx = 0.0f, sy = 0.0f;
        const bool vis = e < N && visible(v, Wf, Hf, ff, pts + 3L * e, sx, sy);
        const unsigned long long m = __ballot(vis);
        __syncthreads();
        if (lane == 0) scnt[wid] = __popcll(m);
        __syncthreads();
        int at = n;
        for (int w = 0; w < 16; w++) {
            if (w < wid) at += scnt[w];
            n += scnt[w];
        }
        if (vis) {
            at += __popcll(m & ((1ull << lane) - 1ull));
            const float ux = (sx - v.lo) / (v.hix - v.lo);
            const float uy = (sy - v.lo) / (v.hiy - v.lo);
            word[at] = morton2(ux, uy) << 12 | (uint32_t)at;
            idAt[at] = e;
        }
    }
    int n2 = 2;
    while (n2 < n) n2 *= 2;
    __syncthreads();
    for (int t = n + tid; t < n2; t += 1024) word[t] = 0xffffffffu;     // positions stay below 4095 where n < n2
    __syncthreads();
    for (int k = 2; k <= n2; k *= 2)
        for (int j = k / 2; j > 0; j /= 2) {
            for (int x = tid; x < n2 / 2; x += 1024) {
                const int i = 2 * x - (x & (j - 1));
                const uint32_t a = word[i], b = word[i + j];
                if ((a > b) == ((i & k) == 0)) { word[i] = b; word[i + j] = a; }
            }
            // 64 neighbouring pairs at a distance of up to 64 cover 128 words of one wavefront
            const int next = j > 1 ? j / 2 : k;
            if (j > 64 || next > 64) __syncthreads();
            else wave_lds_fence();
        }
    __syncthreads();
    for (int t = tid; t < n; t += 1024) {
        keys[t] = word[t] >> 12;
        ids[t] = idAt[word[t] & (kFrontSplats - 1)];
    }
    if (tid == 0) vs->nc = n;
}

// ---------------------------------------------------------------------------
// Karras hierarchy on 64-bit unique keys (buildRadixTree.cuh:76-167).
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t key64(const uint32_t* k, int i) { return ((uint64_t)k[i] << 32) | (uint32_t)i; }

__device__ __forceinline__ int delta(const uint32_t* k, int n, int i, int j)
{
    if (j < 0 || j >= n) return -1;
    return __clzll(key64(k, i) ^ key64(k, j));
}

__device__ float trunc_r2(float h, float prec, int cnt)
{
    float v = -2.0f * (h * h);
    v = v * plogf(prec / (float)cnt);
    float R = sqrtf(v);
    return R * R;
}

__global__ __launch_bounds__(256) void k_hierarchy(float Wf, float Hf, float ff, const float* __restrict__ pts,
                                                   const ViewState* __restrict__ vs, const uint32_t* __restrict__ keys,
                                                   const int32_t* __restrict__ ids, NodeGeo* __restrict__ geo,
                                                   NodeLnk* __restrict__ lnk, NodeAux* __restrict__ aux,
                                                   float2* __restrict__ leafXY, int* __restrict__ flags, VStride vsd)
{
    pts = vw(pts, vsd.pts);
    vs = vw(vs, vsd.ws);
    keys = vw(keys, vsd.ws);
    ids = vw(ids, vsd.ws);
    geo = vw(geo, vsd.ws);
    lnk = vw(lnk, vsd.ws);
    aux = vw(aux, vsd.ws);
    leafXY = vw(leafXY, vsd.ws);
    flags = vw(flags, vsd.ws);
    int n = vs->nc;
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int L0 = n - 1;
    float h = vs->h, prec = vs->prec;
    // leaf t
    {
        int nd = L0 + t;
        float sx, sy;
        screen_f32(Wf, Hf, ff, pts + 3L * ids[t], sx, sy);
        NodeGeo g;
        g.lox = sx; g.loy = sy; g.hix = sx; g.hiy = sy; g.cx = sx; g.cy = sy;
        g.r2 = trunc_r2(h, prec, 1);
        g.deg = 0;
        geo[nd] = g;
        leafXY[t] = make_float2(sx, sy);
        lnk[nd].left = -1; lnk[nd].right = -1; lnk[nd].count = 1;
        NodeAux a; a.off = 0; a.first = t; a.last = t; a.pad = ids[t];   // pad: the leaf's splat id
        aux[nd] = a;
    }
    if (t == 0) lnk[0].parent = -1;
    if (t >= n - 1) return;
    flags[t] = 0;                                  // fan-in arrival count of internal node t
    // internal node t
    int i0, j0;
    if (t == 0) { i0 = 0; j0 = n - 1; }
    else {
        int dl = delta(keys, n, t, t - 1), dr = delta(keys, n, t, t + 1);
        int d = dr > dl ? 1 : -1;
        int dmin = dl < dr ? dl : dr;
        int lmax = 2;
        while (delta(keys, n, t, t + d * lmax) > dmin) lmax <<= 1;
        int l = 0;
        for (int s = lmax >> 1; s > 0; s >>= 1)
            if (delta(keys, n, t, t + (l + s) * d) > dmin) l += s;
        int jdx = t + l * d;
        i0 = d < 0 ? jdx : t;
        j0 = d < 0 ? t : jdx;
    }
    uint64_t fc = key64(keys, i0), lc = key64(keys, j0);
    int sp;
    if (fc == lc) sp = (i0 + j0) >> 1;
    else {
        int dn = __clzll(fc ^ lc);
        sp = i0;
        int stride = j0 - i0;
        do {
            stride = (stride + 1) >> 1;
            int mid = sp + stride;
            if (mid < j0 && __clzll(fc ^ key64(keys, mid)) > dn) sp = mid;
        } while (stride > 1);
    }
    int lc_ = sp, rc_ = sp + 1;
    if (i0 == sp) lc_ += L0;
    if (j0 == sp + 1) rc_ += L0;
    lnk[t].left = lc_; lnk[t].right = rc_;
    lnk[lc_].parent = t; lnk[rc_].parent = t;
    aux[t].first = i0; aux[t].last = j0;
    // what the bottom-up pass needs of the count alone, kept off its serial chain
    lnk[t].count = j0 - i0 + 1;
    geo[t].r2 = trunc_r2(h, prec, j0 - i0 + 1);
}

// hermiteError (hermitefmm.cuh:184-195), integer powers by repeated products
__device__ float hermite_error(float r, float nr, int p)
{
    if (r >= 1.0f) return r;
    float om = 1.0f - r;
    float a = nr / (om * om);
    float rp = 1.0f;
    for (int i = 0; i < p; i++) rp = rp * r;
    float fac = 1.0f;
    for (int i = 1; i <= p; i++) fac = fac * (float)i;
    float b = rp / sqrtf(fac);
    float c = b * b;
    float d = 2.0f * (1.0f - rp) * b;
    return a * (c + d);
}

// sqrtf(d!) of every degree, with hermite_error's operations: entry d of a table in LDS
constexpr int kRootFact = kMaxDegree + 2;
__device__ __forceinline__ void root_fact_fill(float* tab)
{
    if ((int)threadIdx.x >= kRootFact) return;
    float fac = 1.0f;
    for (int i = 1; i <= (int)threadIdx.x; i++) fac = fac * (float)i;
    tab[threadIdx.x] = sqrtf(fac);
}

// The record of an internal node from its two complete children, left then
// right (buildDynamicRadixTree.cuh:126-223, with the children's own centres); r2 is the
// node's already.  The pass is a chain of these merges, so this is bound by their latency.
__device__ __forceinline__ NodeGeo merge_geo(const NodeGeo& gl, int cl, const NodeGeo& gr, int cr, float h,
                                             float prec, float r2, const float* rootFact)
{
    NodeGeo g;
    g.r2 = r2;
    g.lox = fminf(gl.lox, gr.lox); g.loy = fminf(gl.loy, gr.loy);
    g.hix = fmaxf(gl.hix, gr.hix); g.hiy = fmaxf(gl.hiy, gr.hiy);
    int cn = cl + cr;
    float num = (float)cl * gl.cx;
    num = num + (float)cr * gr.cx;
    g.cx = num / (float)cn;
    num = (float)cl * gl.cy;
    num = num + (float)cr * gr.cy;
    g.cy = num / (float)cn;
    float mn = 0.0f;
    mn = fmaxf(mn, fmaxf(g.cx - g.lox, g.hix - g.cx));
    mn = fmaxf(mn, fmaxf(g.cy - g.loy, g.hiy - g.cy));
    float rr = mn / h;
    int deg;
    if (gl.deg < 0 && gr.deg < 0) deg = -1;
    else if (!(rr < 1.0f)) deg = -1;
    else {
        // the lowest degree from the children's up whose hermiteError meets the
        // precision; the error's power r^d is carried from one degree to the next, with
        // the same products as hermite_error evaluates
        int d = gl.deg > gr.deg ? gl.deg : gr.deg;
        float root = rootFact[d];
        const float om = 1.0f - rr;
        const float a = (float)cn / (om * om);
        float rp = 1.0f;
        for (int i = 0; i < d; i++) rp = rp * rr;
        while (d <= kMaxDegree) {
            const float b = rp / root;
            const float c = b * b;
            const float e = 2.0f * (1.0f - rp) * b;
            if (!(a * (c + e) > prec)) break;
            d++;
            rp = rp * rr;
            root = rootFact[d];                     // d <= kMaxDegree + 1: inside the table
        }
        deg = d <= kMaxDegree ? d : -1;
    }
    g.deg = deg;
    return g;
}

// Bottom-up pass, level 1: one workgroup per block of 1024 sorted leaves.  The
// second thread to reach a node whose leaf range lies inside the block merges
// it.  Such a node's index lies inside the block too (a Karras node's index is
// one end of its range), so the block's internal nodes are staged in LDS first
// (links and leaf ranges in, merged records out, one arrival counter each) and
// the fan-in never waits on device memory: both arrivals come from the same
// workgroup, so workgroup-scope fences order the exchange.  Merged records are
// also stored to device memory for the later passes.  The chain of merges bounds it:
// factorials from a table, counts and truncation radii from k_hierarchy take 1M splats
// from 87 to 59 us.  A thread that reaches a
// node spanning the block's boundary hands its (complete) node to level 2.
constexpr int kFanBlock = 1024;
__global__ __launch_bounds__(kFanBlock) void k_bottom_up_local(ViewState* vs, NodeGeo* geo,
                                                               const NodeLnk* __restrict__ lnk,
                                                               const NodeAux* __restrict__ aux, int* seeds, VStride vsd)
{
    __shared__ int arrivals[kFanBlock];
    __shared__ float2 sLeaf[kFanBlock];          // the block's leaf positions
    __shared__ NodeGeo sNode[kFanBlock];         // merged records of internal nodes b0 + i
    __shared__ int4 sLink[kFanBlock];            // left, right, parent, first leaf of node b0 + i
    __shared__ int sLast[kFanBlock];             // last leaf of node b0 + i
    __shared__ int sSeeds[kFanBlock];            // nodes handed to level 2
    __shared__ int nSeeds, seedBase;
    __shared__ float rootFact[kRootFact];
    vs = vw(vs, vsd.ws);
    geo = vw(geo, vsd.ws);
    lnk = vw(lnk, vsd.ws);
    root_fact_fill(rootFact);
    aux = vw(aux, vsd.ws);
    seeds = vw(seeds, vsd.ws);
    const int n = vs->nc;
    const int L0 = n - 1;
    const int b0 = blockIdx.x * kFanBlock;
    const int tid = threadIdx.x;
    const int pos = b0 + tid;
    arrivals[tid] = 0;
    if (tid == 0) nSeeds = 0;
    NodeGeo g;
    int p = -1;
    if (pos < n && n >= 2) {
        g = geo[L0 + pos];
        sLeaf[tid] = make_float2(g.cx, g.cy);
        p = lnk[L0 + pos].parent;
    }
    if (pos < L0) {
        const NodeLnk L = lnk[pos];
        const NodeAux a = aux[pos];
        sLink[tid] = make_int4(L.left, L.right, L.parent, a.first);
        sLast[tid] = a.last;
        sNode[tid].r2 = geo[pos].r2;
    }
    __syncthreads();
    const float h = vs->h, prec = vs->prec;
    int nd = L0 + pos;
    int cnt = 1;
    if (pos >= n || n < 2) p = -1;
    while (p >= 0) {
        const int pi = p - b0;
        const int4 Lk = (pi >= 0 && pi < kFanBlock) ? sLink[pi] : make_int4(0, 0, 0, -1);
        const int last = (pi >= 0 && pi < kFanBlock) ? sLast[pi] : b0 + kFanBlock;
        if (Lk.w < b0 || last >= b0 + kFanBlock) {   // p spans the block's boundary
            sSeeds[atomicAdd(&nSeeds, 1)] = nd;       // at most one per thread
            break;
        }
        __threadfence_block();
        int old = atomicAdd(&arrivals[pi], 1);
        if (old == 0) break;
        __threadfence_block();
        const bool isLeft = Lk.x == nd;
        const int sib = isLeft ? Lk.y : Lk.x;
        NodeGeo gs;
        if (sib >= L0) {                             // a leaf: its box and centre are its position
            const float2 q = sLeaf[sib - L0 - b0];
            gs.lox = q.x; gs.loy = q.y; gs.hix = q.x; gs.hiy = q.y; gs.cx = q.x; gs.cy = q.y;
            gs.r2 = 0.0f; gs.deg = 0;
        } else {
            gs = sNode[sib - b0];
        }
        const int cs = (last - Lk.w + 1) - cnt;
        const NodeGeo gl = isLeft ? g : gs, gr = isLeft ? gs : g;
        const int cl = isLeft ? cnt : cs, cr = isLeft ? cs : cnt;
        const NodeGeo m = merge_geo(gl, cl, gr, cr, h, prec, sNode[pi].r2, rootFact);
        sNode[pi] = m;
        geo[p] = m;
        g = m;
        cnt = cl + cr;
        nd = p;
        p = Lk.z;
    }
    // one device-wide slot reservation per workgroup (thousands of single-word
    // atomics on one counter would serialize)
    __syncthreads();
    if (tid == 0) seedBase = nSeeds ? atomicAdd(&vs->nseeds, nSeeds) : 0;
    __syncthreads();
    if (tid < nSeeds) seeds[seedBase + tid] = sSeeds[tid];
}

// A node's record between workgroups of one launch: stores and loads that bypass the
// caches that are not coherent between XCDs.
__device__ __forceinline__ void store_shared(NodeGeo* p, const NodeGeo& g)
{
    unsigned long long w[4];
    __builtin_memcpy(w, &g, sizeof(g));
    for (int q = 0; q < 4; q++)
        __hip_atomic_store((unsigned long long*)p + q, w[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ NodeGeo load_shared(const NodeGeo* p)
{
    unsigned long long w[4];
    for (int q = 0; q < 4; q++)
        w[q] = __hip_atomic_load((const unsigned long long*)p + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    NodeGeo g;
    __builtin_memcpy(&g, w, sizeof(g));
    return g;
}

// Bottom-up pass, level 2: the few block-spanning nodes, device-scope fan-in.  The second
// thread to arrive at a parent merges it.  A thread's record is stored past the caches and
// has arrived (s_waitcnt) before its arrival is counted, and the sibling's is loaded past
// them after: agent-scope fences instead, which write back and invalidate an L2 at every
// step, made this pass 87 us at 1M splats
// (now 47) and 379 us for 16 views of 2M (now 85).
__global__ __launch_bounds__(256) void k_bottom_up_global(const ViewState* __restrict__ vs, NodeGeo* geo,
                                                          const NodeLnk* __restrict__ lnk,
                                                          const NodeAux* __restrict__ aux, int* flags,
                                                          const int* __restrict__ seeds, VStride vsd)
{
    __shared__ float rootFact[kRootFact];
    vs = vw(vs, vsd.ws);
    geo = vw(geo, vsd.ws);
    lnk = vw(lnk, vsd.ws);
    aux = vw(aux, vsd.ws);
    flags = vw(flags, vsd.ws);
    seeds = vw(seeds, vsd.ws);
    const int nseeds = vs->nseeds;
    if ((int)(blockIdx.x * blockDim.x) >= nseeds) return;      // uniform over the workgroup
    root_fact_fill(rootFact);
    __syncthreads();
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nseeds) return;
    const float h = vs->h, prec = vs->prec;
    int nd = seeds[t];
    NodeGeo g = geo[nd];
    NodeLnk own = lnk[nd];
    int cnt = own.count, p = own.parent;
    while (p >= 0) {
        const NodeLnk L = lnk[p];
        const float r2 = geo[p].r2;
        const int old = __hip_atomic_fetch_add(&flags[p], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (old == 0) return;
        asm volatile("" ::: "memory");
        const bool isLeft = L.left == nd;
        const NodeGeo gs = load_shared(geo + (isLeft ? L.right : L.left));
        const int cs = L.count - cnt;
        const NodeGeo gl = isLeft ? g : gs, gr = isLeft ? gs : g;
        g = merge_geo(gl, isLeft ? cnt : cs, gr, isLeft ? cs : cnt, h, prec, r2, rootFact);
        store_shared(geo + p, g);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        cnt = L.count;
        nd = p;
        p = L.parent;
    }
}

// Coefficient blocks.  FGT walks start at the root and at the children of
// nodes with more than k sources (the capacity descent asks for their weights);
// a walk stops at the first node with an expansion.  An internal node below an
// expanded node, with no start in between, is therefore never evaluated and
// gets no block.  The leaves' single coefficients lie first, in leaf order; a workgroup
// reserves its nodes' list entries and blocks behind them with one atomic (where a block
// lies changes no value), which takes the place of a scan over all nodes in three launches.
// The atomics of one word follow one another: workgroups of 1024, 1M splats 81 -> 24 us
// against 256 with an atomic for each of the two counts.
constexpr int kCoefThreads = 1024;
__global__ __launch_bounds__(kCoefThreads) void k_coef_blocks(ViewState* vs, const NodeGeo* __restrict__ geo,
                                                     const NodeLnk* __restrict__ lnk, NodeAux* __restrict__ aux, int k,
                                                     int* momList, VStride vsd)
{
    vs = vw(vs, vsd.ws);
    geo = vw(geo, vsd.ws);
    lnk = vw(lnk, vsd.ws);
    aux = vw(aux, vsd.ws);
    momList = vw(momList, vsd.ws);
    const int n = vs->nc;
    const int nn = 2 * n - 1;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    int d = t < n - 1 ? geo[t].deg : -1;
    if (d >= 0) {
        int x = t;
        while (true) {
            const int p = lnk[x].parent;
            if (p < 0 || lnk[p].count > k) break;           // x starts a walk
            if (geo[p].deg >= 0) { d = -1; break; }          // every walk stops at p
            x = p;
        }
    }
    // list the internal nodes that need moments: one slot reservation per workgroup
    __shared__ unsigned long long sums[kCoefThreads / 64];
    __shared__ unsigned long long base;
    const bool want = d >= 0;
    const unsigned long long m = __ballot(want);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int incl = wave_incl_scan(want ? (d + 1) * (d + 1) : 0);
    if (lane == 63) sums[wid] = (unsigned long long)incl << 32 | (unsigned)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long tot = 0ull;
        for (int q = 0; q < kCoefThreads / 64; q++) tot += sums[q];
        base = tot ? atomicAdd(&vs->blocks, tot) : 0ull;
    }
    __syncthreads();
    unsigned long long at = base;
    for (int q = 0; q < wid; q++) at += sums[q];
    if (want) momList[(int)(unsigned)at + __popcll(m & ((1ull << lane) - 1ull))] = t;
    if (t < nn) aux[t].off = t >= n - 1 ? t - (n - 1) : want ? n + (int)(at >> 32) + incl - (d + 1) * (d + 1) : 0;
}

// Children records of the sampler's walk, one per internal node (after the tree's
// degrees and coefficient offsets are final).
__device__ __forceinline__ SampChild samp_child(int c, const NodeGeo* __restrict__ geo,
                                                const NodeLnk* __restrict__ lnk, const NodeAux* __restrict__ aux)
{
    const NodeGeo g = geo[c];
    SampChild r;
    r.lox = g.lox; r.loy = g.loy; r.hix = g.hix; r.hiy = g.hiy;
    r.cx = g.cx; r.cy = g.cy; r.r2 = g.r2; r.deg = g.deg;
    const NodeAux a = aux[c];
    r.off = a.off; r.count = lnk[c].count; r.id = c; r.first = a.first;
    return r;
}

__device__ __forceinline__ SampRec samp_record(int p, const NodeGeo* __restrict__ geo, const NodeLnk* __restrict__ lnk,
                                               const NodeAux* __restrict__ aux)
{
    const NodeLnk lk = lnk[p];
    SampRec r;
    r.l = samp_child(lk.left, geo, lnk, aux);
    r.r = samp_child(lk.right, geo, lnk, aux);
    return r;
}

// Hermite moments A[a][b] = sum_leaves tx^a ty^b / (a! b!), t = (x - c) / sqrt(2 h^2)
// (hermitefmm.cuh:119-138).  Leaves carry the single coefficient 1.  Internal
// nodes with an expansion are listed by k_coef_blocks; thread (node, row a)
// computes row a of one node, accumulating in FP64 in leaf order.  A workgroup
// of 255 threads covers 15 nodes x 17 rows.
constexpr int kMomNodes = 15;

// 1 / a! as correctly rounded doubles (IEEE division, evaluated at compile time)
constexpr double ifact_c(int a) { double f = 1.0; for (int q = 2; q <= a; q++) f = f * q; return 1.0 / f; }
__constant__ double kInvFact[kMaxDegree + 1] = {
    ifact_c(0), ifact_c(1), ifact_c(2), ifact_c(3), ifact_c(4), ifact_c(5), ifact_c(6), ifact_c(7), ifact_c(8),
    ifact_c(9), ifact_c(10), ifact_c(11), ifact_c(12), ifact_c(13), ifact_c(14), ifact_c(15), ifact_c(16) };
// Row ax of kMomLeaves leaves from position pos on: x^ax / ax! and y.  The leaves' reads are
// in flight together and their power chains interleave; a leaf at a time, each waited for
// its read and then for its own chain (the two bands' degree-6 moments of 1M splats
// 100 -> 63 us, with both bands in one launch).
constexpr int kMomLeaves = 4;
__device__ __forceinline__ void moment_leaves(const float2* __restrict__ leafXY, int pos, int last, const NodeGeo& g,
                                              float is2h, int ax, double ifx, double* mx, double* ty)
{
    double tx[kMomLeaves];
#pragma unroll
    for (int u = 0; u < kMomLeaves; u++) {
        const float2 q = leafXY[pos + u < last ? pos + u : last];
        tx[u] = (double)((q.x - g.cx) * is2h);
        ty[u] = (double)((q.y - g.cy) * is2h);
        mx[u] = 1.0;
    }
    for (int q = 0; q < ax; q++)
#pragma unroll
        for (int u = 0; u < kMomLeaves; u++) mx[u] = mx[u] * tx[u];
#pragma unroll
    for (int u = 0; u < kMomLeaves; u++) mx[u] = mx[u] * ifx;
}

__global__ __launch_bounds__(256) void k_moments(const ViewState* __restrict__ vs, const NodeGeo* __restrict__ geo,
                                                 const NodeAux* __restrict__ aux, const int* __restrict__ momList,
                                                 float* __restrict__ coef, const float2* __restrict__ leafXY,
                                                 const NodeLnk* __restrict__ lnk,
                                                 SampRec* __restrict__ rec, int* __restrict__ walkQueue,
                                                 int* __restrict__ tieQueue, VStride vsd)
{
    vs = vw(vs, vsd.ws);
    geo = vw(geo, vsd.ws);
    aux = vw(aux, vsd.ws);
    momList = vw(momList, vsd.ws);
    coef = vw(coef, vsd.ws);
    leafXY = vw(leafXY, vsd.ws);
    const int n = vs->nc;
    const int L0 = n - 1;
    const int t = threadIdx.x;
    // leaves: 256 per workgroup
    {
        long lf = (long)blockIdx.x * 256 + t;
        if (lf < n) coef[aux[L0 + lf].off] = 1.0f;
        // and the children's record of an internal node for the walks, with empty queues
        if (lf < L0) vw(rec, vsd.ws)[lf] = samp_record((int)lf, geo, vw(lnk, vsd.ws), aux);
        if (lf == 0) { *vw(walkQueue, vsd.ws) = 0; *vw(tieQueue, vsd.ws) = 0; }
    }
    if (t >= kMomNodes * (kMaxDegree + 1)) return;
    const long slot = (long)blockIdx.x * kMomNodes + t / (kMaxDegree + 1);
    const int ax = t % (kMaxDegree + 1);
    if (slot >= (int)(unsigned)vs->blocks) return;
    const int nd = momList[slot];
    NodeGeo g = geo[nd];
    const int p = g.deg;
    if (ax > p) return;
    const float is2h = vs->is2h;
    NodeAux a = aux[nd];
    const int P1 = p + 1;
    const double ifx = kInvFact[ax];
    double acc[kMaxDegree + 1];
#pragma unroll
    for (int bb = 0; bb <= kMaxDegree; bb++) acc[bb] = 0.0;
    for (int pos = a.first; pos <= a.last; pos += kMomLeaves) {
        double mx[kMomLeaves], ty[kMomLeaves];
        moment_leaves(leafXY, pos, a.last, g, is2h, ax, ifx, mx, ty);
#pragma unroll
        for (int u = 0; u < kMomLeaves; u++) {
            if (pos + u > a.last) break;
            double py = 1.0;
#pragma unroll
            for (int bb = 0; bb <= kMaxDegree; bb++) {
                if (bb <= p) {
                    acc[bb] += mx[u] * (py * ifact_c(bb));
                    py = py * ty[u];
                }
            }
        }
    }
#pragma unroll
    for (int bb = 0; bb <= kMaxDegree; bb++)
        if (bb <= p) coef[a.off + ax * P1 + bb] = (float)acc[bb];
}

// ---------------------------------------------------------------------------
// FGT evaluation (evaluateDynamicRadixTree.cuh:128-242, hermitefmm.cuh:35-47, 213-237)
// ---------------------------------------------------------------------------
typedef float f4v __attribute__((ext_vector_type(4)));
typedef int i4v __attribute__((ext_vector_type(4)));

struct TreeView {
    const NodeGeo UD_GLOBAL* geo;
    const NodeLnk UD_GLOBAL* lnk;
    const NodeAux UD_GLOBAL* aux;
    const float UD_GLOBAL* coef;
    float s2h, is2h;
};

__device__ __forceinline__ NodeGeo ld_geo(const TreeView& T, int i)
{
    const f4v UD_GLOBAL* q = (const f4v UD_GLOBAL*)(T.geo + i);
    f4v a = q[0], b = q[1];
    NodeGeo g;
    g.lox = a.x; g.loy = a.y; g.hix = a.z; g.hiy = a.w;
    g.cx = b.x; g.cy = b.y; g.r2 = b.z; g.deg = __float_as_int(b.w);
    return g;
}

__device__ __forceinline__ NodeLnk ld_lnk(const TreeView& T, int i)
{
    i4v a = *(const i4v UD_GLOBAL*)(T.lnk + i);
    NodeLnk l;
    l.left = a.x; l.right = a.y; l.parent = a.z; l.count = a.w;
    return l;
}

__device__ __forceinline__ float eval_node(const TreeView& T, const NodeGeo& g, int nd, float qx, float qy)
{
    int p = g.deg;
    float tx = (qx - g.cx) * T.is2h;
    float ty = (qy - g.cy) * T.is2h;
    float ex = pexpf(-(tx * tx)), ey = pexpf(-(ty * ty));
    const float UD_GLOBAL* c = T.coef + T.aux[nd].off;
    if (p == 0) {
        float w = 0.0f;
        w = w + (c[0] * ex) * ey;
        return w;
    }
    // Hermite functions h_n(t) = 2t h_{n-1} - 2(n-1) h_{n-2}, h_0 = e^{-t^2}
    // (loops unrolled to the maximum degree and predicated, so hy stays in registers).
    // Each term of the series is added with one fused multiply-add,
    // w = fma(c[a][b] h_a, h_b, w): the reference's `weight += coeffs[index] *
    // hermiteX[a] * hermiteY[b]` (hermitefmm.cuh:233) as nvcc's default
    // contraction (-fmad=true) compiles it; each recurrence step is
    // h_n = fma(2t, h_{n-1}, -(2(n-1) h_{n-2})) (hermitefmm.cuh:45), the form
    // of the fixed-order densities below.
    float hy[kMaxDegree + 1];
    hy[0] = ey;
    hy[1] = (2.0f * ty) * ey;
#pragma unroll
    for (int n = 2; n <= kMaxDegree; n++)
        hy[n] = (n <= p) ? __builtin_fmaf(2.0f * ty, hy[n - 1], -((2.0f * (float)(n - 1)) * hy[n - 2])) : 0.0f;
    // a row's loads are issued together, past its end with the last element again
    // (predicated loads would wait for each other)
    float w = 0.0f;
    float hprev = 0.0f, ha = ex;
    for (int a = 0; a <= p; a++) {
        const float UD_GLOBAL* at = c + a * (p + 1);
        float row[kMaxDegree + 1];
#pragma unroll
        for (int b = 0; b <= kMaxDegree; b++) row[b] = at[b < p ? b : p];
        if (a == 1) { hprev = ex; ha = (2.0f * tx) * ex; }
        else if (a >= 2) {
            float hn = __builtin_fmaf(2.0f * tx, ha, -((2.0f * (float)(a - 1)) * hprev));
            hprev = ha; ha = hn;
        }
#pragma unroll
        for (int b = 0; b <= kMaxDegree; b++) {
            const float t = __builtin_fmaf(row[b] * ha, hy[b], w);
            w = b <= p ? t : w;
        }
    }
    return w;
}

// Hermite evaluation with the coefficient block staged in LDS: called by all 64
// lanes of a wavefront for the same node (uniform p and block), so the block
// is fetched with one coalesced load per 64 coefficients and then read with
// LDS broadcasts.  Lanes with act == false only help with the load.
// the degree-P series sum_a sum_b c[a][b] h_a(tx) h_b(ty) with the loops of
// eval_node unrolled exactly (same operation order)
template <int P>
__device__ __forceinline__ float hermite_series(const float* sc, float tx, float ty, float ex, float ey)
{
    float hy[P + 1];
    hy[0] = ey;
    if (P >= 1) hy[P >= 1 ? 1 : 0] = (2.0f * ty) * ey;
#pragma unroll
    for (int n = 2; n <= P; n++) hy[n] = __builtin_fmaf(2.0f * ty, hy[n - 1], -((2.0f * (float)(n - 1)) * hy[n - 2]));
    float w = 0.0f, hprev = 0.0f, ha = ex;
#pragma unroll
    for (int a = 0; a <= P; a++) {
        if (a == 1) { hprev = ex; ha = (2.0f * tx) * ex; }
        else if (a >= 2) {
            float hn = __builtin_fmaf(2.0f * tx, ha, -((2.0f * (float)(a - 1)) * hprev));
            hprev = ha; ha = hn;
        }
#pragma unroll
        for (int b = 0; b <= P; b++) w = __builtin_fmaf(sc[a * (P + 1) + b] * ha, hy[b], w);
    }
    return w;
}

// hermite_series for the higher degrees: the rows in a loop (unrolling 100 and more
// terms makes the compiler hoist their LDS reads into 256 registers), the terms of
// a row unrolled exactly
template <int P>
__device__ __forceinline__ float hermite_rows(const float* sc, float tx, float ty, float ex, float ey)
{
    float hy[P + 1];
    hy[0] = ey;
    hy[1] = (2.0f * ty) * ey;
#pragma unroll
    for (int n = 2; n <= P; n++) hy[n] = __builtin_fmaf(2.0f * ty, hy[n - 1], -((2.0f * (float)(n - 1)) * hy[n - 2]));
    float w = 0.0f, hprev = ex, ha = (2.0f * tx) * ex;
#pragma unroll
    for (int b = 0; b <= P; b++) w = __builtin_fmaf(sc[b] * ex, hy[b], w);
#pragma unroll 1
    for (int a = 1; a <= P; a++) {
        const float* row = sc + a * (P + 1);
#pragma unroll
        for (int b = 0; b <= P; b++) w = __builtin_fmaf(row[b] * ha, hy[b], w);
        const float hn = __builtin_fmaf(2.0f * tx, ha, -((2.0f * (float)a) * hprev));
        hprev = ha; ha = hn;
    }
    return w;
}

// the degree-p expansion at scaled offset (tx, ty), its coefficients in LDS (read by
// broadcast; p wave-uniform), the series unrolled for its degree
__device__ __forceinline__ float hermite_at(const float* sc, int p, float tx, float ty)
{
    const float ex = pexpf(-(tx * tx)), ey = pexpf(-(ty * ty));
    switch (p) {
#define UD_SERIES(P) case P: return hermite_series<P>(sc, tx, ty, ex, ey);
    UD_SERIES(0) UD_SERIES(1) UD_SERIES(2) UD_SERIES(3) UD_SERIES(4) UD_SERIES(5) UD_SERIES(6) UD_SERIES(7)
#undef UD_SERIES
#define UD_SERIES(P) case P: return hermite_rows<P>(sc, tx, ty, ex, ey);
    UD_SERIES(8) UD_SERIES(9) UD_SERIES(10) UD_SERIES(11) UD_SERIES(12) UD_SERIES(13) UD_SERIES(14) UD_SERIES(15)
#undef UD_SERIES
    default: return hermite_rows<kMaxDegree>(sc, tx, ty, ex, ey);
    }
}

__device__ __forceinline__ bool truncated(const NodeGeo& g, float qx, float qy)
{
    float cx = fminf(fmaxf(qx, g.lox), g.hix);
    float cy = fminf(fmaxf(qy, g.loy), g.hiy);
    float dx = qx - cx, dy = qy - cy;
    float d2 = dx * dx;
    d2 = d2 + dy * dy;
    return !(d2 < g.r2);
}

__device__ __forceinline__ float tree_weight(const TreeView& T, int entry, float qx, float qy)
{
    NodeGeo g = ld_geo(T, entry);
    if (g.deg >= 0) return eval_node(T, g, entry, qx, qy);
    int rootparent = T.lnk[entry].parent;
    int nd = entry;
    float w = 0.0f;
    while (true) {
        while (g.deg < 0 && !truncated(g, qx, qy)) { nd = T.lnk[nd].left; g = ld_geo(T, nd); }
        if (g.deg >= 0) w = w + eval_node(T, g, nd, qx, qy);
        int pr = T.lnk[nd].parent;
        while (pr != rootparent && nd == T.lnk[pr].right) { nd = pr; pr = T.lnk[pr].parent; }
        if (pr != rootparent) { nd = T.lnk[pr].right; g = ld_geo(T, nd); }
        else break;   // climbed back to the entry node
    }
    return w;
}


__device__ __forceinline__ float key_of(unsigned long long v) { return __uint_as_float((uint32_t)(v >> 32)); }

// Sampler: one lane per pixel, 8x8 pixel tile per wavefront.
//
// Every FGT weight the descents need is a sequential sum over a subset of the
// frontier of the root's walk (nodes with degree >= 0, or truncated ones that
// contribute 0): the walk from any node n stops exactly where the root's walk
// stops inside n's subtree, because the stop rule depends only on the node and
// the pixel.  So the frontier values of the root's walk, added up for each
// ancestor in traversal order, give W(n) for every node on it bit for bit as the
// reference's per-call walks (evaluateDynamicRadixTree.cuh:128-174) would.  The pass
// records, for each walked node with more than k sources, the weights of its
// two children in a trie of descent states; the ceil(sqrt(k)) descents then
// read weights and capacities from the trie and evaluate the few remaining
// weights (below clusters that were not walked) on demand.  The reference
// keeps the k smallest keys in a sorted insertion list (ties keep insertion
// order, sequentialPoissonRadixTree.cuh:15-41), which k_sample_draw selects.

// An entry holds the weights of its node's two children and their capacities, so
// a descent step reads everything it compares in one round of loads:
// field 0 the left child's capacity, 1 / 2 the left / right weight, 3 the child
// entries, 4 the right child's capacity.  Each wavefront owns one contiguous
// block of the workspace ([tile][entry][field][lane]): lanes that walk the same
// nodes create their entries in step, so their accesses coalesce, and a
// wavefront's whole trie (under 1 MB) sits in one or two pages, so its loads do
// not miss the address-translation caches (with the fields of all tiles
// interleaved, consecutive fields of one entry lay 1 MB apart).
struct TrieRef {
    float UD_GLOBAL* base;          // this lane's slot in its tile's block
    __device__ float get(int e, int f) const { return base[(kTrieFields * e + f) * 64]; }
    __device__ void set(int e, int f, float v) const { base[(kTrieFields * e + f) * 64] = v; }
    __device__ int kids(int e) const { return __float_as_int(get(e, 3)); }
    __device__ void setKids(int e, int v) const { set(e, 3, __int_as_float(v)); }
    // one half of field 3 (left child entry + 1 in the low half, right in the high
    // half), stored alone so that no load of the other half is needed
    __device__ void setKidHalf(int e, bool right, int v) const
    {
        unsigned short UD_GLOBAL* h = (unsigned short UD_GLOBAL*)(base + (kTrieFields * e + 3) * 64);
        h[right ? 1 : 0] = (unsigned short)v;
    }
    __device__ void init(int e, float wUnset) const
    {
        set(e, 0, 1.0f); set(e, 1, wUnset); set(e, 2, wUnset); setKids(e, 0); set(e, 4, 1.0f);
    }
};

// The path of a descent: entry << 1 | side (-1: no capacity to update), probability of
// the step, capacity before it.  The first kPathLds steps in LDS ([step][lane]; a
// descent has about 4 at 1M splats), the rest in private memory.
constexpr int kPathLds = 8;
struct PathStep {
    int at;
    float prob, cap;
};
struct DescentPath {
    int* lds;                       // [3][kPathLds][64], offset by the lane
    int at[kMaxDepth - kPathLds];
    float prob[kMaxDepth - kPathLds], cap[kMaxDepth - kPathLds];
    __device__ void set(int q, int a, float p, float c)
    {
        if (q < kPathLds) {
            lds[q * 64] = a;
            lds[(kPathLds + q) * 64] = __float_as_int(p);
            lds[(2 * kPathLds + q) * 64] = __float_as_int(c);
        } else {
            at[q - kPathLds] = a; prob[q - kPathLds] = p; cap[q - kPathLds] = c;
        }
    }
    __device__ PathStep get(int q) const
    {
        if (q < kPathLds)
            return PathStep{ lds[q * 64], __int_as_float(lds[(kPathLds + q) * 64]),
                             __int_as_float(lds[(2 * kPathLds + q) * 64]) };
        return PathStep{ at[q - kPathLds], prob[q - kPathLds], cap[q - kPathLds] };
    }
};

// The ceil(sqrt(k)) capacity descents of one pixel over its tile's trie (nt entries so
// far), recording each launch's reached leaf range; returns the launches recorded (bad: a
// path or the trie grew past its bound).  The tile's entries are described in LDS: info[e] holds the entries + 1 of its children (left |
// right << 10) and which of them hold rows of the walk (bit 20 left, 21 right),
// node[e] its tree node.
//
// Where only one child of an entry holds rows, its sibling weighs exactly 0 for
// every pixel that reaches the entry, so that child has its parent's weight W, the
// step to it has probability W / W = 1, and the capacities along a run of such
// entries are all the same number: 1 less the probabilities below the run of the
// launches that took it.  A pixel with W > 0 therefore crosses the run in LDS with
// the capacity of its first child (rootCap, or the one in the entry that branches
// above it) and no memory access: a left step always goes left (1 cap < 0 cr never
// holds), a right step goes right while cap > 0 and otherwise left, into a child of
// weight 0, where the general descent goes on.  Entries where both children hold rows
// are stepped as ever; at 1M splats, 512x512 they are 3.6 of the 14.6 steps of a
// descent.  A pixel that steps into a child of weight <= 0 stays with the general
// descent there, in this launch and every other (its weight is fixed), so the
// capacities of a run are kept in one place.  A general part whose steps all find
// weights 0 / 0 goes left at each of them whatever the capacities are, and ends at the
// same leaves with probability NaN each time: it is remembered (memo*).
__device__ __forceinline__ int tile_descents(const TreeView& T, const SampRec UD_GLOBAL* srec, const TrieRef& tr,
                                             int tileEnts, int nt, int TMAX, int k, int L, int L0, float qx, float qy,
                                             float total, const uint32_t* info, const int* node, int* ldsPath,
                                             int2* rch, bool& bad)
{
    const float unset = __builtin_nanf("");              // weight not computed yet
    const float inf = __builtin_huge_valf();
    DescentPath path;
    path.lds = ldsPath;
    float rootCap = 1.0f;
    int memoKey = -1, memoFirst = 0, memoCnt = 0;
    // a tree of at most k leaves is one subtree: no step is taken in it
    const bool inTile = tileEnts > 0 && L0 + 1 > k && total > 0.0f && total < inf;
    int drawn = 0;
    for (int la = 0; la < L; la++) {
        int np = 0, depth = 0, e = 0, side = 0;
        float cap = rootCap, own = total;                // own: clamped weight of the node reached
        i4v ref = { 0, L0 + 1, 0, 0 };                   // the root: all leaves from the first
        while (inTile) {
            const uint32_t inf_ = info[e];
            const uint32_t type = (inf_ >> 20) & 3u;
            depth++;
            if (type == 3u) {
                float wl = fmaxf(0.0f, tr.get(e, 1)), wr = fmaxf(0.0f, tr.get(e, 2));
                const float cl = tr.get(e, 0), cr = tr.get(e, 4);
                const float l0 = wl, r0 = wr, sum = wl + wr;
                wl = wl / sum; wr = wr / sum;
                side = wl * cl < wr * cr ? 1 : 0;
                own = side ? r0 : l0;
                cap = side ? cr : cl;
                path.set(np++, e << 1 | side, side ? wr : wl, cap);
            } else if (type == 2u && !(cap > 0.0f)) {
                path.set(np++, -1, 0.0f, 0.0f);
                side = 0;
                own = 0.0f;
                break;
            } else {
                side = type == 2u ? 1 : 0;
            }
            const int kid = (int)((inf_ >> (10 * side)) & 1023u);
            if (kid == 0 || !(own > 0.0f && own < inf)) break;
            e = kid - 1;
        }
        // child `side` of entry e (or the root): a subtree of at most k leaves, or the
        // general descent
        if (inTile) ref = *((const i4v UD_GLOBAL*)(srec + node[e]) + 3 * side + 2);
        int first = ref.w, cnt = ref.y;
        float prob = 1.0f;
        if (cnt > k && memoKey == (e << 1 | side)) {
            first = memoFirst; cnt = memoCnt; prob = unset;
        } else if (cnt > k) {
            const int key = e << 1 | side;
            int ge = 0, nd = ref.z;
            bool fresh = false;                           // an entry of this step: nothing to load
            if (inTile) {
                const int kids = tr.kids(e);
                ge = (side ? kids >> 16 : kids & 0xffff) - 1;
                if (ge < 0) {
                    if (nt >= TMAX) { bad = true; break; }
                    ge = nt++;
                    fresh = true;
                    tr.setKidHalf(e, side, ge + 1);
                }
            }
            bool still = true;                            // every step so far found 0 / 0
            while (cnt > k) {
                // one round of loads: the children's records and, of an entry that is
                // there already, its weights, children and capacities
                const f4v UD_GLOBAL* rec = (const f4v UD_GLOBAL*)(srec + nd);
                const i4v lref = *(const i4v UD_GLOBAL*)(rec + 2), rref = *(const i4v UD_GLOBAL*)(rec + 5);
                float wl = unset, wr = unset, cl = 1.0f, cr = 1.0f;
                int gk = 0;
                if (!fresh) {
                    wl = tr.get(ge, 1); wr = tr.get(ge, 2);
                    cl = tr.get(ge, 0); cr = tr.get(ge, 4);
                    gk = tr.kids(ge);
                }
                if (wl != wl) {
                    // a child truncated for this pixel weighs 0; others are walked
                    f4v box[2], mid[2];
#pragma unroll
                    for (int c = 0; c < 2; c++) { box[c] = rec[3 * c]; mid[c] = rec[3 * c + 1]; }
                    bool zero[2];
#pragma unroll
                    for (int c = 0; c < 2; c++) {
                        NodeGeo g;
                        g.lox = box[c].x; g.loy = box[c].y; g.hix = box[c].z; g.hiy = box[c].w;
                        g.r2 = mid[c].z;
                        zero[c] = __float_as_int(mid[c].w) < 0 && truncated(g, qx, qy);
                    }
#pragma unroll 1
                    for (int c = 0; c < 2; c++) {              // one copy of the inlined walk
                        float w = 0.0f;
                        if (!(c ? zero[1] : zero[0])) w = tree_weight(T, c ? rref.z : lref.z, qx, qy);
                        tr.set(ge, 1 + c, w);
                        if (c) wr = w; else wl = w;
                    }
                    if (fresh) { tr.set(ge, 0, 1.0f); tr.set(ge, 4, 1.0f); }
                }
                wl = fmaxf(0.0f, wl); wr = fmaxf(0.0f, wr);
                if (ge < tileEnts && wl == 0.0f && wr == 0.0f) {
                    // an entry of the tile whose rows one child holds is stored as 0, 0
                    // (the pixel reached it): that child's weight is the entry's own
                    const uint32_t type = (info[ge] >> 20) & 3u;
                    if (type == 1u) wl = own;
                    if (type == 2u) wr = own;
                }
                const float l0 = wl, r0 = wr, sum = wl + wr;
                wl = wl / sum; wr = wr / sum;
                still = still && wl != wl && wr != wr;
                const bool right = wl * cl < wr * cr;
                own = right ? r0 : l0;
                const i4v to = right ? rref : lref;
                nd = to.z; cnt = to.y; first = to.w;
                int ce = (right ? gk >> 16 : gk & 0xffff) - 1;
                const bool was = fresh;
                fresh = false;
                if (ce < 0) {
                    if (nt >= TMAX) { bad = true; break; }
                    ce = nt++;
                    fresh = true;
                    if (was) tr.setKids(ge, right ? (ce + 1) << 16 : ce + 1);
                    else tr.setKidHalf(ge, right, ce + 1);
                }
                depth++;
                if (depth >= kMaxDepth) { bad = true; break; }
                path.set(np++, ge << 1 | (right ? 1 : 0), right ? wr : wl, right ? cr : cl);
                ge = ce;
            }
            if (bad) break;
            if (still) { memoKey = key; memoFirst = first; memoCnt = cnt; }
        }
        for (int q = np - 1; q >= 0; q--) {
            const PathStep st = path.get(q);
            if (st.at >= 0) tr.set(st.at >> 1, (st.at & 1) ? 4 : 0, fmaxf(0.0f, st.cap - prob));
            prob = prob * st.prob;
        }
        rootCap = fmaxf(0.0f, rootCap - prob);
        rch[(long)la * 64] = make_int2(first, cnt);
        drawn = la + 1;
    }
    return drawn;
}

// Sampler walk: one workgroup of four wavefronts per 8x8 pixel tile, one lane per
// pixel for the weights and the descents.
//
// The union of the 64 pixels' FGT walks is traversed level by level, eight walked
// nodes per wavefront and step: eight lanes take a node, four of them each of its
// children (one 48 B SampChild load), and test the child against 16 pixels each, so a
// step settles 64 children with one round of loads.  A child is evaluated (it carries
// an expansion or is a leaf), walked (some pixel's walk goes below it) or dropped
// (truncated for every pixel that reaches it: it adds nothing).  Both kinds go to LDS
// lists.  The evaluated ones are shared out over the wavefronts (records and
// coefficients fetched ahead); their values for the pixels that reach them are
// stored as rows of 64 floats, 0 for the other pixels.  What the reference asks for
// are sums of those rows in depth-first order: with every node's count of evaluated
// nodes below its left and right child (bottom-up over the levels) and its first
// place in that order (top-down), W of a child is the sum of a contiguous run of rows,
// in order, from 0.  Walked nodes with more than k sources get a trie entry with
// both children's weights, for the descents (k_sample_descend).
//
// One depth-first walk per wavefront waits for a record or a coefficient block at nearly
// every one of its steps, 250 of them per tile on average at 1M splats, 512x512 (555 in the
// densest tile, which set the kernel's time), and its descents load every node of a path:
// walk and descents 1912 us against 464 + 394 us (128x128, 4096 splats: 235 us against
// 47 + 46 us).  Four wavefronts share a tile because a dense tile's own time ends the
// kernel and a small image has fewer tiles than the chip has SIMDs (one wavefront per
// tile, its descents in the same kernel: 1173 us and 118 us).
//
// A tile that outgrows the lists is queued, and the PASSES form, launched next with a
// workgroup for every tile of which those past the queue's end leave at once, takes its
// walk in passes over the leaves: each traverses the tree for the leaves [a, b) only,
// b found by halving, with the walked nodes that reach into them and the evaluated ones
// that begin in them.  In depth-first order a pass's rows follow those of the passes
// before, so the sums go on where those left them: the total in registers, those of the
// walked nodes that reach over a (one per level at most, sPath) in their trie entries.
// Bit for bit the sums of one pass.  A kernel of its own, so that the single pass keeps its
// registers.  Bound by the levels' latency, some 20 levels in each pass.  sampling.sample with
// these tiles walked depth-first by one wavefront each against passes, at 512x512: 4M splats
// a third of the usual size, a few tiles 7.76 -> 4.26 ms, an eighth, half of the tiles 17.1 ->
// 7.5 ms (depth-first throughout 6.2 and 18.2).
constexpr int kWalkWaves = 4;
constexpr int kWalkNodes = 448;      // walked nodes a tile's lists hold (277 in that densest tile)
constexpr int kWalkRows = 448;       // evaluated nodes (220); the trie has rows for as many (walk_extra)
constexpr int kWalkTake = 8;         // evaluated nodes a wavefront takes at a time
constexpr uint32_t kEntOpen = 1u << 22;   // sInfo: the entry's node reaches over an end of a pass

// OR over the four lanes of a quad
__device__ __forceinline__ uint32_t quad_or(uint32_t v)
{
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, false);   // lane ^ 1
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, false);   // lane ^ 2
    return v;
}

// a Hermite coefficient block on its way from memory to LDS (up to 289 floats)
struct CoefFetch {
    float c[5];
    int np;
    __device__ void load(const float UD_GLOBAL* p, int np_, int lane)
    {
        np = np_;
        // every lane loads (the last element past the end), so no lane waits for a branch
        c[0] = p[lane < np ? lane : np - 1];
        c[1] = p[lane + 64 < np ? lane + 64 : np - 1];
        if (np > 128) {
#pragma unroll
            for (int q = 2; q < 5; q++) c[q] = p[lane + 64 * q < np ? lane + 64 * q : np - 1];
        }
    }
    __device__ void store(float* sc, int lane) const
    {
        if (lane < np) sc[lane] = c[0];
        if (lane + 64 < np) sc[lane + 64] = c[1];
        if (np > 128) {
#pragma unroll
            for (int q = 2; q < 5; q++)
                if (lane + 64 * q < np) sc[lane + 64 * q] = c[q];
        }
    }
};

template <bool PASSES>
__global__ __launch_bounds__(64 * kWalkWaves, PASSES ? 4 : 6) void k_sample_walk(int W, int H, int k, int L,
                                                                 const ViewState* __restrict__ vs, const NodeGeo* geo,
                                                                 const NodeLnk* lnk, const NodeAux* aux,
                                                                 const float* coef, const SampRec* __restrict__ srec_,
                                                                 float* trieWs, int tcap,
                                                                 int* __restrict__ tileInfo,
                                                                 int* __restrict__ walkQueue, VStride vsd)
{
    int blk = (int)blockIdx.x;
    if constexpr (PASSES) {
        const int* q = vw(walkQueue, vsd.ws);
        if (blk >= q[0]) return;
        blk = q[1 + blk];
    }
    // walked nodes in level order: the pixels walking below it; its index; parent place
    // | side << 9 | (trie entry + 1) << 10 | first place in depth-first order << 19; its
    // evaluated nodes below the left | right << 16 child
    __shared__ unsigned long long sMask[kWalkNodes];
    __shared__ int sNode[kWalkNodes];
    __shared__ uint32_t sLink[kWalkNodes];
    __shared__ uint32_t sBelow[kWalkNodes];
    __shared__ unsigned short sRowLink[kWalkRows];         // evaluated: parent place | side << 9
    __shared__ unsigned short sRowAt[kWalkRows];           // row at each depth-first place
    __shared__ uint32_t sInfo[kWalkEntries];               // trie entries: children, which hold rows (tile_descents)
    __shared__ int sEntNode[kWalkEntries];                 // their tree nodes
    __shared__ unsigned short sEntAt[kWalkEntries];        // their places among the walked nodes
    __shared__ unsigned short sLevel[kMaxDepth + 1];       // first walked node of each level
    __shared__ float sCoef[kWalkWaves][(kMaxDegree + 1) * (kMaxDegree + 1)];
    __shared__ unsigned long long sCount;                  // walked | evaluated << 20 | entries << 40
    __shared__ int sTicket;
    // passes: trie entry + 1 (0: none) of the walked node of each level that reaches over
    // the first leaf, and over the end; the last leaf at which a node begins
    __shared__ int sPath[PASSES ? kMaxDepth : 1], sNext[PASSES ? kMaxDepth : 1];
    __shared__ int sLast;
    vs = vw(vs, vsd.ws);
    trieWs = vw(trieWs, vsd.ws);
    const SampRec UD_GLOBAL* srec = (const SampRec UD_GLOBAL*)vw(srec_, vsd.ws);
    TreeView T;
    T.geo = (const NodeGeo UD_GLOBAL*)vw(geo, vsd.ws);
    T.lnk = (const NodeLnk UD_GLOBAL*)vw(lnk, vsd.ws);
    T.aux = (const NodeAux UD_GLOBAL*)vw(aux, vsd.ws);
    T.coef = (const float UD_GLOBAL*)vw(coef, vsd.ws);
    T.s2h = vs->s2h;
    T.is2h = vs->is2h;
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int entMax = tcap - walk_extra(L);              // entries the walk may create
    TrieRef tr;
    tr.base = (float UD_GLOBAL*)trieWs + (long)blk * kTrieFields * tcap * 64 + lane;
    float UD_GLOBAL* rows = tr.base + (long)kTrieFields * entMax * 64;     // entries only the descents create
    const int tilesY = (H + 7) >> 3;
    const uint32_t tile = xcd_chunk_remap<kSampTileRun>((uint32_t)blk, gridDim.x);
    const int ti = tile / tilesY, tj = tile - (tile / tilesY) * tilesY;
    const int i = ti * 8 + (lane >> 3), j = tj * 8 + (lane & 7);
    const bool valid = (i < W) && (j < H);
    if (vs->nc <= 0) return;                               // uniform over the launch
    const float qx = (float)i, qy = (float)j;
    const float unset = __builtin_nanf("");              // weight not computed yet
    const unsigned long long lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    bool bad = false;
    float total = 0.0f;
    // value of an expansion or leaf for the pixels of mask, the coefficients in f
    auto eval = [&](const CoefFetch& f, int p, float cx, float cy, unsigned long long mask) {
        f.store(sCoef[wv], lane);
        wave_lds_fence();
        float w = 0.0f;
        if ((mask >> lane) & 1ull) w = hermite_at(sCoef[wv], p, (qx - cx) * T.is2h, (qy - cy) * T.is2h);
        wave_lds_fence();
        return w;
    };
    // ---- the root ----
    const NodeGeo g0 = ld_geo(T, 0);
    const unsigned long long wm0 = __ballot(valid && g0.deg < 0 && !truncated(g0, qx, qy));
    int* tileOut = vw(tileInfo, vsd.ws) + (long)blk * kTileInfo;
    // a tile that evaluates nothing: its weights, 0, start no descent, so that it needs no trie
    auto nothing = [&]() {
        if (wv == 0) {
            if (lane < 2) tileOut[lane] = 0;
            tileOut[64 + lane] = __float_as_int(0.0f);
        }
    };
    const bool skips = !PASSES && g0.deg < 0 && vs->prec > 0.0f;          // uniform
    if (skips && wm0 == 0ull) { nothing(); return; }
    if (threadIdx.x == 0) {
        sMask[0] = wm0; sNode[0] = 0; sLink[0] = 1u << 10;
        sInfo[0] = PASSES ? kEntOpen : 0u; sEntNode[0] = 0; sEntAt[0] = 0;
        sCount = (wm0 ? 1ull : 0ull) | (1ull << 40);
        sTicket = 0;
    }
    if constexpr (PASSES)
        if (threadIdx.x < kMaxDepth) sPath[threadIdx.x] = threadIdx.x == 0 ? 1 : 0;
    __syncthreads();
    int levels = 0, nodes = wm0 ? 1 : 0, evals = 0, nt = 1;
    // passes: this one's leaves are [a, b); entries below nt0 are earlier passes'
    const int leaves = vs->nc;
    int a = 0, b = leaves, nt0 = 1;
    while (true) {
        // ---- traversal ----
        {
            if constexpr (PASSES) {
                // the root again, no node over the end yet
                if (threadIdx.x == 0) {
                    sLink[0] = 1u << 10;
                    sCount = 1ull | ((unsigned long long)nt0 << 40);
                    sTicket = 0;
                    sLast = a;
                }
                if (threadIdx.x < kMaxDepth) sNext[threadIdx.x] = 0;
                __syncthreads();
                levels = evals = 0;
                nodes = 1;
            }
            bool over = false;                                // uniform over the workgroup
            const int slot = lane >> 3, side = (lane >> 2) & 1, quad = lane & 3;
            const float x0 = (float)(ti * 8), y0 = (float)(tj * 8 + 2 * quad);
            int lo = 0, hi = nodes;                           // the level's walked nodes
            while (lo < hi) {
                if (levels >= kMaxDepth - 1) { bad = true; break; }       // a walk below the depth bound
                if (threadIdx.x == 0) sLevel[levels] = (unsigned short)lo;
                levels++;
                for (int b0 = lo + 8 * wv; b0 < hi; b0 += 8 * kWalkWaves) {
                    const int at = b0 + slot;
                    const bool on = at < hi;
                    const f4v UD_GLOBAL* rec = (const f4v UD_GLOBAL*)(srec + (on ? sNode[at] : 0)) + 3 * side;
                    const f4v box = rec[0], mid = rec[1];
                    const i4v ref = *(const i4v UD_GLOBAL*)(rec + 2);
                    const unsigned long long act = on ? sMask[at] : 0ull;
                    const int parentEnt = on ? (int)((sLink[at] >> 10) & 511u) - 1 : -1;
                    const int deg = __float_as_int(mid.w);
                    // !truncated for the 8 x 2 pixels of this lane (same operations per pixel)
                    float dx2[8];
#pragma unroll
                    for (int x = 0; x < 8; x++) {
                        const float px = x0 + (float)x;
                        const float dx = px - fminf(fmaxf(px, box.x), box.z);
                        dx2[x] = dx * dx;
                    }
                    uint32_t in[2] = { 0u, 0u };
#pragma unroll
                    for (int y = 0; y < 2; y++) {
                        const float py = y0 + (float)y;
                        const float dy = py - fminf(fmaxf(py, box.y), box.w);
                        const float dy2 = dy * dy;
#pragma unroll
                        for (int x = 0; x < 8; x++) in[x >> 2] |= dx2[x] + dy2 < mid.z ? 1u << (8 * (x & 3) + y) : 0u;
                    }
                    const uint32_t inLo = quad_or(in[0] << (2 * quad)), inHi = quad_or(in[1] << (2 * quad));
                    const unsigned long long walk = act & (((unsigned long long)inHi << 32) | inLo);
                    const bool lead = on && quad == 0;
                    bool isEval = lead && deg >= 0;
                    bool isWalk = lead && deg < 0 && walk != 0ull;
                    bool wantEnt = isWalk && ref.y > k && parentEnt >= 0;
                    const int from = ref.w, upto = ref.w + ref.y;             // the child's leaves
                    if constexpr (PASSES) {
                        isEval &= from >= a && from < b;
                        isWalk &= from < b && upto > a;
                        wantEnt &= isWalk && from >= a;
                        if (isEval || isWalk) atomicMax(&sLast, from);
                    }
                    const unsigned long long bw = __ballot(isWalk), be = __ballot(isEval), bt = __ballot(wantEnt);
                    unsigned long long base = 0;
                    if (lane == 0)
                        base = atomicAdd(&sCount, (unsigned long long)__popcll(bw) | ((unsigned long long)__popcll(be) << 20) |
                                                      ((unsigned long long)__popcll(bt) << 40));
                    base = ((unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane((int)(base >> 32)) << 32) |
                           (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
                    const int to = (int)(base & 0xfffffu) + __popcll(bw & lt);
                    const int row = (int)((base >> 20) & 0xfffffu) + __popcll(be & lt);
                    int ent = wantEnt ? (int)(base >> 40) + __popcll(bt & lt) : -1;
                    if (ent >= entMax) ent = -1;
                    const bool fresh = ent >= 0;
                    if constexpr (PASSES)
                        if (isWalk && from < a) ent = sPath[levels] - 1;
                    if (isWalk && to < kWalkNodes) {
                        sMask[to] = walk;
                        sNode[to] = ref.z;
                        sLink[to] = (uint32_t)at | ((uint32_t)side << 9) | ((uint32_t)(ent + 1) << 10);
                        if (fresh) {
                            sInfo[ent] = PASSES && upto > b ? kEntOpen : 0u;
                            sEntNode[ent] = ref.z;
                            sEntAt[ent] = (unsigned short)to;
                            atomicOr(&sInfo[parentEnt], (uint32_t)(ent + 1) << (10 * side));
                        }
                        if constexpr (PASSES)
                            if (upto > b) sNext[levels] = ent + 1;
                    }
                    if (isEval && row < kWalkRows) sRowLink[row] = (unsigned short)(at | (side << 9));
                }
                __syncthreads();
                const unsigned long long c = sCount;
                nodes = (int)(c & 0xfffffu);
                evals = (int)((c >> 20) & 0xfffffu);
                nt = (int)(c >> 40);
                if (nodes > kWalkNodes || evals > kWalkRows) {
                    if constexpr (!PASSES) {                              // left to the passes
                        if (threadIdx.x == 0) {
                            int* q = vw(walkQueue, vsd.ws);
                            q[1 + atomicAdd(q, 1)] = blk;
                        }
                        return;
                    }
                    over = true;
                    break;
                }
                lo = hi;
                hi = nodes;
                __syncthreads();                               // sCount is read before the next level adds to it
            }
            if constexpr (PASSES) {
                if (over) {
                    // half the leaves at which nodes begin.  A list of 448 overflows over at
                    // least 7 of them, since at most 64 nodes begin at one: a < b < the old b
                    b = a + (sLast - a + 1) / 2;
                    if (b <= a) { bad = true; nt = nt0; break; }
                    // the links to this traversal's entries go
                    if (threadIdx.x < kMaxDepth && sPath[threadIdx.x] > 0) {
                        uint32_t& x = sInfo[sPath[threadIdx.x] - 1];
                        if ((int)(x & 1023u) > nt0) x &= ~1023u;
                        if ((int)((x >> 10) & 1023u) > nt0) x &= ~(1023u << 10);
                    }
                    __syncthreads();
                    continue;
                }
            }
            if (nt > entMax) nt = entMax;
        }
        if (skips && evals == 0 && !bad) { nothing(); return; }
        if (nodes > 0 && !bad) {
            // the trie entries by number, in a pass those of its walked nodes
            const int items = PASSES ? nodes : nt;
            auto entry_of = [&](int it) { return PASSES ? (int)((sLink[it] >> 10) & 511u) - 1 : it; };
            auto place_of = [&](int it) { return PASSES ? it : (int)sEntAt[it]; };
            // ---- places (first wavefront) ----
            if (wv == 0) {
                if (lane == 0) sLevel[levels] = (unsigned short)nodes;
                for (int x = lane; x < nodes; x += 64) sBelow[x] = 0u;
                wave_lds_fence();
                // evaluated nodes below each side, bottom-up
                for (int e = lane; e < evals; e += 64) {
                    const uint32_t l = sRowLink[e];
                    atomicAdd(&sBelow[l & 511u], 1u << (16 * (l >> 9)));
                }
                wave_lds_fence();
                for (int d = levels - 1; d > 0; d--) {
                    for (int x = sLevel[d] + lane; x < sLevel[d + 1]; x += 64) {
                        const uint32_t l = sLink[x], c = sBelow[x];
                        atomicAdd(&sBelow[l & 511u], ((c & 0xffffu) + (c >> 16)) << (16 * ((l >> 9) & 1u)));
                    }
                    wave_lds_fence();
                }
                // first places in depth-first order, top-down (the root's is 0)
                for (int d = 1; d < levels; d++) {
                    for (int x = sLevel[d] + lane; x < sLevel[d + 1]; x += 64) {
                        const uint32_t l = sLink[x], up = l & 511u;
                        const uint32_t first = (sLink[up] >> 19) + (((l >> 9) & 1u) ? sBelow[up] & 0xffffu : 0u);
                        sLink[x] = l | (first << 19);
                    }
                    wave_lds_fence();
                }
                for (int e = lane; e < evals; e += 64) {
                    const uint32_t l = sRowLink[e], up = l & 511u;
                    sRowAt[(sLink[up] >> 19) + ((l >> 9) ? sBelow[up] & 0xffffu : 0u)] = (unsigned short)e;
                }
                for (int t = lane; t < items; t += 64) {
                    const int ent = entry_of(t);
                    if (PASSES && ent < 0) continue;
                    const uint32_t c = sBelow[place_of(t)];
                    sInfo[ent] |= ((c & 0xffffu) ? 1u << 20 : 0u) | ((c >> 16) ? 1u << 21 : 0u);
                }
            }
            // ---- values: kWalkTake nodes at a time, the next ones' records in flight ----
            {
                struct Take {
                    f4v mid;
                    int off, first, num;
                    unsigned long long mask;
                };
                auto take = [&]() {
                    Take t;
                    int b = 0;
                    if (lane == 0) b = atomicAdd(&sTicket, kWalkTake);
                    t.first = __builtin_amdgcn_readfirstlane(b);
                    t.num = evals - t.first < kWalkTake ? evals - t.first : kWalkTake;
                    const uint32_t l = lane < t.num ? sRowLink[t.first + lane] : 0u;
                    const f4v UD_GLOBAL* rec = (const f4v UD_GLOBAL*)(srec + sNode[l & 511u]) + 3 * (l >> 9);
                    t.mid = rec[1];
                    t.off = ((const i4v UD_GLOBAL*)(rec + 2))->x;
                    t.mask = sMask[l & 511u];
                    return t;
                };
                Take next = take();
                while (next.num > 0) {                         // wave-uniform
                    const Take t = next;
                    next = take();
                    auto coefs = [&](int q, CoefFetch& f) {
                        const int p = __builtin_amdgcn_readlane(__float_as_int(t.mid.w), q);
                        f.load(T.coef + __builtin_amdgcn_readlane(t.off, q), (p + 1) * (p + 1), lane);
                    };
                    CoefFetch f;
                    coefs(0, f);
                    for (int q = 0; q < t.num; q++) {
                        const CoefFetch cur = f;
                        if (q + 1 < t.num) coefs(q + 1, f);
                        const unsigned long long m =
                            ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(t.mask >> 32), q) << 32) |
                            (uint32_t)__builtin_amdgcn_readlane((int)t.mask, q);
                        rows[(long)(t.first + q) * 64] =
                            eval(cur, __builtin_amdgcn_readlane(__float_as_int(t.mid.w), q),
                                 __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t.mid.x), q)),
                                 __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t.mid.y), q)), m);
                    }
                }
            }
            __syncthreads();
            // ---- sums ----
            // N sums of rows at once, num[q] of them from place at[q] on, each in order
            auto sums = [&](auto count, const int* at, const int* num, float* out) {
                constexpr int N = decltype(count)::value;
                int m = 0;
#pragma unroll
                for (int q = 0; q < N; q++) m = num[q] > m ? num[q] : m;
                for (int r = 0; r < m; r += 16 / N) {
                    float v[N][16 / N];
#pragma unroll
                    for (int u = 0; u < 16 / N; u++)
#pragma unroll
                        for (int q = 0; q < N; q++)
                            v[q][u] = r + u < num[q] ? rows[(long)sRowAt[at[q] + r + u] * 64] : 0.0f;
#pragma unroll
                    for (int u = 0; u < 16 / N; u++)           // adding 0 past the end changes nothing
#pragma unroll
                        for (int q = 0; q < N; q++) out[q] = out[q] + v[q][u];
                }
            };
            if (wv == 0) {
                const int at0 = 0;
                sums(std::integral_constant<int, 1>{}, &at0, &evals, &total);
            } else {
                // trie entries.  Where one child holds all rows, only pixels of weight <= 0
                // there read the weights (tile_descents): 0 and 0 for a pixel that reached it
                auto put = [&](int ent, bool mine, float wl, float wr) {
                    const uint32_t kids = sInfo[ent];
                    tr.set(ent, 0, 1.0f);
                    tr.set(ent, 1, mine ? wl : unset);
                    tr.set(ent, 2, mine ? wr : unset);
                    tr.setKids(ent, (int)((kids & 1023u) | (((kids >> 10) & 1023u) << 16)));
                    tr.set(ent, 4, 1.0f);
                };
                for (int c0 = 0; c0 < items; c0 += 64 * (kWalkWaves - 1)) {
                    const int mine = c0 + lane * (kWalkWaves - 1) + wv - 1;       // this lane's entry
                    const bool has = mine < items && (!PASSES || entry_of(mine) >= 0);
                    const uint32_t type = sInfo[has ? entry_of(mine) : 0] >> 20;
                    // one that reaches over an end of the pass keeps its sums
                    const bool both = has && (PASSES ? (type & 3u) == 3u || type >= kEntOpen >> 20 : type == 3u);
                    unsigned long long plain = __ballot(has && !both), branch = __ballot(both);
                    auto item = [&](int q) { return c0 + q * (kWalkWaves - 1) + wv - 1; };
                    while (plain) {
                        const int it = item(__builtin_ctzll(plain));
                        plain &= plain - 1;
                        put(entry_of(it), (sMask[place_of(it)] >> lane) & 1ull, 0.0f, 0.0f);
                    }
                    while (branch) {                                // two at a time: 16 row loads in flight
                        int it[2], ent[2], at[4], num[4];
                        float w[4] = { 0.0f, 0.0f, 0.0f, 0.0f };
                        it[0] = item(__builtin_ctzll(branch));
                        branch &= branch - 1;
                        const bool two = branch != 0ull;
                        it[1] = two ? item(__builtin_ctzll(branch)) : it[0];
                        branch &= branch - 1;
#pragma unroll
                        for (int q = 0; q < 2; q++) {
                            ent[q] = __builtin_amdgcn_readfirstlane(entry_of(it[q]));
                            const int x = __builtin_amdgcn_readfirstlane(place_of(it[q]));
                            if (PASSES && a > 0 && ent[q] < nt0 && ((sMask[x] >> lane) & 1ull)) {
                                w[2 * q] = tr.get(ent[q], 1);           // of the passes before
                                w[2 * q + 1] = tr.get(ent[q], 2);
                            }
                            const uint32_t below = __builtin_amdgcn_readfirstlane(sBelow[x]);
                            at[2 * q] = (int)(__builtin_amdgcn_readfirstlane(sLink[x]) >> 19);
                            num[2 * q] = q == 0 || two ? (int)(below & 0xffffu) : 0;
                            at[2 * q + 1] = at[2 * q] + num[2 * q];
                            num[2 * q + 1] = q == 0 || two ? (int)(below >> 16) : 0;
                        }
                        sums(std::integral_constant<int, 4>{}, at, num, w);
                        put(ent[0], (sMask[place_of(it[0])] >> lane) & 1ull, w[0], w[1]);
                        if (two) put(ent[1], (sMask[place_of(it[1])] >> lane) & 1ull, w[2], w[3]);
                    }
                }
            }
            __syncthreads();
        }
        if (!PASSES || bad || b >= leaves) break;
        if constexpr (PASSES) {
            // as many leaves again, more after a pass that left room
            const int span = b - a, used = nodes > evals ? nodes : evals;
            const long more = (long)span * (used < kWalkNodes / 8 ? 16 : used < kWalkNodes / 2 ? 2 : 1);
            a = b;
            b = more < leaves - a ? a + (int)more : leaves;
            nt0 = nt;
            if (threadIdx.x < kMaxDepth) sPath[threadIdx.x] = threadIdx.x == 0 ? 1 : sNext[threadIdx.x];
        }
    }
    // ---- for k_sample_descend: the pixels' totals, the entries of the trie ----
    const int tileEnts = nodes > 0 ? nt : 0;
    for (int t = threadIdx.x; t < tileEnts; t += 64 * kWalkWaves) {
        tileOut[128 + t] = (int)(sInfo[t] & ~kEntOpen);
        tileOut[128 + kWalkEntries + t] = sEntNode[t];
    }
    if (wv > 0) return;
    if (nodes == 0) {
        if (g0.deg >= 0) {
            CoefFetch f;
            f.load(T.coef + T.aux[0].off, (g0.deg + 1) * (g0.deg + 1), lane);
            total = eval(f, g0.deg, g0.cx, g0.cy, __ballot(valid));
        }
        tr.init(0, unset);
    }
    if (lane == 0) { tileOut[0] = tileEnts; tileOut[1] = bad ? 1 : 0; }
    tileOut[64 + lane] = __float_as_int(total);
}

// The capacity descents of every tile k_sample_walk finished, one lane per pixel.  A
// pass of its own: a tile's descents take one wavefront where its walk takes four,
// and as long as both together (the slowest tile, whose pixels weigh subtrees on
// demand, sets this pass's time: all tiles are in flight at once at 512x512).
__global__ __launch_bounds__(64, 4) void k_sample_descend(int W, int H, int k, int L, const ViewState* __restrict__ vs,
                                                       const NodeGeo* geo, const NodeLnk* lnk, const NodeAux* aux,
                                                       const float* coef, const SampRec* __restrict__ srec,
                                                       float* trieWs, int tcap, const int* __restrict__ tileInfo,
                                                       int2* __restrict__ reach, int* __restrict__ errOut,
                                                       VStride vsd)
{
    __shared__ uint32_t sInfo[kWalkEntries];
    __shared__ int sEntNode[kWalkEntries];
    __shared__ int sPath[3 * kPathLds * 64];
    vs = vw(vs, vsd.ws);
    trieWs = vw(trieWs, vsd.ws);
    reach = vw(reach, vsd.ws);
    const int* tile_ = vw(tileInfo, vsd.ws) + (long)blockIdx.x * kTileInfo;
    TreeView T;
    T.geo = (const NodeGeo UD_GLOBAL*)vw(geo, vsd.ws);
    T.lnk = (const NodeLnk UD_GLOBAL*)vw(lnk, vsd.ws);
    T.aux = (const NodeAux UD_GLOBAL*)vw(aux, vsd.ws);
    T.coef = (const float UD_GLOBAL*)vw(coef, vsd.ws);
    T.s2h = vs->s2h;
    T.is2h = vs->is2h;
    const int lane = threadIdx.x;
    const int n = vs->nc;
    const bool runTree = n > 0;
    const int ents = runTree ? tile_[0] : 0;
    for (int t = lane; t < ents; t += 64) {
        sInfo[t] = (uint32_t)tile_[128 + t];
        sEntNode[t] = tile_[128 + kWalkEntries + t];
    }
    wave_lds_fence();
    TrieRef tr;
    tr.base = (float UD_GLOBAL*)trieWs + (long)blockIdx.x * kTrieFields * tcap * 64 + lane;
    const int tilesY = (H + 7) >> 3;
    const uint32_t tile = xcd_chunk_remap<kSampTileRun>(blockIdx.x, gridDim.x);
    const int ti = tile / tilesY, tj = tile - (tile / tilesY) * tilesY;
    const int i = ti * 8 + (lane >> 3), j = tj * 8 + (lane & 7);
    const bool valid = (i < W) && (j < H);
    int2* rch = reach + (long)blockIdx.x * L * 64 + lane;   // [launch][lane] of this tile
    int drawn = 0;                                      // launches whose leaf range is recorded
    if (valid && runTree) {
        const float total = fmaxf(0.0f, __int_as_float(tile_[64 + lane]));
        bool bad = tile_[1] != 0;
        if (!bad && total >= vs->prec)
            drawn = tile_descents(T, (const SampRec UD_GLOBAL*)vw(srec, vsd.ws), tr, ents, ents > 0 ? ents : 1, tcap, k, L,
                                  n - 1, (float)i, (float)j, total, sInfo, sEntNode, sPath + lane, rch, bad);
        if (bad) atomicOr(errOut, 1);
    }
    for (int la = drawn; la < L; la++) rch[(long)la * 64] = make_int2(0, 0);
}

// The key u / E(leaf) of one candidate as its bit pattern (keys are positive, so
// the patterns order like the floats); kNoKey where the key is not finite (E = 0:
// never inserted).
constexpr uint32_t kNoKey = 0xffffffffu;
constexpr uint32_t kInfKey = 0x7f800000u;
__device__ __forceinline__ uint32_t draw_key(float qx, float qy, float2 xy, float is2h, uint32_t x)
{
    float tx = (qx - xy.x) * is2h;
    float ty = (qy - xy.y) * is2h;
    float ex = pexpf(-(tx * tx)), ey = pexpf(-(ty * ty));
    float wgt = 0.0f;
    wgt = wgt + (1.0f * ex) * ey;
    float p = fmaxf(0.0f, wgt);
    float key = u01(x) / p;
    return key < __builtin_huge_valf() ? __float_as_uint(key) : kNoKey;
}

// draw_key and the draw number (launch << 16 | ordinal) as one word (replay)
__device__ __forceinline__ bool draw_word(float qx, float qy, float2 xy, float is2h, uint32_t x, int la, int ord,
                                          unsigned long long& ent)
{
    const uint32_t key = draw_key(qx, qy, xy, is2h, x);
    if (key == kNoKey) return false;
    ent = ((unsigned long long)key << 32) | (uint32_t)((la << 16) | ord);
    return true;
}

// Sequential Poisson keys over the leaves each launch reached (the walk's
// capacity descents do not depend on the keys, so they run first, in
// k_sample_descend): in a Karras tree the leaves of a subtree are the contiguous
// sorted range [first, first + count), in the left-to-right order nextLeaf visits
// (sequentialPoissonDynamicTree.cuh:16-53), and every leaf carries the single
// Hermite coefficient 1, so E(leaf) = e^{-tx^2} e^{-ty^2}.  Key u / E with u the
// Philox word of (leaf ordinal, launch, pixel, view).  The reference keeps the
// keys in a sorted list of k slots, inserting with a strict < and carrying each
// displaced entry down (insertSample, sequentialPoissonRadixTree.cuh:15-41); with
// distinct keys that list is the k smallest keys in order.
//
// One wavefront per pixel.  A lane keys one Philox block (four leaves of one
// launch) per iteration: at most L ceil(k / 4) blocks, since a descent stops at a
// subtree of at most k leaves, so all keys of a pixel stay in 4 IT registers.  A
// threshold that between k and 64 ROWS keys meet is found by galloping and
// bisection on the key bits (ballots and scalar counts, a few steps); the keys
// below it are compacted into LDS, ranked by comparison with LDS broadcasts, and
// written in rank order as one coalesced row.  A lane per pixel with its k best
// keys in an LDS heap ran the pixel's about 210 candidates and 120 heap
// replacements as one serial chain at 2 wavefronts per SIMD (the heap's 20 KB):
// 673 us at 1M splats, 512x512, k = 40 (now 261 us) and 226 us at 128x128, where
// 256 wavefronts left most of the chip idle (now 19 us).
//
// Equal keys are where the reference's list differs from a sort: a carried entry
// passes over entries equal to it, so an insertion ahead of a run of equal keys
// moves the run's first entry to the run's end, and a full list drops the front
// of its last run.  A pixel with two equal keys among those at or below the
// threshold queues itself (tieQueue: its sampler lane and its k-th smallest key,
// infinite with fewer than k keys), and k_sample_replay redraws it through the
// reference's insertion.
//
// A pixel that no launch drew for gets its empty slots at once.  From kDrawManyTiles tiles on a
// wavefront takes 16 pixels of a tile one after another, the empty ones found for all of them
// with one load (up to two rows of keys; with four the loop's registers cost more).  2048x1024
// under 6400 splats, k = 40, 4 % of the pixels not empty: 1420 -> 190 us; under 16, k = 8: 641
// -> 52.  At 512x512, half the line's tiles, turns save nothing under 100 000 splats at k = 40
// and cost 7 % at k = 64.
constexpr int kDrawWaves = 4;
constexpr int kDrawTurns = 16;
constexpr long kDrawManyTiles = 8192;

// pixels of the tile that some launch drew for: where one did, the first did
__device__ __forceinline__ unsigned long long drawn_pixels(const int2* __restrict__ reach, int blk, int L, int lane)
{
    return __ballot(reach[(long)blk * L * 64 + lane].y > 0);
}

// empty slots for the 16 pixels from pl on of a tile: two of its columns, each contiguous
__device__ __forceinline__ void empty_columns(int W, int H, int k, int ti, int tj, int pl, int lane, int32_t* out)
{
    const int j = tj * 8, n = min(8, H - j) * k;
    for (int c = 0; c < 2; c++) {
        const int i = ti * 8 + (pl >> 3) + c;
        if (i >= W) break;
        for (int x = lane; x < n; x += 64) out[((long)j + (long)H * i) * k + x] = -1;
    }
}

template <int ROWS, int IT, int TURNS>
__global__ __launch_bounds__(64 * kDrawWaves) void k_sample_draw(int W, int H, int k, int L, int tiles,
                                                                 uint32_t seedLo, uint32_t seedHi, uint32_t view,
                                                                 const ViewState* __restrict__ vs,
                                                                 const float2* __restrict__ leafXY,
                                                                 const int32_t* __restrict__ leafId,
                                                                 const int2* __restrict__ reach,
                                                                 int32_t* __restrict__ out, int* __restrict__ tieQueue,
                                                                 VStride vsd)
{
    vs = vw(vs, vsd.ws);
    leafXY = vw(leafXY, vsd.ws);
    leafId = vw(leafId, vsd.ws);
    reach = vw(reach, vsd.ws);
    tieQueue = vw(tieQueue, vsd.ws);
    view += blockIdx.y;
    out += (long)blockIdx.y * W * H * k;
    constexpr int CAP = 64 * ROWS;
    __shared__ __align__(16) uint32_t sKey[kDrawWaves][CAP];
    __shared__ int sPos[kDrawWaves][CAP];
    __shared__ int sOwner[kDrawWaves][CAP];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    // the blocks of a sampler tile run on the XCD its walk ran on (tile t was
    // workgroup t of the walk: XCD t mod 8), whose L2 holds its reached ranges and
    // most of its leaves
    constexpr int per = 64 / (kDrawWaves * TURNS);      // workgroups per tile
    const int full = tiles & ~7, d = blockIdx.x;
    const int blk = d < full * per ? (d >> 3) / per * 8 + (d & 7) : d / per;
    const int pl0 = ((d < full * per ? (d >> 3) % per : d % per) * kDrawWaves + wv) * TURNS;
    const int tilesY = (H + 7) >> 3;
    const uint32_t tile = xcd_chunk_remap<kSampTileRun>((uint32_t)blk, (uint32_t)tiles);
    const int ti = tile / tilesY, tj = tile - (tile / tilesY) * tilesY;
    const float is2h = vs->is2h;
    const unsigned long long some = TURNS > 1 ? drawn_pixels(reach, blk, L, lane) : ~0ull;
    if (TURNS > 1 && some == 0ull) { empty_columns(W, H, k, ti, tj, pl0, lane, out); return; }
#pragma unroll 1
    for (int turn = 0; turn < TURNS; turn++) {
        const int pl = pl0 + turn;
        const int i = ti * 8 + (pl >> 3), j = tj * 8 + (pl & 7);
        if (i >= W || j >= H) continue;                     // wave-uniform
        const float qx = (float)i, qy = (float)j;
        const uint32_t pixel = (uint32_t)(j + H * i);
        int2 fc = make_int2(0, 0);
        if (((some >> pl) & 1ull) && lane < L) fc = reach[((long)blk * L + lane) * 64 + pl];
        if (__ballot(fc.y > 0) == 0ull) {
            for (int s = lane; s < k; s += 64) out[(long)pixel * k + s] = -1;
            continue;
        }
        uint32_t key[4 * IT];
        int pos[IT];
        int blocks = 0;                                     // Philox blocks of the pixel
#pragma unroll
        for (int it = 0; it < IT; it++) {
            if (it > 0 && blocks <= 64 * it) {              // wave-uniform
#pragma unroll
                for (int q = 0; q < 4; q++) key[4 * it + q] = kNoKey;
                pos[it] = 0;
                continue;
            }
            const int t = it * 64 + lane;
            int la = 0, kk0 = 0, first = 0, cnt = 0;
            blocks = 0;
            for (int l = 0; l < L; l++) {
                const int f = __builtin_amdgcn_readlane(fc.x, l), c = __builtin_amdgcn_readlane(fc.y, l);
                const int nb = (c + 3) >> 2;
                if (t >= blocks && t < blocks + nb) { la = l; kk0 = 4 * (t - blocks); first = f; cnt = c; }
                blocks += nb;
            }
            const u32x4 rnd = philox4x32_10(u32x4{ (uint32_t)(kk0 >> 2), (uint32_t)la, pixel, view }, seedLo, seedHi);
            pos[it] = first + kk0;
            float2 xy[4];
#pragma unroll
            for (int q = 0; q < 4; q++) xy[q] = kk0 + q < cnt ? leafXY[pos[it] + q] : make_float2(0.0f, 0.0f);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t kb = draw_key(qx, qy, xy[q], is2h,
                                             (q == 0) ? rnd.x : (q == 1) ? rnd.y : (q == 2) ? rnd.z : rnd.w);
                key[4 * it + q] = kk0 + q < cnt ? kb : kNoKey;
            }
        }
        auto count = [&](uint32_t x) {
            int c = 0;
#pragma unroll
            for (int e = 0; e < 4 * IT; e++) c += __popcll(__ballot(key[e] <= x));
            return c;
        };
        // threshold: every finite key if at most CAP, else one that k .. CAP keys meet
        uint32_t thr = kInfKey - 1;
        int m = count(thr);
        bool tie = false;
        uint32_t kth = kInfKey;                             // the k-th smallest key
        if (m > CAP) {
            uint32_t lo = 0, hi = kInfKey - 1, step = 1u << 23;   // count(lo) < k, count(hi) > CAP
            uint32_t mid = 0x3f800000u;                     // keys lie around 1: gallop by octaves from there
            while (true) {
                m = count(mid);
                if (m >= k && m <= CAP) { thr = mid; break; }
                const bool up = m < k;
                if (up) lo = mid; else hi = mid;
                if (hi - lo <= 1) { tie = true; kth = hi; break; }    // more than CAP - k keys equal hi
                if (up && hi == kInfKey - 1) mid = hi - mid > step ? mid + step : lo + ((hi - lo) >> 1);
                else if (!up && lo == 0) mid = mid > step ? mid - step : hi >> 1;
                else mid = lo + ((hi - lo) >> 1);
                if (step < 1u << 30) step <<= 1;            // 2^30 spans the keys above 1; past that, halve
            }
        }
        if (!tie) {
            uint32_t* sk = sKey[wv];
            int base = 0;
#pragma unroll
            for (int e = 0; e < 4 * IT; e++) {
                const bool in = key[e] <= thr;
                const unsigned long long mk = __ballot(in);
                const int at = base + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(mk >> 32),
                                                                     __builtin_amdgcn_mbcnt_lo((unsigned)mk, 0));
                if (in) { sk[at] = key[e]; sPos[wv][at] = pos[e >> 2] + (e & 3); }
                base += __popcll(mk);
            }
#pragma unroll
            for (int r = 0; r < ROWS; r++)
                if (r * 64 + lane >= m) sk[r * 64 + lane] = kNoKey;
            wave_lds_fence();
            uint32_t mine[ROWS];
            int id[ROWS], rank[ROWS];
#pragma unroll
            for (int r = 0; r < ROWS; r++) {
                const int e = r * 64 + lane;
                mine[r] = sk[e];
                id[r] = e < m ? leafId[sPos[wv][e]] : -1;
                rank[r] = 0;
            }
            for (int q0 = 0; q0 < CAP; q0 += 16) {
                if (q0 >= m) break;                         // wave-uniform
                uint32_t o[16];
#pragma unroll
                for (int q = 0; q < 16; q += 4) {
                    const uint4 v = *(const uint4*)(sk + q0 + q);
                    o[q] = v.x; o[q + 1] = v.y; o[q + 2] = v.z; o[q + 3] = v.w;
                }
#pragma unroll
                for (int q = 0; q < 16; q++)
#pragma unroll
                    for (int r = 0; r < ROWS; r++) rank[r] += o[q] < mine[r];
            }
            // equal keys share a rank: of the lanes writing one place, one reads its own entry back
#pragma unroll
            for (int r = 0; r < ROWS; r++)
                if (r * 64 + lane < m) sOwner[wv][rank[r]] = r * 64 + lane;
            wave_lds_fence();
            bool dup = false;
            uint32_t top = 0;
#pragma unroll
            for (int r = 0; r < ROWS; r++) {
                if (r * 64 + lane >= m) continue;
                dup |= sOwner[wv][rank[r]] != r * 64 + lane;
                if (rank[r] < k && mine[r] > top) top = mine[r];
            }
            tie = __ballot(dup) != 0ull;
            if (tie && m >= k) {
                for (int o = 32; o > 0; o >>= 1) {
                    const uint32_t x = (uint32_t)__shfl_xor((int)top, o, 64);
                    top = x > top ? x : top;
                }
                kth = top;
            }
            wave_lds_fence();
            int32_t* o = out + (long)pixel * k;
            if (!tie) {
                int* so = sOwner[wv];                       // ids in rank order
#pragma unroll
                for (int r = 0; r < ROWS; r++)
                    if (r * 64 + lane < m) so[rank[r]] = id[r];
                wave_lds_fence();
                for (int s = lane; s < k; s += 64) o[s] = s < m ? so[s] : -1;
            }
        }
        if (tie && lane == 0) {
            const int e = atomicAdd(tieQueue, 1);
            tieQueue[1 + 2 * e] = blk * 64 + pl;
            tieQueue[2 + 2 * e] = (int)kth;
        }
        wave_lds_fence();
    }
}

// The same with two pixels per wavefront, in halves, where a pixel has at most 32 Philox
// blocks and slots (up to k = 24: five launches of six): 32 lanes key and select.  The
// threshold lies between k and 32 keys, searched for both halves together.  640x480,
// k = 24: 271 -> 166 us.
inline bool draw_halves(int k, int L) { return k <= 32 && L * ((k + 3) / 4) <= 32; }

template <int TURNS>
__global__ __launch_bounds__(64 * kDrawWaves) void k_sample_draw_halves(int W, int H, int k, int L, int tiles,
                                                                        uint32_t seedLo, uint32_t seedHi,
                                                                        uint32_t view, const ViewState* __restrict__ vs,
                                                                        const float2* __restrict__ leafXY,
                                                                        const int32_t* __restrict__ leafId,
                                                                        const int2* __restrict__ reach,
                                                                        int32_t* __restrict__ out,
                                                                        int* __restrict__ tieQueue, VStride vsd)
{
    vs = vw(vs, vsd.ws);
    leafXY = vw(leafXY, vsd.ws);
    leafId = vw(leafId, vsd.ws);
    reach = vw(reach, vsd.ws);
    tieQueue = vw(tieQueue, vsd.ws);
    view += blockIdx.y;
    out += (long)blockIdx.y * W * H * k;
    __shared__ __align__(16) uint32_t sKey[kDrawWaves][64];
    __shared__ int sPos[kDrawWaves][64];
    __shared__ int sOwner[kDrawWaves][64];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int s = lane & 31, h0 = lane & 32;            // lane of the pixel, its first lane
    constexpr int per = 32 / (kDrawWaves * TURNS);      // workgroups per tile, as above
    const int full = tiles & ~7, d = blockIdx.x;
    const int blk = d < full * per ? (d >> 3) / per * 8 + (d & 7) : d / per;
    const int pl0 = 2 * TURNS * ((d < full * per ? (d >> 3) % per : d % per) * kDrawWaves + wv) + (h0 >> 5);
    const int tilesY = (H + 7) >> 3;
    const uint32_t tile = xcd_chunk_remap<kSampTileRun>((uint32_t)blk, (uint32_t)tiles);
    const int ti = tile / tilesY, tj = tile - (tile / tilesY) * tilesY;
    const float is2h = vs->is2h;
    const unsigned long long some = TURNS > 1 ? drawn_pixels(reach, blk, L, lane) : ~0ull;
    if (TURNS > 1 && some == 0ull) { empty_columns(W, H, k, ti, tj, pl0 - (h0 >> 5), lane, out); return; }
#pragma unroll 1
    for (int turn = 0; turn < TURNS; turn++) {
        const int pl = pl0 + 2 * turn;
        const int i = ti * 8 + (pl >> 3), j = tj * 8 + (pl & 7);
        const bool in = i < W && j < H;
        if (!__ballot(in)) continue;                        // wave-uniform
        const float qx = (float)i, qy = (float)j;
        const uint32_t pixel = in ? (uint32_t)(j + H * i) : 0u;
        int2 fc = make_int2(0, 0);
        if (in && ((some >> pl) & 1ull) && s < L) fc = reach[((long)blk * L + s) * 64 + pl];
        if (__ballot(fc.y > 0) == 0ull) {                   // both pixels are empty
            if (in && s < k) out[(long)pixel * k + s] = -1;
            continue;
        }
        auto half_of = [&](unsigned long long m) { return h0 ? (uint32_t)(m >> 32) : (uint32_t)m; };
        int la = 0, kk0 = 0, first = 0, cnt = 0, blocks = 0;
        for (int l = 0; l < L; l++) {
            const int f = __shfl(fc.x, h0 + l, 64), c = __shfl(fc.y, h0 + l, 64);
            const int nb = (c + 3) >> 2;
            if (s >= blocks && s < blocks + nb) { la = l; kk0 = 4 * (s - blocks); first = f; cnt = c; }
            blocks += nb;
        }
        const u32x4 rnd = philox4x32_10(u32x4{ (uint32_t)(kk0 >> 2), (uint32_t)la, pixel, view }, seedLo, seedHi);
        const int pos = first + kk0;
        uint32_t key[4];
        {
            float2 xy[4];
#pragma unroll
            for (int q = 0; q < 4; q++) xy[q] = kk0 + q < cnt ? leafXY[pos + q] : make_float2(0.0f, 0.0f);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t kb = draw_key(qx, qy, xy[q], is2h,
                                             (q == 0) ? rnd.x : (q == 1) ? rnd.y : (q == 2) ? rnd.z : rnd.w);
                key[q] = kk0 + q < cnt ? kb : kNoKey;
            }
        }
        auto count = [&](uint32_t x) {
            int c = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) c += __popc(half_of(__ballot(key[e] <= x)));
            return c;
        };
        // threshold: every finite key if at most 32, else one that k .. 32 keys meet; the search
        // of k_sample_draw, each half with its own interval
        uint32_t thr = kInfKey - 1;
        int m = count(thr);
        bool tie = false, search = m > 32;
        uint32_t kth = kInfKey;                             // the k-th smallest key
        uint32_t lo = 0, hi = kInfKey - 1, step = 1u << 23, mid = 0x3f800000u;
        while (__ballot(search)) {
            const int c = count(mid);
            if (!search) continue;
            if (c >= k && c <= 32) { thr = mid; m = c; search = false; continue; }
            const bool up = c < k;
            if (up) lo = mid; else hi = mid;
            if (hi - lo <= 1) { tie = true; kth = hi; search = false; continue; }
            if (up && hi == kInfKey - 1) mid = hi - mid > step ? mid + step : lo + ((hi - lo) >> 1);
            else if (!up && lo == 0) mid = mid > step ? mid - step : hi >> 1;
            else mid = lo + ((hi - lo) >> 1);
            if (step < 1u << 30) step <<= 1;
        }
        uint32_t* sk = sKey[wv] + h0;
        int* so = sOwner[wv] + h0;
        sKey[wv][lane] = kNoKey;
        wave_lds_fence();
        int base = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const bool take = !tie && key[e] <= thr;
            const uint32_t mk = half_of(__ballot(take));
            const int at = base + __popc(mk & ((1u << s) - 1u));
            if (take) { sk[at] = key[e]; sPos[wv][h0 + at] = pos + e; }
            base += __popc(mk);
        }
        wave_lds_fence();
        const bool held = !tie && s < m;
        const uint32_t mine = sk[s];
        const int id = held ? leafId[sPos[wv][lane]] : -1;
        int rank = 0;
        for (int q0 = 0; q0 < 32; q0 += 16) {
            if (!__ballot(held && q0 < m)) break;
            uint32_t o[16];
#pragma unroll
            for (int q = 0; q < 16; q += 4) {
                const uint4 v = *(const uint4*)(sk + q0 + q);
                o[q] = v.x; o[q + 1] = v.y; o[q + 2] = v.z; o[q + 3] = v.w;
            }
#pragma unroll
            for (int q = 0; q < 16; q++) rank += o[q] < mine;
        }
        // equal keys share a rank: of the lanes writing one place, one reads its own entry back
        if (held) so[rank] = s;
        wave_lds_fence();
        const bool dup = held && so[rank] != s;
        uint32_t top = held && rank < k ? mine : 0u;
        if (half_of(__ballot(dup))) {
            tie = true;
            kth = kInfKey;
        }
        for (int o = 16; o > 0; o >>= 1) {
            const uint32_t x = (uint32_t)__shfl_xor((int)top, o, 64);
            top = x > top ? x : top;
        }
        if (tie && m >= k && top > 0u) kth = top;           // equal keys among those held
        wave_lds_fence();
        if (held && !tie) so[rank] = id;                    // ids in rank order
        wave_lds_fence();
        if (in && !tie && s < k) out[(long)pixel * k + s] = s < m ? so[s] : -1;
        if (in && tie && s == 0) {
            const int e = atomicAdd(tieQueue, 1);
            tieQueue[1 + 2 * e] = blk * 64 + pl;
            tieQueue[2 + 2 * e] = (int)kth;
        }
        wave_lds_fence();
    }
}

// The pixels k_sample_draw queued, drawn again through the reference's insertion,
// one wavefront per pixel: list position s lives in row s / 64 of lane s % 64
// (k <= 256: at most 4 rows).  Inserting word c with the strict < of the reference
// puts c at s0, the count of keys <= c's; behind it a displaced entry is carried
// on and passes over entries of its own key, so each run of equal keys behind s0
// keeps its entries in place except its first, which moves to the position after
// the run (and the first entry of the last run leaves a full list; a carried
// empty slot ends the insertion, and the empty slots form the last run).  So
// position s > s0 keeps its entry inside a run and otherwise takes the first
// entry of the run ending at s - 1; s0 takes c.  Candidates are keyed 64 at a
// time, one per lane, and inserted in the reference's order; one whose key is
// above the final list's largest (k_sample_draw queued the pixel's k-th smallest
// key) is skipped, as it only ever joins runs the list drops whole.
// A persistent grid drains the queue.
constexpr int kReplayRows = 4;
__global__ __launch_bounds__(64) void k_sample_replay(int W, int H, int k, int L, unsigned drawBlocks, uint32_t seedLo,
                                                      uint32_t seedHi, uint32_t view, const ViewState* __restrict__ vs,
                                                      const float2* __restrict__ leafXY,
                                                      const int32_t* __restrict__ leafId,
                                                      const int2* __restrict__ reach, const int* __restrict__ tieQueue,
                                                      int32_t* __restrict__ out, VStride vsd)
{
    tieQueue = vw(tieQueue, vsd.ws);
    const int lane = threadIdx.x;
    const int count = tieQueue[0];
    vs = vw(vs, vsd.ws);
    leafXY = vw(leafXY, vsd.ws);
    leafId = vw(leafId, vsd.ws);
    reach = vw(reach, vsd.ws);
    view += blockIdx.y;
    out += (long)blockIdx.y * W * H * k;
    const unsigned long long empty = ((unsigned long long)0x7f800000u << 32) | 0xffffffffull;
    const int R = (k + 63) >> 6;
    for (int e = blockIdx.x; e < count; e += gridDim.x) {
        const int sl = tieQueue[1 + 2 * e];             // sampler lane: draw block * 64 + lane
        const float kmax = __uint_as_float((uint32_t)tieQueue[2 + 2 * e]);
        const int blk = sl >> 6, pl = sl & 63;
        const int tilesY = (H + 7) >> 3;
        const uint32_t tile = xcd_chunk_remap<kSampTileRun>((uint32_t)blk, drawBlocks);
        const int ti = tile / tilesY, tj = tile - (tile / tilesY) * tilesY;
        const int i = ti * 8 + (pl >> 3), j = tj * 8 + (pl & 7);
        const float is2h = vs->is2h;
        const float qx = (float)i, qy = (float)j;
        const uint32_t pixel = (uint32_t)(j + H * i);
        const int2* rch = reach + (long)blk * L * 64 + pl;
        unsigned long long v[kReplayRows];
#pragma unroll
        for (int r = 0; r < kReplayRows; r++) v[r] = empty;
        for (int la = 0; la < L; la++) {
            const int2 fc = rch[(long)la * 64];
            const int first = fc.x, cnt = fc.y;
            for (int c0 = 0; c0 < cnt; c0 += 64) {
                // this lane's candidate of the chunk
                const int kk = c0 + lane;
                unsigned long long mine = empty;
                bool okc = false;
                if (kk < cnt) {
                    const u32x4 rnd = philox4x32_10(u32x4{ (uint32_t)(kk >> 2), (uint32_t)la, pixel, view }, seedLo,
                                                    seedHi);
                    const int q = kk & 3;
                    okc = draw_word(qx, qy, leafXY[first + kk], is2h,
                                    (q == 0) ? rnd.x : (q == 1) ? rnd.y : (q == 2) ? rnd.z : rnd.w, la, kk, mine) &&
                          !(key_of(mine) > kmax);
                }
                const unsigned long long okm = __ballot(okc);
                const int nc = cnt - c0 < 64 ? cnt - c0 : 64;
                for (int t = 0; t < nc; t++) {
                    if (!((okm >> t) & 1ull)) continue;       // key not finite (never inserted) or above kmax
                    const unsigned long long c = __shfl(mine, t, 64);
                    const float kc = key_of(c);
                    int s0 = 0;
#pragma unroll
                    for (int r = 0; r < kReplayRows; r++)
                        if (r < R) s0 += __popcll(__ballot(r * 64 + lane < k && !(kc < key_of(v[r]))));
                    if (s0 >= k) continue;                                // not below any key: not inserted
                    // run starts at or after s0 (s0 itself is one), prefix maximum over positions
                    // every shuffle runs on all 64 lanes; lane 0 then takes row r - 1's
                    // lane 63 (or nothing in row 0) as its predecessor
                    int start[kReplayRows];
                    unsigned long long before[kReplayRows];               // the entry ahead of each
                    int carry = -1;
#pragma unroll
                    for (int r = 0; r < kReplayRows; r++) {
                        if (r >= R) break;                                // wave-uniform
                        const int pos = r * 64 + lane;
                        const unsigned long long up = __shfl_up(v[r], 1, 64);
                        const unsigned long long wrap = __shfl(v[r > 0 ? r - 1 : 0], 63, 64);
                        const unsigned long long prev = lane > 0 ? up : r > 0 ? wrap : empty;
                        before[r] = prev;
                        const bool st = pos >= s0 && pos < k && (pos == s0 || key_of(v[r]) != key_of(prev));
                        const unsigned long long sm = __ballot(st), upto = sm & ((2ull << lane) - 1ull);
                        start[r] = upto ? r * 64 + 63 - __clzll((long long)upto) : carry;
                        if (sm) carry = r * 64 + 63 - __clzll((long long)sm);
                    }
                    // the first entry of the run ending at pos - 1: start of pos - 1, then its entry
                    unsigned long long nv[kReplayRows];
#pragma unroll
                    for (int r = 0; r < kReplayRows; r++) {
                        if (r >= R) break;
                        const int pos = r * 64 + lane;
                        const int spUp = __shfl_up(start[r], 1, 64);
                        const int spWrap = __shfl(start[r > 0 ? r - 1 : 0], 63, 64);
                        const int sp = lane > 0 ? spUp : r > 0 ? spWrap : -1;
                        unsigned long long from = empty;
#pragma unroll
                        for (int rr = 0; rr < kReplayRows; rr++) {
                            if (rr >= R) break;
                            const unsigned long long g = __shfl(v[rr], sp & 63, 64);
                            if (sp >= 0 && (sp >> 6) == rr) from = g;
                        }
                        // inside a run (the empty slots, which end a list that is not full,
                        // are one run: a carried empty slot ends the insertion there)
                        const bool inside = pos > s0 && key_of(v[r]) == key_of(before[r]);
                        nv[r] = pos >= k ? empty : pos < s0 ? v[r] : pos == s0 ? c : inside ? v[r] : from;
                    }
#pragma unroll
                    for (int r = 0; r < kReplayRows; r++)
                        if (r < R) v[r] = nv[r];
                }
            }
        }
        int32_t* o = out + ((long)j + (long)H * i) * k;
#pragma unroll
        for (int r = 0; r < kReplayRows; r++) {
            const int pos = r * 64 + lane;
            if (pos < k) {
                const uint32_t dn = (uint32_t)(v[r] & 0xffffffffull);
                o[pos] = dn == 0xffffffffu ? -1 : leafId[rch[(long)(dn >> 16) * 64].x + (int)(dn & 0xffffu)];
            }
        }
    }
}

__global__ void k_fill_f32(float* p, long n, float v)
{
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = v;
}

__global__ void k_fill_idx(int32_t* p, long n)
{
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = -1;
}

// ---------------------------------------------------------------------------
// Fixed-order (degree 6) Hermite densities D_b(q) = c_b sum_i exp(-|q - s_i|^2 /
// 2 h_b^2) on the shared tree: approximateFMMWeights (band 0, the tree's h;
// sampling.cpp:136-175, samplingCuda.cu:398-493, buildRadixTree.cuh:449-606,
// transformRadixTree.cuh:15-69, 152-222) and the normalisers of Poisson-rate
// sampling (bands 0 and 1).
// ---------------------------------------------------------------------------

// Internal nodes whose degree-6 truncation bound at band b meets the
// precision, and whose parent's does not, carry an expansion: a 49-float
// block at fixOff[node].  A workgroup reserves its slots of both bands with one atomic:
// those of one word follow one another, and 1M splats took 45 us with one per band and 256
// nodes (now 23).
constexpr int kSelectThreads = 1024;
__global__ __launch_bounds__(kSelectThreads) void k_fixed_select(ViewState* vs, int nbands, int p, const NodeGeo* __restrict__ geo,
                                                      const NodeLnk* __restrict__ lnk, int* fixOff0, int* fixOff1,
                                                      int* list0, int* list1, VStride vsd)
{
    vs = vw(vs, vsd.ws);
    geo = vw(geo, vsd.ws);
    lnk = vw(lnk, vsd.ws);
    fixOff0 = vw(fixOff0, vsd.ws);
    fixOff1 = vw(fixOff1, vsd.ws);
    list0 = vw(list0, vsd.ws);
    list1 = vw(list1, vsd.ws);
    __shared__ unsigned long long wcnt[kSelectThreads / 64];
    __shared__ unsigned long long first;
    const int n = vs->nc;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const float prec = vs->prec;
    bool acc[2] = { false, false };
    unsigned long long m[2] = { 0ull, 0ull };
    for (int b = 0; b < nbands; b++) {
        const float hb = vs->band[b].h;
        auto meets = [&](int nd) {
            NodeGeo g = geo[nd];
            float mn = 0.0f;
            mn = fmaxf(mn, fmaxf(g.cx - g.lox, g.hix - g.cx));
            mn = fmaxf(mn, fmaxf(g.cy - g.loy, g.hiy - g.cy));
            float rr = mn / hb;
            return hermite_error(rr, (float)lnk[nd].count, p) <= prec;
        };
        // the walk from the root evaluates the first node on its path that meets the
        // bound and skips its subtree, so only those nodes need an expansion
        if (t < n - 1) acc[b] = meets(t) && (t == 0 || !meets(lnk[t].parent));
        m[b] = __ballot(acc[b]);
    }
    if (lane == 0) wcnt[wid] = (unsigned long long)__popcll(m[1]) << 32 | (unsigned)__popcll(m[0]);
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long tot = 0ull;
        for (int q = 0; q < kSelectThreads / 64; q++) tot += wcnt[q];
        first = tot ? atomicAdd(&vs->nfix, tot) : 0ull;
    }
    __syncthreads();
    unsigned long long at = first;
    for (int q = 0; q < wid; q++) at += wcnt[q];
    if (t >= n - 1) return;
    for (int b = 0; b < nbands; b++) {
        const int slot = (int)(unsigned)(b ? at >> 32 : at) + __popcll(m[b] & ((1ull << lane) - 1ull));
        int* fixOff = b ? fixOff1 : fixOff0;
        int* list = b ? list1 : list0;
        fixOff[t] = acc[b] ? slot * (p + 1) * (p + 1) : -1;
        if (acc[b]) list[slot] = t;
    }
}

// Degree-P moments at band b, scaled by the band's leaf coefficient: thread
// (node, row a) sums row a over the node's leaf range in FP64 (leaf order).
// 256 / (P + 1) nodes x (P + 1) rows per 256-thread workgroup.
template <int P>
__global__ __launch_bounds__(256) void k_fixed_moments(const ViewState* __restrict__ vs,
                                                       const NodeGeo* __restrict__ geo, const NodeAux* __restrict__ aux,
                                                       const float2* __restrict__ leafXY,
                                                       const int* __restrict__ list0, const int* __restrict__ list1,
                                                       const int* __restrict__ fixOff0, const int* __restrict__ fixOff1,
                                                       float* __restrict__ coef0, float* __restrict__ coef1, VStride vsd)
{
    const int b = blockIdx.z;
    vs = vw(vs, vsd.ws);
    geo = vw(geo, vsd.ws);
    aux = vw(aux, vsd.ws);
    leafXY = vw(leafXY, vsd.ws);
    const int* list = vw(b ? list1 : list0, vsd.ws);
    const int* fixOff = vw(b ? fixOff1 : fixOff0, vsd.ws);
    float* coef = vw(b ? coef1 : coef0, vsd.ws);
    const int t = threadIdx.x;
    if (t >= (256 / (P + 1)) * (P + 1)) return;
    const long slot = (long)blockIdx.x * (256 / (P + 1)) + t / (P + 1);
    const int ax = t % (P + 1);
    if (slot >= (int)(unsigned)(b ? vs->nfix >> 32 : vs->nfix)) return;
    const int nd = list[slot];
    const float is2h = vs->band[b].is2h;
    const double c = (double)vs->band[b].c;
    NodeGeo g = geo[nd];
    NodeAux a = aux[nd];
    const int off = fixOff[nd];
    const double ifx = kInvFact[ax];
    double acc[P + 1];
#pragma unroll
    for (int bb = 0; bb <= P; bb++) acc[bb] = 0.0;
    for (int pos = a.first; pos <= a.last; pos += kMomLeaves) {
        double mx[kMomLeaves], ty[kMomLeaves];
        moment_leaves(leafXY, pos, a.last, g, is2h, ax, ifx, mx, ty);
#pragma unroll
        for (int u = 0; u < kMomLeaves; u++) {
            if (pos + u > a.last) break;
            double py = 1.0;
#pragma unroll
            for (int bb = 0; bb <= P; bb++) {
                acc[bb] += mx[u] * (py * ifact_c(bb));
                py = py * ty[u];
            }
        }
    }
#pragma unroll
    for (int bb = 0; bb <= P; bb++)
        coef[off + ax * (P + 1) + bb] = (float)(c * acc[bb]);
}

__device__ __forceinline__ bool box_meets_disc(const NodeGeo& g, float qx, float qy, float rad)
{
    float cx = fminf(fmaxf(qx, g.lox), g.hix);
    float cy = fminf(fmaxf(qy, g.loy), g.hiy);
    float dx = qx - cx, dy = qy - cy;
    float d2 = 0.0f;
    d2 = d2 + dx * dx;
    d2 = d2 + dy * dy;
    return d2 < rad * rad;
}

// c exp(-tx^2) exp(-ty^2), t = (q - x) / sqrt(2 h^2), in leaf-evaluation order
__device__ __forceinline__ float band_point(const Band& B, float qx, float qy, float x, float y)
{
    float tx = (qx - x) * B.is2h;
    float ty = (qy - y) * B.is2h;
    float ex = pexpf(-(tx * tx)), ey = pexpf(-(ty * ty));
    float v = 0.0f;
    v = v + (B.c * ex) * ey;
    return v;
}

// ---------------------------------------------------------------------------
// Launch shape of the per-pixel passes (k_fmm_eval, k_poisson): one wavefront
// per pixel tile of tw x 2^lth pixels (tw 2^lth = 64), wpb wavefronts per
// workgroup, and optionally an XCD-grouped block order: workgroups are handed
// to the 8 XCDs round-robin, so block b runs on XCD b mod 8; with xcd set,
// block b takes the tile range of position b / 8 within XCD b mod 8's
// contiguous share, so each XCD's L2 serves one band of the image (and of the
// leaves under it).  A pixel's result does not depend on the shape.
// The views of a batch are blockIdx.y; their workspaces lie vstride bytes apart.
// ---------------------------------------------------------------------------
struct TileCfg {
    int tw, lth, wpb, xcd;
};
constexpr int kMaxWavesPerBlock = 8;


// pixel (i, j) of this lane; false for a wavefront past the last tile (wave-uniform)
__device__ __forceinline__ bool tile_lane(const TileCfg& c, int W, int H, int lane, int& i, int& j)
{
    const int blk = c.xcd ? (int)xcd_remap(blockIdx.x, gridDim.x) : (int)blockIdx.x;
    const int tile = blk * c.wpb + (int)(threadIdx.x >> 6);
    const int th = 1 << c.lth;
    const int tilesY = (H + th - 1) >> c.lth;
    const int ntiles = ((W + c.tw - 1) / c.tw) * tilesY;
    if (tile >= ntiles) return false;
    const int ti = tile / tilesY, tj = tile - ti * tilesY;
    i = ti * c.tw + (lane >> c.lth);
    j = (tj << c.lth) + (lane & (th - 1));
    return true;
}


// children record of internal node p for the density walk (after the expansions
// of every band are selected)
__device__ __forceinline__ FmmRec fmm_record(int p, int L0, const NodeGeo* __restrict__ geo,
                                             const NodeLnk* __restrict__ lnk, const int* __restrict__ fixOff0,
                                             const int* __restrict__ fixOff1)
{
    const NodeLnk lk = lnk[p];
    const NodeGeo gl = geo[lk.left], gr = geo[lk.right];
    FmmRec r;
    r.lbox[0] = gl.lox; r.lbox[1] = gl.loy; r.lbox[2] = gl.hix; r.lbox[3] = gl.hiy;
    r.rbox[0] = gr.lox; r.rbox[1] = gr.loy; r.rbox[2] = gr.hix; r.rbox[3] = gr.hiy;
    r.lc[0] = gl.cx; r.lc[1] = gl.cy; r.rc[0] = gr.cx; r.rc[1] = gr.cy;
    r.left = lk.left; r.right = lk.right;
    r.lfix[0] = lk.left < L0 ? fixOff0[lk.left] : -1;
    r.rfix[0] = lk.right < L0 ? fixOff0[lk.right] : -1;
    r.lfix[1] = (fixOff1 && lk.left < L0) ? fixOff1[lk.left] : -1;
    r.rfix[1] = (fixOff1 && lk.right < L0) ? fixOff1[lk.right] : -1;
    r.pad[0] = r.pad[1] = 0;
    return r;
}

// children records of the internal nodes for the density walk
__global__ __launch_bounds__(256) void k_fmm_records(const ViewState* __restrict__ vs, const NodeGeo* __restrict__ geo,
                                                     const NodeLnk* __restrict__ lnk,
                                                     const int* __restrict__ fixOff0,
                                                     const int* __restrict__ fixOff1, FmmRec* __restrict__ rec, VStride vsd)
{
    vs = vw(vs, vsd.ws);
    geo = vw(geo, vsd.ws);
    lnk = vw(lnk, vsd.ws);
    fixOff0 = vw(fixOff0, vsd.ws);
    fixOff1 = vw(fixOff1, vsd.ws);
    rec = vw(rec, vsd.ws);
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    const int L0 = vs->nc - 1;
    if (p >= L0) return;
    rec[p] = fmm_record(p, L0, geo, lnk, fixOff0, fixOff1);
}

__device__ __forceinline__ bool box4_meets_disc(const float* bx, float qx, float qy, float rad)
{
    float cx = fminf(fmaxf(qx, bx[0]), bx[2]);
    float cy = fminf(fmaxf(qy, bx[1]), bx[3]);
    float dx = qx - cx, dy = qy - cy;
    float d2 = 0.0f;
    d2 = d2 + dx * dx;
    d2 = d2 + dy * dy;
    return d2 < rad * rad;
}

// Densities: one lane per pixel, one pixel tile per wavefront (TileCfg), bands on
// blockIdx.y (nbands per view).
// The reference walks each pixel with an explicit stack: pop a node; evaluate
// it if it is a leaf or carries an expansion, else push its left child and then
// its right child, each only if its box meets the query disc
// (transformRadixTree.cuh:15-69).  The terms of a pixel are therefore the leaves and
// expansions whose boxes meet its disc, rightmost first (a child's box lies in its
// parent's, and rounding keeps that order: a pixel that meets the child meets the parent).
// A workgroup finds the terms of its tiles level by level: a list of nodes in walk order,
// each node without a term replaced by its children that meet some pixel's disc, one
// thread per node, so a level's record loads are in flight together.  A level that runs
// over the list is cut there; once the terms of what was kept are added, the walk starts
// again from the root without the leaves up to the cut.  Then
// kFmmTerms terms at a time come to LDS, each wavefront evaluates the (term, pixel) pairs
// that meet, 64 at a time, and each pixel adds its values in order: bit for bit the
// reference's sums.  (A term meets 9 of a tile's 64 pixels in the narrow band, 28 to 49 in
// the wide one: a lane per pixel left most lanes idle.)
// Bound by the latency of the levels' and terms' loads (62 % miss L2 in the larger case),
// then by instruction issue.  Both bands of 512x512 under 1M splats 676 -> 493 us against
// one wavefront's walk with a stack; 16 views of 640x480 under 2M splats 3.53 -> 3.27 ms;
// 8 views of 64x145 under 600K splats, up to ten thousand terms to a tile, 2.46 -> 1.89 ms
// (putting the later half of a long level off in LDS, and a stack where that room ran out,
// 3.78 ms).  Lists of 704 and 1024 take 516 us and 3.30 ms, two wavefronts per workgroup
// 554 us and 4.63 ms, 32 terms at a time 672 us and 3.12 ms, one lane per pixel over its
// own terms 1023 us and 3.34 ms.
constexpr int kFmmTerms = 64, kFmmList = 1536, kFmmPairs = 384;
// Where a tile reaches few leaves each wavefront walks for itself (fmm_stack): the level form's
// barriers then cost more than the walk's waits, which other wavefronts hide.  The line is the
// number of leaves in reach if they lie evenly in the root's box, 6 to 16 with the band's
// wavefronts.  Level form against stack, us: 4096x2160 under 64 / 6400 / 256 000 / 1M / 3M
// splats 214 / 484 / 844 / 1149 / 1788 and 117 / 249 / 470 / 820 / 1850 (of the last 22 leaves
// per tile); 16 views of 640x480 under 6400, two bands, 700 and 430; 512x512 under 20 000, both
// ways 109; 256x256 under 6400, 49 and 63.  The lists are short where splats are few, so that
// five workgroups of four wavefronts fit a CU's LDS instead of four (4096x2160 under 64 000,
// stack, 409 us with long lists, 358).
constexpr float kFmmReachLow = 6.0f, kFmmReachHigh = 16.0f, kFmmReachPerWave = 1.0f / 512.0f;
constexpr int kFmmListShort = 512, kFmmListShortSplats = 14;     // splats per 64 pixels


// each active lane's word goes to LDS at the wavefront's base plus its lane's word
__device__ __forceinline__ void load_to_lds(const float UD_GLOBAL* from, float* base)
{
    __builtin_amdgcn_global_load_lds((const void UD_GLOBAL*)from, (void __attribute__((address_space(3)))*)(base), 4, 0, 0);
}
// those loads have arrived (a barrier alone does not wait for them)
__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

__device__ __forceinline__ unsigned long long uniform64(unsigned long long m)
{
    return (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(m >> 32)) << 32 |
           (unsigned)__builtin_amdgcn_readfirstlane((int)m);
}

// bits of m below this lane's
__device__ __forceinline__ int wave_rank(unsigned long long m)
{
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
}

// A fixed-order expansion at scaled offset t = (q - c) / sqrt(2 h^2):
// sum_a h_a(tx) sum_b C_ab h_b(ty), Hermite functions by their three-term
// recurrence from ex = e^{-tx^2}, ey = e^{-ty^2}, every product-sum one fused multiply-add
// (the oracle uses fmaf in the same order).
template <int P>
__device__ __forceinline__ float fixed_series(const float4* co, float tx, float ty, float ex, float ey)
{
    float hx[P + 1], hy[P + 1];
    hx[0] = ex; hy[0] = ey;
    hx[1] = (2.0f * tx) * ex; hy[1] = (2.0f * ty) * ey;
#pragma unroll
    for (int q = 2; q <= P; q++) {
        hx[q] = __builtin_fmaf(2.0f * tx, hx[q - 1], -((2.0f * (float)(q - 1)) * hx[q - 2]));
        hy[q] = __builtin_fmaf(2.0f * ty, hy[q - 1], -((2.0f * (float)(q - 1)) * hy[q - 2]));
    }
    float val = 0.0f, sa = 0.0f;
#pragma unroll
    for (int q4 = 0; q4 < ((P + 1) * (P + 1) + 3) / 4; q4++) {
        const float4 c4 = co[q4];
        const float c[4] = { c4.x, c4.y, c4.z, c4.w };
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int q = 4 * q4 + e, a = q / (P + 1), b = q - a * (P + 1);
            if (a > P) break;
            sa = __builtin_fmaf(c[e], hy[b], b == 0 ? 0.0f : sa);
            if (b == P) val = __builtin_fmaf(hx[a], sa, val);
        }
    }
    return val;
}

// words of an expansion's block in LDS: whole float4 words, an odd number of them, so
// that lanes reading different blocks meet different banks
constexpr int fmm_block(int p)
{
    const int q = ((p + 1) * (p + 1) + 3) / 4;
    return 4 * (q | 1);
}
// LDS bytes of a workgroup of wpb wavefronts: the terms' blocks, boxes, centres, block
// offsets and each wavefront's masks of them, two lists of nodes, the wavefronts' pairs
constexpr size_t fmm_lds(int p, int wpb, int list)
{
    return (size_t)kFmmTerms * (4 * fmm_block(p) + 28 + 8 * wpb) + 2 * (size_t)list * 4 + (size_t)kFmmPairs * 6 * wpb;
}

// |q - closest point of [lo, hi]| for the closest whole q in [a, b]
__device__ __forceinline__ float pixel_gap(float lo, float hi, float a, float b)
{
    const float p = fminf(fmaxf(ceilf(lo), a), b), q = fminf(fmaxf(floorf(hi), a), b);
    const float dp = p - fminf(fmaxf(p, lo), hi), dq = q - fminf(fmaxf(q, lo), hi);
    return fminf(fabsf(dp), fabsf(dq));
}

// some pixel of the tile (x, y the first and last i, z, w of j) meets the box within rad
__device__ __forceinline__ bool box4_meets_tile(const float4& bx, const float4& tile, float rad)
{
    const float dx = pixel_gap(bx.x, bx.z, tile.x, tile.y), dy = pixel_gap(bx.y, bx.w, tile.z, tile.w);
    float d2 = 0.0f;
    d2 = d2 + dx * dx;
    d2 = d2 + dy * dy;
    return d2 < rad * rad;
}

// The reference's walk by one wavefront for the union of its 64 pixels: stack entries carry
// the mask of pixels for which the node was pushed, so each pixel sees its own nodes in its
// own order (the shared stack is its stack with other pixels' entries interleaved, in the same
// last-in-first-out order).  A pushed entry also carries the child's centre and expansion
// offset from its parent's FmmRec, so leaves and expansions need no node load and a descent
// needs one wave-uniform record load.  An internal entry just below the top is handled in the
// same step as the top entry, its children pushed in the order that popping one after the
// other leaves.  Karras trees on 64-bit keys are at most 64 levels deep; a level keeps at most
// two entries pending, so the stack stays within 2 * 64 + 4.
constexpr int kFmmStack = 136;
struct FmmEntry {
    int node, off;                   // its expansion's offset, -1 for none / a leaf
    float2 c;
    unsigned long long mask;
};

template <int P>
__device__ __forceinline__ float fmm_stack(const Band& B, int L0, int b, const FmmRec* __restrict__ frec,
                                           const int* __restrict__ fixOff, const NodeGeo* __restrict__ geo,
                                           const float UD_GLOBAL* cf, float qx, float qy, bool valid, FmmEntry* stack,
                                           int lane)
{
    constexpr int NC = (P + 1) * (P + 1), Q = (NC + 3) / 4;
    float w = 0.0f;
    const unsigned long long all = __ballot(valid);
    if (lane == 0) stack[0] = FmmEntry{ 0, L0 > 0 ? fixOff[0] : -1, make_float2(geo[0].cx, geo[0].cy), all };
    int sp = 1;
    while (sp > 0) {
        sp--;
        wave_lds_fence();
        const FmmEntry top = stack[sp], low = stack[sp > 0 ? sp - 1 : 0];
        wave_lds_fence();
        const int nd = __builtin_amdgcn_readfirstlane(top.node), off = __builtin_amdgcn_readfirstlane(top.off);
        const int nd2 = __builtin_amdgcn_readfirstlane(low.node), off2 = __builtin_amdgcn_readfirstlane(low.off);
        const bool act = (top.mask >> lane) & 1ull;
        // the term of a leaf or an expansion on top of the stack
        auto add_top = [&]() {
            const float tx = (qx - top.c.x) * B.is2h, ty = (qy - top.c.y) * B.is2h;
            const float ex = pexpf(-(tx * tx)), ey = pexpf(-(ty * ty));
            if (nd >= L0) {
                if (act) w = w + (0.0f + (B.c * ex) * ey);
                return;
            }
            // wave-uniform block, fetched by broadcast vector loads issued together
            const float UD_GLOBAL* cc = cf + off;
            float4 co[Q];
#pragma unroll
            for (int q = 0; q < Q; q++)
                co[q] = make_float4(cc[4 * q], 4 * q + 1 < NC ? cc[4 * q + 1] : 0.0f, 4 * q + 2 < NC ? cc[4 * q + 2] : 0.0f,
                                    4 * q + 3 < NC ? cc[4 * q + 3] : 0.0f);
            if (act) w = w + fixed_series<P>(co, tx, ty, ex, ey);
        };
        const bool topInt = nd < L0 && off < 0;
        const bool lowInt = sp > 0 && nd2 < L0 && off2 < 0;
        if (!topInt && !lowInt) {
            add_top();
            continue;
        }
        if (lowInt) sp--;
        const bool two = topInt && lowInt;
        const int ndA = topInt ? nd : nd2;                   // the upper internal entry
        const FmmRec r = frec[ndA];
        const FmmRec r2 = frec[two ? nd2 : ndA];
        if (!topInt) add_top();
        const bool actA = topInt ? act : (bool)((low.mask >> lane) & 1ull);
        const bool act2 = two && ((low.mask >> lane) & 1ull);
        const unsigned long long ml = __ballot(actA && box4_meets_disc(r.lbox, qx, qy, B.radius));
        const unsigned long long mr = __ballot(actA && box4_meets_disc(r.rbox, qx, qy, B.radius));
        const unsigned long long ml2 = __ballot(act2 && box4_meets_disc(r2.lbox, qx, qy, B.radius));
        const unsigned long long mr2 = __ballot(act2 && box4_meets_disc(r2.rbox, qx, qy, B.radius));
        if (sp + 4 > kFmmStack) break;                       // unreachable for trees of depth <= 64
        auto push = [&](unsigned long long m, int node, int fix, float cx, float cy) {
            if (!m) return;
            if (lane == 0) stack[sp] = FmmEntry{ node, fix, make_float2(cx, cy), m };
            sp++;
        };
        push(ml2, r2.left, b ? r2.lfix[1] : r2.lfix[0], r2.lc[0], r2.lc[1]);
        push(mr2, r2.right, b ? r2.rfix[1] : r2.rfix[0], r2.rc[0], r2.rc[1]);
        push(ml, r.left, b ? r.lfix[1] : r.lfix[0], r.lc[0], r.lc[1]);
        push(mr, r.right, b ? r.rfix[1] : r.rfix[0], r.rc[0], r.rc[1]);
    }
    return w;
}

template <int P>
__global__ __launch_bounds__(64 * kMaxWavesPerBlock) void k_fmm_eval(TileCfg cfg, int W, int H, int listLen,
                                                                    const ViewState* __restrict__ vs, size_t vstride,
                                                                    int nbands, const NodeGeo* geo,
                                                                    const NodeAux* aux,
                                                                    const FmmRec* __restrict__ frec,
                                                                    const int* __restrict__ fixOff0,
                                                                    const int* __restrict__ fixOff1,
                                                                    const float* coef0, const float* coef1,
                                                                    float* __restrict__ out, size_t outStride,
                                                                    size_t bandStride)
{
    constexpr int NC = (P + 1) * (P + 1), BLK = fmm_block(P), T = kFmmTerms;
    extern __shared__ __align__(16) unsigned char fmmLds[];
    float* tB = (float*)fmmLds;                              // [T][BLK]
    float4* tBox = (float4*)(tB + T * BLK);
    float2* tC = (float2*)(tBox + T);
    unsigned long long* tMask = (unsigned long long*)(tC + T);   // [wpb][T]
    int* tOff = (int*)(tMask + T * cfg.wpb);                 // -1: a leaf
    int* list = tOff + T;                                    // two of listLen
    __shared__ float4 area[kMaxWavesPerBlock];               // the tiles, joined down a column
    __shared__ int areas;
    __shared__ int total[2][kMaxWavesPerBlock];
    __shared__ int cutAt;
    const int tid = threadIdx.x, lane = tid & 63, wpb = cfg.wpb;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    int i = W, j = H;
    const bool has = tile_lane(cfg, W, H, lane, i, j);       // wave-uniform
    const bool valid = has && i < W && j < H;
    const int b = (int)blockIdx.y % nbands;                  // band
    const size_t v = blockIdx.y / nbands;                    // view
    vs = (const ViewState*)((const char*)vs + v * vstride);
    geo = (const NodeGeo*)((const char*)geo + v * vstride);
    aux = (const NodeAux*)((const char*)aux + v * vstride);
    frec = (const FmmRec*)((const char*)frec + v * vstride);
    const int* fixOff = (const int*)((const char*)(b ? fixOff1 : fixOff0) + v * vstride);
    const float* coef = (const float*)((const char*)(b ? coef1 : coef0) + v * vstride);
    out = (float*)((char*)out + v * outStride + (size_t)b * bandStride);
    const int n = vs->nc;
    float w = 0.0f;
    const Band B = vs->band[b];
    const float UD_GLOBAL* cf = (const float UD_GLOBAL*)coef;
    const float qx = (float)i, qy = (float)j;
    const int L0 = n - 1;
    // the leaves that a tile reaches if they lie evenly in the root's box (uniform over the
    // band's workgroups)
    const float4 root = *(const float4*)&geo[0].lox;
    const float reach = (float)n * ((float)cfg.tw + 2.0f * B.radius) * ((float)(1 << cfg.lth) + 2.0f * B.radius) /
                        ((fminf(root.z, (float)W) - fmaxf(root.x, 0.0f) + 2.0f * B.radius) *
                         (fminf(root.w, (float)H) - fmaxf(root.y, 0.0f) + 2.0f * B.radius));
    const float waves = (float)gridDim.x * (float)gridDim.y * (float)wpb;
    if (n > 0 && reach < fminf(fmaxf(waves * kFmmReachPerWave, kFmmReachLow), kFmmReachHigh)) {
        if (has)
            w = fmm_stack<P>(B, L0, b, frec, fixOff, geo, cf, qx, qy, valid, (FmmEntry*)fmmLds + kFmmStack * wid, lane);
    } else if (n > 0) {
        const int i0 = __builtin_amdgcn_readfirstlane(i), j0 = __builtin_amdgcn_readfirstlane(j);
        const int i1 = min(i0 + cfg.tw, W) - 1, j1 = min(j0 + (1 << cfg.lth), H) - 1;
        const float4 own = make_float4((float)i0, (float)i1, (float)j0, (float)j1);   // if has
        if (lane == 0) total[0][wid] = has ? 1 : 0;
        if (lane == 0) area[wid] = own;
        __syncthreads();
        if (tid == 0) {
            int m = 0;                                       // the wavefronts with a tile come first
            for (int q = 0; q < wpb && total[0][q]; q++) {
                const float4 t = area[q];
                if (m > 0 && area[m - 1].x == t.x) area[m - 1].w = t.w;
                else area[m++] = t;
            }
            areas = m;
        }
        // entries: a node to be replaced by its children, or ~(2 parent + side) of a term
        const int rootOff = L0 > 0 ? fixOff[0] : -1;
        const bool rootTerm = L0 == 0 || rootOff >= 0;
        int* A = list;
        int* O = list + listLen;
        float* val = (float*)(list + 2 * listLen) + kFmmPairs * wid;        // this wavefront's pairs
        uint16_t* pair = (uint16_t*)((float*)(list + 2 * listLen) + kFmmPairs * wpb) + kFmmPairs * wid;
        if (tid == 0) A[0] = 0;
        int F = 1, end = n, cut = 0;                         // entries; leaves from end on are added, from cut on kept
        bool more = !rootTerm;
        int turn = 1;
        __syncthreads();
        while (true) {
            while (more) {
                more = false;
                int kept = 0;
                for (int c0 = 0; c0 < F; c0 += 64 * wpb) {
                    const int at = c0 + tid;
                    const int e = at < F ? A[at] : -1;
                    bool f1 = at < F, f2 = false;
                    int o1 = e, o2 = 0;
                    if (at < F && e >= 0) {
                        const FmmRec UD_GLOBAL* r = (const FmmRec UD_GLOBAL*)(frec + e);
                        const float4 lb = make_float4(r->lbox[0], r->lbox[1], r->lbox[2], r->lbox[3]);
                        const float4 rb = make_float4(r->rbox[0], r->rbox[1], r->rbox[2], r->rbox[3]);
                        const int cl = r->left, cr = r->right, fl = r->lfix[b], fr = r->rfix[b];
                        f1 = false;
                        for (int t = 0; t < areas; t++) {
                            f1 |= box4_meets_tile(rb, area[t], B.radius);
                            f2 |= box4_meets_tile(lb, area[t], B.radius);
                        }
                        f1 &= (cl >= L0 ? cl - L0 : cl) + 1 < end;           // the right child's first leaf
                        o1 = cr >= L0 || fr >= 0 ? ~(2 * e + 1) : cr;
                        o2 = cl >= L0 || fl >= 0 ? ~(2 * e) : cl;
                    }
                    const unsigned long long m1 = __ballot(f1), m2 = __ballot(f2);
                    const int inner = __ballot((f1 && o1 >= 0) || (f2 && o2 >= 0)) ? 1 << 16 : 0;
                    if (lane == 0) total[turn][wid] = (__popcll(m1) + __popcll(m2)) | inner;
                    __syncthreads();
                    int base = kept;
                    for (int q = 0; q < wpb; q++) {
                        const int x = total[turn][q];
                        more |= (x >> 16) != 0;
                        if (q < wid) base += x & 0xffff;
                        kept += x & 0xffff;
                    }
                    turn ^= 1;
                    const int p = base + wave_rank(m1) + wave_rank(m2), p2 = p + (f1 ? 1 : 0);
                    if (f1 && p < listLen) O[p] = o1;
                    if (f2 && p2 < listLen) O[p2] = o2;
                    if (kept > listLen) {
                        // one past the last leaf of the first entry that is left out
                        if ((f1 && p == listLen) || (f2 && p2 == listLen)) {
                            const bool second = !(f1 && p == listLen);
                            const int parent = e >= 0 ? e : ~e >> 1;
                            if (second || (e < 0 && !(~e & 1))) {            // a left child
                                const int cl = frec[parent].left;
                                cutAt = (cl >= L0 ? cl - L0 : cl) + 1;
                            } else cutAt = aux[parent].last + 1;
                        }
                        break;
                    }
                }
                __syncthreads();
                if (kept > listLen) cut = cutAt;
                F = min(kept, listLen);
                int* t = A; A = O; O = t;
            }
            for (int t0 = 0; t0 < F; t0 += T) {
                const int nt = min(T, F - t0);
                for (int t = tid; t < nt; t += 64 * wpb) {
                    if (rootTerm) {
                        tC[0] = make_float2(geo[0].cx, geo[0].cy);
                        tOff[0] = rootOff;
                        tBox[0] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    } else {
                        const int e = ~A[t0 + t];
                        const FmmRec UD_GLOBAL* r = (const FmmRec UD_GLOBAL*)(frec + (e >> 1));
                        const float UD_GLOBAL* bx = e & 1 ? r->rbox : r->lbox;
                        const float UD_GLOBAL* cc = e & 1 ? r->rc : r->lc;
                        tBox[t] = make_float4(bx[0], bx[1], bx[2], bx[3]);
                        tC[t] = make_float2(cc[0], cc[1]);
                        tOff[t] = (e & 1 ? r->right : r->left) >= L0 ? -1 : (e & 1 ? r->rfix[b] : r->lfix[b]);
                    }
                }
                __syncthreads();
                // the blocks, a wavefront per term, straight to LDS
                for (int t = wid; t < nt; t += wpb) {
                    const int off = __builtin_amdgcn_readfirstlane(tOff[t]);
                    if (off < 0) continue;
#pragma unroll
                    for (int q = 0; q < NC; q += 64)
                        if (lane + q < NC) load_to_lds(cf + off + q + lane, tB + t * BLK + q);
                }
                wait_loads();
                // the terms that some pixel of this tile meets
                unsigned long long todo =
                    __ballot(has && lane < nt && (rootTerm || box4_meets_tile(tBox[lane], own, B.radius)));
                __syncthreads();
                while (todo) {
                    // (term, pixel) pairs of the next terms, as many as there is room for
                    int pairs = 0, nm = 0;
                    while (todo && pairs <= kFmmPairs - 256) {
                        // four terms at a time, their box reads in flight together
                        unsigned long long m[4];
                        int t[4];
                        bool mine[4];
#pragma unroll
                        for (int u = 0; u < 4; u++) {
                            t[u] = todo ? __builtin_amdgcn_readfirstlane(__ffsll(todo) - 1) : -1;
                            todo &= todo - 1ull;
                        }
#pragma unroll
                        for (int u = 0; u < 4; u++) {
                            const float4 bx = tBox[t[u] < 0 ? 0 : t[u]];
                            const float q[4] = { bx.x, bx.y, bx.z, bx.w };
                            mine[u] = t[u] >= 0 && valid && (rootTerm || box4_meets_disc(q, qx, qy, B.radius));
                            m[u] = __ballot(mine[u]);
                        }
#pragma unroll
                        for (int u = 0; u < 4; u++) {
                            if (!m[u]) continue;
                            if (mine[u]) pair[pairs + wave_rank(m[u])] = (uint16_t)(t[u] << 6 | lane);
                            if (lane == 0) tMask[wid * T + nm] = m[u];
                            pairs += __popcll(m[u]);
                            nm++;
                        }
                    }
                    wave_lds_fence();
                    for (int k0 = 0; k0 < pairs; k0 += 64) {
                        const int k = k0 + lane;
                        if (k < pairs) {
                            const int e = pair[k], t = e >> 6, px = e & 63;
                            const float2 c = tC[t];
                            const float x = (float)(i0 + (px >> cfg.lth)), y = (float)(j0 + (px & ((1 << cfg.lth) - 1)));
                            const float tx = (x - c.x) * B.is2h, ty = (y - c.y) * B.is2h;
                            const float ex = pexpf(-(tx * tx)), ey = pexpf(-(ty * ty));
                            if (tOff[t] < 0) val[k] = 0.0f + (B.c * ex) * ey;       // band_point
                            else val[k] = fixed_series<P>((const float4*)(tB + t * BLK), tx, ty, ex, ey);
                        }
                    }
                    wave_lds_fence();
                    // each pixel adds its terms in order
                    for (int k0 = 0, at = 0; k0 < nm; k0 += 4) {
                        float x[4];
                        unsigned long long m[4];
#pragma unroll
                        for (int u = 0; u < 4; u++) m[u] = k0 + u < nm ? tMask[wid * T + k0 + u] : 0ull;
#pragma unroll
                        for (int u = 0; u < 4; u++) {
                            m[u] = uniform64(m[u]);
                            x[u] = (m[u] >> lane) & 1ull ? val[at + wave_rank(m[u])] : 0.0f;
                            at += __popcll(m[u]);
                        }
#pragma unroll
                        for (int u = 0; u < 4; u++)
                            if ((m[u] >> lane) & 1ull) w = w + x[u];
                    }
                    wave_lds_fence();
                }
                __syncthreads();
            }
            if (cut == 0) break;
            end = cut;
            cut = 0;
            if (tid == 0) A[0] = 0;
            F = 1;
            more = true;
            __syncthreads();
        }
    }
    if (valid) out[(long)j + (long)H * i] = w;
}

// ---------------------------------------------------------------------------
// Poisson-rate sampling with inclusion probabilities (no reference kernel; its
// dead plain-Poisson kernel, poissonRadixTree.cuh:70-200, draws Bernoulli(k p)
// only inside the reached subtree, which leaves the inclusion probabilities
// unknown).  Every culled splat i is included at pixel q independently with the
// defensive-mixture probability (Hesterberg 1995)
//   pi_i = min(1, lambda p_i(q)),  p_i = (g0_i(q) / N0(q) + g1_i(q) / N1(q)) / 2,
// g_b = c_b exp(-|q - s_i|^2 / 2 h_b^2) for the tree bandwidth h_0 = h and the
// wide bandwidth h_1 = max(h, 99.9th percentile of the visible splats' own
// bandwidths sqrt(lambda_max(V_i))), and N_b = max(D_b, c_b) with D_b the
// fixed-order density of band b: the expected count stays near lambda, and EWA
// weight / pi stays bounded for splats not wider than h_1.  Pixels with
// D_0 < precision draw nothing.  The support is the set of pairs with
// p >= 1e-4 (independent of the rate), so 1 / pi <= 1e4 / lambda: far tails of
// splats wider than h_1, whose weights there would be multiplied by huge
// 1 / pi, are outside it.
// ---------------------------------------------------------------------------
constexpr float kProposalHCap = 16.0f;
constexpr float kProposalPMin = 1e-4f;   // support: pairs whose rate-free proposal p >= 1e-4

// histogram of the visible splats' proposal bandwidths (1/16 px bins, the
// last bin holds everything >= 16; degenerate splats are skipped)
__global__ __launch_bounds__(256) void k_wide_hist(ViewState* vs, const int32_t* __restrict__ ids,
                                                   const float* __restrict__ hraw, VStride vsd)
{
    vs = vw(vs, vsd.ws);
    ids = vw(ids, vsd.ws);
    hraw = vw(hraw, vsd.ws);
    __shared__ int sh[256];
    sh[threadIdx.x] = 0;
    __syncthreads();
    const int nc = vs->nc;
    for (int pos = blockIdx.x * blockDim.x + threadIdx.x; pos < nc; pos += gridDim.x * blockDim.x) {
        float hi = hraw[ids[pos]];
        if (hi >= 0.0f) atomicAdd(&sh[hi < kProposalHCap ? (int)(hi * 16.0f) : 255], 1);
    }
    __syncthreads();
    if (sh[threadIdx.x]) atomicAdd(&vs->hhist[threadIdx.x], sh[threadIdx.x]);
}

// wide band: h_1 = max(h, 99.9th percentile of the histogram, rounded up to 1/16 px)
// (one workgroup of 256 threads, a thread per bin: the chosen bin is the first
// whose inclusive count reaches the target, 0 when the histogram is empty)
__global__ __launch_bounds__(256) void k_wide_band(ViewState* vs, VStride vsd)
{
    vs = vw(vs, vsd.ws);
    __shared__ int wsum[4];
    __shared__ int qbs;
    const int t = threadIdx.x, wid = t >> 6;
    const int c = vs->hhist[t];
    const int inc = wave_incl_scan(c);
    if ((t & 63) == 63) wsum[wid] = inc;
    if (t == 0) qbs = 0;
    __syncthreads();
    int base = 0;
    for (int q = 0; q < wid; q++) base += wsum[q];
    const long cum = (long)base + inc;
    const long total = (long)wsum[0] + wsum[1] + wsum[2] + wsum[3];
    const long target = total - total / 1000;
    if (cum >= target && cum - c < target) qbs = t;
    __syncthreads();
    if (t != 0) return;
    const float hw = fmaxf(vs->h, (float)(qbs + 1) * 0.0625f);
    vs->band[1] = make_band(hw, (double)vs->prec);
}

// rate-free mixture proposal t0 g0 + t1 g1 at (x, y)
// The proposal mixture at squared distance d2: k0 e^{-a0 d2} + k1 e^{-a1 d2},
// with k_b = t_b c_b and a_b = is2h_b^2 = 1 / 2h_b^2 (one exponential per band).
__device__ __forceinline__ float mix_d2(float k0, float a0, float k1, float a1, float d2)
{
    const float e0 = pexpf(-(d2 * a0));
    const float e1 = pexpf(-(d2 * a1));
    float m = k0 * e0;
    m = m + k1 * e1;
    return m;
}

// wide-band half plus footprint half: k1 e^{-a1 d2} + kf f (same order as mix_d2)
__device__ __forceinline__ float foot_mix(float k0, float a0, float kf, float d2, float f)
{
    const float e0 = pexpf(-(d2 * a0));
    float m = k0 * e0;
    m = m + kf * f;
    return m;
}

__device__ __forceinline__ float dist2(float qx, float qy, float x, float y)
{
    const float dx = qx - x, dy = qy - y;
    float d2 = dx * dx;
    d2 = d2 + dy * dy;
    return d2;
}

// Walk records of the Poisson pass, and (for internal nodes) the density walk's
// children records, in one launch after the expansions are selected.  The
// escape pointer of a node is the right sibling of its first ancestor-or-self
// that is a left child (-1 on the rightmost path).  That sibling's leaf range
// starts at m = last + 1, and in a Karras tree a right child's index is the
// first leaf of its range, so it is internal node m when node m's range starts
// at m and leaf m otherwise (no climb over parent links).
__global__ __launch_bounds__(256) void k_walk_records(const ViewState* __restrict__ vs,
                                                      const NodeGeo* __restrict__ geo,
                                                      const NodeLnk* __restrict__ lnk,
                                                      const NodeAux* __restrict__ aux,
                                                      const int* __restrict__ fixOff0,
                                                      const int* __restrict__ fixOff1, PNode* __restrict__ pnode,
                                                      FmmRec* __restrict__ frec, VStride vsd)
{
    vs = vw(vs, vsd.ws);
    geo = vw(geo, vsd.ws);
    lnk = vw(lnk, vsd.ws);
    aux = vw(aux, vsd.ws);
    fixOff0 = vw(fixOff0, vsd.ws);
    fixOff1 = vw(fixOff1, vsd.ws);
    pnode = vw(pnode, vsd.ws);
    frec = vw(frec, vsd.ws);
    const int nd = blockIdx.x * blockDim.x + threadIdx.x;
    const int nc = vs->nc;
    if (nc <= 0 || nd >= 2 * nc - 1) return;
    const int L0 = nc - 1;
    const NodeGeo g = geo[nd];
    const NodeAux a = aux[nd];
    const int m = a.last + 1;
    int esc = -1;
    if (m < nc) esc = (m < L0 && aux[m].first == m) ? m : L0 + m;
    PNode q;
    q.lox = g.lox; q.loy = g.loy; q.hix = g.hix; q.hiy = g.hiy;
    q.left = nd < L0 ? lnk[nd].left : -1;
    q.esc = esc;
    q.first = a.first; q.last = a.last;
    pnode[nd] = q;
    if (nd < L0) frec[nd] = fmm_record(nd, L0, geo, lnk, fixOff0, fixOff1);
}

// Footprint records of the sorted leaves, and the sum of the visible splats'
// footprint masses (integrals of min(w, 1)) for the normaliser of the footprint
// half (footSum starts at zero).
__global__ __launch_bounds__(256) void k_foot_leaves(float Wf, float Hf, float ff, float smoothing,
                                                     const float* __restrict__ pts, const float* __restrict__ nrm,
                                                     const float* __restrict__ sd, const ViewState* __restrict__ vs,
                                                     const int32_t* __restrict__ ids,
                                                     const float2* __restrict__ leafXY, FootLeaf* __restrict__ footLeaf,
                                                     double* footSum, VStride vsd)
{
    pts = vw(pts, vsd.pts);
    nrm = vw(nrm, vsd.pts);
    sd = vw(sd, vsd.sd);
    vs = vw(vs, vsd.ws);
    ids = vw(ids, vsd.ws);
    leafXY = vw(leafXY, vsd.ws);
    footLeaf = vw(footLeaf, vsd.ws);
    footSum = vw(footSum, vsd.ws);
    __shared__ double sm[4];
    const int n = vs->nc;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    double mass = 0.0;
    if (t < n) {
        const int id = ids[t];
        FootLeaf L;
        const float2 xy = leafXY[t];
        L.x = xy.x; L.y = xy.y;
        float m, ms;
        foot_f32(Wf, Hf, ff, pts + 3L * id, nrm + 3L * id, sd + 2L * id, smoothing, L.t00, L.t01, L.t11, L.amp, m,
                 ms);
        L.pad[0] = L.pad[1] = 0.0f;
        footLeaf[t] = L;
        mass = (double)ms;
    }
    for (int o = 32; o > 0; o >>= 1) mass += __shfl_xor(mass, o, 64);
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = mass;
    __syncthreads();
    if (threadIdx.x == 0) {
        const double b = (sm[0] + sm[1]) + (sm[2] + sm[3]);
        if (b != 0.0) atomicAdd(footSum, b);
    }
}

__global__ void k_zero_f64(double* p, size_t stride, int views)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v < views) *(double*)((char*)p + stride * v) = 0.0;
}

// One lane per pixel (one pixel tile per wavefront, TileCfg).  The walk
// visits nodes left to right; a node's bound U (the mixture at the point of its
// box closest to q) is >= pi_i of each of its leaves.  U = 0: skip the
// subtree.  A leaf, or a node with count U <= 1, is thinned: candidate leaves at
// rate U by geometric skips over its contiguous leaf range (skip = floor(log u /
// log(1 - U))), each kept with probability pi_i / U, i.e. included with
// probability pi_i, independently.  Uniforms are Philox4x32-10 words at counter
// (step, 0x80000000, pixel, view), one block per geometric-skip step of the
// pixel (word x the skip, word y the acceptance test).  A skipped or thinned
// subtree is left through its escape pointer.
// Walking and thinning alternate: a lane queues its ranges in registers and thins them
// in the order found, and each turn of the wavefront takes the step that more lanes can
// take.  A pixel at 512x512 under 1M splats visits 109 nodes and takes 59 thinning steps
// (tile maxima 130 and 75), but the pixels find their ranges at different nodes: thinned
// on the spot, every visit waited for some lane's steps.  Bound by instruction issue (a
// thinning step is a Philox block, a logarithm and a mixture).  16 views of 640x480 under
// 2M splats: 5.85 -> 3.47 ms (512x512, 1M: 578 -> 322 us); queues of 2, 4, 6 ranges take
// 3.63, 3.49, 3.74 ms, walking only at 4/3 of the thinning lanes (or already at 3/4)
// is 1 % slower.  One walk over the union of the tile's nodes with scalar loads visits
// 392 nodes: 7.24 ms.
// The first kPoissonStage samples of each lane are staged in LDS (slot-major,
// [slot][lane], so the stores hit 64 distinct banks) and written out at
// the end together with the empty slots, one tile row (2^lth contiguous pixels
// x kcap slots) per coalesced pass of the wavefront; only samples past the
// staged ones are stored directly.  A lane's scattered 4-byte stores would
// otherwise leave partly written lines in L2 for the length of the walk.
constexpr int kPoissonQueue = 3;

constexpr int kPoissonStage = 16;
constexpr size_t kPoissonStageBytes = (size_t)kPoissonStage * 64 * 8;    // per wavefront

__global__ __launch_bounds__(64 * kMaxWavesPerBlock) void k_poisson(TileCfg cfg, int W, int H, int kcap, float rate,
                                                                   const float* __restrict__ tscale, int tsH,
                                                                   uint32_t seedLo, uint32_t seedHi,
                                                                   const uint64_t* __restrict__ seedDev,
                                                                   uint32_t view0, const ViewState* __restrict__ vs,
                                                                   size_t vstride, const PNode* __restrict__ pnode,
                                                                   const float2* __restrict__ leafXY,
                                                                   const int32_t* __restrict__ leafId,
                                                                   const float* __restrict__ dens0,
                                                                   const float* __restrict__ dens1, size_t densStride,
                                                                   int32_t* __restrict__ outIds,
                                                                   float* __restrict__ outIpi, int* err, int fmode,
                                                                   float fscale, const FootLeaf* __restrict__ footLeaf,
                                                                   const double* __restrict__ footSum)
{
    extern __shared__ int32_t stage[];
    const int lane = threadIdx.x & 63;
    int i, j;
    if (!tile_lane(cfg, W, H, lane, i, j)) return;           // wave-uniform
    int32_t* sid = stage + (threadIdx.x >> 6) * (2 * kPoissonStage * 64);
    float* sip = (float*)(sid + kPoissonStage * 64);
    const bool valid = i < W && j < H;
    const uint32_t view = view0 + blockIdx.y;
    if (seedDev) {
        const uint64_t sd = *seedDev;
        seedLo = (uint32_t)sd;
        seedHi = (uint32_t)(sd >> 32);
    }
    vs = vw(vs, vstride);
    pnode = vw(pnode, vstride);
    leafXY = vw(leafXY, vstride);
    leafId = vw(leafId, vstride);
    dens0 = vw(dens0, densStride);
    dens1 = vw(dens1, densStride);
    if (fmode) {
        footLeaf = vw(footLeaf, vstride);
        footSum = vw(footSum, vstride);
    }
    const long perView = (long)W * H;
    outIds += (long)blockIdx.y * perView * kcap;
    outIpi += (long)blockIdx.y * perView * kcap;
    if (tscale) tscale += (long)blockIdx.y * ((W + 15) / 16) * tsH;
    const long pix = valid ? (long)j + (long)H * i : 0;
    int32_t* oid = outIds + pix * kcap;
    float* oip = outIpi + pix * kcap;
    int ns = 0;
    bool over = false;
    const int n = vs->nc;
    const float D0 = (n > 0 && valid) ? dens0[pix] : 0.0f;
    const bool draws = valid && n > 0 && D0 >= vs->prec;
    if (__ballot(draws)) {
        const Band B0 = vs->band[0], B1 = vs->band[1];
        float lam = rate;
        if (tscale && draws) lam = lam * tscale[(long)(i >> 4) * tsH + (j >> 4)];
        // a negative or non-finite multiplier would make every candidate's pi 1
        // (fminf drops a NaN): draw nothing there and say so
        if (draws && !(lam >= 0.0f && lam <= 3.0e38f)) { atomicOr(err, 16); lam = 0.0f; }
        const float t0 = 0.5f / fmaxf(D0, B0.c);
        const float t1 = 0.5f / fmaxf(draws ? dens1[pix] : 0.0f, B1.c);
        const float k0 = t0 * B0.c, k1 = t1 * B1.c;
        const float a0 = B0.is2h * B0.is2h, a1 = B1.is2h * B1.is2h;
        // footprint mode: the wide band's half as above, and in place of band 0
        // f_i(q) / (kw max(D1, c1)), kw = the visible splats' mean footprint mass
        // over h_1^1.5 (so that both halves expect about lam / 2 samples), or the
        // caller's scale
        float kf = 0.0f;
        if (fmode) {
            float kw = fscale;
            if (!(kw > 0.0f)) {
                const double hh = (double)B1.h;
                kw = (float)((*footSum / (double)n) / (hh * sqrt(hh)));
            }
            if (kw > 0.0f && kw < 3.0e38f) kf = t1 / kw;
        }
        const float qx = (float)i, qy = (float)j;
        const uint32_t pixel = (uint32_t)pix;
        uint32_t step = 0;                            // geometric-skip steps of this pixel
        // the ranges still to be thinned, the current one (from its last candidate on) in slot 0
        int qpos[kPoissonQueue], qlast[kPoissonQueue];
        float qU[kPoissonQueue], il1 = 0.0f;
#pragma unroll
        for (int q = 0; q < kPoissonQueue; q++) { qpos[q] = qlast[q] = 0; qU[q] = 0.5f; }
        int cnt = 0;
        bool fresh = true;                            // il1 is not slot 0's yet
        int nd = draws ? 0 : -1;
        int visits = 0;                               // a preorder walk visits each node at most once
        PNode pn = pnode[0];
        // Both steps run in all lanes and select what a lane keeps: branches around the state
        // (queue, node record) copied it at every join (3.78 ms).
        while (true) {
            const bool walks = nd >= 0 && cnt < kPoissonQueue, thins = cnt > 0;
            const unsigned long long mw = __ballot(walks), mt = __ballot(thins);
            if (!(mw | mt)) break;
            if (__popcll(mw) >= __popcll(mt)) {
                float cx = fminf(fmaxf(qx, pn.lox), pn.hix);
                float cy = fminf(fmaxf(qy, pn.loy), pn.hiy);
                const float d2b = dist2(qx, qy, cx, cy);
                // proposal bound over the node
                float pB = fmode ? foot_mix(k1, a1, kf, d2b, foot_bound(a1, d2b)) : mix_d2(k0, a0, k1, a1, d2b);
                const float U = fminf(1.0f, lam * pB);
                // outside the support: past the subtree; a leaf or few enough: thinned
                const bool in = pB >= kProposalPMin && U > 0.0f;
                const bool push = walks && in && (pn.left < 0 || !((float)(pn.last - pn.first + 1) * U > 1.0f));
                const int to = in && !push ? pn.left : pn.esc;
#pragma unroll
                for (int q = 0; q < kPoissonQueue; q++) {
                    const bool here = push && cnt == q;
                    qpos[q] = here ? pn.first - 1 : qpos[q];
                    qlast[q] = here ? pn.last : qlast[q];
                    qU[q] = here ? U : qU[q];
                }
                cnt += push;
                nd = walks ? to : nd;
                visits += walks;
                if (__ballot(visits > 2 * n)) {              // never
                    if (visits > 2 * n) { atomicOr(err, 8); nd = -1; }
                }
                pn = pnode[nd >= 0 ? nd : 0];                // on its way while others thin
            } else {
                // one Philox block per step: word x draws the skip, word y the acceptance test
                if (thins && fresh) { il1 = 1.0f / plog1mf(qU[0]); fresh = false; }
                const u32x4 blk = philox4x32_10(u32x4{ step, 0x80000000u, pixel, view }, seedLo, seedHi);
                step += thins;
                const float r = plogf_normal(u01(blk.x)) * il1;       // failures before the next candidate
                const bool cand = thins && r < (float)(qlast[0] - qpos[0]), pop = thins && !cand;
                const int pos = cand ? qpos[0] + (int)r + 1 : 0;
                if (cand) {
                    float pl;
                    if (fmode) {
                        const FootLeaf L = footLeaf[pos];
                        const float d2 = dist2(qx, qy, L.x, L.y);
                        pl = foot_mix(k1, a1, kf, d2, foot_leaf(L, a1, qx, qy, d2));
                    } else {
                        const float2 lp = leafXY[pos];
                        pl = mix_d2(k0, a0, k1, a1, dist2(qx, qy, lp.x, lp.y));
                    }
                    const float pi = fminf(1.0f, lam * pl);
                    const float a = u01(blk.y);
                    // in the support, and P = pi / U, exactly 1 when pi = U
                    if (pl >= kProposalPMin && a * qU[0] <= pi) {
                        if (ns < kcap) {
                            const int32_t id = leafId[pos];
                            const float ip = 1.0f / pi;
                            if (ns < kPoissonStage) { sid[ns * 64 + lane] = id; sip[ns * 64 + lane] = ip; }
                            else { oid[ns] = id; oip[ns] = ip; }
                            ns++;
                        } else over = true;
                    }
                }
                qpos[0] = cand ? pos : qpos[0];
#pragma unroll
                for (int q = 0; q + 1 < kPoissonQueue; q++) {
                    qpos[q] = pop ? qpos[q + 1] : qpos[q];
                    qlast[q] = pop ? qlast[q + 1] : qlast[q];
                    qU[q] = pop ? qU[q + 1] : qU[q];
                }
                cnt -= pop;
                fresh = fresh || pop;
            }
        }
    }
    // staged samples and empty slots: a row of the tile (2^lth pixels) is contiguous
    // in memory and is written by the whole wavefront, so the stores coalesce
    __builtin_amdgcn_wave_barrier();
    const int th = 1 << cfg.lth;
    for (int r = 0; r < (64 >> cfg.lth); r++) {
        const int l0 = r << cfg.lth;
        const int ir = __shfl(i, l0, 64), jr = __shfl(j, l0, 64);
        const int cnt = ir < W ? (H - jr < th ? H - jr : th) : 0;          // wave-uniform
        if (cnt <= 0) continue;
        int32_t* rid = outIds + ((long)jr + (long)H * ir) * kcap;
        float* rip = outIpi + ((long)jr + (long)H * ir) * kcap;
        const int total = cnt * kcap;
        for (int e0 = 0; e0 < total; e0 += 64) {
            const int e = e0 + lane;
            const int c = e < total ? e / kcap : 0;
            const int nsc = __shfl(ns, l0 + c, 64);
            const int q = e - c * kcap;                   // slot of pixel l0 + c
            if (e < total) {
                if (q >= nsc) { rid[e] = -1; rip[e] = 0.0f; }
                else if (q < kPoissonStage) { rid[e] = sid[q * 64 + l0 + c]; rip[e] = sip[q * 64 + l0 + c]; }
            }
        }
    }
    if (over) atomicOr(err, 4);
}

// ---------------------------------------------------------------------------
// Per-tile features for the rate network (no reference counterpart): 16x16
// pixel tiles, 32 features each (layout in ude_tile_features).  Splat
// statistics are accumulated in fixed point with integer atomics, pixel
// statistics by fixed-order reductions, so the features are reproducible.
// ---------------------------------------------------------------------------
constexpr int kTileFeat = 32;
constexpr double kFix = 1048576.0;          // 2^20 fixed-point unit

struct TileAcc {
    unsigned long long cnt, sz, szz, sh;
    unsigned int hmax, pad;
};

__global__ __launch_bounds__(256) void k_tile_splats(int N, int W, int H, float ff, float smoothing,
                                                     const float* __restrict__ pts, const float* __restrict__ nrm,
                                                     const float* __restrict__ sd, TileAcc* acc)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= N) return;
    const float* p = pts + 3L * t;
    if (!(p[2] < 0.0f)) return;
    float sx, sy;
    screen_f32((float)W, (float)H, ff, p, sx, sy);
    if (!(sx >= 0.0f && sx < (float)W && sy >= 0.0f && sy < (float)H)) return;
    const int tH = (H + 15) / 16;
    TileAcc* a = acc + (long)((int)sx >> 4) * tH + ((int)sy >> 4);
    float z = -p[2];
    float h = prop_h((float)W, (float)H, ff, p, nrm + 3L * t, sd + 2L * t, smoothing);
    if (!(h >= 0.0f)) h = 0.0f;
    h = fminf(h, kProposalHCap);
    atomicAdd(&a->cnt, 1ull);
    atomicAdd(&a->sz, (unsigned long long)((double)z * kFix));
    atomicAdd(&a->szz, (unsigned long long)((double)z * (double)z * kFix));
    atomicAdd(&a->sh, (unsigned long long)((double)h * kFix));
    atomicMax(&a->hmax, __float_as_uint(h));
}

// block-wide sum / max / min over 256 threads, fixed order
__device__ __forceinline__ float blk_sum(float v, float* sh)
{
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) sh[threadIdx.x] = sh[threadIdx.x] + sh[threadIdx.x + s];
        __syncthreads();
    }
    float r = sh[0];
    __syncthreads();
    return r;
}

__device__ __forceinline__ float blk_max(float v, float* sh)
{
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) sh[threadIdx.x] = fmaxf(sh[threadIdx.x], sh[threadIdx.x + s]);
        __syncthreads();
    }
    float r = sh[0];
    __syncthreads();
    return r;
}

// one workgroup per tile, one thread per pixel
__global__ __launch_bounds__(256) void k_tile_pixels(int W, int H, float prec, const float* __restrict__ dens,
                                                     const float* __restrict__ gimg, const TileAcc* __restrict__ acc,
                                                     float* __restrict__ out)
{
    __shared__ float sh[256];
    const int tH = (H + 15) / 16;
    const int tile = blockIdx.x;
    const int ti = tile / tH, tj = tile - (tile / tH) * tH;
    const int i = ti * 16 + (threadIdx.x >> 4), j = tj * 16 + (threadIdx.x & 15);
    const bool in = i < W && j < H;
    const long pix = (long)j + (long)H * i;
    const float d0 = in ? log1pf(fmaxf(dens[pix], 0.0f)) : 0.0f;
    const float d1 = in ? log1pf(fmaxf(dens[(long)W * H + pix], 0.0f)) : 0.0f;
    float gm = 0.0f;
    if (in && gimg) {
        const float* g = gimg + 3 * pix;
        float s2 = g[0] * g[0];
        s2 = s2 + g[1] * g[1];
        s2 = s2 + g[2] * g[2];
        gm = sqrtf(s2);
    }
    const float np = blk_sum(in ? 1.0f : 0.0f, sh);
    const float inv = 1.0f / fmaxf(np, 1.0f);
    float f[kTileFeat];
    // splat statistics
    const TileAcc a = acc[tile];
    const float cnt = (float)a.cnt;
    const float ic = a.cnt ? 1.0f / cnt : 0.0f;
    const float mz = (float)((double)a.sz / kFix) * ic;
    const float mzz = (float)((double)a.szz / kFix) * ic;
    f[0] = log1pf(cnt);
    f[1] = mz;
    f[2] = sqrtf(fmaxf(mzz - mz * mz, 0.0f));
    f[3] = (float)((double)a.sh / kFix) * ic;
    f[4] = __uint_as_float(a.hmax);
    // densities (log1p), coverage, gradient magnitudes
    const float m0 = blk_sum(d0, sh) * inv, m1 = blk_sum(d1, sh) * inv;
    f[5] = m0;
    f[6] = blk_max(in ? d0 : 0.0f, sh);
    f[7] = -blk_max(in ? -d0 : -1e30f, sh);
    f[8] = sqrtf(fmaxf(blk_sum(in ? (d0 - m0) * (d0 - m0) : 0.0f, sh) * inv, 0.0f));
    f[9] = m1;
    f[10] = blk_max(in ? d1 : 0.0f, sh);
    f[11] = -blk_max(in ? -d1 : -1e30f, sh);
    f[12] = sqrtf(fmaxf(blk_sum(in ? (d1 - m1) * (d1 - m1) : 0.0f, sh) * inv, 0.0f));
    f[13] = blk_sum((in && dens[pix] >= prec) ? 1.0f : 0.0f, sh) * inv;
    const float mg = blk_sum(gm, sh) * inv;
    f[14] = mg;
    f[15] = blk_max(gm, sh);
    f[16] = sqrtf(fmaxf(blk_sum(in ? (gm - mg) * (gm - mg) : 0.0f, sh) * inv, 0.0f));
    f[17] = log1pf(blk_sum(gm * gm, sh));
    // quadrants: mean log density and mean gradient magnitude
    const int quad = ((threadIdx.x >> 7) << 1) | ((threadIdx.x >> 3) & 1);
    for (int q = 0; q < 4; q++) {
        const bool mine = quad == q && in;
        const float nq = fmaxf(blk_sum(mine ? 1.0f : 0.0f, sh), 1.0f);
        f[18 + 2 * q] = blk_sum(mine ? d0 : 0.0f, sh) / nq;
        f[19 + 2 * q] = blk_sum(mine ? gm : 0.0f, sh) / nq;
    }
    f[26] = ((float)ti * 16.0f + 8.0f) / (float)W;
    f[27] = ((float)tj * 16.0f + 8.0f) / (float)H;
    f[28] = log1pf(blk_sum(in ? fmaxf(dens[pix], 0.0f) : 0.0f, sh));
    f[29] = log1pf(blk_sum(in ? gm * fmaxf(dens[pix], 0.0f) : 0.0f, sh));
    f[30] = np * (1.0f / 256.0f);
    f[31] = log1pf(cnt * np * (1.0f / 256.0f));
    if (threadIdx.x < kTileFeat) out[(long)tile * kTileFeat + threadIdx.x] = f[threadIdx.x];
}

__global__ void k_zero_u64(unsigned long long* p, long n)
{
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = 0ull;
}

inline unsigned grid1(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// Tree structure of one view: bandwidth, cull, sort, hierarchy, bottom-up
// boxes / centres / counts / dynamic degrees.
int build_structure(int N, int W, int H, double f, double smoothing, double prec, const float* pts, const float* nrm,
                    const float* sd, const TreeWs& w, hipStream_t st, int views = 1, VStride vsd = VStride{})
{
    float Wf = (float)W, Hf = (float)H, ff = (float)f;
    if (N <= kFrontSplats) {
        k_front_small<<<dim3(1, views), 1024, 0, st>>>(N, Wf, Hf, ff, (float)smoothing, prec, pts, nrm, sd, w.vs, w.hraw,
                                                       w.keysA, w.idsA, vsd);
    } else {
        long nCull = (N + kCullTile - 1) / kCullTile;
        const bool small = sort_tile(N) == kSortTileSmall;
        long nSort = (N + sort_tile(N) - 1) / sort_tile(N);
        k_zero_state<<<dim3(1, views), 64, 0, st>>>(w.vs, vsd);
        // 256 workgroups of 1024 threads per view: 16 waves per CU stream the splats,
        // and the two sums take 512 device atomics (1M splats: 23.7 -> 17.2 us)
        const unsigned bwBlocks = grid1(N, 1024) < 256u ? grid1(N, 1024) : 256u;
        k_bandwidth<<<dim3(bwBlocks, views), 1024, 0, st>>>(N, Wf, Hf, ff, (float)smoothing, pts, nrm, sd, w.vs, w.hraw,
                                                           vsd);
        k_view_params<<<dim3(1, views), 64, 0, st>>>(w.vs, Wf, Hf, prec, vsd);
        k_cull_count<<<dim3((unsigned)nCull, views), 256, 0, st>>>(N, Wf, Hf, ff, pts, w.vs, w.cullCounts, vsd);
        // up to 256 counts the workgroups of the next launch add up themselves
        if (nCull > 256) k_scan_small<<<dim3(1, views), 1024, 0, st>>>(w.cullCounts, (int)nCull, &w.vs->nc, vsd);
        k_cull_scatter<<<dim3((unsigned)nCull, views), 256, 0, st>>>(N, Wf, Hf, ff, pts, w.vs, w.cullCounts, w.keysB, w.idsB, vsd);
        uint32_t* kin = w.keysB; uint32_t* kout = w.keysA;
        int32_t* iin = w.idsB; int32_t* iout = w.idsA;
        for (int shift = 0; shift < 24; shift += 8) {                  // 20-bit keys
            const dim3 grid((unsigned)nSort, views);
            if (small) {
                k_sort_hist<kSortTileSmall><<<grid, 256, 0, st>>>(w.vs, kin, shift, (int)nSort, w.sortHist, vsd);
                k_sort_scatter<kSortTileSmall><<<grid, 256, 0, st>>>(w.vs, kin, iin, shift, (int)nSort, w.sortHist,
                                                                     nullptr, kout, iout, vsd);
            } else {
                k_sort_hist<kSortTile><<<grid, 256, 0, st>>>(w.vs, kin, shift, (int)nSort, w.sortHist, vsd);
                k_sort_scan_digits<<<dim3(256, views), 256, 0, st>>>(w.sortHist, (int)nSort, w.scanBlocks, vsd);
                k_sort_scatter<kSortTile><<<grid, 256, 0, st>>>(w.vs, kin, iin, shift, (int)nSort, w.sortHist,
                                                                w.scanBlocks, kout, iout, vsd);
            }
            uint32_t* tk = kin; kin = kout; kout = tk;
            int32_t* ti = iin; iin = iout; iout = ti;
        }
    }
    // the sorted data is in keysA / idsA (three passes)
    k_hierarchy<<<dim3(grid1(N, 256), views), 256, 0, st>>>(Wf, Hf, ff, pts, w.vs, w.keysA, w.idsA, w.geo, w.lnk, w.aux, w.leafXY,
                                                            w.flags, vsd);
    k_bottom_up_local<<<dim3(grid1(N, kFanBlock), views), kFanBlock, 0, st>>>(w.vs, w.geo, w.lnk, w.aux, w.seeds, vsd);
    k_bottom_up_global<<<dim3(grid1(N, 256), views), 256, 0, st>>>(w.vs, w.geo, w.lnk, w.aux, w.flags, w.seeds, vsd);
    hipError_t e0 = hipGetLastError();
    return e0 == hipSuccess ? UDE_OK : UDE_ERR_LAUNCH;
}

// Dynamic-degree Hermite moments of the sampler's tree.
int build_moments(int N, int k, const TreeWs& w, hipStream_t st, int views, VStride vsd)
{
    k_coef_blocks<<<dim3(grid1(2L * N, kCoefThreads), views), kCoefThreads, 0, st>>>(w.vs, w.geo, w.lnk, w.aux, k, w.momList, vsd);
    // enough workgroups for max(N leaves / 256, N nodes / 15)
    k_moments<<<dim3(grid1(N, kMomNodes), views), 256, 0, st>>>(w.vs, w.geo, w.aux, w.momList, w.coef, w.leafXY, w.lnk, w.srec,
                                                                w.walkQueue, w.tieQueue, vsd);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? UDE_OK : UDE_ERR_LAUNCH;
}

int num_launches(int k)
{
    int L = 0;
    while ((double)L < sqrt((double)k)) L++;
    return L;
}

// trie entries per lane: room for the walk plus what the descents may add
int trie_entries(int k) { return kWalkEntries + walk_extra(num_launches(k)); }

// Optional timing of one sampling kernel (0 the walk + draw pair of
// sampling.sample, 1 k_fmm_eval, 2 k_poisson): while enabled, its launches are
// bracketed by pairs of HIP events recorded on their stream (single host
// thread; events are pooled and reused across profiling windows).
struct SamplerTiming {
    bool on = false;
    int kernel = 0;
    int used = 0;
    std::vector<std::pair<hipEvent_t, hipEvent_t>> pool;
};
SamplerTiming g_timing;

bool timing_pair(int kernel, hipEvent_t* a, hipEvent_t* b)
{
    if (!g_timing.on || g_timing.kernel != kernel) return false;
    if (g_timing.used == (int)g_timing.pool.size()) {
        hipEvent_t x, y;
        if (hipEventCreate(&x) != hipSuccess) return false;
        if (hipEventCreate(&y) != hipSuccess) { (void)hipEventDestroy(x); return false; }
        g_timing.pool.push_back({x, y});
    }
    *a = g_timing.pool[g_timing.used].first;
    *b = g_timing.pool[g_timing.used].second;
    g_timing.used++;
    return true;
}

// The sampler's per-pixel passes over `views` views (workspaces vsd.ws bytes apart).
void launch_sample(int N, int W, int H, int k, uint32_t seedLo, uint32_t seedHi, uint32_t view, const TreeWs& w,
                   int32_t* out, int* err, hipStream_t st, int views, VStride vsd)
{
    const unsigned tiles = (unsigned)(((W + 7) / 8) * ((H + 7) / 8));
    const int L = num_launches(k);
    hipEvent_t e0, e1;
    bool timed = timing_pair(0, &e0, &e1);
    if (timed) (void)hipEventRecord(e0, st);
    const dim3 wg(tiles, views);
    k_sample_walk<false><<<wg, 64 * kWalkWaves, 0, st>>>(W, H, k, L, w.vs, w.geo, w.lnk, w.aux, w.coef, w.srec, w.trie,
                                                         trie_entries(k), w.tileInfo, w.walkQueue, vsd);
    k_sample_walk<true><<<wg, 64 * kWalkWaves, 0, st>>>(W, H, k, L, w.vs, w.geo, w.lnk, w.aux, w.coef, w.srec, w.trie,
                                                        trie_entries(k), w.tileInfo, w.walkQueue, vsd);
    k_sample_descend<<<wg, 64, 0, st>>>(W, H, k, L, w.vs, w.geo, w.lnk, w.aux, w.coef, w.srec, w.trie, trie_entries(k),
                                        w.tileInfo, w.reach, err, vsd);
    // a pixel has at most L ceil(k / 4) Philox blocks, 64 per iteration: 8 x 16, 12 x 32
    // and 16 x 64 at k = 64, 128 and 256
    auto draw = [&](auto turns) {
        constexpr int T = decltype(turns)::value;
        const dim3 dg(tiles * (64 / (kDrawWaves * T)), views);
#define UD_DRAW(R, I) k_sample_draw<R, I, T><<<dg, 64 * kDrawWaves, 0, st>>>(                                         \
        W, H, k, L, (int)tiles, seedLo, seedHi, view, w.vs, w.leafXY, w.idsA, w.reach, out, w.tieQueue, vsd)
        if (draw_halves(k, L)) {
            constexpr int TH = T > 8 ? 8 : T;
            k_sample_draw_halves<TH><<<dim3(tiles * (32 / (kDrawWaves * TH)), views), 64 * kDrawWaves, 0, st>>>(
                W, H, k, L, (int)tiles, seedLo, seedHi, view, w.vs, w.leafXY, w.idsA, w.reach, out, w.tieQueue, vsd);
        } else if (k <= 64) UD_DRAW(1, 2);
        else if (k <= 128) UD_DRAW(2, 6);
        else UD_DRAW(4, 16);
    };
    if ((long)tiles * views >= kDrawManyTiles && k <= 128) draw(std::integral_constant<int, kDrawTurns>{});
    else draw(std::integral_constant<int, 1>{});
#undef UD_DRAW
    k_sample_replay<<<dim3(64, views), 64, 0, st>>>(W, H, k, L, tiles, seedLo, seedHi, view, w.vs, w.leafXY, w.idsA,
                                                    w.reach, w.tieQueue, out, vsd);
    if (timed) (void)hipEventRecord(e1, st);
}

// proposal of ude_sample_poisson: 0 the two density bands, 1 the wide band plus the
// footprint half; scale 0 = normaliser from the view, > 0 the caller's
int g_pois_mode = 0;
double g_pois_scale = 0.0;

// launch shapes of k_fmm_eval (0) and k_poisson (1); set by ude_set_tile_config
TileCfg g_tile[2] = {{8, 3, 4, 0}, {8, 3, 4, 0}};

dim3 tile_grid(const TileCfg& c, int W, int H, int views)
{
    const int th = 1 << c.lth;
    const long ntiles = (long)((W + c.tw - 1) / c.tw) * ((H + th - 1) / th);
    return dim3((unsigned)((ntiles + c.wpb - 1) / c.wpb), (unsigned)views);
}

// degree-6 expansions of bands 0 .. nbands-1 on one view's tree (or a batch)
void fixed_expansions(int N, int nbands, int p, const TreeWs& w, hipStream_t st, int views = 1,
                      VStride vsd = VStride{})
{
    k_fixed_select<<<dim3(grid1(N, kSelectThreads), views), kSelectThreads, 0, st>>>(
        w.vs, nbands, p, w.geo, w.lnk, w.fixOff[0], nbands > 1 ? w.fixOff[1] : nullptr, w.fixList[0],
        nbands > 1 ? w.fixList[1] : nullptr, vsd);
    const dim3 grid(grid1(N, 256 / (p + 1)), views, nbands);
    switch (p) {
#define UD_MOMENTS(P) case P: k_fixed_moments<P><<<grid, 256, 0, st>>>(w.vs, w.geo, w.aux, w.leafXY, w.fixList[0], \
                                                                        w.fixList[1], w.fixOff[0], w.fixOff[1],    \
                                                                        w.fixCoef[0], w.fixCoef[1], vsd); break;
    UD_MOMENTS(4) UD_MOMENTS(5) UD_MOMENTS(6) UD_MOMENTS(7) UD_MOMENTS(8)
#undef UD_MOMENTS
    default: break;
    }
}

// densities of bands 0 .. nbands-1 of `views` views in one launch: w is the
// first view's workspace, the others follow vstride bytes apart; view v writes
// band b to out + v outStride + b bandStride bytes
void fmm_eval(int N, int W, int H, int views, int nbands, int p, const TreeWs& w, size_t vstride, float* out,
              size_t outStride, size_t bandStride, hipStream_t st)
{
    const TileCfg c = g_tile[0];
    hipEvent_t e0, e1;
    bool timed = timing_pair(1, &e0, &e1);
    if (timed) (void)hipEventRecord(e0, st);
    const dim3 grid = tile_grid(c, W, H, views * nbands);
    const int list = N < kFmmListShortSplats * (((long)W * H + 63) / 64) ? kFmmListShort : kFmmList;
    switch (p) {
#define UD_EVAL(P) case P: k_fmm_eval<P><<<grid, 64 * c.wpb, fmm_lds(P, c.wpb, list), st>>>(                       \
        c, W, H, list, w.vs, vstride, nbands, w.geo, w.aux, w.frec, w.fixOff[0], nbands > 1 ? w.fixOff[1] : nullptr,            \
        w.fixCoef[0], nbands > 1 ? w.fixCoef[1] : nullptr, out, outStride, bandStride); break;
    UD_EVAL(4) UD_EVAL(5) UD_EVAL(6) UD_EVAL(7) UD_EVAL(8)
#undef UD_EVAL
    default: break;
    }
    if (timed) (void)hipEventRecord(e1, st);
}

// degree of the fixed-order expansions; set by ude_set_fixed_degree
int g_fixed_p = kFixedDegree;

} // namespace

extern "C" {

size_t ude_sample_workspace_bytes(int N, int W, int H, int k)
{
    return carve(nullptr, N, W, H, k, kModeSample, nullptr) + 256;
}

int ude_sample(int bn, int N, int W, int H, int k, double f, double smoothing, double prec,
               const float* pts, const float* nrm, const float* sd, int sdBatch,
               uint64_t seed, int32_t* out, int* errFlag, void* ws, size_t wsBytes, hipStream_t st)
{
    if (bn <= 0 || W <= 0 || H <= 0 || k <= 0 || N < 0) return UDE_ERR_ARG;
    if (k > 256) return UDE_ERR_ARG;
    long perView = (long)W * H * k;
    if (N == 0) {
        k_fill_idx<<<grid1(perView * bn, 256), 256, 0, st>>>(out, perView * bn);
        return UDE_OK;
    }
    if (wsBytes < ude_sample_workspace_bytes(N, W, H, k)) return UDE_ERR_WORKSPACE;
    // as many views at once as the workspace holds
    TreeWs w;
    const size_t per = carve(ws, N, W, H, k, kModeSample, &w);
    const size_t most = bn < 65535 ? bn : 65535;             // views are the grid's second dimension
    const int span = (int)((wsBytes - 256) / per < most ? (wsBytes - 256) / per : most);
    uint32_t sLo = (uint32_t)seed, sHi = (uint32_t)(seed >> 32);
    for (int b = 0; b < bn; b += span) {
        const int views = span < bn - b ? span : bn - b;
        const VStride vsd{per, sizeof(float) * 3 * (size_t)N, sdBatch > 1 ? sizeof(float) * 2 * (size_t)N : 0};
        const float* pb = pts + 3L * N * b;
        const float* nb = nrm + 3L * N * b;
        const float* sb = sd + (sdBatch > 1 ? 2L * N * b : 0);
        int rc = build_structure(N, W, H, f, smoothing, prec, pb, nb, sb, w, st, views, vsd);
        if (rc == UDE_OK) rc = build_moments(N, k, w, st, views, vsd);
        if (rc != UDE_OK) return rc;
        launch_sample(N, W, H, k, sLo, sHi, (uint32_t)b, w, out + perView * b, errFlag, st, views, vsd);
    }
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? UDE_OK : UDE_ERR_LAUNCH;
}

size_t ude_fmm_weights_workspace_bytes(int N, int W, int H)
{
    return carve(nullptr, N, W, H, 0, kModeFixed, nullptr) + 256;
}

int ude_fmm_weights(int bn, int N, int W, int H, double f, double smoothing, double prec,
                    const float* pts, const float* nrm, const float* sd, int sdBatch,
                    float* out, void* ws, size_t wsBytes, hipStream_t st)
{
    if (bn <= 0 || W <= 0 || H <= 0 || N < 0) return UDE_ERR_ARG;
    long perView = (long)W * H;
    if (N == 0) {
        k_fill_f32<<<grid1(perView * bn, 256), 256, 0, st>>>(out, perView * bn, 0.0f);
        hipError_t e = hipGetLastError();
        return e == hipSuccess ? UDE_OK : UDE_ERR_LAUNCH;
    }
    if (wsBytes < ude_fmm_weights_workspace_bytes(N, W, H)) return UDE_ERR_WORKSPACE;
    const int p = g_fixed_p;
    TreeWs w;
    carve(ws, N, W, H, 0, kModeFixed, &w);
    for (int b = 0; b < bn; b++) {
        const float* pb = pts + 3L * N * b;
        const float* nb = nrm + 3L * N * b;
        const float* sb = sd + (sdBatch > 1 ? 2L * N * b : 0);
        int rc = build_structure(N, W, H, f, smoothing, prec, pb, nb, sb, w, st);
        if (rc != UDE_OK) return rc;
        fixed_expansions(N, 1, p, w, st);
        k_fmm_records<<<grid1(N, 256), 256, 0, st>>>(w.vs, w.geo, w.lnk, w.fixOff[0], nullptr, w.frec, VStride{});
        fmm_eval(N, W, H, 1, 1, p, w, 0, out + perView * b, 0, 0, st);
    }
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? UDE_OK : UDE_ERR_LAUNCH;
}

size_t ude_poisson_workspace_bytes(int bn, int N, int W, int H)
{
    return carve(nullptr, N, W, H, 0, kModePoisson, nullptr) * (size_t)(bn > 1 ? bn : 1) + 256;
}

int ude_sample_poisson(int bn, int N, int W, int H, int kcap, double f, double smoothing, double prec,
                       double rate, const float* tileScale, const float* pts, const float* nrm, const float* sd,
                       int sdBatch, uint64_t seed, const uint64_t* seedDev, int32_t* outIds, float* outIpi,
                       float* densOut, int* errFlag, void* ws, size_t wsBytes, hipStream_t st)
{
    if (bn <= 0 || W <= 0 || H <= 0 || kcap <= 0 || N < 0 || !(rate >= 0.0)) return UDE_ERR_ARG;
    long perView = (long)W * H;
    if (N == 0) {
        k_fill_idx<<<grid1(perView * kcap * bn, 256), 256, 0, st>>>(outIds, perView * kcap * bn);
        k_fill_f32<<<grid1(perView * kcap * bn, 256), 256, 0, st>>>(outIpi, perView * kcap * bn, 0.0f);
        if (densOut) k_fill_f32<<<grid1(perView * 2 * bn, 256), 256, 0, st>>>(densOut, perView * 2 * bn, 0.0f);
        hipError_t e = hipGetLastError();
        return e == hipSuccess ? UDE_OK : UDE_ERR_LAUNCH;
    }
    // all views' trees resident at once when the workspace holds them: every
    // per-pixel pass is then one launch over the whole batch; otherwise view by view
    const size_t per = carve(nullptr, N, W, H, 0, kModePoisson, nullptr);
    const bool batched = bn > 1 && wsBytes >= per * (size_t)bn + 256;
    if (!batched && wsBytes < per + 256) return UDE_ERR_WORKSPACE;
    const int span = batched ? bn : 1;
    const int tsW = (W + 15) / 16, tsH = (H + 15) / 16;
    const uint32_t sLo = (uint32_t)seed, sHi = (uint32_t)(seed >> 32);
    const TileCfg pc = g_tile[1];
    const int p = g_fixed_p;
    const int fmode = g_pois_mode;
    const float fscale = (float)g_pois_scale;
    for (int g = 0; g < bn; g += span) {
        // every view of the group in one launch per build stage (view = blockIdx.y)
        TreeWs w;
        carve(ws, N, W, H, 0, kModePoisson, &w);
        const VStride vsd{per, sizeof(float) * 3 * (size_t)N, sdBatch > 1 ? sizeof(float) * 2 * (size_t)N : 0};
        const float* pb = pts + 3L * N * g;
        const float* nb = nrm + 3L * N * g;
        const float* sb = sd + (sdBatch > 1 ? 2L * N * g : 0);
        int rc = build_structure(N, W, H, f, smoothing, prec, pb, nb, sb, w, st, span, vsd);
        if (rc != UDE_OK) return rc;
        k_wide_hist<<<dim3(grid1(N, 256) < 256u ? grid1(N, 256) : 256u, span), 256, 0, st>>>(w.vs, w.idsA, w.hraw,
                                                                                          vsd);
        k_wide_band<<<dim3(1, span), 256, 0, st>>>(w.vs, vsd);
        fixed_expansions(N, 2, p, w, st, span, vsd);
        k_walk_records<<<dim3(grid1(2L * N, 256), span), 256, 0, st>>>(w.vs, w.geo, w.lnk, w.aux, w.fixOff[0],
                                                                       w.fixOff[1], w.pnode, w.frec, vsd);
        // footprint proposal: the leaves' footprint records and their node bounds
        if (fmode) {
            k_zero_f64<<<(span + 63) / 64, 64, 0, st>>>(w.footSum, per, span);
            k_foot_leaves<<<dim3(grid1(N, 256), span), 256, 0, st>>>((float)W, (float)H, (float)f, (float)smoothing,
                                                                     pb, nb, sb, w.vs, w.idsA, w.leafXY, w.footLeaf,
                                                                     w.footSum, vsd);
        }
        float* d0 = densOut ? densOut + perView * 2 * g : w.dens[0];
        float* d1 = densOut ? d0 + perView : w.dens[1];
        const size_t dstride = densOut ? sizeof(float) * 2 * perView : per;
        fmm_eval(N, W, H, span, 2, p, w, per, d0, dstride, (size_t)((char*)d1 - (char*)d0), st);
        const float* ts = tileScale ? tileScale + (long)tsW * tsH * g : nullptr;
        hipEvent_t e0, e1;
        bool timed = timing_pair(2, &e0, &e1);
        if (timed) (void)hipEventRecord(e0, st);
        k_poisson<<<tile_grid(pc, W, H, span), 64 * pc.wpb, kPoissonStageBytes * pc.wpb, st>>>(
            pc, W, H, kcap, (float)rate, ts, tsH, sLo, sHi, seedDev, (uint32_t)g, w.vs, per, w.pnode, w.leafXY,
            w.idsA, d0, d1, dstride, outIds + perView * kcap * g, outIpi + perView * kcap * g, errFlag, fmode,
            fscale, w.footLeaf, w.footSum);
        if (timed) (void)hipEventRecord(e1, st);
    }
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? UDE_OK : UDE_ERR_LAUNCH;
}

int ude_set_poisson_proposal(int mode, double footprintScale)
{
    if (mode != 0 && mode != 1) return UDE_ERR_ARG;
    if (!(footprintScale <= 3.0e38)) return UDE_ERR_ARG;          // NaN or too large for float
    g_pois_mode = mode;
    g_pois_scale = footprintScale > 0.0 ? footprintScale : 0.0;
    return UDE_OK;
}

int ude_get_poisson_proposal(double* footprintScale)
{
    if (footprintScale) *footprintScale = g_pois_scale;
    return g_pois_mode;
}

int ude_set_fixed_degree(int p)
{
    if (p < kFixedPMin || p > kFixedPMax) return UDE_ERR_ARG;
    g_fixed_p = p;
    return UDE_OK;
}

int ude_get_fixed_degree(void)
{
    return g_fixed_p;
}

int ude_set_tile_config(int kernel, int tileW, int tileH, int wavesPerBlock, int xcdOrder)
{
    if (kernel < 0 || kernel > 1) return UDE_ERR_ARG;
    if (tileW <= 0 || tileH <= 0 || tileW * tileH != 64 || (tileW & (tileW - 1))) return UDE_ERR_ARG;
    if (wavesPerBlock != 1 && wavesPerBlock != 2 && wavesPerBlock != 4 && wavesPerBlock != 8) return UDE_ERR_ARG;
    if (xcdOrder != 0 && xcdOrder != 1) return UDE_ERR_ARG;
    int lth = 0;
    while ((1 << lth) < tileH) lth++;
    g_tile[kernel] = TileCfg{tileW, lth, wavesPerBlock, xcdOrder};
    return UDE_OK;
}

int ude_get_tile_config(int kernel, int* cfg)
{
    if (kernel < 0 || kernel > 1 || !cfg) return UDE_ERR_ARG;
    const TileCfg c = g_tile[kernel];
    cfg[0] = c.tw; cfg[1] = 1 << c.lth; cfg[2] = c.wpb; cfg[3] = c.xcd;
    return UDE_OK;
}

size_t ude_tile_features_workspace_bytes(int W, int H)
{
    return sizeof(TileAcc) * (size_t)((W + 15) / 16) * ((H + 15) / 16) + 256;
}

int ude_tile_features(int bn, int N, int W, int H, double f, double smoothing, double prec, const float* pts,
                      const float* nrm, const float* sd, int sdBatch, const float* dens, const float* gimg,
                      float* out, void* ws, size_t wsBytes, hipStream_t st)
{
    if (bn <= 0 || W <= 0 || H <= 0 || N < 0 || !dens) return UDE_ERR_ARG;
    if (wsBytes < ude_tile_features_workspace_bytes(W, H)) return UDE_ERR_WORKSPACE;
    const int tiles = ((W + 15) / 16) * ((H + 15) / 16);
    TileAcc* acc = (TileAcc*)ws;
    const long perView = (long)W * H;
    for (int b = 0; b < bn; b++) {
        k_zero_u64<<<grid1((long)tiles * 5, 256), 256, 0, st>>>((unsigned long long*)acc, (long)tiles * 5);
        if (N > 0)
            k_tile_splats<<<grid1(N, 256), 256, 0, st>>>(N, W, H, (float)f, (float)smoothing, pts + 3L * N * b,
                                                         nrm + 3L * N * b, sd + (sdBatch > 1 ? 2L * N * b : 0), acc);
        k_tile_pixels<<<tiles, 256, 0, st>>>(W, H, (float)prec, dens + 2 * perView * b,
                                             gimg ? gimg + 3 * perView * b : nullptr, acc,
                                             out + (long)tiles * kTileFeat * b);
    }
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? UDE_OK : UDE_ERR_LAUNCH;
}

int ude_profile_sampler_begin(int kernel)
{
    if (kernel < 0 || kernel > 2) return UDE_ERR_ARG;
    g_timing.kernel = kernel;
    g_timing.on = true;
    g_timing.used = 0;
    return UDE_OK;
}

int ude_profile_sampler_end(double* totalMs, int* launches)
{
    double tot = 0.0;
    int n = g_timing.used;
    g_timing.on = false;
    for (int q = 0; q < n; q++) {
        float ms = 0.0f;
        if (hipEventSynchronize(g_timing.pool[q].second) != hipSuccess) return UDE_ERR_LAUNCH;
        if (hipEventElapsedTime(&ms, g_timing.pool[q].first, g_timing.pool[q].second) != hipSuccess)
            return UDE_ERR_LAUNCH;
        tot += ms;
    }
    g_timing.used = 0;
    if (totalMs) *totalMs = tot;
    if (launches) *launches = n;
    return UDE_OK;
}

} // extern "C"
