// ud_gather.hip -- the pixelgather and nearestsamples op surfaces (gfx950):
//   pixelgather.scatter  per-slot copy of the sampled splats' attribute rows
//   pixelgather.gather   its adjoint: per-splat sums of per-slot rows
//   (splatting/extensions/pixelGather.cpp:10-23, pixelGatherCuda.cu:7-152)
//   nearestsamples.nearest  per splat, its nearest co-sampled splats
//   (FMMKdTreeSampling/nearestSamples.cpp:30-75, nearestSamplesCuda.cu:290-564)
//
// Slot tensors are x-major (bn, W, H, k) with pixel (i, j) at j + H (i + W b);
// a slot's row of C channels is contiguous, so the scatter output
// (bn, W, H, k, C) is written by consecutive threads at consecutive addresses
// and the kernels are bound by HBM streaming plus the row gathers.
#include "ud_device.h"
#include "../../include/udsplat.h"

#include <climits>
#include <hip/hip_fp16.h>

namespace {

inline unsigned grid1(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

inline int launch_status()
{
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? UDE_OK : UDE_ERR_LAUNCH;
}

// orders the wavefront's LDS accesses (its LDS operations execute in order)
__device__ __forceinline__ void wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// One thread per output element (slot, channel): out = values[b, id, c] or 0.
template <class T>
__global__ __launch_bounds__(256) void k_pixel_scatter(long nslots, int WHk, int N, int C,
                                                       const int32_t* __restrict__ idx,
                                                       const T* __restrict__ values, T* __restrict__ out)
{
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nslots * C) return;
    const long slot = e / C;
    const int c = (int)(e - slot * C);
    const int id = idx[slot];
    const long b = slot / WHk;
    out[e] = id >= 0 ? values[((long)b * N + id) * C + c] : T(0);
}

// One thread per (slot, channel) input element, added into the splat's row.
// Zero entries add nothing and are skipped (the sums are the same).  Bound by the
// atomics, one per element.
template <class T>
__global__ __launch_bounds__(256) void k_pixel_gather(long nslots, int WHk, int N, int C,
                                                      const int32_t* __restrict__ idx,
                                                      const T* __restrict__ values, T* __restrict__ out)
{
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nslots * C) return;
    const long slot = e / C;
    const int c = (int)(e - slot * C);
    const int id = idx[slot];
    if (id < 0) return;
    const T v = values[e];
    if (v == T(0)) return;
    const long b = slot / WHk;
    atomicAdd(out + ((long)b * N + id) * C + c, v);
}

// The rows of a tile of pixels are summed in LDS first: neighbouring pixels draw from the
// same splats, so a tile's slots name far fewer splats than there are slots and the global
// atomics drop by that factor.  The sums live in a hash table of the splats' indices.  A
// chunk of 1024 slots looks its entries up, one slot per thread, then adds its elements,
// one per thread, so that rows are read and written by consecutive lanes; a slot that
// finds no entry within kGatherProbes steps adds to global memory.  A chunk in which more
// than 7 slots of 8 met a splat for the first time, or found no entry, shows that the
// tile's slots share little: the rest of the tile then adds to global memory.  A workgroup
// fills half a CU, and its table half of what LDS that leaves.
// 100 000 splats, 2 x 256x256 x 16 slots of three channels, drawn from 390 splats per tile:
// 51 us, where one global atomic per element took 108 us; slots drawn from all splats, which
// a tile cannot sum: 71 us for one view against 63 us.
constexpr int kGatherProbes = 8, kGatherLds = 64 * 1024, kGatherMinEntries = 512, kGatherThreads = 1024;

// entries of the table: the largest power of two that fits
inline int gather_entries(size_t rowBytes)
{
    int e = 4096;
    while (e >= kGatherMinEntries && e * (rowBytes + sizeof(int32_t)) > kGatherLds) e /= 2;
    return e;
}

// Where a tile's sums gain.  Setting up and writing out the tables takes some 6 us more than
// the atomics of a small call, the more the wider the rows.  Atomics against tiles, us:
//   float, one channel:   200x150 of 8 slots 21 / 10, 40x30 of 40 5 / 11
//   three:                200x150 of 8 23 / 17, 2 x 100x100 of 16 20 / 24, 64x64 of 24 15 / 17
//   six:                  200x150 of 24 54 / 37, 100x80 of 40 23 / 33
//   eight:                512x512 of 40 473 / 477, 300x300 of 40 142 / 168 (rows of 32 bytes
//                         reach memory as whole sectors, which sums by element do not beat)
//   twelve:               400x300 of 24 233 / 194, 2 x 250x250 of 16 122 / 151
//   double, three:        200x150 of 8 18 / 16, 40x30 of 40 16 / 17
//   six:                  512x512 of 2 37 / 25, 8 x 40x30 of 40 16 / 19
// One slot per pixel has nothing to share within it (512x512, three channels, 18 / 22).
template <class T>
inline bool gather_by_tiles(long nslots, int k, int C)
{
    if (k < 2) return false;
    if (sizeof(T) == 8) return nslots >= (C <= 3 ? 200000 : 500000);
    if (C >= 8) return C >= 12 && nslots >= 2500000;
    return nslots >= (C <= 3 ? 200000 : 700000);
}

template <class T>
__global__ __launch_bounds__(kGatherThreads) void k_pixel_gather_tile(int W, int H, int k, int N, int C, int side,
                                                                     int entries, const int32_t* __restrict__ idx,
                                                                     const T* __restrict__ values,
                                                                     T* __restrict__ out)
{
    extern __shared__ __align__(16) unsigned char gatherLds[];
    T* sum = (T*)gatherLds;                             // [entries][C]
    int32_t* key = (int32_t*)(sum + entries * C);
    __shared__ int slotEntry[kGatherThreads];           // the chunk's slots: entry, -1 none, -2 empty slot
    __shared__ int slotId[kGatherThreads];
    __shared__ int fresh[2], used[2];                   // of the chunk, alternating
    const int t = threadIdx.x;
    for (int e = t; e < entries * C; e += kGatherThreads) sum[e] = T(0);
    for (int e = t; e < entries; e += kGatherThreads) key[e] = -1;
    if (t < 2) { fresh[t] = 0; used[t] = 0; }
    __syncthreads();
    const int tilesH = (H + side - 1) / side, ti = blockIdx.x / tilesH, tj = blockIdx.x - ti * tilesH;
    const int w = min(side, W - side * ti), h = min(side, H - side * tj);
    const long b = blockIdx.y;
    T* o = out + b * N * C;
    const int line = h * k;                             // slots of one i: contiguous
    const int shift = __clz(entries) + 1;               // the hash's top log2(entries) bits
    bool direct = false;
    for (int c0 = 0, turn = 0; c0 < w * line; c0 += kGatherThreads, turn ^= 1) {
        const int n = min(kGatherThreads, w * line - c0);
        if (t < n) {
            const int di = (c0 + t) / line, q = c0 + t - di * line;
            const int id = idx[((b * W + side * ti + di) * H + side * tj) * k + q];
            int found = id < 0 ? -2 : -1;
            bool first = id >= 0;
            if (id >= 0 && !direct) {
                int e = (int)(((unsigned)id * 2654435769u) >> shift);
                for (int probe = 0; probe < kGatherProbes; probe++) {
                    int old = key[e];
                    if (old == -1) old = atomicCAS(key + e, -1, id);
                    if (old == -1 || old == id) { found = e; first = old == -1; break; }
                    e = (e + 1) & (entries - 1);
                }
            }
            slotEntry[t] = found;
            slotId[t] = id;
            const unsigned long long mf = __ballot(first), mu = __ballot(id >= 0);
            if ((t & 63) == 0) { atomicAdd(fresh + turn, __popcll(mf)); atomicAdd(used + turn, __popcll(mu)); }
        }
        __syncthreads();
        for (int x = t; x < n * C; x += kGatherThreads) {
            const int s = x / C, c = x - s * C, e = slotEntry[s];
            if (e == -2) continue;
            const int di = (c0 + s) / line, q = c0 + s - di * line;
            const T v = values[(((b * W + side * ti + di) * H + side * tj) * k + q) * C + c];
            if (v == T(0)) continue;
            if (e >= 0) atomicAdd(sum + e * C + c, v);
            else atomicAdd(o + (long)slotId[s] * C + c, v);
        }
        direct = direct || 8 * fresh[turn] > 7 * used[turn];
        if (t == 0) { fresh[turn ^ 1] = 0; used[turn ^ 1] = 0; }
        __syncthreads();
    }
    for (int x = t; x < entries * C; x += kGatherThreads) {
        const T v = sum[x];
        if (v == T(0)) continue;
        const int e = x / C;
        atomicAdd(o + (long)key[e] * C + (x - e * C), v);
    }
}

template <class T>
int scatter_t(int bn, int W, int H, int k, int N, int C, const int32_t* idx, const T* values, T* out, hipStream_t st)
{
    if (bn <= 0 || W <= 0 || H <= 0 || k <= 0 || N < 0 || C <= 0) return UDE_ERR_ARG;
    const long nslots = (long)bn * W * H * k;
    k_pixel_scatter<T><<<grid1(nslots * C, 256), 256, 0, st>>>(nslots, W * H * k, N, C, idx, values, out);
    return launch_status();
}

template <class T>
int gather_t(int bn, int W, int H, int k, int N, int C, const int32_t* idx, const T* values, T* out, hipStream_t st)
{
    if (bn <= 0 || W <= 0 || H <= 0 || k <= 0 || N < 0 || C <= 0) return UDE_ERR_ARG;
    if (N == 0) return UDE_OK;
    const long nslots = (long)bn * W * H * k;
    // tiles of 16x16 where they keep most of the 256 CUs at two workgroups, else of 8x8 (three
    // channels: 280x290 pixels, 342 tiles, 101 us against 69; 400x300, 475 tiles, 72 against 77)
    auto tiles = [&](int side) { return (long)((W + side - 1) / side) * ((H + side - 1) / side); };
    const int side = tiles(16) * bn >= 400 ? 16 : 8;
    const int entries = gather_entries((size_t)C * sizeof(T));
    if (gather_by_tiles<T>(nslots, k, C) && entries >= kGatherMinEntries && k <= 1024 && tiles(side) <= INT_MAX &&
        bn <= 65535)
        k_pixel_gather_tile<T><<<dim3((unsigned)tiles(side), bn), kGatherThreads,
                                 entries * (C * sizeof(T) + sizeof(int32_t)), st>>>(W, H, k, N, C, side, entries, idx,
                                                                                    values, out);
    else
        k_pixel_gather<T><<<grid1(nslots * C, 256), 256, 0, st>>>(nslots, W * H * k, N, C, idx, values, out);
    return launch_status();
}

// ---------------------------------------------------------------------------
// nearestsamples.nearest.  A pixel's surface splat is the first slot of largest
// weight (nearestSamplesCuda.cu:306-321); every other splat sampled at the pixel
// is a candidate neighbour of the surface splat at squared distance d2 (float32,
// ((dx dx + dy dy) + dz dz)).  Each splat keeps the K smallest (d2, index) words
// (distance bits high, index low: ties by index) in a sorted row of K 64-bit
// slots.  A candidate enters by a cascade of atomicMin over the row: each slot
// keeps the smaller word and the larger one moves on to the next slot, so every
// word that leaves slot j reaches slot j + 1; a slot returning the candidate's
// own word means another pixel inserted the same neighbour, and the copy is
// dropped.  The final rows are the K nearest distinct candidates in order,
// whatever order the pixels ran in (the reference merges under a spin lock per
// splat, nearestSamplesCuda.cu:370-404).
// ---------------------------------------------------------------------------
constexpr unsigned long long kNearestEmpty = ~0ull;

__global__ void k_fill_u64(unsigned long long* __restrict__ p, long n, unsigned long long v)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = v;
}

// lanes of a pixel: the power of two that holds its slots, at most a wavefront
inline int nearest_lanes(int k)
{
    int p = 1;
    while (p < k && p < 64) p *= 2;
    return p;
}

// `lanes` lanes per pixel, one candidate each (lanes strided by `lanes` when k > 64).
// A candidate's cascade starts at a slot that its final one is not before: the number of
// words known to be smaller, those of the row as read and those that the pixel's other
// candidates bring.  (Word j of the final order then never leaves slot j once there: only
// smaller words could displace it, and those settle before.)  The count holds only if no
// word enters it twice, so all lanes of a pixel work on one copy of the row: lane q loads
// words q, q + lanes, ... and hands them round in LDS.  Each candidate is then in that copy
// for every lane (and dropped), or for none (and counted as a mate's); with a row read per
// lane, one could find a mate's word in the row that the mate itself had read too early to
// find.  Words that move on while the copy is made are seen once at most, since only a word
// above all before it counts.  A pixel that finds an empty row writes each word once, and
// one that finds a full row writes only what enters.  Bound by the latency of reading the
// row and of the atomics.  One thread per pixel, each candidate starting at slot 0, took
// 419 us at 2 x 256x256 pixels of 16 slots, 100 000 splats, K = 10 (now 48 us).
template <class T>
__global__ __launch_bounds__(256) void k_nearest_insert(long npix, int k, int lanes, int K, int N,
                                                        const int32_t* __restrict__ idx, const T* __restrict__ wts,
                                                        const T* __restrict__ pts, unsigned long long* rows)
{
    __shared__ unsigned long long keys[256];
    const int lane = threadIdx.x & (lanes - 1), grp = (int)threadIdx.x - lane;
    const long pix = ((long)blockIdx.x * 256 + threadIdx.x) / lanes;
    const bool in = pix < npix;                         // uniform over a pixel's lanes
    const long base = in ? pix * k : 0;
    // the first slot of largest weight; a NaN beyond slot 0 never wins, one in slot 0 stays
    T bw = T(0);
    int bs = INT_MAX;                                   // no slot yet
    if (in)
        for (int q = lane; q < k; q += lanes) {
            T w = wts[base + q];
            if (w != w) { if (q) continue; w = (T)INFINITY; }
            if (bs == INT_MAX || w > bw) { bw = w; bs = q; }
        }
    for (int m = lanes >> 1; m > 0; m >>= 1) {
        const T ow = __shfl_xor(bw, m, 64);
        const int os = __shfl_xor(bs, m, 64);
        if (os != INT_MAX && (bs == INT_MAX || ow > bw || (ow == bw && os < bs))) { bw = ow; bs = os; }
    }
    const int s = in && bs != INT_MAX ? idx[base + bs] : -1;
    const bool live = s >= 0 && s < N;
    T sx = T(0), sy = T(0), sz = T(0);
    if (live) { sx = pts[3L * s]; sy = pts[3L * s + 1]; sz = pts[3L * s + 2]; }
    unsigned long long* row = rows + (live ? (long)s * K : 0);
    for (int q0 = 0; q0 < k; q0 += lanes) {
        const int q = q0 + lane, c = live && q < k ? idx[base + q] : -1;
        unsigned long long key = kNearestEmpty;
        if (c >= 0 && c != s && c < N) {
            const float dx = (float)(sx - pts[3L * c]), dy = (float)(sy - pts[3L * c + 1]),
                        dz = (float)(sz - pts[3L * c + 2]);
            float d2 = dx * dx;
            d2 = d2 + dy * dy;
            d2 = d2 + dz * dz;
            key = ((unsigned long long)__float_as_uint(d2) << 32) | (uint32_t)c;
        }
        if (__ballot(key != kNearestEmpty) == 0ull) continue;   // the wavefront brings nothing
        int pos = 0;
        bool there = false;
        unsigned long long top = 0ull;                  // the largest word seen
        for (int j0 = 0; j0 < K; j0 += lanes) {
            const int n = min(lanes, K - j0);
            keys[threadIdx.x] = live && lane < n
                                    ? __hip_atomic_load(row + j0 + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                                    : kNearestEmpty;
            wave_order();
            for (int t = 0; t < n; t++) {
                const unsigned long long v = keys[grp + t];
                pos += v < key && (j0 + t == 0 || v > top);
                there |= v == key;
                top = v > top ? v : top;
            }
            wave_order();
        }
        if (there) key = kNearestEmpty;                 // a copy is there, or was and was moved on
        keys[threadIdx.x] = key;
        wave_order();
        bool copy = false;
        for (int t = 0; t < lanes; t++) copy |= keys[grp + t] == key && t < lane;
        if (copy) key = kNearestEmpty;                  // a pixel-mate brings it
        wave_order();
        keys[threadIdx.x] = key;
        wave_order();
        for (int t = 0; t < lanes; t++) pos += keys[grp + t] < key;
        wave_order();
        if (key == kNearestEmpty) continue;
        for (int j = pos; j < K; j++) {
            const unsigned long long old = atomicMin(row + j, key);
            if (old == key || old == kNearestEmpty) break;   // a copy already there / an empty slot filled
            if (old > key) key = old;                        // carry the displaced word on
        }
    }
}

__global__ void k_nearest_finish(long n, const unsigned long long* __restrict__ rows, int32_t* __restrict__ out)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const unsigned long long v = rows[t];
    out[t] = v == kNearestEmpty ? -1 : (int32_t)(uint32_t)(v & 0xffffffffull);
}

template <class T>
int nearest_t(int bn, int W, int H, int k, int N, int K, const int32_t* idx, const T* wts, const T* pts,
              int32_t* out, void* ws, size_t wsBytes, hipStream_t st)
{
    if (bn <= 0 || W <= 0 || H <= 0 || k <= 0 || N < 0 || K <= 0) return UDE_ERR_ARG;
    if (N == 0) return UDE_OK;
    if (wsBytes < (size_t)N * K * 8) return UDE_ERR_WORKSPACE;
    unsigned long long* rows = (unsigned long long*)ws;
    const long n = (long)N * K, npix = (long)bn * W * H;
    k_fill_u64<<<grid1(n, 256), 256, 0, st>>>(rows, n, kNearestEmpty);
    const int lanes = nearest_lanes(k);
    k_nearest_insert<T><<<grid1(npix, 256 / lanes), 256, 0, st>>>(npix, k, lanes, K, N, idx, wts, pts, rows);
    k_nearest_finish<<<grid1(n, 256), 256, 0, st>>>(n, rows, out);
    return launch_status();
}

} // namespace

extern "C" {

size_t ude_nearest_workspace_bytes(int N, int K) { return (size_t)(N > 0 ? N : 1) * (K > 0 ? K : 1) * 8 + 256; }

int ude_nearest_samples(int bn, int W, int H, int k, int N, int K, const int32_t* idx, const float* wts,
                        const float* pts, int32_t* out, void* ws, size_t wsBytes, hipStream_t st)
{
    return nearest_t<float>(bn, W, H, k, N, K, idx, wts, pts, out, ws, wsBytes, st);
}

int ude_nearest_samples_f64(int bn, int W, int H, int k, int N, int K, const int32_t* idx, const double* wts,
                            const double* pts, int32_t* out, void* ws, size_t wsBytes, hipStream_t st)
{
    return nearest_t<double>(bn, W, H, k, N, K, idx, wts, pts, out, ws, wsBytes, st);
}


int ude_pixel_scatter(int bn, int W, int H, int k, int N, int C, const int32_t* idx, const float* values,
                      float* out, hipStream_t st)
{
    return scatter_t<float>(bn, W, H, k, N, C, idx, values, out, st);
}

int ude_pixel_scatter_f64(int bn, int W, int H, int k, int N, int C, const int32_t* idx, const double* values,
                          double* out, hipStream_t st)
{
    return scatter_t<double>(bn, W, H, k, N, C, idx, values, out, st);
}

int ude_pixel_scatter_f16(int bn, int W, int H, int k, int N, int C, const int32_t* idx, const void* values,
                          void* out, hipStream_t st)
{
    return scatter_t<__half>(bn, W, H, k, N, C, idx, (const __half*)values, (__half*)out, st);
}

int ude_pixel_gather(int bn, int W, int H, int k, int N, int C, const int32_t* idx, const float* values, float* out,
                     hipStream_t st)
{
    return gather_t<float>(bn, W, H, k, N, C, idx, values, out, st);
}

int ude_pixel_gather_f64(int bn, int W, int H, int k, int N, int C, const int32_t* idx, const double* values,
                         double* out, hipStream_t st)
{
    return gather_t<double>(bn, W, H, k, N, C, idx, values, out, st);
}

} // extern "C"
