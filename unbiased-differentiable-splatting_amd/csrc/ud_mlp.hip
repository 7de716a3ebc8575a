// ud_mlp.hip -- per-tile rate network for Poisson-rate sampling (gfx950).
//
// A 32 -> 64 -> 64 -> 1 perceptron (ReLU hidden layers) maps 32 features of a
// 16x16 pixel tile to the logarithm of its sampling-rate multiplier.  Weights
// and activations enter the matrix cores as bfloat16 and accumulate in FP32
// (v_mfma_f32_16x16x16_bf16); biases, the output layer's dot product, the
// loss and the optimiser run in FP32.  Forward, backward and Adam are all
// kernels here, so the network trains on the GPU with no library GEMM.
//
// A wavefront takes 16 rows (tiles) through the whole network: the weights sit in
// LDS as bfloat16, the activations pass from one layer's accumulator layout to the
// next one's operand layout through 2 KB of LDS, and the weight gradients of all its
// rows accumulate in registers (the accumulator layout of H1 and dZ2 is the operand
// layout of H1^T dZ2).  One kernel per layer and direction took 15 launches per
// training evaluation, and its weight-gradient products walked all T rows in one
// wavefront per 16x16 weights: 1310 us at T = 20480 (now 51 us).
//
// Parameter block (FP32, 6337 floats): W1 [32][64], b1 [64], W2 [64][64],
// b2 [64], W3 [64], b3 [1] (row-major, input index first).
#include "ud_device.h"
#include "../../include/udsplat.h"

using namespace ud;

namespace {

constexpr int kIn = 32, kHid = 64;
constexpr int kOffW1 = 0, kOffB1 = kIn * kHid, kOffW2 = kOffB1 + kHid, kOffB2 = kOffW2 + kHid * kHid;
constexpr int kOffW3 = kOffB2 + kHid, kOffB3 = kOffW3 + kHid, kParams = kOffB3 + 1;

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// FP32 -> bfloat16, round to nearest even (NaN stays NaN)
__device__ __forceinline__ uint16_t f2bf(float x)
{
    uint32_t u = __float_as_uint(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

__device__ __forceinline__ float bfr(float x) { return bf2f(f2bf(x)); }

constexpr int kWaves = 4;                    // wavefronts per workgroup
constexpr int kPad1 = kIn + 4, kPad2 = kHid + 4;      // LDS row strides (8-byte fragments, spread over the banks)
constexpr int kTrainBlocks = 128;            // workgroups of the training pass (partial gradients)
constexpr int kPartial = kParams + 1;        // gradient and loss

struct Weights {
    uint16_t w1t[kHid * kPad1];              // W1 transposed: [out][in]
    uint16_t w2t[kHid * kPad2];              // W2 transposed: [out][in]
    uint16_t w2[kHid * kPad2];               // W2: [in][out]
    float b1[kHid], b2[kHid];
    __align__(16) float w3[kHid];            // rounded to bfloat16
    float b3;
};

__device__ __forceinline__ void load_weights(const float* __restrict__ P, Weights& w, bool back)
{
    for (int e = threadIdx.x; e < kIn * kHid; e += blockDim.x)
        w.w1t[(e % kHid) * kPad1 + e / kHid] = f2bf(P[kOffW1 + e]);
    for (int e = threadIdx.x; e < kHid * kHid; e += blockDim.x) {
        const uint16_t x = f2bf(P[kOffW2 + e]);
        w.w2t[(e % kHid) * kPad2 + e / kHid] = x;
        if (back) w.w2[(e / kHid) * kPad2 + e % kHid] = x;
    }
    if (threadIdx.x < kHid) {
        w.b1[threadIdx.x] = P[kOffB1 + threadIdx.x];
        w.b2[threadIdx.x] = P[kOffB2 + threadIdx.x];
        w.w3[threadIdx.x] = bfr(P[kOffW3 + threadIdx.x]);
    }
    if (threadIdx.x == 0) w.b3 = P[kOffB3];
}

__device__ __forceinline__ f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// four consecutive bfloat16 of an LDS row (8-byte aligned)
__device__ __forceinline__ bf16x4 frag(const uint16_t* p) { return *(const bf16x4*)p; }

__device__ __forceinline__ void lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// an accumulator tile set (rows 4g + v, columns 16c + r) as operand rows (row r,
// columns 16s + 4g ...), through the wavefront's 16 x kPad2 LDS buffer
__device__ __forceinline__ void to_rows(uint16_t* buf, const bf16x4 (&x)[4], bf16x4 (&out)[4], int r, int g)
{
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
        for (int v = 0; v < 4; v++) buf[(4 * g + v) * kPad2 + 16 * c + r] = (uint16_t)x[c][v];
    lds_fence();
#pragma unroll
    for (int s = 0; s < 4; s++) out[s] = frag(buf + r * kPad2 + 16 * s + 4 * g);
    lds_fence();
}

// H1, H2 (bfloat16, accumulator layout) and y (rows 4g + v, in every lane of a row
// group) of the 16 rows from t0 on; feature k is (X[k] - mean[k]) / std[k], or X[k].
// y is summed in the order of the hidden units: dZ2 = dy W3 rounds to bfloat16, where a
// last bit of y that depends on the split moves a term by 2^-9 (one of 317 x 64 changed
// the gradient by 1.7e-5).  Sixteen lanes side by side cost k_mlp_train 39 -> 42 us at T = 20480.
__device__ __forceinline__ void forward16(int T, const float* __restrict__ X, const float* __restrict__ mean,
                                          const float* __restrict__ std, long t0, const Weights& w, uint16_t* buf,
                                          int r, int g, bf16x4 (&h1)[4], bf16x4 (&h2)[4], float (&y)[4])
{
    const long row = t0 + r;
    bf16x4 a[2];
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int k = 16 * s + 4 * g + v;
            float x = row < T ? X[row * kIn + k] : 0.0f;
            if (mean) x = (x - mean[k]) / std[k];
            a[s][v] = (short)f2bf(x);
        }
#pragma unroll
    for (int c = 0; c < 4; c++) {
        f32x4 z = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
        for (int s = 0; s < 2; s++) z = mfma(a[s], frag(w.w1t + (16 * c + r) * kPad1 + 16 * s + 4 * g), z);
#pragma unroll
        for (int v = 0; v < 4; v++) h1[c][v] = (short)f2bf(fmaxf(z[v] + w.b1[16 * c + r], 0.0f));
    }
    bf16x4 rows[4];
    to_rows(buf, h1, rows, r, g);
#pragma unroll
    for (int c = 0; c < 4; c++) {
        f32x4 z = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
        for (int s = 0; s < 4; s++) z = mfma(rows[s], frag(w.w2t + (16 * c + r) * kPad2 + 16 * s + 4 * g), z);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const uint16_t h = f2bf(fmaxf(z[v] + w.b2[16 * c + r], 0.0f));
            h2[c][v] = (short)h;
            buf[(4 * g + v) * kPad2 + 16 * c + r] = h;
        }
    }
    lds_fence();
    float s = 0.0f;                          // row r
#pragma unroll
    for (int k = 0; k < kHid; k += 4) {
        const bf16x4 h = frag(buf + r * kPad2 + k);
        const f32x4 q = *(const f32x4*)(w.w3 + k);
#pragma unroll
        for (int v = 0; v < 4; v++) s = s + bf2f((uint16_t)h[v]) * q[v];
    }
    s = s + w.b3;
    lds_fence();
#pragma unroll
    for (int v = 0; v < 4; v++) y[v] = __shfl(s, 4 * g + v, 64);
}

__global__ __launch_bounds__(64 * kWaves) void k_mlp_forward(int T, const float* __restrict__ X,
                                                             const float* __restrict__ mean,
                                                             const float* __restrict__ std,
                                                             const float* __restrict__ P, float* __restrict__ y)
{
    __shared__ __align__(16) Weights w;
    __shared__ __align__(16) uint16_t buf[kWaves][16 * kPad2];
    load_weights(P, w, false);
    __syncthreads();
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    for (long t0 = ((long)blockIdx.x * kWaves + wv) * 16; t0 < T; t0 += (long)gridDim.x * kWaves * 16) {
        bf16x4 h1[4], h2[4];
        float o[4];
        forward16(T, X, mean, std, t0, w, buf[wv], r, g, h1, h2, o);
#pragma unroll
        for (int v = 0; v < 4; v++)
            if (r == v && t0 + 4 * g + v < T) y[t0 + 4 * g + v] = o[v];
    }
}

// sum of the loss weights (T without weights): 1024 strided sums, added pairwise from the
// furthest apart on (dy takes its order from here, see forward16); its inverse, 0 for no weight
__global__ __launch_bounds__(1024) void k_weight_sum(int T, const float* __restrict__ weight, float* __restrict__ inv)
{
    __shared__ float sw[1024];
    float s = 0.0f;
    for (int t = threadIdx.x; t < T; t += 1024) s = s + (weight ? weight[t] : 1.0f);
    sw[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x >= 64) return;
    float p[16];
#pragma unroll
    for (int q = 0; q < 16; q++) p[q] = sw[threadIdx.x + 64 * q];
#pragma unroll
    for (int o = 8; o > 0; o >>= 1)
#pragma unroll
        for (int q = 0; q < o; q++) p[q] = p[q] + p[q + o];
    for (int o = 32; o > 0; o >>= 1) p[0] = p[0] + __shfl_down(p[0], o, 64);
    if (threadIdx.x == 0) inv[0] = p[0] > 0.0f ? 1.0f / p[0] : 0.0f;
}

// Forward and backward of the weighted mean-square loss, dy = 2 w (y - target) / sum(w):
// the gradient and loss of this workgroup's rows to part[blockIdx.x].
__global__ __launch_bounds__(64 * kWaves) void k_mlp_train(int T, const float* __restrict__ X,
                                                           const float* __restrict__ P,
                                                           const float* __restrict__ target,
                                                           const float* __restrict__ weight,
                                                           const float* __restrict__ inv, float* __restrict__ part)
{
    // the weights, then (after the last row) the workgroup's gradient
    __shared__ __align__(16) union { Weights w; float sum[kPartial]; } u;
    __shared__ __align__(16) uint16_t buf[kWaves][16 * kPad2];
    load_weights(P, u.w, true);
    __syncthreads();
    const Weights& w = u.w;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const float iw = inv[0];
    f32x4 gW1[2][4], gW2[4][4];
    float gb1[4], gb2[4], gw3[4], gb3 = 0.0f, loss = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        gb1[c] = gb2[c] = gw3[c] = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; q++) gW2[q][c] = f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
        for (int q = 0; q < 2; q++) gW1[q][c] = f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
    }
    for (long t0 = ((long)blockIdx.x * kWaves + wv) * 16; t0 < T; t0 += (long)gridDim.x * kWaves * 16) {
        bf16x4 h1[4], h2[4], z[4], rows[4];
        float y[4], dy[4];
        forward16(T, X, nullptr, nullptr, t0, w, buf[wv], r, g, h1, h2, y);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const long t = t0 + 4 * g + v;
            const float wt = t < T ? (weight ? weight[t] : 1.0f) : 0.0f;
            const float e = t < T ? y[v] - target[t] : 0.0f;
            dy[v] = (2.0f * wt) * e * iw;
            if (r == 0) { loss += wt * (e * e); gb3 += dy[v]; }
        }
        // dZ2 = dy W3^T where H2 > 0
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float h = bf2f((uint16_t)h2[c][v]);
                const float x = h > 0.0f ? dy[v] * w.w3[16 * c + r] : 0.0f;
                gw3[c] += dy[v] * h;
                gb2[c] += x;
                z[c][v] = (short)f2bf(x);
            }
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int c = 0; c < 4; c++) gW2[q][c] = mfma(h1[q], z[c], gW2[q][c]);
        // dZ1 = dZ2 W2^T where H1 > 0
        to_rows(buf[wv], z, rows, r, g);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            f32x4 d = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
            for (int s = 0; s < 4; s++) d = mfma(rows[s], frag(w.w2 + (16 * c + r) * kPad2 + 16 * s + 4 * g), d);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float x = bf2f((uint16_t)h1[c][v]) > 0.0f ? d[v] : 0.0f;
                gb1[c] += x;
                z[c][v] = (short)f2bf(x);
            }
        }
#pragma unroll
        for (int q = 0; q < 2; q++) {
            bf16x4 xt;                                   // X^T: row 16 q + r of the features, rows 4g + v
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const long t = t0 + 4 * g + v;
                xt[v] = (short)f2bf(t < T ? X[t * kIn + 16 * q + r] : 0.0f);
            }
#pragma unroll
            for (int c = 0; c < 4; c++) gW1[q][c] = mfma(xt, z[c], gW1[q][c]);
        }
    }
    // column sums over the row groups (lanes of equal r), the loss over all lanes
#pragma unroll
    for (int c = 0; c < 4; c++)
        for (int o = 16; o < 64; o <<= 1) {
            gb1[c] += __shfl_xor(gb1[c], o, 64);
            gb2[c] += __shfl_xor(gb2[c], o, 64);
            gw3[c] += __shfl_xor(gw3[c], o, 64);
        }
    gb3 = wave_sum(gb3);
    loss = wave_sum(loss);
    __syncthreads();                                     // the weights are no longer read
    for (int q = 0; q < kWaves; q++) {                   // the wavefronts' sums, in order
        if (wv == q) {
            auto add = [&](int at, float x) { u.sum[at] = q ? u.sum[at] + x : x; };
#pragma unroll
            for (int c = 0; c < 4; c++) {
#pragma unroll
                for (int v = 0; v < 4; v++) {
#pragma unroll
                    for (int i = 0; i < 2; i++) add(kOffW1 + (16 * i + 4 * g + v) * kHid + 16 * c + r, gW1[i][c][v]);
#pragma unroll
                    for (int i = 0; i < 4; i++) add(kOffW2 + (16 * i + 4 * g + v) * kHid + 16 * c + r, gW2[i][c][v]);
                }
                if (g == 0) {
                    add(kOffB1 + 16 * c + r, gb1[c]);
                    add(kOffB2 + 16 * c + r, gb2[c]);
                    add(kOffW3 + 16 * c + r, gw3[c]);
                }
            }
            if (lane == 0) { add(kOffB3, gb3); add(kParams, loss); }
        }
        __syncthreads();
    }
    for (int e = threadIdx.x; e < kPartial; e += blockDim.x) part[(long)blockIdx.x * kPartial + e] = u.sum[e];
}

// grad = the workgroups' partial gradients added in order, loss = their losses / sum(w)
__global__ __launch_bounds__(256) void k_mlp_reduce(int blocks, const float* __restrict__ part,
                                                    const float* __restrict__ inv, float* __restrict__ grad,
                                                    float* __restrict__ loss)
{
    __shared__ float sh[4][64];
    const int e = blockIdx.x * 64 + (threadIdx.x & 63), q = threadIdx.x >> 6;
    float s = 0.0f;
    if (e < kPartial) {
#pragma unroll 8
        for (int b = q; b < blocks; b += 4) s += part[(long)b * kPartial + e];
    }
    sh[q][threadIdx.x & 63] = s;
    __syncthreads();
    if (q == 0 && e < kPartial) {
        s = ((sh[0][threadIdx.x] + sh[1][threadIdx.x]) + sh[2][threadIdx.x]) + sh[3][threadIdx.x];
        if (e < kParams) grad[e] = s;
        else if (loss) loss[0] = s * inv[0];
    }
}

// Rate multipliers from the predictions (ude_rate_scale), one workgroup: about 30
// elementwise and reduction kernels of a tensor library otherwise (8 us here at 1024
// tiles, about 100 us of launches there).
__device__ __forceinline__ double block_sum(double x, double* sh)
{
    x = wave_sum_d(x);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = x;
    __syncthreads();
    double s = sh[0];
    for (int q = 1; q < 16; q++) s += sh[q];
    __syncthreads();
    return s;
}

// a NaN stays a NaN
__device__ __forceinline__ double clamp_d(double x, double lo, double hi)
{
    x = x < lo ? lo : x;
    return x > hi ? hi : x;
}

__global__ __launch_bounds__(1024) void k_rate_scale(int T, const float* __restrict__ y, const double* __restrict__ count,
                                                     double lo, double hi, double* __restrict__ s,
                                                     float* __restrict__ out)
{
    __shared__ double sh[16];
    const double inf = __builtin_huge_val();
    auto at = [&](int t) {
        const double v = (double)y[t];
        return v != v ? 0.0 : v == inf ? 20.0 : v == -inf ? -20.0 : v;
    };
    double c = 0.0, yc = 0.0;
    for (int t = threadIdx.x; t < T; t += 1024) c += count[t];
    const double sum = block_sum(c, sh);
    const double tot = sum < 1e-30 ? 1e-30 : sum;
    for (int t = threadIdx.x; t < T; t += 1024) yc += at(t) * count[t];
    const double mean = block_sum(yc, sh) / tot;
    for (int t = threadIdx.x; t < T; t += 1024) s[t] = exp(clamp_d(at(t) - mean, -20.0, 20.0));
    for (int it = 0; it < 3; it++) {
        double a = 0.0;
        for (int t = threadIdx.x; t < T; t += 1024) a += s[t] * count[t];
        const double b = block_sum(a, sh);
        const double f = tot / (b < 1e-30 ? 1e-30 : b);
        for (int t = threadIdx.x; t < T; t += 1024) s[t] = clamp_d(s[t] * f, lo, hi);
    }
    for (int t = threadIdx.x; t < T; t += 1024) out[t] = (float)s[t];
}

// Adam (Kingma & Ba 2015) with bias correction, FP32 master parameters
__global__ __launch_bounds__(256) void k_adam(int n, float* __restrict__ p, const float* __restrict__ g,
                                              float* __restrict__ m, float* __restrict__ v, float lr, float b1,
                                              float b2, float eps, float c1, float c2)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    float gt = g[t];
    float mt = b1 * m[t] + (1.0f - b1) * gt;
    float vt = b2 * v[t] + (1.0f - b2) * (gt * gt);
    m[t] = mt;
    v[t] = vt;
    p[t] = p[t] - lr * (mt / c1) / (sqrtf(vt / c2) + eps);
}

inline size_t a256(size_t x) { return (x + 255) & ~(size_t)255; }
inline unsigned g256(long n) { return (unsigned)((n + 255) / 256); }

// workgroups for T rows, 16 per wavefront and pass
inline unsigned row_blocks(int T, unsigned most)
{
    const unsigned b = (unsigned)((T + 16 * kWaves - 1) / (16 * kWaves));
    return b < most ? b : most;
}

inline int launch_status()
{
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? UDE_OK : UDE_ERR_LAUNCH;
}

} // namespace

extern "C" {

int ude_mlp_param_count(void) { return kParams; }

// training: the inverse weight sum, the partial gradients
size_t ude_mlp_workspace_bytes(int T)
{
    return 256 + a256(sizeof(float) * (size_t)kPartial * row_blocks(T > 0 ? T : 1, kTrainBlocks)) + 256;
}

int ude_mlp_forward(int T, const float* X, const float* params, float* y, void* ws, size_t wsBytes, hipStream_t st)
{
    if (T <= 0) return UDE_OK;
    if (wsBytes < ude_mlp_workspace_bytes(T)) return UDE_ERR_WORKSPACE;
    k_mlp_forward<<<row_blocks(T, 1024), 64 * kWaves, 0, st>>>(T, X, nullptr, nullptr, params, y);
    return launch_status();
}

int ude_mlp_loss_grad(int T, const float* X, const float* params, const float* target, const float* weight,
                      float* grad, float* loss, void* ws, size_t wsBytes, hipStream_t st)
{
    if (T <= 0) return UDE_ERR_ARG;
    if (wsBytes < ude_mlp_workspace_bytes(T)) return UDE_ERR_WORKSPACE;
    float* inv = (float*)ws;
    float* part = (float*)((char*)ws + 256);
    const unsigned blocks = row_blocks(T, kTrainBlocks);
    k_weight_sum<<<1, 1024, 0, st>>>(T, weight, inv);
    k_mlp_train<<<blocks, 64 * kWaves, 0, st>>>(T, X, params, target, weight, inv, part);
    k_mlp_reduce<<<(kPartial + 63) / 64, 256, 0, st>>>((int)blocks, part, inv, grad, loss);
    return launch_status();
}

size_t ude_rate_scale_workspace_bytes(int T) { return 12 * (size_t)(T > 0 ? T : 0) + 512; }

int ude_rate_scale(int T, const float* feats, const float* mean, const float* std, const float* params,
                   const double* counts, double lo, double hi, float* out, void* ws, size_t wsBytes, hipStream_t st)
{
    if (T < 0 || !mean || !std) return UDE_ERR_ARG;
    if (T == 0) return UDE_OK;
    if (wsBytes < ude_rate_scale_workspace_bytes(T)) return UDE_ERR_WORKSPACE;
    double* s = (double*)ws;
    float* y = (float*)(s + T);
    k_mlp_forward<<<row_blocks(T, 1024), 64 * kWaves, 0, st>>>(T, feats, mean, std, params, y);
    k_rate_scale<<<1, 1024, 0, st>>>(T, y, counts, lo, hi, s, out);
    return launch_status();
}

int ude_adam_step(int n, float* params, const float* grad, float* m, float* v, float lr, float beta1, float beta2,
                  float eps, int step, hipStream_t st)
{
    if (n <= 0 || step <= 0) return UDE_ERR_ARG;
    float c1 = 1.0f - powf(beta1, (float)step), c2 = 1.0f - powf(beta2, (float)step);
    k_adam<<<g256(n), 256, 0, st>>>(n, params, grad, m, v, lr, beta1, beta2, eps, c1, c2);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? UDE_OK : UDE_ERR_LAUNCH;
}

} // extern "C"
