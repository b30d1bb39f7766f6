// Learned edge prior: features, MLP forward / backward on the matrix cores,
// Adam, minibatch training and the dense prior for aco_problem.prior.
//
// No counterpart in the reference (its eta is 1/(d+0.1)^beta from the
// distance alone, kernel.cl:672-679,782-789).
//
// MLP 12 -> 64 -> 64 -> 1 with ReLU.  BF16 operands, FP32 accumulation on
// the matrix cores.  One wave processes 16 edges per tile with the edges on
// the N dimension of every product: the accumulator layout of one layer
// (lane l holds rows 4*(l/16)+j, column l%16) is exactly the B-operand
// layout of the next, so the forward pass needs no data movement between
// layers.  The weight gradients contract over edges, which needs the
// transposed layout: 16x16 tiles go through a per-wave LDS buffer.
//
// Layer 1 (K = 12 features, padded to 16) and the weight gradients (K = the
// 16 edges of a tile) use v_mfma_f32_16x16x16_bf16.  The 64-deep products
// (layer 2 and dH1 = W2^T dz2) use gfx950's v_mfma_f32_16x16x32_bf16, two
// per 16-row block: its A and B operands are two 4-element halves put side
// by side, each half one 16-deep slice in the layout above.  Element i of a
// lane's A operand and element i of its B operand carry the same index of
// the contraction, so the product sums exactly the slices' terms, whatever
// order the unit adds them in.
//
// Determinism: a partial row of the gradient holds four consecutive tiles,
// added one after another, and the reduce kernel sums the rows in a fixed
// order (runs of consecutive rows, then the runs); there are no atomics.

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>
#include <vector>

#include "aco_internal.h"
#include "cvrp_aco.h"
#include "cvrp_prior.h"

namespace cvrp {
namespace prior {

constexpr int NF = 12, NFP = 16, H = 64;
constexpr int OFF_W1 = 0, OFF_B1 = H * NF, OFF_W2 = OFF_B1 + H, OFF_B2 = OFF_W2 + H * H,
              OFF_W3 = OFF_B2 + H, OFF_B3 = OFF_W3 + H, NP = OFF_B3 + 1;
static_assert(NP == ACO_PRIOR_PARAMS, "parameter layout");
constexpr int NPL = NP + 1;         // partial row: gradient, then the loss sum
constexpr int kThreads = 256, kWaves = kThreads / 64;
constexpr int kMaxBatch = 65536;

typedef short v4s __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

__host__ __device__ inline unsigned short f2bf(float f)
{
    // round to nearest even (finite inputs)
    unsigned u;
    memcpy(&u, &f, 4);
    u = u + 0x7FFFu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

__device__ __forceinline__ float bf2f(unsigned short b) { return __uint_as_float((unsigned)b << 16); }

__device__ __forceinline__ v4s ld4(const unsigned short *p) { return *reinterpret_cast<const v4s *>(p); }

__device__ __forceinline__ v4f mfma(v4s a, v4s b, v4f c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// c + [a0 a1] x [b0; b1]: two 16-deep slices in one 32-deep product.
__device__ __forceinline__ v4f mfma2(v4s a0, v4s a1, v4s b0, v4s b1, v4f c)
{
    const v8s a = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
    const v8s b = {b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]};
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c,
                                                    0, 0, 0);
}

// Block-resident network: bf16 weights (W2 also transposed, for dH1),
// fp32 biases, w3 rounded to bf16 and widened.
struct NetLds {
    alignas(16) unsigned short w1[H][NFP];
    alignas(16) unsigned short w2[H][H];
    alignas(16) unsigned short w2t[H][H];
    alignas(16) float b1[H];
    alignas(16) float b2[H];
    alignas(16) float w3[H];
    float b3;
};

// Every global read is requested before the first LDS write (8 or 16 bytes
// each): an element at a time, a block waited for twenty of them in turn.
__device__ void load_net(NetLds &S, const unsigned short *wb, const float *pf)
{
    typedef unsigned short v8u __attribute__((ext_vector_type(8)));
    static_assert(H == 64 && NF == 12 && NFP == 16 && kThreads == 256, "one pass of the block");
    static_assert(OFF_W1 % 8 == 0 && OFF_W2 % 8 == 0, "aligned vector reads");
    const int t = threadIdx.x;
    const v8u *w2 = reinterpret_cast<const v8u *>(wb + OFF_W2);
    const v8u a0 = w2[t], a1 = w2[t + kThreads];
    const v4s c = reinterpret_cast<const v4s *>(wb + OFF_W1)[t < H * NF / 4 ? t : 0];
    const int q = t & (H - 1), part = t / H;
    const float b = part < 2 ? pf[(part == 0 ? OFF_B1 : OFF_B2) + q] : 0.0f;
    const unsigned short w3 = wb[OFF_W3 + q];
    const float b3 = pf[OFF_B3];
    auto put = [&](int e, v8u a) {   // elements 8e .. 8e + 7
        const int o = e / (H / 8), i0 = 8 * (e % (H / 8));
        *reinterpret_cast<v8u *>(&S.w2[o][i0]) = a;
#pragma unroll
        for (int k = 0; k < 8; ++k) S.w2t[i0 + k][o] = a[k];
    };
    put(t, a0);
    put(t + kThreads, a1);
    if (t < H * NF / 4) *reinterpret_cast<v4s *>(&S.w1[t / 3][4 * (t % 3)]) = c;
    if (part == 0) S.b1[q] = b;
    else if (part == 1) S.b2[q] = b;
    else if (part == 2) S.w3[q] = bf2f(w3);
    else *reinterpret_cast<v4s *>(&S.w1[q][NF]) = v4s{0, 0, 0, 0};
    if (t == 0) S.b3 = b3;
    __syncthreads();
}

struct Fwd {
    v4f z1[4];
    v4s h1[4];
    v4f z2[4];
    float z;
};

// The weights one lane feeds to the matrix cores (row r = l%16, slice
// g = l/16 of every 16-deep operand), read from the block's LDS copy at
// each use ...
struct LdsWeights {
    const NetLds &S;
    int r, g;
    __device__ v4s w1(int t) const { return ld4(&S.w1[16 * t + r][4 * g]); }
    __device__ v4s w2(int mt, int kt) const { return ld4(&S.w2[16 * mt + r][16 * kt + 4 * g]); }
    __device__ v4f b1(int t) const { return *reinterpret_cast<const v4f *>(&S.b1[16 * t + 4 * g]); }
    __device__ v4f b2(int mt) const { return *reinterpret_cast<const v4f *>(&S.b2[16 * mt + 4 * g]); }
    __device__ float w3(int mt, int j) const { return S.w3[16 * mt + 4 * g + j]; }
    __device__ float b3() const { return S.b3; }
};

// ... or from the parameter buffers in global memory (bf16 weights, W1
// rows of 12 features zero-padded to 16 here; fp32 biases; w3 widened from
// its bf16 copy) ...
struct GlobalWeights {
    const unsigned short *wb;
    const float *pf;
    int r, g;
    __device__ v4s w1(int t) const
    {
        if (g * 4 >= NF) return v4s{0, 0, 0, 0};
        return ld4(wb + OFF_W1 + (16 * t + r) * NF + 4 * g);
    }
    __device__ v4s w2(int mt, int kt) const { return ld4(wb + OFF_W2 + (16 * mt + r) * H + 16 * kt + 4 * g); }
    __device__ v4f b1(int t) const { return *reinterpret_cast<const v4f *>(pf + OFF_B1 + 16 * t + 4 * g); }
    __device__ v4f b2(int mt) const { return *reinterpret_cast<const v4f *>(pf + OFF_B2 + 16 * mt + 4 * g); }
    __device__ float w3(int mt, int j) const { return bf2f(wb[OFF_W3 + 16 * mt + 4 * g + j]); }
    __device__ float b3() const { return pf[OFF_B3]; }
};

// ... or held in registers for a whole loop over tiles (about 90 VGPRs: the
// inference kernel, whose waves run many tiles each).
struct RegWeights {
    v4s w1_[4], w2_[4][4];
    v4f b1_[4], b2_[4];
    float w3_[16], b3_;
    template <typename Src>
    __device__ explicit RegWeights(const Src &L)
    {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            w1_[t] = L.w1(t);
            b1_[t] = L.b1(t);
            b2_[t] = L.b2(t);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                w2_[t][k] = L.w2(t, k);
                w3_[4 * t + k] = L.w3(t, k);
            }
        }
        b3_ = L.b3();
    }
    __device__ v4s w1(int t) const { return w1_[t]; }
    __device__ v4s w2(int mt, int kt) const { return w2_[mt][kt]; }
    __device__ v4f b1(int t) const { return b1_[t]; }
    __device__ v4f b2(int mt) const { return b2_[mt]; }
    __device__ float w3(int mt, int j) const { return w3_[4 * mt + j]; }
    __device__ float b3() const { return b3_; }
};

// x: B operand of layer 1 (lane: features 4*(l/16)+j of edge l%16).
template <typename Wt>
__device__ __forceinline__ void fwd_tile(const Wt &W, v4s x, Fwd &F)
{
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        F.z1[t] = mfma(W.w1(t), x, W.b1(t));
        v4s h;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float z = F.z1[t][j];
            h[j] = (short)f2bf(z > 0.0f ? z : 0.0f);
        }
        F.h1[t] = h;
    }
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
        v4f c = mfma2(W.w2(mt, 0), W.w2(mt, 1), F.h1[0], F.h1[1], W.b2(mt));
        F.z2[mt] = mfma2(W.w2(mt, 2), W.w2(mt, 3), F.h1[2], F.h1[3], c);
    }
    float s = 0.0f;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float h = F.z2[mt][j] > 0.0f ? F.z2[mt][j] : 0.0f;
            s += W.w3(mt, j) * h;
        }
    s += __shfl_xor(s, 16);
    s += __shfl_xor(s, 32);
    F.z = s + W.b3();
}

// Accumulator-layout tile (rows 4g+j, column r) -> LDS ...
__device__ __forceinline__ void put_tile(unsigned short (*T)[16], v4s d, int lane)
{
    const int r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) T[4 * g + j][r] = (unsigned short)d[j];
}

// ... read back as the operand of a product contracting over the former
// columns: lane gets row r, columns 4g..4g+3.
__device__ __forceinline__ v4s take_tile(unsigned short (*T)[16], int lane)
{
    return ld4(&T[lane & 15][4 * (lane >> 4)]);
}

__device__ __forceinline__ v4s pack_bf16(v4f v)
{
    v4s h;
#pragma unroll
    for (int j = 0; j < 4; ++j) h[j] = (short)f2bf(v[j]);
    return h;
}

__device__ __forceinline__ v4s load_x(const unsigned short *xb, long long e, bool valid, int g)
{
    if (!valid) return v4s{0, 0, 0, 0};
    return ld4(xb + (size_t)e * NFP + 4 * g);
}

// ---------------------------------------------------------------- kernels --

// Inference: each wave takes tiles tile, tile + waves, ... with its weight
// fragments in registers (read once from global memory: no LDS, no block
// barrier) and the next tile's features requested before the current
// tile's products.
__global__ __launch_bounds__(kThreads) void k_forward(const unsigned short *xb, long long E,
                                                      const unsigned short *wb, const float *pf,
                                                      float *logits)
{
    const int lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
    const long long tiles = (E + 15) / 16;
    const long long waves = (long long)gridDim.x * kWaves;
    long long tile = (long long)blockIdx.x * kWaves + (threadIdx.x >> 6);
    if (tile >= tiles) return;   // wave-uniform
    const RegWeights W(GlobalWeights{wb, pf, r, g});
    v4s x = load_x(xb, tile * 16 + r, tile * 16 + r < E, g);
    for (; tile < tiles; tile += waves) {
        const long long e = tile * 16 + r;
        const long long en = (tile + waves) * 16 + r;
        const v4s xn = load_x(xb, en, en < E, g);
        Fwd F;
        fwd_tile(W, x, F);
        if (g == 0 && e < E) logits[e] = F.z;
        x = xn;
    }
}

// Fused forward + backward (positions [0, Eb) of idx, or of the data in order
// without one).  Four tiles of 16 edges make one partial row: their products
// are accumulated tile after tile, which fixes the order of every sum, but
// the chain of a tile up to that point is the launch's length, so each wave
// of a block runs it for one of the four.  The tiles' operands (bf16) and
// bias terms (fp32) pass through LDS; then wave w accumulates rows 16w ..
// 16w+15 of both weight gradients, and the bias terms of the same rows, over
// the four tiles in order.  A CU holds one block (LDS), and one that takes
// every kTrainBlocks-th group reads the network once.  With a wave for all
// four tiles of a row 16384 edges took 35.7 us on 64 of the CUs, now 13.7 us on
// all (1024 edges 32.0, 11.3; 65536, where every CU is busy either way, 43.9,
// 42.5).
struct TrainLds {
    alignas(16) unsigned short tr[kWaves][13][16][16];   // dz2, h1, x, dz1 of a wave's tile
    alignas(16) float terms[3][4][kWaves][64][4];        // of b1, b2, w3: row block, tile, lane
    float out[2][kWaves][16];                            // of b3 and the loss
};
constexpr int kTrainBlocks = 256;   // one per CU
static int train_rows(int Eb) { return (Eb + 16 * kWaves - 1) / (16 * kWaves); }

__global__ __launch_bounds__(kThreads) void k_train(const unsigned short *xb, const float *label,
                                                    const int *idx, int Eb,
                                                    const unsigned short *wb, const float *pf,
                                                    float pos_weight, float invE, float *partials)
{
    __shared__ NetLds S;
    __shared__ TrainLds B;
    load_net(S, wb, pf);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, r = lane & 15;
    const int tiles = (Eb + 15) / 16, groups = (tiles + kWaves - 1) / kWaves;
    const v4f zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int group = blockIdx.x; group < groups; group += gridDim.x) {
        const int tile = group * kWaves + w, count = min(kWaves, tiles - group * kWaves);
        if (w < count) {
            unsigned short(*T)[16][16] = B.tr[w];
            const int pos = tile * 16 + r;
            const bool valid = pos < Eb;
            const int e = !valid ? 0 : idx ? idx[pos] : pos;
            const v4s x = load_x(xb, e, valid, g);
            const float y = valid ? label[e] : 0.0f;
            Fwd F;
            fwd_tile(LdsWeights{S, r, g}, x, F);
            const float we = valid ? (y > 0.5f ? pos_weight : 1.0f) : 0.0f;
            const float sig = 1.0f / (1.0f + expf(-F.z));
            const float ge = we * (sig - y) * invE;
            if (g == 0) {
                B.out[0][w][r] = valid ? ge : 0.0f;
                B.out[1][w][r] =
                    valid ? we * ((fmaxf(F.z, 0.0f) - y * F.z) + log1pf(expf(-fabsf(F.z)))) : 0.0f;
            }
            put_tile(T[8], x, lane);
            // layer 3 and the ReLU of layer 2
            v4s dz2b[4];
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) {
                v4f d, d3;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const bool on = F.z2[mt][j] > 0.0f;
                    d3[j] = ge * (on ? F.z2[mt][j] : 0.0f);
                    d[j] = on ? S.w3[16 * mt + 4 * g + j] * ge : 0.0f;
                }
                *reinterpret_cast<v4f *>(B.terms[1][mt][w][lane]) = d;
                *reinterpret_cast<v4f *>(B.terms[2][mt][w][lane]) = d3;
                dz2b[mt] = pack_bf16(d);
                put_tile(T[mt], dz2b[mt], lane);
                put_tile(T[4 + mt], F.h1[mt], lane);
            }
            // dH1 = W2^T dz2 (dz2 is already the B operand), ReLU of layer 1
#pragma unroll
            for (int it = 0; it < 4; ++it) {
                v4f c = mfma2(ld4(&S.w2t[16 * it + r][4 * g]), ld4(&S.w2t[16 * it + r][16 + 4 * g]), dz2b[0],
                              dz2b[1], zero4);
                c = mfma2(ld4(&S.w2t[16 * it + r][32 + 4 * g]), ld4(&S.w2t[16 * it + r][48 + 4 * g]), dz2b[2],
                          dz2b[3], c);
                v4f d;
#pragma unroll
                for (int j = 0; j < 4; ++j) d[j] = F.z1[it][j] > 0.0f ? c[j] : 0.0f;
                *reinterpret_cast<v4f *>(B.terms[0][it][w][lane]) = d;
                put_tile(T[9 + it], pack_bf16(d), lane);
            }
        }
        __syncthreads();
        // weight gradients contract over the 16 edges of each tile
        v4f dW2[4], dW1 = zero4, db[3];
#pragma unroll
        for (int it = 0; it < 4; ++it) dW2[it] = zero4;
#pragma unroll
        for (int q = 0; q < 3; ++q) db[q] = zero4;
        float o0 = 0.0f, o1 = 0.0f;
#pragma unroll
        for (int t = 0; t < kWaves; ++t) {
            if (t >= count) break;
            unsigned short(*T)[16][16] = B.tr[t];
            const v4s aT = take_tile(T[w], lane);
#pragma unroll
            for (int it = 0; it < 4; ++it) dW2[it] = mfma(aT, take_tile(T[4 + it], lane), dW2[it]);
            dW1 = mfma(take_tile(T[9 + w], lane), take_tile(T[8], lane), dW1);
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const v4f d = *reinterpret_cast<const v4f *>(B.terms[q][w][t][lane]);
#pragma unroll
                for (int j = 0; j < 4; ++j) db[q][j] += d[j];
            }
            o0 += B.out[0][t][r];
            o1 += B.out[1][t][r];
        }
        float *P = partials + (size_t)group * NPL;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = 16 * w + 4 * g + j;
#pragma unroll
            for (int it = 0; it < 4; ++it) P[OFF_W2 + row * H + 16 * it + r] = dW2[it][j];
            if (r < NF) P[OFF_W1 + row * NF + r] = dW1[j];
            // bias / w3 gradients: sum over the 16 edge lanes of each row group
#pragma unroll
            for (int q = 0; q < 3; ++q)
#pragma unroll
                for (int o = 1; o < 16; o <<= 1) db[q][j] += __shfl_xor(db[q][j], o);
            if (r == 0) {
                P[OFF_B1 + row] = db[0][j];
                P[OFF_B2 + row] = db[1][j];
                P[OFF_W3 + row] = db[2][j];
            }
        }
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
            o0 += __shfl_xor(o0, o);
            o1 += __shfl_xor(o1, o);
        }
        if (threadIdx.x == 0) {
            P[OFF_B3] = o0;
            P[NP] = o1 * invE;
        }
        if (group + (int)gridDim.x < groups) __syncthreads();   // the buffers are read
    }
}

// Per parameter: the sum of the partial rows in a fixed order (runs of
// consecutive rows, then the runs in order), then (update != 0) Adam in
// fp32.  Parameter NP is the loss.
struct AdamArgs {
    float lr, beta1, om_beta1, beta2, om_beta2, c1, c2, eps;
};

// A block takes kReduceParams parameters; each is summed by kReduceGroups
// threads over consecutive runs of the partial rows, then the runs' sums are
// added in run order (a fixed order: runs are deterministic).
// Sixteen rows are requested together (same order of additions): 256 rows
// 10.0 -> 4.0 us, 1024 rows 37.7 -> 7.3, which was bound by one row's latency
// after another.
constexpr int kReduceParams = 32, kReduceGroups = 8;
// Rows per run for a batch: its partial rows rounded up to fours.
static int train_run(int rows) { return ((rows + kWaves - 1) / kWaves * kWaves + kReduceGroups - 1) / kReduceGroups; }

__global__ __launch_bounds__(kReduceParams * kReduceGroups) void k_reduce_adam(
    const float *partials, int W, int run, float *pf, float *m, float *v, unsigned short *wb, float *grad_out,
    float *loss_out, int update, AdamArgs a)
{
    __shared__ float red[kReduceGroups][kReduceParams];
    const int i = threadIdx.x % kReduceParams, q = threadIdx.x / kReduceParams;
    const int p = blockIdx.x * kReduceParams + i;
    const int w0 = q * run, w1 = min(W, w0 + run);
    float part = 0.0f;
    if (p <= NP)
#pragma unroll 16
        for (int w = w0; w < w1; ++w) part += partials[(size_t)w * NPL + p];
    red[q][i] = part;
    __syncthreads();
    if (q != 0 || p > NP) return;
    float s = red[0][i];
    for (int g = 1; g < kReduceGroups && g * run < W; ++g) s += red[g][i];
    if (p == NP) {
        if (loss_out) *loss_out = s;
        return;
    }
    if (grad_out) grad_out[p] = s;
    if (!update) return;
    const float mm = a.beta1 * m[p] + a.om_beta1 * s;
    const float vv = a.beta2 * v[p] + a.om_beta2 * (s * s);
    const float mh = mm / a.c1, vh = vv / a.c2;
    const float np = pf[p] - a.lr * (mh / (sqrtf(vh) + a.eps));
    m[p] = mm;
    v[p] = vv;
    pf[p] = np;
    wb[p] = f2bf(np);
}

__global__ void k_to_bf16(const float *pf, unsigned short *wb, int count)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < count) wb[p] = f2bf(pf[p]);
}

// Features -> bf16 rows of 16 (features 12..15 zero), labels copied along:
// four threads per edge, 16 bytes each.  The inputs may lie in pinned host
// memory (read once, in order, over the link).
__global__ void k_pack_features(const float *feat, const float *label, long long E, unsigned short *xb, float *lab)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long e = t >> 2;
    const int q = (int)(t & 3);
    if (e >= E) return;
    ushort4 o = {0, 0, 0, 0};
    if (q < 3) {
        const float4 f = *reinterpret_cast<const float4 *>(feat + e * NF + 4 * q);
        o = ushort4{f2bf(f.x), f2bf(f.y), f2bf(f.z), f2bf(f.w)};
    } else if (label) {
        lab[e] = label[e];
    }
    *reinterpret_cast<ushort4 *>(xb + e * NFP + 4 * q) = o;
}

// Distances of one instance: the whole matrix with row pitch P (>= n), or
// its depot row and candidate edges only.
struct DistMatrix {
    const float *d;
    int P;
    __device__ __forceinline__ float edge(int i, int, int j) const { return d[(size_t)i * P + j]; }
    __device__ __forceinline__ float depot(int i) const { return d[i]; }
};
struct DistEdges {
    const float *d0, *e;   // n, n x k
    int k;
    __device__ __forceinline__ float edge(int i, int r, int) const { return e[(size_t)i * k + r]; }
    __device__ __forceinline__ float depot(int i) const { return d0[i]; }
};

template <class D>
__global__ void k_node_stats(int n, const float *x, const float *y, D dist,
                             const int *nn, int nnw, int k, float *rad, float *ang, float *kd)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    const float dx = x[v] - x[0], dy = y[v] - y[0];
    rad[v] = sqrtf(dx * dx + dy * dy);
    ang[v] = atan2f(dy, dx) / 3.14159265358979323846f;
    kd[v] = dist.edge(v, k - 1, nn[(size_t)v * nnw + k - 1]);
}

// One block: R = max radius (1 if 0), mkd = mean k-th candidate distance
// (summed in double, 1 if 0).
__global__ void k_node_reduce(int n, const float *rad, const float *kd, float *out)
{
    __shared__ double s[256];
    __shared__ float mx[256];
    const int t = threadIdx.x;
    double a = 0.0;
    float m = 0.0f;
    for (int v = t; v < n; v += 256) {
        a += (double)kd[v];
        m = fmaxf(m, rad[v]);
    }
    s[t] = a;
    mx[t] = m;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (t < o) {
            s[t] += s[t + o];
            mx[t] = fmaxf(mx[t], mx[t + o]);
        }
        __syncthreads();
    }
    if (t == 0) {
        const float R = mx[0] > 0.0f ? mx[0] : 1.0f;
        const float mkd = (float)(s[0] / (double)n);
        out[0] = R;
        out[1] = mkd > 0.0f ? mkd : 1.0f;
    }
}

template <class D>
__global__ void k_edge_features(int n, int k, D dist, const int *nn, int nnw,
                                const int *dem, float Q, const float *rad, const float *ang,
                                const float *kd, const float *Rm, float *feat, unsigned short *xb)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)n * k) return;
    const int i = (int)(t / k), r = (int)(t % k);
    const int j = nn[(size_t)i * nnw + r];
    const float R = Rm[0], mkd = Rm[1];
    const float dij = dist.edge(i, r, j);
    float f[NF];
    f[0] = dij / mkd;
    f[1] = (float)r / (float)k;
    f[2] = (float)dem[i] / Q;
    f[3] = (float)dem[j] / Q;
    f[4] = ang[i];
    f[5] = ang[j];
    f[6] = rad[i] / R;
    f[7] = rad[j] / R;
    f[8] = kd[i] / mkd;
    f[9] = kd[j] / mkd;
    f[10] = ((dist.depot(i) + dist.depot(j)) - dij) / R;
    bool mutual = false;
    for (int q = 0; q < k; ++q) mutual |= nn[(size_t)j * nnw + q] == i;
    f[11] = mutual ? 1.0f : 0.0f;
    if (feat)
        for (int q = 0; q < NF; ++q) feat[t * NF + q] = f[q];
    if (xb)
        for (int q = 0; q < NFP; ++q) xb[t * NFP + q] = q < NF ? f2bf(f[q]) : (unsigned short)0;
}

__device__ __forceinline__ float prior_pow(float p, float ex)
{
    if (ex == 1.0f) return p;
    if (ex == 2.0f) return p * p;
    return powf(p, ex);
}

__global__ void k_prior_fill(long long cnt, float val, float *out)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < cnt) out[t] = val;
}

__global__ void k_prior_scatter(int n, int k, const int *nn, int nnw, const float *logits, float ex,
                                float *out)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)n * k) return;
    const int i = (int)(t / k), r = (int)(t % k);
    const int j = nn[(size_t)i * nnw + r];
    const float p = 1.0f / (1.0f + expf(-logits[t]));
    out[(size_t)i * n + j] = prior_pow(p, ex);
}

// Rows row0 .. row0 + gridDim.x of the dense multiplier, one block each,
// written once and in order (out may be pinned host memory): `val` except at
// the row's candidates.  LDS: n floats where they fit (staged), otherwise
// the candidates are written after the fill.
template <bool STAGED>
__global__ __launch_bounds__(256) void k_prior_rows(int n, int row0, int k, const int *nn, int nnw, const float *logits,
                                                    float ex, float val, float *out)
{
    extern __shared__ float row[];
    const int i = row0 + blockIdx.x;
    float *o = out + (size_t)blockIdx.x * n, *w = STAGED ? row : o;
    for (int j = threadIdx.x; j < n; j += 256) w[j] = val;
    if (!STAGED) __threadfence_system();   // another thread writes the candidate's entry again
    __syncthreads();
    for (int r = threadIdx.x; r < k; r += 256) {
        const float p = 1.0f / (1.0f + expf(-logits[(size_t)i * k + r]));
        w[nn[(size_t)i * nnw + r]] = prior_pow(p, ex);
    }
    if (!STAGED) return;
    __syncthreads();
    for (int j = threadIdx.x; j < n; j += 256) o[j] = row[j];
}
constexpr int kPriorRowLds = 4096;   // floats: 16 KB, several rows per CU

// Fisher-Yates swap targets of draws draw0 .. draw0 + count of a SplitMix64
// stream: draw d swaps index i = last - (d - draw0) with out = x % (i + 1).
__global__ void k_swap_targets(unsigned long long seed, unsigned long long draw0, int last, int count, int *out)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count) return;
    unsigned long long z = seed + 0x9E3779B97F4A7C15ull * (draw0 + (unsigned long long)t + 1ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    out[t] = (int)(z % (unsigned long long)(last - t + 1));
}

// heur[i][j] (pitch P) *= prior[i][j] (pitch n), j < n
__global__ void k_heur_mul(int n, int P, const float *prior, float *heur)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)n * n) return;
    const int i = (int)(t / n), j = (int)(t % n);
    const size_t e = (size_t)i * P + j;
    heur[e] = heur[e] * prior[t];
}

// ------------------------------------------------------------------- host --

struct DevBuf {
    void *p = nullptr;
    ~DevBuf() { if (p) (void)hipFree(p); }
    template <class T> T *as() const { return static_cast<T *>(p); }
};

static hipError_t dalloc(DevBuf &b, size_t bytes)
{
    return hipMalloc(&b.p, bytes ? bytes : 16);
}

}  // namespace prior
}  // namespace cvrp

using namespace cvrp;
using namespace cvrp::prior;

// Working memory of a network's calls, kept between them (one call at a
// time): one device allocation, given back after a call that needed more
// than kKeep, and one pinned one: one or two parts for inputs, then results.
// Pageable copies of this size cost 25 to 60 us each whatever they hold,
// allocations of 2 MB and more 25 us; a gradient made six of the first and two
// of the second.  Gradient over 16384 edges 202 -> 75 us, multiplier of 501
// nodes 200 -> 115 us, eight training steps of 16384 edges 932 -> 500 us; what
// is left is the copy into the buffers, the launches and the kernels (25 us
// of the gradient).
// Parts are as large as the largest call so far needs, up to kPart, and a call
// that fits one makes one: a network that is made, used once and dropped pays
// for pinning, 25 us a block with its end while the runtime has a freed one
// and 100 to 300 us and more when not.  A part is a chunk of the pipeline and
// each costs about 15 us: with parts of 256, 128 and 64 KB the gradient of
// 65536 edges takes 229, 328 and 499 us, with 512 KB 194 us.
struct PriorSpace {
    static constexpr size_t kPart = size_t(512) << 10, kLeast = size_t(32) << 10, kKeep = size_t(64) << 20;
    std::mutex mutex;
    unsigned char *dev = nullptr;
    size_t dev_bytes = 0;
    unsigned char *pin = nullptr;
    size_t part = 0, results = 0;   // bytes of a part, and behind the parts
    int parts = 0;
    hipEvent_t done[2] = {nullptr, nullptr};
    bool busy[2] = {false, false};
    int cur = 0;
    hipStream_t side = nullptr;   // swap targets, beside the training stream

    hipError_t init(size_t bytes)
    {
        if (bytes <= dev_bytes) return hipSuccess;
        release();
        const hipError_t e = hipMalloc((void **)&dev, bytes);
        if (e == hipSuccess) dev_bytes = bytes;
        return e;
    }
    // for a call that moves `bytes` through the parts, rows of `row` bytes
    // whole, and takes `res` bytes of results; nothing is in use yet
    hipError_t pinned(size_t bytes, size_t row, size_t res)
    {
        size_t want = std::max(part, kLeast);
        while ((want < bytes && want < kPart) || want < row) want *= 2;
        const int count = std::max(parts, bytes > want ? 2 : 1);
        if (want == part && count == parts && res <= results) return hipSuccess;
        res = std::max(res, results);
        unpin();
        const hipError_t e = hipHostMalloc((void **)&pin, want * count + res, hipHostMallocDefault);
        if (e != hipSuccess) return e;
        part = want;
        parts = count;
        results = res;
        return hipSuccess;
    }
    unsigned char *result() const { return pin + part * parts; }
    void unpin()
    {
        if (pin) (void)hipHostFree(pin);
        pin = nullptr;
        part = results = 0;
        parts = 0;
    }
    void release()
    {
        if (dev) (void)hipFree(dev);
        dev = nullptr;
        dev_bytes = 0;
    }
    ~PriorSpace()
    {
        release();
        unpin();
        for (hipEvent_t e : done)
            if (e) (void)hipEventDestroy(e);
        if (side) (void)hipStreamDestroy(side);
    }
    // input part to fill next, once its last reader on the device is done
    hipError_t take(unsigned char *&p)
    {
        hipError_t e = hipSuccess;
        if (!done[cur]) e = hipEventCreateWithFlags(&done[cur], hipEventDisableTiming);
        if (e == hipSuccess && busy[cur]) e = hipEventSynchronize(done[cur]);
        busy[cur] = false;
        p = pin + cur * part;
        return e;
    }
    hipError_t used(hipStream_t st)
    {
        const hipError_t e = hipEventRecord(done[cur], st);
        busy[cur] = true;
        cur = parts - 1 - cur;
        return e;
    }
};

// One call's use of a PriorSpace: pieces of the device allocation, and at the
// end nothing of the call in flight.
struct SpaceUse {
    PriorSpace &s;
    hipStream_t st;
    std::lock_guard<std::mutex> lock;
    size_t off = 0;
    SpaceUse(PriorSpace &sp, hipStream_t stream) : s(sp), st(stream), lock(sp.mutex) {}
    ~SpaceUse()
    {
        (void)hipStreamSynchronize(st);
        if (s.side) (void)hipStreamSynchronize(s.side);
        s.busy[0] = s.busy[1] = false;
        s.cur = 0;
        if (s.dev_bytes > PriorSpace::kKeep) s.release();
    }
    static size_t round(size_t bytes) { return (bytes + 255) & ~size_t(255); }
    template <class T> T *take(size_t count)
    {
        T *p = reinterpret_cast<T *>(s.dev + off);
        off += round(count * sizeof(T));
        return p;
    }
};

struct aco_prior {
    hipStream_t stream = nullptr;
    PriorSpace space;
    float *pf = nullptr, *m = nullptr, *v = nullptr;
    unsigned short *wb = nullptr;
    int step = 0;
};

#define PCHK(expr)                                                                               \
    do {                                                                                         \
        hipError_t e_ = (expr);                                                                  \
        if (e_ != hipSuccess)                                                                    \
            return set_error(ACO_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));   \
    } while (0)

static uint64_t mix64(uint64_t z)
{
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// SplitMix64 (Steele, Lea & Flood, 2014): state += golden; output mix(state)
static uint64_t sm_next(uint64_t &s)
{
    s += 0x9E3779B97F4A7C15ull;
    return mix64(s);
}

static void glorot_init(uint64_t seed, std::vector<float> &p)
{
    p.assign(NP, 0.0f);
    uint64_t s = seed;
    const int offs[3] = {OFF_W1, OFF_W2, OFF_W3}, cnts[3] = {H * NF, H * H, H};
    const int fin[3] = {NF, H, H}, fout[3] = {H, H, 1};
    for (int q = 0; q < 3; ++q) {
        const float bound = sqrtf(6.0f / (float)(fin[q] + fout[q]));
        for (int t = 0; t < cnts[q]; ++t) {
            const float u = (float)(sm_next(s) >> 40) * (1.0f / 16777216.0f);
            p[offs[q] + t] = (2.0f * u - 1.0f) * bound;
        }
    }
}

static int upload_params(aco_prior *net, const float *params)
{
    PCHK(hipMemcpyAsync(net->pf, params, NP * sizeof(float), hipMemcpyHostToDevice, net->stream));
    PCHK(hipMemsetAsync(net->m, 0, NP * sizeof(float), net->stream));
    PCHK(hipMemsetAsync(net->v, 0, NP * sizeof(float), net->stream));
    hipLaunchKernelGGL(k_to_bf16, dim3((NP + 255) / 256), dim3(256), 0, net->stream, net->pf, net->wb, NP);
    PCHK(hipGetLastError());
    PCHK(hipStreamSynchronize(net->stream));
    net->step = 0;
    return ACO_OK;
}

static AdamArgs adam_args(int step, float lr, float b1, float b2, float eps)
{
    // bias corrections and (1 - beta) in double from the fp32 betas, rounded once
    AdamArgs a;
    a.lr = lr;
    a.beta1 = b1;
    a.beta2 = b2;
    a.om_beta1 = (float)(1.0 - (double)b1);
    a.om_beta2 = (float)(1.0 - (double)b2);
    a.c1 = (float)(1.0 - pow((double)b1, (double)step));
    a.c2 = (float)(1.0 - pow((double)b2, (double)step));
    a.eps = eps;
    return a;
}

static int pack_features(aco_prior *net, const float *feat, const float *label, long long count, unsigned short *xb,
                         float *lab)
{
    hipLaunchKernelGGL(k_pack_features, dim3((unsigned)((4 * count + 255) / 256)), dim3(256), 0, net->stream, feat,
                       label, count, xb, lab);
    PCHK(hipGetLastError());
    return ACO_OK;
}

// bf16 features and labels of `count` edges into device arrays: rows pass
// through the pinned input buffers, from which the packing kernel reads them
// while the next buffer is filled.
static int stage_features(aco_prior *net, const float *feat, const float *label, long long count, unsigned short *xb,
                          float *lab)
{
    PriorSpace &sp = net->space;
    const long long per = (long long)(sp.part / ((NF + 1) * sizeof(float)));
    for (long long e = 0; e < count; e += per) {
        const long long c = std::min(per, count - e);
        unsigned char *b = nullptr;
        PCHK(sp.take(b));
        float *f = reinterpret_cast<float *>(b), *l = f + c * NF;
        memcpy(f, feat + e * NF, (size_t)c * NF * sizeof(float));
        memcpy(l, label + e, (size_t)c * sizeof(float));
        const int rc = pack_features(net, f, l, c, xb + e * NFP, lab + e);
        if (rc != ACO_OK) return rc;
        PCHK(sp.used(net->stream));
    }
    return ACO_OK;
}

// bf16 features alone, from pageable memory through f32, which holds
// kForwardRows rows: one plain copy for most calls.  Without labels there is
// one array to move, and the runtime's copy of it is faster than a memcpy into
// pinned buffers from some 8000 edges on (forward of 16384 edges 75 against
// 87 us, 65536: 229, 305), and for fewer a new network pins nothing.
constexpr long long kForwardRows = 131072;   // 6 MB
static int stage_features_only(aco_prior *net, const float *feat, long long count, unsigned short *xb, float *f32)
{
    for (long long e = 0; e < count; e += kForwardRows) {
        const long long c = std::min(kForwardRows, count - e);
        PCHK(hipMemcpyAsync(f32, feat + e * NF, (size_t)c * NF * sizeof(float), hipMemcpyHostToDevice, net->stream));
        const int rc = pack_features(net, f32, nullptr, c, xb + e * NFP, nullptr);
        if (rc != ACO_OK) return rc;
    }
    return ACO_OK;
}

// Bytes put one after another, sent to the device through the pinned input
// buffers.
struct PinnedStream {
    aco_prior *net;
    unsigned char *dst, *buf = nullptr;
    size_t fill = 0;
    int flush()
    {
        if (!fill) return ACO_OK;
        PCHK(hipMemcpyAsync(dst, buf, fill, hipMemcpyHostToDevice, net->stream));
        PCHK(net->space.used(net->stream));
        dst += fill;
        fill = 0;
        buf = nullptr;
        return ACO_OK;
    }
    int put(const void *src, size_t bytes)
    {
        const unsigned char *s = static_cast<const unsigned char *>(src);
        while (bytes) {
            if (fill == net->space.part) {
                const int rc = flush();
                if (rc != ACO_OK) return rc;
            }
            if (!buf) PCHK(net->space.take(buf));
            const size_t c = std::min(bytes, net->space.part - fill);
            memcpy(buf + fill, s, c);
            fill += c;
            s += c;
            bytes -= c;
        }
        return ACO_OK;
    }
};

static int launch_forward(aco_prior *net, const unsigned short *xb, long long count, float *logits,
                          hipStream_t st = nullptr)
{
    const long long tiles = (count + 15) / 16;
    long long blocks = (tiles + kWaves - 1) / kWaves;
    if (blocks > 2048) blocks = 2048;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_forward, dim3((unsigned)blocks), dim3(kThreads), 0, st ? st : net->stream, xb,
                       count, net->wb, net->pf, logits);
    PCHK(hipGetLastError());
    return ACO_OK;
}

static float floor_pow(float floor, float exponent)
{
    return exponent == 1.0f ? floor : exponent == 2.0f ? floor * floor : powf(floor, exponent);
}

// One batch: fused forward/backward, then the ordered reduce (+ Adam).
static int launch_batch(aco_prior *net, const unsigned short *xb, const float *label, const int *idx,
                        int Eb, float pos_weight, float *partials, float *grad_out, float *loss_out,
                        bool update, const AdamArgs &aa)
{
    const int rows = train_rows(Eb);
    hipLaunchKernelGGL(k_train, dim3(std::min(rows, kTrainBlocks)), dim3(kThreads), 0, net->stream, xb, label, idx, Eb,
                       net->wb, net->pf, pos_weight, 1.0f / (float)Eb, partials);
    PCHK(hipGetLastError());
    hipLaunchKernelGGL(k_reduce_adam, dim3((NPL + kReduceParams - 1) / kReduceParams),
                       dim3(kReduceParams * kReduceGroups), 0, net->stream, partials,
                       rows, train_run(rows), net->pf, net->m, net->v, net->wb, grad_out, loss_out,
                       update ? 1 : 0, aa);
    PCHK(hipGetLastError());
    return ACO_OK;
}

static size_t partial_bytes(int Eb)
{
    return (size_t)train_rows(Eb) * NPL * sizeof(float);
}

extern "C" {

void aco_prior_default_train_params(aco_prior_train_params *tp)
{
    if (!tp) return;
    tp->epochs = 4;
    tp->batch = 16384;
    tp->lr = 3e-3f;
    tp->lr_final = 3e-4f;
    tp->pos_weight = 4.0f;
    tp->beta1 = 0.9f;
    tp->beta2 = 0.999f;
    tp->eps = 1e-8f;
    tp->shuffle_seed = 1;
}

int aco_prior_create(uint64_t seed, aco_prior **out)
{
    if (!out) return set_error(ACO_ERR_ARG, "null output handle");
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
        return set_error(ACO_ERR_NODEV, "no HIP device");
    aco_prior *net = new aco_prior();
    auto fail = [&](int rc) {
        aco_prior_destroy(net);
        return rc;
    };
    if (hipStreamCreateWithFlags(&net->stream, hipStreamNonBlocking) != hipSuccess ||
        hipMalloc((void **)&net->pf, NP * sizeof(float)) != hipSuccess ||
        hipMalloc((void **)&net->m, NP * sizeof(float)) != hipSuccess ||
        hipMalloc((void **)&net->v, NP * sizeof(float)) != hipSuccess ||
        hipMalloc((void **)&net->wb, NP * sizeof(unsigned short)) != hipSuccess)
        return fail(set_error(ACO_ERR_HIP, "aco_prior_create: device allocation failed"));
    std::vector<float> p;
    glorot_init(seed, p);
    const int rc = upload_params(net, p.data());
    if (rc != ACO_OK) return fail(rc);
    *out = net;
    return ACO_OK;
}

int aco_prior_destroy(aco_prior *net)
{
    if (!net) return ACO_OK;
    if (net->stream) (void)hipStreamSynchronize(net->stream);
    if (net->pf) (void)hipFree(net->pf);
    if (net->m) (void)hipFree(net->m);
    if (net->v) (void)hipFree(net->v);
    if (net->wb) (void)hipFree(net->wb);
    if (net->stream) (void)hipStreamDestroy(net->stream);
    delete net;
    return ACO_OK;
}

int aco_prior_get_params(aco_prior *net, float *params, int32_t count)
{
    if (!net || !params) return set_error(ACO_ERR_ARG, "null argument");
    if (count != NP) return set_error(ACO_ERR_ARG, "count must be ACO_PRIOR_PARAMS");
    PCHK(hipMemcpyAsync(params, net->pf, NP * sizeof(float), hipMemcpyDeviceToHost, net->stream));
    PCHK(hipStreamSynchronize(net->stream));
    return ACO_OK;
}

int aco_prior_set_params(aco_prior *net, const float *params, int32_t count)
{
    if (!net || !params) return set_error(ACO_ERR_ARG, "null argument");
    if (count != NP) return set_error(ACO_ERR_ARG, "count must be ACO_PRIOR_PARAMS");
    for (int i = 0; i < NP; ++i)
        if (!std::isfinite(params[i])) return set_error(ACO_ERR_ARG, "non-finite parameter");
    return upload_params(net, params);
}

static int check_instance_args(int32_t n, const float *x, const float *y, const int32_t *demand,
                               int32_t capacity, const float *dist, const int32_t *nn,
                               int32_t nn_width, int32_t k)
{
    if (n < 2 || n > 65536) return set_error(ACO_ERR_ARG, "n must be in [2, 65536]");
    if (!x || !y || !demand || !dist || !nn) return set_error(ACO_ERR_ARG, "null array");
    if (capacity <= 0) return set_error(ACO_ERR_ARG, "capacity must be positive");
    if (k < 1 || k > nn_width || k > n - 1) return set_error(ACO_ERR_ARG, "need 1 <= k <= nn_width, k < n");
    for (long long t = 0; t < (long long)n * nn_width; ++t)
        if (nn[t] < 0 || nn[t] >= n) return set_error(ACO_ERR_ARG, "nn list entry out of range");
    return ACO_OK;
}

// Device features of one instance, fp32 rows.
static int device_features(hipStream_t st, int32_t n, const float *x, const float *y,
                           const int32_t *demand, int32_t capacity, const float *dist,
                           const int32_t *nn, int32_t nnw, int32_t k, DevBuf &feat_d)
{
    DevBuf xd, yd, dd, demd, nn_d, rad, ang, kd, Rm;
    const size_t N = (size_t)n, E = N * (size_t)k;
    PCHK(dalloc(xd, N * 4));
    PCHK(dalloc(yd, N * 4));
    PCHK(dalloc(dd, N * N * 4));
    PCHK(dalloc(demd, N * 4));
    PCHK(dalloc(nn_d, N * nnw * 4));
    PCHK(dalloc(rad, N * 4));
    PCHK(dalloc(ang, N * 4));
    PCHK(dalloc(kd, N * 4));
    PCHK(dalloc(Rm, 16));
    PCHK(dalloc(feat_d, E * NF * 4));
    PCHK(hipMemcpyAsync(xd.p, x, N * 4, hipMemcpyHostToDevice, st));
    PCHK(hipMemcpyAsync(yd.p, y, N * 4, hipMemcpyHostToDevice, st));
    PCHK(hipMemcpyAsync(dd.p, dist, N * N * 4, hipMemcpyHostToDevice, st));
    PCHK(hipMemcpyAsync(demd.p, demand, N * 4, hipMemcpyHostToDevice, st));
    PCHK(hipMemcpyAsync(nn_d.p, nn, N * nnw * 4, hipMemcpyHostToDevice, st));
    const DistMatrix D = {dd.as<float>(), n};
    hipLaunchKernelGGL(k_node_stats<DistMatrix>, dim3((n + 255) / 256), dim3(256), 0, st, n, xd.as<float>(),
                       yd.as<float>(), D, nn_d.as<int>(), nnw, k, rad.as<float>(), ang.as<float>(),
                       kd.as<float>());
    PCHK(hipGetLastError());
    hipLaunchKernelGGL(k_node_reduce, dim3(1), dim3(256), 0, st, n, rad.as<float>(), kd.as<float>(),
                       Rm.as<float>());
    PCHK(hipGetLastError());
    hipLaunchKernelGGL(k_edge_features<DistMatrix>, dim3((unsigned)((E + 255) / 256)), dim3(256), 0, st, n, k, D,
                       nn_d.as<int>(), nnw, demd.as<int>(), (float)capacity, rad.as<float>(), ang.as<float>(),
                       kd.as<float>(), Rm.as<float>(), feat_d.as<float>(), (unsigned short *)nullptr);
    PCHK(hipGetLastError());
    PCHK(hipStreamSynchronize(st));
    return ACO_OK;
}

int aco_prior_features(int32_t n, const float *x, const float *y, const int32_t *demand,
                       int32_t capacity, const float *dist, const int32_t *nn, int32_t nn_width,
                       int32_t k, float *feat)
{
    int rc = check_instance_args(n, x, y, demand, capacity, dist, nn, nn_width, k);
    if (rc != ACO_OK) return rc;
    if (!feat) return set_error(ACO_ERR_ARG, "null feature buffer");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return set_error(ACO_ERR_NODEV, "no HIP device");
    hipStream_t st;
    PCHK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    {
        DevBuf fd;
        rc = device_features(st, n, x, y, demand, capacity, dist, nn, nn_width, k, fd);
        if (rc == ACO_OK) {
            const hipError_t e = hipMemcpy(feat, fd.p, (size_t)n * k * NF * 4, hipMemcpyDeviceToHost);
            if (e != hipSuccess) rc = set_error(ACO_ERR_HIP, std::string("feature readback: ") + hipGetErrorString(e));
        }
    }
    (void)hipStreamDestroy(st);
    return rc;
}

int aco_prior_forward(aco_prior *net, const float *feat, int64_t count, float *logits)
{
    if (!net || !feat || !logits) return set_error(ACO_ERR_ARG, "null argument");
    if (count < 1 || count > (1ll << 31)) return set_error(ACO_ERR_ARG, "count out of range");
    SpaceUse use(net->space, net->stream);
    const size_t rows = (size_t)std::min<long long>(count, kForwardRows);
    PCHK(net->space.init(SpaceUse::round((size_t)count * NFP * 2) + SpaceUse::round((size_t)count * 4) +
                         SpaceUse::round(rows * NF * 4)));
    unsigned short *xb = use.take<unsigned short>((size_t)count * NFP);
    float *out = use.take<float>((size_t)count);
    int rc = stage_features_only(net, feat, count, xb, use.take<float>(rows * NF));
    if (rc != ACO_OK) return rc;
    rc = launch_forward(net, xb, count, out);
    if (rc != ACO_OK) return rc;
    PCHK(hipMemcpyAsync(logits, out, (size_t)count * 4, hipMemcpyDeviceToHost, net->stream));
    PCHK(hipStreamSynchronize(net->stream));
    return ACO_OK;
}

int aco_prior_gradient(aco_prior *net, const float *feat, const float *label, int64_t count,
                       float pos_weight, float *grad, float *loss)
{
    if (!net || !feat || !label || !grad) return set_error(ACO_ERR_ARG, "null argument");
    if (count < 1 || count > kMaxBatch) return set_error(ACO_ERR_ARG, "count must be in [1, 65536]");
    if (!(pos_weight > 0.0f) || !std::isfinite(pos_weight)) return set_error(ACO_ERR_ARG, "pos_weight must be positive");
    SpaceUse use(net->space, net->stream);
    const size_t E = (size_t)count;
    PCHK(net->space.init(SpaceUse::round(E * NFP * 2) + SpaceUse::round(E * 4) + partial_bytes((int)count)));
    PCHK(net->space.pinned(E * (NF + 1) * sizeof(float), 0, NPL * sizeof(float)));
    unsigned short *xb = use.take<unsigned short>(E * NFP);
    float *lab = use.take<float>(E), *part = use.take<float>(partial_bytes((int)count) / 4);
    int rc = stage_features(net, feat, label, count, xb, lab);
    if (rc != ACO_OK) return rc;
    // the reduction writes the gradient and the loss to host memory
    float *g = reinterpret_cast<float *>(net->space.result());
    rc = launch_batch(net, xb, lab, nullptr, (int)count, pos_weight, part, g, g + NP, false,
                      adam_args(1, 0, 0.9f, 0.999f, 1e-8f));
    if (rc != ACO_OK) return rc;
    PCHK(hipStreamSynchronize(net->stream));
    memcpy(grad, g, NP * sizeof(float));
    if (loss) *loss = g[NP];
    return ACO_OK;
}

int aco_prior_adam_step(aco_prior *net, const float *grad, float lr, float beta1, float beta2, float eps)
{
    if (!net || !grad) return set_error(ACO_ERR_ARG, "null argument");
    // a single partial row holding the gradient (loss slot zero)
    DevBuf part;
    PCHK(dalloc(part, NPL * 4));
    PCHK(hipMemsetAsync(part.p, 0, NPL * 4, net->stream));
    PCHK(hipMemcpyAsync(part.p, grad, NP * 4, hipMemcpyHostToDevice, net->stream));
    net->step += 1;
    hipLaunchKernelGGL(k_reduce_adam, dim3((NPL + kReduceParams - 1) / kReduceParams),
                       dim3(kReduceParams * kReduceGroups), 0, net->stream, part.as<float>(), 1, 1,
                       net->pf, net->m, net->v, net->wb, nullptr, nullptr, 1,
                       adam_args(net->step, lr, beta1, beta2, eps));
    PCHK(hipGetLastError());
    PCHK(hipStreamSynchronize(net->stream));
    return ACO_OK;
}

constexpr long long kDeviceDraws = 4096;

int aco_prior_train(aco_prior *net, const float *feat, const float *label, int64_t count,
                    const aco_prior_train_params *tp, float *epoch_loss)
{
    if (!net || !feat || !label || !tp) return set_error(ACO_ERR_ARG, "null argument");
    if (count < 1 || count >= (1ll << 31)) return set_error(ACO_ERR_ARG, "count out of range");
    if (tp->epochs < 1 || tp->batch < 16 || tp->batch > kMaxBatch)
        return set_error(ACO_ERR_ARG, "epochs >= 1 and batch in [16, 65536] required");
    if (!(tp->lr > 0.0f) || !(tp->lr_final >= 0.0f) || !(tp->pos_weight > 0.0f))
        return set_error(ACO_ERR_ARG, "lr, lr_final, pos_weight must be positive");
    const long long nb = (count + tp->batch - 1) / tp->batch;
    const long long total = nb * tp->epochs;
    SpaceUse use(net->space, net->stream);
    PriorSpace &sp = net->space;
    const size_t E = (size_t)count;
    PCHK(sp.init(SpaceUse::round(E * NFP * 2) + 2 * SpaceUse::round(E * 4) + SpaceUse::round(partial_bytes(tp->batch)) +
                 SpaceUse::round((size_t)total * 4)));
    unsigned short *xb = use.take<unsigned short>(E * NFP);
    float *lab = use.take<float>(E);
    int *idx = use.take<int>(E);
    float *part = use.take<float>(partial_bytes(tp->batch) / 4), *losses = use.take<float>((size_t)total);
    // The order of an epoch is a Fisher-Yates shuffle, which only the host can
    // make (65536 swaps: 0.1 ms), but the swap targets are one 64-bit remainder
    // each (0.3 ms) of a counter-based stream, so the device draws them, two
    // buffers ahead of the swaps.  On the training stream, while nothing is
    // trained yet, and where a buffer holds an epoch (then its next one is
    // needed an epoch later); else beside the training, on a stream of its
    // own, which takes 0.4 to 3 ms to make (one epoch over 513024 edges on a
    // new network: 4.1 ms with host draws, 6.7 to 7.8 with that stream, 3.4
    // so).  Epochs of fewer than kDeviceDraws draws draw on the host, where
    // they cost less (5 ns each) than a launch and its wait (about 20 us).
    const long long per_epoch = count - 1, draws = per_epoch * tp->epochs;
    const bool device = per_epoch >= kDeviceDraws;
    const int chunk = (int)std::min<long long>(std::max(per_epoch, 1ll), PriorSpace::kPart / sizeof(int));
    const size_t span = SpaceUse::round((size_t)chunk * sizeof(int));
    PCHK(sp.pinned(E * (NF + 1) * sizeof(float), 0, device ? 2 * span : 0));
    auto targets = [&](int i) { return reinterpret_cast<int *>(sp.result() + i * span); };
    long long step = 0;    // batches launched
    long long drawn = 0;   // draws requested so far
    int requests = 0;      // request r fills buffer r % 2
    hipEvent_t ready[2] = {nullptr, nullptr};
    struct Events {
        hipEvent_t *e;
        ~Events()
        {
            for (int i = 0; i < 2; ++i)
                if (e[i]) (void)hipEventDestroy(e[i]);
        }
    } events{ready};
    auto request = [&]() -> int {   // never across an epoch's end
        if (!device || drawn == draws) return ACO_OK;
        const long long in = drawn % per_epoch;
        const int c = (int)std::min<long long>(chunk, per_epoch - in), at = requests & 1;
        if (!ready[at]) PCHK(hipEventCreateWithFlags(&ready[at], hipEventDisableTiming));
        const bool beside = step > 0 && per_epoch > chunk;
        if (beside && !sp.side) PCHK(hipStreamCreateWithFlags(&sp.side, hipStreamNonBlocking));
        const hipStream_t on = beside ? sp.side : net->stream;
        hipLaunchKernelGGL(k_swap_targets, dim3((c + 255) / 256), dim3(256), 0, on, tp->shuffle_seed,
                           (unsigned long long)drawn, (int)(per_epoch - in), c, targets(at));
        PCHK(hipGetLastError());
        PCHK(hipEventRecord(ready[at], on));
        drawn += c;
        ++requests;
        return ACO_OK;
    };
    int rc = request();
    if (rc == ACO_OK) rc = request();
    if (rc != ACO_OK) return rc;
    rc = stage_features(net, feat, label, count, xb, lab);
    if (rc != ACO_OK) return rc;
    std::vector<int> perm((size_t)count);
    int from = 0;   // buffer the next targets come from
    uint64_t seed = tp->shuffle_seed;
    for (int ep = 0; ep < tp->epochs; ++ep) {
        for (long long i = 0; i < count; ++i) perm[(size_t)i] = (int)i;
        for (long long i = count - 1; !device && i > 0; --i)
            std::swap(perm[(size_t)i], perm[(size_t)(sm_next(seed) % (uint64_t)(i + 1))]);
        for (long long i = count - 1; device && i > 0;) {
            PCHK(hipEventSynchronize(ready[from]));
            const int *j = targets(from);
            const long long c = std::min<long long>(chunk, i);
            for (long long t = 0; t < c; ++t) std::swap(perm[(size_t)(i - t)], perm[(size_t)j[t]]);
            i -= c;
            rc = request();   // refills this buffer
            if (rc != ACO_OK) return rc;
            from ^= 1;
        }
        PinnedStream up = {net, reinterpret_cast<unsigned char *>(idx)};   // behind the epoch that reads idx now
        rc = up.put(perm.data(), E * sizeof(int));
        if (rc == ACO_OK) rc = up.flush();
        if (rc != ACO_OK) return rc;
        for (long long b = 0; b < nb; ++b, ++step) {
            const long long lo = b * tp->batch;
            const int Eb = (int)std::min<long long>(tp->batch, count - lo);
            const double frac = total > 1 ? (double)step / (double)(total - 1) : 0.0;
            const float lr = (float)(tp->lr_final + 0.5 * (tp->lr - tp->lr_final) * (1.0 + cos(M_PI * frac)));
            net->step += 1;
            rc = launch_batch(net, xb, lab, idx + lo, Eb, tp->pos_weight, part, nullptr, losses + step, true,
                              adam_args(net->step, lr, tp->beta1, tp->beta2, tp->eps));
            if (rc != ACO_OK) return rc;
        }
    }
    std::vector<float> lh((size_t)total);
    PCHK(hipMemcpyAsync(lh.data(), losses, (size_t)total * 4, hipMemcpyDeviceToHost, net->stream));
    PCHK(hipStreamSynchronize(net->stream));
    if (epoch_loss)
        for (int ep = 0; ep < tp->epochs; ++ep) {
            double a = 0.0;
            for (long long b = 0; b < nb; ++b) a += lh[(size_t)(ep * nb + b)];
            epoch_loss[ep] = (float)(a / (double)nb);
        }
    return ACO_OK;
}

int aco_prior_build(aco_prior *net, int32_t n, const float *x, const float *y,
                    const int32_t *demand, int32_t capacity, const float *dist, const int32_t *nn,
                    int32_t nn_width, int32_t k, float exponent, float floor, float *prior)
{
    if (!net || !prior) return set_error(ACO_ERR_ARG, "null argument");
    int rc = check_instance_args(n, x, y, demand, capacity, dist, nn, nn_width, k);
    if (rc != ACO_OK) return rc;
    if (!(exponent >= 0.0f) || !std::isfinite(exponent)) return set_error(ACO_ERR_ARG, "exponent must be >= 0");
    if (!(floor > 0.0f && floor <= 1.0f)) return set_error(ACO_ERR_ARG, "floor must be in (0, 1]");
    // The device needs the depot row and the candidate edges of the distance
    // matrix, not the matrix, and returns the multiplier row by row into the
    // pinned buffers, each copied out while the next is written.
    SpaceUse use(net->space, net->stream);
    PriorSpace &sp = net->space;
    hipStream_t st = net->stream;
    const size_t N = (size_t)n, E = N * (size_t)k;
    // x, y, demand, depot row, lists and edges in one block, in this order
    const size_t block = 4 * N + 2 * E;
    PCHK(sp.init(SpaceUse::round(block * 4) + 3 * SpaceUse::round(N * 4) + 256 + SpaceUse::round(E * NFP * 2) +
                 SpaceUse::round(E * 4)));
    float *xd = use.take<float>(block), *yd = xd + N, *d0 = yd + 2 * N, *de = d0 + N + E;
    const int *demd = reinterpret_cast<int *>(yd + N), *nnd = reinterpret_cast<int *>(d0 + N);
    float *rad = use.take<float>(N), *ang = use.take<float>(N), *kd = use.take<float>(N), *Rm = use.take<float>(64);
    unsigned short *xb = use.take<unsigned short>(E * NFP);
    float *lg = use.take<float>(E);
    PCHK(sp.pinned(std::max(block, N * N) * 4, N * 4, 0));
    PinnedStream up = {net, reinterpret_cast<unsigned char *>(xd)};
    const struct { const void *p; } heads[4] = {{x}, {y}, {demand}, {dist}};   // dist: its first row
    for (const auto &h : heads)
        if ((rc = up.put(h.p, N * 4)) != ACO_OK) return rc;
    for (size_t i = 0; i < N; ++i)
        if ((rc = up.put(nn + i * nn_width, (size_t)k * 4)) != ACO_OK) return rc;
    std::vector<float> edges((size_t)k);
    for (size_t i = 0; i < N; ++i) {
        for (int r = 0; r < k; ++r) edges[r] = dist[i * N + (size_t)nn[i * nn_width + r]];
        if ((rc = up.put(edges.data(), (size_t)k * 4)) != ACO_OK) return rc;
    }
    if ((rc = up.flush()) != ACO_OK) return rc;
    const DistEdges D = {d0, de, k};
    hipLaunchKernelGGL(k_node_stats<DistEdges>, dim3((n + 255) / 256), dim3(256), 0, st, n, xd, yd, D, nnd, k, k, rad,
                       ang, kd);
    PCHK(hipGetLastError());
    hipLaunchKernelGGL(k_node_reduce, dim3(1), dim3(256), 0, st, n, rad, kd, Rm);
    PCHK(hipGetLastError());
    hipLaunchKernelGGL(k_edge_features<DistEdges>, dim3((unsigned)((E + 255) / 256)), dim3(256), 0, st, n, k, D, nnd, k,
                       demd, (float)capacity, rad, ang, kd, Rm, (float *)nullptr, xb);
    PCHK(hipGetLastError());
    rc = launch_forward(net, xb, (long long)E, lg);
    if (rc != ACO_OK) return rc;
    const float fl = floor_pow(floor, exponent);
    const int per = (int)std::min<size_t>(N, sp.part / (N * 4));
    struct { int row, rows, buf; } out = {0, 0, 0};   // rows on their way
    auto collect = [&]() -> int {
        if (!out.rows) return ACO_OK;
        // rows that all fit one part: the stream itself (11 us less than an
        // event's wait where it is the only one, 11 us more behind others; and
        // a stream whose last wait was an event's costs the next one made 100 us)
        PCHK(out.rows == n ? hipStreamSynchronize(st) : hipEventSynchronize(sp.done[out.buf]));
        sp.busy[out.buf] = false;
        memcpy(prior + (size_t)out.row * N, sp.pin + out.buf * sp.part, (size_t)out.rows * N * 4);
        return ACO_OK;
    };
    for (int row = 0; row < n; row += per) {
        const int rows = std::min(per, n - row), buf = sp.cur;
        unsigned char *b = nullptr;
        PCHK(sp.take(b));
        if (n <= kPriorRowLds)
            hipLaunchKernelGGL(k_prior_rows<true>, dim3(rows), dim3(256), N * 4, st, n, row, k, nnd, k, lg, exponent, fl,
                               reinterpret_cast<float *>(b));
        else
            hipLaunchKernelGGL(k_prior_rows<false>, dim3(rows), dim3(256), 0, st, n, row, k, nnd, k, lg, exponent, fl,
                               reinterpret_cast<float *>(b));
        PCHK(hipGetLastError());
        PCHK(sp.used(st));
        if ((rc = collect()) != ACO_OK) return rc;
        out = {row, rows, buf};
    }
    return collect();
}

int aco_prior_apply(aco_ctx *ctx, aco_prior *net, const float *const *x, const float *const *y,
                    int32_t k, float exponent, float floor)
{
    if (!ctx || !net || !x || !y) return set_error(ACO_ERR_ARG, "null argument");
    if (!(exponent >= 0.0f) || !std::isfinite(exponent)) return set_error(ACO_ERR_ARG, "exponent must be >= 0");
    if (!(floor > 0.0f && floor <= 1.0f)) return set_error(ACO_ERR_ARG, "floor must be in (0, 1]");
    std::vector<CtxInstanceView> views;
    void *sv = nullptr;
    int rc = ctx_prior_view(ctx, views, &sv);
    if (rc != ACO_OK) return rc;
    hipStream_t st = (hipStream_t)sv;
    int max_n = 0;
    for (size_t b = 0; b < views.size(); ++b) {
        const CtxInstanceView &v = views[b];
        if (!x[b] || !y[b]) return set_error(ACO_ERR_ARG, "null coordinates for instance " + std::to_string(b));
        if (k < 1 || k > v.n - 1) return set_error(ACO_ERR_ARG, "need 1 <= k < n");
        if (!((v.nnk && k <= v.k_ctx) || k <= v.nn_ls))
            return set_error(ACO_ERR_ARG, "k exceeds the context's candidate and neighbour lists");
        max_n = std::max(max_n, v.n);
    }
    const size_t N = (size_t)max_n, E = N * (size_t)k;
    DevBuf xd, yd, rad, ang, kd, Rm, xb, lg, dense;
    PCHK(dalloc(xd, N * 4));
    PCHK(dalloc(yd, N * 4));
    PCHK(dalloc(rad, N * 4));
    PCHK(dalloc(ang, N * 4));
    PCHK(dalloc(kd, N * 4));
    PCHK(dalloc(Rm, 16));
    PCHK(dalloc(xb, E * NFP * 2));
    PCHK(dalloc(lg, E * 4));
    PCHK(dalloc(dense, N * N * 4));
    const float fl = floor_pow(floor, exponent);
    for (size_t b = 0; b < views.size(); ++b) {
        const CtxInstanceView &v = views[b];
        const int n = v.n;
        const bool use_k = v.nnk && k <= v.k_ctx;
        const int *nn = use_k ? v.nnk : v.nnls;
        const int nnw = use_k ? v.k_ctx : v.nnP;
        const long long En = (long long)n * k, NN = (long long)n * n;
        PCHK(hipMemcpyAsync(xd.p, x[b], (size_t)n * 4, hipMemcpyHostToDevice, st));
        PCHK(hipMemcpyAsync(yd.p, y[b], (size_t)n * 4, hipMemcpyHostToDevice, st));
        const DistMatrix D = {v.dist, v.P};
        hipLaunchKernelGGL(k_node_stats<DistMatrix>, dim3((n + 255) / 256), dim3(256), 0, st, n, xd.as<float>(),
                           yd.as<float>(), D, nn, nnw, k, rad.as<float>(), ang.as<float>(), kd.as<float>());
        PCHK(hipGetLastError());
        hipLaunchKernelGGL(k_node_reduce, dim3(1), dim3(256), 0, st, n, rad.as<float>(), kd.as<float>(),
                           Rm.as<float>());
        PCHK(hipGetLastError());
        hipLaunchKernelGGL(k_edge_features<DistMatrix>, dim3((unsigned)((En + 255) / 256)), dim3(256), 0, st, n, k,
                           D, nn, nnw, v.dem, (float)v.Q, rad.as<float>(), ang.as<float>(), kd.as<float>(),
                           Rm.as<float>(), (float *)nullptr, xb.as<unsigned short>());
        PCHK(hipGetLastError());
        rc = launch_forward(net, xb.as<unsigned short>(), En, lg.as<float>(), st);
        if (rc != ACO_OK) return rc;
        hipLaunchKernelGGL(k_prior_fill, dim3((unsigned)((NN + 255) / 256)), dim3(256), 0, st, NN, fl,
                           dense.as<float>());
        PCHK(hipGetLastError());
        hipLaunchKernelGGL(k_prior_scatter, dim3((unsigned)((En + 255) / 256)), dim3(256), 0, st, n, k, nn,
                           nnw, lg.as<float>(), exponent, dense.as<float>());
        PCHK(hipGetLastError());
        hipLaunchKernelGGL(k_heur_mul, dim3((unsigned)((NN + 255) / 256)), dim3(256), 0, st, n, v.P,
                           dense.as<float>(), v.heur);
        PCHK(hipGetLastError());
    }
    PCHK(hipStreamSynchronize(st));
    return ACO_OK;
}

}  // extern "C"
