// harm_mlp.hip -- the learned Newton seed: GPU training (FP32 MFMA GEMMs,
// Adam), packing of the BF16 inference operands, and its C ABI.
//
// No counterpart in the reference (the seed replaces utoprim_2d.c:268-307).
// Training works on batches of B standardized rows:
//   forward   H1 = tanh(X W1^T + b1), H2, H3 likewise, O = H3 W4^T + b4
//   loss      L = 1/(2B) sum_b mask_b |O_b - T_b|^2
//   backward  dO = mask (O - T) / B;  dW_l = dZ_l^T H_{l-1};  db_l = dZ_l^T 1
//             dZ_{l-1} = (dZ_l W_l) * (1 - H_{l-1}^2)
// One launch (k_train) takes the batch through all of that with the activations
// in registers and LDS, every product on v_mfma_f32_16x16x4_f32; a second
// (k_adam_gather) folds the blocks' gradients in a fixed order, so that a training
// step is deterministic, applies Adam, and draws the next step's rows.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "harm_host.hpp"
#include "harm_phys.hpp"
#include "harm_mlp.hpp"

using namespace harm;

struct harm_mlp {
    int device;
    hipStream_t stream;
    float *params, *adam_m, *adam_v, *grad;
    uint4 *wpack;
    float *bias;
    double *norm;
    int vsq_from_W;
    float loss_w[2];  // weights of the two outputs in the training loss
    long long adam_t;
    // training workspace: the drawn rows of a batch (wsB of them), the blocks'
    // gradients, the losses of the steps not yet copied to the host
    int wsB;
    float *X, *T, *part;
    uint8_t *M;
    float4 *rec;  // a training set's records, recN of them
    size_t recN;
    double *lossd;
    double *normp;
};

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define MCHK(x)                                                                                            \
    do {                                                                                                   \
        hipError_t e_ = (x);                                                                               \
        if (e_ != hipSuccess)                                                                              \
            return harm_host::set_error(std::string(#x) + ": " + hipGetErrorString(e_) + " @harm_mlp.hip:" + \
                                            std::to_string(__LINE__),                                      \
                                        2);                                                                \
    } while (0)

// k_train: one block of 8 wavefronts per CU, each wavefront on 16 batch rows at a
// time.  A layer's activations are kept transposed (neurons x rows): with q = lane /
// 16 and c = lane % 16 the D layout of a 16x16 tile (register r: neuron 4q + r of row
// c) is the B operand of the next product for the contraction order {4q + r : q}, so
// the forward and the backward chain run from register to register, the weights
// coming from LDS (rows of TR_LD floats: 16-byte reads along a row and 4-byte reads
// across rows both touch every bank once).  A weight gradient contracts over the batch
// rows, for which D would have to be rows x neurons: each layer's h and dZ pass
// through LDS once and are read back in that order.  The 36 accumulator tiles of a
// wavefront (dW1 with db1 as its ninth column, dW2, dW3: 144 registers) are kept over all
// its rows; with the products' operands 60 of its registers go to scratch (136 B a lane).
//
// Bound by the FP32 matrix cores: 408 MFMA of 32 cycles per 16 rows.  Two wavefronts
// a SIMD (256 registers each) let one's 48 tanhf a lane run beside the other's
// products.  A batch of 65536 rows (two passes of a wavefront): 56 us, about 22 of
// them at the matrix cores' rate, 10 for the weights' staging and the fold at the end; the
// same step as 24 launches of one product or reduction each took 860 us.
constexpr int TR_WAVES = 8, TR_BLOCKS = 256;
constexpr int TR_LD = MLP_NH + 4;
constexpr int TR_W1 = 0, TR_W2 = TR_W1 + MLP_NH * MLP_NIN, TR_W3 = TR_W2 + MLP_NH * TR_LD,
              TR_BIAS = TR_W3 + MLP_NH * TR_LD, TR_W4 = TR_BIAS + 3 * MLP_NH, TR_B4 = TR_W4 + MLP_NOUT * MLP_NH,
              TR_SCR = TR_B4 + 4;
constexpr int TR_TILE = 16 * TR_LD, TR_SCRATCH = 3 * TR_TILE + 2 * 16;  // per wavefront: h1, h2, h3 or dZ; dO
// A wavefront's gradient as rows of 64 lanes: dW2 64, dW3 64, dW1 16, dW4 8, db2 4,
// db3 4, db4 2, loss 1.  The block's waves are added 55 rows at a time.
constexpr int TR_ROWS = 163, TR_FOLD = 55;
static_assert(TR_WAVES * TR_FOLD * 64 <= TR_SCR + TR_WAVES * TR_SCRATCH && 3 * TR_FOLD >= TR_ROWS, "fold buffer");
static_assert((TR_SCR + TR_WAVES * TR_SCRATCH) * 4 <= 160 * 1024, "LDS");

// LDS written by some lanes of a wavefront and read by others of the same one: its
// LDS operations complete in order, so only the compiler has to keep it.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ f32x4 lds4(const float *p) { return *reinterpret_cast<const f32x4 *>(p); }

// Keeps the scheduler from gathering the loads of several products in registers.
__device__ __forceinline__ void tr_stage() { __builtin_amdgcn_sched_barrier(0); }

// a = b + W h: a, h in D layout, 64 neurons each.
__device__ __forceinline__ void tr_dense(const float *W, const float *b, int q, int c, const f32x4 (&h)[4],
                                         f32x4 (&a)[4])
{
#pragma unroll
    for (int t = 0; t < 4; t++) a[t] = lds4(b + 16 * t + 4 * q);
#pragma unroll
    for (int s = 0; s < 4; s++) {
        if (s == 2) tr_stage();
        f32x4 w[4];
#pragma unroll
        for (int t = 0; t < 4; t++) w[t] = lds4(W + (16 * t + c) * TR_LD + 16 * s + 4 * q);
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int t = 0; t < 4; t++) a[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[t][r], h[s][r], a[t], 0, 0, 0);
    }
}

// a = W^T dz
__device__ __forceinline__ void tr_dense_t(const float *W, int q, int c, const f32x4 (&dz)[4], f32x4 (&a)[4])
{
#pragma unroll
    for (int t = 0; t < 4; t++) a[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; s++) {
        tr_stage();
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int t = 0; t < 4; t++)
                a[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(W[(16 * s + 4 * q + r) * TR_LD + 16 * t + c], dz[s][r],
                                                            a[t], 0, 0, 0);
    }
}

// dW += dZ^T h and db += dZ^T 1 over the 16 rows of two LDS tiles.
__device__ __forceinline__ void tr_wgrad(const float *dz, const float *h, int q, int c, f32x4 (&dW)[4][4],
                                         float (&db)[4])
{
#pragma unroll
    for (int r = 0; r < 4; r++) {
        if (r == 2) tr_stage();
        float a[4], b[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            a[t] = dz[(4 * q + r) * TR_LD + 16 * t + c];
            b[t] = h[(4 * q + r) * TR_LD + 16 * t + c];
            db[t] += a[t];
        }
#pragma unroll
        for (int o = 0; o < 4; o++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                dW[o][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[o], b[i], dW[o][i], 0, 0, 0);
    }
}

// tanh without a branch (the library's takes one of two per lane, so a wavefront runs
// both and the loads around them wait): an odd polynomial below 0.9, fitted there to a
// relative error of 6e-9, and 1 - 2 / (exp(2|x|) + 1) above.  Relative error against 64 bits
// over 4e6 arguments in [-12, 12]: 1.73e-8 rms, 1.06e-7 at most (the library's: 1.76e-8,
// 1.42e-7); over 4e6 in [1e-30, 1] 8.9e-9 and 1.06e-7 (9.2e-9 and 1.41e-7).
__device__ __forceinline__ float tr_tanhf(float x)
{
    const float ax = __builtin_fabsf(x), y = x * x;
    float p = -0.000455460249f;
    p = __builtin_fmaf(p, y, 0.00258266856f);
    p = __builtin_fmaf(p, y, -0.00826454442f);
    p = __builtin_fmaf(p, y, 0.0216635428f);
    p = __builtin_fmaf(p, y, -0.0539293028f);
    p = __builtin_fmaf(p, y, 0.133329779f);
    p = __builtin_fmaf(p, y, -0.333333224f);
    const float lo = __builtin_fmaf(ax * y, p, ax);
    const float e = __builtin_amdgcn_exp2f(ax * 2.88539008f) + 1.f;  // 2 log2(e)
    float r = __builtin_amdgcn_rcpf(e);
    r = e < 1e30f ? __builtin_fmaf(__builtin_fmaf(-e, r, 1.f), r, r) : r;
    const float hi = __builtin_fmaf(-2.f, r, 1.f);
    return __builtin_copysignf(ax < 0.9f ? lo : hi, x);
}

// h = tanh(a), also into the LDS tile (rows x neurons)
__device__ __forceinline__ void tr_tanh(const f32x4 (&a)[4], f32x4 (&h)[4], float *tile, int q, int c)
{
    tr_stage();
#pragma unroll
    for (int t = 0; t < 4; t++) {
#pragma unroll
        for (int r = 0; r < 4; r++) h[t][r] = tr_tanhf(a[t][r]);
        if (tile) *reinterpret_cast<f32x4 *>(tile + c * TR_LD + 16 * t + 4 * q) = h[t];
    }
}

// dz = a (1 - h^2) with h from its LDS tile, into the tile dzt
__device__ __forceinline__ void tr_dtanh(const f32x4 (&a)[4], const float *ht, f32x4 (&dz)[4], float *dzt, int q,
                                         int c)
{
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const f32x4 h = lds4(ht + c * TR_LD + 16 * t + 4 * q);
#pragma unroll
        for (int r = 0; r < 4; r++) dz[t][r] = a[t][r] * (1.f - h[r] * h[r]);
        *reinterpret_cast<f32x4 *>(dzt + c * TR_LD + 16 * t + 4 * q) = dz[t];
    }
}

// GRAD: the blocks' gradients and losses into part[block][TR_ROWS][64]; otherwise the
// outputs Y[B][2].  Any grid of at most TR_BLOCKS blocks covers the batch.
template <bool GRAD>
__global__ void __launch_bounds__(TR_WAVES * 64) __attribute__((amdgpu_waves_per_eu(2)))
k_train(const float *__restrict__ P, const float *__restrict__ X, const float *__restrict__ T,
        const uint8_t *__restrict__ M, int B, float lw0, float lw1, float *__restrict__ part, float *__restrict__ Y)
{
    __shared__ __attribute__((aligned(16))) float lds[TR_SCR + (GRAD ? TR_WAVES * TR_SCRATCH : 0)];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = lane >> 4, c = lane & 15;
    for (int k = tid; k < MLP_NH * MLP_NH; k += TR_WAVES * 64) {
        lds[TR_W2 + (k >> 6) * TR_LD + (k & 63)] = P[MLP_W2 + k];
        lds[TR_W3 + (k >> 6) * TR_LD + (k & 63)] = P[MLP_W3 + k];
    }
    for (int k = tid; k < MLP_NH * MLP_NIN; k += TR_WAVES * 64) lds[TR_W1 + k] = P[MLP_W1 + k];
    if (tid < MLP_NH) {
        lds[TR_BIAS + tid] = P[MLP_B1 + tid];
        lds[TR_BIAS + MLP_NH + tid] = P[MLP_B2 + tid];
        lds[TR_BIAS + 2 * MLP_NH + tid] = P[MLP_B3 + tid];
    } else if (tid < MLP_NH + MLP_NOUT * MLP_NH + MLP_NOUT) {
        lds[TR_W4 + tid - MLP_NH] = P[MLP_W4 + tid - MLP_NH];  // W4 and b4 follow each other in both
    }
    __syncthreads();

    float *t1 = lds + TR_SCR + (GRAD ? wave * TR_SCRATCH : 0), *t2 = t1 + TR_TILE, *t3 = t2 + TR_TILE,
          *tdo = t3 + TR_TILE;
    f32x4 dW1[4], dW2[4][4], dW3[4][4];
    float dW4[2][4], db2[4], db3[4], db4[2] = {0.f, 0.f}, loss = 0.f;
#pragma unroll
    for (int o = 0; o < 4; o++) {
        dW1[o] = f32x4{0.f, 0.f, 0.f, 0.f};
        db2[o] = db3[o] = dW4[0][o] = dW4[1][o] = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) dW2[o][i] = dW3[o][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    const int ntile = (B + 15) / 16;
    for (int tile = blockIdx.x + gridDim.x * wave; tile < ntile; tile += gridDim.x * TR_WAVES) {
        asm volatile("" ::: "memory");  // weights are read where they are used, not kept in registers over the rows
        const int z = 16 * tile + c;
        const bool in = z < B;
        f32x4 a[4], h[4];
        {
            const float x0 = in ? X[(size_t)z * MLP_NIN + 2 * q] : 0.f;
            const float x1 = in ? X[(size_t)z * MLP_NIN + 2 * q + 1] : 0.f;
#pragma unroll
            for (int t = 0; t < 4; t++) {
                a[t] = lds4(lds + TR_BIAS + 16 * t + 4 * q);
                const float *w = lds + TR_W1 + (16 * t + c) * MLP_NIN + 2 * q;
                a[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[0], x0, a[t], 0, 0, 0);
                a[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[1], x1, a[t], 0, 0, 0);
            }
        }
        tr_tanh(a, h, GRAD ? t1 : nullptr, q, c);
        tr_dense(lds + TR_W2, lds + TR_BIAS + MLP_NH, q, c, h, a);
        tr_tanh(a, h, GRAD ? t2 : nullptr, q, c);
        tr_dense(lds + TR_W3, lds + TR_BIAS + 2 * MLP_NH, q, c, h, a);
        tr_tanh(a, h, GRAD ? t3 : nullptr, q, c);
        float o0 = 0.f, o1 = 0.f;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const f32x4 w0 = lds4(lds + TR_W4 + 16 * t + 4 * q), w1 = lds4(lds + TR_W4 + MLP_NH + 16 * t + 4 * q);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                o0 += w0[r] * h[t][r];
                o1 += w1[r] * h[t][r];
            }
        }
        o0 += __shfl_xor(o0, 16, 64);
        o1 += __shfl_xor(o1, 16, 64);
        o0 += __shfl_xor(o0, 32, 64);
        o1 += __shfl_xor(o1, 32, 64);
        o0 += lds[TR_B4];
        o1 += lds[TR_B4 + 1];
        if (!GRAD) {
            if (q == 0 && in) {
                Y[(size_t)z * MLP_NOUT] = o0;
                Y[(size_t)z * MLP_NOUT + 1] = o1;
            }
            continue;
        }
        float d0 = 0.f, d1 = 0.f;
        if (in) {
            const float w = M ? (float)M[z] : 1.f;
            const float e0 = o0 - T[(size_t)z * MLP_NOUT], e1 = o1 - T[(size_t)z * MLP_NOUT + 1];
            d0 = w * lw0 * e0 / (float)B;
            d1 = w * lw1 * e1 / (float)B;
            if (q == 0) {
                loss += w * (lw0 * e0 * e0 + lw1 * e1 * e1);
                db4[0] += d0;
                db4[1] += d1;
            }
        }
        if (q == 0) {
            tdo[2 * c] = d0;
            tdo[2 * c + 1] = d1;
        }
        wave_lds_fence();
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float e0 = tdo[2 * (4 * q + r)], e1 = tdo[2 * (4 * q + r) + 1];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const float hz = t3[(4 * q + r) * TR_LD + 16 * t + c];
                dW4[0][t] += e0 * hz;
                dW4[1][t] += e1 * hz;
            }
        }
        f32x4 dz[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const f32x4 w0 = lds4(lds + TR_W4 + 16 * t + 4 * q), w1 = lds4(lds + TR_W4 + MLP_NH + 16 * t + 4 * q);
#pragma unroll
            for (int r = 0; r < 4; r++) a[t][r] = w0[r] * d0 + w1[r] * d1;
        }
        wave_lds_fence();
        tr_dtanh(a, t3, dz, t3, q, c);
        wave_lds_fence();
        tr_wgrad(t3, t2, q, c, dW3, db3);
        tr_dense_t(lds + TR_W3, q, c, dz, a);
        wave_lds_fence();
        tr_dtanh(a, t2, dz, t3, q, c);
        wave_lds_fence();
        tr_wgrad(t3, t1, q, c, dW2, db2);
        tr_dense_t(lds + TR_W2, q, c, dz, a);
        wave_lds_fence();
        tr_dtanh(a, t1, dz, t3, q, c);
        wave_lds_fence();
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int zr = 16 * tile + 4 * q + r;
            const float x = c < MLP_NIN ? (zr < B ? X[(size_t)zr * MLP_NIN + c] : 0.f) : (c == MLP_NIN ? 1.f : 0.f);
#pragma unroll
            for (int t = 0; t < 4; t++)
                dW1[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(t3[(4 * q + r) * TR_LD + 16 * t + c], x, dW1[t], 0, 0, 0);
        }
        wave_lds_fence();  // the next rows write the tiles that were read here
    }
    if (!GRAD) return;

    auto over_q = [](float v) {
        v += __shfl_xor(v, 16, 64);
        return v + __shfl_xor(v, 32, 64);
    };
    auto over_lanes = [](float v) {
#pragma unroll
        for (int s = 1; s < 64; s <<= 1) v += __shfl_xor(v, s, 64);
        return v;
    };
#pragma unroll
    for (int t = 0; t < 4; t++) {
        dW4[0][t] = over_q(dW4[0][t]);
        dW4[1][t] = over_q(dW4[1][t]);
        db2[t] = over_q(db2[t]);
        db3[t] = over_q(db3[t]);
    }
    db4[0] = over_lanes(db4[0]);
    db4[1] = over_lanes(db4[1]);
    loss = over_lanes(loss);
    auto row = [&](int k) -> float {  // k is a constant after unrolling
        if (k < 64) return dW2[k >> 4][(k >> 2) & 3][k & 3];
        if (k < 128) return dW3[(k - 64) >> 4][(k >> 2) & 3][k & 3];
        if (k < 144) return dW1[(k - 128) >> 2][k & 3];
        if (k < 152) return dW4[(k - 144) >> 2][k & 3];
        if (k < 156) return db2[k & 3];
        if (k < 160) return db3[k & 3];
        return k == 160 ? db4[0] : k == 161 ? db4[1] : loss;
    };
    float *out = part + (size_t)blockIdx.x * (TR_ROWS * 64);
#pragma unroll
    for (int f = 0; f < 3; f++) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < TR_FOLD; k++)
            if (f * TR_FOLD + k < TR_ROWS) lds[(wave * TR_FOLD + k) * 64 + lane] = row(f * TR_FOLD + k);
        __syncthreads();
        const int n = (f == 2 ? TR_ROWS - 2 * TR_FOLD : TR_FOLD) * 64;
        for (int k = tid; k < n; k += TR_WAVES * 64) {
            float s = 0.f;
#pragma unroll
            for (int w = 0; w < TR_WAVES; w++) s += lds[w * TR_FOLD * 64 + k];
            out[f * TR_FOLD * 64 + k] = s;
        }
    }
}

// Packs the BF16 A operands and the bias table of harm_mlp.hpp from the
// master parameters: one thread per (chunk, lane).
__global__ void k_pack(const float *__restrict__ P, uint4 *__restrict__ wpack, float *__restrict__ bias)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < MLP_CHUNKS * 64) {
        const int chunk = t / 64, lane = t % 64, row = lane & 15, gq = lane >> 4;
        bf16x8_t v;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            float w = 0.f;
            if (chunk < 4) {
                const int o = 16 * chunk + row;
                if (gq < 2 && i < 4) w = P[MLP_W1 + o * MLP_NIN + 4 * gq + i];
            } else if (chunk < 20) {
                const int base = (chunk < 12) ? MLP_W2 : MLP_W3;
                const int rel = (chunk < 12) ? chunk - 4 : chunk - 12;
                const int mt = rel / 2, c = rel % 2;
                w = P[base + (16 * mt + row) * MLP_NH + mlp_perm(c, gq, i)];
            } else {
                const int c = chunk - 20;
                if (row < MLP_NOUT) w = P[MLP_W4 + row * MLP_NH + mlp_perm(c, gq, i)];
            }
            v[i] = (__bf16)w;
        }
        wpack[t] = __builtin_bit_cast(uint4, v);
    }
    if (t < MLP_BIAS_LEN) {
        float b = 0.f;
        if (t < MLP_NH)
            b = P[MLP_B1 + t];
        else if (t < 2 * MLP_NH)
            b = P[MLP_B2 + t - MLP_NH];
        else if (t < 3 * MLP_NH)
            b = P[MLP_B3 + t - 2 * MLP_NH];
        else if (t < 3 * MLP_NH + MLP_NOUT)
            b = P[MLP_B4 + t - 3 * MLP_NH];
        bias[t] = b;
    }
}

// splitmix64 finalizer: the row drawn for (seed, step, b).
__device__ __forceinline__ unsigned long long mix64(unsigned long long x)
{
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

// A training set and the draw of one batch from it.  A row lies in eleven arrays, and
// at random rows each of its numbers costs a cache line: where a call draws enough of
// them (see harm_mlp_train) the set is first written as records of the very floats
// that a draw forms, 8 inputs, 2 targets and the mask in 48 bytes.
struct Draw {
    const double *feat, *targ;
    const uint8_t *valid;
    const float4 *rec;  // the records, or null
    size_t n;
    int B;
    unsigned long long seed;
};

__device__ __forceinline__ void row_floats(const Draw &d, const double *__restrict__ norm, size_t r, float (&x)[12])
{
    const size_t n = d.n;
#pragma unroll
    for (int k = 0; k < MLP_NIN; k++) x[k] = (float)((d.feat[k * n + r] - norm[k]) * norm[8 + k]);
    const bool ok = d.valid ? d.valid[r] != 0 : true;
    x[8] = ok ? (float)((d.targ[r] - norm[16]) / norm[18]) : 0.f;
    x[9] = ok ? (float)((d.targ[n + r] - norm[17]) / norm[19]) : 0.f;
    x[10] = ok ? 1.f : 0.f;
    x[11] = 0.f;
}

__global__ void __launch_bounds__(256) k_records(Draw d, const double *__restrict__ norm, float4 *__restrict__ rec)
{
    const size_t r = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (r >= d.n) return;
    float x[12];
    row_floats(d, norm, r, x);
#pragma unroll
    for (int k = 0; k < 3; k++) rec[3 * r + k] = make_float4(x[4 * k], x[4 * k + 1], x[4 * k + 2], x[4 * k + 3]);
}

__device__ __forceinline__ void draw_row(const Draw &d, const double *__restrict__ norm, int b, float *__restrict__ X,
                                         float *__restrict__ T, uint8_t *__restrict__ M)
{
    const size_t r = (size_t)(mix64(d.seed ^ mix64((unsigned long long)b)) % d.n);
    float x[12];
    if (d.rec) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const float4 v = d.rec[3 * r + k];
            x[4 * k] = v.x;
            x[4 * k + 1] = v.y;
            x[4 * k + 2] = v.z;
            x[4 * k + 3] = v.w;
        }
    } else {
        row_floats(d, norm, r, x);
    }
#pragma unroll
    for (int k = 0; k < MLP_NIN; k++) X[(size_t)b * MLP_NIN + k] = x[k];
    T[(size_t)b * MLP_NOUT] = x[8];
    T[(size_t)b * MLP_NOUT + 1] = x[9];
    M[b] = x[10] != 0.f ? 1 : 0;
}

// Parameter of row/lane of k_train's gradients; -1 where there is none.
__device__ __forceinline__ int tr_param(int row, int lane)
{
    const int q = lane >> 4, c = lane & 15;
    if (row < 128) {
        const int o = (row >> 4) & 3, i = (row >> 2) & 3, r = row & 3;
        return (row < 64 ? MLP_W2 : MLP_W3) + (16 * o + 4 * q + r) * MLP_NH + 16 * i + c;
    }
    if (row < 144) {
        const int n = 16 * ((row - 128) >> 2) + 4 * q + (row & 3);
        return c < MLP_NIN ? MLP_W1 + n * MLP_NIN + c : c == MLP_NIN ? MLP_B1 + n : -1;
    }
    if (row < 160) {
        if (q) return -1;
        const int t = row & 3;
        if (row < 152) return MLP_W4 + ((row - 144) >> 2) * MLP_NH + 16 * t + c;
        return (row < 156 ? MLP_B2 : MLP_B3) + 16 * t + c;
    }
    return lane == 0 && row < 162 ? MLP_B4 + row - 160 : -1;
}

// Blocks [0, nfold): one row of k_train's gradients each, the nb blocks' values added
// in 64 bits in a fixed order (8 wavefronts a share each, then those), into grad, and
// an Adam step where asked; row 162 is the loss.  The other blocks draw the rows of
// the next step's batch, which does not depend on the parameters: its scattered
// 8-byte loads run beside the fold, and a step is two launches.
constexpr int AG_THREADS = 512;
__global__ void __launch_bounds__(AG_THREADS)
k_adam_gather(const float *__restrict__ part, int nfold, int nb, int B, float *__restrict__ p, float *__restrict__ m,
              float *__restrict__ v, float *__restrict__ grad, double *__restrict__ loss, int step, float lr, float bc1,
              float bc2, Draw d, const double *__restrict__ norm, float *__restrict__ X, float *__restrict__ T,
              uint8_t *__restrict__ M)
{
    const int row = blockIdx.x;
    if (row >= nfold) {
        const long long b = (long long)(row - nfold) * AG_THREADS + threadIdx.x;
        if (b < d.B) draw_row(d, norm, (int)b, X, T, M);
        return;
    }
    __shared__ double red[AG_THREADS / 64][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    double s = 0.;
#pragma unroll 8
    for (int z = w; z < nb; z += AG_THREADS / 64) s += (double)part[((size_t)z * TR_ROWS + row) * 64 + lane];
    red[w][lane] = s;
    __syncthreads();
    if (w) return;
#pragma unroll
    for (int k = 1; k < AG_THREADS / 64; k++) s += red[k][lane];
    if (row == TR_ROWS - 1) {
        if (lane == 0) *loss = s / (2. * B);
        return;
    }
    const int i = tr_param(row, lane);
    if (i < 0) return;
    const float gi = (float)s;
    grad[i] = gi;
    if (!step) return;
    const float mi = 0.9f * m[i] + 0.1f * gi;
    const float vi = 0.999f * v[i] + 0.001f * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float mh = mi / bc1, vh = vi / bc2;
    p[i] -= lr * mh / (sqrtf(vh) + 1e-8f);
}

// Partial sums over valid rows for the normalization: pass 0 sums x, pass 1
// sums (x - mean)^2; 10 variables (8 features, 2 targets) and the row count.
__global__ void __launch_bounds__(256) k_norm_partials(const double *__restrict__ feat,
                                                       const double *__restrict__ targ,
                                                       const uint8_t *__restrict__ valid, size_t n, int pass,
                                                       const double *__restrict__ mean, double *__restrict__ part)
{
    __shared__ double red[11][256];
    double acc[11];
#pragma unroll
    for (int k = 0; k < 11; k++) acc[k] = 0.;
    for (size_t r = (size_t)blockIdx.x * 256 + threadIdx.x; r < n; r += (size_t)gridDim.x * 256) {
        if (valid && !valid[r]) continue;
#pragma unroll
        for (int k = 0; k < 10; k++) {
            const double x = (k < 8) ? feat[k * n + r] : targ[(k - 8) * n + r];
            const double d = pass ? x - mean[k] : x;
            acc[k] += pass ? d * d : d;
        }
        acc[10] += 1.;
    }
#pragma unroll
    for (int k = 0; k < 11; k++) red[k][threadIdx.x] = acc[k];
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s)
#pragma unroll
            for (int k = 0; k < 11; k++) red[k][threadIdx.x] += red[k][threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x < 11) part[blockIdx.x * 11 + threadIdx.x] = red[threadIdx.x][0];
}

constexpr int NORM_BLOCKS = 512;

// Single thread: fold the partials in block order into the mean (pass 0) or
// into the normalization block (pass 1).
__global__ void k_norm_finish(const double *__restrict__ part, int pass, double *__restrict__ mean,
                              double *__restrict__ norm)
{
    double s[11];
    for (int k = 0; k < 11; k++) s[k] = 0.;
    for (int b = 0; b < NORM_BLOCKS; b++)
        for (int k = 0; k < 11; k++) s[k] += part[b * 11 + k];
    const double cnt = s[10] > 0. ? s[10] : 1.;
    if (pass == 0) {
        for (int k = 0; k < 10; k++) mean[k] = s[k] / cnt;
        return;
    }
    for (int k = 0; k < 10; k++) {
        double sd = sqrt(s[k] / cnt);
        if (!(sd > 1e-12)) sd = 1.;
        if (k < 8) {
            norm[k] = mean[k];
            norm[8 + k] = 1. / sd;
        } else {
            norm[16 + (k - 8)] = mean[k];
            norm[18 + (k - 8)] = sd;
        }
    }
}

// BF16 inference on standardized inputs (rows beyond n are zero inputs).
__global__ void __launch_bounds__(256) k_forward_bf16(MlpDev m, const float *__restrict__ X, float *__restrict__ Y,
                                                      int n)
{
    const int b = blockIdx.x * 256 + threadIdx.x;
    float x[MLP_NIN];
#pragma unroll
    for (int k = 0; k < MLP_NIN; k++) x[k] = (b < n) ? X[b * MLP_NIN + k] : 0.f;
    float y0, y1;
    mlp_forward_wave(m, x, y0, y1);
    if (b < n) {
        Y[2 * b] = y0;
        Y[2 * b + 1] = y1;
    }
}

// Features and seeds of a zone batch (SoA as harm_utoprim2d_batch).
__global__ void __launch_bounds__(256) k_seed(MlpDev m, const double *__restrict__ U, const double *__restrict__ gcov,
                                              const double *__restrict__ gcon, const double *__restrict__ gdet,
                                              size_t n, double *__restrict__ feat, double *__restrict__ W0,
                                              double *__restrict__ vsq0)
{
    const size_t z = (size_t)blockIdx.x * 256 + threadIdx.x;
    const bool act = z < n;
    double f[MLP_NIN], D = 1.;
    bool ok = false;
    if (act) {
        Geom geom;
#pragma unroll
        for (int a = 0; a < 16; a++) {
            geom.gcov[a / 4][a % 4] = gcov[(size_t)a * n + z];
            geom.gcon[a / 4][a % 4] = gcon[(size_t)a * n + z];
        }
        geom.g = gdet[z];
        geom_derive(geom);
        double Uz[NPR];
#pragma unroll
        for (int k = 0; k < NPR; k++) Uz[k] = U[(size_t)k * n + z];
        ok = mlp_features_U(Uz, geom, f);
        if (ok) D = mlp_wref(f);
        if (feat)
#pragma unroll
            for (int k = 0; k < MLP_NIN; k++) feat[(size_t)k * n + z] = f[k];
    }
    if (!W0) return;  // uniform over the grid: no MFMA below
    float x[MLP_NIN];
    if (ok)
        mlp_standardize(m, f, x);
    else
#pragma unroll
        for (int k = 0; k < MLP_NIN; k++) x[k] = 0.f;
    float y0, y1;
    mlp_forward_wave(m, x, y0, y1);
    if (act) {
        double w, v;
        mlp_unstandardize(m, y0, y1, D, w, v);
        W0[z] = ok ? w : 0.;
        if (vsq0) vsq0[z] = ok ? v : 0.;
    }
}

// Training pairs from solved zones: features of U, targets from the converged
// primitives (W = (rho + gam u) (1 + utsq), v^2 = utsq / (1 + utsq)).
__global__ void __launch_bounds__(256) k_pairs(const double *__restrict__ U, const double *__restrict__ gcov,
                                               const double *__restrict__ gcon, const double *__restrict__ gdet,
                                               const double *__restrict__ prim, const int8_t *__restrict__ ret,
                                               size_t n, double gam, double *__restrict__ feat,
                                               double *__restrict__ targ, uint8_t *__restrict__ valid)
{
    const size_t z = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (z >= n) return;
    Geom geom;
#pragma unroll
    for (int a = 0; a < 16; a++) {
        geom.gcov[a / 4][a % 4] = gcov[(size_t)a * n + z];
        geom.gcon[a / 4][a % 4] = gcon[(size_t)a * n + z];
    }
    geom.g = gdet[z];
    geom_derive(geom);
    double Uz[NPR], pr[NPR], f[MLP_NIN];
#pragma unroll
    for (int k = 0; k < NPR; k++) {
        Uz[k] = U[(size_t)k * n + z];
        pr[k] = prim[(size_t)k * n + z];
    }
    const bool ok = mlp_features_U(Uz, geom, f) && ret[z] == 0 && mlp_wref(f) > 0.;
    double t0 = 0., t1 = 0.;
    if (ok) {
        const double utsq = utsq_of(geom, pr);
        t0 = log((pr[RHO] + gam * pr[UU]) * (1. + utsq)) - log(mlp_wref(f));
        t1 = utsq / (1. + utsq);
    }
#pragma unroll
    for (int k = 0; k < MLP_NIN; k++) feat[(size_t)k * n + z] = f[k];
    targ[z] = t0;
    targ[n + z] = t1;
    valid[z] = ok ? 1 : 0;
}

inline unsigned cdiv(size_t a, size_t b) { return (unsigned)((a + b - 1) / b); }

template <class T>
int dalloc(T **p, size_t n)
{
    *p = nullptr;
    if (n == 0) return 0;
    MCHK(hipMalloc((void **)p, n * sizeof(T)));
    return 0;
}

// Training sets of at most REC_MAX rows (0.8 GB of records, kept with the network) are
// drawn from records where a call draws more than one row in REC_ROWS of the set.
constexpr size_t REC_MAX = (size_t)1 << 24, REC_ROWS = 8;

// Steps whose losses wait on the device for one copy.
constexpr int LOSS_KEEP = 1024;

int ensure_ws(harm_mlp *m, int B)
{
    if (B <= m->wsB) return 0;
    m->wsB = 0;
    void **bufs[] = {(void **)&m->X, (void **)&m->T, (void **)&m->M};
    for (auto p : bufs) {
        if (*p) (void)hipFree(*p);
        *p = nullptr;
    }
    const size_t b = (size_t)B;
    int rc;
    if ((rc = dalloc(&m->X, b * MLP_NIN)) || (rc = dalloc(&m->T, b * MLP_NOUT)) || (rc = dalloc(&m->M, b))) return rc;
    m->wsB = B;
    return 0;
}

// Room for a training set of n rows as records; false where there is none.
bool ensure_records(harm_mlp *m, size_t n)
{
    if (n <= m->recN) return true;
    if (m->rec) (void)hipFree(m->rec);
    m->rec = nullptr;
    m->recN = 0;
    if (hipMalloc((void **)&m->rec, n * 3 * sizeof(float4)) != hipSuccess) {
        (void)hipGetLastError();
        m->rec = nullptr;
        return false;
    }
    m->recN = n;
    return true;
}

// A batch's 16-row tiles go to the blocks in turn, so a small one takes a wavefront
// on each of as many CUs as it has tiles.
int train_blocks(int B) { return (int)std::min<unsigned>(TR_BLOCKS, cdiv(B, 16)); }

int launch_forward(harm_mlp *m, const float *X, float *Y, int B)
{
    hipLaunchKernelGGL(k_train<false>, dim3(train_blocks(B)), dim3(TR_WAVES * 64), 0, m->stream, m->params, X,
                       (const float *)nullptr, (const uint8_t *)nullptr, B, 0.f, 0.f, (float *)nullptr, Y);
    MCHK(hipGetLastError());
    return 0;
}

// Forward, loss and gradient of B standardized rows into m->part.
int launch_train(harm_mlp *m, const float *X, const float *T, const uint8_t *M, int B)
{
    hipLaunchKernelGGL(k_train<true>, dim3(train_blocks(B)), dim3(TR_WAVES * 64), 0, m->stream, m->params, X, T, M, B,
                       m->loss_w[0], m->loss_w[1], m->part, (float *)nullptr);
    MCHK(hipGetLastError());
    return 0;
}

int launch_draw(harm_mlp *m, const Draw &d)
{
    hipLaunchKernelGGL(k_adam_gather, dim3(cdiv(d.B, AG_THREADS)), dim3(AG_THREADS), 0, m->stream, m->part, 0, 0, 0,
                       m->params, m->adam_m, m->adam_v, m->grad, m->lossd, 0, 0.f, 1.f, 1.f, d, m->norm, m->X, m->T, m->M);
    MCHK(hipGetLastError());
    return 0;
}

// The gradient of launch_train's batch into m->grad and its loss into *loss (m->lossd
// if null); an Adam step where loss is given; the rows of *next drawn where that is.
int launch_adam(harm_mlp *m, int B, double *loss, float lr, const Draw *next)
{
    float bc1 = 1.f, bc2 = 1.f;
    const bool step = loss != nullptr;
    if (step) {
        m->adam_t++;
        bc1 = (float)(1. - std::pow(0.9, (double)m->adam_t));
        bc2 = (float)(1. - std::pow(0.999, (double)m->adam_t));
    }
    const Draw d = next ? *next : Draw{};
    hipLaunchKernelGGL(k_adam_gather, dim3(TR_ROWS + cdiv(d.B, AG_THREADS)), dim3(AG_THREADS), 0, m->stream, m->part,
                       TR_ROWS, train_blocks(B), B, m->params, m->adam_m, m->adam_v, m->grad,
                       step ? loss : m->lossd, (int)step, lr, bc1, bc2, d, m->norm, m->X, m->T, m->M);
    MCHK(hipGetLastError());
    return 0;
}

int repack(harm_mlp *m)
{
    hipLaunchKernelGGL(k_pack, dim3(cdiv(MLP_CHUNKS * 64, 256)), dim3(256), 0, m->stream, m->params, m->wpack,
                       m->bias);
    MCHK(hipGetLastError());
    return 0;
}

struct DevGuard {
    int prev = -1;
    explicit DevGuard(int d)
    {
        (void)hipGetDevice(&prev);
        if (prev != d) (void)hipSetDevice(d);
    }
    ~DevGuard()
    {
        int cur;
        if (hipGetDevice(&cur) == hipSuccess && cur != prev && prev >= 0) (void)hipSetDevice(prev);
    }
};

int check_batch(int n)
{
    if (n <= 0 || n > (1 << 24)) return harm_host::set_error("batch size must be in [1, 2^24]", 4);
    return 0;
}

}  // namespace

harm::MlpDev harm_mlp_view(const harm_mlp *m)
{
    harm::MlpDev d;
    d.wpack = m->wpack;
    d.bias = m->bias;
    d.norm = m->norm;
    d.vsq_from_W = m->vsq_from_W;
    return d;
}
int harm_mlp_device(const harm_mlp *m) { return m->device; }

extern "C" {

harm_mlp *harm_mlp_create(int device)
{
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) {
        harm_host::set_error("no HIP device available: libharmcool.so runs only on a gfx950 GPU", 2);
        return nullptr;
    }
    if (device >= 0 && hipSetDevice(device) != hipSuccess) {
        harm_host::set_error("hipSetDevice failed", 2);
        return nullptr;
    }
    harm_mlp *m = new harm_mlp();
    std::memset(m, 0, sizeof(*m));
    (void)hipGetDevice(&m->device);
    m->vsq_from_W = 1;
    m->loss_w[0] = m->loss_w[1] = 1.f;
    bool ok = hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) == hipSuccess;
    ok = ok && !dalloc(&m->params, MLP_NPARAMS) && !dalloc(&m->adam_m, MLP_NPARAMS) &&
         !dalloc(&m->adam_v, MLP_NPARAMS) && !dalloc(&m->grad, MLP_NPARAMS) && !dalloc(&m->wpack, MLP_CHUNKS * 64) &&
         !dalloc(&m->bias, MLP_BIAS_LEN) && !dalloc(&m->norm, MLP_NORM_LEN) && !dalloc(&m->normp, NORM_BLOCKS * 11 + 16) &&
         !dalloc(&m->part, (size_t)TR_BLOCKS * TR_ROWS * 64) && !dalloc(&m->lossd, LOSS_KEEP);
    if (!ok) {
        harm_mlp_destroy(m);
        return nullptr;
    }
    std::vector<double> nrm(MLP_NORM_LEN, 0.);
    for (int k = 0; k < 8; k++) nrm[8 + k] = 1.;
    nrm[18] = nrm[19] = 1.;
    if (harm_mlp_set_norm(m, nrm.data()) || harm_mlp_init(m, 1)) {
        harm_mlp_destroy(m);
        return nullptr;
    }
    return m;
}

void harm_mlp_destroy(harm_mlp *m)
{
    if (!m) return;
    DevGuard dg(m->device);
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    void *bufs[] = {m->params, m->adam_m, m->adam_v, m->grad, m->wpack, m->bias, m->norm, m->normp,
                    m->X,      m->T,      m->M,      m->part, m->lossd, m->rec};
    for (void *p : bufs)
        if (p) (void)hipFree(p);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
}

int harm_mlp_init(harm_mlp *m, uint64_t seed)
{
    if (!m) return harm_host::set_error("null network", 1);
    std::vector<float> P(MLP_NPARAMS, 0.f);
    unsigned long long s = seed * 0x9E3779B97F4A7C15ull + 1;
    auto next = [&]() {
        s ^= s << 13;
        s ^= s >> 7;
        s ^= s << 17;
        return (double)(s >> 11) * (1.0 / 9007199254740992.0);
    };
    auto fill = [&](int off, int nout, int nin) {
        const double a = std::sqrt(3.0 / nin);
        for (int i = 0; i < nout * nin; i++) P[off + i] = (float)((2. * next() - 1.) * a);
    };
    fill(MLP_W1, MLP_NH, MLP_NIN);
    fill(MLP_W2, MLP_NH, MLP_NH);
    fill(MLP_W3, MLP_NH, MLP_NH);
    fill(MLP_W4, MLP_NOUT, MLP_NH);
    return harm_mlp_set_params(m, P.data());
}

int harm_mlp_set_params(harm_mlp *m, const float *params)
{
    if (!m || !params) return harm_host::set_error("null argument", 1);
    DevGuard dg(m->device);
    MCHK(hipMemcpyAsync(m->params, params, MLP_NPARAMS * sizeof(float), hipMemcpyHostToDevice, m->stream));
    MCHK(hipMemsetAsync(m->adam_m, 0, MLP_NPARAMS * sizeof(float), m->stream));
    MCHK(hipMemsetAsync(m->adam_v, 0, MLP_NPARAMS * sizeof(float), m->stream));
    m->adam_t = 0;
    int rc = repack(m);
    if (rc) return rc;
    MCHK(hipStreamSynchronize(m->stream));
    return 0;
}

int harm_mlp_get_params(harm_mlp *m, float *params)
{
    if (!m || !params) return harm_host::set_error("null argument", 1);
    DevGuard dg(m->device);
    MCHK(hipMemcpyAsync(params, m->params, MLP_NPARAMS * sizeof(float), hipMemcpyDeviceToHost, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    return 0;
}

int harm_mlp_set_norm(harm_mlp *m, const double *norm)
{
    if (!m || !norm) return harm_host::set_error("null argument", 1);
    for (int k = 8; k < 16; k++)
        if (!(norm[k] > 0.) || !std::isfinite(norm[k])) return harm_host::set_error("feature 1/std must be > 0", 4);
    if (!(norm[18] > 0.) || !(norm[19] > 0.)) return harm_host::set_error("output std must be > 0", 4);
    DevGuard dg(m->device);
    MCHK(hipMemcpyAsync(m->norm, norm, MLP_NORM_LEN * sizeof(double), hipMemcpyHostToDevice, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    return 0;
}

int harm_mlp_get_norm(harm_mlp *m, double *norm)
{
    if (!m || !norm) return harm_host::set_error("null argument", 1);
    DevGuard dg(m->device);
    MCHK(hipMemcpyAsync(norm, m->norm, MLP_NORM_LEN * sizeof(double), hipMemcpyDeviceToHost, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    return 0;
}

int harm_mlp_set_vsq_from_w(harm_mlp *m, int on)
{
    if (!m) return harm_host::set_error("null network", 1);
    m->vsq_from_W = on ? 1 : 0;
    return 0;
}

int harm_mlp_set_loss_weights(harm_mlp *m, float w_logw, float w_vsq)
{
    if (!m) return harm_host::set_error("null network", 1);
    if (!(w_logw >= 0.f) || !(w_vsq >= 0.f)) return harm_host::set_error("loss weights must be >= 0", 4);
    m->loss_w[0] = w_logw;
    m->loss_w[1] = w_vsq;
    return 0;
}

int harm_mlp_fit_norm(harm_mlp *m, const double *feat, const double *targ, const uint8_t *valid, size_t n)
{
    if (!m || !feat || !targ) return harm_host::set_error("null argument", 1);
    if (n == 0) return harm_host::set_error("empty training set", 4);
    DevGuard dg(m->device);
    double *mean = m->normp + NORM_BLOCKS * 11;
    for (int pass = 0; pass < 2; pass++) {
        hipLaunchKernelGGL(k_norm_partials, dim3(NORM_BLOCKS), dim3(256), 0, m->stream, feat, targ, valid, n, pass,
                           mean, m->normp);
        MCHK(hipGetLastError());
        hipLaunchKernelGGL(k_norm_finish, dim3(1), dim3(1), 0, m->stream, m->normp, pass, mean, m->norm);
        MCHK(hipGetLastError());
    }
    MCHK(hipStreamSynchronize(m->stream));
    return 0;
}

int harm_mlp_grad(harm_mlp *m, const float *X, const float *T, const uint8_t *mask, int n, float *grad, double *loss)
{
    if (!m || !X || !T) return harm_host::set_error("null argument", 1);
    int rc;
    if ((rc = check_batch(n))) return rc;
    DevGuard dg(m->device);
    if ((rc = launch_train(m, X, T, mask, n)) || (rc = launch_adam(m, n, nullptr, 0.f, nullptr))) return rc;
    double l = 0.;
    MCHK(hipMemcpyAsync(&l, m->lossd, sizeof(l), hipMemcpyDeviceToHost, m->stream));
    if (grad) MCHK(hipMemcpyAsync(grad, m->grad, MLP_NPARAMS * sizeof(float), hipMemcpyDeviceToHost, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    if (loss) *loss = l;
    return 0;
}

int harm_mlp_train_batch(harm_mlp *m, const float *X, const float *T, const uint8_t *mask, int n, float lr)
{
    if (!m || !X || !T) return harm_host::set_error("null argument", 1);
    int rc;
    if ((rc = check_batch(n))) return rc;
    DevGuard dg(m->device);
    if ((rc = launch_train(m, X, T, mask, n)) || (rc = launch_adam(m, n, m->lossd, lr, nullptr)) || (rc = repack(m)))
        return rc;
    MCHK(hipStreamSynchronize(m->stream));
    return 0;
}

int harm_mlp_train(harm_mlp *m, const double *feat, const double *targ, const uint8_t *valid, size_t n, int batch,
                   int steps, float lr0, float lr1, uint64_t seed, float *loss_trace)
{
    if (!m || !feat || !targ) return harm_host::set_error("null argument", 1);
    if (n == 0) return harm_host::set_error("empty training set", 4);
    int rc;
    if ((rc = check_batch(batch))) return rc;
    if (steps < 0 || !(lr0 > 0.f) || !(lr1 > 0.f)) return harm_host::set_error("bad training schedule", 4);
    DevGuard dg(m->device);
    if ((rc = ensure_ws(m, batch))) return rc;
    Draw d = {feat, targ, valid, nullptr, n, batch, 0};
    if (n <= REC_MAX && (size_t)steps * batch >= n / REC_ROWS && ensure_records(m, n)) {
        hipLaunchKernelGGL(k_records, dim3(cdiv(n, 256)), dim3(256), 0, m->stream, d, m->norm, m->rec);
        MCHK(hipGetLastError());
        d.rec = m->rec;
    }
    auto draw_seed = [&](int s) { return (unsigned long long)seed * 0x100000001B3ull + (unsigned long long)s; };
    std::vector<double> lp(LOSS_KEEP);
    d.seed = draw_seed(0);
    if (steps > 0 && (rc = launch_draw(m, d))) return rc;
    for (int s = 0; s < steps; s++) {
        const double fr = steps > 1 ? (double)s / (steps - 1) : 0.;
        const float lr = (float)(lr0 * std::pow((double)lr1 / lr0, fr));
        d.seed = draw_seed(s + 1);
        const int k = s % LOSS_KEEP;
        if ((rc = launch_train(m, m->X, m->T, m->M, batch)) ||
            (rc = launch_adam(m, batch, m->lossd + k, lr, s + 1 < steps ? &d : nullptr)))
            return rc;
        if (loss_trace && (k == LOSS_KEEP - 1 || s == steps - 1)) {
            MCHK(hipMemcpyAsync(lp.data(), m->lossd, (k + 1) * sizeof(double), hipMemcpyDeviceToHost, m->stream));
            MCHK(hipStreamSynchronize(m->stream));
            for (int i = 0; i <= k; i++) loss_trace[s - k + i] = (float)lp[i];
        }
    }
    if ((rc = repack(m))) return rc;
    MCHK(hipStreamSynchronize(m->stream));
    return 0;
}

int harm_mlp_forward(harm_mlp *m, const float *X, float *Y, int n, int bf16)
{
    if (!m || !X || !Y) return harm_host::set_error("null argument", 1);
    int rc;
    if ((rc = check_batch(n))) return rc;
    DevGuard dg(m->device);
    if (bf16) {
        hipLaunchKernelGGL(k_forward_bf16, dim3(cdiv(n, 256)), dim3(256), 0, m->stream, harm_mlp_view(m), X, Y, n);
        MCHK(hipGetLastError());
    } else {
        if ((rc = launch_forward(m, X, Y, n))) return rc;
    }
    MCHK(hipStreamSynchronize(m->stream));
    return 0;
}

int harm_mlp_seed(harm_mlp *m, const double *U, const double *gcov, const double *gcon, const double *gdet, size_t n,
                  double *feat, double *W0, double *vsq0, void *stream)
{
    if (!m || !U || !gcov || !gcon || !gdet) return harm_host::set_error("null argument", 1);
    if (n == 0) return 0;
    if (n > ((size_t)1 << 31)) return harm_host::set_error("batch too large", 4);
    DevGuard dg(m->device);
    hipStream_t st = stream ? (hipStream_t)stream : m->stream;
    hipLaunchKernelGGL(k_seed, dim3(cdiv(n, 256)), dim3(256), 0, st, harm_mlp_view(m), U, gcov, gcon, gdet, n, feat,
                       W0, vsq0);
    MCHK(hipGetLastError());
    MCHK(hipStreamSynchronize(st));
    return 0;
}

int harm_mlp_pairs(const double *U, const double *gcov, const double *gcon, const double *gdet, const double *prim,
                   const int8_t *ret, size_t n, double gam, double *feat, double *targ, uint8_t *valid, void *stream)
{
    if (!U || !gcov || !gcon || !gdet || !prim || !ret || !feat || !targ || !valid)
        return harm_host::set_error("null argument", 1);
    if (n == 0) return 0;
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(k_pairs, dim3(cdiv(n, 256)), dim3(256), 0, st, U, gcov, gcon, gdet, prim, ret, n, gam, feat,
                       targ, valid);
    MCHK(hipGetLastError());
    MCHK(hipStreamSynchronize(st));
    return 0;
}

}  // extern "C"
