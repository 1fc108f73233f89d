// cts_mlp.hip -- training and inference of the field surrogate (gfx950).
//
// The two 64x64 products of every forward and backward pass run on the
// bf16 matrix cores (v_mfma_f32_16x16x32_bf16, FP32 accumulate) with each
// operand split into a bf16 high and low part (three products per tile), so
// the products carry ~16 significant bits; the 3-input first layer, the
// 2-output last layer and the activations are FP32 vector code.
//
// MFMA 16x16x32 operand layout (one wave, lane l):
//   A (16 x 32, row-major):  row l % 16, columns 8 (l / 16) .. +7
//   B (32 x 16):             column l % 16, rows 8 (l / 16) .. +7
//   D (16 x 16):             rows 4 (l / 16) + t, column l % 16, t = 0..3
#include "cts_internal.hpp"
#include "cts_mlp.hpp"

namespace cts {

// ---------------------------------------------------------------- samples
// Training / validation samples: |u|, |v| uniform in (0, 6], r log-uniform
// in [0.02, 1] from Philox4x32-10 (key = seed, counter = {i, 0, 0, tag});
// the field is the FP64 Bassetti-Erskine path (sigma_x = 1, sigma_y = r).
// Each record: a0 a1 a2 t0 t1 with t = log(G / (u b)) (see cts_mlp.hpp).
__global__ void __launch_bounds__(256)
k_mlp_samples(int64_t n, uint64_t seed, uint32_t tag, float *out, double *exact)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const u32x4 o = philox4x32_10((uint32_t)i, (uint32_t)(i >> 32), 0u, tag, (uint32_t)seed,
                                  (uint32_t)(seed >> 32));
    // |u|, |v| >= kSurZero / 2 keeps every sample off the zero-field branch
    const double lo = 0.5 * kSurZero;
    const double au = lo + (kSurUMax - lo) * (((double)(o.v[0] >> 8) + 0.5) * 0x1p-24);
    const double av = lo + (kSurUMax - lo) * (((double)(o.v[1] >> 8) + 0.5) * 0x1p-24);
    const double r = exp(log(kSurRMin) * (1.0 - ((double)(o.v[2] >> 8) + 0.5) * 0x1p-24));
    double gx, gy;
    ion_field(au, av * r, 1.0, r, gx, gy);
    float a[3];
    sur_features(au, av, r, a);
    float bx, by;
    sur_envelope((float)au, (float)av, (float)r, bx, by);
    float *rec = out + i * 5;
    rec[0] = a[0];
    rec[1] = a[1];
    rec[2] = a[2];
    rec[3] = (float)log(gx / (au * (double)bx));
    rec[4] = (float)log(gy / (av * (double)by));
    if (exact) {
        exact[i * 5 + 0] = au;
        exact[i * 5 + 1] = av;
        exact[i * 5 + 2] = r;
        exact[i * 5 + 3] = gx;
        exact[i * 5 + 4] = gy;
    }
}

// ------------------------------------------------------------- training
// Gradient of the mean squared error of the normalized targets.  A block of
// four waves runs `chunks` batches of 64 samples and writes its partial
// gradient (+ loss) to part[block].  Each wave takes 16 samples of a batch
// through the network and back; then the sums over the batch's 64 samples are
// shared out: every wave forms a quarter of dW2 on the matrix cores and one
// or two of the per-feature sums (lane = feature, samples in order).
//
// Register layouts follow the MFMA operands (lane l: lr = l % 16, lg = l / 16):
//   rows   A operand: sample lr, features 32 kb + 8 lg + i
//   cols   result: samples 4 lg + t, feature 16 fb + lr
// H1 is computed in both (three multiply-adds and a GELU per element, and the
// cols need GELU' anyway), dZ2 passes from cols to rows through LDS, and the
// split weights of both products stay in registers.
//
// What it is bound by: the chain of a batch (record gather, two layers, the
// sums in order) on one or two waves per SIMD.  One wave per 64-sample batch
// with every operand staged in 145 KB of LDS, one wave on a compute unit, took
// 126 us for 512 blocks of two batches; this takes 33 us (two blocks on a
// compute unit, each with its two batches one after the other; 256 blocks of
// one batch 18) and gives the same gradients, since every sum keeps its order.
// With the waves' sums joined only once, over 32 samples each, 24 us, but the
// weights of a long training run drift from the others'.
struct MlpTrainParams {
    const float *params;    // kMlpParams
    const float *samples;   // [n][5]
    int64_t n;
    float *part;            // [grid][kMlpParams + 1]
    float norm[4];          // mu_x, s_x, mu_y, s_y of the targets
    float inv_batch;
    uint64_t seed;
    uint32_t step;
    int32_t chunks;
    int32_t random;         // 0: samples taken in order (gradient checks)
};

constexpr int kTrainBlock = 256;
constexpr int kRow = 68;  // pitch of a row of 64 dwords in LDS

// order between a wave's own LDS writes and reads
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__global__ void __launch_bounds__(kTrainBlock, 2)
k_mlp_train(MlpTrainParams P)
{
#pragma clang fp contract(fast)
    // the operands of dW2: dZ2^T[n][s] and H1^T[k][s], split; W2 is staged in
    // their place at the start
    __shared__ __attribute__((aligned(16))) __bf16 tr[4][64 * kPb];
    __bf16 *d2th = tr[0], *d2tl = tr[1], *h1th = tr[2], *h1tl = tr[3];
    __shared__ __attribute__((aligned(16))) uint32_t dzs[64 * kRow];  // dZ2[s][n] (hi, lo), then dZ1[s][k]
    __shared__ __attribute__((aligned(16))) float h2s[64 * kRow];     // H2[s][n]
    __shared__ __attribute__((aligned(16))) float recs[64 * 8];       // a0 a1 a2 valid y0 y1 - -
    __shared__ float dos[64 * 2];                                     // d loss / d output
    __shared__ float w1s[64 * 4], w3s[64 * 4];                        // W1[k], b1[k]; b2[n], W3[0][n], W3[1][n]
    const int tid = threadIdx.x, l = tid & 63, wv = tid >> 6;
    const int lr = l & 15, lg = l >> 4;
    const float *W = P.params;
    float *dz1s = reinterpret_cast<float *>(dzs);

    // the record of sample gid (lanes below 16 of each wave: 16 wv + l)
    float rc[5] = {0, 0, 0, 0, 0};
    bool valid = false;
    auto fetch = [&](int c) {
        const int64_t gid = ((int64_t)blockIdx.x * P.chunks + c) * 64 + 16 * wv + l;
        int64_t idx;
        if (P.random) {
            const u32x4 o = philox4x32_10((uint32_t)gid, (uint32_t)(gid >> 32), P.step, 0x4d4c5054u,
                                          (uint32_t)P.seed, (uint32_t)(P.seed >> 32));
            idx = (int64_t)(((uint64_t)o.v[0] * (uint64_t)P.n) >> 32);
        } else {
            idx = gid < P.n ? gid : P.n - 1;
        }
        valid = P.random || gid < P.n;
        const float *rec = P.samples + idx * 5;
#pragma unroll
        for (int j = 0; j < 5; j++) rc[j] = rec[j];
    };
    if (l < 16) fetch(0);

    // the weights: W2 through LDS into this lane's operands of H1 W2^T and
    // dZ2 W2 (feature 16 fb + lr, 8 of the other index)
    float *w2s = reinterpret_cast<float *>(&tr[0][0]);
    for (int i = tid; i < 4096; i += kTrainBlock) w2s[(i >> 6) * kRow + (i & 63)] = W[MP_W2 + i];
    if (tid < 64) {
        for (int j = 0; j < 3; j++) w1s[4 * tid + j] = W[MP_W1 + 3 * tid + j];
        w1s[4 * tid + 3] = W[MP_B1 + tid];
        w3s[4 * tid] = W[MP_B2 + tid];
        w3s[4 * tid + 1] = W[MP_W3 + tid];
        w3s[4 * tid + 2] = W[MP_W3 + 64 + tid];
        w3s[4 * tid + 3] = 0.0f;
    }
    __syncthreads();
    v8bf w2h[4][2], w2l[4][2], w2th[4][2], w2tl[4][2];
#pragma unroll
    for (int fb = 0; fb < 4; fb++)
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
#pragma unroll
            for (int i = 0; i < 8; i++) {
                __bf16 hi, lo;
                split_bf16(w2s[(16 * fb + lr) * kRow + 32 * kb + 8 * lg + i], hi, lo);
                w2h[fb][kb][i] = hi; w2l[fb][kb][i] = lo;
                split_bf16(w2s[(32 * kb + 8 * lg + i) * kRow + 16 * fb + lr], hi, lo);
                w2th[fb][kb][i] = hi; w2tl[fb][kb][i] = lo;
            }
    __syncthreads();

    const float b3 = W[MP_B3 + (lg & 1)];  // output lg of sample lr (lanes below 32)
    v4f gw2[4];
#pragma unroll
    for (int nb = 0; nb < 4; nb++) gw2[nb] = (v4f){0, 0, 0, 0};
    float s0 = 0, s1 = 0;       // wave 0: dW3, wave 1: db2, wave 2: dW1[0], [1], wave 3: dW1[2], db1
    float gb3 = 0, loss = 0;    // sample lr: db3 of output lg, and the loss (lg = 0)

    for (int c = 0; c < P.chunks; c++) {
        if (l < 16) {
            float *d = recs + (16 * wv + l) * 8;
            d[0] = rc[0]; d[1] = rc[1]; d[2] = rc[2];
            d[3] = valid ? 1.0f : 0.0f;
            d[4] = (rc[3] - P.norm[0]) / P.norm[1];
            d[5] = (rc[4] - P.norm[2]) / P.norm[3];
            if (c + 1 < P.chunks) fetch(c + 1);
        }
        wave_sync();
        // layer 1, rows
        v8bf ah[2], al[2];
        {
            const float4 x = *reinterpret_cast<const float4 *>(recs + (16 * wv + lr) * 8);
#pragma unroll
            for (int kb = 0; kb < 2; kb++)
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const float4 w = *reinterpret_cast<const float4 *>(&w1s[4 * (32 * kb + 8 * lg + i)]);
                    const float z = w.w + w.x * x.x + w.y * x.y + w.z * x.z;
                    __bf16 hi, lo;
                    split_bf16(gelu_only(z), hi, lo);
                    ah[kb][i] = hi;
                    al[kb][i] = lo;
                }
        }
        // layer 2, cols: Z2[s][n] = sum_k H1[s][k] W2[n][k]
        float dg2[4][4];
#pragma unroll
        for (int fb = 0; fb < 4; fb++) {
            v4f acc = {0, 0, 0, 0};
#pragma unroll
            for (int kb = 0; kb < 2; kb++) acc = mfma3(ah[kb], al[kb], w2h[fb][kb], w2l[fb][kb], acc);
            const float b2 = w3s[4 * (16 * fb + lr)];
#pragma unroll
            for (int t = 0; t < 4; t++)
                h2s[(16 * wv + 4 * lg + t) * kRow + 16 * fb + lr] = gelu_f(acc[t] + b2, dg2[fb][t]);
        }
        wave_sync();
        // the outputs, features in order (lane = sample lr, output lg), the
        // loss and its derivative
        if (l < 32) {
            float o = b3;
            const float *h = h2s + (16 * wv + lr) * kRow;
            for (int n = 0; n < 64; n += 4) {
                const float4 v = *reinterpret_cast<const float4 *>(h + n);
                o += w3s[4 * n + 1 + lg] * v.x;
                o += w3s[4 * n + 5 + lg] * v.y;
                o += w3s[4 * n + 9 + lg] * v.z;
                o += w3s[4 * n + 13 + lg] * v.w;
            }
            const float *d = recs + (16 * wv + lr) * 8;
            const float e = d[3] != 0.0f ? o - d[4 + lg] : 0.0f;
            dos[2 * (16 * wv + lr) + lg] = 2.0f * e * P.inv_batch;
            gb3 = __builtin_fmaf(2.0f * e, P.inv_batch, gb3);
            loss += e * e;
        }
        wave_sync();
        // dZ2, cols: to LDS as rows (for dH1) and transposed (for dW2)
        float dt[4][2];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            dt[t][0] = dos[2 * (16 * wv + 4 * lg + t)];
            dt[t][1] = dos[2 * (16 * wv + 4 * lg + t) + 1];
        }
#pragma unroll
        for (int fb = 0; fb < 4; fb++) {
            const float4 e = *reinterpret_cast<const float4 *>(&w3s[4 * (16 * fb + lr)]);
            v4bf vh, vl;
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const float dz = (dt[t][0] * e.y + dt[t][1] * e.z) * dg2[fb][t];
                __bf16 hi, lo;
                split_bf16(dz, hi, lo);
                vh[t] = hi;
                vl[t] = lo;
                dzs[(16 * wv + 4 * lg + t) * kRow + 16 * fb + lr] =
                    (uint32_t)__builtin_bit_cast(uint16_t, hi) | ((uint32_t)__builtin_bit_cast(uint16_t, lo) << 16);
            }
            *reinterpret_cast<v4bf *>(&d2th[(16 * fb + lr) * kPb + 16 * wv + 4 * lg]) = vh;
            *reinterpret_cast<v4bf *>(&d2tl[(16 * fb + lr) * kPb + 16 * wv + 4 * lg]) = vl;
        }
        wave_sync();
#pragma unroll
        for (int kb = 0; kb < 2; kb++) {
            const uint4 *q = reinterpret_cast<const uint4 *>(&dzs[(16 * wv + lr) * kRow + 32 * kb + 8 * lg]);
            const uint4 q0 = q[0], q1 = q[1];
            const uint32_t w[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
#pragma unroll
            for (int i = 0; i < 8; i++) {
                ah[kb][i] = __builtin_bit_cast(__bf16, (uint16_t)(w[i] & 0xffffu));
                al[kb][i] = __builtin_bit_cast(__bf16, (uint16_t)(w[i] >> 16));
            }
        }
        wave_sync();
        // H1 again, cols; dH1 = dZ2 W2 -> dZ1 = dH1 GELU'(z1)
        float4 xt[4];
#pragma unroll
        for (int t = 0; t < 4; t++) xt[t] = *reinterpret_cast<const float4 *>(recs + (16 * wv + 4 * lg + t) * 8);
#pragma unroll
        for (int fb = 0; fb < 4; fb++) {
            v4f acc = {0, 0, 0, 0};
#pragma unroll
            for (int kb = 0; kb < 2; kb++) acc = mfma3(ah[kb], al[kb], w2th[fb][kb], w2tl[fb][kb], acc);
            const float4 w = *reinterpret_cast<const float4 *>(&w1s[4 * (16 * fb + lr)]);
            v4bf vh, vl;
#pragma unroll
            for (int t = 0; t < 4; t++) {
                float dg;
                const float z = w.w + w.x * xt[t].x + w.y * xt[t].y + w.z * xt[t].z;
                __bf16 hi, lo;
                split_bf16(gelu_f(z, dg), hi, lo);
                vh[t] = hi;
                vl[t] = lo;
                dz1s[(16 * wv + 4 * lg + t) * kRow + 16 * fb + lr] = acc[t] * dg;
            }
            *reinterpret_cast<v4bf *>(&h1th[(16 * fb + lr) * kPb + 16 * wv + 4 * lg]) = vh;
            *reinterpret_cast<v4bf *>(&h1tl[(16 * fb + lr) * kPb + 16 * wv + 4 * lg]) = vl;
        }
        __syncthreads();
        // sums over the batch: dW2 += dZ2^T H1, rows n of block wv, ...
#pragma unroll
        for (int nb = 0; nb < 4; nb++)
#pragma unroll
            for (int kb = 0; kb < 2; kb++) {
                const int ao = (16 * wv + lr) * kPb + 32 * kb + 8 * lg, bo = (16 * nb + lr) * kPb + 32 * kb + 8 * lg;
                gw2[nb] = mfma3(frag(d2th + ao), frag(d2tl + ao), frag(h1th + bo), frag(h1tl + bo), gw2[nb]);
            }
        // ... and the per-feature sums (lane = feature), samples in order
        if (wv == 0) {
#pragma unroll 8
            for (int s = 0; s < 64; s++) {
                const float h = h2s[s * kRow + l];
                s0 += dos[2 * s] * h;
                s1 += dos[2 * s + 1] * h;
            }
        } else if (wv == 1) {
#pragma unroll 4
            for (int s = 0; s < 64; s += 4) {
                const v4bf vh = *reinterpret_cast<const v4bf *>(&d2th[l * kPb + s]);
                const v4bf vl = *reinterpret_cast<const v4bf *>(&d2tl[l * kPb + s]);
#pragma unroll
                for (int t = 0; t < 4; t++) s0 += (float)vh[t] + (float)vl[t];
            }
        } else if (wv == 2) {
#pragma unroll 8
            for (int s = 0; s < 64; s++) {
                const float dz = dz1s[s * kRow + l];
                s0 += dz * recs[8 * s];
                s1 += dz * recs[8 * s + 1];
            }
        } else {
#pragma unroll 8
            for (int s = 0; s < 64; s++) {
                const float dz = dz1s[s * kRow + l];
                s0 += dz * recs[8 * s + 2];
                s1 += dz;
            }
        }
        __syncthreads();
    }
    float *out = P.part + (int64_t)blockIdx.x * (kMlpParams + 1);
#pragma unroll
    for (int nb = 0; nb < 4; nb++)
#pragma unroll
        for (int t = 0; t < 4; t++) out[MP_W2 + (16 * wv + 4 * lg + t) * 64 + 16 * nb + lr] = gw2[nb][t];
    if (wv == 0) {
        out[MP_W3 + l] = s0;
        out[MP_W3 + 64 + l] = s1;
    } else if (wv == 1) {
        out[MP_B2 + l] = s0;
    } else if (wv == 2) {
        out[MP_W1 + 3 * l] = s0;
        out[MP_W1 + 3 * l + 1] = s1;
    } else {
        out[MP_W1 + 3 * l + 2] = s0;
        out[MP_B1 + l] = s1;
    }
    // db3 and the loss: sums over the samples
    if (l < 32) {
        dos[2 * (16 * wv + lr) + lg] = gb3;
        recs[8 * (16 * wv + lr) + lg] = loss;
    }
    __syncthreads();
    if (wv == 0) {
        float a0 = dos[2 * l], a1 = dos[2 * l + 1], sl = recs[8 * l] + recs[8 * l + 1];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            a0 += __shfl_xor(a0, o, 64);
            a1 += __shfl_xor(a1, o, 64);
            sl += __shfl_xor(sl, o, 64);
        }
        if (l == 0) {
            out[MP_B3] = a0;
            out[MP_B3 + 1] = a1;
            out[kMlpParams] = sl;
        }
    }
}

// Sum of the workgroup partials (in order) and one Adam step: a block takes 64
// parameters; its waves bring up to kAdamTile partials to LDS at once, then
// the first one adds them.  (One thread per parameter walking 512 partials in
// memory took 118 us, this 6.7.)
constexpr int kAdamTile = 512;
__global__ void __launch_bounds__(kAdamBlock)
k_mlp_adam(float *params, float *m, float *v, const float *part, int nwg, float lr, float b1, float b2,
           float eps, float bc1, float bc2, float *grad_out, float *loss_out)
{
    __shared__ float tile[kAdamTile][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int p = blockIdx.x * 64 + lane;
    const bool in = p <= kMlpParams, mine = wv == 0 && p < kMlpParams;
    float m0 = 0, v0 = 0, p0 = 0;
    if (mine) { m0 = m[p]; v0 = v[p]; p0 = params[p]; }
    float g = 0.0f;
    for (int w0 = 0; w0 < nwg; w0 += kAdamTile) {
        constexpr int nw = kAdamBlock / 64, per = kAdamTile / nw;
        float x[per];
#pragma unroll
        for (int j = 0; j < per; j++) {
            const int w = w0 + wv + j * nw;
            x[j] = (in && w < nwg) ? part[(int64_t)w * (kMlpParams + 1) + p] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < per; j++) tile[wv + j * nw][lane] = x[j];
        __syncthreads();
        if (wv == 0) {
            const int n = nwg - w0 < kAdamTile ? nwg - w0 : kAdamTile;
            int j = 0;
            for (; j + 32 <= n; j += 32) {
                float y[32];
#pragma unroll
                for (int u = 0; u < 32; u++) y[u] = tile[j + u][lane];
#pragma unroll
                for (int u = 0; u < 32; u++) g += y[u];
            }
            for (; j < n; j++) g += tile[j][lane];
        }
        __syncthreads();
    }
    if (wv != 0 || p > kMlpParams) return;
    if (p == kMlpParams) {
        if (loss_out) *loss_out = g;
        return;
    }
    if (grad_out) grad_out[p] = g;
    if (lr == 0.0f) return;
    const float mm = b1 * m0 + (1.0f - b1) * g;
    const float vv = b2 * v0 + (1.0f - b2) * g * g;
    m[p] = mm;
    v[p] = vv;
    params[p] = p0 - lr * (mm / bc1) / (sqrtf(vv / bc2) + eps);
}

// Raw network outputs for n feature vectors (tests and validation).
__global__ void __launch_bounds__(256)
k_mlp_eval(const float *W, const float *feat, int64_t n, int32_t stride, float *out)
{
    __shared__ __attribute__((aligned(16))) MlpLds L;
    load_mlp_lds(L, W, threadIdx.x, blockDim.x);
    __syncthreads();
    for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < n; base += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = base + threadIdx.x;
        float a0 = 0, a1 = 0, a2 = 0;
        if (i < n) {
            a0 = feat[i * stride];
            a1 = feat[i * stride + 1];
            a2 = feat[i * stride + 2];
        }
        float o0, o1;
        mlp_forward_wave(L, a0, a1, a2, o0, o1);  // the whole wave takes part
        if (i < n) {
            out[2 * i] = o0;
            out[2 * i + 1] = o1;
        }
    }
}

// Field error of the surrogate against the exact FP64 values in
// exact[n][5] = |u| |v| r Gx Gy: per point |G_sur - G| / |G| (vector norm),
// written to err[n].
__global__ void __launch_bounds__(256)
k_mlp_field_error(const float *W, const double *exact, int64_t n, float4 norm, double *err)
{
    __shared__ __attribute__((aligned(16))) MlpLds L;
    load_mlp_lds(L, W, threadIdx.x, blockDim.x);
    __syncthreads();
    for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < n; base += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = base + threadIdx.x;
        double au = 1, av = 1, r = 1;
        if (i < n) { au = exact[i * 5]; av = exact[i * 5 + 1]; r = exact[i * 5 + 2]; }
        float a[3];
        sur_features(au, av, r, a);
        float o0, o1;
        mlp_forward_wave(L, a[0], a[1], a[2], o0, o1);
        if (i < n) {
            float bx, by;
            sur_envelope((float)au, (float)av, (float)r, bx, by);
            const double gx = au * (double)bx * exp((double)(norm.x + norm.y * o0));
            const double gy = av * (double)by * exp((double)(norm.z + norm.w * o1));
            const double ex = exact[i * 5 + 3], ey = exact[i * 5 + 4];
            err[i] = sqrt(((gx - ex) * (gx - ex) + (gy - ey) * (gy - ey)) / (ex * ex + ey * ey));
        }
    }
}

hipError_t launch_mlp_samples(int64_t n, uint64_t seed, uint32_t tag, float *out, double *exact, hipStream_t st)
{
    hipLaunchKernelGGL(k_mlp_samples, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, seed, tag, out, exact);
    return hipGetLastError();
}

hipError_t launch_mlp_train(const float *params, const float *samples, int64_t n, float *part, const float norm[4],
                            float inv_batch, uint64_t seed, uint32_t step, int chunks, int random, int nwg,
                            hipStream_t st)
{
    MlpTrainParams P;
    P.params = params; P.samples = samples; P.n = n; P.part = part;
    for (int i = 0; i < 4; i++) P.norm[i] = norm[i];
    P.inv_batch = inv_batch; P.seed = seed; P.step = step; P.chunks = chunks; P.random = random;
    hipLaunchKernelGGL(k_mlp_train, dim3(nwg), dim3(kTrainBlock), 0, st, P);
    return hipGetLastError();
}

hipError_t launch_mlp_adam(float *params, float *m, float *v, const float *part, int nwg, float lr, float b1,
                           float b2, float eps, float bc1, float bc2, float *grad_out, float *loss_out,
                           hipStream_t st)
{
    hipLaunchKernelGGL(k_mlp_adam, dim3(kMlpParams / 64 + 1), dim3(kAdamBlock), 0, st, params, m, v, part,
                       nwg, lr, b1, b2, eps, bc1, bc2, grad_out, loss_out);
    return hipGetLastError();
}

hipError_t launch_mlp_eval(const float *W, const float *feat, int64_t n, int stride, float *out, hipStream_t st)
{
    int64_t nwg = (n + 255) / 256;
    if (nwg > 2048) nwg = 2048;
    if (nwg < 1) nwg = 1;
    hipLaunchKernelGGL(k_mlp_eval, dim3((unsigned)nwg), dim3(256), 0, st, W, feat, n, stride, out);
    return hipGetLastError();
}

hipError_t launch_mlp_field_error(const float *W, const double *exact, int64_t n, const float norm[4], double *err,
                                  hipStream_t st)
{
    int64_t nwg = (n + 255) / 256;
    if (nwg > 2048) nwg = 2048;
    if (nwg < 1) nwg = 1;
    const float4 nm = make_float4(norm[0], norm[1], norm[2], norm[3]);
    hipLaunchKernelGGL(k_mlp_field_error, dim3((unsigned)nwg), dim3(256), 0, st, W, exact, n, nm, err);
    return hipGetLastError();
}

hipError_t upload_faddeeva_tables_mlp(const FadTables &t)
{
    return hipMemcpyToSymbol(HIP_SYMBOL(c_weid), t.weid, kFadConst * sizeof(double));
}

}  // namespace cts
