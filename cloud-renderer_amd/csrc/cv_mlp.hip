// Far-field MLP kernels: batched inference, training step (forward with saved
// activations, backward, per-workgroup gradient partials), deterministic
// reduction + Adam, and weight packing for the matrix cores.
//
// Training loss per row (weight w = remaining transmittance 1 - a_k):
//     w^2 * sum_c (y_c - t_c)^2   +   (y_4 - e)^2,
//     e = max_c |clamp(y_c, 0, 1) - t_c|   (treated as a constant),
// averaged over the batch.  The first term is the squared error the far
// field adds to the fragment colour; the second trains the error estimate
// that decides the fallback.
#include "cv_mlp.h"
#include "cv_mlp_launch.h"

namespace cv {

// ---------------------------------------------------------------------------
// batched inference: rows X[n][17] -> Y[n][5], one wave per 32 rows
//
// Bound by the GELUs (128 per lane and tile, two of their eight instructions at
// a fraction of the rate) and, for fewer rows than fill the device, by the
// chain of layers: 32 rows per wave are one chain and twice the waves of 64.
// The 544 features of a tile are contiguous, so the loads are whole lines.
// ---------------------------------------------------------------------------
constexpr int kFwdWaves = 4;
__global__ void __launch_bounds__(64 * kFwdWaves) k_mlp_forward(MlpDev w, const float* __restrict__ X, int n,
                                                                float* __restrict__ Y) {
    __shared__ __align__(16) uint16_t xs[kFwdWaves][32 * kMlpInPad];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int row0 = (blockIdx.x * kFwdWaves + wave) * 32;
    uint16_t* tile = xs[wave];
    const size_t base = (size_t)row0 * kMlpIn, end = (size_t)n * kMlpIn;
#pragma unroll
    for (int q = 0; q < 8; ++q) ((uint32_t*)tile)[q * 64 + lane] = 0u;  // the pads, and rows past n
    __syncthreads();
#pragma unroll
    for (int q = 0; q < (32 * kMlpIn + 63) / 64; ++q) {
        const int i = q * 64 + lane;
        if (i < 32 * kMlpIn && base + i < end) tile[(i / kMlpIn) * kMlpInPad + i % kMlpIn] = (uint16_t)f2bf_bits(X[base + i]);
    }
    __syncthreads();
    if (row0 >= n) return;
    const cv_f32x16 y = mlp_forward_tile(w, tile, 0, lane);
    // outputs 0..3 in registers 0..3 of half 0, output 4 in register 0 of half 1
    const int row = row0 + (lane & 31);
    if (row >= n) return;
    float* o = Y + (size_t)row * kMlpOut;
    if (lane < 32) {
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = y[q];
    } else {
        o[4] = y[0];
    }
}

// ---------------------------------------------------------------------------
// training: a workgroup per 64 rows; writes every parameter's partial gradient
// of this workgroup (no atomics) and its partial loss
//
// Four waves: wave (mt, nt) holds output units 32 mt .. + 31 of rows
// 32 nt .. + 31 of every layer.  A wave's accumulators are half of the next
// layer's B operand for its rows; the halves are exchanged through LDS (two
// 16-byte words per lane and layer).  Z stays in the waves' registers for the
// backward pass.  The work is a chain of layers, so what counts is how little
// of it one wave does and that 16384 rows are one workgroup per CU: with one
// wave per 64 rows a step took 105 us of this kernel, of which the matrix
// instructions were 3.
// ---------------------------------------------------------------------------
struct TrainLds {
    uint16_t xs[64 * kMlpInPad];        // layer-0 input, row-major
    uint16_t hs[5][64 * 64];            // H_l as [unit][row] (l = 0 uses 32 units)
    uint16_t gs[64 * 64];               // dL/dZ_l as [unit][row]
    cv_u32x4 xch[2][2][4][64];          // B operands [buffer][nt][step][lane]
    float fx[2][2][8][64];              // [mt][from nt]: the half of a wave's gradients whose row sums the other takes
    float loss[64];
};

__device__ __forceinline__ cv_u32x4 lds_row8(const uint16_t* base) { return *(const cv_u32x4*)base; }

template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
// sum over the 32 lanes of each half (rows of the batch): the butterfly over
// lane distances 1, 2, 4, 8, 16, on lane permutes inside a row of 16 (mirrors
// serve for 4 and 8, where the groups they swap already hold equal sums)
__device__ __forceinline__ float half_sum(float v) {
    v = dpp_add<0xB1>(v);   // quad_perm 1 0 3 2
    v = dpp_add<0x4E>(v);   // quad_perm 2 3 0 1
    v = dpp_add<0x141>(v);  // row_half_mirror
    v = dpp_add<0x140>(v);  // row_mirror
    return v + __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x401F));  // lane ^ 16
}

// the wave's gradients (accumulator registers) into LDS: bf16 for the weight
// gradients, the next layer's B operand, and the half of the bias terms that
// the wave of the other rows sums
__device__ __forceinline__ void store_grad(const cv_f32x16& g, TrainLds& S, int buf, int mt, int nt, int lane) {
    const int h = lane >> 5, c = lane & 31;
#pragma unroll
    for (int j = 0; j < 16; ++j) S.gs[(32 * mt + mlp_crow(h, j)) * 64 + 32 * nt + c] = (uint16_t)f2bf_bits(g[j]);
#pragma unroll
    for (int s = 0; s < 2; ++s) S.xch[buf][nt][2 * mt + s][lane] = chain_b(g, s);
#pragma unroll
    for (int q = 0; q < 8; ++q) S.fx[mt][nt][q][lane] = nt == 0 ? g[8 + q] : g[q];
}
// bias gradients: registers 0..7 by the wave of rows 0..31, 8..15 by the other
__device__ __forceinline__ void bias_grad(const cv_f32x16& g, int l, const TrainLds& S, float* __restrict__ part,
                                          int mt, int nt, int lane) {
    const int h = lane >> 5, c = lane & 31;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const float own = nt == 0 ? g[q] : g[8 + q];
        const float sm = half_sum(own + S.fx[mt][nt ^ 1][q][lane]);
        const int unit = 32 * mt + (nt == 0 ? mlp_crow(h, q) : mlp_crow(h, 8 + q));
        if (c == 0 && unit < mlp_out(l)) part[mlp_boff(l) + unit] = sm;
    }
}

// dW_l = G H_l^T over the 64 rows (K = rows), outputs 32 mt .., inputs
// 32 nt .., written to the partials
__device__ __forceinline__ void weight_grad(int l, const TrainLds& S, float* __restrict__ part, int mt, int nt,
                                            int lane) {
    const int h = lane >> 5, c = lane & 31;
    const int nin = mlp_in(l), nout = mlp_out(l);
    cv_f32x16 acc;
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = 0.0f;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        cv_u32x4 a = lds_row8(S.gs + (32 * mt + c) * 64 + 16 * s + 8 * h);
        cv_u32x4 b = lds_row8(S.hs[l] + (32 * nt + c) * 64 + 16 * s + 8 * h);
        acc = mfma_bf16(a, b, acc);
    }
    const int in = 32 * nt + c;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int out = 32 * mt + mlp_crow(h, j);
        if (out < nout && in < nin) part[mlp_woff(l) + out * nin + in] = acc[j];
    }
}

// dH_l = W_l^T G_l (layers 1..4), then G_{l-1} = dH_l * GELU'(Z_{l-1})
template <int KS>
__device__ __forceinline__ void back_layer(const MlpDev& w, int l, const TrainLds& S, int buf, const cv_f32x16& z,
                                           cv_f32x16& g, int mt, int nt, int lane) {
    cv_f32x16 d;
#pragma unroll
    for (int j = 0; j < 16; ++j) d[j] = 0.0f;
#pragma unroll
    for (int s = 0; s < KS; ++s)
        d = mfma_bf16(load_blk(w.bwd, mlp_bblk0(l) + mt * KS + s, lane), S.xch[buf][nt][s][lane], d);
#pragma unroll
    for (int j = 0; j < 16; ++j) g[j] = d[j] * gelu_grad(z[j]);
}

__global__ void __launch_bounds__(256) k_mlp_train(MlpDev w, const float* __restrict__ X, const float* __restrict__ T,
                                                   int n, float inv_n, float* __restrict__ partial,
                                                   float* __restrict__ loss_part) {
    __shared__ __align__(16) TrainLds S;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int mt = wave >> 1, nt = wave & 1;
    const int h = lane >> 5, c = lane & 31;
    const int row0 = blockIdx.x * 64;
    float* part = partial + (size_t)blockIdx.x * kMlpParamsPad;
    {
        // features 8 wave .. + 7 of row `lane`
        const int row = row0 + lane, k0 = 8 * wave;
        float v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = row < n && k0 + q < kMlpIn ? X[(size_t)row * kMlpIn + k0 + q] : 0.0f;
        cv_u32x4 b;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            b[q] = pack_bf2(v[2 * q], v[2 * q + 1]);
            S.hs[0][(k0 + 2 * q) * 64 + lane] = (uint16_t)b[q];
            S.hs[0][(k0 + 2 * q + 1) * 64 + lane] = (uint16_t)(b[q] >> 16);
        }
        *(cv_u32x4*)(S.xs + lane * kMlpInPad + k0) = b;
    }
    __syncthreads();

    // ---- forward, keeping Z_l and storing H_{l+1}
    cv_f32x16 z[4];
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        const int KS = l == 0 ? 2 : 4;
        cv_f32x16 a = bias_init(w.bias, mlp_bpad0(l) + 32 * mt, h);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const cv_u32x4 B = l == 0 ? x_operand(S.xs, 32 * nt + c, s, h) : S.xch[l & 1][nt][s][lane];
            a = mfma_bf16(load_blk(w.fwd, mlp_fblk0(l) + mt * KS + s, lane), B, a);
        }
        z[l] = a;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            a[j] = gelu_f(a[j]);
            S.hs[l + 1][(32 * mt + mlp_crow(h, j)) * 64 + 32 * nt + c] = (uint16_t)f2bf_bits(a[j]);
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) S.xch[(l + 1) & 1][nt][2 * mt + s][lane] = chain_b(a, s);
        __syncthreads();
    }

    // ---- output layer and loss gradient (the waves of units 0..31), in
    // accumulator layout: rows 0..3 in registers 0..3 of half 0, row 4 in
    // register 0 of half 1
    cv_f32x16 g;
#pragma unroll
    for (int j = 0; j < 16; ++j) g[j] = 0.0f;
    float d4[4] = {0.0f, 0.0f, 0.0f, 0.0f}, w2 = 0.0f;  // loss terms w2 d4^2
    if (mt == 0) {
        cv_f32x16 y = bias_init(w.bias, mlp_bpad0(4), h);
#pragma unroll
        for (int s = 0; s < 4; ++s) y = mfma_bf16(load_blk(w.fwd, mlp_fblk0(4) + s, lane), S.xch[0][nt][s][lane], y);
        const int row = row0 + 32 * nt + c;
        const bool valid = row < n;
        float e = 0.0f;
        if (h == 0 && valid) {
            const float* t = T + (size_t)row * kMlpOut;
            w2 = t[4] * t[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                d4[q] = y[q] - t[q];
                e = fmaxf(e, fabsf(fminf(fmaxf(y[q], 0.0f), 1.0f) - t[q]));
            }
        }
        const float e_hi = __shfl(e, c, 64);
        if (valid) {
            if (h == 0) {
#pragma unroll
                for (int q = 0; q < 4; ++q) g[q] = 2.0f * w2 * d4[q] * inv_n;
            } else {
                const float de = y[0] - e_hi;
                g[0] = 2.0f * de * inv_n;
                d4[0] = de;
                w2 = 1.0f;
            }
        }
        if (nt == 0) {
            float lsum = 0.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q) lsum = fmaf(w2 * d4[q], d4[q], lsum);
            S.loss[lane] = lsum;
        }
    }

    // ---- backward
    store_grad(g, S, 1, mt, nt, lane);
    __syncthreads();
    if (wave == 1) {
        // rows 32..63 go on from the sums of rows 0..31
        float lsum = S.loss[lane];
#pragma unroll
        for (int q = 0; q < 4; ++q) lsum = fmaf(w2 * d4[q], d4[q], lsum);
        float tot = lsum;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) tot += __shfl_xor(tot, off, 64);
        if (lane == 0) loss_part[blockIdx.x] = tot * inv_n;
    }
    if (mt == 0) {
        weight_grad(4, S, part, 0, nt, lane);
        bias_grad(g, 4, S, part, mt, nt, lane);
    }
    back_layer<2>(w, 4, S, 1, z[3], g, mt, nt, lane);
    __syncthreads();
#pragma unroll
    for (int l = 3; l >= 1; --l) {
        store_grad(g, S, l & 1, mt, nt, lane);
        __syncthreads();
        weight_grad(l, S, part, mt, nt, lane);
        bias_grad(g, l, S, part, mt, nt, lane);
        back_layer<4>(w, l, S, l & 1, z[l - 1], g, mt, nt, lane);
        __syncthreads();
    }
    store_grad(g, S, 0, mt, nt, lane);
    __syncthreads();
    if (nt == 0) weight_grad(0, S, part, mt, 0, lane);
    bias_grad(g, 0, S, part, mt, nt, lane);
}

// where parameter p's bf16 value goes in the packed blocks (k_mlp_pack's inverse)
__device__ __forceinline__ void pack_param(int p, float v, uint16_t* __restrict__ fwd, uint16_t* __restrict__ bwd,
                                           float* __restrict__ bias) {
    int l = 0;
    while (l < 4 && p >= mlp_woff(l + 1)) ++l;
    if (p >= mlp_boff(l)) {
        bias[mlp_bpad0(l) + p - mlp_boff(l)] = v;
        return;
    }
    const int nin = mlp_in(l), m = (p - mlp_woff(l)) / nin, k = (p - mlp_woff(l)) % nin;
    const uint16_t b = (uint16_t)f2bf_bits(v);
    // slot q of lane half h holds offset 8 (q / 4) + 4 h + q % 4 of its 16-wide step
    auto at = [](int blk, int row, int kk) {
        const int q = ((kk >> 3) << 2) | (kk & 3), h = (kk >> 2) & 1;
        return blk * 512 + (32 * h + (row & 31)) * 8 + q;
    };
    fwd[at(mlp_fblk0(l) + (m >> 5) * (mlp_kpad(l) / 16) + (k >> 4), m, k & 15)] = b;
    if (l > 0) bwd[at(mlp_bblk0(l) + (k >> 5) * (mlp_mpad(l) / 16) + (m >> 4), k, m & 15)] = b;
}

// ---------------------------------------------------------------------------
// gradient reduction (fixed order over workgroups), Adam and the packed weights
// of the next step
//
// 14 MB of partials for 16384 rows: 64 parameters per workgroup spread them
// over 219 CUs; what bounds it is latency.  A workgroup brings kAdamRows
// partials of each parameter into LDS in one round trip, and one wave adds them
// in order from there; the loss partials likewise, a workgroup's own (added by
// readlane they were the longest chain).  10.6 -> 6.7 us at 16384 rows.
// ---------------------------------------------------------------------------
constexpr int kAdamRows = 256;
static_assert(kMlpParamsPad % 4 == 0, "rows are read 16 bytes at a time");
__global__ void __launch_bounds__(256) k_mlp_adam(const float* __restrict__ partial, int nwg,
                                                 const float* __restrict__ loss_part, float* __restrict__ master,
                                                 float* __restrict__ m1, float* __restrict__ m2,
                                                 float* __restrict__ grad_out, float* __restrict__ loss_out,
                                                 AdamStep st, MlpPacked pk) {
    __shared__ __align__(16) float rows[kAdamRows * 64];
    const int tid = threadIdx.x;
    if (blockIdx.x == gridDim.x - 1) {
        // the loss partials, added in order by every thread alike
        float s = 0.0f;
        for (int i0 = 0; i0 < nwg; i0 += 256) {
            rows[tid] = i0 + tid < nwg ? loss_part[i0 + tid] : 0.0f;
            __syncthreads();
            const int m = min(256, nwg - i0);
#pragma unroll 16
            for (int q = 0; q < m; ++q) s += rows[q];
            __syncthreads();
        }
        if (tid == 0 && loss_out) *loss_out = s;
        return;
    }
    // 16 threads a row, 16 bytes each
    const float4* src = (const float4*)(partial + blockIdx.x * 64) + (tid & 15);
    const int r = tid >> 4;
    const bool in_row = blockIdx.x * 64 + 4 * (tid & 15) < kMlpParamsPad;
    float gsum = 0.0f;
    for (int i0 = 0; i0 < nwg; i0 += kAdamRows) {
        float4 v[kAdamRows / 16];
#pragma unroll
        for (int q = 0; q < kAdamRows / 16; ++q) {
            const int i = i0 + r + 16 * q;
            v[q] = in_row && i < nwg ? src[(size_t)i * (kMlpParamsPad / 4)] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
#pragma unroll
        for (int q = 0; q < kAdamRows / 16; ++q) ((float4*)rows)[(r + 16 * q) * 16 + (tid & 15)] = v[q];
        __syncthreads();
        if (tid < 64) {
            const int m = min(kAdamRows, nwg - i0);
#pragma unroll 16
            for (int k = 0; k < m; ++k) gsum += rows[k * 64 + tid];
        }
        __syncthreads();
    }
    const int p = blockIdx.x * 64 + tid;
    if (tid >= 64 || p >= kMlpParams) return;
    if (grad_out) grad_out[p] = gsum;
    if (st.apply) {
        float a = fmaf(st.beta1, m1[p], (1.0f - st.beta1) * gsum);
        float b = fmaf(st.beta2, m2[p], (1.0f - st.beta2) * gsum * gsum);
        m1[p] = a;
        m2[p] = b;
        float mh = a / st.bc1, vh = b / st.bc2;
        const float v = master[p] - st.lr * mh / (sqrtf(vh) + st.eps);
        master[p] = v;
        pack_param(p, v, pk.fwd, pk.bwd, pk.bias);
    }
}

// ---------------------------------------------------------------------------
// packing: FP32 master -> bf16 A blocks (forward W, backward W^T), padded biases
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_mlp_pack(const float* __restrict__ master, uint16_t* __restrict__ fwd,
                                                  uint16_t* __restrict__ bwd, float* __restrict__ bias) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int nf = kMlpFwdBlocks * 512, nb = kMlpBwdBlocks * 512;
    if (t < nf) {
        const int blk = t >> 9, lane = (t >> 3) & 63, q = t & 7;
        int l = 0;
        while (l < 4 && blk >= mlp_fblk0(l + 1)) ++l;
        const int KS = mlp_kpad(l) / 16;
        const int local = blk - mlp_fblk0(l), mt = local / KS, s = local % KS;
        const int m = 32 * mt + (lane & 31);
        const int k = 16 * s + mlp_kperm(lane >> 5, q);
        float v = (m < mlp_out(l) && k < mlp_in(l)) ? master[mlp_woff(l) + m * mlp_in(l) + k] : 0.0f;
        fwd[t] = (uint16_t)f2bf_bits(v);
    } else if (t < nf + nb) {
        const int u = t - nf;
        const int blk = u >> 9, lane = (u >> 3) & 63, q = u & 7;
        int l = 1;
        while (l < 4 && blk >= mlp_bblk0(l + 1)) ++l;
        const int KS = mlp_mpad(l) / 16;
        const int local = blk - mlp_bblk0(l), mt = local / KS, s = local % KS;
        const int m = 32 * mt + (lane & 31);           // input unit of layer l
        const int k = 16 * s + mlp_kperm(lane >> 5, q);  // output unit of layer l
        float v = (k < mlp_out(l) && m < mlp_in(l)) ? master[mlp_woff(l) + k * mlp_in(l) + m] : 0.0f;
        bwd[u] = (uint16_t)f2bf_bits(v);
    } else if (t < nf + nb + kMlpBiasPad) {
        const int u = t - nf - nb;
        const int l = u / 64, r = u % 64;
        bias[u] = (l < 5 && r < mlp_out(l)) ? master[mlp_boff(l) + r] : 0.0f;
    }
}

// ---------------------------------------------------------------------------
// launch wrappers
// ---------------------------------------------------------------------------
void launch_mlp_pack(const float* master, uint16_t* fwd, uint16_t* bwd, float* bias, hipStream_t s) {
    const int total = kMlpFwdBlocks * 512 + kMlpBwdBlocks * 512 + kMlpBiasPad;
    hipLaunchKernelGGL(k_mlp_pack, dim3((total + 255) / 256), dim3(256), 0, s, master, fwd, bwd, bias);
}

void launch_mlp_forward(const MlpDev& w, const float* X, int n, float* Y, hipStream_t s) {
    if (n <= 0) return;
    // a launch takes fewer than 2^32 threads, two of them per row
    constexpr int per = 32 * kFwdWaves, kMaxRows = 1 << 30;
    for (int64_t i = 0; i < n; i += kMaxRows) {
        const int m = n - i < kMaxRows ? (int)(n - i) : kMaxRows;
        hipLaunchKernelGGL(k_mlp_forward, dim3((m + per - 1) / per), dim3(64 * kFwdWaves), 0, s, w, X + i * kMlpIn, m,
                           Y + i * kMlpOut);
    }
}

int mlp_train_groups(int n) { return (n + 63) / 64; }

void launch_mlp_train(const MlpDev& w, const float* X, const float* T, int n, float* partial, float* loss_part,
                      hipStream_t s) {
    const int nwg = mlp_train_groups(n);
    hipLaunchKernelGGL(k_mlp_train, dim3(nwg), dim3(256), 0, s, w, X, T, n, 1.0f / (float)n, partial,
                       loss_part);
}

void launch_mlp_adam(const float* partial, int nwg, const float* loss_part, float* master, float* m1, float* m2,
                     float* grad_out, float* loss_out, const AdamStep& st, const MlpPacked& pk, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_adam, dim3((kMlpParams + 63) / 64 + 1), dim3(256), 0, s, partial, nwg, loss_part, master,
                       m1, m2, grad_out, loss_out, st, pk);
}

}  // namespace cv
