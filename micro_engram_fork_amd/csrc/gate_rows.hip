// Stage 3 on gfx950 from key and value projections that are already computed: the scalar /
// scalar_sqrt gate and the residual add, and their backward.
//
// Reference (micro_engram/module.py:239-261), per token with hidden x (d wide), K = round_T(W_K
// e) and V = round_T(W_V e):
//   h = rms_norm(x) * q_scale, k = rms_norm(K) * k_scale        (scales only for scalar_sqrt)
//   s = sum(h * k) / sqrt(d); scalar_sqrt: s = sign(s) * sqrt(max(|s|, 1e-6))
//   alpha = sigmoid(s); out = x + round_H(alpha * V * keep)
//
// The fused two-pass kernel (gate.hip) computes K and V tile by tile on 256-token MFMA tiles, in
// whole rounds of the CUs per pass, and its backward computes them again. Small batches, batches
// whose rounds it fills badly and forwards with gradients run the projections in a GEMM of their
// own (me_kv_proj) and these kernels do the rest in one pass over the rows: a workgroup per token,
// 8 columns per lane with 16-byte loads of hidden, K and V issued together (V and hidden stay in
// registers for the output, so the row's only memory round trip is before the reduction), the
// three sums sum K^2, sum x (1 + dq) (1 + dk) K and sum x^2 reduced across the workgroup, the gate,
// then x + round_H(alpha V) written with 16-byte stores.
//
// Any width: rows whose model dim, row stride or addresses do not allow 16-byte accesses take a
// kernel that walks one column per lane and step (scalar loads and stores; 8 columns for rows over
// 8064 columns), so an engram of any
// model dim and memory width runs (its projections then come from a library GEMM, the nn.Linear
// of module.py:245, 254, since the MFMA kernels need whole 16-byte rows).
//
// The backward of this stage from the same K and V rows (the autograd of module.py:239-261, what
// me_gate_backward computes on MFMA tiles for the shapes those take): per token, from the
// forward's row statistics (sum x^2, sum K^2, sck = sum x qs ks K, alpha),
//   dV = round_T(alpha keep g);  d alpha = keep sum g V;  ds = d alpha alpha (1 - alpha)
//   ds0 = ds / (2 sqrt|s0|) where |s0| >= 1e-6, else 0 (scalar_sqrt); ds0 = ds (scalar)
//   a = ds0 r_h r_k / sqrt(d), c2 = a r_h^2 sck / d, c3 = a r_k^2 sck / d
//   d hidden = g + round_H(a w K - c2 x), dK = round_T(a w x - c3 K)   (w = qs ks)
// then d q_scale_j = ks_j P_j and d k_scale_j = qs_j P_j with P_j = sum over tokens of a x_j K_j.
// Rows of up to 8064 columns with 16-byte accesses take gate_rows_grad_block_kernel (a run of tokens
// per workgroup, every row read once, P summed in registers, then over the workgroups in a fixed
// order); others one workgroup per token, P per 256-token block and then over the blocks in order.
#include "me_common.h"

#include <algorithm>
#include <cmath>
#include <initializer_list>

namespace me {
namespace {

constexpr int kThreads = 256;  // one token per workgroup
constexpr int kKeep = 3;      // steps kept in registers: rows up to 3 * 256 * LC columns
constexpr int kScaleBlock = 256;  // tokens per partial of the scale gradients

struct RowArgs {
    const uint8_t *hidden;  // [n, d] of H
    const uint8_t *k;       // [n, *] of T, row stride kv_stride elements
    const uint8_t *v;       // [n, *] of T, row stride kv_stride elements
    const uint8_t *q_delta; // [d] scale - 1 (nullable: scalar gate)
    const uint8_t *k_delta;
    const uint8_t *keep;    // [n] (nullable)
    uint8_t *out;           // [n, d] of H
    float *alpha_out;       // [n] (nullable)
    float *row_stats;       // [n, 4] (nullable): sum x^2, sum K^2, sum x qs ks K, alpha
    int64_t n, d, kv_stride;
    int scale_bf16, sqrt_mode;
    float inv_d, inv_sqrt_d;
    // backward
    const uint8_t *grad_out;  // [n, d] of H
    const float *stats_in;    // [n, 4] the forward's row statistics
    uint8_t *grad_hidden;     // [n, d] of H
    uint8_t *grad_k;          // [n, d] of T
    uint8_t *grad_v;          // [n, d] of T
    float *coef;              // [n] the token's a (workspace)
    float *col_part;          // [ceil(n / kScaleBlock)][d] (workspace)
};

// LC consecutive elements of X as floats: 16-byte accesses for LC = 8, single elements for 1.
template <typename X, int LC>
__device__ __forceinline__ void loadn(const uint8_t *p, float (&v)[LC]) {
    if constexpr (LC == 1) {
        if constexpr (sizeof(X) == 2) v[0] = bf16_bits_to_float(*as_global(reinterpret_cast<const uint16_t *>(p)));
        else v[0] = *as_global(reinterpret_cast<const float *>(p));
    } else if constexpr (sizeof(X) == 2) {
        const u32x4_v w = *as_global(reinterpret_cast<const u32x4_v *>(p));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[2 * e] = bf16_bits_to_float(static_cast<uint16_t>(w[e]));
            v[2 * e + 1] = bf16_bits_to_float(static_cast<uint16_t>(w[e] >> 16));
        }
    } else {
        const f32x4_v a = *as_global(reinterpret_cast<const f32x4_v *>(p));
        const f32x4_v b = *as_global(reinterpret_cast<const f32x4_v *>(p + 16));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = a[e];
            v[4 + e] = b[e];
        }
    }
}

// Stores LC values rounded to X (round to nearest even for bf16).
template <typename X, int LC>
__device__ __forceinline__ void storen(uint8_t *p, const float (&v)[LC]) {
    if constexpr (LC == 1) {
        if constexpr (sizeof(X) == 2) *as_global(reinterpret_cast<uint16_t *>(p)) = float_to_bf16_bits_rne(v[0]);
        else *as_global(reinterpret_cast<float *>(p)) = v[0];
    } else if constexpr (sizeof(X) == 2) {
        u32x4_v w;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            w[e] = static_cast<uint32_t>(float_to_bf16_bits_rne(v[2 * e])) |
                   (static_cast<uint32_t>(float_to_bf16_bits_rne(v[2 * e + 1])) << 16);
        *as_global(reinterpret_cast<u32x4_v *>(p)) = w;
    } else {
        *as_global(reinterpret_cast<f32x4_v *>(p)) = f32x4_v{v[0], v[1], v[2], v[3]};
        *as_global(reinterpret_cast<f32x4_v *>(p + 16)) = f32x4_v{v[4], v[5], v[6], v[7]};
    }
}

// storen<X, 8> past the caches.
template <typename X>
__device__ __forceinline__ void store8_nt(uint8_t *p, const float (&v)[8]) {
    if constexpr (sizeof(X) == 2) {
        u32x4_v w;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            w[e] = static_cast<uint32_t>(float_to_bf16_bits_rne(v[2 * e])) |
                   (static_cast<uint32_t>(float_to_bf16_bits_rne(v[2 * e + 1])) << 16);
        __builtin_nontemporal_store(w, as_global(reinterpret_cast<u32x4_v *>(p)));
    } else {
        __builtin_nontemporal_store(f32x4_v{v[0], v[1], v[2], v[3]}, as_global(reinterpret_cast<f32x4_v *>(p)));
        __builtin_nontemporal_store(f32x4_v{v[4], v[5], v[6], v[7]}, as_global(reinterpret_cast<f32x4_v *>(p + 16)));
    }
}

// w = (1 + q delta)(1 + k delta) of LC columns from j (1 without scales).
template <int LC>
__device__ __forceinline__ void scale_products(const RowArgs &a, int64_t j, float (&w)[LC]) {
    if (a.q_delta != nullptr) {
        float qd[LC], kd[LC];
        if (a.scale_bf16) {
            loadn<uint16_t, LC>(a.q_delta + j * 2, qd);
            loadn<uint16_t, LC>(a.k_delta + j * 2, kd);
        } else {
            loadn<float, LC>(a.q_delta + j * 4, qd);
            loadn<float, LC>(a.k_delta + j * 4, kd);
        }
#pragma unroll
        for (int e = 0; e < LC; ++e) w[e] = (1.f + qd[e]) * (1.f + kd[e]);
    } else {
#pragma unroll
        for (int e = 0; e < LC; ++e) w[e] = 1.f;
    }
}

template <typename X>
__device__ __forceinline__ float round_to(float v) {
    if constexpr (sizeof(X) == 2) return round_to_bf16(v);
    return v;
}

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off, 64);
    return x;
}

// Sums of a block's threads, in wave order, the same in every thread.
template <int N>
__device__ __forceinline__ void block_sums(float (&v)[N], float (*s_part)[4]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = wave_sum(v[i]);
    if (lane == 0)
#pragma unroll
        for (int i = 0; i < N; ++i) s_part[wave][i] = v[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
        v[i] = 0.f;
#pragma unroll
        for (int w = 0; w < kThreads / 64; ++w) v[i] += s_part[w][i];
    }
}

// Eight columns kept as loaded (bf16: one 16-byte register quad, fp32: two) until they are used.
template <typename X>
struct Raw8 {
    u32x4_v w[sizeof(X) / 2];
    __device__ __forceinline__ void load(const uint8_t *p) {
#pragma unroll
        for (int q = 0; q < static_cast<int>(sizeof(X)) / 2; ++q)
            w[q] = as_global(reinterpret_cast<const u32x4_v *>(p))[q];
    }
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int q = 0; q < static_cast<int>(sizeof(X)) / 2; ++q) w[q] = u32x4_v{0u, 0u, 0u, 0u};
    }
    __device__ __forceinline__ float at(int e) const {
        if constexpr (sizeof(X) == 2)
            return __uint_as_float((e & 1) ? (w[0][e >> 1] & 0xffff0000u) : (w[0][e >> 1] << 16));
        else
            return __uint_as_float(w[e >> 2][e & 3]);
    }
};

// Column layout of the 16-byte row kernels: a group is 16 lanes, of which 14 hold 8 columns each
// (112 columns), so a token's sums add up in the order of the fused kernel's 224-column tiles
// (gate.hip: a lane's 8 columns in order, the 16 lanes by row shifts, the two halves of a tile, the
// tiles in order) and both paths give the same bits. Four groups are 896 contiguous bytes of a
// bf16 row, so the two idle lanes cost no memory traffic.
constexpr int kGroupCols = 112;
constexpr int kMaxGroups = 72;  // 8064 columns

__device__ __forceinline__ float row16_sum(float v) {  // exact in lane 16i + 15, as gate.hip adds
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x111, 0xf, 0xf, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x112, 0xf, 0xf, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x114, 0xf, 0xf, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x118, 0xf, 0xf, true));
    return v;
}

// Sums over a token's groups (s_half[group][N], an even number of groups), the same in every lane
// of the calling wave: lane i adds up sum i % N tile by tile.
template <int N>
__device__ __forceinline__ void tile_sums(const float *s_half, int tiles, float (&out)[N]) {
    const float *p = s_half + (threadIdx.x & 63) % N;
    float acc = 0.f;
#pragma unroll 8
    for (int t = 0; t < tiles; ++t) acc += p[2 * t * N] + p[(2 * t + 1) * N];
#pragma unroll
    for (int i = 0; i < N; ++i)
        out[i] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(acc), i));
}

__device__ __forceinline__ float row_gate(const RowArgs &a, float sx2, float sk2, float sck) {
    constexpr float kEps = 1.1920928955078125e-07f;  // torch.finfo(float32).eps: rms_norm default
    const float rh = 1.0f / sqrtf(sx2 * a.inv_d + kEps);
    const float rk = 1.0f / sqrtf(sk2 * a.inv_d + kEps);
    float s = rh * rk * sck * a.inv_sqrt_d;
    if (a.sqrt_mode) {
        const float sg = s > 0.f ? 1.f : (s < 0.f ? -1.f : 0.f);
        s = sg * sqrtf(fmaxf(fabsf(s), 1e-6f));
    }
    return 1.0f / (1.0f + expf(-s));
}

// The forward on 16-byte rows of at most kSteps * kRowThreads / 16 groups: one workgroup per token,
// every load of the token's three rows issued before the first use, hidden and V kept as loaded
// until the output, which is written past the caches. HBM-bound for many tokens (8192 x 5376 in
// bf16: 352 MB in 63 us, 5.6 TB/s; 67 us in the kernel that loads a step at a time), one memory
// round trip and two reductions for few (256 tokens: 5.0 us against 5.4).
template <typename H, typename T, int kRowThreads, int kSteps>
__global__ __launch_bounds__(kRowThreads) void gate_row_kernel(const RowArgs a) {
    constexpr int kGroups = kSteps * kRowThreads / 16;
    __shared__ float s_half[kGroups * 3];
    const int tid = threadIdx.x, l16 = tid & 15;
    const int64_t n = blockIdx.x;
    const uint8_t *x = a.hidden + n * a.d * static_cast<int64_t>(sizeof(H));
    const uint8_t *kr = a.k + n * a.kv_stride * static_cast<int64_t>(sizeof(T));
    const uint8_t *vr = a.v + n * a.kv_stride * static_cast<int64_t>(sizeof(T));
    Raw8<H> xk[kSteps];
    Raw8<T> kk[kSteps], vk[kSteps];
    int col[kSteps];
    bool in[kSteps];
#pragma unroll
    for (int q = 0; q < kSteps; ++q) {
        col[q] = ((q * kRowThreads + tid) >> 4) * kGroupCols + l16 * 8;
        in[q] = l16 < kGroupCols / 8 && col[q] < a.d;
        if (in[q]) {
            xk[q].load(x + col[q] * sizeof(H));
            kk[q].load(kr + col[q] * sizeof(T));
        } else {
            xk[q].zero();
            kk[q].zero();
        }
    }
#pragma unroll
    for (int q = 0; q < kSteps; ++q)
        if (in[q]) vk[q].load(vr + col[q] * sizeof(T));
#pragma unroll
    for (int q = 0; q < kSteps; ++q) {
        float w[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = 1.f;
        if (in[q]) scale_products<8>(a, col[q], w);
        float sk2 = 0.f, sck = 0.f, sx2 = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float kv = kk[q].at(e), xv = xk[q].at(e);
            sk2 += kv * kv;
            sck += xv * w[e] * kv;
            sx2 += xv * xv;
        }
        sk2 = row16_sum(sk2);
        sck = row16_sum(sck);
        sx2 = row16_sum(sx2);
        if (l16 == 15) {
            float *p = s_half + ((q * kRowThreads + tid) >> 4) * 3;
            p[0] = sk2;
            p[1] = sck;
            p[2] = sx2;
        }
    }
    __syncthreads();
    float sums[3];
    tile_sums<3>(s_half, static_cast<int>(ceil_div(a.d, 2 * kGroupCols)), sums);
    float alpha = row_gate(a, sums[2], sums[0], sums[1]);
    if (tid == 0) {
        if (a.alpha_out != nullptr) a.alpha_out[n] = alpha;
        if (a.row_stats != nullptr) {
            float *st = a.row_stats + n * 4;
            st[0] = sums[2];
            st[1] = sums[0];
            st[2] = sums[1];
            st[3] = alpha;
        }
    }
    if (a.keep != nullptr && a.keep[n] == 0) alpha = 0.f;
    uint8_t *o = a.out + n * a.d * static_cast<int64_t>(sizeof(H));
#pragma unroll
    for (int q = 0; q < kSteps; ++q) {
        if (!in[q]) continue;
        float ov[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) ov[e] = xk[q].at(e) + round_to<H>(alpha * vk[q].at(e));
        store8_nt<H>(o + col[q] * sizeof(H), ov);
    }
}

template <typename H, typename T, int kLaneCols>
__global__ __launch_bounds__(kThreads) void gate_rows_kernel(const RowArgs a) {
    constexpr float kEps = 1.1920928955078125e-07f;  // torch.finfo(float32).eps: rms_norm default
    __shared__ float s_part[kThreads / 64][3];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t n = blockIdx.x;
    const uint8_t *x = a.hidden + n * a.d * static_cast<int64_t>(sizeof(H));
    const uint8_t *kr = a.k + n * a.kv_stride * static_cast<int64_t>(sizeof(T));
    const uint8_t *vr = a.v + n * a.kv_stride * static_cast<int64_t>(sizeof(T));
    float sk2 = 0.f, sck = 0.f, sx2 = 0.f;
    // the row's hidden and V values of the first kKeep steps stay in registers for the output
    float xk[kKeep][kLaneCols], vk[kKeep][kLaneCols];
    int it = 0;
    for (int64_t j = static_cast<int64_t>(tid) * kLaneCols; j < a.d; j += kThreads * kLaneCols, ++it) {
        float xv[kLaneCols], kv[kLaneCols], w[kLaneCols];
        loadn<H, kLaneCols>(x + j * sizeof(H), xv);
        loadn<T, kLaneCols>(kr + j * sizeof(T), kv);
#pragma unroll
        for (int q = 0; q < kKeep; ++q)
            if (q == it) {
#pragma unroll
                for (int e = 0; e < kLaneCols; ++e) xk[q][e] = xv[e];
                loadn<T, kLaneCols>(vr + j * sizeof(T), vk[q]);
            }
        scale_products<kLaneCols>(a, j, w);
#pragma unroll
        for (int e = 0; e < kLaneCols; ++e) {
            sk2 += kv[e] * kv[e];
            sck += xv[e] * w[e] * kv[e];
            sx2 += xv[e] * xv[e];
        }
    }
    sk2 = wave_sum(sk2);
    sck = wave_sum(sck);
    sx2 = wave_sum(sx2);
    if (lane == 0) {
        s_part[wave][0] = sk2;
        s_part[wave][1] = sck;
        s_part[wave][2] = sx2;
    }
    __syncthreads();
    sk2 = sck = sx2 = 0.f;
#pragma unroll
    for (int w = 0; w < kThreads / 64; ++w) {  // in wave order: the same sums in every thread
        sk2 += s_part[w][0];
        sck += s_part[w][1];
        sx2 += s_part[w][2];
    }
    const float rh = 1.0f / sqrtf(sx2 * a.inv_d + kEps);
    const float rk = 1.0f / sqrtf(sk2 * a.inv_d + kEps);
    float s = rh * rk * sck * a.inv_sqrt_d;
    if (a.sqrt_mode) {
        const float sg = s > 0.f ? 1.f : (s < 0.f ? -1.f : 0.f);
        s = sg * sqrtf(fmaxf(fabsf(s), 1e-6f));
    }
    float alpha = 1.0f / (1.0f + expf(-s));
    if (tid == 0) {
        if (a.alpha_out != nullptr) a.alpha_out[n] = alpha;
        if (a.row_stats != nullptr) {
            float *st = a.row_stats + n * 4;
            st[0] = sx2;
            st[1] = sk2;
            st[2] = sck;
            st[3] = alpha;
        }
    }
    if (a.keep != nullptr && a.keep[n] == 0) alpha = 0.f;
    uint8_t *o = a.out + n * a.d * static_cast<int64_t>(sizeof(H));
    it = 0;
    for (int64_t j = static_cast<int64_t>(tid) * kLaneCols; j < a.d; j += kThreads * kLaneCols, ++it) {
        float xv[kLaneCols], vv[kLaneCols], ov[kLaneCols];
        if (it < kKeep) {
#pragma unroll
            for (int q = 0; q < kKeep; ++q)
                if (q == it)
#pragma unroll
                    for (int e = 0; e < kLaneCols; ++e) {
                        xv[e] = xk[q][e];
                        vv[e] = vk[q][e];
                    }
        } else {  // rows wider than kKeep steps: the rest is read again
            loadn<H, kLaneCols>(x + j * sizeof(H), xv);
            loadn<T, kLaneCols>(vr + j * sizeof(T), vv);
        }
#pragma unroll
        for (int e = 0; e < kLaneCols; ++e) ov[e] = xv[e] + round_to<H>(alpha * vv[e]);
        storen<H, kLaneCols>(o + j * sizeof(H), ov);
    }
}

// Backward per token (see the file comment): dV and the row sum of g V, the token's
// coefficients, then d hidden and dK; the token's a goes to the workspace for the scale
// gradients.
template <typename H, typename T, int kLaneCols>
__global__ __launch_bounds__(kThreads) void gate_rows_grad_kernel(const RowArgs a) {
    constexpr float kEps = 1.1920928955078125e-07f;
    __shared__ float s_part[kThreads / 64][4];
    const int tid = threadIdx.x;
    const int64_t n = blockIdx.x;
    const int64_t hrow = n * a.d, krow = n * a.kv_stride;
    const uint8_t *x = a.hidden + hrow * static_cast<int64_t>(sizeof(H));
    const uint8_t *g = a.grad_out + hrow * static_cast<int64_t>(sizeof(H));
    const uint8_t *kr = a.k + krow * static_cast<int64_t>(sizeof(T));
    const uint8_t *vr = a.v + krow * static_cast<int64_t>(sizeof(T));
    const float *st = a.stats_in + n * 4;
    const float sx2 = st[0], sk2 = st[1], sck = st[2], alpha = st[3];
    const bool kept = a.keep == nullptr || a.keep[n] != 0;
    const float alpha_eff = kept ? alpha : 0.f;
    // dV = round_T(alpha keep g) and sum g V
    float gv[1] = {0.f};
    for (int64_t j = static_cast<int64_t>(tid) * kLaneCols; j < a.d; j += kThreads * kLaneCols) {
        float gg[kLaneCols], vv[kLaneCols], dv[kLaneCols];
        loadn<H, kLaneCols>(g + j * sizeof(H), gg);
        loadn<T, kLaneCols>(vr + j * sizeof(T), vv);
#pragma unroll
        for (int e = 0; e < kLaneCols; ++e) {
            gv[0] += gg[e] * vv[e];
            dv[e] = alpha_eff * gg[e];
        }
        storen<T, kLaneCols>(a.grad_v + (n * a.d + j) * static_cast<int64_t>(sizeof(T)), dv);
    }
    block_sums<1>(gv, s_part);
    const float dalpha = kept ? gv[0] : 0.f;
    const float ds = dalpha * alpha * (1.f - alpha);
    const float rh = 1.0f / sqrtf(sx2 * a.inv_d + kEps);
    const float rk = 1.0f / sqrtf(sk2 * a.inv_d + kEps);
    const float s0 = rh * rk * sck * a.inv_sqrt_d;
    float ds0 = ds;
    if (a.sqrt_mode) ds0 = fabsf(s0) >= 1e-6f ? ds / (2.f * sqrtf(fabsf(s0))) : 0.f;
    const float ca = ds0 * rh * rk * a.inv_sqrt_d;
    const float c2 = ca * rh * rh * sck * a.inv_d;
    const float c3 = ca * rk * rk * sck * a.inv_d;
    if (tid == 0) a.coef[n] = ca;
    for (int64_t j = static_cast<int64_t>(tid) * kLaneCols; j < a.d; j += kThreads * kLaneCols) {
        float xv[kLaneCols], kv[kLaneCols], gg[kLaneCols], w[kLaneCols], dx[kLaneCols], dk[kLaneCols];
        loadn<H, kLaneCols>(x + j * sizeof(H), xv);
        loadn<T, kLaneCols>(kr + j * sizeof(T), kv);
        loadn<H, kLaneCols>(g + j * sizeof(H), gg);
        scale_products<kLaneCols>(a, j, w);
#pragma unroll
        for (int e = 0; e < kLaneCols; ++e) {
            dx[e] = gg[e] + round_to<H>(ca * w[e] * kv[e] - c2 * xv[e]);
            dk[e] = ca * w[e] * xv[e] - c3 * kv[e];
        }
        storen<H, kLaneCols>(a.grad_hidden + (hrow + j) * static_cast<int64_t>(sizeof(H)), dx);
        storen<T, kLaneCols>(a.grad_k + (n * a.d + j) * static_cast<int64_t>(sizeof(T)), dk);
    }
}

// The backward in one pass over the rows, for 16-byte rows of at most kSteps * kRowThreads / 16 groups.
// HBM-bound (four rows read and three written per token): a workgroup takes `per` tokens one after the other, every load of a token's four rows
// issued before the first use and the rows kept as loaded across the reduction, so each row is read
// once; with scales (kScaled) each lane sums a x K of its columns over the workgroup's tokens in
// registers and the workgroup writes one row of partials (the token at a time kernel above re-reads
// hidden, g and K after the reduction, and a kernel of its own reads hidden and K again for the
// scale gradients). 8192 tokens x 5376 in bf16, 616 MB: 246 us with that kernel, 132 with this one
// (4.7 TB/s; a copy of 1 GiB reaches 5.1); 2048 x 1024 in fp32: 85 and 18. Hidden states of another dtype than the
// projections gain as much (forward and backward with the projections and products, fp32 hidden and a bf16
// engram, 5320 x 136, 8192 tokens: 780 us with that kernel, 633 with this one). The stores are
// non-temporal (2048 x 5376: 36.5 us through the caches, 32 past them).
template <typename H, typename T, int kRowThreads, int kSteps, bool kScaled>
__global__ __launch_bounds__(kRowThreads) void gate_rows_grad_block_kernel(const RowArgs a, int per) {
    constexpr float kEps = 1.1920928955078125e-07f;
    constexpr int kGroups = kSteps * kRowThreads / 16;
    __shared__ float s_half[2][kGroups];
    const int tid = threadIdx.x, l16 = tid & 15;
    const int tiles = static_cast<int>(ceil_div(a.d, 2 * kGroupCols));
    const int64_t n0 = static_cast<int64_t>(blockIdx.x) * per, n1 = min(n0 + per, a.n);
    float w[kSteps][8], colp[kSteps][8];
    int col[kSteps];
    bool in[kSteps];
#pragma unroll
    for (int q = 0; q < kSteps; ++q) {
        col[q] = ((q * kRowThreads + tid) >> 4) * kGroupCols + l16 * 8;
        in[q] = l16 < kGroupCols / 8 && col[q] < a.d;
        if constexpr (kScaled) {
            if (in[q]) scale_products<8>(a, col[q], w[q]);
#pragma unroll
            for (int e = 0; e < 8; ++e) colp[q][e] = 0.f;
        }
    }
    int buf = 0;
    for (int64_t n = n0; n < n1; ++n, buf ^= 1) {
        const int64_t hrow = n * a.d, krow = n * a.kv_stride;
        Raw8<H> g[kSteps], x[kSteps];
        Raw8<T> v[kSteps], k[kSteps];
#pragma unroll
        for (int q = 0; q < kSteps; ++q) {
            const int64_t j = col[q];
            if (in[q]) {
                g[q].load(a.grad_out + (hrow + j) * static_cast<int64_t>(sizeof(H)));
                v[q].load(a.v + (krow + j) * static_cast<int64_t>(sizeof(T)));
            } else {
                g[q].zero();
                v[q].zero();
            }
        }
#pragma unroll
        for (int q = 0; q < kSteps; ++q) {
            const int64_t j = col[q];
            if (in[q]) {
                x[q].load(a.hidden + (hrow + j) * static_cast<int64_t>(sizeof(H)));
                k[q].load(a.k + (krow + j) * static_cast<int64_t>(sizeof(T)));
            }
        }
        const f32x4_v st = *as_global(reinterpret_cast<const f32x4_v *>(a.stats_in + n * 4));
        const bool kept = a.keep == nullptr || a.keep[n] != 0;
        const float sx2 = st[0], sk2 = st[1], sck = st[2], alpha = st[3];
        const float alpha_eff = kept ? alpha : 0.f;
        // dV = round_T(alpha keep g) and sum g V
#pragma unroll
        for (int q = 0; q < kSteps; ++q) {
            float dv[8], part = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                part += g[q].at(e) * v[q].at(e);
                dv[e] = alpha_eff * g[q].at(e);
            }
            part = row16_sum(part);
            if (l16 == 15) s_half[buf][(q * kRowThreads + tid) >> 4] = part;
            if (in[q]) store8_nt<T>(a.grad_v + (hrow + col[q]) * static_cast<int64_t>(sizeof(T)), dv);
        }
        __syncthreads();  // two buffers: a wave one token ahead writes the other one
        float gv[1];
        tile_sums<1>(s_half[buf], tiles, gv);
        const float dalpha = kept ? gv[0] : 0.f;
        const float ds = dalpha * alpha * (1.f - alpha);
        const float rh = 1.0f / sqrtf(sx2 * a.inv_d + kEps);
        const float rk = 1.0f / sqrtf(sk2 * a.inv_d + kEps);
        const float s0 = rh * rk * sck * a.inv_sqrt_d;
        float ds0 = ds;
        if (a.sqrt_mode) ds0 = fabsf(s0) >= 1e-6f ? ds / (2.f * sqrtf(fabsf(s0))) : 0.f;
        const float ca = ds0 * rh * rk * a.inv_sqrt_d;
        const float c2 = ca * rh * rh * sck * a.inv_d;
        const float c3 = ca * rk * rk * sck * a.inv_d;
#pragma unroll
        for (int q = 0; q < kSteps; ++q) {
            const int64_t j = col[q];
            if (!in[q]) continue;
            float dx[8], dk[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float xv = x[q].at(e), kv = k[q].at(e);
                const float cw = kScaled ? ca * w[q][e] : ca;
                dx[e] = g[q].at(e) + round_to<H>(cw * kv - c2 * xv);
                dk[e] = cw * xv - c3 * kv;
                if constexpr (kScaled) colp[q][e] += ca * xv * kv;
            }
            store8_nt<H>(a.grad_hidden + (hrow + j) * static_cast<int64_t>(sizeof(H)), dx);
            store8_nt<T>(a.grad_k + (hrow + j) * static_cast<int64_t>(sizeof(T)), dk);
        }
    }
    if constexpr (kScaled) {
#pragma unroll
        for (int q = 0; q < kSteps; ++q) {
            const int64_t j = col[q];
            if (in[q]) storen<float, 8>(reinterpret_cast<uint8_t *>(a.col_part + blockIdx.x * a.d + j), colp[q]);
        }
    }
}

// The workgroups' partials of gate_rows_grad_block_kernel added up, times the other scale: 64
// columns per workgroup, wave w takes partials w, w + 16, ... (loads of 256 contiguous bytes, all
// independent), then the waves' sums in order.
constexpr int kSumWaves = 16;
__global__ __launch_bounds__(64 * kSumWaves) void gate_rows_scale_sum_kernel(const RowArgs a, int64_t parts,
                                                                            float *grad_q, float *grad_k) {
    __shared__ float s_sum[kSumWaves][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t j = static_cast<int64_t>(blockIdx.x) * 64 + lane;
    float p = 0.f;
    if (j < a.d) {
#pragma unroll 8
        for (int64_t b = wave; b < parts; b += kSumWaves) p += a.col_part[b * a.d + j];
    }
    s_sum[wave][lane] = p;
    __syncthreads();
    if (wave != 0 || j >= a.d) return;
    p = 0.f;
#pragma unroll
    for (int i = 0; i < kSumWaves; ++i) p += s_sum[i][lane];
    float q, k;
    if (a.scale_bf16) {
        q = bf16_bits_to_float(reinterpret_cast<const uint16_t *>(a.q_delta)[j]);
        k = bf16_bits_to_float(reinterpret_cast<const uint16_t *>(a.k_delta)[j]);
    } else {
        q = reinterpret_cast<const float *>(a.q_delta)[j];
        k = reinterpret_cast<const float *>(a.k_delta)[j];
    }
    grad_q[j] = (1.f + k) * p;
    grad_k[j] = (1.f + q) * p;
}

// Scale gradients, first level: column j of token block b, sum over the block's tokens (in
// order) of a x_j K_j; one thread per column, consecutive threads on consecutive columns.
template <typename H, typename T>
__global__ __launch_bounds__(kThreads) void gate_rows_scale_part_kernel(const RowArgs a) {
    const int64_t j = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    const int64_t b = blockIdx.y;
    if (j >= a.d) return;
    const int64_t n0 = b * kScaleBlock, n1 = min(n0 + kScaleBlock, a.n);
    float p = 0.f;
    for (int64_t n = n0; n < n1; ++n) {
        float xv[1], kv[1];
        loadn<H, 1>(a.hidden + (n * a.d + j) * static_cast<int64_t>(sizeof(H)), xv);
        loadn<T, 1>(a.k + (n * a.kv_stride + j) * static_cast<int64_t>(sizeof(T)), kv);
        p += a.coef[n] * xv[0] * kv[0];
    }
    a.col_part[b * a.d + j] = p;
}

// Second level: the blocks' partials in order, times the other scale.
__global__ __launch_bounds__(kThreads) void gate_rows_scale_kernel(const RowArgs a, int64_t blocks,
                                                                   float *grad_q, float *grad_k) {
    const int64_t j = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (j >= a.d) return;
    float p = 0.f;
    for (int64_t b = 0; b < blocks; ++b) p += a.col_part[b * a.d + j];
    float q, k;
    if (a.scale_bf16) {
        q = bf16_bits_to_float(reinterpret_cast<const uint16_t *>(a.q_delta)[j]);
        k = bf16_bits_to_float(reinterpret_cast<const uint16_t *>(a.k_delta)[j]);
    } else {
        q = reinterpret_cast<const float *>(a.q_delta)[j];
        k = reinterpret_cast<const float *>(a.k_delta)[j];
    }
    grad_q[j] = (1.f + k) * p;
    grad_k[j] = (1.f + q) * p;
}

bool aligned16(const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace
}  // namespace me

using namespace me;

namespace me {
namespace {

// The argument checks and fields shared by the forward and the backward of the row kernels.
int rows_common(RowArgs &a, const void *hidden, int hidden_dtype, int64_t n, int64_t model_dim,
                const void *k_proj, const void *v_proj, int64_t kv_stride, int dtype,
                const void *q_scale_delta, const void *k_scale_delta, int scale_dtype, int gate_mode,
                const uint8_t *keep) {
    ME_CHECK_ARG(n >= 0 && n < (int64_t{1} << 31), "bad token count %lld", (long long)n);
    ME_CHECK_ARG(model_dim >= 1, "model_dim must be positive, got %lld", (long long)model_dim);
    ME_CHECK_ARG(hidden_dtype == ME_BF16 || hidden_dtype == ME_F32, "hidden dtype must be bf16 or fp32");
    ME_CHECK_ARG(dtype == ME_BF16 || dtype == ME_F32, "projection dtype must be bf16 or fp32");
    ME_CHECK_ARG(gate_mode == ME_GATE_SCALAR || gate_mode == ME_GATE_SCALAR_SQRT, "unknown gate mode %d",
                 gate_mode);
    ME_CHECK_ARG(kv_stride >= model_dim, "kv_stride %lld < model_dim %lld", (long long)kv_stride,
                 (long long)model_dim);
    a.hidden = static_cast<const uint8_t *>(hidden);
    a.k = static_cast<const uint8_t *>(k_proj);
    a.v = static_cast<const uint8_t *>(v_proj);
    a.keep = keep;
    a.n = n;
    a.d = model_dim;
    a.kv_stride = kv_stride;
    a.sqrt_mode = gate_mode == ME_GATE_SCALAR_SQRT;
    if (a.sqrt_mode) {
        ME_CHECK_ARG(q_scale_delta && k_scale_delta, "scalar_sqrt needs both scale deltas");
        ME_CHECK_ARG(scale_dtype == ME_BF16 || scale_dtype == ME_F32, "scale dtype must be bf16 or fp32");
        a.q_delta = static_cast<const uint8_t *>(q_scale_delta);
        a.k_delta = static_cast<const uint8_t *>(k_scale_delta);
        a.scale_bf16 = scale_dtype == ME_BF16;
    }
    a.inv_d = 1.0f / static_cast<float>(model_dim);
    a.inv_sqrt_d = static_cast<float>(1.0 / std::sqrt(static_cast<double>(model_dim)));
    return ME_OK;
}

// 16-byte accesses of 8 columns when every row start allows them, else one column per step.
bool wide_rows(const RowArgs &a, std::initializer_list<const void *> ptrs) {
    if (a.d % 8 != 0 || a.kv_stride % 8 != 0) return false;
    for (const void *p : ptrs)
        if (p != nullptr && !aligned16(p)) return false;
    return true;
}

#define ME_ROWS_DISPATCH(KERNEL, LC, grid, s, a)                                                     \
    do {                                                                                            \
        if (hidden_dtype == ME_BF16) {                                                              \
            if (dtype == ME_BF16) hipLaunchKernelGGL((KERNEL<uint16_t, uint16_t, LC>), grid, dim3(kThreads), 0, s, a); \
            else hipLaunchKernelGGL((KERNEL<uint16_t, float, LC>), grid, dim3(kThreads), 0, s, a); \
        } else {                                                                                    \
            if (dtype == ME_BF16) hipLaunchKernelGGL((KERNEL<float, uint16_t, LC>), grid, dim3(kThreads), 0, s, a); \
            else hipLaunchKernelGGL((KERNEL<float, float, LC>), grid, dim3(kThreads), 0, s, a);    \
        }                                                                                           \
    } while (0)

// Workgroups of gate_rows_grad_block_kernel, each a run of whole tokens. One row of partials per
// workgroup is written and read again, so there are only as many as keep the memory busy: 512 (8192
// tokens x 5376 in bf16: 131 us with 256, 512 or 1024; 2048 tokens: 35.9 / 31.8 / 35.0), or 1024 for
// narrow rows of many tokens (8192 x 2048: 70.5 / 56.8 / 48.5).
constexpr int64_t kGradGroups = 1024;
int64_t grad_groups(int64_t n, int64_t d) { return d <= 2048 && n >= 4096 ? kGradGroups : kGradGroups / 2; }

// The token's coefficient and the scale gradients' partials of either backward kernel.
size_t rows_grad_workspace(int64_t n, int64_t d) {
    const size_t coef = (static_cast<size_t>(n) * 4 + 255) & ~size_t{255};
    const int64_t parts = std::max(ceil_div(n, kScaleBlock), std::min(n, grad_groups(n, d)));
    return coef + static_cast<size_t>(parts) * static_cast<size_t>(d) * 4;
}

// Whether the one-pass kernels take these rows: at most kMaxGroups groups.
bool one_pass(const RowArgs &a) { return a.d <= kMaxGroups * kGroupCols; }

template <typename H, typename T, int kRowThreads, int kSteps>
void launch_row(const RowArgs &a, int per, unsigned groups, hipStream_t s) {
    if (a.grad_out == nullptr)
        hipLaunchKernelGGL((gate_row_kernel<H, T, kRowThreads, kSteps>), dim3(groups), dim3(kRowThreads), 0, s, a);
    else if (a.sqrt_mode)
        hipLaunchKernelGGL((gate_rows_grad_block_kernel<H, T, kRowThreads, kSteps, true>), dim3(groups),
                           dim3(kRowThreads), 0, s, a, per);
    else
        hipLaunchKernelGGL((gate_rows_grad_block_kernel<H, T, kRowThreads, kSteps, false>), dim3(groups),
                           dim3(kRowThreads), 0, s, a, per);
}

// The fewest steps with at most 24 groups (384 threads) each, and as few waves as hold them: every
// load of a token in flight and few idle lanes (8192 tokens in bf16: 5376 columns, 48 groups, 63 us on
// 2 x 384 threads and 77 on 1024; 1024 columns, 17 us on 256 threads and 46 on 1024).
template <typename H, typename T>
void launch_rows(const RowArgs &a, int per, unsigned groups, hipStream_t s) {
    const int g = static_cast<int>(ceil_div(a.d, 2 * kGroupCols)) * 2;
    const int steps = (g + 23) / 24;
    const int waves = static_cast<int>(ceil_div(ceil_div(g, steps), 4));
    if (steps == 1) {
        if (waves <= 2) launch_row<H, T, 128, 1>(a, per, groups, s);
        else if (waves == 3) launch_row<H, T, 192, 1>(a, per, groups, s);
        else if (waves == 4) launch_row<H, T, 256, 1>(a, per, groups, s);
        else if (waves == 5) launch_row<H, T, 320, 1>(a, per, groups, s);
        else launch_row<H, T, 384, 1>(a, per, groups, s);
    } else if (steps == 2) {
        if (waves <= 4) launch_row<H, T, 256, 2>(a, per, groups, s);
        else if (waves == 5) launch_row<H, T, 320, 2>(a, per, groups, s);
        else launch_row<H, T, 384, 2>(a, per, groups, s);
    } else {
        if (waves <= 5) launch_row<H, T, 320, 3>(a, per, groups, s);
        else launch_row<H, T, 384, 3>(a, per, groups, s);
    }
}

void launch_rows(const RowArgs &a, int hidden_dtype, int dtype, int per, unsigned groups, hipStream_t s) {
    if (hidden_dtype == ME_BF16) {
        if (dtype == ME_BF16) launch_rows<uint16_t, uint16_t>(a, per, groups, s);
        else launch_rows<uint16_t, float>(a, per, groups, s);
    } else {
        if (dtype == ME_BF16) launch_rows<float, uint16_t>(a, per, groups, s);
        else launch_rows<float, float>(a, per, groups, s);
    }
}

}  // namespace
}  // namespace me

extern "C" int me_gate_rows(const void *hidden, int hidden_dtype, int64_t n, int64_t model_dim,
                            const void *k_proj, const void *v_proj, int64_t kv_stride, int dtype,
                            const void *q_scale_delta, const void *k_scale_delta, int scale_dtype,
                            int gate_mode, const uint8_t *keep, void *out, float *alpha_out,
                            float *row_stats, void *stream) {
    RowArgs a{};
    const int st = rows_common(a, hidden, hidden_dtype, n, model_dim, k_proj, v_proj, kv_stride, dtype,
                               q_scale_delta, k_scale_delta, scale_dtype, gate_mode, keep);
    if (st != ME_OK) return st;
    if (n == 0) return ME_OK;
    ME_CHECK_ARG(hidden && k_proj && v_proj && out, "null tensor pointer");
    a.out = static_cast<uint8_t *>(out);
    a.alpha_out = alpha_out;
    a.row_stats = row_stats;
    const dim3 grid(static_cast<unsigned>(n));
    hipStream_t s = as_stream(stream);
    if (!wide_rows(a, {hidden, k_proj, v_proj, out, a.q_delta, a.k_delta}))
        ME_ROWS_DISPATCH(gate_rows_kernel, 1, grid, s, a);
    else if (!one_pass(a))
        ME_ROWS_DISPATCH(gate_rows_kernel, 8, grid, s, a);
    else
        launch_rows(a, hidden_dtype, dtype, 1, static_cast<unsigned>(n), s);
    return check_launch("me_gate_rows");
}

extern "C" int me_gate_rows_backward_workspace_size(int64_t n, int64_t model_dim, size_t *bytes) {
    ME_CHECK_ARG(bytes != nullptr, "bytes is null");
    ME_CHECK_ARG(n >= 0 && model_dim >= 1, "bad shape n=%lld d=%lld", (long long)n, (long long)model_dim);
    *bytes = rows_grad_workspace(n, model_dim);
    return ME_OK;
}

extern "C" int me_gate_rows_backward(const void *hidden, int hidden_dtype, int64_t n, int64_t model_dim,
                                     const void *k_proj, const void *v_proj, int64_t kv_stride, int dtype,
                                     const void *q_scale_delta, const void *k_scale_delta, int scale_dtype,
                                     int gate_mode, const uint8_t *keep, const void *grad_out,
                                     const float *row_stats, void *grad_hidden, void *grad_key,
                                     void *grad_value, float *grad_q_scale, float *grad_k_scale,
                                     void *workspace, size_t workspace_size, void *stream) {
    RowArgs a{};
    const int st = rows_common(a, hidden, hidden_dtype, n, model_dim, k_proj, v_proj, kv_stride, dtype,
                               q_scale_delta, k_scale_delta, scale_dtype, gate_mode, keep);
    if (st != ME_OK) return st;
    hipStream_t s = as_stream(stream);
    if (n == 0) {  // no tokens: zero scale gradients (a fill kernel: nothing for a captured graph to memset)
        if (a.sqrt_mode && grad_q_scale && grad_k_scale) {
            hipLaunchKernelGGL(gate_rows_scale_kernel, dim3(static_cast<unsigned>(ceil_div(model_dim, kThreads))),
                               dim3(kThreads), 0, s, a, int64_t{0}, grad_q_scale, grad_k_scale);
            return check_launch("me_gate_rows_backward (zero scale gradients)");
        }
        return ME_OK;
    }
    ME_CHECK_ARG(hidden && k_proj && v_proj && grad_out && row_stats && grad_hidden && grad_key && grad_value,
                 "null tensor pointer");
    if (a.sqrt_mode) ME_CHECK_ARG(grad_q_scale && grad_k_scale, "scalar_sqrt needs the scale gradient outputs");
    const size_t need = rows_grad_workspace(n, model_dim);
    if (workspace == nullptr || workspace_size < need) {
        set_error("me_gate_rows_backward: workspace of %zu bytes needed, got %zu", need, workspace_size);
        return ME_ERR_WORKSPACE;
    }
    a.grad_out = static_cast<const uint8_t *>(grad_out);
    a.stats_in = row_stats;
    a.grad_hidden = static_cast<uint8_t *>(grad_hidden);
    a.grad_k = static_cast<uint8_t *>(grad_key);
    a.grad_v = static_cast<uint8_t *>(grad_value);
    a.coef = static_cast<float *>(workspace);
    a.col_part = reinterpret_cast<float *>(static_cast<uint8_t *>(workspace) +
                                           ((static_cast<size_t>(n) * 4 + 255) & ~size_t{255}));
    const dim3 grid(static_cast<unsigned>(n));
    const bool wide = wide_rows(a, {hidden, k_proj, v_proj, grad_out, grad_hidden, grad_key, grad_value, a.q_delta,
                                    a.k_delta});
    if (wide && aligned16(row_stats) && one_pass(a)) {
        const int per = static_cast<int>(ceil_div(n, grad_groups(n, model_dim)));
        const unsigned groups = static_cast<unsigned>(ceil_div(n, per));
        launch_rows(a, hidden_dtype, dtype, per, groups, s);
        const int bs = check_launch("me_gate_rows_backward (rows)");
        if (bs != ME_OK || !a.sqrt_mode) return bs;
        hipLaunchKernelGGL(gate_rows_scale_sum_kernel, dim3(static_cast<unsigned>(ceil_div(model_dim, 64))),
                           dim3(64 * kSumWaves), 0, s, a, static_cast<int64_t>(groups), grad_q_scale, grad_k_scale);
        return check_launch("me_gate_rows_backward (scale gradients)");
    }
    if (wide)
        ME_ROWS_DISPATCH(gate_rows_grad_kernel, 8, grid, s, a);
    else
        ME_ROWS_DISPATCH(gate_rows_grad_kernel, 1, grid, s, a);
    int st_ = check_launch("me_gate_rows_backward (rows)");
    if (st_ != ME_OK || !a.sqrt_mode) return st_;
    const int64_t blocks = ceil_div(n, kScaleBlock);
    const dim3 pgrid(static_cast<unsigned>(ceil_div(model_dim, kThreads)), static_cast<unsigned>(blocks));
    if (hidden_dtype == ME_BF16) {
        if (dtype == ME_BF16) hipLaunchKernelGGL((gate_rows_scale_part_kernel<uint16_t, uint16_t>), pgrid, dim3(kThreads), 0, s, a);
        else hipLaunchKernelGGL((gate_rows_scale_part_kernel<uint16_t, float>), pgrid, dim3(kThreads), 0, s, a);
    } else {
        if (dtype == ME_BF16) hipLaunchKernelGGL((gate_rows_scale_part_kernel<float, uint16_t>), pgrid, dim3(kThreads), 0, s, a);
        else hipLaunchKernelGGL((gate_rows_scale_part_kernel<float, float>), pgrid, dim3(kThreads), 0, s, a);
    }
    st_ = check_launch("me_gate_rows_backward (scale partials)");
    if (st_ != ME_OK) return st_;
    hipLaunchKernelGGL(gate_rows_scale_kernel, dim3(static_cast<unsigned>(ceil_div(model_dim, kThreads))),
                       dim3(kThreads), 0, s, a, blocks, grad_q_scale, grad_k_scale);
    return check_launch("me_gate_rows_backward (scale gradients)");
}
