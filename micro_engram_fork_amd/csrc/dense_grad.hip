// Dense gradients of plain embedding tables on gfx950, from the coalesced row gradients of a row
// lookup's backward: every row of a table is the summed gradient of its lookups, or zero -- what the
// autograd of nn.Embedding leaves in weight.grad (micro_engram/module.py:146-154).
//
// Write-bound: a table's gradient is as large as the table (the small fp32 engram: 16 tables of 65,536
// x 64, 268 MB), the rows it has values for are a few per cent of that. So all tables are written in
// one launch, each 16-byte chunk once, in the table's dtype and past the caches: a workgroup owns
// about 32 KB of consecutive rows of one table, finds its part of the table's ascending unique rows
// (64 probes per step of the search, so three dependent reads for 8192 rows), maps them in LDS and
// streams its rows out. 16 x 65,536 x 64 in fp32: 51 us, 5.2 TB/s (a zero fill and an indexed write per
// table before: 170 us of kernels, and the host time of four times as many calls).
// 24 x 50,000 x 64 in bf16: 32 us (before, also through fp32 copies of every table).
#include "me_common.h"

namespace me {
namespace {

constexpr int kThreads = 256;
constexpr int kChunkBytes = 32 * 1024;  // rows of one workgroup
constexpr int kMaxRows = 1024;          // at most this many rows (their map is in LDS)

struct DenseArgs {
    const int64_t *rows;  // unique rows in their tables, ascending per table
    const float *sums;    // [count, dim] their summed gradients
    const int64_t *info;  // [nt + 2] count, first unique row of each table, count
    uint8_t *out[ME_MAX_TABLES];       // [n_rows[k], dim] of T
    int64_t n_rows[ME_MAX_TABLES];
    int32_t table[ME_MAX_TABLES];      // the table's place in info
    uint32_t first_block[ME_MAX_TABLES + 1];
    int nt;                            // tables written
    int dim, rows_per_block;
};

// The first index in [lo, hi) whose row is at least `target` (rows ascending), by a whole wave.
__device__ __forceinline__ int64_t wave_lower_bound(const int64_t *rows, int64_t lo, int64_t hi, int64_t target) {
    const int lane = threadIdx.x & 63;
    while (hi - lo > 64) {  // at least halves every time: the probes are under half the range apart
        const int64_t step = (hi - lo) / 64;
        const int m = __popcll(__ballot(rows[lo + lane * step] < target));  // a prefix of the lanes
        if (m == 0) return lo;
        if (m < 64) hi = lo + m * step;
        lo += (m - 1) * step + 1;
    }
    return lo + __popcll(__ballot(lo + lane < hi && rows[min(lo + lane, hi - 1)] < target));
}

// kWide: 16-byte chunks (dim a multiple of 4, or 8 in bf16); else one element at a time.
template <typename T, bool kWide>
__global__ __launch_bounds__(kThreads) void dense_grad_kernel(const DenseArgs a) {
    constexpr int kElems = kWide ? 16 / static_cast<int>(sizeof(T)) : 1;  // elements per chunk
    __shared__ int32_t s_map[kMaxRows];
    __shared__ int64_t s_bound[2];
    const int tid = threadIdx.x, wave = tid >> 6;
    int k = 0;
    while (k + 1 < a.nt && blockIdx.x >= a.first_block[k + 1]) ++k;
    const int64_t r0 = static_cast<int64_t>(blockIdx.x - a.first_block[k]) * a.rows_per_block;
    const int n = static_cast<int>(min(a.n_rows[k] - r0, static_cast<int64_t>(a.rows_per_block)));
    if (wave < 2) {
        const int64_t b0 = a.info[1 + a.table[k]], b1 = a.info[2 + a.table[k]];
        const int64_t b = b1 > b0 ? wave_lower_bound(a.rows, b0, b1, r0 + (wave == 0 ? 0 : n)) : b0;
        if ((tid & 63) == 0) s_bound[wave] = b;
    }
    for (int i = tid; i < n; i += kThreads) s_map[i] = -1;
    __syncthreads();
    for (int64_t u = s_bound[0] + tid; u < s_bound[1]; u += kThreads)
        s_map[a.rows[u] - r0] = static_cast<int32_t>(u);
    __syncthreads();
    const int per_row = a.dim / kElems;
    int row = tid / per_row, c = tid % per_row;
    const int drow = kThreads / per_row, dc = kThreads % per_row;
    uint8_t *out = a.out[k] + (r0 * a.dim) * static_cast<int64_t>(sizeof(T));
    while (row < n) {
        const int32_t u = s_map[row];
        uint8_t *p = out + (static_cast<int64_t>(row) * a.dim + c * kElems) * static_cast<int64_t>(sizeof(T));
        const float *s = a.sums + static_cast<int64_t>(u) * a.dim + c * kElems;
        if constexpr (!kWide) {
            const float v = u >= 0 ? *as_global(s) : 0.f;
            if constexpr (sizeof(T) == 2) *as_global(reinterpret_cast<uint16_t *>(p)) = float_to_bf16_bits_rne(v);
            else *as_global(reinterpret_cast<float *>(p)) = v;
        } else {
            u32x4_v w = {0u, 0u, 0u, 0u};
            if (u >= 0) {
                if constexpr (sizeof(T) == 4) {
                    w = *as_global(reinterpret_cast<const u32x4_v *>(s));
                } else {
                    const f32x4_v lo = *as_global(reinterpret_cast<const f32x4_v *>(s));
                    const f32x4_v hi = *as_global(reinterpret_cast<const f32x4_v *>(s + 4));
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        w[e] = static_cast<uint32_t>(float_to_bf16_bits_rne(lo[2 * e])) |
                               (static_cast<uint32_t>(float_to_bf16_bits_rne(lo[2 * e + 1])) << 16);
                        w[2 + e] = static_cast<uint32_t>(float_to_bf16_bits_rne(hi[2 * e])) |
                                   (static_cast<uint32_t>(float_to_bf16_bits_rne(hi[2 * e + 1])) << 16);
                    }
                }
            }
            __builtin_nontemporal_store(w, as_global(reinterpret_cast<u32x4_v *>(p)));
        }
        row += drow;
        c += dc;
        if (c >= per_row) {
            c -= per_row;
            ++row;
        }
    }
}

}  // namespace
}  // namespace me

using namespace me;

extern "C" int me_dense_table_grads(const int64_t *local_rows, const float *sums, const int64_t *info,
                                    int32_t n_tables, const int64_t *table_rows, int32_t dim, int dtype,
                                    void *const *grads, void *stream) {
    ME_CHECK_ARG(n_tables >= 1 && n_tables <= ME_MAX_TABLES, "n_tables must be in [1, %d]", ME_MAX_TABLES);
    ME_CHECK_ARG(dim >= 1, "dim must be positive");
    ME_CHECK_ARG(dtype == ME_BF16 || dtype == ME_F32, "table dtype must be bf16 or fp32");
    ME_CHECK_ARG(info && table_rows && grads, "null pointer");
    const int64_t es = static_cast<int64_t>(dtype_size(dtype));
    DenseArgs a{};
    a.rows = local_rows;
    a.sums = sums;
    a.info = info;
    a.dim = dim;
    a.rows_per_block = static_cast<int>(kChunkBytes / (dim * es));
    if (a.rows_per_block < 1) a.rows_per_block = 1;
    if (a.rows_per_block > kMaxRows) a.rows_per_block = kMaxRows;
    bool wide = (dim * es) % 16 == 0 && reinterpret_cast<uintptr_t>(sums) % 16 == 0;
    int64_t blocks = 0;
    for (int k = 0; k < n_tables; ++k) {
        ME_CHECK_ARG(table_rows[k] >= 0, "table %d: bad row count", k);
        if (grads[k] == nullptr || table_rows[k] == 0) continue;
        a.out[a.nt] = static_cast<uint8_t *>(grads[k]);
        a.n_rows[a.nt] = table_rows[k];
        a.table[a.nt] = k;
        wide = wide && reinterpret_cast<uintptr_t>(grads[k]) % 16 == 0;
        a.first_block[a.nt++] = static_cast<uint32_t>(blocks);
        blocks += ceil_div(table_rows[k], a.rows_per_block);
        ME_CHECK_ARG(blocks < (int64_t{1} << 31), "tables too large");
    }
    if (a.nt == 0) return ME_OK;
    a.first_block[a.nt] = static_cast<uint32_t>(blocks);
    const dim3 grid(static_cast<unsigned>(blocks));
    hipStream_t s = as_stream(stream);
    if (dtype == ME_BF16) {
        if (wide) hipLaunchKernelGGL((dense_grad_kernel<uint16_t, true>), grid, dim3(kThreads), 0, s, a);
        else hipLaunchKernelGGL((dense_grad_kernel<uint16_t, false>), grid, dim3(kThreads), 0, s, a);
    } else {
        if (wide) hipLaunchKernelGGL((dense_grad_kernel<float, true>), grid, dim3(kThreads), 0, s, a);
        else hipLaunchKernelGGL((dense_grad_kernel<float, false>), grid, dim3(kThreads), 0, s, a);
    }
    return check_launch("me_dense_table_grads");
}
