// Stage 3 on gfx950: the key and value projections of the memory vectors,
//   kv[n][j]     = round_T(sum_m mem[n][m] W_K[j][m])        j < d
//   kv[n][d + j] = round_T(sum_m mem[n][m] W_V[j][m])        j < d
// the two nn.Linear calls of MicroEngram.inject (micro_engram/module.py:245, 254). me_gate_rows
// then does the gate and the residual add from kv. Batches that fill the part with the fused gate
// kernel's 256 x 224 tiles take those (gate.hip); the tiles here are for smaller ones (a serving
// decode step: 256 tokens against 10,752 output columns of K = 1536).
//
// At that size the GEMM is bound by moving operands into the CUs: the weights (33 MB at the
// Gemma-scale shape) are read once per token tile, the memory vectors once per column tile.
// Measured on MI355X, loads that ask each 128-byte line for half of it (what an MFMA fragment
// loaded straight into registers is: 16 rows x 64 bytes) move the same bytes 1.5x slower than
// loads of whole lines. So operands go through LDS as in the fused gate kernel: a workgroup owns
// a TM-token x TN-column output tile, its K loop streams 128-byte k-slabs (one line of each of
// the TM + TN rows) into a ring of LDS slots with buffer_load ... lds (8 whole rows per
// instruction, no register staging), and its four waves, 2 x 2 over the tile, read their MFMA
// fragments back with ds_read_b128. Rows are XOR-swizzled by (row >> 1) & 7 over their eight
// 16-byte chunks, so a fragment read of 16 consecutive rows covers all LDS banks. R - 1 slabs are
// in flight while one is consumed; one barrier per slab. The tile is then staged in LDS (rounded
// to T) and written as 16-byte row segments.
//
// Output columns are laid out virtually as [K block | V block], each block padded to a multiple
// of 16 columns, so a 16-column MFMA block and an 8-row load read one weight matrix. Rows past the
// token count, padding columns and k past mem_dim read as zeros (per-lane offsets past the
// buffer); nothing outside the real output is stored.
//
// bf16: v_mfma_f32_16x16x32_bf16, a slab is 2 k-steps of 32. fp32, few tiles: v_mfma_f32_16x16x4f32, a
// slab is 2 k-steps of 16: each lane reads 4 consecutive values and the four MFMAs of the step take
// component i of every lane (the sum runs over the same k in a permuted order in both operands).
// fp32, many tiles: the fp32 matrix rate (157 TFLOP/s) bounds those, so a slab is one k-step of 32 on the
// bf16 matrix cores. Each value is split exactly into three bf16 parts as its fragment is read (11
// vector instructions per pair and one that checks the parts), and six of the nine products of the parts are
// accumulated in fp32; the other three are below 2^-26 of each term. 2-norm error against 64 bits, normal
// values, memory dim 512 / 1024 / 1536: 3.4e-7 / 4.8e-7 / 6.0e-7 (fp32 MFMAs 4.1e-7 / 5.7e-7 / 7.0e-7). Blocks of
// 16 x 16 outputs with values that have no such parts (not finite, or so tiny, under about 2^-110, that the last
// part ends below the smallest bf16) are made again in fp32 MFMAs: slower, 2048 tokens with one tiny weight
// 107 us where they take 68 without. The splitting and the MFMAs take turns on a SIMD (2048
// tokens at 1024 x 1024: 61.6 us, 24 of them MFMAs at their full rate): one wave with the next
// slab's splitting placed between its MFMAs, 16x16x32 or 32x32x16, took as long.
#include "me_common.h"

namespace me {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef int int32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kSlab = 128;        // bytes of k per row per slab (a cache line)
constexpr int kXcds = 8;
constexpr uint32_t kBufferConfig = 0x00020000u;  // raw buffer descriptor word 3 (gfx9 family)
constexpr int kLdsBytes = 160 * 1024;

struct ProjArgs {
    const uint8_t *mem;   // [n, m] of T
    const uint8_t *wk;    // [d, m] of T
    const uint8_t *wv;    // [d, m] of T
    uint8_t *kv;          // [n, 2d] of T
    int64_t n, d, m;
    int64_t d_pad;        // d rounded up to 16: the V block starts at virtual column d_pad
    uint32_t mem_bytes, w_bytes, row_bytes;
    int slabs;            // ceil(row_bytes / 128)
    int tiles_tok, tiles_total, per_xcd;
};

__device__ __forceinline__ int32x4 rsrc_of(const void *base, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    int32x4 r;
    r.x = static_cast<int>(static_cast<uint32_t>(a));
    r.y = static_cast<int>(static_cast<uint32_t>(a >> 32) & 0xffffu);  // stride 0
    r.z = static_cast<int>(bytes);
    r.w = static_cast<int>(kBufferConfig);
    return r;
}

// 64 lanes x 16 bytes from the buffer (lane's byte voffset; at or past the range: zeros) into
// LDS at lds_base + 16 * lane. Counted by vmcnt, which the caller waits for explicitly.
__device__ __forceinline__ void dma16(const int32x4 &rsrc, uint32_t lds_base, uint32_t voffset) {
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :
                 : "s"(lds_base), "v"(voffset), "s"(rsrc)
                 : "memory");
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

__device__ __forceinline__ uint32_t lds_addr(const void *p) {
    return static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) uint8_t *)p));
}

template <typename T>
struct Mma;
template <>
struct Mma<uint16_t> {  // a 16-byte fragment is one k-step of 32
    __device__ __forceinline__ static void run(floatx4 &acc, const u32x4_v &a, const u32x4_v &b) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                      __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
    }
};
template <>
struct Mma<float> {  // a 16-byte fragment is four k values of each lane group: four MFMAs
    __device__ __forceinline__ static void run(floatx4 &acc, const u32x4_v &a, const u32x4_v &b) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[i]), __uint_as_float(b[i]), acc,
                                                       0, 0, 0);
    }
};

// Eight fp32 values of a lane as three bf16 fragments that add up to them exactly: each value rounded to
// the nearest bf16, then what remains, twice (24 bits of significand in three times 8).
struct Split {
    u32x4_v p[3];
};

// `rest` collects the bits of what is left for the third part: that part is exact where the low half of
// its fp32 is zero, which values under about 2^-110 may miss (the smallest bf16 is 2^-133).
__device__ __forceinline__ Split split_of(const u32x4_v &lo, const u32x4_v &hi, uint32_t &rest) {
    Split s;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float x = __uint_as_float(i < 2 ? lo[2 * i] : hi[2 * i - 4]);
        float y = __uint_as_float(i < 2 ? lo[2 * i + 1] : hi[2 * i - 3]);
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            // one v_cvt_pk_bf16_f32 for the pair
            const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2){x, y}, bf16x2));
            s.p[t][i] = w;
            if (t == 2) rest |= __float_as_uint(x) | __float_as_uint(y);
            x -= __uint_as_float(w << 16);
            y -= __uint_as_float(w & 0xffff0000u);
        }
    }
    return s;
}

// T: element type; BA x BB 16-row blocks per wave (tokens x columns); WA x 2 waves; R ring slots.
// SPLIT (fp32): the products on the bf16 matrix cores.
template <typename T, int BA, int BB, int R, bool SPLIT, int WA>
__global__ __launch_bounds__(128 * WA) void proj_kernel(const ProjArgs a) {
    constexpr int kEs = sizeof(T);
    constexpr int kWaves = 2 * WA, kBlock = 64 * kWaves;
    constexpr int TM = WA * 16 * BA;              // tokens per tile
    constexpr int TN = 2 * 16 * BB;               // columns per tile
    constexpr int kRows = TM + TN;                // rows per slab: A (tokens) then B (columns)
    constexpr int kDmaWave = (kRows / 8 + kWaves - 1) / kWaves;  // 8-row loads per wave and slab (past kRows: zeros)
    constexpr int kSlot = kDmaWave * kWaves * 8 * kSlab;         // bytes per ring slot
    static_assert(R >= 3 && R * kSlot <= kLdsBytes, "ring must fit in LDS");
    static_assert(!SPLIT || kEs == 4, "fp32 values are split");
    static_assert((R - 2) * kDmaWave <= 63, "vmcnt counts up to 63");
    constexpr int kStagePitch = TN * kEs + 16;    // epilogue staging row: TN values + pad
    static_assert(TM * kStagePitch <= R * kSlot, "epilogue staging must fit in the ring");
    __shared__ __attribute__((aligned(16))) uint8_t ring[R * kSlot];

    const int b = blockIdx.x;  // XCD x takes tiles [x per_xcd, (x+1) per_xcd), token tiles fastest
    const int tile = (b % kXcds) * a.per_xcd + b / kXcds;
    if (tile >= a.tiles_total) return;
    const int tok_tile = tile % a.tiles_tok;
    const int col_tile = tile / a.tiles_tok;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wa = wave % WA, wb = wave / WA;     // the wave's part of the tile
    const int64_t tok0 = static_cast<int64_t>(tok_tile) * TM;
    const int64_t col0 = static_cast<int64_t>(col_tile) * TN;

    const int32x4 rm = rsrc_of(a.mem, a.mem_bytes);
    const int32x4 rk = rsrc_of(a.wk, a.w_bytes);
    const int32x4 rv = rsrc_of(a.wv, a.w_bytes);

    // Load i of this wave fills slab rows 8 (kWaves i + wave) + [0, 8): lane l takes row + l / 8 at
    // physical chunk l % 8, i.e. logical chunk (l % 8) ^ ((row >> 1) & 7). A lane's row offset
    // and chunk are fixed for the whole K loop; per slab the k offset is added, and a chunk past
    // the row (k tail), a token past n or a padding column reads past its buffer (zeros).
    uint32_t roff[kDmaWave], chk[kDmaWave], lim[kDmaWave];
    int src[kDmaWave];  // 0: mem, 1: W_K, 2: W_V (uniform per load)
#pragma unroll
    for (int i = 0; i < kDmaWave; ++i) {
        const int g8 = 8 * (kWaves * i + wave);    // first slab row of the load (uniform)
        const int row = g8 + (lane >> 3);
        chk[i] = static_cast<uint32_t>((lane & 7) ^ ((row >> 1) & 7)) * 16u;
        if (g8 < TM) {
            src[i] = 0;
            lim[i] = a.mem_bytes;
            const int64_t r = tok0 + row;
            roff[i] = r < a.n ? static_cast<uint32_t>(r) * a.row_bytes : a.mem_bytes;
        } else {
            const int64_t vc0 = col0 + (g8 - TM);  // virtual column of the load's 8 rows
            src[i] = vc0 < a.d_pad ? 1 : 2;
            lim[i] = a.w_bytes;
            const int64_t jr = (vc0 < a.d_pad ? vc0 : vc0 - a.d_pad) + (lane >> 3);
            roff[i] = (g8 < kRows && jr < a.d && vc0 < 2 * a.d_pad) ? static_cast<uint32_t>(jr) * a.row_bytes : a.w_bytes;
        }
    }
    const uint32_t ring_lds = lds_addr(ring);
    auto issue = [&](int sl) {
        const uint32_t slot = ring_lds + static_cast<uint32_t>(sl % R) * kSlot;
        const uint32_t kb = static_cast<uint32_t>(sl) * kSlab;
#pragma unroll
        for (int i = 0; i < kDmaWave; ++i) {
            const uint32_t dst = __builtin_amdgcn_readfirstlane(slot + static_cast<uint32_t>(kWaves * i + wave) * 1024u);
            const bool in = roff[i] < lim[i] && chk[i] + kb < a.row_bytes;
            const uint32_t vo = in ? roff[i] + chk[i] + kb : lim[i];
            dma16(src[i] == 0 ? rm : (src[i] == 1 ? rk : rv), dst, vo);
        }
    };

    floatx4 acc[BA][BB];
#pragma unroll
    for (int i = 0; i < BA; ++i)
#pragma unroll
        for (int j = 0; j < BB; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    // fragment reads: k-step ks of the slab in `slot`; lane l reads row (l & 15) of a 16-row block
    // at logical chunk 4 ks + (l >> 4)
    const int fr = lane & 15;
    const int fq = lane >> 4;
    auto frag = [&](const uint8_t *slot, int row, int ks) {
        const int c = ((4 * ks + fq) ^ ((row >> 1) & 7)) << 4;
        return *reinterpret_cast<const u32x4_v *>(slot + row * kSlab + c);
    };

    const int slabs = a.slabs;
    uint32_t rest_a[BA] = {}, rest_b[BB] = {};  // split_of's, of this lane's row of each block
#pragma unroll
    for (int sl = 0; sl < R - 1; ++sl)
        if (sl < slabs) issue(sl);
    for (int sl = 0; sl < slabs; ++sl) {
        // slab sl landed for this wave (later slabs may fly), then for every wave
        if (sl + R - 2 < slabs)
            wait_vmcnt<(R - 2) * kDmaWave>();
        else
            wait_vmcnt<0>();
        __syncthreads();
        // the slot of slab sl - 1 is free: every wave read it before this barrier
        if (sl + R - 1 < slabs) issue(sl + R - 1);
        const uint8_t *slot = ring + (sl % R) * kSlot;
        if constexpr (SPLIT) {  // one k-step of 32: chunks fq and 4 + fq of both operands
            Split fa[BA], fb[BB];
#pragma unroll
            for (int i = 0; i < BA; ++i) {
                const int row = wa * 16 * BA + 16 * i + fr;
                fa[i] = split_of(frag(slot, row, 0), frag(slot, row, 1), rest_a[i]);
            }
#pragma unroll
            for (int j = 0; j < BB; ++j) {
                const int row = TM + wb * 16 * BB + 16 * j + fr;
                fb[j] = split_of(frag(slot, row, 0), frag(slot, row, 1), rest_b[j]);
            }
            // of the nine products of the parts the three below 2^-26 of the first are left out; the small
            // ones come first, each over every block before the next: an MFMA waits for its accumulator
            constexpr int kA[6] = {2, 0, 1, 1, 0, 0}, kB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
            for (int t = 0; t < 6; ++t)
#pragma unroll
                for (int i = 0; i < BA; ++i)
#pragma unroll
                    for (int j = 0; j < BB; ++j) Mma<uint16_t>::run(acc[i][j], fa[i].p[kA[t]], fb[j].p[kB[t]]);
        } else {
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                u32x4_v fa[BA], fb[BB];
#pragma unroll
                for (int i = 0; i < BA; ++i) fa[i] = frag(slot, wa * 16 * BA + 16 * i + fr, ks);
#pragma unroll
                for (int j = 0; j < BB; ++j) fb[j] = frag(slot, TM + wb * 16 * BB + 16 * j + fr, ks);
#pragma unroll
                for (int i = 0; i < BA; ++i)
#pragma unroll
                    for (int j = 0; j < BB; ++j) Mma<T>::run(acc[i][j], fa[i], fb[j]);
            }
        }
    }
    if constexpr (SPLIT) {
        // A value that is not finite has no such parts (its remainder is NaN; that of a value whose rounding
        // overflows is infinite), and a tiny one not all of them: blocks whose sums are not finite and blocks
        // with parts that are not exact are made again from the values themselves, in fp32 MFMAs.
#pragma unroll
        for (int i = 0; i < BA; ++i)
#pragma unroll
            for (int j = 0; j < BB; ++j) {
                bool bad = ((rest_a[i] | rest_b[j]) & 0xffffu) != 0;
#pragma unroll
                for (int r = 0; r < 4; ++r) bad |= (__float_as_uint(acc[i][j][r]) & 0x7f800000u) == 0x7f800000u;
                if (__any(bad)) {
                    const int64_t tok = tok0 + wa * 16 * BA + 16 * i + fr;
                    const int64_t vc = col0 + wb * 16 * BB + 16 * j + fr;
                    const int64_t jr = vc < a.d_pad ? vc : vc - a.d_pad;
                    const bool live_t = tok < a.n, live_c = jr < a.d && vc < 2 * a.d_pad;
                    const float *pt = reinterpret_cast<const float *>(a.mem) + (live_t ? tok : 0) * a.m;
                    const float *pc = reinterpret_cast<const float *>(vc < a.d_pad ? a.wk : a.wv) + (live_c ? jr : 0) * a.m;
                    floatx4 sum = floatx4{0.f, 0.f, 0.f, 0.f};
                    for (int64_t k0 = 0; k0 < a.m; k0 += 32) {  // m % 4 == 0; eight steps' loads in flight
                        float x[8], y[8];
#pragma unroll
                        for (int u = 0; u < 8; ++u) {
                            const bool in = k0 + 4 * u < a.m;
                            x[u] = in && live_t ? *as_global(pt + k0 + 4 * u + fq) : 0.f;
                            y[u] = in && live_c ? *as_global(pc + k0 + 4 * u + fq) : 0.f;
                        }
#pragma unroll
                        for (int u = 0; u < 8; ++u)
                            sum = __builtin_amdgcn_mfma_f32_16x16x4f32(x[u], y[u], sum, 0, 0, 0);
                    }
                    acc[i][j] = sum;
                }
            }
    }
    __syncthreads();  // every wave is done with the ring (and no load is in flight): stage there

    // acc[i][j] lane l: token 16 i + 4 (l >> 4) + r and column 16 j + (l & 15) of the wave's
    // quarter; staged rounded to T as [TM][TN]
#pragma unroll
    for (int i = 0; i < BA; ++i)
#pragma unroll
        for (int j = 0; j < BB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = wa * 16 * BA + 16 * i + 4 * fq + r;
                const int col = wb * 16 * BB + 16 * j + fr;
                uint8_t *p = ring + row * kStagePitch + col * kEs;
                if constexpr (kEs == 2)
                    *reinterpret_cast<uint16_t *>(p) = float_to_bf16_bits_rne(acc[i][j][r]);
                else
                    *reinterpret_cast<float *>(p) = acc[i][j][r];
                // one store at a time: this compiler has merged two of these into a ds_write2_b32 with a wrong
                // offset (tiles of 64 fp32 columns: 51 for 204), which the GPU tests of those tiles show
                asm volatile("" : : : "memory");
            }
    __syncthreads();
    // 16-byte row segments: TM rows x (TN * kEs / 16) segments
    constexpr int kSegs = TN * kEs / 16;
    constexpr int kPerSeg = 16 / kEs;
    const int64_t stride = 2 * a.d;
    for (int it = threadIdx.x; it < TM * kSegs; it += kBlock) {
        const int row = it / kSegs;
        const int seg = it % kSegs;
        const int64_t tok = tok0 + row;
        const int64_t vc = col0 + seg * kPerSeg;  // virtual column: K block, then V block
        const int64_t jr = vc < a.d_pad ? vc : vc - a.d_pad;
        if (tok >= a.n || jr >= a.d || vc >= 2 * a.d_pad) continue;
        const int64_t oc = vc < a.d_pad ? jr : a.d + jr;
        const u32x4_v v = *reinterpret_cast<const u32x4_v *>(ring + row * kStagePitch + seg * 16);
        *as_global(reinterpret_cast<u32x4_v *>(a.kv + (tok * stride + oc) * kEs)) = v;
    }
}

// ---- a few tokens: every weight byte in flight at once ---------------------------------------------
// For a few tokens (takes_few) the GEMM is one read of the weights (33 MB at the Gemma-scale shape) and next to
// no arithmetic, so what counts is how soon all of it is in flight: a tile's ring (above) keeps three
// slabs of its rows in flight and walks 24, a chain of eight memory latencies. Here a workgroup takes
// 16 columns whole: its four waves split the slabs, each wave asks for all of its rows' lines at
// once (buffer_load ... lds, whole lines) and for its token fragments (into registers; a few KB
// that every workgroup reads, so L2 has them), waits once, multiplies, and the waves' partial tiles
// are added in wave order. At 24 slabs a workgroup holds 48 KB of LDS, so three share a CU and the
// 672 workgroups of the Gemma-scale shape are all resident. One token there: 7.3 us, 4.5 TB/s of weights
// with the launch in it (10.2 us in 32 x 96 ring tiles); at 2048 x 1024 3.8 us (7.6), at 1024 x 1024 in
// fp32 4.7 (16.0).
// SW: slabs per wave at most; B: 16-token blocks.
template <typename T, int SW, int B>
__global__ __launch_bounds__(kThreads) void proj_few_kernel(const ProjArgs a) {
    constexpr int kEs = sizeof(T);
    constexpr int kOwn = SW * 2048;  // bytes of a wave's rows
    __shared__ __attribute__((aligned(16))) uint8_t lds[4 * kOwn];
    static_assert(4 * kOwn <= kLdsBytes, "rows fit LDS");
    static_assert(kOwn >= B * 1024, "a wave's partial tiles fit where its rows were");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t vc0 = static_cast<int64_t>(blockIdx.x) * 16;  // virtual column: K block, then V block
    const bool is_v = vc0 >= a.d_pad;
    const int64_t j0 = is_v ? vc0 - a.d_pad : vc0;
    const int32x4 rw = rsrc_of(is_v ? a.wv : a.wk, a.w_bytes);
    const __amdgpu_buffer_rsrc_t rm = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(a.mem), 0, static_cast<int>(a.mem_bytes), kBufferConfig);
    const int sw = (a.slabs + 3) / 4;
    const int s0 = wave * sw, ns = min(sw, a.slabs - s0);  // this wave's slabs (none if ns <= 0)
    // token fragments: lane l holds token 16 b + (l & 15), chunk 4 ks + (l >> 4) of a slab
    const int fr = lane & 15, fq = lane >> 4;
    u32x4_v fa[B][SW][2];
#pragma unroll
    for (int b = 0; b < B; ++b)
#pragma unroll
        for (int i = 0; i < SW; ++i)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const int64_t t = 16 * b + fr;
                const uint32_t kb = static_cast<uint32_t>(s0 + i) * kSlab + static_cast<uint32_t>(4 * ks + fq) * 16u;
                const uint32_t off = t < a.n && i < ns && kb < a.row_bytes ? static_cast<uint32_t>(t) * a.row_bytes + kb
                                                                          : a.mem_bytes;
                fa[b][i][ks] = __builtin_bit_cast(u32x4_v, __builtin_amdgcn_raw_buffer_load_b128(rm, off, 0, 0));
            }
    __builtin_amdgcn_sched_barrier(0);
    uint8_t *own = lds + wave * kOwn;
    const uint32_t own_lds = lds_addr(own);
#pragma unroll
    for (int i = 0; i < 2 * SW; ++i) {  // 8 rows of a slab: lane l takes row 8 (i & 1) + l / 8, chunk swizzled
        if (i / 2 < ns) {
            const int row = 8 * (i & 1) + (lane >> 3);
            const uint32_t kb = static_cast<uint32_t>(s0 + i / 2) * kSlab +
                                static_cast<uint32_t>((lane & 7) ^ ((row >> 1) & 7)) * 16u;
            const uint32_t off = j0 + row < a.d && kb < a.row_bytes
                                     ? static_cast<uint32_t>(j0 + row) * a.row_bytes + kb
                                     : a.w_bytes;
            dma16(rw, __builtin_amdgcn_readfirstlane(own_lds + static_cast<uint32_t>(i) * 1024u), off);
        }
    }
    floatx4 acc[B];
#pragma unroll
    for (int b = 0; b < B; ++b) acc[b] = floatx4{0.f, 0.f, 0.f, 0.f};
    wait_vmcnt<0>();  // the wave's own rows and fragments; no other wave reads them
#pragma unroll
    for (int i = 0; i < SW; ++i)
        if (i < ns)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const int c = ((4 * ks + fq) ^ ((fr >> 1) & 7)) << 4;
                const u32x4_v fb = *reinterpret_cast<const u32x4_v *>(own + i * 2048 + fr * kSlab + c);
#pragma unroll
                for (int b = 0; b < B; ++b) Mma<T>::run(acc[b], fa[b][i][ks], fb);
            }
    // partial tiles [16 B tokens][16 columns] where the wave's rows were (its reads are done: the
    // MFMAs above used them)
#pragma unroll
    for (int b = 0; b < B; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            reinterpret_cast<float *>(own)[(16 * b + 4 * fq + r) * 16 + fr] = acc[b][r];
    __syncthreads();
    for (int e = threadIdx.x; e < B * 128; e += kThreads) {  // two columns of a token
        const int tok = e >> 3, col = (e & 7) * 2;
        if (tok >= a.n || j0 + col >= a.d) continue;
        float v0 = 0.f, v1 = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float *p = reinterpret_cast<const float *>(lds + w * kOwn) + tok * 16 + col;
            v0 += p[0];
            v1 += p[1];
        }
        uint8_t *o = a.kv + (tok * 2 * a.d + (is_v ? a.d : 0) + j0 + col) * kEs;
        if constexpr (kEs == 2)
            *as_global(reinterpret_cast<uint32_t *>(o)) =
                static_cast<uint32_t>(float_to_bf16_bits_rne(v0)) |
                (static_cast<uint32_t>(float_to_bf16_bits_rne(v1)) << 16);
        else
            *as_global(reinterpret_cast<u32x2_v *>(o)) = u32x2_v{__float_as_uint(v0), __float_as_uint(v1)};
    }
}

template <typename T, int B>
int launch_few(const ProjArgs &a, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>(2 * a.d_pad / 16));
    const int sw = (a.slabs + 3) / 4;
    if (sw <= 2) hipLaunchKernelGGL((proj_few_kernel<T, 2, B>), grid, dim3(kThreads), 0, s, a);
    else if (sw <= 4) hipLaunchKernelGGL((proj_few_kernel<T, 4, B>), grid, dim3(kThreads), 0, s, a);
    else if (sw <= 6) hipLaunchKernelGGL((proj_few_kernel<T, 6, B>), grid, dim3(kThreads), 0, s, a);
    else if (sw <= 8) hipLaunchKernelGGL((proj_few_kernel<T, 8, B>), grid, dim3(kThreads), 0, s, a);
    else hipLaunchKernelGGL((proj_few_kernel<T, 12, B>), grid, dim3(kThreads), 0, s, a);
    return check_launch("me_kv_proj (few tokens)");
}

// Every workgroup reads every token's row, so the kernel pays while those reads are few (us, few / ring tiles
// of 32 x 32; model dim x memory dim, bf16: 5376 x 1536, 8 tokens 7.9 / 9.2, 16: 9.2 / 9.2, 32: 13.6 / 9.2;
// 2048 x 1024, 32: 5.2 / 6.1; 8192 x 512, 20: 6.2 / 5.3) and its token blocks are at most two: from 33 tokens bf16
// takes the ring tiles (48 tokens: 2560 x 640 8.1 / 5.7, 5320 x 136 5.4 / 4.4, 1024 x 1024 6.7 / 6.5), fp32, whose
// ring tiles are bound by their MFMAs, from 65 (2048 x 1024, 48: 14.2 / 17.2). Past 50 MB the weights take as
// long either way (8192 x 2048 in bf16, 1 token: 13.6 / 12.6). Rows have at most 48 slabs (96 KB of LDS).
bool takes_few(const ProjArgs &a, int dtype) {
    if (a.n > (dtype == ME_BF16 ? 32 : 64) || a.slabs > 48) return false;
    if (2 * a.d_pad * a.row_bytes > 50'000'000) return false;
    return 2 * a.d_pad / 16 * a.n * a.row_bytes <= (a.n <= 16 || dtype != ME_BF16 ? 22'000'000 : 17'000'000);
}

template <typename T>
int few(const ProjArgs &a, hipStream_t s) {
    if (a.n <= 16) return launch_few<T, 1>(a, s);
    if constexpr (sizeof(T) == 4)
        if (a.n > 32) return launch_few<T, 4>(a, s);
    return launch_few<T, 2>(a, s);
}

template <typename T, int BA, int BB, int R, bool SPLIT = false, int WA = 2>
int launch(ProjArgs a, hipStream_t s) {
    constexpr int TM = 16 * WA * BA, TN = 32 * BB;
    a.tiles_tok = static_cast<int>(ceil_div(a.n, TM));
    const int tiles_col = static_cast<int>(ceil_div(2 * a.d_pad, TN));
    a.tiles_total = a.tiles_tok * tiles_col;
    a.per_xcd = static_cast<int>(ceil_div(a.tiles_total, kXcds));
    hipLaunchKernelGGL((proj_kernel<T, BA, BB, R, SPLIT, WA>), dim3(static_cast<unsigned>(a.per_xcd * kXcds)),
                       dim3(128 * WA), 0, s, a);
    return check_launch("me_kv_proj");
}

}  // namespace
}  // namespace me

using namespace me;

extern "C" int me_kv_proj(const void *mem, int64_t n, int64_t mem_dim, const void *w_key,
                          const void *w_value, int64_t model_dim, int dtype, void *kv,
                          void *stream) {
    ME_CHECK_ARG(dtype == ME_BF16 || dtype == ME_F32, "dtype must be bf16 or fp32");
    ME_CHECK_ARG(n >= 0 && mem_dim >= 1 && model_dim >= 1, "bad shape");
    if (n == 0) return ME_OK;
    ME_CHECK_ARG(mem && w_key && w_value && kv, "null tensor pointer");
    const int64_t es = static_cast<int64_t>(dtype_size(dtype));
    ME_CHECK_ARG(model_dim % 8 == 0, "model_dim must be a multiple of 8");
    ME_CHECK_ARG((mem_dim * es) % 16 == 0, "mem_dim * element size must be a multiple of 16 bytes");
    ME_CHECK_ARG(n * mem_dim * es < (int64_t{1} << 31) && model_dim * mem_dim * es < (int64_t{1} << 31),
                 "mem and each weight must be under 2 GiB");
    ME_CHECK_ARG(n < (int64_t{1} << 24), "too many tokens: at most 2^24 - 1");
    auto al16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    ME_CHECK_ARG(al16(mem) && al16(w_key) && al16(w_value) && al16(kv), "tensors must be 16-byte aligned");
    ProjArgs a{};
    a.mem = static_cast<const uint8_t *>(mem);
    a.wk = static_cast<const uint8_t *>(w_key);
    a.wv = static_cast<const uint8_t *>(w_value);
    a.kv = static_cast<uint8_t *>(kv);
    a.n = n;
    a.d = model_dim;
    a.m = mem_dim;
    a.d_pad = (model_dim + 15) / 16 * 16;
    a.row_bytes = static_cast<uint32_t>(mem_dim * es);
    a.slabs = static_cast<int>(ceil_div(a.row_bytes, kSlab));
    a.mem_bytes = static_cast<uint32_t>(n * mem_dim * es);
    a.w_bytes = static_cast<uint32_t>(model_dim * mem_dim * es);
    hipStream_t s = as_stream(stream);
    // Tiles (measured on MI355X at model dim 5376, mem dim 1536, bf16, unless said otherwise): small
    // batches are bound by how many bytes each CU keeps in flight from L2, so they take the
    // smallest tile whose tiles all find a place at once, two workgroups per CU: 32 x 32 with six slots of
    // 128-byte slabs (19 tokens: 9.2 us; 10.4 with 32 x 96 and four slots; at 2048 x 1024, 128
    // tokens: 6.9, 8.9), 64 x 64 with four (192 tokens: 13.2; 15.6 with 64 x 96; at 3584 x 1536, 256
    // tokens: 12.7, 15.4), 64 x 96 with four (256 tokens: 16.0; 64 x 64 20.3, 128 x 96 17.6, with eight
    // waves 14.8 by itself but 0.2 us more in a decode step; also where they make one round, 128 tokens: 12.8,
    // 64 x 64 13.9). Tiles of one round, one to a CU, take eight
    // waves, two per SIMD as two smaller workgroups are, with fewer bytes for the same outputs: 64 x 64 with
    // six slots (48 tokens: 9.8, 10.5 with four waves, the decode step 24.6 -> 23.7; at 2048 x 1024, 256
    // tokens: 7.8, 8.2), 256 x 96 (512 tokens: 24.4, 29.1 in 64 x 128; the decode step of 500 tokens 46.7 ->
    // 42.8) and 256 x 128 with three (700 tokens: 28.2, 33.6; at 3584 x 1536, 1024 tokens: 27.9, 33.8; at
    // 2048 x 1024, 2042 tokens: 22.2, 25.5). Larger batches take the gate's 256 x 224 tiles (one
    // workgroup per CU, a matrix core's worth of work per barrier)
    // or 64 x 128 ones (three slots, two workgroups per CU), whichever needs the less time for the
    // whole rounds its tiles make on 256 CUs: a round of the first takes about 7 us and 1.25 us per
    // slab, 256 tiles of the second 1.2 us and 0.33 us per slab, but never under 1.6 such (512
    // tokens: 33.4 and 30.5 us; 768: 33.7, 36.7; 1237: 39.0, 61.6; 2048: 69.9, 101; 8192: 233, 398;
    // at 2048 x 1024, 1024 tokens: 24.8, 14.9; 2048: 25.7, 27.1; 8192: 76.7, 107; at 1024 x 512, 2048
    // tokens: 16.9, 10.6). 64 x 128 also where the memory width rules the first out (5320 x 136, 4096 tokens:
    // 43.2; 55.5 on 128 x 192 tiles, which were slower than one of the others for every shape measured).
    // fp32: fp32 MFMAs on 32 x 64 and 32 x 128 tiles, split products on 64 x 64 and 64 x 128 ones, whichever the
    // rule below takes least time for: with c tiles on the fullest CU (two at a time) they take about 11, 19, 17.5
    // and 29 us per c at a memory dim of 1024, and as much less or more as that is shorter or longer (us in that
    // order, model dim x memory dim: 1024 x 1024, 200 tokens 17.4, 24.7, 27.2, 38.7, 512: 26.2, 25.5, 28.4, 39.5,
    // 1000: 46.7, 41.5, 39.8, 40.6, 2048: 89.9, 78.4, 75.4, 63.1, where 64 x 128 tiles of fp32 MFMAs took 76-82;
    // 3584 x 1536, 257: 65.7, 58.9, 81.2, 82.9; 2560 x 640, 800: 58.4, 50.6, 57.8, 58.0).
    if (takes_few(a, dtype)) return dtype == ME_BF16 ? few<uint16_t>(a, s) : few<float>(a, s);
    constexpr int64_t kCus = 256;
    auto tiles = [&](int tokens, int cols) { return ceil_div(n, tokens) * ceil_div(2 * a.d_pad, cols); };
    if (dtype == ME_BF16) {
        if (tiles(32, 32) <= 2 * kCus) return launch<uint16_t, 1, 1, 6>(a, s);
        if (tiles(64, 64) <= kCus) return launch<uint16_t, 1, 2, 6, false, 4>(a, s);
        if (tiles(64, 64) <= 2 * kCus && tiles(64, 96) > kCus) return launch<uint16_t, 2, 2, 4>(a, s);
        if (tiles(64, 96) <= 2 * kCus) return launch<uint16_t, 2, 3, 4>(a, s);
        if (tiles(64, 128) > 2 * kCus) {  // three rounds and more of those below
            if (tiles(256, 96) <= kCus) return launch<uint16_t, 4, 3, 3, false, 4>(a, s);
            if (tiles(256, 128) <= kCus) return launch<uint16_t, 4, 4, 3, false, 4>(a, s);
        }
        const float small = static_cast<float>(ceil_div(tiles(64, 128), kCus));
        if (a.row_bytes % kSlab == 0 && a.slabs >= 3 && n * model_dim * 4 < (int64_t{1} << 31)) {
            const float large = static_cast<float>(ceil_div(ceil_div(n, 256) * 2 * ceil_div(model_dim, 224), kCus));
            if (large * (7.f + 1.25f * a.slabs) <= 2.f + fmaxf(small, 1.6f) * (1.2f + 0.33f * a.slabs))
                return kv_proj_224(mem, n, mem_dim, w_key, w_value, model_dim, kv, s);
        }
        return launch<uint16_t, 2, 4, 3>(a, s);
    }
    // a tile alone on its CU takes longer than its share of two
    auto per_cu = [&](int tokens, int cols) { return fmaxf(1.3f, static_cast<float>(ceil_div(tiles(tokens, cols), kCus))); };
    const float t32x64 = 11.f * per_cu(32, 64) + 3.5f, t32x128 = 19.f * per_cu(32, 128) + 4.5f;
    const float t64x64 = 17.5f * per_cu(64, 64) + 5.f, t64x128 = 29.f * per_cu(64, 128) + 3.f;
    const float least = fminf(fminf(t32x64, t32x128), fminf(t64x64, t64x128));
    if (t32x64 == least) return launch<float, 1, 2, 5>(a, s);
    if (t64x64 == least) return launch<float, 2, 2, 4, true>(a, s);
    if (t64x128 == least) return launch<float, 2, 4, 3, true>(a, s);
    return launch<float, 1, 4, 4>(a, s);
}
