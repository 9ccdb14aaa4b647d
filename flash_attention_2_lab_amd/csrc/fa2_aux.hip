// The reference module's other operators, for gfx950: a device copy, FP32 attention
// scores, FP32 attention forwards (kernels in fa2_forward_f32.h) and a 16x64x16 FP16 matrix
// product, both on MFMA. Any pointer aligned to its element type works (views with offsets
// included).
//
// Entry points (include/fa2_mi355x.h):
//   fa2_copy                    <- copy_cuda (reference csrc/copy_kernel.cu:23-53)
//   fa2_attention_scores_f32    <- naive_attention_scores (csrc/naive_attention.cu:174-201, 330-418)
//   fa2_attention_forward_f32   <- naive_attention_forward, block_attention_forward
//                                  (csrc/naive_attention.cu:48-172, 249-328, 420-502),
//                                  tiled_attention_forward (csrc/tiled_attention.cu:273-333),
//                                  tilewise_attention_forward (csrc/tilewise_attention.cu:337-388)
//   fa2_matmul_16x64x16_f16     <- wmma_matmul_16x64x16 (csrc/wmma_matmul.cu:51-193, 250-315)

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <math.h>

#include "fa2_mi355x.h"
#include "fa2_forward_f32.h"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

int hip_status(hipError_t err) {
    return err == hipSuccess ? FA2_STATUS_SUCCESS : FA2_STATUS_HIP_ERROR_BASE + (int)err;
}

bool aligned_to(const void* p, uintptr_t bytes) {
    return (reinterpret_cast<uintptr_t>(p) & (bytes - 1)) == 0;
}

// ---------------------------------------------------------------------------
// Copy: grid-stride over elements of the widest size (16, 8, 4, 2 or 1 bytes)
// that divides both addresses and the byte count.
template <typename T>
__global__ __launch_bounds__(256) void copy_kernel(const T* __restrict__ src, T* __restrict__ dst,
                                                   int64_t count) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride)
        dst[i] = src[i];
}

template <typename T>
hipError_t launch_copy(const void* src, void* dst, int64_t bytes, hipStream_t stream) {
    const int64_t count = bytes / (int64_t)sizeof(T);
    const int64_t blocks = count / 256 + (count % 256 != 0);
    const unsigned grid = (unsigned)(blocks < 65536 ? blocks : 65536);
    hipLaunchKernelGGL((copy_kernel<T>), dim3(grid), dim3(256), 0, stream, static_cast<const T*>(src),
                       static_cast<T*>(dst), count);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Scores S[bh][i][j] = scale * sum_d Q[bh][i][d] K[bh][j][d], FP32, any seq_len and
// head_dim. A workgroup of 4 waves owns 64 rows and a range of 64-column blocks of S; a wave
// computes 32 x 32 of a block on v_mfma_f32_32x32x2_f32 (A = Q rows, B = K rows; lane (m, h)
// gives row m of its operand, k = h; in group j of 8 dimensions half h takes dimensions
// 8j + 4h .. +3). Operands go through LDS by LDS-DMA in chunks of 64 dimensions: units of 32
// rows, 8 KiB, 16-byte chunk c of row r at c ^ (r % 16), which keeps the 16-byte reads free
// of bank conflicts. Rows past seq_len and dimensions past head_dim are fetched as zeros. Two
// accumulators, as in the forward.
//
// Bound at head_dim 64 by the FP32 MFMA rate and the write of S about equally (7 us each at
// B1 H8 N1024): a step (one chunk of one block) fetches the next step's operands before its
// products, and the stores of a block run beside the products of the next. kSingle
// (head_dim <= 64) keeps Q in registers, so that a step fetches K alone and 32 KiB of LDS
// are enough; 112 VGPRs leave room for four workgroups per CU. A register of the accumulator is
// stored as two 128-byte row segments; rows and columns past seq_len fall outside num_records.
// Measured on MI355X (graph replays, FP32 VALU tile with 4-byte LDS reads -> this): B1 H8
// N1024 D64 31.5 -> 15.6 us, D16 12.4 -> 9.4 us; B1 H8 N2048 D64 95 -> 47 us; B4 H8 N2048
// D128 634 -> 348 us; B1 H1 N64 D64 9.6 -> 3.3 us. One block per workgroup, its phases in
// turn, took 17.2 us at B1 H8 N1024 D64.
//
// kWide: head_dim a multiple of 4 and at most 2^16, and 16-byte aligned pointers: 16-byte
// LDS-DMA, four rows an instruction. Otherwise 4-byte LDS-DMA, one row an instruction with a
// descriptor of its own, for any head_dim and alignment. kNarrow (head_dim at most 16): rows of
// 16 dimensions in LDS, four to a 4-byte LDS-DMA. The fetch instructions are what small
// operands cost, so kNarrow, the one-row fetch of kSingle and any one-row fetch of a unit of up to
// kFewRows rows issue none for rows past seq_len, whose products are not stored. FP32 VALU tile ->
// all 32 rows of a unit, one an instruction -> this: B1 H8 N1024 D3 11.5 -> 11.9 -> 8.8 us, 2048
// heads of N7 D3 6.8 -> 11.4 -> 5.2, of N7 D17 11.5 -> 12.9 -> 7.9, 4096 heads of N1 D4 on 4-byte
// aligned storage 11.4 -> 20.6 -> 8.1, of N1 D65 47.2 -> 52.3 -> 33.4, 2048 of N16 D65 26.4 -> 27.5 ->
// 22.4. Past 64 dimensions a loop to the last row alone lost at 32 rows (8 heads of N1000 D65 33.7
// -> 28.6 -> 30.7, with this rule 29.0) and at 48 keys (700 heads 15.1 -> 12.6 -> 13.9, with it 12.4).
constexpr int kScoreTile = 64;
constexpr int kNarrowDims = 16;
constexpr int kFewRows = 24;

template <bool kWide, bool kSingle, bool kNarrow = false>
__global__ __launch_bounds__(256) void scores_f32_kernel(const float* __restrict__ query,
                                                         const float* __restrict__ key,
                                                         float* __restrict__ scores, int seq_len,
                                                         int head_dim, uint32_t tiles, uint32_t ranges,
                                                         uint32_t total_blocks, float scale) {
    static_assert(!kNarrow || (kSingle && !kWide), "the narrow fetch");
    constexpr int kPitch = kNarrow ? kNarrowDims * 4 : 256;  // bytes of a row in LDS
    constexpr int kGroups = kPitch / 32;                      // of 8 dimensions
    constexpr int kUnitBytes = 32 * kPitch;
    constexpr int kOutOfRange = 0x40000000;  // past every num_records here (a row of S is at most 2 MiB in HBM's 288 GB)
    constexpr int kParts = kSingle ? 2 : 1;  // waves that share the fetch of a unit
    constexpr int kSlotBytes = (kSingle ? 2 : 4) * kUnitBytes;  // K alone, or K and Q
    __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * kSlotBytes];
    const uint32_t id = blockIdx.y * gridDim.x + blockIdx.x;
    if (id >= total_blocks) return;
    const uint32_t logical = xcd_contiguous(id, total_blocks);
    // Uniform values, but divided on the VALU: back to SGPRs, which the descriptors need.
    const uint32_t bh = __builtin_amdgcn_readfirstlane(logical / (tiles * ranges));
    const uint32_t rem = logical - bh * (tiles * ranges);
    const uint32_t row_block = __builtin_amdgcn_readfirstlane(rem / ranges);
    const uint32_t range = rem - row_block * ranges;
    const int row0 = (int)row_block * kScoreTile;
    const int col_begin = (int)__builtin_amdgcn_readfirstlane(range * tiles / ranges);  // tiles * ranges < 2^32
    const int col_end = (int)__builtin_amdgcn_readfirstlane((range + 1) * tiles / ranges);

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int m = lane & 31;
    const int h = lane >> 5;
    const int chunks = kSingle ? 1 : (int)(((int64_t)head_dim + 63) / 64);
    const int64_t row_bytes = (int64_t)head_dim * 4;
    const uint32_t smem_addr = lds_address(smem);

    // Share `part` of the unit of rows `first`.. `first`+31 and dimensions 64 * chunk.. of
    // `source`, to the unit at `lds`.
    auto fetch_unit = [&](const float* source, int first, int chunk, uint32_t lds, int part) {
        const uint32_t d0 = (uint32_t)chunk * 64u;
        const uint64_t base = reinterpret_cast<uint64_t>(source) + ((uint64_t)bh * seq_len + first) * row_bytes + (uint64_t)d0 * 4;
        const int rows = min(32, seq_len - first);  // may be negative: nothing to fetch
        u32x4 d;
        d[3] = 0x00020000u;
        if (kNarrow && rows <= 0) return;
        if (kWide || kNarrow) {
            d[0] = __builtin_amdgcn_readfirstlane((uint32_t)base);
            d[1] = __builtin_amdgcn_readfirstlane((uint32_t)(base >> 32) & 0xffffu);
            d[2] = __builtin_amdgcn_readfirstlane(rows > 0 ? (uint32_t)(rows * row_bytes) - d0 * 4u : 0u);
#pragma unroll
            for (int i = 0; i < 8 / kParts; ++i) {
                const int n = i * kParts + part;
                if (kNarrow && 4 * n >= rows) break;
                const int row = 4 * n + (lane >> 4);
                if (kNarrow) {
                    const int dim = (lane & 15) ^ ((n & 3) << 2);
                    dma4(d, lds + n * 256, dim < head_dim ? (int)(row * row_bytes) + 4 * dim : kOutOfRange);
                } else {
                    const int chunk16 = (lane & 15) ^ (row & 15);
                    const bool in = d0 + 4u * chunk16 < (uint32_t)head_dim;
                    dma16(d, lds + n * 1024, in ? (int)(row * row_bytes) + 16 * chunk16 : kOutOfRange);
                }
            }
        } else {
            auto fetch_row = [&](int row, bool exists) {
                const uint64_t a = base + (uint64_t)row * row_bytes;
                d[0] = __builtin_amdgcn_readfirstlane((uint32_t)a);
                d[1] = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu);
                d[2] = __builtin_amdgcn_readfirstlane(exists ? min(64u, (uint32_t)head_dim - d0) * 4u : 0u);
                dma4(d, lds + row * 256, (lane << 2) ^ ((row & 15) << 4));
            };
            if (kSingle || rows <= kFewRows) {
                for (int row = part; row < rows; row += kParts) fetch_row(row, true);
            } else {
                for (int row = 0; row < 32; ++row) fetch_row(row, row < rows);
            }
        }
    };
    // A step's operands into ring slot `slot`. kSingle: waves 2u and 2u+1 fetch half of K's
    // unit u each. Otherwise wave w fetches unit w: K, K, Q, Q.
    auto fetch = [&](int col, int chunk, int slot) {
        const uint32_t lds = smem_addr + (uint32_t)(slot * kSlotBytes);
        if (kSingle) fetch_unit(key, col * kScoreTile + 32 * (wave >> 1), chunk, lds + (wave >> 1) * kUnitBytes, wave & 1);
        else fetch_unit(wave < 2 ? key : query, (wave < 2 ? col * kScoreTile : row0) + 32 * (wave & 1), chunk,
                        lds + wave * kUnitBytes, 0);
    };
    // The wave's fetches have landed and its LDS reads are done: behind the barrier the other
    // waves read the one slot and refill the other.
    auto landed = [&]() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    const uint32_t lane_read = smem_addr + (uint32_t)(m * kPitch + ((h ^ (kNarrow ? (m >> 2) & 3 : m & 15)) << 4));
    auto read = [&](int slot, int unit, int j) {
        return *reinterpret_cast<const FA2_LDS f32x4*>(
            (size_t)((lane_read ^ (uint32_t)(j << 5)) + (uint32_t)(slot * kSlotBytes + unit * kUnitBytes)));
    };
    f32x4 qf[8];
    if (kSingle) {
        // Q through slot 1, which is free until the second step's fetch.
        fetch_unit(query, row0 + 32 * (wave >> 1), 0, smem_addr + (uint32_t)(kSlotBytes + (wave >> 1) * kUnitBytes), wave & 1);
        fetch(col_begin, 0, 0);
        landed();
#pragma unroll
        for (int j = 0; j < kGroups; ++j) qf[j] = read(1, wave >> 1, j);
        // Every wave has read its Q before any wave's fetch refills slot 1. (The compiler may
        // sink LDS reads past a plain barrier; the asm takes their results.)
#pragma unroll
        for (int j = 0; j < kGroups; ++j) asm volatile("" : "+v"(qf[j]));
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    } else {
        fetch(col_begin, 0, 0);
        landed();
    }

    // S rows of this wave through a descriptor of its own: rows past seq_len are outside it.
    const int out_row = row0 + 32 * (wave >> 1);
    const uint64_t out_base = reinterpret_cast<uint64_t>(scores) + ((uint64_t)bh * seq_len + out_row) * (uint64_t)seq_len * 4u;
    // readfirstlane returns a signed int: back to unsigned before it is widened.
    const uint32_t out_lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)out_base);
    const uint32_t out_hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(out_base >> 32));
    const uint32_t out_bytes = (uint32_t)max(0, min(32, seq_len - out_row)) * (uint32_t)seq_len * 4u;
    const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(
        reinterpret_cast<void*>((uint64_t)out_hi << 32 | out_lo), (short)0,
        (int)__builtin_amdgcn_readfirstlane(out_bytes), 0x00020000);

    int slot = 0;
    for (int col = col_begin; col < col_end; ++col) {
        f32x16 acc[2];
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[0][i] = acc[1][i] = 0.0f;
        auto multiply = [&](f32x4 q, f32x4 k) {
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(q[e], k[e], acc[e & 1], 0, 0, 0);
        };
        for (int chunk = 0; chunk < chunks; ++chunk) {
            if (chunk + 1 < chunks) fetch(col, chunk + 1, slot ^ 1);
            else if (col + 1 < col_end) fetch(col + 1, 0, slot ^ 1);
            const int groups = (int)min(8u, ((uint32_t)head_dim - (uint32_t)chunk * 64u + 7u) / 8u);  // of 8 dimensions
            if (!kNarrow && groups == 8) {
                f32x4 kf[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) kf[j] = read(slot, wave & 1, j);
                __builtin_amdgcn_sched_barrier(0);  // all reads in flight before the first product
#pragma unroll
                for (int j = 0; j < 8; ++j) multiply(kSingle ? qf[j] : read(slot, 2 + (wave >> 1), j), kf[j]);
            } else {
#pragma unroll
                for (int j = 0; j < min(7, kGroups); ++j)
                    if (j < groups) multiply(kSingle ? qf[j] : read(slot, 2 + (wave >> 1), j), read(slot, wave & 1, j));
            }
            if (chunk + 1 < chunks) landed();
            slot ^= 1;
        }
        // The next block's operands have landed before the stores are issued, so that the
        // wait does not include them.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const int out_col = col * kScoreTile + 32 * (wave & 1) + m;
        const int lane_offset = out_col < seq_len ? 4 * h * seq_len * 4 + out_col * 4 : kOutOfRange;
#pragma unroll
        for (int i = 0; i < 16; ++i)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint((acc[0][i] + acc[1][i]) * scale), out,
                                                  lane_offset + (8 * (i >> 2) + (i & 3)) * seq_len * 4, 0, 0);
        if (col + 1 < col_end) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
}

// ---------------------------------------------------------------------------
// C = A B for one 16x64 (A) by 64x16 (B) FP16 pair per wavefront, FP32 result, as
// two v_mfma_f32_16x16x32_f16. Operand layout of that instruction: lane l holds,
// for A, row l%16 and reduction indices 8(l/16)..8(l/16)+7; for B, column l%16
// and the same reduction indices; the 16x16 FP32 result gives lane l column l%16,
// rows 4(l/16)..4(l/16)+3.
__global__ __launch_bounds__(64) void matmul_16x64x16_kernel(const _Float16* __restrict__ a,
                                                             const _Float16* __restrict__ b,
                                                             float* __restrict__ c) {
    const int64_t m = blockIdx.x;
    const int lane = threadIdx.x;
    const int rc = lane & 15;       // row of A, column of B and of C
    const int kg = lane >> 4;       // reduction group
    const _Float16* a_m = a + m * 16 * 64;
    const _Float16* b_m = b + m * 64 * 16;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        f16x8 av, bv;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int k = 32 * h + 8 * kg + j;
            av[j] = a_m[rc * 64 + k];
            bv[j] = b_m[k * 16 + rc];
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bv, acc, 0, 0, 0);
    }
    float* c_m = c + m * 16 * 16;
#pragma unroll
    for (int i = 0; i < 4; ++i) c_m[(4 * kg + i) * 16 + rc] = acc[i];
}

}  // namespace

extern "C" int fa2_copy(const void* src, void* dst, int64_t bytes, void* stream) {
    if (bytes < 0) return FA2_STATUS_NEGATIVE_DIMENSION;
    if (bytes == 0) return FA2_STATUS_SUCCESS;
    if (!src || !dst) return FA2_STATUS_NULL_POINTER;
    const uintptr_t bits = reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst) |
                           static_cast<uintptr_t>(bytes);
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipError_t err;
    if ((bits & 15) == 0) err = launch_copy<u32x4>(src, dst, bytes, s);
    else if ((bits & 7) == 0) err = launch_copy<uint64_t>(src, dst, bytes, s);
    else if ((bits & 3) == 0) err = launch_copy<uint32_t>(src, dst, bytes, s);
    else if ((bits & 1) == 0) err = launch_copy<uint16_t>(src, dst, bytes, s);
    else err = launch_copy<uint8_t>(src, dst, bytes, s);
    return hip_status(err);
}

extern "C" int fa2_attention_scores_f32(const float* query, const float* key, float* scores,
                                        int64_t batch_heads, int64_t seq_len, int64_t head_dim,
                                        void* stream) {
    if (batch_heads < 0 || seq_len < 0 || head_dim < 0) return FA2_STATUS_NEGATIVE_DIMENSION;
    if (batch_heads == 0 || seq_len == 0) return FA2_STATUS_SUCCESS;
    if (!query || !key || !scores) return FA2_STATUS_NULL_POINTER;
    if (!aligned_to(query, 4) || !aligned_to(key, 4) || !aligned_to(scores, 4)) return FA2_STATUS_MISALIGNED;
    if (seq_len > INT32_MAX || head_dim > INT32_MAX) return FA2_STATUS_TOO_LARGE;
    const int64_t tiles = (seq_len + kScoreTile - 1) / kScoreTile;  // seq_len <= INT32_MAX: no overflow
    if (batch_heads > (int64_t)UINT32_MAX / (tiles * tiles)) return FA2_STATUS_TOO_LARGE;
    // scale = 1/sqrt(head_dim) in FP32, as the reference's host code computes it
    // (head_dim 0 gives +inf and scores of 0 * inf = NaN there too).
    const float scale = 1.0f / sqrtf((float)head_dim);
    // Workgroups per row of blocks: enough for four workgroups per CU, and at most 8 blocks a
    // workgroup, so that the last round is short. At B1 H8 N1024, 15.6 us at 1024 workgroups
    // against 16.0, 18.3 and 16.8 at 512, 1280 and 2048.
    const int64_t rows = batch_heads * tiles;
    const int64_t wanted = (1024 + rows - 1) / rows;
    int64_t ranges = (tiles + 7) / 8 > wanted ? (tiles + 7) / 8 : wanted;
    if (ranges > tiles) ranges = tiles;
    const int64_t total = rows * ranges;
    constexpr int64_t kMaxX = (int64_t)1 << 22;  // a grid's x dimension times 256 stays below 2^32
    const int64_t x = total < kMaxX ? total : kMaxX;
    const dim3 grid((unsigned)x, (unsigned)((total + x - 1) / x));
    const bool wide = head_dim % 4 == 0 && head_dim <= 65536 && aligned_to(query, 16) && aligned_to(key, 16);
    // Up to 16 keys the narrow fetch also beats the wide one (2048 heads of D8 at N7 6.5 -> 5.1 us,
    // at N16 6.5 -> 5.6), beyond no longer (B1 H8 N1024 D8 8.5 -> 8.6).
    const auto kernel = head_dim <= kNarrowDims && (!wide || seq_len <= 16) ? scores_f32_kernel<false, true, true>
                        : head_dim <= 64 ? (wide ? scores_f32_kernel<true, true> : scores_f32_kernel<false, true>)
                                         : (wide ? scores_f32_kernel<true, false> : scores_f32_kernel<false, false>);
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, static_cast<hipStream_t>(stream), query, key, scores, (int)seq_len,
                       (int)head_dim, (uint32_t)tiles, (uint32_t)ranges, (uint32_t)total, scale);
    return hip_status(hipGetLastError());
}

extern "C" int fa2_attention_forward_f32(const float* query, const float* key, const float* value,
                                         float* output, int64_t batch_heads, int64_t seq_len,
                                         int64_t head_dim, void* stream) {
    if (batch_heads < 0 || seq_len < 0 || head_dim < 0) return FA2_STATUS_NEGATIVE_DIMENSION;
    if (head_dim != 64 && head_dim != 128) return FA2_STATUS_BAD_HEAD_DIM;
    if (batch_heads == 0 || seq_len == 0) return FA2_STATUS_SUCCESS;
    if (!query || !key || !value || !output) return FA2_STATUS_NULL_POINTER;
    if (!aligned_to(query, 4) || !aligned_to(key, 4) || !aligned_to(value, 4) || !aligned_to(output, 4))
        return FA2_STATUS_MISALIGNED;
    if (seq_len > INT32_MAX) return FA2_STATUS_TOO_LARGE;
    const int64_t tiles = (seq_len + 63) / 64;  // seq_len <= INT32_MAX: no overflow
    if (batch_heads > (int64_t)UINT32_MAX / tiles) return FA2_STATUS_TOO_LARGE;
    const float scale_log2 = 1.0f / sqrtf((float)head_dim) * 1.4426950408889634074f;
    hipStream_t s = static_cast<hipStream_t>(stream);
    // 4-byte aligned pointers (views with an offset) take the instantiations with 4-byte
    // LDS-DMA.
    const bool wide = aligned_to(query, 16) && aligned_to(key, 16) && aligned_to(value, 16) && aligned_to(output, 16);
    const auto run = head_dim == 64 ? (wide ? launch_f32_forward<64, true> : launch_f32_forward<64, false>)
                                    : (wide ? launch_f32_forward<128, true> : launch_f32_forward<128, false>);
    const hipError_t err = run(query, key, value, output, batch_heads, seq_len, scale_log2, s);
    return err == hipSuccess ? FA2_STATUS_SUCCESS : FA2_STATUS_HIP_ERROR_BASE + (int)err;
}

extern "C" int fa2_matmul_16x64x16_f16(const void* a, const void* b, float* c, int64_t batch,
                                       void* stream) {
    if (batch < 0) return FA2_STATUS_NEGATIVE_DIMENSION;
    if (batch == 0) return FA2_STATUS_SUCCESS;
    if (!a || !b || !c) return FA2_STATUS_NULL_POINTER;
    if (!aligned_to(a, 2) || !aligned_to(b, 2) || !aligned_to(c, 4)) return FA2_STATUS_MISALIGNED;
    if (batch > (int64_t)UINT32_MAX) return FA2_STATUS_TOO_LARGE;
    hipLaunchKernelGGL(matmul_16x64x16_kernel, dim3((unsigned)batch), dim3(64), 0,
                       static_cast<hipStream_t>(stream), static_cast<const _Float16*>(a),
                       static_cast<const _Float16*>(b), c);
    return hip_status(hipGetLastError());
}
