// RMSNorm + Linear as ONE kernel on the matrix cores (gfx950), optionally over gathered rows.
//
//   n   = x[row] * rsqrt(mean(x[row]^2) + eps) * w_norm               x fp32 or bf16, 128 channels
//   out = bf16(n W^T + bias)                                          W (N, 128) bf16, N % 64 == 0
// Reference: `self.kv_bullet(self.norm_bullet(bullets))` (models/yemong/attention.py:150-151),
// `self.qkv(self.norm1(x))` (:94-96,132) and the temporal block's `linear1(norm1(x))`
// (models/yemong/griffin.py:269-272) as they run under bf16 autocast: nn.RMSNorm, autocast's
// cast, nn.Linear.
//
// With `row_index` the kernel reads row row_index[r] of x for output row r, and with `n_rows`
// (a device-side count) it stops after that many rows: the projection then runs over the
// bullets in flight only (a compact list built on the device), never over the empty slots,
// without the host ever learning how many there are.
//
// A wave owns 32 rows.  Rows come in as whole 256-byte runs through LDS (two passes of 64
// channels), each lane ends up with its row's channels in the k-slot order
//   ch(ks, h, e) = 16ks + 8(e/4) + 4h + e%4      (lane = 32h + m, k-slot e of step ks)
// which is the B operand of out^T = W n^T on v_mfma_f32_32x32x16_bf16.  The packed weights
// list output features so that a lane's 16 results per 32-feature block are two runs of 8
// consecutive features (16-byte stores, the two lanes of a row side by side):
//   [fb][ks][l][e] = W[32fb + 16((r/8)/2) + 8((r/4)%2) + 4((r/8)%2) + r%4][ch(ks, l/32, e)],  r = l%32
// Weights stream through LDS in chunks of 64 features (16 KB), double-buffered.  A work-group takes chunks_per_group of them
// (blockIdx.y names which): all of them when the rows fill the chip, few when they do not, so that a small call is not one
// work-group's walk through every chunk.  16 environments x 12 tokens, 384 features: 10.6 -> 7.4 us.
//
// bf16 rows (what an encoder under bf16 autocast hands over) are 256 bytes: one pass brings them in whole, and the
// staging area holds them as they are.  The kernel is bound by its bytes, so they are read in the type they have and only
// where a bullet is in flight; the library's norm and projection over every slot that they went through before took 1.6 of
// the 2.23 ms of a rollout step of 7808 environments x 80 slots (now 0.86 ms).

#include "common.h"

namespace bnb {

constexpr int kNlD = 128;
constexpr int kNlWaves = 4;
constexpr int kNlThreads = kNlWaves * kWave;
constexpr int kNlChunkFeatures = 64;
constexpr int kNlChunkHalfs = kNlChunkFeatures * kNlD;                 // 8192 bf16 = 16 KB
constexpr int kNlPrefetch = kNlChunkHalfs / 8 / kNlThreads;           // 16-byte pieces per thread per chunk
constexpr int kNlHalfPitch = 64 + 4;                                   // floats per staged half row (bank spread)
constexpr int kNlRowPitch = kNlD + 8;                                  // halfs per staged bf16 row
static_assert(kNlRowPitch * 2 <= kNlHalfPitch * 4, "a staged bf16 row fits the slice's row pitch");

// KEEP: n leaves as well (n_out, the update's form; float32 rows, no list, no bias).  Held to the registers of three work-groups
// per CU, as many as the other forms have.  The row waits in float32 for its factor, which costs 1 to 5 us a launch beside
// rounding the bf16 operand once more: 93,696 rows x 384 features 28.8 -> 29.9 us, 393,216 rows 122 -> 128 us.
template <typename XT, bool KEEP>
__global__ __launch_bounds__(kNlThreads, KEEP ? 3 : 1) void norm_linear_kernel(
    const XT *__restrict__ x, int64_t x_stride, const int32_t *__restrict__ row_index,
    const int32_t *__restrict__ n_rows, const float *__restrict__ norm_w, float eps,
    const uint16_t *__restrict__ wpack, const float *__restrict__ bias, uint16_t *__restrict__ out, int64_t R, int N,
    int chunks_per_group, uint16_t *__restrict__ n_out)
{
    // staging area for the rows (prologue) and the two weight buffers (loop) share this space
    constexpr int kStageFloats = kNlWaves * 32 * kNlHalfPitch;                       // 8704 floats = 34 KB
    constexpr int kLdsBytes = kStageFloats * 4 > 2 * kNlChunkHalfs * 2 ? kStageFloats * 4 : 2 * kNlChunkHalfs * 2;
    __shared__ __align__(16) unsigned char s_raw[kLdsBytes];
    float *s_stage = reinterpret_cast<float *>(s_raw);
    uint16_t *s_w = reinterpret_cast<uint16_t *>(s_raw);

    const int64_t rows = !KEEP && n_rows != nullptr ? (int64_t)*n_rows : R;
    const int64_t block_row0 = (int64_t)blockIdx.x * (kNlWaves * 32);
    if (block_row0 >= rows) return;  // whole work-group past the end of the (device-side) row count

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 31;
    const int half = lane >> 5;

    u32x4 pre[kNlPrefetch];
    auto fetch = [&](int c) {
        const u32x4 *src = reinterpret_cast<const u32x4 *>(wpack + (int64_t)c * kNlChunkHalfs);
#pragma unroll
        for (int q = 0; q < kNlPrefetch; ++q) pre[q] = src[tid + q * kNlThreads];
    };
    auto stash = [&](int buf) {
        u32x4 *dst = reinterpret_cast<u32x4 *>(s_w + buf * kNlChunkHalfs);
#pragma unroll
        for (int q = 0; q < kNlPrefetch; ++q) dst[tid + q * kNlThreads] = pre[q];
    };
    const int c0 = blockIdx.y * chunks_per_group, c_end = c0 + chunks_per_group;  // the launcher divides the chunks evenly
    if (!KEEP) fetch(c0);

    // ---- rows in: a quarter-wave per 256-byte half row, two passes over the channels ----
    const int64_t row0 = block_row0 + wave * 32;
    float *stage = s_stage + wave * (32 * kNlHalfPitch);
    const int io_row = lane >> 4;        // 4 rows per instruction
    const int io_col = (lane & 15) * 4;  // this lane's four channels within the half row
    int64_t src_row[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        int64_t r = row0 + 4 * j + io_row;
        r = r < rows ? r : rows - 1;
        src_row[j] = !KEEP && row_index != nullptr ? (int64_t)row_index[r] : r;
    }
    // The per-row factor rsqrt(mean(x^2) + eps) is a scalar of the output row, so it is applied
    // to the products instead of the operand: the operand is bf16(x * w_norm), formed as the
    // channels arrive (the row never sits in registers as fp32), same relative rounding.
    bf16x8 nb[8];
    float ss = 0.0f;
    [[maybe_unused]] float kept[8][8];  // KEEP: the row itself, until its factor is known
    auto operand = [&](int ks, const float (&t)[8]) {  // k-slots of contraction step ks: channels 16 ks + ...
        if constexpr (KEEP) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                kept[ks][e] = t[e];
                ss = fmaf(t[e], t[e], ss);
            }
            return;
        }
        const f32x4 wl = *reinterpret_cast<const f32x4 *>(norm_w + 16 * ks + 4 * half);
        const f32x4 wh = *reinterpret_cast<const f32x4 *>(norm_w + 16 * ks + 8 + 4 * half);
        const float wv[8] = {wl.x, wl.y, wl.z, wl.w, wh.x, wh.y, wh.z, wh.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            nb[ks][e] = (__bf16)(t[e] * wv[e]);
            ss = fmaf(t[e], t[e], ss);
        }
    };
    if constexpr (is_bf16<XT>::value) {
        uint16_t *stage_x = reinterpret_cast<uint16_t *>(stage);  // 32 x 136 halfs fill the slice's 32 x 68 floats
        u32x4 xv[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            xv[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(x + src_row[j] * x_stride + 2 * io_col));
#pragma unroll
        for (int j = 0; j < 8; ++j)
            *reinterpret_cast<u32x4 *>(stage_x + (4 * j + io_row) * kNlRowPitch + 2 * io_col) = xv[j];
        wave_lds_handover();
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            const uint16_t *sp = stage_x + m * kNlRowPitch + 16 * ks + 4 * half;
            const Row4 lo = load4<false>(sp), hi = load4<false>(sp + 8);
            const float t[8] = {lo.v[0], lo.v[1], lo.v[2], lo.v[3], hi.v[0], hi.v[1], hi.v[2], hi.v[3]};
            operand(ks, t);
        }
        __syncthreads();  // the slices are read out before the weights move in
    } else {
        // both passes' rows are requested before the first one is staged: one round trip to memory instead of two
        f32x4 xv[2][8];
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                xv[pass][j] = __builtin_nontemporal_load(
                    reinterpret_cast<const f32x4 *>(x + src_row[j] * x_stride + 64 * pass + io_col));
        }
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                *reinterpret_cast<f32x4 *>(stage + (4 * j + io_row) * kNlHalfPitch + io_col) = xv[pass][j];
            __syncthreads();
#pragma unroll
            for (int k4 = 0; k4 < 4; ++k4) {
                const float *sp = stage + m * kNlHalfPitch + 16 * k4 + 4 * half;
                const f32x4 lo = *reinterpret_cast<const f32x4 *>(sp);
                const f32x4 hi = *reinterpret_cast<const f32x4 *>(sp + 8);
                const float t[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
                operand(4 * pass + k4, t);
            }
            __syncthreads();
        }
    }
    ss += __shfl_xor(ss, 32);
    const float rstd = rsqrtf(ss * (1.0f / kNlD) + eps);

    if constexpr (KEEP) {
        // The update keeps the normalised rows for the weight gradient, rounded once from float32 (the operand is bf16 before its
        // factor and would be rounded a second time).  They leave as whole 256-byte rows through this wave's slice of the
        // staging area (32 rows x 136 halfs fit in the 32 x 68 floats of the slice).
        uint16_t *stage_n = reinterpret_cast<uint16_t *>(stage);
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            const f32x4 wl = *reinterpret_cast<const f32x4 *>(norm_w + 16 * ks + 4 * half);
            const f32x4 wh = *reinterpret_cast<const f32x4 *>(norm_w + 16 * ks + 8 + 4 * half);
            const float wv[8] = {wl.x, wl.y, wl.z, wl.w, wh.x, wh.y, wh.z, wh.w};
            float t[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                nb[ks][e] = (__bf16)(kept[ks][e] * wv[e]);
                t[e] = (kept[ks][e] * rstd) * wv[e];
            }
            uint16_t *sp = stage_n + m * kNlRowPitch + 16 * ks + 4 * half;
            *reinterpret_cast<u32x2 *>(sp) = u32x2{pack_bf16x2(t[0], t[1]), pack_bf16x2(t[2], t[3])};
            *reinterpret_cast<u32x2 *>(sp + 8) = u32x2{pack_bf16x2(t[4], t[5]), pack_bf16x2(t[6], t[7])};
            if (ks & 1) __builtin_amdgcn_sched_barrier(0);  // the norm's weights in four portions beside the kept row
        }
        fetch(c0);  // now that the row has left its registers
        wave_lds_handover();
        if (blockIdx.y == 0) {
            const int a_row = lane >> 4, a_col = (lane & 15) * 8;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int64_t r = row0 + 4 * j + a_row;
                const u32x4 v = *reinterpret_cast<const u32x4 *>(stage_n + (4 * j + a_row) * kNlRowPitch + a_col);
                if (r < rows) __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(n_out + r * kNlD + a_col));
            }
        }
        __syncthreads();  // the slices are read out before the weights move in
    }

    stash(0);
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();

    const int64_t row = row0 + m;
    for (int c = c0; c < c_end; ++c) {
        const int buf = (c - c0) & 1;
        if (c + 1 < c_end) fetch(c + 1);
        const uint16_t *wb = s_w + buf * kNlChunkHalfs + lane * 8;
        f32x16 z0 = {0.0f}, z1 = {0.0f};
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            const bf16x8 a0 = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(wb + ks * 512));
            const bf16x8 a1 = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(wb + 4096 + ks * 512));
            z0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, nb[ks], z0, 0, 0, 0);
            z1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, nb[ks], z1, 0, 0, 0);
        }
        if (row < rows) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const f32x16 &z = b ? z1 : z0;
                const int f0 = c * kNlChunkFeatures + 32 * b + 8 * half;  // first feature of this lane's first run
#pragma unroll
                for (int run = 0; run < 2; ++run) {
                    float r[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) r[e] = z[8 * run + e] * rstd;
                    if (!KEEP && bias != nullptr) {
                        const f32x4 bl = *reinterpret_cast<const f32x4 *>(bias + f0 + 16 * run);
                        const f32x4 bh = *reinterpret_cast<const f32x4 *>(bias + f0 + 16 * run + 4);
                        r[0] += bl.x; r[1] += bl.y; r[2] += bl.z; r[3] += bl.w;
                        r[4] += bh.x; r[5] += bh.y; r[6] += bh.z; r[7] += bh.w;
                    }
                    const u32x4 w = {pack_bf16x2(r[0], r[1]), pack_bf16x2(r[2], r[3]), pack_bf16x2(r[4], r[5]),
                                     pack_bf16x2(r[6], r[7])};
                    *reinterpret_cast<u32x4 *>(out + row * N + f0 + 16 * run) = w;
                }
            }
        }
        if (c + 1 < c_end) stash(buf ^ 1);
        __syncthreads();
    }
}

// ------------------------------------------------------------------------------------
// compact list of the rows whose mask byte is set (the bullets in flight)
// ------------------------------------------------------------------------------------

// Flags of four mask bytes j .. j+3 of a row as bits 0..3; `words`: the rows are whole aligned dwords.
__device__ __forceinline__ uint32_t mask_flags(const uint8_t *row, int j, int n, bool words)
{
    uint32_t f = 0;
    if (words) {
        if (j < n) {
            const uint32_t w = *reinterpret_cast<const uint32_t *>(row + j);
#pragma unroll
            for (int k = 0; k < 4; ++k) f |= (w >> (8 * k)) & 0xffu ? 1u << k : 0u;
        }
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) f |= j + k < n && row[j + k] != 0 ? 1u << k : 0u;
    }
    return f;
}

static bool mask_words(const uint8_t *mask, int n) { return n % 4 == 0 && (reinterpret_cast<uintptr_t>(mask) & 3u) == 0; }

// counts[b] = number of set bytes in mask row b (one wave per row).
__global__ __launch_bounds__(256) void mask_count_kernel(const uint8_t *__restrict__ mask, int32_t *__restrict__ counts,
                                                         int B, int n, bool words)
{
    const int b = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (b >= B) return;
    const uint8_t *row = mask + (int64_t)b * n;
    int c = 0;
    for (int j = (threadIdx.x & 63) * 4; j < n; j += 256) c += __popc(mask_flags(row, j, n, words));
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
    if ((threadIdx.x & 63) == 0) counts[b] = c;
}

// One wave lists the set entries of mask row b, ascending, from index[base] on.
__device__ __forceinline__ void mask_fill_row(const uint8_t *__restrict__ mask, int32_t *__restrict__ index, int b, int n, bool words,
                                              int base, int lane)
{
    const uint8_t *row = mask + (int64_t)b * n;
    const uint64_t below = (1ull << lane) - 1ull;
    for (int j0 = 0; j0 < n; j0 += 256) {
        const int j = j0 + 4 * lane;
        const uint32_t f = mask_flags(row, j, n, words);
        uint64_t set[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) set[k] = __ballot((f >> k) & 1u);
        int at = base;
#pragma unroll
        for (int k = 0; k < 4; ++k) at += (int)__popcll(set[k] & below);
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if ((f >> k) & 1u) index[at++] = b * n + j + k;
#pragma unroll
        for (int k = 0; k < 4; ++k) base += (int)__popcll(set[k]);
    }
}

// index[offsets[b] + k] = b*n + j for the k-th set byte j of mask row b (one wave per row).
__global__ __launch_bounds__(256) void mask_fill_kernel(const uint8_t *__restrict__ mask, const int32_t *__restrict__ offsets,
                                                        int32_t *__restrict__ index, int B, int n, bool words)
{
    const int b = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (b < B) mask_fill_row(mask, index, b, n, words, offsets[b], threadIdx.x & 63);
}

// The same with the offsets formed on the way: a work-group lists ROWS rows and sums the counts of all rows before them
// itself.  A launch reads B^2 / (2 ROWS) counts out of L2 for that, which is less time than a scan between the two kernels
// takes as launches of its own: the list of 16 x 80 slots cost 9.7 us as torch's fill, count, scan and fill, each behind the
// one before; 6.6 us now.  16 rows per group up to 8192 rows (4096 x 1520 slots: 8.9 us, with 64 rows 22 us: too few
// work-groups), 64 beyond, where the counts would be what it reads (537 MB at 65536 rows with 16, 134 MB with 64).
template <int ROWS>
__global__ __launch_bounds__(1024) void mask_list_kernel(const uint8_t *__restrict__ mask, const int32_t *__restrict__ counts,
                                                         int32_t *__restrict__ offsets, int32_t *__restrict__ index, int B, int n,
                                                         bool words)
{
    __shared__ int s_part[16];
    __shared__ int s_count[ROWS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int b0 = blockIdx.x * ROWS;
    int c = 0;
    for (int i = tid; i < b0; i += 1024) c += counts[i];
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
    if (lane == 0) s_part[wave] = c;
    if (tid < ROWS) s_count[tid] = b0 + tid < B ? counts[b0 + tid] : 0;
    __syncthreads();
    int base = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) base += s_part[w];
    for (int i = 0; i < ROWS / 16; ++i) {  // wave w lists rows w, w + 16, ...
        const int q = 16 * i + wave, b = b0 + q;
        int part = lane < q ? s_count[lane] : 0;
        for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off);
        const int before = base + part;
        if (b < B) {
            if (lane == 0) {
                offsets[b] = before;
                if (b == B - 1) offsets[B] = before + s_count[q];
            }
            mask_fill_row(mask, index, b, n, words, before, lane);
        }
    }
}

}  // namespace bnb

namespace bnb {

// Work-groups along the features: the chunks are halved (or thirded, ...) while the grid stays within what the chip holds at
// once, three work-groups per CU.  A listed launch is sized for every slot, of which a quarter is in flight as a rule.
static int nl_feature_groups(int64_t row_groups, int N, bool listed)
{
    const int chunks = N / kNlChunkFeatures;
    const int64_t room = (listed ? 4 : 1) * 3 * (int64_t)cu_count();
    for (int g = chunks; g > 1; --g)
        if (chunks % g == 0 && row_groups * g <= room) return g;
    return 1;
}

template <typename XT>
static int launch_norm_linear(const XT *x, int64_t x_row_stride, const int32_t *row_index, const int32_t *n_rows,
                              const float *norm_weight, float eps, const void *weight_packed, const float *bias, void *out,
                              int64_t R, int D, int N, void *stream)
{
    if (R < 0 || x_row_stride < D || N < 1) return BNB_ERR_BAD_SHAPE;
    if (D != kNlD || N % kNlChunkFeatures != 0) return BNB_ERR_UNSUPPORTED;
    if (R == 0) return 0;
    if (!x || !norm_weight || !weight_packed || !out) return BNB_ERR_NULL_POINTER;
    if (!aligned16(x) || !aligned16(out) || !aligned16(norm_weight) || !aligned16(weight_packed) ||
        (bias && !aligned16(bias)) || (x_row_stride * sizeof(XT)) % 16 != 0)
        return BNB_ERR_MISALIGNED;
    if ((reinterpret_cast<uintptr_t>(row_index) | reinterpret_cast<uintptr_t>(n_rows)) & 3u) return BNB_ERR_MISALIGNED;
    const int64_t blocks = (R + kNlWaves * 32 - 1) / (kNlWaves * 32);
    if (blocks > 0x7fffffffLL) return BNB_ERR_UNSUPPORTED;
    const int groups = nl_feature_groups(blocks, N, n_rows != nullptr);
    hipLaunchKernelGGL((norm_linear_kernel<XT, false>), dim3((unsigned)blocks, groups), dim3(kNlThreads), 0, (hipStream_t)stream,
                       x, x_row_stride, row_index, n_rows, norm_weight, eps, (const uint16_t *)weight_packed, bias,
                       (uint16_t *)out, R, N, N / kNlChunkFeatures / groups, (uint16_t *)nullptr);
    return (int)hipGetLastError();
}

}  // namespace bnb

extern "C" int bnb_norm_linear_fwd(const float *x, int64_t x_row_stride, const int32_t *row_index,
                                   const int32_t *n_rows, const float *norm_weight, float eps,
                                   const void *weight_packed, const float *bias, void *out, int64_t R, int D, int N,
                                   void *stream)
{
    return bnb::launch_norm_linear(x, x_row_stride, row_index, n_rows, norm_weight, eps, weight_packed, bias, out, R, D, N,
                                   stream);
}

extern "C" int bnb_norm_linear_bf16_fwd(const void *x, int64_t x_row_stride, const int32_t *row_index,
                                        const int32_t *n_rows, const float *norm_weight, float eps,
                                        const void *weight_packed, const float *bias, void *out, int64_t R, int D, int N,
                                        void *stream)
{
    return bnb::launch_norm_linear((const uint16_t *)x, x_row_stride, row_index, n_rows, norm_weight, eps, weight_packed,
                                   bias, out, R, D, N, stream);
}

extern "C" int bnb_norm_linear_train_fwd(const float *x, int64_t x_row_stride, const float *norm_weight, float eps,
                                         const void *weight_packed, void *out, void *n_out, int64_t R, int D, int N,
                                         void *stream)
{
    using namespace bnb;
    if (R < 0 || x_row_stride < D || N < 1) return BNB_ERR_BAD_SHAPE;
    if (D != kNlD || N % kNlChunkFeatures != 0) return BNB_ERR_UNSUPPORTED;
    if (R == 0) return 0;
    if (!x || !norm_weight || !weight_packed || !out || !n_out) return BNB_ERR_NULL_POINTER;
    if (!aligned16(x) || !aligned16(out) || !aligned16(n_out) || !aligned16(norm_weight) || !aligned16(weight_packed) ||
        (x_row_stride % 4) != 0)
        return BNB_ERR_MISALIGNED;
    const int64_t blocks = (R + kNlWaves * 32 - 1) / (kNlWaves * 32);
    if (blocks > 0x7fffffffLL) return BNB_ERR_UNSUPPORTED;
    const int groups = nl_feature_groups(blocks, N, false);
    hipLaunchKernelGGL((norm_linear_kernel<float, true>), dim3((unsigned)blocks, groups), dim3(kNlThreads), 0, (hipStream_t)stream, x,
                       x_row_stride, (const int32_t *)nullptr, (const int32_t *)nullptr, norm_weight, eps,
                       (const uint16_t *)weight_packed, (const float *)nullptr, (uint16_t *)out, R, N,
                       N / kNlChunkFeatures / groups, (uint16_t *)n_out);
    return (int)hipGetLastError();
}

extern "C" int bnb_mask_count(const uint8_t *mask, int32_t *counts, int B, int n, void *stream)
{
    using namespace bnb;
    if (B < 0 || n < 1) return BNB_ERR_BAD_SHAPE;
    if (B == 0) return 0;
    if (!mask || !counts) return BNB_ERR_NULL_POINTER;
    hipLaunchKernelGGL(mask_count_kernel, dim3((unsigned)((B + 3) / 4)), dim3(256), 0, (hipStream_t)stream, mask, counts, B, n, mask_words(mask, n));
    return (int)hipGetLastError();
}

extern "C" int bnb_mask_fill(const uint8_t *mask, const int32_t *offsets, int32_t *index, int B, int n, void *stream)
{
    using namespace bnb;
    if (B < 0 || n < 1 || (int64_t)B * n > 0x7fffffffLL) return BNB_ERR_BAD_SHAPE;
    if (B == 0) return 0;
    if (!mask || !offsets || !index) return BNB_ERR_NULL_POINTER;
    hipLaunchKernelGGL(mask_fill_kernel, dim3((unsigned)((B + 3) / 4)), dim3(256), 0, (hipStream_t)stream, mask, offsets, index, B, n, mask_words(mask, n));
    return (int)hipGetLastError();
}

extern "C" int bnb_mask_rows(const uint8_t *mask, int32_t *counts, int32_t *offsets, int32_t *index, int B, int n, void *stream)
{
    using namespace bnb;
    if (B < 1 || n < 1 || (int64_t)B * n > 0x7fffffffLL) return BNB_ERR_BAD_SHAPE;
    if (!mask || !counts || !offsets || !index) return BNB_ERR_NULL_POINTER;
    hipLaunchKernelGGL(mask_count_kernel, dim3((unsigned)((B + 3) / 4)), dim3(256), 0, (hipStream_t)stream, mask, counts, B, n,
                       mask_words(mask, n));
    if (B <= 8192)
        hipLaunchKernelGGL(mask_list_kernel<16>, dim3((unsigned)((B + 15) / 16)), dim3(1024), 0, (hipStream_t)stream, mask, counts,
                           offsets, index, B, n, mask_words(mask, n));
    else
        hipLaunchKernelGGL(mask_list_kernel<64>, dim3((unsigned)((B + 63) / 64)), dim3(1024), 0, (hipStream_t)stream, mask, counts,
                           offsets, index, B, n, mask_words(mask, n));
    return (int)hipGetLastError();
}
