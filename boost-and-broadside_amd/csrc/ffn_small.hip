// The sublayer tail of ffn_fused.hip for few rows: one work-group per 32 tokens, the hidden units split over its waves.
//
// The wide kernel gives a wave 32 tokens and all 512 hidden units, 16 dependent rounds of gate / up products, GELU and down
// projection: 25 us however few the tokens are, and with less than a work-group of 128 tokens per CU most of the chip is
// idle meanwhile.  Here the eight waves of a work-group hold the same 32 tokens and take 64 hidden units each.  No weight is
// used by two waves, so the operands go from L2 straight into registers (the packed stream already lists every operand as
// one contiguous kilobyte), requested before the rows they will meet have arrived; the eight partial results of the down
// projection meet in LDS and are added in wave order.  The projection's four channel blocks go to four waves, the next
// sublayer's head is split over the waves by feature blocks.
//
// What bounds it is latency (five barriers, three dependent round trips to L2 or memory) and, per CU, the 0.5 MB of weights
// at 64 bytes a clock.  With the next sublayer's head (384 features), replayed back to back, against the wide kernel:
//   192 rows 11.2 us (26.7), 4096 rows 12.1 us (27.5), 8192 rows 13.5 us (28.2), 16384 rows 24.4 us (30.2).
//
// Layouts (operand order, channel order of a lane, pack) are those of ffn_fused.hip; s, n and the head's normalised rows are
// the same bits, only the order in which the hidden units' contributions are added differs.

#include "ffn_small.h"
#include "ffn_math.h"

namespace bnb {

constexpr int kFsWaves = 8;
constexpr int kFsThreads = kFsWaves * kWave;
constexpr int kFsPitch = kFfnD + 4;                                // floats per staged fp32 row
constexpr int kFsOperandPitch = kFfnD + 8;                         // halfs per staged operand row
constexpr int kFsTile = 32 * kFsPitch;                             // floats of one wave's partial result
constexpr int kFsChunkHalfs = 3 * 32 * kFfnD;
static_assert(kFfnChunks == 2 * kFsWaves, "two chunks of 32 hidden units per wave");

template <bool GATE, bool HEAD, bool TRAIN>
__global__ __launch_bounds__(kFsThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void ffn_small_kernel(
    const float *__restrict__ x, int64_t x_stride, const uint16_t *__restrict__ rows_a, int64_t rows_a_stride,
    const uint16_t *__restrict__ rows_b, int64_t rows_b_stride, const uint16_t *__restrict__ wproj,
    const float *__restrict__ norm_w, float eps, const uint16_t *__restrict__ wpack, float *__restrict__ out, int64_t R,
    const float *__restrict__ next_norm_w, float next_eps, const uint16_t *__restrict__ next_wpack,
    uint16_t *__restrict__ next_out, int next_features, float *__restrict__ s_out, uint16_t *__restrict__ n_out)
{
    __shared__ __align__(16) float s_part[kFsWaves * kFsTile];  // the waves' partial results; the first tile holds s before
    __shared__ __align__(16) float s_norm[2][kFfnD];
    uint16_t *s_rows = reinterpret_cast<uint16_t *>(s_part + kFsTile);  // operand rows of the projection, before the partials

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 31;
    const int half = lane >> 5;
    const int64_t row0 = (int64_t)blockIdx.x * 32;

    // ---- the rows, then the first operands: everything is on its way before anything is waited for ----
    const int a_row = tid >> 4, a_col = (tid & 15) * 8;  // one 16-byte piece of an operand row per thread
    const int x_row = tid >> 5, x_col = (tid & 31) * 4;  // two pieces of the residual rows per thread, 16 rows apart
    const int64_t ra = row0 + a_row < R ? row0 + a_row : R - 1;
    u32x4 av = *reinterpret_cast<const u32x4 *>(rows_a + ra * rows_a_stride + a_col);
    u32x4 bv = {0u, 0u, 0u, 0u};
    if (GATE) bv = *reinterpret_cast<const u32x4 *>(rows_b + ra * rows_b_stride + a_col);
    f32x4 xv[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int64_t r = row0 + x_row + 16 * j < R ? row0 + x_row + 16 * j : R - 1;
        xv[j] = *reinterpret_cast<const f32x4 *>(x + r * x_stride + x_col);
    }
    bf16x8 wp[8];
    if (wave < 4) {
#pragma unroll
        for (int ks = 0; ks < 8; ++ks)
            wp[ks] = *reinterpret_cast<const bf16x8 *>(wproj + ((wave * 8 + ks) * 64 + lane) * 8);
    }
    const uint16_t *wc = wpack + (int64_t)(2 * wave) * kFsChunkHalfs + lane * 8;  // this wave's two chunks
    bf16x8 wg[8], wu[8];
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
        wg[ks] = *reinterpret_cast<const bf16x8 *>(wc + ks * 512);
        wu[ks] = *reinterpret_cast<const bf16x8 *>(wc + 4096 + ks * 512);
    }

    if (tid < kFfnD) s_norm[0][tid] = norm_w[tid];
    else if (HEAD && tid < 2 * kFfnD) s_norm[1][tid - kFfnD] = next_norm_w[tid - kFfnD];
    if (GATE) {
        const Row8 g = load8(reinterpret_cast<const uint16_t *>(&av)), y = load8(reinterpret_cast<const uint16_t *>(&bv));
        float p[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) p[e] = round_to_bf16(gelu_phi(g.v[e])) * y.v[e];
        av = u32x4{pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3]), pack_bf16x2(p[4], p[5]), pack_bf16x2(p[6], p[7])};
    }
    *reinterpret_cast<u32x4 *>(s_rows + a_row * kFsOperandPitch + a_col) = av;
#pragma unroll
    for (int j = 0; j < 2; ++j) *reinterpret_cast<f32x4 *>(s_part + (x_row + 16 * j) * kFsPitch + x_col) = xv[j];
    __syncthreads();

    // ---- s = x + rows Wp^T: waves 0..3 form one block of 32 channels each, in place ----
    if (wave < 4) {
        f32x16 z;
        float *sp = s_part + m * kFsPitch + 32 * wave + 4 * half;
#pragma unroll
        for (int v = 0; v < 16; v += 4) {
            const f32x4 t = *reinterpret_cast<const f32x4 *>(sp + 2 * v);
#pragma unroll
            for (int e = 0; e < 4; ++e) z[v + e] = t[e];
        }
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            const uint16_t *op = s_rows + m * kFsOperandPitch + 16 * ks + 4 * half;
            const u32x2 lo = *reinterpret_cast<const u32x2 *>(op), hi = *reinterpret_cast<const u32x2 *>(op + 8);
            z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wp[ks], __builtin_bit_cast(bf16x8, u32x4{lo.x, lo.y, hi.x, hi.y}), z, 0, 0, 0);
        }
#pragma unroll
        for (int v = 0; v < 16; v += 4) *reinterpret_cast<f32x4 *>(sp + 2 * v) = f32x4{z[v], z[v + 1], z[v + 2], z[v + 3]};
    }
    __syncthreads();

    // ---- every wave: its token's s in the accumulator layout, n = rmsnorm(s) as B operand ----
    f32x16 acc[4];
    bf16x8 nb[8];
    auto rows_in = [&]() {
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            const float *sp = s_part + m * kFsPitch + 16 * ks + 4 * half;
            const f32x4 lo = *reinterpret_cast<const f32x4 *>(sp), hi = *reinterpret_cast<const f32x4 *>(sp + 8);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[ks >> 1][8 * (ks & 1) + e] = lo[e], acc[ks >> 1][8 * (ks & 1) + 4 + e] = hi[e];
        }
    };
    auto normalise = [&](const float *w, float ep) {
        float ss = 0.0f;
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
#pragma unroll
            for (int v = 0; v < 16; ++v) ss = fmaf(acc[cb][v], acc[cb][v], ss);
        }
        ss += __shfl_xor(ss, 32);
        const float rstd = rsqrtf(ss * (1.0f / kFfnD) + ep);
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            const f32x4 wl = *reinterpret_cast<const f32x4 *>(w + 16 * ks + 4 * half);
            const f32x4 wh = *reinterpret_cast<const f32x4 *>(w + 16 * ks + 8 + 4 * half);
            const float wv[8] = {wl.x, wl.y, wl.z, wl.w, wh.x, wh.y, wh.z, wh.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) nb[ks][e] = (__bf16)((acc[ks >> 1][8 * (ks & 1) + e] * rstd) * wv[e]);
            asm volatile("" : "+v"(nb[ks]));  // formed here: left to the first product, s would stay in registers beside the sums
        }
    };
    rows_in();
    normalise(s_norm[0], eps);
    if constexpr (TRAIN) {
        // what the update keeps: s as it stands in LDS, and n, whose step ks comes from wave ks, as whole rows
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            if (ks != wave) continue;
            const u32x4 v = __builtin_bit_cast(u32x4, nb[ks]);
            uint16_t *op = s_rows + m * kFsOperandPitch + 16 * ks + 4 * half;
            *reinterpret_cast<u32x2 *>(op) = u32x2{v.x, v.y};
            *reinterpret_cast<u32x2 *>(op + 8) = u32x2{v.z, v.w};
        }
        __syncthreads();
        if (row0 + a_row < R)
            *reinterpret_cast<u32x4 *>(n_out + (row0 + a_row) * kFfnD + a_col) =
                *reinterpret_cast<const u32x4 *>(s_rows + a_row * kFsOperandPitch + a_col);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (row0 + x_row + 16 * j < R)
                *reinterpret_cast<f32x4 *>(s_out + (row0 + x_row + 16 * j) * kFfnD + x_col) =
                    *reinterpret_cast<const f32x4 *>(s_part + (x_row + 16 * j) * kFsPitch + x_col);
        }
    }
    __syncthreads();  // also keeps the operand loads that follow behind the norm, whose registers they take over
    bf16x8 wd[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) wd[q] = *reinterpret_cast<const bf16x8 *>(wc + 8192 + q * 512);
    if (wave != 0) {  // s enters the sum once
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[cb][v] = 0.0f;
        }
    }

    // ---- two chunks of 32 hidden units; the second one's operands arrive under the first one's arithmetic ----
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        f32x16 g = {0.0f}, u = {0.0f};
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            g = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wg[ks], nb[ks], g, 0, 0, 0);
            u = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wu[ks], nb[ks], u, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (c == 0) {
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) wg[ks] = *reinterpret_cast<const bf16x8 *>(wc + kFsChunkHalfs + ks * 512);
        }
        bf16x8 hb[2];
#pragma unroll
        for (int v = 0; v < 16; ++v) hb[v >> 3][v & 7] = (__bf16)(gelu_phi(g[v]) * u[v]);
        __builtin_amdgcn_sched_barrier(0);
        if (c == 0) {
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) wu[ks] = *reinterpret_cast<const bf16x8 *>(wc + kFsChunkHalfs + 4096 + ks * 512);
        }
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wd[cb * 2 + t], hb[t], acc[cb], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (c == 0) {
#pragma unroll
            for (int q = 0; q < 8; ++q) wd[q] = *reinterpret_cast<const bf16x8 *>(wc + kFsChunkHalfs + 8192 + q * 512);
        }
    }

    // ---- the partial results meet (everyone has s out of the first tile); out leaves as whole rows ----
    float *mine = s_part + wave * kFsTile;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
        const f32x16 &a = acc[ks >> 1];
        const int v0 = 8 * (ks & 1);
        float *sp = mine + m * kFsPitch + 16 * ks + 4 * half;
        *reinterpret_cast<f32x4 *>(sp) = f32x4{a[v0], a[v0 + 1], a[v0 + 2], a[v0 + 3]};
        *reinterpret_cast<f32x4 *>(sp + 8) = f32x4{a[v0 + 4], a[v0 + 5], a[v0 + 6], a[v0 + 7]};
    }
    const int blocks = HEAD ? next_features >> 5 : 0;  // the head's blocks of 32 features go round the waves
    if (HEAD && wave < blocks) {
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) wg[ks] = *reinterpret_cast<const bf16x8 *>(next_wpack + ((int64_t)(wave * 8 + ks) * 64 + lane) * 8);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        float *sp = s_part + (x_row + 16 * j) * kFsPitch + x_col;
        f32x4 t = *reinterpret_cast<const f32x4 *>(sp);
#pragma unroll
        for (int w = 1; w < kFsWaves; ++w) t += *reinterpret_cast<const f32x4 *>(sp + w * kFsTile);
        if (row0 + x_row + 16 * j < R) *reinterpret_cast<f32x4 *>(out + (row0 + x_row + 16 * j) * kFfnD + x_col) = t;
        if (HEAD) *reinterpret_cast<f32x4 *>(sp) = t;  // only this thread reads these four sums
    }
    if constexpr (HEAD) {
        __syncthreads();
        if (wave >= blocks) return;  // no barrier follows
        rows_in();
        normalise(s_norm[1], next_eps);
        const int64_t out_row = row0 + (m & 15);
        for (int b = wave; b < blocks; b += kFsWaves) {
            f32x16 z = {0.0f};
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wg[ks], nb[ks], z, 0, 0, 0);
            if (b + kFsWaves < blocks) {
#pragma unroll
                for (int ks = 0; ks < 8; ++ks)
                    wg[ks] = *reinterpret_cast<const bf16x8 *>(next_wpack + ((int64_t)((b + kFsWaves) * 8 + ks) * 64 + lane) * 8);
            }
            u32x4 w[2];
#pragma unroll
            for (int t = 0; t < 2; ++t)
                w[t] = u32x4{pack_bf16x2(z[8 * t], z[8 * t + 1]), pack_bf16x2(z[8 * t + 2], z[8 * t + 3]),
                             pack_bf16x2(z[8 * t + 4], z[8 * t + 5]), pack_bf16x2(z[8 * t + 6], z[8 * t + 7])};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const u32x2 t = __builtin_amdgcn_permlane16_swap(w[0][q], w[1][q], false, false);
                w[0][q] = t.x, w[1][q] = t.y;
            }
            uint16_t *p = next_out + out_row * next_features + 32 * b + 16 * (m >> 4) + 8 * half;
            *reinterpret_cast<u32x4 *>(p) = w[0];
            *reinterpret_cast<u32x4 *>(p + 16 * (int64_t)next_features) = w[1];
        }
    }
}

// A work-group takes a CU's LDS, so 32 rows for each of 256 CUs are one round (13.5 us against the wide kernel's 28.2 us
// at 8192 rows) and two rounds still win (24.4 us against 30.2 us at 16384 rows); a third would not (the wide kernel takes
// 31.5 us at 24576 rows).
int64_t ffn_small_rows_limit() { return (int64_t)64 * cu_count(); }

int launch_ffn_small(const FfnSmallArgs &a, hipStream_t s)
{
    const dim3 grid((unsigned)((a.R + 31) / 32)), block(kFsThreads);
#define BNB_FFN_SMALL(GATE, HEAD, TRAIN)                                                                                     \
    hipLaunchKernelGGL((ffn_small_kernel<GATE, HEAD, TRAIN>), grid, block, 0, s, a.x, a.x_stride, a.rows_a, a.rows_a_stride, \
                       a.rows_b, a.rows_b_stride, a.wproj, a.norm_w, a.eps, a.wpack, a.out, a.R, a.next_norm_w, a.next_eps,  \
                       a.next_wpack, a.next_out, a.next_features, a.s_out, a.n_out)
    if (a.s_out) BNB_FFN_SMALL(false, false, true);
    else if (a.rows_b && a.next_out) BNB_FFN_SMALL(true, true, false);
    else if (a.rows_b) BNB_FFN_SMALL(true, false, false);
    else if (a.next_out) BNB_FFN_SMALL(false, true, false);
    else BNB_FFN_SMALL(false, false, false);
#undef BNB_FFN_SMALL
    return (int)hipGetLastError();
}

}  // namespace bnb
