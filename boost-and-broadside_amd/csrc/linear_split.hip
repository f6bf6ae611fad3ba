// Float32 Linear layers of the trunk with their neighbours folded in, on the bf16 matrix cores (gfx950):
//
//     out[r, :] = ( A[r, :] W^T + bias ) (+ resid[r, :])        A = x                     plain
//                                                                  | rmsnorm(x) * norm_w     NORM
//                                                                  | gelu(x) * x2            MULGELU
//     GATE: W = [gate rows ; up rows] interleaved by blocks of 32, out[r, u] = gelu(g[r, u]) * up[r, u]
//
// (models/yemong/attention.py:21-37,60-74; models/yemong/griffin.py:165-167,238-247 run without autocast,
// evaluation/agents.py:214-219), but a float32 operand enters as three bf16 pieces, v = h + m / 128 + l / 128^2, each
// the rounded rest of the ones before.  The rests are carried larger because bf16 ends where float32 does: unscaled, the
// last piece of a value below 8e-34 would have no exponent left.  So a value is carried exactly from 4.7e-38 on, and
// within 3e-7 down to the smallest normal one.  Of the nine piece products the three of at most 2^-25 of the whole, half a
// float32 rounding each (m l, l m, l l), are left out; the other six run on v_mfma_f32_32x32x16_bf16, which does in 32
// cycles what v_mfma_f32_32x32x2_f32 needs 512 for: 192 cycles per 32 x 32 x 16 block instead of 512.  The products of
// each size have an accumulator of their own, so the sum of K products is rounded K/16 times at full size and not K/2
// times: the relative 2-norm error of a launch against float64 is 0.5e-7 .. 1.8e-7 (fp32 matrix cores 1.2e-7 .. 3.4e-7),
// at 1e-36 times the usual size as well (unscaled pieces: 4e-5 with tiny rows, 6e-4 with tiny weights).
// What the pieces cannot carry (infinities, a row value above 3.39e38, products beyond the range) shows as a result that is
// not finite, and such a result is formed once more from whole values in float32.
//
// Time, fp32 matrix cores -> here: 12288 rows norm + 384 features 33 -> 17 us, norm + 2 x 512 + gate 53 -> 30 us,
// 512 -> 128 32 -> 26 us; 65760 rows 108 -> 59, 219 -> 120, 118 -> 84 us (with unscaled pieces on the same boxes 52, 113 and
// 78 us: two more multiplications per value of a row and two more per result).  Matrix cores busy 33 to 50 % of the
// large launches' time; the rest is the split of the rows, the gate and the row loads (64-byte pieces a row apart).
//
// A wave owns 32 rows, four waves share a stream of 32-feature x 128-channel weight chunks (24 KB with the
// three pieces) that goes L2 -> LDS directly through three buffers, one barrier per chunk.  A row's three pieces
// of one 128-channel slab stay in registers across all feature blocks of the work-group.  Channel order of a
// product as everywhere: k-slot e of step ks in a lane of half h is channel 16 ks + 8 (e/4) + 4 h + e%4.

#include "split_math.h"

namespace bnb {

constexpr int kLsWaves = 4;
// Rows per CU up to which a contraction of 512 or more is split over waves.  The one such layer of the trunk is 512 -> 128, us of this
// form and of the other on 256 CUs: 2000 rows 9 / 21, 8192 17 / 23, 12288 26 / 25, 27680 50 / 35; other N were not measured.
constexpr int kLsFewRowsPerCu = 40;

struct LinearSplitArgs {
    const float *x;
    int64_t x_stride;
    const float *x2;  // gelu(x) * x2 when given
    int64_t x2_stride;
    const float *norm_w;  // rmsnorm(x) * norm_w when given (K == 128)
    float eps;
    const uint16_t *w;  // [fb][K/128][ks][piece][lane][8], fb < n_blocks
    const float *bias, *resid;
    int64_t resid_stride;
    float *out;
    int64_t out_stride, R;
    int K, n_blocks;
};

enum { kLsPlain = 0, kLsNorm = 1, kLsMulGelu = 2 };

// this lane's 64 channels (of half `half`) of slab t of a row
__device__ __forceinline__ void load_rows(const LinearSplitArgs &p, int64_t row, int t, int half, float (&a)[8][8])
{
    const float *xp = p.x + row * p.x_stride + t * 128 + 4 * half;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
        const f32x4 lo = *reinterpret_cast<const f32x4 *>(xp + 16 * ks), hi = *reinterpret_cast<const f32x4 *>(xp + 16 * ks + 8);
#pragma unroll
        for (int e = 0; e < 4; ++e) a[ks][e] = lo[e], a[ks][4 + e] = hi[e];
    }
}

// ... through the prologue and into pieces
template <int PRO>
__device__ __forceinline__ void form_operand(const LinearSplitArgs &p, int64_t row, int t, int half, float (&a)[8][8],
                                         bf16x8 (&ah)[8], bf16x8 (&am)[8], bf16x8 (&al)[8], float &rstd)
{
    const float *nw = nullptr;
    if (PRO == kLsNorm) {
        float ss = 0.0f;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
#pragma unroll
            for (int e = 0; e < 8; ++e) ss = fmaf(a[ks][e], a[ks][e], ss);
        }
        ss += __shfl_xor(ss, 32);
        rstd = rsqrtf(ss * (1.0f / 128) + p.eps);
        nw = p.norm_w + 4 * half;
        __builtin_amdgcn_sched_barrier(0);  // the norm's weights come in after the rows: both at once do not fit the registers
    }
    if (PRO == kLsMulGelu) {
        const float *yp = p.x2 + row * p.x2_stride + t * 128 + 4 * half;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            const f32x4 lo = *reinterpret_cast<const f32x4 *>(yp + 16 * ks), hi = *reinterpret_cast<const f32x4 *>(yp + 16 * ks + 8);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                a[ks][e] = gelu_erf_ls(a[ks][e]) * lo[e], a[ks][4 + e] = gelu_erf_ls(a[ks][4 + e]) * hi[e];
        }
    }
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
        if (PRO == kLsNorm) {
            const f32x4 lo = *reinterpret_cast<const f32x4 *>(nw + 16 * ks), hi = *reinterpret_cast<const f32x4 *>(nw + 16 * ks + 8);
#pragma unroll
            for (int e = 0; e < 4; ++e) a[ks][e] = a[ks][e] * rstd * lo[e], a[ks][4 + e] = a[ks][4 + e] * rstd * hi[e];
        }
        split8(a[ks], ah[ks], am[ks], al[ks]);
        if (PRO == kLsNorm && (ks & 3) == 3) __builtin_amdgcn_sched_barrier(0);
    }
}

// Operand value k of row r in float32
template <int PRO>
__device__ __forceinline__ float operand_f32(const LinearSplitArgs &p, int64_t r, int k, float rstd)
{
    float av = p.x[r * p.x_stride + k];
    if (PRO == kLsNorm) av = av * rstd * p.norm_w[k];
    if (PRO == kLsMulGelu) av = gelu_erf_ls(av) * p.x2[r * p.x2_stride + k];
    return av;
}

// One element in float32, from whole values: row r, feature m of block `block`
template <int PRO>
__device__ __forceinline__ float dot_f32(const LinearSplitArgs &p, int64_t r, int block, int m, float rstd)
{
    float sum = 0.0f;
#pragma unroll 1
    for (int k = 0; k < p.K; ++k) {
        sum = fmaf(operand_f32<PRO>(p, r, k, rstd), whole_weight(p.w, p.K >> 7, block, m, k), sum);
    }
    return sum;
}

// A result that is not finite is formed once more in float32, from whole values: an infinite or nearly infinite operand, or a
// product beyond the range, meets the other pieces as inf - inf or inf * 0, where float32 products have a value.  Only a row
// that holds a NaN is left alone.  Called by whole half-waves (row r, lane m: its 32 channels in turn).
template <int PRO>
__device__ __forceinline__ bool row_has_nan(const LinearSplitArgs &p, int64_t r, int m, float rstd)
{
    bool nan = false;
#pragma unroll 1
    for (int k = m; k < p.K; k += 32) {
        const float av = operand_f32<PRO>(p, r, k, rstd);
        nan = nan || av != av;
    }
    return (uint32_t)(__ballot(nan) >> (threadIdx.x & 32)) != 0;
}

// one contraction step: the six piece products
__device__ __forceinline__ void products(bf16x8 ah, bf16x8 am, bf16x8 al, const u32x4 (&w)[3], Sums &s)
{
    const bf16x8 wh = __builtin_bit_cast(bf16x8, w[0]), wm = __builtin_bit_cast(bf16x8, w[1]), wl = __builtin_bit_cast(bf16x8, w[2]);
    s.small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, wh, s.small, 0, 0, 0);
    s.mid = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am, wh, s.mid, 0, 0, 0);
    s.big = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, wh, s.big, 0, 0, 0);
    s.small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am, wm, s.small, 0, 0, 0);
    s.mid = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, wm, s.mid, 0, 0, 0);
    s.small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, wl, s.small, 0, 0, 0);
}

template <int N>
__device__ __forceinline__ void wait_vmcnt()
{
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
}

// NB weight blocks of 32 features are accumulated side by side (GATE: the gate and the up block)
// LONG: a contraction of more than 128 channels
template <int PRO, bool GATE, int NB, bool LONG>
__global__ __launch_bounds__(kLsWaves * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void linear_split_kernel(LinearSplitArgs p, int tiles, int splits,
                                                                                                     int groups_per_wg)
{
    __shared__ __align__(16) uint16_t s_w[3][kLsChunkHalfs];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 31, half = lane >> 5;
    // the work-groups that share a row tile (each a run of feature blocks) go to one XCD: its L2 reads the rows once
    const int sp = (int)(blockIdx.x / 8) % splits;
    const int tile = (int)(blockIdx.x / 8) / splits * 8 + (int)(blockIdx.x % 8);
    const int groups = p.n_blocks / NB;
    const int g0 = sp * groups_per_wg;
    const int g1 = g0 + groups_per_wg < groups ? g0 + groups_per_wg : groups;
    if (tile >= tiles || g0 >= g1) return;
    const int slabs = LONG ? p.K >> 7 : 1;
    const int64_t row0 = (int64_t)tile * (32 * kLsWaves) + wave * 32;
    const int64_t row = row0 + m < p.R ? row0 + m : p.R - 1;  // rows past the end repeat the last one and are not stored

    const uint32_t lds_w = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t *)&s_w[0][0];
    constexpr int OUT_BLOCKS = GATE ? 1 : NB, kStores = 16 * OUT_BLOCKS;
    // every row of this wave exists: exactly kStores stores a group, at 32-bit offsets
    const bool full = row0 + 32 <= p.R && p.out_stride < (1 << 24) && p.resid_stride < (1 << 24);
    bool counted = full;  // the last group's results left as kStores stores
    constexpr int kDma = kLsChunkHalfs / 512 / kLsWaves;  // 1 KB pieces per wave and chunk: 6
    // the chunk that is requested next: block b of group g, slab t
    int rg = g0, rt = 0, rb = 0, rbuf = 0;
    auto request = [&]() -> bool {
        if (rg >= g1) return false;
        const uint16_t *src = p.w + ((int64_t)(rg * NB + rb) * slabs + rt) * kLsChunkHalfs + wave * (kDma * 512);
        const uint32_t dst = lds_w + (uint32_t)(rbuf * kLsChunkHalfs * 2 + wave * (kDma * 1024));
#pragma unroll
        for (int q = 0; q < kDma; ++q)
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %0"
                         :
                         : "s"(src + q * 512), "v"((uint32_t)(lane * 16)), "s"(dst + (uint32_t)(q * 1024))
                         : "memory", "m0");
        rbuf = rbuf == 2 ? 0 : rbuf + 1;
        if (++rb == NB) {
            rb = 0;
            if (++rt == slabs) rt = 0, ++rg;
        }
        return true;
    };
    request();
    request();

    bf16x8 ah[8], am[8], al[8];
    float rstd = 0.0f;
    auto load_slab = [&](int t) {
        float a[8][8];
        load_rows(p, row, t, half, a);
        form_operand<PRO>(p, row, t, half, a, ah, am, al, rstd);
    };
    load_slab(0);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's parts of the first two chunks are in LDS
    __syncthreads();

    int buf = 0;
    for (int g = g0; g < g1; ++g) {
        f32x16 big[NB];
        for (int t = 0; t < slabs; ++t) {
            if (LONG && (t > 0 || g > g0)) load_slab(t);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const bool more = request();  // two chunks ahead, into the buffer of the chunk before this one
                Sums sums;  // of this chunk alone: its three accumulators give way to one
                sums.clear();
                const uint16_t *wb = s_w[buf] + lane * 8;
                u32x4 w[2][3];
#pragma unroll
                for (int q = 0; q < 3; ++q) w[0][q] = *reinterpret_cast<const u32x4 *>(wb + q * 512);
#pragma unroll
                for (int ks = 0; ks < 8; ++ks) {
                    if (ks < 7) {
#pragma unroll
                        for (int q = 0; q < 3; ++q) w[(ks + 1) & 1][q] = *reinterpret_cast<const u32x4 *>(wb + ((ks + 1) * 3 + q) * 512);
                    }
                    __builtin_amdgcn_sched_barrier(0);  // the next step's operands are requested before this step's products
                    products(ah[ks], am[ks], al[ks], w[ks & 1], sums);
                }
#pragma unroll
                for (int v = 0; v < 16; ++v) big[b][v] = LONG && t > 0 ? big[b][v] + sums.total(v) : sums.total(v);
                buf = buf == 2 ? 0 : buf + 1;
                // This wave's part of the next chunk has landed once nothing older than the request above and, behind a
                // group's end, than its kStores result stores (issued between the two requests) is outstanding: the
                // counter runs in issue order.  A result store has a whole chunk's time to be acknowledged this way.
                if (!counted) {
                    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): such a wave leaves stores out
                } else if (t == 0 && b == 0 && g > g0) {
                    if (more) wait_vmcnt<kStores + kDma>();
                    else wait_vmcnt<kStores>();
                } else if (more) {
                    wait_vmcnt<kDma>();
                } else {
                    wait_vmcnt<0>();
                }
                __syncthreads();
            }
        }
        // ---- epilogue: the lane holds feature m of each block, rows 8 i + 4 half + j ----
        float zero = 0.0f;  // a NaN once some result is not finite
#pragma unroll
        for (int b = 0; b < NB; ++b) {
#pragma unroll
            for (int v = 0; v < 16; ++v) zero = fmaf(big[b][v], 0.0f, zero);
        }
        const bool any_off = __any(zero != zero);
        uint32_t off[OUT_BLOCKS] = {};  // bit v: result v is not finite
        if (any_off) {
#pragma unroll
            for (int b = 0; b < OUT_BLOCKS; ++b) {
#pragma unroll
                for (int v = 0; v < 16; ++v) off[b] |= not_finite(big[b][v]) || (GATE && not_finite(big[NB - 1][v])) ? 1u << v : 0u;
            }
        }
        counted = full && !any_off;
#pragma unroll
        for (int b = 0; b < OUT_BLOCKS; ++b) {
            const int feat = (g * OUT_BLOCKS + b) * 32 + m;
            const float bv = p.bias != nullptr ? p.bias[feat] : 0.0f;
            if (counted) {
                // 32-bit lane offsets, formed here and not kept across the chunk loop (the empty asm hides that they do not change)
                uint32_t o_off = 4u * half * (uint32_t)p.out_stride + m, r_off = 4u * half * (uint32_t)p.resid_stride + m;
                asm volatile("" : "+v"(o_off), "+v"(r_off));
                const float *rp = p.resid + row0 * p.resid_stride + (g * OUT_BLOCKS + b) * 32;
                float *op = p.out + row0 * p.out_stride + (g * OUT_BLOCKS + b) * 32;
                auto leave = [&](int v, float more) {
                    float o = big[b][v] + bv;
                    if (GATE) o = gelu_erf_ls(o) * big[NB - 1][v];
                    op[o_off] = o + more;
                    o_off += (v & 3) == 3 ? 5u * (uint32_t)p.out_stride : (uint32_t)p.out_stride;
                };
                if (p.resid != nullptr) {
                    // all sixteen requests first: one round trip instead of sixteen
                    float res[16];
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        res[v] = rp[r_off];
                        r_off += (v & 3) == 3 ? 5u * (uint32_t)p.resid_stride : (uint32_t)p.resid_stride;
                    }
#pragma unroll
                    for (int v = 0; v < 16; ++v) leave(v, res[v]);
                } else {
#pragma unroll
                    for (int v = 0; v < 16; ++v) leave(v, 0.0f);
                }
            } else {
                int rr0 = 4 * half;
                asm volatile("" : "+v"(rr0));  // sixteen row addresses are not kept across the chunk loop for this path either
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int64_t r = row0 + 8 * (v >> 2) + rr0 + (v & 3);
                    float o = big[b][v] + bv;
                    if (GATE) o = gelu_erf_ls(o) * big[NB - 1][v];
                    if (p.resid != nullptr && r < p.R) o += p.resid[r * p.resid_stride + feat];
                    if (r < p.R && !(off[b] >> v & 1u)) p.out[r * p.out_stride + feat] = o;
                }
            }
        }
        if (any_off) {
#pragma unroll
            for (int b = 0; b < OUT_BLOCKS; ++b) {
                const int feat = (g * OUT_BLOCKS + b) * 32 + m;
                const float bv = p.bias != nullptr ? p.bias[feat] : 0.0f;
#pragma unroll 1
                for (int v = 0; v < 16; ++v) {
                    if (!__any(off[b] >> v & 1u)) continue;
                    const int rr = 8 * (v >> 2) + 4 * half + (v & 3);
                    const int64_t r = row0 + rr < p.R ? row0 + rr : p.R - 1;
                    const float rs = __shfl(rstd, rr);
                    const bool nan = row_has_nan<PRO>(p, r, m, rs);
                    if (!(off[b] >> v & 1u) || row0 + rr >= p.R) continue;
                    float o = __builtin_nanf("");
                    if (!nan) {
                        o = dot_f32<PRO>(p, r, g * NB + b, m, rs) + bv;
                        if (GATE) o = gelu_erf_ls(o) * dot_f32<PRO>(p, r, g * NB + NB - 1, m, rs);
                    }
                    if (p.resid != nullptr) o += p.resid[r * p.resid_stride + feat];
                    p.out[r * p.out_stride + feat] = o;
                }
            }
            __builtin_amdgcn_s_waitcnt(0x0f70);  // nothing of this path is left for the chunk loop to wait for
        }
    }
}

// Few rows and a long contraction: the four waves of a work-group take one 128-channel slab each of the SAME 32 rows
// and add up in LDS, so that the slabs' row loads and splits, a serial chain of latencies in the kernel above,
// run side by side.  Nothing of the weights is shared then, they go from L2 straight into registers.
template <int PRO, int NB>
__global__ __launch_bounds__(kLsWaves * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void linear_split_k_kernel(LinearSplitArgs p, int groups)
{
    __shared__ __align__(16) float s_part[kLsWaves][NB * 16][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = lane & 31, half = lane >> 5;
    const int g = (int)(blockIdx.x % groups);
    const int64_t row0 = (int64_t)(blockIdx.x / groups) * 32;
    const int64_t row = row0 + m < p.R ? row0 + m : p.R - 1;
    const int slabs = p.K >> 7;
    f32x16 big[NB];
    float rstd = 0.0f;
    for (int t = wave; t < slabs; t += kLsWaves) {
        float a[8][8];
        load_rows(p, row, t, half, a);
        bf16x8 ah[8], am[8], al[8];
        form_operand<PRO>(p, row, t, half, a, ah, am, al, rstd);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const uint16_t *wb = p.w + ((int64_t)(g * NB + b) * slabs + t) * kLsChunkHalfs + lane * 8;
            Sums sums;
            sums.clear();
            u32x4 w[4][3];  // three steps ahead
#pragma unroll
            for (int ks = 0; ks < 3; ++ks) {
#pragma unroll
                for (int q = 0; q < 3; ++q) w[ks][q] = *reinterpret_cast<const u32x4 *>(wb + (ks * 3 + q) * 512);
            }
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) {
                if (ks < 5) {
#pragma unroll
                    for (int q = 0; q < 3; ++q) w[(ks + 3) & 3][q] = *reinterpret_cast<const u32x4 *>(wb + ((ks + 3) * 3 + q) * 512);
                }
                __builtin_amdgcn_sched_barrier(0);
                products(ah[ks], am[ks], al[ks], w[ks & 3], sums);
            }
#pragma unroll
            for (int v = 0; v < 16; ++v) big[b][v] = t >= kLsWaves ? big[b][v] + sums.total(v) : sums.total(v);
        }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
        for (int v = 0; v < 16; ++v) s_part[wave][b * 16 + v][lane] = big[b][v];
    }
    __syncthreads();
    // each wave adds up and writes four of a lane's sixteen rows: 8 wave + 4 half + 0..3
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int feat = (g * NB + b) * 32 + m;
        const float bv = p.bias != nullptr ? p.bias[feat] : 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t r = row0 + 8 * wave + 4 * half + j;
            float o = 0.0f;
#pragma unroll
            for (int q = 0; q < kLsWaves; ++q) o += s_part[q][b * 16 + 4 * wave + j][lane];
            if (__any(not_finite(o)) && !row_has_nan<PRO>(p, r < p.R ? r : p.R - 1, m, 0.0f) && not_finite(o))
                o = dot_f32<PRO>(p, r < p.R ? r : p.R - 1, g * NB + b, m, 0.0f);
            if (r >= p.R) continue;
            o += bv;
            if (p.resid != nullptr) o += p.resid[r * p.resid_stride + feat];
            p.out[r * p.out_stride + feat] = o;
        }
    }
}

template <int PRO, bool GATE, int NB, bool LONG>
static int launch_nb(const LinearSplitArgs &p, hipStream_t stream)
{
    const int64_t tiles = (p.R + 32 * kLsWaves - 1) / (32 * kLsWaves);
    const int groups = p.n_blocks / NB, slabs = p.K / 128, cus = cu_count();
    // Feature blocks per work-group: the split whose slowest CU has the least to do.  A work-group's time in chunks:
    // its products, and the load + split of its rows (about 1.5 chunks a slab); two work-groups share a CU, and an odd
    // one left over runs at 0.65 of a pair's time.
    int best = groups;
    double best_t = 0.0;
    for (int per = groups; per >= 1; --per) {
        const int splits = (groups + per - 1) / per;
        const int64_t n = (tiles * splits + cus - 1) / cus;
        const double unit = slabs == 1 ? 1.5 + per * NB : per * slabs * (1.5 + NB);
        const double t = unit * ((double)(n / 2) + (n & 1 ? 0.65 : 0.0));
        if (per == groups || t < best_t) best = per, best_t = t;
    }
    const int splits = (groups + best - 1) / best;
    const int64_t grid = (tiles + 7) / 8 * 8 * splits;
    if (grid > 0x7fffffffLL) return BNB_ERR_UNSUPPORTED;
    hipLaunchKernelGGL((linear_split_kernel<PRO, GATE, NB, LONG>), dim3((unsigned)grid), dim3(kLsWaves * 64), 0, stream, p, (int)tiles, splits, best);
    return (int)hipGetLastError();
}

template <int PRO, bool GATE>
static int launch_pro(const LinearSplitArgs &p, hipStream_t stream)
{
    constexpr int NB = GATE ? 2 : 1;
    if constexpr (PRO != kLsNorm) {
        if (p.K > 128) {
            if constexpr (!GATE) {
                if (p.K >= 512 && p.R <= (int64_t)kLsFewRowsPerCu * cu_count()) {
                    const int64_t tiles = (p.R + 31) / 32;
                    if (p.n_blocks % 2 == 0)
                        hipLaunchKernelGGL((linear_split_k_kernel<PRO, 2>), dim3((unsigned)(tiles * (p.n_blocks / 2))), dim3(256), 0, stream, p, p.n_blocks / 2);
                    else
                        hipLaunchKernelGGL((linear_split_k_kernel<PRO, 1>), dim3((unsigned)(tiles * p.n_blocks)), dim3(256), 0, stream, p, p.n_blocks);
                    return (int)hipGetLastError();
                }
            }
            // a longer contraction re-reads its rows for every group of blocks: two blocks at a time where they pair up
            if (GATE || p.n_blocks % 2 == 0) return launch_nb<PRO, GATE, 2, true>(p, stream);
            return launch_nb<PRO, GATE, NB, true>(p, stream);
        }
    }
    return launch_nb<PRO, GATE, NB, false>(p, stream);
}

static int launch_linear_split(const LinearSplitArgs &p, bool gate, hipStream_t stream)
{
    if (p.norm_w != nullptr) return gate ? launch_pro<kLsNorm, true>(p, stream) : launch_pro<kLsNorm, false>(p, stream);
    if (p.x2 != nullptr) return launch_pro<kLsMulGelu, false>(p, stream);
    return gate ? launch_pro<kLsPlain, true>(p, stream) : launch_pro<kLsPlain, false>(p, stream);
}

// 0 = nothing to do, 1 = go on, anything else an error
static int linear_split_checks(const float *x, int64_t x_row_stride, const float *x2, int64_t x2_row_stride, const float *norm_weight,
                             const void *weight_packed, const float *bias, const float *resid, int64_t resid_row_stride,
                             const float *out, int64_t out_row_stride, int64_t R, int K, int N, int gate)
{
    if (R < 0 || K < 1 || N < 1) return BNB_ERR_BAD_SHAPE;
    if (K % 128 != 0 || N % 32 != 0 || (gate && N % 64 != 0)) return BNB_ERR_UNSUPPORTED;
    if (norm_weight != nullptr && (K != 128 || x2 != nullptr)) return BNB_ERR_UNSUPPORTED;
    if (gate && (bias != nullptr || x2 != nullptr)) return BNB_ERR_UNSUPPORTED;
    if (R == 0) return 0;
    if (!x || !weight_packed || !out) return BNB_ERR_NULL_POINTER;
    const int n_out = gate ? N / 2 : N;
    if (x_row_stride < K || out_row_stride < n_out || (x2 && x2_row_stride < K) || (resid && resid_row_stride < n_out))
        return BNB_ERR_BAD_SHAPE;
    if (!aligned16(x) || !aligned16(weight_packed) || x_row_stride % 4 != 0 || (x2 && (!aligned16(x2) || x2_row_stride % 4 != 0)) ||
        (norm_weight && !aligned16(norm_weight)))
        return BNB_ERR_MISALIGNED;
    return 1;
}

}  // namespace bnb

extern "C" int bnb_linear_f32_fwd(const float *x, int64_t x_row_stride, const float *x2, int64_t x2_row_stride,
                                  const float *norm_weight, float eps, const void *weight_packed, const float *bias,
                                  const float *resid, int64_t resid_row_stride, float *out, int64_t out_row_stride, int64_t R,
                                  int K, int N, int gate, void *stream)
{
    using namespace bnb;
    const int rc = linear_split_checks(x, x_row_stride, x2, x2_row_stride, norm_weight, weight_packed, bias, resid, resid_row_stride, out,
                                       out_row_stride, R, K, N, gate);
    if (rc != 1) return rc;
    return launch_linear_split({x, x_row_stride, x2, x2_row_stride, norm_weight, eps, (const uint16_t *)weight_packed, bias, resid,
                                resid_row_stride, out, out_row_stride, R, K, N / 32}, gate != 0, (hipStream_t)stream);
}
