// The tail of a sublayer in float32 (evaluation without autocast) as one kernel on the bf16 matrix cores:
//
//     s   = x + A Wp^T                                   A = rows | gelu(rows) * rows2
//     out = s + (gelu(n Wg^T) * (n Wu^T)) Wd^T           n = rmsnorm(s) * norm_w
//     HEAD: head1 = n' W1^T, head2 = n' W2^T             n' = rmsnorm(out) * next norm_w: what the next sublayer starts with
//
// (models/yemong/attention.py:21-37,97-98,132,169; models/yemong/griffin.py:238-247,269-287).  Operands as three bf16 pieces and
// products by size as in linear_split.hip; the float32 rows s, the hidden units and out never leave the work-group, where as
// separate launches the 512-wide hidden units went to memory and back and each launch filled the chip for one round.
//
// Eight waves hold 32 rows.  No weight is used by two waves: operands go from L2 straight into registers, a few steps ahead of
// their products.  Projection and down projection: four blocks of 32 channels x two halves of the contraction; gate / up: 64 hidden
// units a wave, split into pieces as they are formed; head: blocks of 32 features in turn.  The rows' pieces lie in LDS (26 KB), the
// hidden units' as well (100 KB): one work-group a CU.  What bounds it: the six products of every contraction step (312 a wave
// without a head, 8 us at two waves a SIMD) and the 1.25 MB of weight pieces a tile at 64 bytes a clock (8 us), one beside the other.
// Measured with a head of 384 features, the launches it replaces -> one kernel, us: 1 row 59 -> 29, 8,191 rows 70 -> 32,
// 12,288 rows 87 -> 54, 16,320 rows 91 -> 58, 27,680 rows 128 -> 105, 60,000 rows 243 -> 216: faster at every size, so it has no
// rule on the row count.  Operand rows read one step further ahead, and the six products in another order: no faster.
// Against float64 the relative error is 1.00e-7 (separate: 1.06e-7), of the heads 1.28e-7 (1.38e-7).
//
// What the pieces cannot carry shows as a value that is not finite: such a row is formed once more from whole float32 values.

#include "split_math.h"
#include "tile_rows.h"

namespace bnb {

constexpr int kTfD = 128, kTfHidden = 512, kTfRows = 32, kTfWaves = 8;
constexpr int kTfPitch = kTfD + 8;            // halfs of an operand row
constexpr int kTfHiddenPitch = kTfHidden + 8;
constexpr int kTfPartPitch = kTfD + 4;        // floats of a row of a partial result
constexpr int kTfPart = kTfRows * kTfPartPitch;

struct TailSplitArgs {
    const float *x, *a, *y;  // y NULL: plain projection
    int64_t x_stride, a_stride, y_stride;
    const uint16_t *wp, *wgu, *wd;
    const float *norm_w;
    float eps;
    float *out;
    const float *head_norm;  // NULL: no head
    float head_eps;
    const uint16_t *head1, *head2;
    float *out1, *out2;
    int blocks1, blocks2;  // of 32 features
    int64_t R;
};

struct TailShared {
    uint16_t n[3][kTfRows * kTfPitch];
    uint16_t h[3][kTfRows * kTfHiddenPitch];
    float part[2 * kTfPart];
    int off[kTfRows];    // the row holds a value that is not finite
    int alone[kTfRows];  // it came with a NaN: left as it is
    int any;
};
static_assert(sizeof(TailShared) <= 160 * 1024, "one work-group a CU");

// six products of one contraction step, weights as the first operand: the lane holds a row, the registers features
__device__ __forceinline__ void products_wn(const bf16x8 (&w)[3], const bf16x8 (&n)[3], Sums &s)
{
    s.small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[0], n[2], s.small, 0, 0, 0);
    s.mid = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[0], n[1], s.mid, 0, 0, 0);
    s.big = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[0], n[0], s.big, 0, 0, 0);
    s.small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[1], n[1], s.small, 0, 0, 0);
    s.mid = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[1], n[0], s.mid, 0, 0, 0);
    s.small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[2], n[0], s.small, 0, 0, 0);
}

template <bool HEAD>
__global__ __launch_bounds__(kTfWaves * kWave) __attribute__((amdgpu_waves_per_eu(2, 2))) void tail_split_kernel(const TailSplitArgs p)
{
    __shared__ __align__(16) TailShared s;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cb = wave & 3, kh = wave >> 2;
    const int m = lane & 31, half = lane >> 5;         // matrix-core mapping
    const int row = tid >> 4, c4 = (tid & 15) * 4;     // row mapping: channels c4 .. +3 and 64 + c4 .. +3
    const int64_t row0 = (int64_t)blockIdx.x * kTfRows;
    const bool valid = row0 + row < p.R;
    const int64_t r = valid ? row0 + row : p.R - 1;    // rows past the end repeat the last one and are not stored

    // the three pieces of a contraction step
    auto weights = [&](const uint16_t *w, bf16x8 (&to)[3]) {
#pragma unroll
        for (int q = 0; q < 3; ++q) to[q] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(w + (q * 512 + lane * 8)));
    };
    auto rows_of = [&](const uint16_t *base, int piece_halfs, int at, bf16x8 (&to)[3]) {
#pragma unroll
        for (int q = 0; q < 3; ++q) to[q] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(base + q * piece_halfs + at));
    };
    // this thread's eight channels as pieces into the operand rows (order of a group of 16 channels: 0-3, 8-11, 4-7, 12-15)
    auto put_pieces = [&](const float (&v)[8]) {
        bf16x8 q[3];
        split8(v, q[0], q[1], q[2]);
        uint16_t *to = s.n[0] + row * kTfPitch + 16 * (c4 >> 4) + ((c4 & 4) << 1) + ((c4 & 8) >> 1);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const u32x4 t = __builtin_bit_cast(u32x4, q[i]);
            *reinterpret_cast<u32x2 *>(to + i * kTfRows * kTfPitch) = u32x2{t.x, t.y};
            *reinterpret_cast<u32x2 *>(to + i * kTfRows * kTfPitch + 64) = u32x2{t.z, t.w};
        }
    };
    auto store_part = [&](const Sums &z) {
        float *to = s.part + kh * kTfPart + m * kTfPartPitch + 32 * cb + 4 * half;
#pragma unroll
        for (int v = 0; v < 16; v += 4)
            *reinterpret_cast<f32x4 *>(to + 2 * v) = f32x4{z.total(v), z.total(v + 1), z.total(v + 2), z.total(v + 3)};
    };
    float x[8];
    auto add_parts = [&]() {  // x += the two halves of the contraction; a row that is not finite any more is noted
        const float *q = s.part + row * kTfPartPitch + c4;
        float odd = 0.0f;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const f32x4 t = *reinterpret_cast<const f32x4 *>(q + 64 * i) + *reinterpret_cast<const f32x4 *>(q + kTfPart + 64 * i);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                x[4 * i + e] = t[e] + x[4 * i + e];
                odd = fmaf(x[4 * i + e], 0.0f, odd);
            }
        }
        if (odd != 0.0f && valid) s.off[row] = 1, s.any = 1;
    };
    float rstd = 0.0f;
    auto norm = [&](const float *w, float eps, float (&v)[8]) {
        const f32x4 wa = *reinterpret_cast<const f32x4 *>(w + c4), wb = *reinterpret_cast<const f32x4 *>(w + 64 + c4);
        float ss = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(x[e], x[e], ss);
        rstd = rsqrtf(sum16(ss) * (1.0f / kTfD) + eps);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = x[e] * rstd * wa[e], v[4 + e] = x[4 + e] * rstd * wb[e];
    };
    auto operand_rows = [&](int64_t at, float (&v)[8]) {
        const Row8 a = load8_split<false>(p.a + at * p.a_stride + c4, 64);
        if (p.y != nullptr) {
            const Row8 y = load8_split<false>(p.y + at * p.y_stride + c4, 64);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = gelu_erf_ls(a.v[e]) * y.v[e];
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = a.v[e];
        }
    };

    // ---- rows, and the projection's operands ----
    {
        float v[8];
        operand_rows(r, v);
        const Row8 t = load8_split<false>(p.x + r * p.x_stride + c4, 64);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = t.v[e];
        bool nan = false;
#pragma unroll
        for (int e = 0; e < 8; ++e) nan = nan || v[e] != v[e] || x[e] != x[e];
        if (tid < kTfRows) s.off[tid] = s.alone[tid] = 0;
        if (tid == 0) s.any = 0;
        bf16x8 w[4][3];
        const uint16_t *wp = p.wp + cb * kLsChunkHalfs + kh * 4 * 1536;
#pragma unroll
        for (int j = 0; j < 4; ++j) weights(wp + j * 1536, w[j]);
        put_pieces(v);
        lds_barrier();
        if (nan) s.alone[row] = 1;
        Sums z;
        z.clear();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            bf16x8 n[3];
            rows_of(s.n[0], kTfRows * kTfPitch, m * kTfPitch + 64 * kh + 16 * j + 8 * half, n);
            products_wn(w[j], n, z);
        }
        store_part(z);
    }
    constexpr int AHEAD = 3;
    // gate / up: the stream holds a gate block and an up block of 32 units in turn
    const uint16_t *wgu = p.wgu + (int64_t)(4 * wave) * kLsChunkHalfs;
    bf16x8 g[AHEAD][3], u[AHEAD][3];
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) weights(wgu + k * 1536, g[k]), weights(wgu + kLsChunkHalfs + k * 1536, u[k]);
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    add_parts();
    {
        float v[8];
        norm(p.norm_w, p.eps, v);
        put_pieces(v);
    }
    lds_barrier();

    bool odd_units = false;
#pragma unroll 1
    for (int c = 0; c < 2; ++c) {
        Sums zg, zu;
        zg.clear(), zu.clear();
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            bf16x8 n[3];
            rows_of(s.n[0], kTfRows * kTfPitch, m * kTfPitch + 16 * ks + 8 * half, n);
            products_wn(g[ks % AHEAD], n, zg);
            products_wn(u[ks % AHEAD], n, zu);
            if (ks + AHEAD < 8) {
                const uint16_t *w = wgu + 2 * c * kLsChunkHalfs + (ks + AHEAD) * 1536;
                weights(w, g[ks % AHEAD]), weights(w + kLsChunkHalfs, u[ks % AHEAD]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (c == 0) {
            const uint16_t *w = wgu + 2 * kLsChunkHalfs;
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) weights(w + k * 1536, g[k]), weights(w + kLsChunkHalfs + k * 1536, u[k]);
            __builtin_amdgcn_sched_barrier(0);
        }
        float odd = 0.0f;
        uint16_t *to = s.h[0] + m * kTfHiddenPitch + 32 * (2 * wave + c) + 8 * half;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            float h[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float a = zg.total(8 * t + e), b = zu.total(8 * t + e);
                odd = fmaf(a, 0.0f, odd), odd = fmaf(b, 0.0f, odd);
                h[e] = gelu_erf_ls(a) * b;
            }
            bf16x8 q[3];
            split8(h, q[0], q[1], q[2]);
#pragma unroll
            for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8 *>(to + i * kTfRows * kTfHiddenPitch + 16 * t) = q[i];
        }
        odd_units = odd_units || odd != 0.0f;
    }
    if (odd_units && row0 + m < p.R) s.off[m] = 1, s.any = 1;
    {
        constexpr int FAR = 6;
        // steps q = 0 .. 15 of this half: hidden units 256 kh + 16 q ..
        const uint16_t *wd = p.wd + (int64_t)(cb * 4 + 2 * kh) * kLsChunkHalfs;
        bf16x8 d[FAR][3];
#pragma unroll
        for (int k = 0; k < FAR; ++k) weights(wd + k * 1536, d[k]);
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier();
        Sums z;
        z.clear();
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            bf16x8 h[3];
            rows_of(s.h[0], kTfRows * kTfHiddenPitch, m * kTfHiddenPitch + 256 * kh + 16 * q + 8 * half, h);
            products_wn(d[q % FAR], h, z);
            if (q + FAR < 16) weights(wd + (q + FAR) * 1536, d[q % FAR]);
            __builtin_amdgcn_sched_barrier(0);
        }
        store_part(z);
    }
    bf16x8 hw[AHEAD][3];
    const int blocks = HEAD ? p.blocks1 + p.blocks2 : 0;
    auto head_stream = [&](int b) { return b < p.blocks1 ? p.head1 + (int64_t)b * kLsChunkHalfs : p.head2 + (int64_t)(b - p.blocks1) * kLsChunkHalfs; };
    if (HEAD) {
        const uint16_t *w = head_stream(wave < blocks ? wave : 0);
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) weights(w + k * 1536, hw[k]);
    }
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    add_parts();
    lds_barrier();

    if (s.any) {
        // ---- rows with a value that is not finite, once more from whole values ----
        float *vec = s.part, *hid = s.part + kTfD;  // s or out of the row; its hidden units, before them its operand
        for (int k = 0; k < kTfRows; ++k) {
            if (!s.off[k] || s.alone[k]) continue;
            const int64_t rk = row0 + k;
            if (row == k) {
                float v[8];
                operand_rows(rk, v);
                const Row8 t = load8_split<false>(p.x + rk * p.x_stride + c4, 64);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int ch = c4 + (e & 3) + 64 * (e >> 2);
                    vec[ch] = t.v[e], hid[ch] = v[e];
                }
            }
            __syncthreads();
            float sum = 0.0f;
            if (tid < kTfD) {
                for (int i = 0; i < kTfD; ++i) sum = fmaf(hid[i], whole_weight(p.wp, 1, tid >> 5, tid & 31, i), sum);
                sum += vec[tid];
            }
            __syncthreads();
            if (tid < kTfD) vec[tid] = sum;
            __syncthreads();
            float ss = 0.0f;
            for (int i = 0; i < kTfD; ++i) ss = fmaf(vec[i], vec[i], ss);
            const float rs = rsqrtf(ss * (1.0f / kTfD) + p.eps);
            float ga = 0.0f, up = 0.0f;
            for (int i = 0; i < kTfD; ++i) {
                const float v = vec[i] * rs * p.norm_w[i];
                ga = fmaf(v, whole_weight(p.wgu, 1, 2 * (tid >> 5), tid & 31, i), ga);
                up = fmaf(v, whole_weight(p.wgu, 1, 2 * (tid >> 5) + 1, tid & 31, i), up);
            }
            hid[tid] = gelu_erf_ls(ga) * up;
            __syncthreads();
            if (tid < kTfD) {
                float o = 0.0f;
                for (int i = 0; i < kTfHidden; ++i) o = fmaf(hid[i], whole_weight(p.wd, 4, tid >> 5, tid & 31, i), o);
                vec[tid] = o + vec[tid];  // read by this thread alone until the barrier
            }
            __syncthreads();
            if (row == k) {
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = vec[c4 + (e & 3) + 64 * (e >> 2)];
            }
            __syncthreads();
        }
    }
    if (valid) store8_split<false>(p.out + r * kTfD + c4, 64, Row8{{x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7]}});

    if constexpr (HEAD) {
        float v[8];
        norm(p.head_norm, p.head_eps, v);
        put_pieces(v);
        float *whole = s.part + row * kTfPartPitch + c4;  // for a result that is not finite
        *reinterpret_cast<f32x4 *>(whole) = f32x4{v[0], v[1], v[2], v[3]};
        *reinterpret_cast<f32x4 *>(whole + 64) = f32x4{v[4], v[5], v[6], v[7]};
        lds_barrier();
#pragma unroll 1
        for (int b = wave; b < blocks; b += kTfWaves) {
            const uint16_t *w = head_stream(b), *wn = head_stream(b + kTfWaves < blocks ? b + kTfWaves : b);
            Sums z;
            z.clear();
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) {
                bf16x8 n[3];
                rows_of(s.n[0], kTfRows * kTfPitch, m * kTfPitch + 16 * ks + 8 * half, n);
                // rows as the first operand: the lane holds a feature, and a store instruction whole runs of 32
                const bf16x8(&q)[3] = hw[ks % AHEAD];
                z.small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(n[2], q[0], z.small, 0, 0, 0);
                z.mid = __builtin_amdgcn_mfma_f32_32x32x16_bf16(n[1], q[0], z.mid, 0, 0, 0);
                z.big = __builtin_amdgcn_mfma_f32_32x32x16_bf16(n[0], q[0], z.big, 0, 0, 0);
                z.small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(n[1], q[1], z.small, 0, 0, 0);
                z.mid = __builtin_amdgcn_mfma_f32_32x32x16_bf16(n[0], q[1], z.mid, 0, 0, 0);
                z.small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(n[0], q[2], z.small, 0, 0, 0);
                if (ks + AHEAD < 8) weights(w + (ks + AHEAD) * 1536, hw[ks % AHEAD]);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) weights(wn + k * 1536, hw[k]);
            __builtin_amdgcn_sched_barrier(0);
            const bool first = b < p.blocks1;
            const int feat = 32 * (first ? b : b - p.blocks1) + m;
            const int width = 32 * (first ? p.blocks1 : p.blocks2);
            float *to = (first ? p.out1 : p.out2) + row0 * width + feat;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int rr = 8 * (v >> 2) + 4 * half + (v & 3);
                float o = z.total(v);
                if (__any(not_finite(o))) {
                    if (not_finite(o)) {
                        const float *n32 = s.part + rr * kTfPartPitch;
                        o = 0.0f;
                        for (int i = 0; i < kTfD; ++i) o = fmaf(n32[i], whole_weight(first ? p.head1 : p.head2, 1, feat >> 5, m, i), o);
                    }
                }
                if (row0 + rr < p.R) to[(int64_t)rr * width] = o;
            }
        }
    }
}

}  // namespace bnb

extern "C" int bnb_tail_f32_fwd(const float *x, int64_t x_row_stride, const float *a, int64_t a_row_stride, const float *y,
                                int64_t y_row_stride, const void *proj_packed, const float *norm_weight, float eps, const void *gate_up_packed,
                                const void *down_packed, float *out, const float *head_norm_weight, float head_eps, const void *head1_packed,
                                float *head1_out, int head1_features, const void *head2_packed, float *head2_out, int head2_features,
                                int64_t R, int D, int hidden, void *stream)
{
    using namespace bnb;
    if (R < 0 || head1_features < 0 || head2_features < 0) return BNB_ERR_BAD_SHAPE;
    if (D != kTfD || hidden != kTfHidden || head1_features % 32 || head2_features % 32) return BNB_ERR_UNSUPPORTED;
    if (R == 0) return 0;
    const bool head = head_norm_weight != nullptr;
    if (!x || !a || !proj_packed || !norm_weight || !gate_up_packed || !down_packed || !out ||
        (head && (!head1_packed || !head1_out || head1_features == 0 || (head2_features > 0 && (!head2_packed || !head2_out)))))
        return BNB_ERR_NULL_POINTER;
    if (x_row_stride < D || a_row_stride < D || (y && y_row_stride < D)) return BNB_ERR_BAD_SHAPE;
    if (!aligned16(x) || !aligned16(a) || !aligned16(y) || !aligned16(out) || !aligned16(proj_packed) || !aligned16(norm_weight) ||
        !aligned16(gate_up_packed) || !aligned16(down_packed) || !aligned16(head_norm_weight) || !aligned16(head1_packed) ||
        !aligned16(head2_packed) || x_row_stride % 4 || a_row_stride % 4 || (y && y_row_stride % 4))
        return BNB_ERR_MISALIGNED;
    const int64_t grid = (R + kTfRows - 1) / kTfRows;
    if (grid > 0x7fffffffLL) return BNB_ERR_UNSUPPORTED;
    TailSplitArgs p{x, a, y, x_row_stride, a_row_stride, y_row_stride, (const uint16_t *)proj_packed, (const uint16_t *)gate_up_packed,
                    (const uint16_t *)down_packed, norm_weight, eps, out, head_norm_weight, head_eps, (const uint16_t *)head1_packed,
                    (const uint16_t *)head2_packed, head1_out, head2_out, head ? head1_features / 32 : 0, head ? head2_features / 32 : 0, R};
    if (head) hipLaunchKernelGGL(tail_split_kernel<true>, dim3((unsigned)grid), dim3(kTfWaves * kWave), 0, (hipStream_t)stream, p);
    else hipLaunchKernelGGL(tail_split_kernel<false>, dim3((unsigned)grid), dim3(kTfWaves * kWave), 0, (hipStream_t)stream, p);
    return (int)hipGetLastError();
}
