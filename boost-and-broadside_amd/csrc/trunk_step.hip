// One timestep of the whole trunk as a single kernel, for small fleets under bfloat16 autocast.
//
// Environments do not see each other, so a work-group takes the environments that fit 32 token rows through every sublayer
// (reference: models/yemong/griffin.py:376-417 over models/yemong/attention.py:89-169 and griffin.py:269-317) and only tokens,
// masks, bullets in flight and the recurrent state come from memory.  Step for step it computes what the separate kernels do
// (norm_linear, sdpa_*, ffn_*, temporal_step), with their rounding points but two: the separate kernels round the merged heads, add the
// read to them and round again, here each of the two is rounded once and the projection adds them (WAVES = 8) or their float32 sum
// is rounded once (WAVES = 4); and a single reader's bullet norm weight is folded into its K and V weights like those of several.  The two forms also add the halves of a contraction in another order, so they agree to a bfloat16
// rounding, not bit for bit.  The residual stream stays in registers, eight channels a thread, and what one wave hands the next goes
// through LDS:
//
//   norm           16 lanes a row, bf16 rows into LDS
//   attention      waves 0..3 one head of the self-attention each, waves 4..7 one head of the bullet read each.  Q, K and V of a
//                  head come out of the products in exactly the registers that the score and value products take (V with the
//                  operands exchanged, which transposes it), so a head never leaves its wave.  The tile holds several
//                  environments: keys of another one carry a score of -inf.
//   projection     four blocks of 32 channels x two halves of the contraction; the merged heads and the read are two
//                  contractions over the same weights
//   recurrence     conv taps and state on the row mapping, the gate products eight blocks of 32 features, one a wave
//   gated MLP      gate / up: 64 hidden units a wave; down: four channel blocks x two halves of the hidden units
//
// What bounds it: every weight of the trunk passes through every work-group once, 0.5 to 0.6 MB a sublayer at the 64 bytes a
// clock that a CU takes from its L2 (22 us of the 61 for two blocks of three sublayers; 27 us with all 256 CUs at it), and the
// phases of a sublayer hang on one another over six to eight barriers: matrix cores and vector ALU of a SIMD are busy for 86,000 of
// 153,000 cycles.  So requests are dealt between matrix products and
// activations (a burst of them stalls the wave that issues it), norm weights are asked for before operands (loads come back in
// order), the barriers wait for LDS traffic only, and nothing may spill: a reload would wait for every operand under way.  In the
// order in which that was found, 16 environments of 12 tokens: 93, 82, 66, 64 us; the separate kernels, 19 launches, 121 us.
// 512 environments of 8 tokens 66 us (143).
//
// Two forms.  WAVES = 8 (one work-group a CU): heads and read, and the halves of a contraction, on different waves.  WAVES = 4 (two
// work-groups a CU, where there are more than CUs): a wave does both one after the other and has twice the rows in the row
// mapping; the first operands are requested where they are used, the neighbour's arithmetic covers the wait.  A wave issues
// 28,000 cycles of matrix products and 52,000 of vector instructions for its tile, which a SIMD does not overlap: busy for 72 % of the
// time.  512 environments of 23 tokens 113 us (243), a rollout of 7808 x 12 760 us in a running loop (880), 50 us for every 32 rows of a
// CU against 62 us with eight waves; 900 us in the first dozen launches after an idle spell, until the clock is up.

#include "common.h"
#include "ffn_math.h"
#include "rglru_math.h"
#include "tile_rows.h"

namespace bnb {

constexpr int kTkD = 128;
constexpr int kTkRows = 32;
constexpr int kTkPitch = kTkD + 8;            // halfs per operand row
constexpr int kTkHiddenPitch = kFfnHidden + 8;
constexpr int kTkHeadPitch = 3 * kTkD + 8;    // [b1 | gate | field rows of y]
constexpr int kTkGatePitch = 2 * kTkD + 8;
constexpr int kTkPartPitch = kTkD + 4;        // floats per row of a partial result
constexpr int kTkPart = kTkRows * kTkPartPitch;
constexpr int kTkSlots = 2048;                // bullet slots of a work-group's environments
constexpr int kTkHeads = 4;
constexpr int kTkDh = 32;
constexpr int kTkChunkHalfs = 3 * 32 * kFfnD;

template <int WAVES>
struct TrunkShared {
    static constexpr int kSegment = 16 * WAVES;  // bullet rows held at a time
    uint16_t n[kTkRows * kTkPitch];
    uint16_t h[kTkRows * kTkHiddenPitch];     // hidden units; merged heads and read; head of the temporal sublayer
    float part[WAVES / 4 * kTkPart];          // (partial) results of a projection; gate pre-activations
    uint16_t bullets[kSegment * kTkPitch];    // normalised rows of the bullets in flight
    uint16_t list[kTkSlots];                  // their positions, relative to the first environment's first slot
    int count[WAVES];
    int off[kTkRows + 1];                     // first list entry of each environment
};
static_assert(2 * kTkRows * kTkPitch <= kTkRows * kTkHiddenPitch && kTkRows * kTkHeadPitch <= kTkRows * kTkHiddenPitch, "overlays of h");
static_assert(kTkRows * kTkGatePitch * 2 <= kTkPart * 4, "gates overlay the first partial result");
static_assert(2 * sizeof(TrunkShared<4>) <= 160 * 1024, "two work-groups of four waves share a CU");

struct TrunkStepArgs {
    bnb_trunk_layer layer[BNB_TRUNK_MAX_LAYERS];
    int n_layers;
    int x_bf16, out_bf16, bullets_bf16;
    const void *x;
    void *out;
    const uint8_t *alive;   // NULL: everyone
    const uint8_t *reset;   // NULL: nobody
    const void *bullets;    // NULL: no read
    const uint8_t *in_flight;  // NULL: every slot
    float bullet_eps;
    int NB, B, NM, n_rec;
    const float *state_in;
    float *state_out;
};

__device__ __forceinline__ bf16x8 lds_operand(const uint16_t *p) { return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(p)); }
__device__ __forceinline__ bf16x8 mem_operand(const uint16_t *p) { return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(p)); }
__device__ __forceinline__ f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ u32x4 pack8(const float *v)
{
    return u32x4{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
}
// all ones where the bit is set
__device__ __forceinline__ uint32_t bit_mask(uint32_t w, int bit) { return (uint32_t)__builtin_amdgcn_sbfe((int)w, bit, 1); }
// bits [lo, hi) of a word, both clamped to it
__device__ __forceinline__ uint32_t bit_range(int lo, int hi)
{
    lo = lo < 0 ? 0 : lo > 32 ? 32 : lo;
    hi = hi < 0 ? 0 : hi > 32 ? 32 : hi;
    return (uint32_t)((1ull << hi) - 1ull) & ~(uint32_t)((1ull << lo) - 1ull);
}

// N times: VALU vector instructions, then one request from memory
template <int N, int VALU>
__device__ __forceinline__ void deal_requests()
{
#pragma unroll
    for (int i = 0; i < N; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x002, VALU, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
    }
}
// N times: one matrix product, then one request from memory
template <int N>
__device__ __forceinline__ void deal_requests_mfma()
{
#pragma unroll
    for (int i = 0; i < N; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
    }
}

template <int WAVES>
__global__ __launch_bounds__(WAVES * kWave) __attribute__((amdgpu_waves_per_eu(2, 2))) void trunk_step_kernel(const TrunkStepArgs a)
{
    constexpr bool SPLIT = WAVES == 8;               // heads and read, and halves of a contraction, on different waves
    constexpr int THREADS = WAVES * kWave;
    constexpr int PASS = THREADS / 16;               // rows of one pass of the row mapping
    constexpr int RP = kTkRows / PASS;               // passes: rows of a thread
    constexpr int CHUNKS = kFfnChunks / WAVES;       // chunks of 32 hidden units of a wave
    constexpr int KS = SPLIT ? 4 : 8;                // contraction steps of a wave's part of the output projection
    constexpr int kSegment = TrunkShared<WAVES>::kSegment;
    __shared__ __align__(16) TrunkShared<WAVES> s;
    int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cb = wave & 3, kh = wave >> 2;  // kh is 0 unless SPLIT
    // Both mappings of a thread, from its number: matrix cores (lane = 32 half + m) and rows (16 lanes a row, channels
    // c4 .. +3 and 64 + c4 .. +3).  `tid` is made opaque once a sublayer, so that the addresses that hang on it are formed
    // where they are used instead of being kept in registers through the loop.
    int lane, m, half, row, c4;
    auto mappings = [&]() {
        asm volatile("" : "+v"(tid));
        lane = tid & 63, m = lane & 31, half = lane >> 5, row = tid >> 4, c4 = (tid & 15) * 4;
    };
    mappings();
    auto operand_col = [&]() { return 16 * (c4 >> 4) + ((c4 & 4) << 1) + ((c4 & 8) >> 1); };  // see norm_rows

    const int NM = a.NM, n_rec = a.n_rec;
    const int envs = kTkRows / NM;  // NM <= 32, checked by the launcher
    const int env0 = blockIdx.x * envs;
    const int here = a.B - env0 < envs ? a.B - env0 : envs;
    const int rows = here * NM;
    const int64_t row0 = (int64_t)env0 * NM;

    // Operands of a sublayer's first phase, and its norm's weights (first: loads come back in order).  Attention: one head's
    // columns of Q, K and V (SPLIT, waves 4..7: of Q and of the read's K and V).  Temporal: the wave's blocks of the head, SPLIT:
    // one or two and in w2 the row's state [h | p0 | p1 | p2], else two or three.  Without branches, so that the requests can be
    // dealt between arithmetic.
    bf16x8 w0[8], w1[8], w2[8];
    f32x4 wn[2];
    struct First {
        const float *norm;
        const uint16_t *p0, *p1;
        const char *p2;
        int off2, step2;
    };
    auto state_row = [&](int r) {  // row of the recurrent state relative to the work-group's first; 0 for a token without one
        const int env = r / NM, tok = r - env * NM;
        return r < rows && tok < n_rec ? env * n_rec + tok : 0;
    };
    auto state_base = [&](const bnb_trunk_layer &L) { return (L.state_slot * ((int64_t)a.B * n_rec) + (int64_t)env0 * n_rec) * (4 * kTkD); };
    auto first_of = [&](const bnb_trunk_layer &L) {
        const uint16_t *head = (const uint16_t *)L.head;
        const bool t = L.temporal != 0;
        First f;
        f.norm = L.norm1;
        f.p0 = head + (t ? wave : cb) * 4096;
        if constexpr (SPLIT) {
            const bool kv = wave >= 4 && L.kv != nullptr;
            f.p1 = t ? (wave + 8 < L.head_blocks ? f.p0 + 8 * 4096 : f.p0) : kv ? (const uint16_t *)L.kv + cb * 4096 : f.p0 + 4 * 4096;
            f.p2 = t ? (const char *)(a.state_in + state_base(L)) : (const char *)(f.p1 + 4 * 4096);
            f.off2 = t ? (state_row(row) * (4 * kTkD) + c4) * 4 : lane * 16;
            f.step2 = t ? 256 : 1024;
        } else {
            f.p1 = f.p0 + 4 * 4096;
            f.p2 = (const char *)(t && L.head_blocks <= 8 ? f.p0 : f.p0 + 8 * 4096);
            f.off2 = lane * 16;
            f.step2 = 1024;
        }
        return f;
    };
    auto first_norm = [&](const First &f) {
        wn[0] = *reinterpret_cast<const f32x4 *>(f.norm + c4);
        wn[1] = *reinterpret_cast<const f32x4 *>(f.norm + 64 + c4);
    };
    auto first_q = [&](const First &f) {
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) w0[ks] = mem_operand(f.p0 + (ks * 512 + lane * 8));
    };
    auto first_kv = [&](const First &f) {
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            w1[ks] = mem_operand(f.p1 + (ks * 512 + lane * 8));
            w2[ks] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(f.p2 + ks * f.step2 + f.off2));
        }
    };

    // ---- what comes from memory first: flags, rows, the first operands ----
    // (an absent or idle lane's byte comes from some other readable place: a branch around it would wait for it on the spot)
    const int slots = a.bullets != nullptr ? here * a.NB : 0;
    const uint8_t *const some = (const uint8_t *)a.x;
    const uint8_t *fl = a.in_flight == nullptr || slots == 0 ? nullptr : a.in_flight + (int64_t)env0 * a.NB;
    uint32_t flag = *(fl != nullptr && tid < slots ? fl + tid : some);
    const uint32_t alive_byte = *(a.alive != nullptr && m < rows ? a.alive + row0 + m : some);
    float x[RP][8];
#pragma unroll
    for (int rp = 0; rp < RP; ++rp) {
        const int r = row + PASS * rp;
        const bool present = r < rows;
        const int at = (present ? r : 0) * kTkD + c4;
        const Row8 t = a.x_bf16 ? load8_split<false>((const uint16_t *)a.x + row0 * kTkD + at, 64)
                                : load8_split<false>((const float *)a.x + row0 * kTkD + at, 64);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[rp][e] = present ? t.v[e] : 0.0f;
    }
    {
        const First f = first_of(a.layer[0]);
        first_norm(f);
        if (SPLIT) first_q(f), first_kv(f);
        __builtin_amdgcn_sched_barrier(0);
    }
    const uint32_t alive_bits = (uint32_t)__ballot(m < rows && (a.alive == nullptr || alive_byte != 0));  // both halves hold the same rows

    // ---- the bullets in flight, in slot order ----
    int total = 0;
    if (slots > 0) {
        if (tid <= here) s.off[tid] = 0;
        lds_barrier();
#pragma unroll 1
        for (int p0 = 0; p0 < slots; p0 += THREADS) {
            const int p = p0 + tid;
            if (p0 > 0) flag = fl != nullptr && p < slots ? fl[p] : 0;
            const bool set = p < slots && (fl == nullptr || flag != 0);
            const uint64_t vote = __ballot(set);
            if (lane == 0) s.count[wave] = (int)__popcll(vote);
            if (set)
                for (int e = p / a.NB + 1; e <= here; ++e) atomicAdd(&s.off[e], 1);
            lds_barrier();
            int before = 0, all = 0;
#pragma unroll
            for (int w = 0; w < WAVES; ++w) {
                const int c = s.count[w];
                before += w < wave ? c : 0;
                all += c;
            }
            if (set) s.list[total + before + (int)__popcll(vote & ((1ull << lane) - 1ull))] = (uint16_t)p;
            total += all;
            lds_barrier();
        }
        total = __builtin_amdgcn_readfirstlane(total);
    }
    const int segments = (total + kSegment - 1) / kSegment;
    // bf16 rows in LDS list the channels of a group of 16 as 0-3, 8-11, 4-7, 12-15: a lane's eight of a contraction step, in the
    // order of the weight streams, are one 16-byte piece
    auto put_rows = [&](uint16_t *p, const float *v) {
        *reinterpret_cast<u32x2 *>(p) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        *reinterpret_cast<u32x2 *>(p + 64) = u32x2{pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
    };
    int held = -1;  // the segment that lies in LDS
    // x / rms(x) of a segment's rows into LDS; rows up to the next multiple of 32 are zero
    auto stage_bullets = [&](int seg) {
        held = seg;
        const int n = total - seg * kSegment < kSegment ? total - seg * kSegment : kSegment;
#pragma unroll 1
        for (int i0 = 0; i0 < n; i0 += 2 * PASS) {
            Row8 t[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int i = i0 + PASS * k + row;
                const int64_t r = (int64_t)env0 * a.NB + s.list[seg * kSegment + (i < n ? i : 0)];
                t[k] = a.bullets_bf16 ? load8_split<false>((const uint16_t *)a.bullets + r * kTkD + c4, 64)
                                      : load8_split<false>((const float *)a.bullets + r * kTkD + c4, 64);
            }
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int i = i0 + PASS * k + row;
                float ss = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) ss = fmaf(t[k].v[e], t[k].v[e], ss);
                const float rstd = rsqrtf(sum16(ss) * (1.0f / kTkD) + a.bullet_eps);
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = i < n ? t[k].v[e] * rstd : 0.0f;
                put_rows(s.bullets + i * kTkPitch + operand_col(), v);
            }
        }
    };

    auto norm_rows = [&](float eps) {  // weights in wn
#pragma unroll
        for (int rp = 0; rp < RP; ++rp) {
            float ss = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) ss = fmaf(x[rp][e], x[rp][e], ss);
            const float rstd = rsqrtf(sum16(ss) * (1.0f / kTkD) + eps);
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = (x[rp][e] * rstd) * wn[e >> 2][e & 3];
            put_rows(s.n + (row + PASS * rp) * kTkPitch + operand_col(), v);
        }
    };
    auto add_parts = [&]() {
#pragma unroll
        for (int rp = 0; rp < RP; ++rp) {
            const float *p = s.part + (row + PASS * rp) * kTkPartPitch + c4;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                f32x4 t = *reinterpret_cast<const f32x4 *>(p + 64 * q);
                if (SPLIT) t += *reinterpret_cast<const f32x4 *>(p + kTkPart + 64 * q);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[rp][4 * q + e] += t[e];
            }
        }
    };
    auto store_part = [&](const f32x16 &z) {
        float *p = s.part + kh * kTkPart + m * kTkPartPitch + 32 * cb + 4 * half;
#pragma unroll
        for (int v = 0; v < 16; v += 4) *reinterpret_cast<f32x4 *>(p + 2 * v) = f32x4{z[v], z[v + 1], z[v + 2], z[v + 3]};
    };
    auto bf16_halves = [&](const f32x16 &z, bf16x8 (&out)[2]) {
#pragma unroll
        for (int v = 0; v < 16; ++v) out[v >> 3][v & 7] = (__bf16)z[v];
    };

#pragma unroll 1
    for (int l = 0; l < a.n_layers; ++l) {
        mappings();
        const bnb_trunk_layer &L = a.layer[l];
        const bool temporal = L.temporal != 0;
        const bool read = !temporal && L.kv != nullptr && a.bullets != nullptr;
        if (l > 0) add_parts();
        norm_rows(L.eps1);
        const uint16_t *proj_rows = s.n;
        if (read && segments > 0 && held != 0) stage_bullets(0);
        // !SPLIT: the first operands are requested here, in each branch by itself (before the branch, the attention's would occupy
        // registers all through the recurrence)
        auto enter = [&]() {
            if constexpr (!SPLIT) {
                const First f = first_of(L);
                first_q(f), first_kv(f);
                __builtin_amdgcn_sched_barrier(0);
            }
            lds_barrier();
        };

        if (!temporal) {
            asm volatile("; attention" ::: "memory");  // keeps the compiler from merging the two branches' requests in front of them
            enter();
            proj_rows = s.h;
            // ---- one head of the self-attention (waves 0..3) or of the read (waves 4..7) ----
            const float scale_log2e = 0.17677669529663687f * kLog2e;
            const bf16x2 ones = {(__bf16)1.0f, (__bf16)1.0f};
            const int q_env = m / NM < here ? m / NM : 0;  // this lane's query is row m of the tile
            bf16x8 qb[2];
            {
                f32x16 z = {0.0f};
#pragma unroll
                for (int ks = 0; ks < 8; ++ks) z = mfma(w0[ks], lds_operand(s.n + m * kTkPitch + 16 * ks + 8 * half), z);
                bf16_halves(z, qb);
            }
            uint16_t *const merged = s.h + m * kTkPitch + kTkDh * cb + 4 * half;
            [[maybe_unused]] f32x16 own;  // !SPLIT: the head's own attention, while the read runs
            // SPLIT: this wave's one of the two; else one after the other
#pragma unroll 1
            for (int src = SPLIT ? kh : 0;; ++src) {
            const bool self = src == 0;
            f32x16 o = {0.0f};
            float mx = -INFINITY, sum = 0.0f;
#pragma unroll 1
            for (int seg = 0;; ++seg) {
                const int first = seg * kSegment;
                const int chunks = self ? (seg == 0 ? 1 : 0) : !read ? 0 : (total - first < kSegment ? total - first + 31 : kSegment) >> 5;
#pragma unroll 1
                for (int c = 0; c < chunks; ++c) {
                    const uint16_t *kr = (self ? s.n : s.bullets + c * 32 * kTkPitch) + m * kTkPitch + 8 * half;
                    f32x16 zk = {0.0f}, zv = {0.0f};
#pragma unroll
                    for (int ks = 0; ks < 8; ++ks) {
                        const bf16x8 kb = lds_operand(kr + 16 * ks);
                        zk = mfma(w1[ks], kb, zk);
                        zv = mfma(kb, w2[ks], zv);
                    }
                    // keys that this lane's query sees, and for the value rows the keys that anyone sees
                    const int base = self ? 0 : first + 32 * c;
                    const int lo = self ? q_env * NM : s.off[q_env], hi = self ? lo + NM : s.off[q_env + 1];
                    uint32_t mine = bit_range(lo - base, hi - base), seen = ~0u;
                    const bf16x8 zero8 = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
                    bf16x8 qs[2] = {qb[0], qb[1]};
                    if (self) {
                        const bool flat = (mine & alive_bits) == 0;  // nobody alive: everyone with the same weight
                        mine = flat ? mine : mine & alive_bits;
                        seen = (uint32_t)__ballot((mine >> m) & 1u);
                        qs[0] = flat ? zero8 : qb[0], qs[1] = flat ? zero8 : qb[1];
                    }
                    bf16x8 va[2];
                    f32x16 z = {0.0f};
                    bf16_halves(zk, va);
                    z = mfma(va[0], qs[0], z);
                    z = mfma(va[1], qs[1], z);
                    const uint32_t mine_h = mine >> (4 * half), seen_h = seen >> (4 * half);
                    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
                    u16x2 largest = {0, 0};  // of the value rows' magnitudes as bf16 patterns
#pragma unroll
                    for (int v = 0; v < 16; ++v)
                        va[v >> 3][v & 7] = (__bf16)__uint_as_float(__float_as_uint(zv[v]) & bit_mask(seen_h, (v & 3) + 8 * (v >> 2)));
#pragma unroll
                    for (int v = 0; v < 8; ++v) {
                        const uint32_t w = __builtin_bit_cast(u32x4, va[v >> 2])[v & 3] & 0x7fff7fffu;
                        largest = __builtin_elementwise_max(largest, __builtin_bit_cast(u16x2, w));
                    }
                    const bool odd = largest.x >= 0x7f80 || largest.y >= 0x7f80;  // not finite
                    float top = -INFINITY;
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const uint32_t k = bit_mask(mine_h, (v & 3) + 8 * (v >> 2));
                        z[v] = __uint_as_float((__float_as_uint(z[v]) & k) | (0xff800000u & ~k));
                        top = fmaxf(top, z[v]);
                    }
                    top = fmaxf(mx, fmaxf(top, __shfl_xor(top, 32)));
                    const float shift = top == -INFINITY ? 0.0f : top * scale_log2e;
                    const float alpha = __builtin_amdgcn_exp2f(fmaf(mx, scale_log2e, -shift));  // 0 the first time
                    mx = top;
                    bf16x8 pb[2];
                    float part = 0.0f;
#pragma unroll
                    for (int v = 0; v < 16; ++v) pb[v >> 3][v & 7] = (__bf16)__builtin_amdgcn_exp2f(fmaf(z[v], scale_log2e, -shift));
#pragma unroll
                    for (int v = 0; v < 16; v += 2)
                        part = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{pb[v >> 3][v & 7], pb[v >> 3][(v & 7) + 1]}, ones, part, false);
                    part += __shfl_xor(part, 32);
                    sum = fmaf(sum, alpha, part);
#pragma unroll
                    for (int v = 0; v < 16; ++v) o[v] *= alpha;
                    if (!__any(odd)) {
                        o = mfma(va[0], pb[0], o);
                        o = mfma(va[1], pb[1], o);
                    } else {
                        // a value row that is not finite spoils its own environment only: 0 * inf must not reach the others
#pragma unroll 1
                        for (int e = 0; e < here; ++e) {
                            const int elo = self ? e * NM : s.off[e], ehi = self ? elo + NM : s.off[e + 1];
                            const uint32_t of_env = bit_range(elo - base, ehi - base) >> (4 * half);
                            bf16x8 ve[2];
#pragma unroll
                            for (int v = 0; v < 16; ++v)
                                ve[v >> 3][v & 7] = (of_env >> ((v & 3) + 8 * (v >> 2))) & 1u ? va[v >> 3][v & 7] : (__bf16)0.0f;
                            f32x16 t = {0.0f};
                            t = mfma(ve[0], pb[0], t);
                            t = mfma(ve[1], pb[1], t);
#pragma unroll
                            for (int v = 0; v < 16; ++v) o[v] = q_env == e ? o[v] + t[v] : o[v];
                        }
                    }
                }
                if (!read || seg + 1 >= segments || (!SPLIT && self)) break;
                lds_barrier();
                stage_bullets(seg + 1);
                lds_barrier();
            }
            // merged heads (SPLIT: and the read behind them) as operand rows of the projection
            const float inv = sum == 0.0f ? 0.0f : __builtin_amdgcn_rcpf(sum);
#pragma unroll
            for (int v = 0; v < 16; ++v) o[v] *= inv;
            if constexpr (!SPLIT) {
                if (self && read) {
                    own = o;
                    const uint16_t *kv = (const uint16_t *)L.kv + cb * 4096;
#pragma unroll
                    for (int ks = 0; ks < 8; ++ks) {
                        w1[ks] = mem_operand(kv + (ks * 512 + lane * 8));
                        w2[ks] = mem_operand(kv + 4 * 4096 + (ks * 512 + lane * 8));
                    }
                    continue;
                }
                if (!self) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) o[v] += own[v];
                }
            }
            uint16_t *p = merged + (SPLIT && !self ? kTkRows * kTkPitch : 0);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                *reinterpret_cast<u32x2 *>(p + 16 * t) = u32x2{pack_bf16x2(o[8 * t], o[8 * t + 1]), pack_bf16x2(o[8 * t + 2], o[8 * t + 3])};
                *reinterpret_cast<u32x2 *>(p + 16 * t + 8) =
                    u32x2{pack_bf16x2(o[8 * t + 4], o[8 * t + 5]), pack_bf16x2(o[8 * t + 6], o[8 * t + 7])};
            }
            break;
            }
        } else {
            asm volatile("; recurrence" ::: "memory");
            enter();
            // ---- the head: [b1 | gate | field rows of y] ----
            auto head_block = [&](const bf16x8 (&w)[8], int b) {
                f32x16 z = {0.0f};
#pragma unroll
                for (int ks = 0; ks < 8; ++ks) z = mfma(w[ks], lds_operand(s.n + m * kTkPitch + 16 * ks + 8 * half), z);
                bf16x8 t[2];
                bf16_halves(z, t);
                uint16_t *p = s.h + m * kTkHeadPitch + 32 * b + 8 * half;
                *reinterpret_cast<bf16x8 *>(p) = t[0];
                *reinterpret_cast<bf16x8 *>(p + 16) = t[1];
            };
            head_block(w0, wave);
            if constexpr (SPLIT) {
                if (wave + 8 < L.head_blocks) head_block(w1, wave + 8);
            } else {
                head_block(w1, wave + 4);
                if (wave + 8 < L.head_blocks) head_block(w2, wave + 8);
                __builtin_amdgcn_sched_barrier(0);
            }
            // state (SPLIT: under way since the last sublayer), taps, and the gate operands: block q = 0, 1 of gate a, 2, 3 of
            // gate x, for half hf of the channels; a wave has one, or the one of each half
            constexpr int GB = SPLIT ? 1 : 2;
            const int gate = (wave & 3) >> 1, gcol = 64 * kh + 32 * (wave & 1);
            f32x4 cw[8], cbias[2], l2sig[2];
#pragma unroll
            for (int e = 0; e < 8; ++e) cw[e] = *reinterpret_cast<const f32x4 *>(L.conv_weight + (4 * c4 + 4 * (e & 3) + 256 * (e >> 2)));
            const float *cbp = L.conv_bias != nullptr ? L.conv_bias : L.conv_weight;
#pragma unroll
            for (int e = 0; e < 2; ++e) cbias[e] = *reinterpret_cast<const f32x4 *>(cbp + (64 * e + c4));
            f32x16 g[GB];
            auto gate_operands = [&]() {
                const uint16_t *gp = (const uint16_t *)L.gates + wave * 4096;
#pragma unroll
                for (int b = 0; b < GB; ++b) {
#pragma unroll
                    for (int v = 0; v < 16; v += 4) {
                        const f32x4 t = *reinterpret_cast<const f32x4 *>(L.gate_bias + gate * kTkD + gcol + 64 * b + (16 * half + v));
#pragma unroll
                        for (int e = 0; e < 4; ++e) g[b][v + e] = t[e];
                    }
                }
#pragma unroll
                for (int ks = 0; ks < 8; ++ks) w0[ks] = mem_operand(gp + (ks * 512 + lane * 8));
                if (!SPLIT) {
#pragma unroll
                    for (int ks = 0; ks < 8; ++ks) w1[ks] = mem_operand(gp + 4 * 4096 + (ks * 512 + lane * 8));
                }
#pragma unroll
                for (int e = 0; e < 2; ++e) l2sig[e] = *reinterpret_cast<const f32x4 *>(L.log2_sigmoid + (64 * e + c4));
                __builtin_amdgcn_sched_barrier(0);
            };
            if (SPLIT) gate_operands();
            uint32_t reset_byte[RP];
#pragma unroll
            for (int rp = 0; rp < RP; ++rp) {
                const int r = row + PASS * rp;
                reset_byte[rp] = *(a.reset != nullptr ? a.reset + env0 + (r < rows ? r / NM : 0) : (const uint8_t *)L.norm1);
            }
            float *so = a.state_out + state_base(L);
            auto ship = [&](int rp) {
                const int r = row + PASS * rp;
                return r < rows && r % NM < n_rec;
            };
            auto state_at = [&](int rp) { return state_row(row + PASS * rp) * (4 * kTkD) + c4; };
            lds_barrier();

            // ---- conv taps and buffer shift ----
            float v[RP][8];
            f32x4 h_in[RP][2];
#pragma unroll
            for (int rp = 0; rp < RP; ++rp) {
                const bool zero = a.reset != nullptr && reset_byte[rp] != 0;
                const float *sin = a.state_in + state_base(L) + state_at(rp);
                f32x4 st[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) st[i] = SPLIT ? __builtin_bit_cast(f32x4, w2[i]) : *reinterpret_cast<const f32x4 *>(sin + 64 * i);
#pragma unroll
                for (int i = 0; i < 8; ++i) st[i] = zero ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : st[i];
                h_in[rp][0] = st[0], h_in[rp][1] = st[1];
                const Row8 cur = load8_split<false>(s.h + (row + PASS * rp) * kTkHeadPitch + c4, 64);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int q = e >> 2, c = e & 3;
                    float t = st[2 + q][c] * cw[e].x;
                    t = fmaf(st[4 + q][c], cw[e].y, t);
                    t = fmaf(st[6 + q][c], cw[e].z, t);
                    t = fmaf(cur.v[e], cw[e].w, t);
                    v[rp][e] = t + (L.conv_bias != nullptr ? cbias[q][c] : 0.0f);
                }
                if (ship(rp)) {
                    float *to = so + state_at(rp);
#pragma unroll
                    for (int i = 0; i < 4; ++i) *reinterpret_cast<f32x4 *>(to + kTkD + 64 * i) = st[4 + i];
                    store8_split<false>(to + 3 * kTkD, 64, cur);
                }
                put_rows(s.n + (row + PASS * rp) * kTkPitch + c4, v[rp]);  // the gate operands list the channels in order
                if (!SPLIT) __builtin_amdgcn_sched_barrier(0);
            }
            if (!SPLIT) {
                __builtin_amdgcn_sched_barrier(0);
                gate_operands();  // here there are registers for them
            }
            lds_barrier();

            // ---- gate pre-activations ----
            uint16_t *const s_g = reinterpret_cast<uint16_t *>(s.part);
#pragma unroll
            for (int b = 0; b < GB; ++b) {
#pragma unroll
                for (int i = 0; i < 16; ++i) g[b][i] = round_to_bf16(g[b][i]);
#pragma unroll
                for (int ks = 0; ks < 8; ++ks)
                    g[b] = mfma(b == 0 ? w0[ks] : w1[ks], lds_operand(s.n + m * kTkPitch + 16 * ks + 8 * half), g[b]);
                bf16x8 t[2];
                bf16_halves(g[b], t);
                uint16_t *p = s_g + m * kTkGatePitch + gate * kTkD + gcol + 64 * b + 16 * half;
                *reinterpret_cast<bf16x8 *>(p) = t[0];
                *reinterpret_cast<bf16x8 *>(p + 8) = t[1];
            }
            lds_barrier();

            // ---- recurrence, and gelu(gate) * y as operand rows of the projection ----
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int rp = 0; rp < RP; ++rp) {
                const uint16_t *gr = s_g + (row + PASS * rp) * kTkGatePitch + c4;
                const uint16_t *hr = s.h + (row + PASS * rp) * kTkHeadPitch + c4;
                const Row8 ga = load8_split<false>(gr, 64), gx = load8_split<false>(gr + kTkD, 64);
                const Row8 gt = load8_split<false>(hr + kTkD, 64);
                Row8 out;
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    out.v[e] = rglru_element<true, false>(v[rp][e], ga.v[e], gx.v[e], l2sig[e >> 2][e & 3], L.c, h_in[rp][e >> 2][e & 3]);
                if (ship(rp)) store8_split<false>(so + state_at(rp), 64, out);
                else if (L.head_blocks > 8) out = load8_split<false>(hr + 2 * kTkD, 64);
                float r[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) r[e] = round_to_bf16(gelu_phi(gt.v[e])) * round_to_bf16(out.v[e]);
                put_rows(s.n + (row + PASS * rp) * kTkPitch + operand_col(), r);
                __builtin_amdgcn_sched_barrier(0);  // one row's temporaries at a time
            }
        }

        // ---- output projection; the first hidden units' operands are on their way behind it ----
        const uint16_t *wc = (const uint16_t *)L.ffn + (int64_t)(CHUNKS * wave) * kTkChunkHalfs;
        bf16x8 wg[2][8], wu[2][8];
        auto hidden_operands = [&](int c) {
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) wg[c & 1][ks] = mem_operand(wc + (c * kTkChunkHalfs + ks * 512 + lane * 8));
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) wu[c & 1][ks] = mem_operand(wc + (c * kTkChunkHalfs + 4096 + ks * 512 + lane * 8));
        };
        bf16x8 wp[KS];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < KS; ++j) wp[j] = mem_operand((const uint16_t *)L.proj + (cb * 8 + kh * 4) * 512 + (j * 512 + lane * 8));
        wn[0] = *reinterpret_cast<const f32x4 *>(L.norm2 + c4);
        wn[1] = *reinterpret_cast<const f32x4 *>(L.norm2 + 64 + c4);
        hidden_operands(0);
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier();
        {
            f32x16 z = {0.0f};
            const uint16_t *p = proj_rows + m * kTkPitch + 64 * kh + 8 * half;
#pragma unroll
            for (int j = 0; j < KS; ++j) z = mfma(wp[j], lds_operand(p + 16 * j), z);
            if (SPLIT && read) {
#pragma unroll
                for (int j = 0; j < KS; ++j) z = mfma(wp[j], lds_operand(p + kTkRows * kTkPitch + 16 * j), z);
            }
            store_part(z);
        }
        lds_barrier();
        add_parts();
        norm_rows(L.eps2);
        lds_barrier();

        // ---- gate / up: the wave's chunks of 32 hidden units; down: a channel block (SPLIT: over half of the hidden units) ----
        const uint16_t *wdp = (const uint16_t *)L.ffn + (int64_t)(8 * kh) * kTkChunkHalfs + 8192 + cb * 1024;
        bf16x8 wd[16], we[16];
        auto down_operands = [&](bf16x8 (&w)[16], int chunk) {
#pragma unroll
            for (int q = 0; q < 16; ++q) w[q] = mem_operand(wdp + ((chunk + (q >> 1)) * kTkChunkHalfs + (q & 1) * 512 + lane * 8));
        };
        bf16x8 nb[8];
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) nb[ks] = lds_operand(s.n + m * kTkPitch + 16 * ks + 8 * half);
        const First next = first_of(a.layer[l + 1 < a.n_layers ? l + 1 : l]);  // behind the last sublayer: any, for nobody
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c) {
            f32x16 g = {0.0f}, u = {0.0f};
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) {
                g = mfma(wg[c & 1][ks], nb[ks], g);
                u = mfma(wu[c & 1][ks], nb[ks], u);
            }
            if (c + 1 < CHUNKS) {
                hidden_operands(c + 1);
                deal_requests_mfma<16>();
            }
            __builtin_amdgcn_sched_barrier(0);
            bf16x8 t[2];
#pragma unroll
            for (int v = 0; v < 16; ++v) t[v >> 3][v & 7] = (__bf16)(gelu_phi(g[v]) * u[v]);
            if (c == (SPLIT ? 0 : CHUNKS - 1)) {
                down_operands(wd, 0);
                deal_requests<16, 9>();
            } else if (SPLIT) {
                first_norm(next), first_q(next);
                deal_requests<10, 14>();
            }
            __builtin_amdgcn_sched_barrier(0);
            uint16_t *p = s.h + m * kTkHiddenPitch + 32 * (CHUNKS * wave + c) + 8 * half;
            *reinterpret_cast<bf16x8 *>(p) = t[0];
            *reinterpret_cast<bf16x8 *>(p + 16) = t[1];
        }
        lds_barrier();
        {
            f32x16 z = {0.0f};
            const uint16_t *p = s.h + m * kTkHiddenPitch + 256 * kh + 8 * half;
#pragma unroll
            for (int q = 0; q < 16; ++q) z = mfma(wd[q], lds_operand(p + 16 * q), z);
            if constexpr (SPLIT) first_kv(next);
            else down_operands(we, 8);
            deal_requests_mfma<16>();
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (!SPLIT) {
#pragma unroll
                for (int q = 0; q < 16; ++q) z = mfma(we[q], lds_operand(p + 256 + 16 * q), z);
                first_norm(next);
            }
            store_part(z);
        }
        lds_barrier();
    }

    mappings();
    add_parts();
#pragma unroll
    for (int rp = 0; rp < RP; ++rp) {
        const int r = row + PASS * rp;
        if (r >= rows) continue;
        Row8 t;
#pragma unroll
        for (int e = 0; e < 8; ++e) t.v[e] = x[rp][e];
        if (a.out_bf16) store8_split<false>((uint16_t *)a.out + row0 * kTkD + (r * kTkD + c4), 64, t);
        else store8_split<false>((float *)a.out + row0 * kTkD + (r * kTkD + c4), 64, t);
    }
}

}  // namespace bnb

extern "C" int bnb_trunk_step_fwd(const bnb_trunk_layer *layers, int n_layers, const void *x, int x_dtype, void *out, int out_dtype,
                                  const uint8_t *alive, const uint8_t *reset, const void *bullets, int bullets_dtype,
                                  const uint8_t *in_flight, float bullet_eps, int NB, const float *state_in, float *state_out,
                                  int B, int NM, int n_rec, int D, int H, int hidden, void *stream)
{
    using namespace bnb;
    if (B < 0 || n_layers < 1 || NM < 1 || n_rec < 1 || n_rec > NM || NB < 0) return BNB_ERR_BAD_SHAPE;
    if (D != kTkD || H != kTkHeads || hidden != kFfnHidden || NM > kTkRows || n_layers > BNB_TRUNK_MAX_LAYERS) return BNB_ERR_UNSUPPORTED;
    if (bullets != nullptr && (int64_t)(kTkRows / NM) * NB > kTkSlots) return BNB_ERR_UNSUPPORTED;
    for (const int t : {x_dtype, out_dtype, bullets != nullptr ? bullets_dtype : BNB_F32})
        if (t != BNB_F32 && t != BNB_BF16) return BNB_ERR_BAD_DTYPE;
    if (B == 0) return 0;
    if (!layers || !x || !out) return BNB_ERR_NULL_POINTER;
    if (!aligned16(x) || !aligned16(out) || !aligned16(state_in) || !aligned16(state_out) || (bullets != nullptr && !aligned16(bullets)))
        return BNB_ERR_MISALIGNED;
    TrunkStepArgs a;
    for (int i = 0; i < n_layers; ++i) {
        const bnb_trunk_layer &L = layers[i];
        if (!L.head || !L.norm1 || !L.proj || !L.norm2 || !L.ffn) return BNB_ERR_NULL_POINTER;
        if (!aligned16(L.head) || !aligned16(L.norm1) || !aligned16(L.proj) || !aligned16(L.norm2) || !aligned16(L.ffn) || !aligned16(L.kv))
            return BNB_ERR_MISALIGNED;
        if (L.temporal) {
            if (!L.conv_weight || !L.gates || !L.gate_bias || !L.log2_sigmoid || !state_in || !state_out) return BNB_ERR_NULL_POINTER;
            if (!aligned16(L.conv_weight) || !aligned16(L.gates) || !aligned16(L.gate_bias) || !aligned16(L.conv_bias) || !aligned16(L.log2_sigmoid)) return BNB_ERR_MISALIGNED;
            if (L.head_blocks != (n_rec < NM ? 12 : 8) || L.state_slot < 0) return BNB_ERR_BAD_SHAPE;
        }
        a.layer[i] = L;
    }
    a.n_layers = n_layers;
    a.x = x, a.x_bf16 = x_dtype == BNB_BF16;
    a.out = out, a.out_bf16 = out_dtype == BNB_BF16;
    a.alive = alive, a.reset = reset;
    a.bullets = NB > 0 ? bullets : nullptr, a.bullets_bf16 = bullets_dtype == BNB_BF16, a.in_flight = in_flight;
    a.bullet_eps = bullet_eps, a.NB = NB;
    a.B = B, a.NM = NM, a.n_rec = n_rec;
    a.state_in = state_in, a.state_out = state_out;
    // As many environments a work-group as fit: with fewer, the weights pass through more CUs (512 environments of 8 tokens:
    // 128 work-groups 70 us, 256 work-groups 74 us; 16 of 12 tokens: 8 or 16 work-groups 64 us).
    const int envs = kTkRows / NM;
    // Up to one work-group a CU: eight waves, the shortest way through a sublayer.  More: four waves and half the LDS, so that two
    // work-groups share a CU and one's arithmetic covers the other's waits; 512 work-groups 112 us against 133, 3904 work-groups
    // 760 against 1000.
    const int64_t groups = (B + envs - 1) / envs;
    if (groups <= cu_count())
        hipLaunchKernelGGL(trunk_step_kernel<8>, dim3((unsigned)groups), dim3(8 * kWave), 0, (hipStream_t)stream, a);
    else
        hipLaunchKernelGGL(trunk_step_kernel<4>, dim3((unsigned)groups), dim3(4 * kWave), 0, (hipStream_t)stream, a);
    return (int)hipGetLastError();
}
