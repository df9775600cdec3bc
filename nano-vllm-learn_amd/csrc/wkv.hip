// Time mixing with a matrix state per head whose rows decay by their own factor at every token:
//   o_t = (S + diag(u) k_t v_t^T)^T r_t          S <- diag(w_t) S + k_t v_t^T          w_t = exp(-exp(z_t + w0))
// and behind it, per head: o / rms(o) * norm * silu(gate).  State, decays and everything between z and the weights are fp32.
//
// Prompt portions (launch_wkv_chunks): a workgroup owns one (segment, head) and takes 64 tokens at a time.  With L the running sum of the log decays over the
// chunk and m its value behind the first 32 tokens,
//   r~_t = r_t e^(L_(t-1) - m)        k~_j = k_j e^(m - L_j)
//   o_t = (e^m S)^T r~_t + sum_{j < t} (r~_t . k~_j) v_j + (r_t . u k_t) v_t          S <- e^L S + e^(L - m) sum_j k~_j v_j^T
// on MFMA tiles: every product that counts has its true size, r~ and k~ enter as bf16 hi + lo halves, S and the weights too.  A chunk in which a channel decays by
// more than 2^100 within 32 tokens would leave the range and is walked token by token on the same registers (no result depends on which way was taken but by
// rounding).  The state stays in fp32 accumulators, laid out so that they are the left operand of S^T r without a shuffle.  Rows go straight to registers, a chunk
// ahead: a thread holds 2 channels of 8 tokens.
// A portion of several segments: a SUMMARY walk leaves every segment's own contribution and the sum of its log decays, a small launch turns those into states at
// segment starts, and the second walk begins there.
// Decoding (launch_wkv_step): one workgroup per (sequence, head) computes the decays from the low-rank row, streams the state once, norms and gates.
// A sequence's first token (position 0) takes the state as zero instead of reading it: slots need no clearing when reused.
#include <type_traits>

#include "api_common.h"
#include "attend_tile.h"
#include "mixers.h"

namespace nvh {

namespace {

using WkvArgs = nvh_wkv_desc;
constexpr int C = 64;                                // tokens per chunk
constexpr int PLD = C + 8;                           // row of the weights in LDS
constexpr float kMaxDecay = 100.f;                   // log2 units a channel may decay in half a chunk on the MFMA way

__device__ __forceinline__ float log2_decay(float z) { return -kLog2e * __expf(z); }

__device__ __forceinline__ void split8(const float (&v)[8], bf16x8& hi, bf16x8& lo) {
    u32x4 h, l;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        h[j] = pack_bf16x2_once(v[2 * j], v[2 * j + 1]);
        l[j] = pack_bf16x2(v[2 * j] - bf16_lo(h[j]), v[2 * j + 1] - bf16_hi(h[j]));
    }
    hi = *reinterpret_cast<const bf16x8*>(&h);
    lo = *reinterpret_cast<const bf16x8*>(&l);
}

// the same number as one the compiler has not seen yet: what is computed from it is computed where it stands, not held in a register over the whole walk
__device__ __forceinline__ int fresh(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// The rows of a chunk, `n` of them from `base` on, of which a thread takes the bytes at `col` of row `row`.  Where offsets fit 32 bits the rows are a raw buffer whose end is the last row's:
// the thread's first row's offset and an addition per load, where the row's clamp and product took 20 cycles; what lies behind reads as zero and is not stored.
template <typename Off>
struct ChunkRows {
    __amdgpu_buffer_rsrc_t buf;
    uint32_t row_bytes;
    __device__ __forceinline__ ChunkRows(const void* base, int64_t bytes, int n, int width)
        : buf(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)((n - 1) * (uint32_t)bytes + width), 0x00020000)), row_bytes((uint32_t)bytes) {}
    __device__ __forceinline__ uint32_t first(int row, int col) const { return row * row_bytes + col; }
    __device__ __forceinline__ uint32_t word(uint32_t at, int i, int, int) const { return __builtin_amdgcn_raw_buffer_load_b32(buf, (int)(at + i * row_bytes), 0, 0); }
    __device__ __forceinline__ u32x4 four(uint32_t at, int i, int, int) const { return __builtin_amdgcn_raw_buffer_load_b128(buf, (int)(at + i * row_bytes), 0, 0); }
    __device__ __forceinline__ void put(uint32_t at, int i, int, int, u32x4 v) const { __builtin_amdgcn_raw_buffer_store_b128(v, buf, (int)(at + i * row_bytes), 0, 0); }
};
// (rows further apart; behind the last row that row again)
template <>
struct ChunkRows<int64_t> {
    unsigned char* base;
    int64_t row_bytes;
    int n;
    __device__ __forceinline__ ChunkRows(const void* base, int64_t bytes, int n, int) : base(static_cast<unsigned char*>(const_cast<void*>(base))), row_bytes(bytes), n(n) {}
    __device__ __forceinline__ uint32_t first(int, int) const { return 0; }
    __device__ __forceinline__ unsigned char* in(int row, int col) const { return base + (int64_t)(row < n ? row : n - 1) * row_bytes + col; }
    __device__ __forceinline__ uint32_t word(uint32_t, int i, int row, int col) const { return *reinterpret_cast<const uint32_t*>(in(fresh(row) + i, col)); }
    __device__ __forceinline__ u32x4 four(uint32_t, int i, int row, int col) const { return *reinterpret_cast<const u32x4*>(in(fresh(row) + i, col)); }
    __device__ __forceinline__ void put(uint32_t, int i, int row, int col, u32x4 v) const {
        if (row + i < n) *reinterpret_cast<u32x4*>(in(row + i, col)) = v;
    }
};

// d[i] summed over the 32 or 64 lanes of a token's channels, for eight tokens at once: every step adds half of one token's lanes to half of another's, so that each lane ends with one token
template <int LANES>
__device__ __forceinline__ float sums_of_eight(float (&d)[8]) {
    float e[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) e[i] = LANES == 64 ? fold32(d[i], d[i + 4]) : fold16(d[i], d[i + 4]);
    if constexpr (LANES == 64) {
        float f[2] = {fold16(e[0], e[2]), fold16(e[1], e[3])};
        asm("s_nop 1\n"
            "v_add_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0x3\n v_add_f32_dpp %0, %1, %1 row_ror:8 row_mask:0xf bank_mask:0xc\n"
            "s_nop 1"
            : "+&v"(f[0]) : "v"(f[1]));
        f[0] += dpp_f32<0x141>(f[0]);                // row_half_mirror
        e[0] = f[0];
    } else {
        asm("s_nop 1\n"
            "v_add_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0x3\n v_add_f32_dpp %0, %2, %2 row_ror:8 row_mask:0xf bank_mask:0xc\n"
            "v_add_f32_dpp %1, %1, %1 row_ror:8 row_mask:0xf bank_mask:0x3\n v_add_f32_dpp %1, %3, %3 row_ror:8 row_mask:0xf bank_mask:0xc\n"
            "s_nop 1\n"
            "v_add_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0x5\n v_add_f32_dpp %0, %1, %1 row_half_mirror row_mask:0xf bank_mask:0xa\n"
            "s_nop 1"
            : "+&v"(e[0]), "+&v"(e[1]) : "v"(e[2]), "v"(e[3]));
    }
    e[0] += dpp_f32<0xB1>(e[0]);                     // quad_perm [1,0,3,2]
    return e[0] + dpp_f32<0x4E>(e[0]);               // quad_perm [2,3,0,1]
}

template <int LANES>
__device__ __forceinline__ int which_of_eight(int lane) {    // the token whose sum this lane has
    return LANES == 64 ? (lane >> 5) * 4 + (lane >> 4 & 1) * 2 + (lane >> 3 & 1) : (lane >> 4 & 1) * 4 + (lane >> 2 & 3);
}

template <int DIM>
struct WkvLds {
    static constexpr int WAVES = DIM / 16, ROW = DIM * 2, IMG = C * ROW;
    unsigned char r_hi[IMG], r_lo[IMG], k_hi[IMG], k_lo[IMG], v[IMG];          // (token by token: w as fp32 over r_hi and r_lo, k and r as they came over k_hi and k_lo)
    uint16_t p[2][C][PLD];                                                     // weights, hi | lo (token by token: outputs, [wave][16][16] fp32)
    float tot[8][DIM];                                                         // log decays by groups of 8 tokens
    float to_mid[DIM], to_end[DIM], mid_to_end[DIM];                           // what a channel decays by up to m, over the chunk, from m on
    float w0[DIM], u[DIM];                                                     // (of the preparing waves' channels, whose registers are full)
    float bonus[C];
    float o[C][DIM + 4];                                                       // outputs on their way from a column of 16 tokens to rows
    int strong;
};

// DIM / 16 waves consume: wave w holds value columns 16 w .., state and outputs of this chunk.  As many prepare the next one: log decays and their sums, r~ and k~,
// weights.  Three parts a chunk, one barrier behind each; the images are written when this chunk's consumers are done with them:
//   consume: outputs, state               | norm, gate, store  | half of the weights of i + 1
//   prepare: values of chunk i + 1        | images, tables     | log decays of chunk i + 2, the other half
// (heads of 128, and rows far apart: | decays of i + 1 | values, images | weights |; the values' registers have no room there).
// What bounds it is issue and latency, not memory: 780 vector instructions a chunk and SIMD, where there were 1240 (rows by a buffer descriptor instead of a clamp and a 64-bit product each,
// masks only in a last chunk, eight tokens' sums at once, halves that are not rounded twice).  Two workgroups per CU (heads of 64: 79 KB and 128 registers each) keep four waves on every
// SIMD; no register of theirs may be spilled inside the loop: a reload waits for every row in flight (four of them: 129 us where none takes 103).
// Gates and results go by whole rows, through LDS: taken where the products leave them, 32 bytes of 16 rows a wave, they were 20 of 103 us.
// Measured, 32 heads of 64, 11 portions of 1090 tokens in the mean, three sets of lengths: 126, 114, 132 -> 97, 83, 110 us; 19 of 500: 74 -> 57; three of 2950, in segments: 100 -> 82.
// 16 heads of 128, 11 of 1090: 445 -> 398, 30 of 550: 405 -> 361 (some registers of 128 are spilled there).
// Two sets of images, one workgroup a CU and two parts a chunk instead: 106, 109, 139.
template <int DIM, bool SUMMARY, typename Off>
__global__ __launch_bounds__(DIM * 8, DIM == 64 ? 4 : 1) void wkv_walk_kernel(const WkvArgs a) {
    using Lds = WkvLds<DIM>;
    constexpr bool AHEAD = DIM == 64 && sizeof(Off) == 4;                // (at 128 more than 128 registers)
    constexpr int ROW = DIM * 2, DT = DIM / 16, CP = DIM / 2, WAVES = Lds::WAVES, T = DIM * 4;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    Lds& lds = *reinterpret_cast<Lds*>(smem);
    auto swz = [](int r) { return ROW == 128 ? (r >> 1) & 7 : r & 15; };       // rows of 256 bytes span all banks
    const int head = blockIdx.x, seg = longest_first<DIM == 64>(a, a.heads);    // heads run fastest: workgroups are dealt round-robin over the XCDs
    const int32_t* ch = a.chunks + 4 * seg;
    const int row0 = ch[0], n_rows = ch[1], seq = ch[2];
    const bool last = seg + 1 == a.n_chunks || a.chunks[4 * (seg + 1) + 3] == 0;
    if (SUMMARY && last) return;                     // (nothing follows it)
    const int wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, lq = lane & 15, lg = lane >> 4;
    const int64_t slot = a.state_slots[seq];
    constexpr int64_t head_state = (int64_t)DIM * DIM;
    if (n_rows <= 0) {
        if (SUMMARY || (last && slot >= 0 && ch[3] > 0))
            pass_segment<SUMMARY>(a.seg_state + ((int64_t)seg * a.heads + head) * head_state, a.state + (slot * a.heads + head) * head_state, DIM, DIM, DIM);
        if (SUMMARY && threadIdx.x < DIM) a.seg_decay[((int64_t)seg * a.heads + head) * DIM + threadIdx.x] = 0.f;
        return;
    }

    // weights D[key 16 jt + 4 lg + r][query 16 qg + lq]: the twelve 16 x 16 tiles the outputs read, dealt to all waves, first those that consume: four on
    // the diagonal, then six below it, then the two above it, which are zero
    auto weights = [&](auto prepares) __attribute__((always_inline)) {
        if (SUMMARY) return;
        constexpr bool P = decltype(prepares)::value;
        const int lane_ = fresh(lane), lq = lane_ & 15, lg = lane_ >> 4;
#pragma unroll
        for (int x0 = P && AHEAD ? WAVES : 0; x0 < 12; x0 += AHEAD ? 2 * WAVES : WAVES) {
            const int x = x0 + (P ? wave_id - WAVES : wave_id), y = x - 4;
            if (x >= 12) break;
            const int qg = x < 4 ? x : y < 6 ? (y > 2) + (y > 0) + 1 : 2 * (y - 6), jt = x < 4 ? x : y < 6 ? y - qg * (qg - 1) / 2 : qg + 1;
            const int q0 = 16 * ROW * qg, k0 = 16 * ROW * jt;
            f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < DIM / 32; ++st) {
                const int at = lq * ROW + ((4 * st + lg) ^ swz(lq)) * 16;  // (of 16 rows further on the same)
                const bf16x8 qh = *reinterpret_cast<const bf16x8*>(lds.r_hi + q0 + at), ql = *reinterpret_cast<const bf16x8*>(lds.r_lo + q0 + at);
                const bf16x8 kh = *reinterpret_cast<const bf16x8*>(lds.k_hi + k0 + at), kl = *reinterpret_cast<const bf16x8*>(lds.k_lo + k0 + at);
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kh, qh, s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kh, ql, s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kl, qh, s, 0, 0, 0);
            }
            float p[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) p[r] = s[r];
            if (x0 == 0 && (WAVES == 4 || x < 4)) {
                const float bonus = lds.bonus[16 * qg + lq];
#pragma unroll
                for (int r = 0; r < 4; ++r) p[r] = lq > 4 * lg + r ? s[r] : lq == 4 * lg + r ? bonus : 0.f;
            } else if (x0 + WAVES > 10) {
#pragma unroll
                for (int r = 0; r < 4; ++r) p[r] = x < 10 ? s[r] : 0.f;
            }
            const u32x2 hi = {pack_bf16x2_once(p[0], p[1]), pack_bf16x2_once(p[2], p[3])};
            const u32x2 lo = {pack_bf16x2(p[0] - bf16_lo(hi[0]), p[1] - bf16_hi(hi[0])), pack_bf16x2(p[2] - bf16_lo(hi[1]), p[3] - bf16_hi(hi[1]))};
            uint16_t* const to = &lds.p[0][lq][8 * lg] + (16 * PLD * qg + 32 * (jt >> 1) + 4 * (jt & 1));
            *reinterpret_cast<u32x2*>(to) = hi;
            *reinterpret_cast<u32x2*>(to + C * PLD) = lo;
        }
    };
    if (wave_id >= WAVES) {
        // ---- this thread's rows of a chunk: channels 2 cp, 2 cp + 1 of tokens 8 tg ..; two 16-byte pieces of values
        const int tid = threadIdx.x - T, wave = wave_id - WAVES, cp = tid % CP, tg = tid / CP;
        const int hc = head * DIM + 2 * cp;
        *reinterpret_cast<f32x2*>(&lds.w0[2 * cp]) = *reinterpret_cast<const f32x2*>(a.w0 + hc);
        if constexpr (!SUMMARY) *reinterpret_cast<f32x2*>(&lds.u[2 * cp]) = *reinterpret_cast<const f32x2*>(a.u + hc);
        uint32_t rr[8], kk[8], zz[8];
        u32x4 vv[2];
        // a chunk's rows.  Every chunk asks for as many rows as any other, in straight line: behind a branch around loads the compiler waits for all that are in flight
        // instead of the ones it needs
        const int t_last = (n_rows - 1) / C * C;
        auto rows_of = [&](const void* p, int64_t stride, int t0) __attribute__((always_inline)) {
            return ChunkRows<Off>(reinterpret_cast<const unsigned char*>(p) + 2 * ((int64_t)(row0 + t0) * stride + head * DIM), stride * 2, n_rows - t0 < C ? n_rows - t0 : C, ROW);
        };
        const int v_row = tid / (DIM / 8), v_col = tid % (DIM / 8) * 16;
        auto fetch_z = [&](int t) __attribute__((always_inline)) {
            const auto z = rows_of(a.z, a.z_stride, t < t_last ? t : t_last);
            const uint32_t at = z.first(fresh(8 * tg), 4 * cp);
#pragma unroll
            for (int i = 0; i < 8; ++i) zz[i] = z.word(at, i, 8 * tg, 4 * cp);
        };
        auto fetch = [&](int t) __attribute__((always_inline)) {
            const int t0 = t < t_last ? t : t_last;
            const auto k = rows_of(a.k, a.stride, t0), r = rows_of(a.r, a.stride, t0);
            const uint32_t at = k.first(fresh(8 * tg), 4 * cp);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                kk[i] = k.word(at, i, 8 * tg, 4 * cp);
                if constexpr (!SUMMARY) rr[i] = r.word(at, i, 8 * tg, 4 * cp);
            }
        };
        auto fetch_v = [&](int t) __attribute__((always_inline)) {
            const auto v = rows_of(a.v, a.stride, t < t_last ? t : t_last);
#pragma unroll
            for (int j = 0; j < 2; ++j) vv[j] = v.four(v.first(fresh(v_row), v_col), j * (T * 8 / DIM), v_row, v_col);
        };
        float la[8], lb[8];                          // sums of log decays up to and with token i of the group
        auto decays = [&](int n) __attribute__((always_inline)) {
            const f32x2 w0 = *reinterpret_cast<const f32x2*>(&lds.w0[2 * cp]);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                la[i] = log2_decay(bf16_lo(zz[i]) + w0[0]);
                lb[i] = log2_decay(bf16_hi(zz[i]) + w0[1]);
            }
            if (n < C) {
                const int left = fresh(n - 8 * tg);
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    la[i] = i < left ? la[i] : 0.f;
                    lb[i] = i < left ? lb[i] : 0.f;
                }
            }
            float sa = 0.f, sb = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                la[i] = sa += la[i];
                lb[i] = sb += lb[i];
            }
            *reinterpret_cast<f32x2*>(&lds.tot[tg][2 * cp]) = f32x2{sa, sb};
        };
        float dec_a = 0.f, dec_b = 0.f, bonus = 0.f;
        f32x2 mid, end;                              // sums of log decays up to m and over the chunk
        bool strong = false;
        uint32_t kh[8], kl[8], rh[8], rl[8];         // k~ and r~ as hi and lo halves; of a strong chunk k and r over kh and kl
        auto values = [&](int n) __attribute__((always_inline)) {
            if (n < C) {                             // keys past the end count nothing
                const int left = fresh(n - 8 * tg);
#pragma unroll
                for (int i = 0; i < 8; ++i) kk[i] = i < left ? kk[i] : 0u;
            }
            float oa = 0.f, ob = 0.f, ma = 0.f, mb = 0.f, fa = 0.f, fb = 0.f;
#pragma unroll
            for (int g = 0; g < 8; ++g) {
                const f32x2 s = *reinterpret_cast<const f32x2*>(&lds.tot[g][2 * cp]);
                oa = g == tg ? fa : oa;
                ob = g == tg ? fb : ob;
                fa += s[0];
                fb += s[1];
                if (g == 3) {
                    ma = fa;
                    mb = fb;
                }
            }
            dec_a += fa;
            dec_b += fb;
            // (every wave holds all channels: they agree)
            strong = __builtin_amdgcn_ballot_w64(!(fminf(fminf(ma, fa - ma), fminf(mb, fb - mb)) >= -kMaxDecay)) != 0;
            mid = f32x2{ma, mb};
            end = f32x2{fa, fb};
            if constexpr (!SUMMARY) {                // r . u k of the 8 tokens: over the lanes that hold a token's channels
                const f32x2 u = *reinterpret_cast<const f32x2*>(&lds.u[2 * cp]);
                const float ua = u[0], ub = u[1];
                float d[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) d[i] = bf16_lo(rr[i]) * ua * bf16_lo(kk[i]) + bf16_hi(rr[i]) * ub * bf16_hi(kk[i]);
                bonus = sums_of_eight<CP>(d);
            }
            if (!strong) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float ia = oa + la[i], ib = ob + lb[i];
                    const float ka = bf16_lo(kk[i]) * fast_exp2(ma - ia), kb = bf16_hi(kk[i]) * fast_exp2(mb - ib);
                    kh[i] = pack_bf16x2_once(ka, kb);
                    kl[i] = pack_bf16x2(ka - bf16_lo(kh[i]), kb - bf16_hi(kh[i]));
                    if constexpr (!SUMMARY) {
                        const float ea = oa + (i ? la[i ? i - 1 : 0] : 0.f), eb = ob + (i ? lb[i ? i - 1 : 0] : 0.f);
                        const float ra = bf16_lo(rr[i]) * fast_exp2(ea - ma), rb = bf16_hi(rr[i]) * fast_exp2(eb - mb);
                        rh[i] = pack_bf16x2_once(ra, rb);
                        rl[i] = pack_bf16x2(ra - bf16_lo(rh[i]), rb - bf16_hi(rh[i]));
                    }
                    if (AHEAD && (i & 1)) __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    kh[i] = kk[i];
                    if constexpr (!SUMMARY) kl[i] = rr[i];
                }
            }
        };
        auto images = [&](int t0, int n) __attribute__((always_inline)) {
            const int tid = fresh(threadIdx.x - T), cp = tid % CP, tg = tid / CP;
            if (n < C) {                             // values past the end count nothing
                const int v_left = fresh(n - tid / (DIM / 8));
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) vv[j][q] = j * (T * 8 / DIM) < v_left ? vv[j][q] : 0u;
            }
            if (!strong) {
                const int pofs = (cp & 3) * 4;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int t = 8 * tg + i, at = t * ROW + (((cp >> 2) ^ swz(t)) * 16) + pofs;
                    *reinterpret_cast<uint32_t*>(lds.k_hi + at) = kh[i];
                    *reinterpret_cast<uint32_t*>(lds.k_lo + at) = kl[i];
                    if constexpr (!SUMMARY) {
                        *reinterpret_cast<uint32_t*>(lds.r_hi + at) = rh[i];
                        *reinterpret_cast<uint32_t*>(lds.r_lo + at) = rl[i];
                    }
                }
            } else {
                // (rare: z is read again, its registers hold the next chunk's)
                float* w_f = reinterpret_cast<float*>(lds.r_hi);
                const auto zs = rows_of(a.z, a.z_stride, t0);
#pragma unroll 1
                for (int i = 0; i < 8; ++i) {
                    const int t = 8 * tg + i;
                    const uint32_t z = zs.word(zs.first(8 * tg, 4 * cp), i, 8 * tg, 4 * cp);
                    const float w0a = lds.w0[2 * cp], w0b = lds.w0[2 * cp + 1];
                    *reinterpret_cast<f32x2*>(w_f + t * DIM + 2 * cp) = f32x2{fast_exp2(log2_decay(bf16_lo(z) + w0a)), fast_exp2(log2_decay(bf16_hi(z) + w0b))};
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int t = 8 * tg + i;
                    *reinterpret_cast<uint32_t*>(lds.k_hi + t * ROW + 4 * cp) = kh[i];
                    if constexpr (!SUMMARY) *reinterpret_cast<uint32_t*>(lds.k_lo + t * ROW + 4 * cp) = kl[i];
                }
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int e = j * T + tid, t = e / (DIM / 8), pc = e % (DIM / 8);
                *reinterpret_cast<u32x4*>(lds.v + t * ROW + (pc ^ swz(t)) * 16) = vv[j];
            }
            if constexpr (!SUMMARY) lds.bonus[8 * tg + which_of_eight<CP>(tid & 63)] = bonus;      // (all lanes of a token hold it)
            if (tg == 0) {
                *reinterpret_cast<f32x2*>(&lds.to_mid[2 * cp]) = f32x2{fast_exp2(mid[0]), fast_exp2(mid[1])};
                *reinterpret_cast<f32x2*>(&lds.to_end[2 * cp]) = f32x2{fast_exp2(end[0]), fast_exp2(end[1])};
                *reinterpret_cast<f32x2*>(&lds.mid_to_end[2 * cp]) = f32x2{fast_exp2(end[0] - mid[0]), fast_exp2(end[1] - mid[1])};
                if (cp == 0) lds.strong = strong;
            }
        };
        auto rows = [&](int t0) { return n_rows - t0 < C ? n_rows - t0 : C; };
        fetch_z(0);
        fetch(0);
        fetch_v(0);
        if constexpr (AHEAD) {
            decays(rows(0));
            fetch_z(C);
        }
        lds_only_barrier();
        for (int t0 = 0; t0 < n_rows + C; t0 += C) {         // prepares the chunk at t0 while the one in front of it is consumed
            const bool there = t0 < n_rows;
            if constexpr (AHEAD) {
                if (there) values(rows(t0));
                fetch(t0 + C);
            } else {
                if (there) decays(rows(t0));
                fetch_z(t0 + C);
            }
            lds_only_barrier();
            if constexpr (!AHEAD) {
                if (there) values(rows(t0));
            }
            if (there) images(t0, rows(t0));
            if constexpr (!AHEAD) fetch(t0 + C);
            fetch_v(t0 + C);
            lds_only_barrier();
            if constexpr (AHEAD) {
                if (t0 + C < n_rows) decays(rows(t0 + C));
                fetch_z(t0 + 2 * C);
            }
            if (there && !strong) weights(std::true_type{});
            lds_only_barrier();
        }
        if constexpr (SUMMARY) {
            if (tg == 0) *reinterpret_cast<f32x2*>(a.seg_decay + (int64_t)seg * a.heads * DIM + hc) = f32x2{dec_a, dec_b};
        }
        return;
    }

    // state: value column 16 wave + lq, key rows 16 t + 4 lg + r
    const int wave = wave_id;
    f32x4 S[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) S[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int sv = 16 * wave + lq;
    if constexpr (!SUMMARY) {
        const float* src = nullptr;
        if (a.summaries) src = a.seg_state + ((int64_t)seg * a.heads + head) * head_state;
        else if (slot >= 0 && a.positions[row0] > 0) src = a.state + (slot * a.heads + head) * head_state;
        if (src) {
#pragma unroll
            for (int t = 0; t < DT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) S[t][r] = src[(16 * t + 4 * lg + r) * DIM + sv];
#pragma unroll
            for (int t = 0; t < DT; ++t) asm volatile("" : "+v"(S[t]));        // (waited for here, not in the loop)
        }
    }
    // this thread's pieces of a chunk's gates and results, 8 columns each: token row + 32 j
    const int row = threadIdx.x / (DIM / 8), col = threadIdx.x % (DIM / 8) * 8;
    f32x8 nw = {};
    if constexpr (!SUMMARY) nw = act_ld8(a.norm + head * DIM + col);
    const float inv_n = 1.f / a.n;
    u32x4 gate[2];
    auto rows_of = [&](const void* p, int64_t stride, int t0) __attribute__((always_inline)) {
        return ChunkRows<Off>(reinterpret_cast<const unsigned char*>(p) + 2 * ((int64_t)(row0 + t0) * stride + head * DIM), stride * 2, n_rows - t0 < C ? n_rows - t0 : C, ROW);
    };
    auto fetch_gate = [&](int t0) __attribute__((always_inline)) {
        if constexpr (!SUMMARY) {
            const auto g = rows_of(a.g, a.stride, t0);
#pragma unroll
            for (int j = 0; j < 2; ++j) gate[j] = g.four(g.first(row, 2 * col), 32 * j, row, 2 * col);
        }
    };
    // transposed reads of columns 16 t ..: row and column quarter this lane addresses (of 16 rows further on the same)
    auto tr_at = [&](int t) __attribute__((always_inline)) {
        const int lane_ = DIM == 64 ? lane : fresh(lane), tr = lane_ >> 2, tp = lane_ & 3;
        return tr * ROW + ((2 * t + (tp >> 1)) ^ swz(tr)) * 16 + (tp & 1) * 8;
    };
    fetch_gate(0);
    lds_only_barrier();                              // the first chunk's decays,
    lds_only_barrier();                              // values,
    lds_only_barrier();                              // images
    if (AHEAD && !__builtin_amdgcn_readfirstlane(lds.strong)) weights(std::false_type{});
    lds_only_barrier();
    for (int t0 = 0; t0 < n_rows; t0 += C) {
        const int n = n_rows - t0 < C ? n_rows - t0 : C;
        f32x4 o[4];                                  // o^T: value 16 wave + 4 lg + r, token 16 it + lq
        if (!__builtin_amdgcn_readfirstlane(lds.strong)) {
            // value fragments: lane = column 16 wave + lq, slots = keys 32 hh + 4 lg + 0..3 and the same + 16
            bf16x8 vf[2];
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                const unsigned char* const at = lds.v + tr_at(wave) + 32 * ROW * hh;
                const u32x2 lo = lds_tr16(at), hi = lds_tr16(at + 16 * ROW);
                const u32x4 raw = {lo[0], lo[1], hi[0], hi[1]};
                vf[hh] = *reinterpret_cast<const bf16x8*>(&raw);
            }
            if constexpr (!SUMMARY) {
                // what the state gives: slots of a 32-wide step are key rows 16 (2 st) + 4 lg + 0..3 and 16 (2 st + 1) + 4 lg + 0..3
#pragma unroll
                for (int it = 0; it < 4; ++it) o[it] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int st = 0; st < DIM / 32; ++st) {
                    float sc[8];
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const f32x4 m4 = *reinterpret_cast<const f32x4*>(&lds.to_mid[16 * (2 * st + q) + 4 * lg]);
#pragma unroll
                        for (int r = 0; r < 4; ++r) sc[4 * q + r] = S[2 * st + q][r] * m4[r];
                    }
                    bf16x8 hi, lo;
                    split8(sc, hi, lo);
                    const int lane_ = AHEAD ? lane : fresh(lane), lq = lane_ & 15, lg = lane_ >> 4;
                    const int pa = lq * ROW + ((4 * st + (lg >> 1)) ^ swz(lq)) * 16 + (lg & 1) * 8, pb = lq * ROW + ((4 * st + 2 + (lg >> 1)) ^ swz(lq)) * 16 + (lg & 1) * 8;
#pragma unroll
                    for (int it = 0; it < 4; ++it) {
                        const int R = 16 * ROW * it;
                        // (kept apart, or two rows' or both images' reads become one, whose halves have to be moved)
                        const u32x2 ha = *reinterpret_cast<const u32x2*>(lds.r_hi + R + pa), hb = *reinterpret_cast<const u32x2*>(lds.r_hi + R + pb);
                        if constexpr (AHEAD) asm volatile("" ::: "memory");
                        const u32x2 xa = *reinterpret_cast<const u32x2*>(lds.r_lo + R + pa), xb = *reinterpret_cast<const u32x2*>(lds.r_lo + R + pb);
                        if constexpr (AHEAD) asm volatile("" ::: "memory");
                        const u32x4 hraw = {ha[0], ha[1], hb[0], hb[1]}, lraw = {xa[0], xa[1], xb[0], xb[1]};
                        const bf16x8 qh = *reinterpret_cast<const bf16x8*>(&hraw), ql = *reinterpret_cast<const bf16x8*>(&lraw);
                        o[it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, qh, o[it], 0, 0, 0);
                        o[it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, ql, o[it], 0, 0, 0);
                        o[it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, qh, o[it], 0, 0, 0);
                    }
                }
#pragma unroll
                for (int it = 0; it < 4; ++it)
#pragma unroll
                    for (int hh = 0; hh <= it / 2; ++hh) {
                        o[it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[hh], *reinterpret_cast<const bf16x8*>(&lds.p[0][16 * it + lq][32 * hh + 8 * lg]), o[it], 0, 0, 0);
                        o[it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[hh], *reinterpret_cast<const bf16x8*>(&lds.p[1][16 * it + lq][32 * hh + 8 * lg]), o[it], 0, 0, 0);
                    }
            }
            // ---- the state behind these tokens
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                const int k_at = tr_at(t);
                f32x4 M = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int hh = 0; hh < 2; ++hh) {
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const unsigned char* const at = (q ? lds.k_lo : lds.k_hi) + k_at + 32 * ROW * hh;
                        const u32x2 ka = lds_tr16(at), kb = lds_tr16(at + 16 * ROW);
                        const u32x4 kraw = {ka[0], ka[1], kb[0], kb[1]};
                        M = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(&kraw), vf[hh], M, 0, 0, 0);
                    }
                }
                const f32x4 e4 = *reinterpret_cast<const f32x4*>(&lds.to_end[16 * t + 4 * lg]), f4 = *reinterpret_cast<const f32x4*>(&lds.mid_to_end[16 * t + 4 * lg]);
#pragma unroll
                for (int r = 0; r < 4; ++r) S[t][r] = e4[r] * S[t][r] + f4[r] * M[r];
            }
        } else {
            // ---- token by token; outputs of 16 tokens change lanes through a few LDS words of the wave
            const float* w_f = reinterpret_cast<const float*>(lds.r_hi);
            float* obuf = reinterpret_cast<float*>(lds.p) + wave * 256;
            const int lane_ = fresh(lane), lq = lane_ & 15, lg = lane_ >> 4, sv = 16 * wave + lq;
#pragma unroll
            for (int it = 0; it < 4; ++it) {
                o[it] = f32x4{0.f, 0.f, 0.f, 0.f};
                for (int i = 0; i < 16 && 16 * it + i < n; ++i) {
                    const int t = 16 * it + i;
                    const float v = act_ld(reinterpret_cast<const uint16_t*>(lds.v + t * ROW + ((sv >> 3) ^ swz(t)) * 16) + (sv & 7));
                    float acc = 0.f;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) {
                        const int key = 16 * dt + 4 * lg;
                        const f32x4 w4 = *reinterpret_cast<const f32x4*>(w_f + t * DIM + key), k4 = act_ld4(reinterpret_cast<const uint16_t*>(lds.k_hi + t * ROW) + key);
                        if constexpr (!SUMMARY) acc += sum4(act_ld4(reinterpret_cast<const uint16_t*>(lds.k_lo + t * ROW) + key) * S[dt]);
                        S[dt] = w4 * S[dt] + k4 * v;
                    }
                    if constexpr (!SUMMARY) {
                        acc = sum_xor16(acc);
                        acc = sum_xor32(acc) + lds.bonus[t] * v;
                        if (lg == 0) obuf[i * 16 + lq] = acc;
                    }
                }
                if constexpr (!SUMMARY) {
                    wave_lds_sync();
                    if (16 * it + lq < n) o[it] = *reinterpret_cast<const f32x4*>(obuf + lq * 16 + 4 * lg);
                    wave_lds_sync();
                }
            }
        }
        if constexpr (!SUMMARY) {
#pragma unroll
            for (int it = 0; it < 4; ++it) *reinterpret_cast<f32x4*>(&lds.o[16 * it + lq][16 * wave + 4 * lg]) = o[it];
        }
        lds_only_barrier();                          // this chunk's images may be replaced; outputs are there
        if constexpr (!SUMMARY) {
            // ---- norm over the head's columns, gate
            const auto out = rows_of(a.out, a.out_stride, t0);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const f32x8 y = act_ld8(&lds.o[row + 32 * j][col]), g = unpack8(gate[j]);
                const float inv = __builtin_amdgcn_rsqf(group_sum<DIM / 8>(sum4(y.a * y.a) + sum4(y.b * y.b)) * inv_n + a.eps);
                f32x8 r;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    r.a[k] = y.a[k] * inv * nw.a[k] * (g.a[k] * fast_rcp(1.f + fast_exp2(-kLog2e * g.a[k])));
                    r.b[k] = y.b[k] * inv * nw.b[k] * (g.b[k] * fast_rcp(1.f + fast_exp2(-kLog2e * g.b[k])));
                }
                out.put(out.first(row, 2 * col), 32 * j, row, 2 * col,
                        u32x4{pack_bf16x2(r.a[0], r.a[1]), pack_bf16x2(r.a[2], r.a[3]), pack_bf16x2(r.b[0], r.b[1]), pack_bf16x2(r.b[2], r.b[3])});
            }
            fetch_gate(t0 + C < n_rows ? t0 + C : t0);
        }
        lds_only_barrier();                          // the next chunk's images
        if (AHEAD && t0 + C < n_rows && !__builtin_amdgcn_readfirstlane(lds.strong)) weights(std::false_type{});
        lds_only_barrier();
    }
    float* dst = nullptr;
    if constexpr (SUMMARY) dst = a.seg_state + ((int64_t)seg * a.heads + head) * head_state;
    else if (last && slot >= 0) dst = a.state + (slot * a.heads + head) * head_state;
    if (dst) {
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) dst[(16 * t + 4 * lg + r) * DIM + sv] = S[t][r];
    }
}

// contributions of the segments -> states at their starts, in place; a thread per four state elements of a portion, walking its segments
__global__ __launch_bounds__(256) void wkv_starts_kernel(const WkvArgs a) {
    const int64_t per = (int64_t)a.heads * a.dim * a.dim, e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    const int first = blockIdx.y;                    // only a portion's first segment starts a walk
    if (a.chunks[4 * first + 3] != 0) return;
    const int count = portion_segments(a.chunks, a.n_chunks, first);
    if (e >= per) return;
    const int64_t ch = e / a.dim, slot = a.state_slots[a.chunks[4 * first + 2]], channels = (int64_t)a.heads * a.dim;
    const f32x4 cur = slot >= 0 && portion_carries(a.chunks, a.n_chunks, first, a.positions) ? *reinterpret_cast<const f32x4*>(a.state + slot * per + e) : f32x4{};
    segment_starts(a.seg_state + first * per + e, per, count, cur, [&](int k) { return a.seg_decay[(first + k) * channels + ch]; }, [](float decay) { return fast_exp2(decay); });
}

// ------------------------------------------------------------------------------------------------ token by token, any type and size
// one workgroup per (portion, head, 32 value columns); the state slice in LDS, 8 groups of key rows x 32 columns; norm and gate in a launch behind
template <typename T>
__global__ __launch_bounds__(256) void wkv_generic_kernel(const WkvArgs a) {
    extern __shared__ float lds_f[];                 // [dim][32] state, [4][dim] w, k, r, u, [8][32] sums
    float *S = lds_f, *wkr = S + a.dim * 32, *red = wkr + 4 * a.dim;
    const int first = blockIdx.x, head = blockIdx.y, tid = threadIdx.x, c = tid & 31, rg = tid >> 5, col = blockIdx.z * 32 + c;
    if (a.chunks[4 * first + 3] != 0) return;        // a portion is walked whole from its first segment
    const int row0 = a.chunks[4 * first];
    int n_rows = a.chunks[4 * first + 1];
    for (int k = first + 1; k < a.n_chunks && a.chunks[4 * k + 3] != 0; ++k) n_rows += a.chunks[4 * k + 1];
    const int64_t slot = a.state_slots[a.chunks[4 * first + 2]], head_state = (int64_t)a.dim * a.dim;
    const bool ok = col < a.dim;
    float* pool = slot >= 0 ? a.state + (slot * a.heads + head) * head_state : nullptr;
    const bool carry = pool && portion_carries(a.chunks, a.n_chunks, first, a.positions);
    for (int r = rg; r < a.dim; r += 8) S[r * 32 + c] = carry && ok ? pool[(int64_t)r * a.dim + col] : 0.f;
    for (int i = tid; i < a.dim; i += 256) wkr[3 * a.dim + i] = a.u[head * a.dim + i];
    for (int t = 0; t < n_rows; ++t) {
        const int64_t at = (int64_t)(row0 + t) * a.stride + head * a.dim;
        for (int i = tid; i < a.dim; i += 256) {
            const float z = act_ld(reinterpret_cast<const T*>(a.z) + (int64_t)(row0 + t) * a.z_stride + head * a.dim + i);
            wkr[i] = fast_exp2(log2_decay(z + a.w0[head * a.dim + i]));
            wkr[a.dim + i] = act_ld(reinterpret_cast<const T*>(a.k) + at + i);
            wkr[2 * a.dim + i] = act_ld(reinterpret_cast<const T*>(a.r) + at + i);
        }
        const float v = ok ? act_ld(reinterpret_cast<const T*>(a.v) + at + col) : 0.f;
        __syncthreads();
        float acc = 0.f;
        for (int r = rg; r < a.dim; r += 8) {
            const float s = S[r * 32 + c], kv = wkr[a.dim + r] * v;
            acc += (s + wkr[3 * a.dim + r] * kv) * wkr[2 * a.dim + r];
            S[r * 32 + c] = wkr[r] * s + kv;
        }
        red[rg * 32 + c] = acc;
        __syncthreads();
        if (rg == 0 && ok) {
            float s = 0.f;
#pragma unroll
            for (int k = 0; k < 8; ++k) s += red[k * 32 + c];
            act_st(reinterpret_cast<T*>(a.out) + (int64_t)(row0 + t) * a.out_stride + head * a.dim + col, s);
        }
    }
    if (pool && ok)
        for (int r = rg; r < a.dim; r += 8) pool[(int64_t)r * a.dim + col] = S[r * 32 + c];
}

// one wave per (row of a portion, head), in place
template <typename T>
__global__ __launch_bounds__(256) void wkv_norm_gate_kernel(const WkvArgs a) {
    const int first = blockIdx.x, lane = threadIdx.x & 63, head = blockIdx.y;
    const int row0 = a.chunks[4 * first], n_rows = a.chunks[4 * first + 1];
    for (int t = blockIdx.z * 4 + (threadIdx.x >> 6); t < n_rows; t += gridDim.z * 4) {
        T* o = reinterpret_cast<T*>(a.out) + (int64_t)(row0 + t) * a.out_stride + head * a.dim;
        const T* g = reinterpret_cast<const T*>(a.g) + (int64_t)(row0 + t) * a.stride + head * a.dim;
        float ss = 0.f;
        for (int c = lane; c < a.dim; c += 64) ss += act_ld(o + c) * act_ld(o + c);
        const float inv = 1.f / sqrtf(wave_sum64(ss) / a.n + a.eps);
        for (int c = lane; c < a.dim; c += 64) act_st(o + c, act_ld(o + c) * inv * a.norm[head * a.dim + c] * silu_f(act_ld(g + c)));
    }
}

// ------------------------------------------------------------------------------------------------ one token per sequence (bf16)
// grid (heads, rows); a thread holds 4 columns of DIM^2 / 1024 state rows; z: the low-rank row in front of its tanh
template <int DIM>
__global__ __launch_bounds__(256) void wkv_step_kernel(const WkvArgs a) {
    constexpr int LN = DIM / 4, RG = 256 / LN, NR = DIM / RG, TPC = 256 / DIM;
    extern __shared__ float low[];                   // [rank]
    __shared__ __attribute__((aligned(16))) float w_s[DIM], k_s[DIM], r_s[DIM], red[RG * DIM], part[4];
    const int head = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, c = (tid % LN) * 4, rg = tid / LN;
    const int64_t slot = a.state_slots[row];
    const bool carry = slot >= 0 && a.positions[row] > 0;
    float* pool = a.state + ((slot >= 0 ? slot : 0) * a.heads + head) * (int64_t)(DIM * DIM) + c;
    f32x4 s[NR];
#pragma unroll
    for (int u = 0; u < NR; ++u)                     // asked for before anything is computed
        s[u] = carry ? *reinterpret_cast<const f32x4*>(pool + (rg + u * RG) * DIM) : f32x4{0.f, 0.f, 0.f, 0.f};
    const int64_t at = (int64_t)row * a.stride + head * DIM;
    const uint16_t* z = reinterpret_cast<const uint16_t*>(a.z) + (int64_t)row * a.z_stride;
    for (int i = tid; i < a.rank; i += 256) low[i] = tanhf(act_ld(z + i));
    const f32x4 v = act_ld4(reinterpret_cast<const uint16_t*>(a.v) + at + c);
    float bonus = 0.f;
    if (tid < DIM) {
        const float k = act_ld(reinterpret_cast<const uint16_t*>(a.k) + at + tid), r = act_ld(reinterpret_cast<const uint16_t*>(a.r) + at + tid);
        k_s[tid] = k;
        r_s[tid] = r;
        bonus = r * a.u[head * DIM + tid] * k;
    }
    bonus = wave_sum64(bonus);
    if ((tid & 63) == 0) part[tid >> 6] = bonus;
    __syncthreads();
    {
        const int chn = tid / TPC, sub = tid % TPC;  // TPC neighbouring lanes share a channel's row of the up-projection
        const uint16_t* w2 = reinterpret_cast<const uint16_t*>(a.w2) + (int64_t)(head * DIM + chn) * a.rank;
        float acc = 0.f;
        for (int p = sub * 8; p < a.rank; p += TPC * 8) {
            const f32x8 w = act_ld8(w2 + p);
            acc += sum4(w.a * *reinterpret_cast<const f32x4*>(low + p)) + sum4(w.b * *reinterpret_cast<const f32x4*>(low + p + 4));
        }
        if constexpr (TPC >= 2) acc += pair_in_row<1>(acc);
        if constexpr (TPC >= 4) acc += pair_in_row<2>(acc);
        if (sub == 0) w_s[chn] = fast_exp2(log2_decay(acc + a.w0[head * DIM + chn]));
    }
    bonus = part[0] + part[1] + part[2] + part[3];
    __syncthreads();
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < NR; ++u) {
        const int r = rg + u * RG;
        acc += s[u] * r_s[r];
        if (slot >= 0) *reinterpret_cast<f32x4*>(pool + r * DIM) = s[u] * w_s[r] + v * k_s[r];
    }
    if (rg == 0) acc += v * bonus;
    *reinterpret_cast<f32x4*>(red + rg * DIM + c) = acc;
    __syncthreads();
    float o = 0.f;
    if (tid < DIM) {
#pragma unroll
        for (int k = 0; k < RG; ++k) o += red[k * DIM + tid];
    }
    const float ss = wave_sum64(o * o);              // (threads past DIM hold zeros)
    if ((tid & 63) == 0) part[tid >> 6] = ss;
    __syncthreads();
    if (tid < DIM) {
        const float inv = 1.f / sqrtf((part[0] + part[1] + part[2] + part[3]) / a.n + a.eps);
        const float y = o * inv * a.norm[head * DIM + tid] * silu_f(act_ld(reinterpret_cast<const uint16_t*>(a.g) + at + tid));
        if (a.out) act_st(reinterpret_cast<uint16_t*>(a.out) + (int64_t)row * a.out_stride + head * DIM + tid, y);
        if (a.out_packed) act_st(reinterpret_cast<uint16_t*>(a.out_packed) + pack_index(row, head * DIM + tid, a.heads * DIM), y);
    }
}

template <int DIM, typename Off>
int walk_off(const WkvArgs& a, hipStream_t stream) {
    constexpr size_t lds = sizeof(WkvLds<DIM>);
    for (const void* fn : {reinterpret_cast<const void*>(wkv_walk_kernel<DIM, true, Off>), reinterpret_cast<const void*>(wkv_walk_kernel<DIM, false, Off>)})
        if (lds > 64 * 1024) (void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    const dim3 grid(a.heads, a.n_chunks);
    if (a.summaries) {
        wkv_walk_kernel<DIM, true, Off><<<grid, DIM * 8, lds, stream>>>(a);
        int rc = check_launch("wkv summary");
        if (rc) return rc;
        const int64_t per = (int64_t)a.heads * DIM * DIM;
        wkv_starts_kernel<<<dim3((unsigned)((per + 1023) / 1024), a.n_chunks), 256, 0, stream>>>(a);
        rc = check_launch("wkv starts");
        if (rc) return rc;
    }
    wkv_walk_kernel<DIM, false, Off><<<grid, DIM * 8, lds, stream>>>(a);
    return check_launch("wkv walk");
}

template <int DIM>
int walk_dim(const WkvArgs& a, hipStream_t stream) {
    constexpr int64_t kNear = 1 << 25;               // row strides with which 63 rows and a piece stay below 2^32 bytes
    return a.stride < kNear && a.z_stride < kNear && a.out_stride < kNear ? walk_off<DIM, uint32_t>(a, stream) : walk_off<DIM, int64_t>(a, stream);
}

template <typename T>
int generic_t(const WkvArgs& a, hipStream_t stream) {
    const size_t lds = ((size_t)a.dim * 36 + 256) * 4;
    if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(wkv_generic_kernel<T>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    wkv_generic_kernel<T><<<dim3(a.n_chunks, a.heads, (a.dim + 31) / 32), 256, lds, stream>>>(a);
    const int rc = check_launch("wkv generic");
    if (rc) return rc;
    wkv_norm_gate_kernel<T><<<dim3(a.n_chunks, a.heads, 16), 256, 0, stream>>>(a);
    return check_launch("wkv norm");
}

bool wkv_supported(int dim) { return dim == 64 || dim == 128; }

int check_wkv(const char* fn, const nvh_wkv_desc* d, int dtype) {
    DTYPE(fn);
    REQUIRE(d->r && d->k && d->v && d->g && d->z && d->w0 && d->u && d->norm && d->positions && d->state_slots && d->state && (d->out || d->out_packed), NVH_E_NULL, "%s: null pointer", fn);
    REQUIRE(d->rows > 0 && d->heads > 0 && d->heads <= 65535 && d->dim > 0 && d->dim % 8 == 0 && d->dim <= 1024 && d->n > 0 && d->n <= d->dim, NVH_E_SHAPE, "%s: heads %d of %d (<= 1024)", fn,
            d->heads, d->dim);
    REQUIRE(d->stride % 8 == 0 && d->stride >= (int64_t)d->heads * d->dim && d->z_stride % 8 == 0 && (!d->out || (d->out_stride % 4 == 0 && d->out_stride >= (int64_t)d->heads * d->dim)),
            NVH_E_STRIDE, "%s: row strides", fn);
    REQUIRE(aligned16(d->r) && aligned16(d->k) && aligned16(d->v) && aligned16(d->g) && aligned16(d->z) && aligned16(d->w0) && aligned16(d->u) && aligned16(d->norm) && aligned16(d->state) &&
            aligned16(d->seg_state) && aligned16(d->seg_decay) && aligned16(d->out) && aligned16(d->out_packed), NVH_E_ALIGN, "%s: pointers must be 16-byte aligned", fn);
    return 0;
}

}  // namespace

}  // namespace nvh

using namespace nvh;

extern "C" {

int nvh_wkv_supported(int dim) { return wkv_supported(dim); }

int nvh_wkv_chunks(const nvh_wkv_desc* d, int generic, int dtype, void* stream) {
    REQUIRE(d, NVH_E_NULL, "wkv_chunks: null descriptor");
    if (d->n_chunks == 0) return 0;
    const int rc = check_wkv("wkv_chunks", d, dtype);
    if (rc) return rc;
    REQUIRE(d->chunks && d->n_chunks > 0 && d->n_chunks <= 65535 && d->out && d->z_stride >= (int64_t)d->heads * d->dim && (!d->summaries || (d->seg_state && d->seg_decay)), NVH_E_NULL,
            "wkv_chunks: %d segments or null pointer", d->n_chunks);
    if (dtype == NVH_F32) return generic_t<float>(*d, (hipStream_t)stream);
    if (generic || !wkv_supported(d->dim)) return generic_t<uint16_t>(*d, (hipStream_t)stream);
    return d->dim == 64 ? walk_dim<64>(*d, (hipStream_t)stream) : walk_dim<128>(*d, (hipStream_t)stream);
}

int nvh_wkv_step(const nvh_wkv_desc* d, int dtype, void* stream) {
    REQUIRE(d, NVH_E_NULL, "wkv_step: null descriptor");
    if (d->rows == 0) return 0;
    const int rc = check_wkv("wkv_step", d, dtype);
    if (rc) return rc;
    REQUIRE(dtype == NVH_BF16 && wkv_supported(d->dim) && d->rows <= 65535 && d->w2 && aligned16(d->w2) && d->rank > 0 && d->rank % 8 == 0 && d->rank <= 8192 && d->z_stride >= d->rank &&
            (!d->out_packed || (d->heads * d->dim) % 32 == 0), NVH_E_SHAPE, "wkv_step: bf16, heads of %d, rank %d (%%8)", d->dim, d->rank);
    const dim3 grid(d->heads, d->rows);
    const size_t lds = (size_t)d->rank * 4;
    if (d->dim == 64) wkv_step_kernel<64><<<grid, 256, lds, (hipStream_t)stream>>>(*d);
    else wkv_step_kernel<128><<<grid, 256, lds, (hipStream_t)stream>>>(*d);
    return check_launch("wkv_step");
}

}  // extern "C"
