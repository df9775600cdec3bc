// Lightning attention: per head a matrix state with a constant decay d,   S = d S + k v^T,   o = S^T q,   q, k, v = silu of the projection's columns.
//
// Prompt portions (launch_lightning_chunks): a workgroup owns one (segment, head, 64 or 128 value columns) and takes 64 tokens at a time,
//   o_i = d^(i+1) S^T q_i + sum_{j <= i} d^(i-j) (q_i . k_j) v_j          S <- d^n S + sum_j d^(n-1-j) k_j v_j^T
// on MFMA tiles.  The state stays in fp32 accumulators, laid out so that they are the left operand of S^T q without a shuffle; everything decays touch
// (weights, state, decayed values) enters the MFMA as bf16 hi + lo halves.  q, k and v go through registers on their way to LDS (silu, one rounding),
// the next step's rows are fetched while this one computes.
// A portion of several segments: a SUMMARY walk leaves every segment's own contribution, a small launch turns those into states at segment starts, and
// the second walk begins there.  State pools are read by the launch in front and written by the last segment: no workgroup sees a half-updated one.
// Decoding (launch_lightning_step): one workgroup per (sequence, head, value slice) streams the state once: read, decay, add, multiply, write.
// A sequence's first token (position 0) takes the state as zero instead of reading it: slots need no clearing when reused.
#include "attend_tile.h"
#include "mixers.h"

namespace nvh {

namespace {

constexpr int C = kLightningChunk, VS = 64;          // tokens per step; value columns of a workgroup of keys of 256
constexpr int PLD = C + 8;                           // row of the weights in LDS

__device__ __forceinline__ void split_hi_lo(const float (&v)[8], bf16x8& hi, bf16x8& lo) {
    u32x4 h, l;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        h[j] = pack_bf16x2_once(v[2 * j], v[2 * j + 1]);
        l[j] = pack_bf16x2(v[2 * j] - bf16_lo(h[j]), v[2 * j + 1] - bf16_hi(h[j]));
    }
    hi = *reinterpret_cast<const bf16x8*>(&h);
    lo = *reinterpret_cast<const bf16x8*>(&l);
}

// (a reciprocal, good to one unit of the last place in 32 bits, in place of a division: half the instructions, and the result is rounded to bf16)
__device__ __forceinline__ float silu_fast(float z) { return z * fast_rcp(1.f + fast_exp2(-kLog2e * z)); }
__device__ __forceinline__ u32x4 silu8(u32x4 r) {
#pragma unroll
    for (int k = 0; k < 4; ++k) r[k] = pack_bf16x2(silu_fast(bf16_lo(r[k])), silu_fast(bf16_hi(r[k])));
    return r;
}

// Keys of 256 (two images of each kind, as the walk below holds, would not fit the LDS, nor rows of a step ahead the registers)
constexpr int kWide = 256;
template <bool SUMMARY>
__global__ __launch_bounds__(256) void lightning_walk_kernel(const LightningArgs a) {
    constexpr int DK = kWide, KP = DK / 8, KROW = DK * 2, NQ = C * KP / 256, NV = C * (VS / 8) / 256, DT = DK / 16;
    constexpr int TB = 8;                            // key tiles read at a time
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char* kimg = smem;                                                // [C][DK] keys
    unsigned char* vimg = kimg + C * KROW;                                     // [C][VS] values
    unsigned char* qimg = vimg + C * VS * 2;                                   // [C][DK] queries
    uint16_t* p_lds = reinterpret_cast<uint16_t*>(qimg + C * KROW);            // [hi | lo][C][PLD] weights
    __shared__ float pw[C + 1];                                                // decay^0 .. decay^C
    auto swz = [](int r) { return r & 7; };
    auto swzv = [](int r) { return (r >> 1) & 7; };
    const int32_t* ch = a.chunks + 4 * blockIdx.x;
    const int row0 = ch[0], n_rows = ch[1], seq = ch[2];
    const int head = blockIdx.y, v0 = blockIdx.z * VS;
    const bool last = blockIdx.x + 1 == (unsigned)a.n_chunks || a.chunks[4 * (blockIdx.x + 1) + 3] == 0;
    if (SUMMARY && last) return;                     // (nothing follows it)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lq = lane & 15, lg = lane >> 4;
    const int64_t slot = a.state_slots[seq];
    const int64_t head_state = (int64_t)a.dk * a.dv;
    if (n_rows <= 0) {
        if (SUMMARY || (last && slot >= 0 && ch[3] > 0))
            pass_segment<SUMMARY>(a.seg_state + ((int64_t)blockIdx.x * a.heads + head) * head_state + v0, a.state + (slot * a.heads + head) * head_state + v0, DK, VS, a.dv);
        return;
    }
    if (tid <= C) pw[tid] = powf(a.decay[head], (float)tid);

    // state: value column v0 + 16 wave + lq, key rows 16 t + 4 lg + r
    f32x4 S[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) S[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int sv = v0 + 16 * wave + lq;
    if constexpr (!SUMMARY) {
        const float* src = nullptr;
        if (a.summaries) src = a.seg_state + ((int64_t)blockIdx.x * a.heads + head) * head_state;
        else if (slot >= 0 && a.positions[row0] > 0) src = a.state + (slot * a.heads + head) * head_state;
        if (src) {
#pragma unroll
            for (int t = 0; t < DT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) S[t][r] = src[(int64_t)(16 * t + 4 * lg + r) * a.dv + sv];
        }
    }
    const uint16_t* qkv = reinterpret_cast<const uint16_t*>(a.qkv);
    const int64_t k_off = (int64_t)a.heads * a.dk + head * DK, v_off = 2 * (int64_t)a.heads * a.dk + (int64_t)head * a.dv + v0, q_off = (int64_t)head * DK;
    u32x4 qr[NQ], kr[NQ], vr[NV];
    const u32x4 zero = {0u, 0u, 0u, 0u};
    auto fetch = [&](int t0) {                       // rows t0 .. of the segment; rows past its end are zero
#pragma unroll
        for (int j = 0; j < NQ; ++j) {
            const int e = j * 256 + tid, r = e / KP, c = (e - r * KP) * 8;
            const bool ok = t0 + r < n_rows;
            const uint16_t* p = qkv + (int64_t)(row0 + (ok ? t0 + r : 0)) * a.qkv_stride + c;
            kr[j] = ok ? *reinterpret_cast<const u32x4*>(p + k_off) : zero;
            if constexpr (!SUMMARY) qr[j] = ok ? *reinterpret_cast<const u32x4*>(p + q_off) : zero;
        }
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int e = j * 256 + tid, r = e >> 3, c = (e & 7) * 8;
            const bool ok = t0 + r < n_rows;
            vr[j] = ok ? *reinterpret_cast<const u32x4*>(qkv + (int64_t)(row0 + t0 + r) * a.qkv_stride + v_off + c) : zero;
        }
    };
    for (int t0 = 0; t0 < n_rows; t0 += C) {
        const int n = n_rows - t0 < C ? n_rows - t0 : C;
        fetch(t0);
        // (silu(0) = 0: rows past the end stay zero)
#pragma unroll
        for (int j = 0; j < NQ; ++j) {
            const int e = j * 256 + tid, r = e / KP, pc = e - r * KP;
            *reinterpret_cast<u32x4*>(kimg + r * KROW + (pc ^ swz(r)) * 16) = silu8(kr[j]);
            if constexpr (!SUMMARY) *reinterpret_cast<u32x4*>(qimg + r * KROW + (pc ^ swz(r)) * 16) = silu8(qr[j]);
        }
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int e = j * 256 + tid, r = e >> 3, pc = e & 7;
            *reinterpret_cast<u32x4*>(vimg + r * VS * 2 + (pc ^ swzv(r)) * 16) = silu8(vr[j]);
        }
        lds_only_barrier();
        const int tr = 4 * lg + (lq >> 2), tp = lq & 3;                        // transposed reads: row and column quarter this lane addresses
        f32x4 o[4];                                  // o^T: value 16 wave + 4 lg + r, token 16 it + lq
        if constexpr (!SUMMARY) {
            // weights of this wave's 16 queries: D[key 16 jt + 4 lg + r][query 16 wave + lq]
            f32x4 s[4];
#pragma unroll
            for (int jt = 0; jt < 4; ++jt) s[jt] = f32x4{0.f, 0.f, 0.f, 0.f};
            const int Rq = 16 * wave + lq;
#pragma unroll
            for (int st = 0; st < DK / 32; ++st) {
                const bf16x8 qf = *reinterpret_cast<const bf16x8*>(qimg + Rq * KROW + ((4 * st + lg) ^ swz(Rq)) * 16);
#pragma unroll
                for (int jt = 0; jt < 4; ++jt) {
                    if (jt > wave) continue;         // keys behind every query of this wave
                    const int Rk = 16 * jt + lq;
                    const bf16x8 kf = *reinterpret_cast<const bf16x8*>(kimg + Rk * KROW + ((4 * st + lg) ^ swz(Rk)) * 16);
                    s[jt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf, s[jt], 0, 0, 0);
                }
            }
#pragma unroll
            for (int jt = 0; jt < 4; ++jt) {
                float p[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int back = Rq - (16 * jt + 4 * lg + r);
                    p[r] = back >= 0 ? s[jt][r] * pw[back >= 0 ? back : 0] : 0.f;
                }
                const u32x2 hi = {pack_bf16x2_once(p[0], p[1]), pack_bf16x2_once(p[2], p[3])};
                const u32x2 lo = {pack_bf16x2(p[0] - bf16_lo(hi[0]), p[1] - bf16_hi(hi[0])), pack_bf16x2(p[2] - bf16_lo(hi[1]), p[3] - bf16_hi(hi[1]))};
                const int at = Rq * PLD + 32 * (jt >> 1) + 8 * lg + 4 * (jt & 1);
                *reinterpret_cast<u32x2*>(p_lds + at) = hi;
                *reinterpret_cast<u32x2*>(p_lds + C * PLD + at) = lo;
            }
            // what the state gives: slots of a 32-wide step are key rows 16 (2 st) + 4 lg + 0..3 and 16 (2 st + 1) + 4 lg + 0..3
#pragma unroll
            for (int it = 0; it < 4; ++it) o[it] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < DK / 32; ++st) {
                const float v[8] = {S[2 * st][0], S[2 * st][1], S[2 * st][2], S[2 * st][3], S[2 * st + 1][0], S[2 * st + 1][1], S[2 * st + 1][2], S[2 * st + 1][3]};
                bf16x8 hi, lo;
                split_hi_lo(v, hi, lo);
#pragma unroll
                for (int it = 0; it < 4; ++it) {
                    const int R = 16 * it + lq;
                    const unsigned char* qrow = qimg + R * KROW + (lg & 1) * 8;
                    const u32x2 qa = *reinterpret_cast<const u32x2*>(qrow + ((4 * st + (lg >> 1)) ^ swz(R)) * 16);
                    const u32x2 qb = *reinterpret_cast<const u32x2*>(qrow + ((4 * st + 2 + (lg >> 1)) ^ swz(R)) * 16);
                    const u32x4 raw = {qa[0], qa[1], qb[0], qb[1]};
                    const bf16x8 qf = *reinterpret_cast<const bf16x8*>(&raw);
                    o[it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, qf, o[it], 0, 0, 0);
                    o[it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, qf, o[it], 0, 0, 0);
                }
            }
#pragma unroll
            for (int it = 0; it < 4; ++it) o[it] *= pw[16 * it + lq + 1];
            lds_only_barrier();                      // all weights are in LDS
        }
        // value fragments: lane = column 16 wave + lq, slots = keys 32 hh + 4 lg + 0..3 and the same + 16
        u32x2 vlo[2], vhi[2];
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            const int ra = 32 * hh + tr, rb = ra + 16, pc = 2 * wave + (tp >> 1);
            vlo[hh] = ds_read_tr16<0>(lds_addr_of(vimg + ra * VS * 2 + (pc ^ swzv(ra)) * 16 + (tp & 1) * 8));
            vhi[hh] = ds_read_tr16<0>(lds_addr_of(vimg + rb * VS * 2 + (pc ^ swzv(rb)) * 16 + (tp & 1) * 8));
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        bf16x8 vf[2];
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            const u32x4 raw = {vlo[hh][0], vlo[hh][1], vhi[hh][0], vhi[hh][1]};
            vf[hh] = *reinterpret_cast<const bf16x8*>(&raw);
        }
        if constexpr (!SUMMARY) {
#pragma unroll
            for (int it = 0; it < 4; ++it)
#pragma unroll
                for (int hh = 0; hh < 2; ++hh) {
                    if (32 * hh > 16 * it + 15) continue;
                    const uint16_t* pr = p_lds + (16 * it + lq) * PLD + 32 * hh + 8 * lg;
                    o[it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[hh], *reinterpret_cast<const bf16x8*>(pr), o[it], 0, 0, 0);
                    o[it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[hh], *reinterpret_cast<const bf16x8*>(pr + C * PLD), o[it], 0, 0, 0);
                }
#pragma unroll
            for (int it = 0; it < 4; ++it) {
                const int t = t0 + 16 * it + lq;
                if (t < n_rows) act_st4(reinterpret_cast<uint16_t*>(a.out) + (int64_t)(row0 + t) * a.out_stride + (int64_t)head * a.dv + v0 + 16 * wave + 4 * lg, o[it]);
            }
        }
        // ---- the state behind these tokens
#pragma unroll
        for (int t = 0; t < DT; ++t) S[t] *= pw[n];
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            const u32x4 raw = *reinterpret_cast<const u32x4*>(&vf[hh]);
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int key = 32 * hh + (j < 4 ? 0 : 16) + 4 * lg + (j & 3);
                v[j] = (j & 1 ? bf16_hi(raw[j >> 1]) : bf16_lo(raw[j >> 1])) * pw[key < n ? n - 1 - key : 0];
            }
            bf16x8 hi, lo;
            split_hi_lo(v, hi, lo);
            const int ra = 32 * hh + tr, rb = ra + 16;
#pragma unroll
            for (int tb = 0; tb < DT; tb += TB) {
                u32x2 klo[TB], khi[TB];
#pragma unroll
                for (int t = 0; t < TB; ++t) {
                    const int pc = 2 * (tb + t) + (tp >> 1);
                    klo[t] = ds_read_tr16<0>(lds_addr_of(kimg + ra * KROW + (pc ^ swz(ra)) * 16 + (tp & 1) * 8));
                    khi[t] = ds_read_tr16<0>(lds_addr_of(kimg + rb * KROW + (pc ^ swz(rb)) * 16 + (tp & 1) * 8));
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < TB; ++t) {
                    const u32x4 kraw = {klo[t][0], klo[t][1], khi[t][0], khi[t][1]};
                    const bf16x8 kf = *reinterpret_cast<const bf16x8*>(&kraw);
                    S[tb + t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, hi, S[tb + t], 0, 0, 0);
                    S[tb + t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, lo, S[tb + t], 0, 0, 0);
                }
            }
        }
        lds_only_barrier();                          // everyone is done with the images
    }
    float* dst = nullptr;
    if constexpr (SUMMARY) dst = a.seg_state + ((int64_t)blockIdx.x * a.heads + head) * head_state;
    else if (last && slot >= 0) dst = a.state + (slot * a.heads + head) * head_state;
    if (dst) {
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) dst[(int64_t)(16 * t + 4 * lg + r) * a.dv + sv] = S[t][r];
    }
}

// ------------------------------------------------------------------------------------------------ the same walk with two kinds of waves
// Four waves prepare: rows of the next chunk from registers through silu into the images, its weights.  The others, four or eight, consume: 16 value columns each,
// state and outputs of this chunk.  Two halves a chunk, one barrier behind each:
//   consume: o(i) = S^T q + weights v                | S(i) behind the chunk
//   prepare: q, k of chunk i + 1 into its images     | weights of chunk i + 1, its values
// Images are double (chunk parity), the weights are written in the half in which nobody reads them; rows are asked for a whole chunk before they are prepared.
// What bounds it is issue (a wave alone issues a vector instruction every 5.5 cycles, three together every 2.7) and, with all CUs busy, the rows that all ask for at
// once; so a workgroup has three waves per SIMD and takes 16 CW columns, 128 where they come in such numbers: queries and keys are prepared once for all of them,
// not for every 64.  A chunk takes 3.8 us alone and 5.0 on all CUs, 9.1 for two workgroups of the 64-column walk; 16 prompts of 1024 tokens on average, 16 heads of
// 128: 251 -> 108 us; 40 prompts of 410: 302 -> 157.  Results leave by whole rows, through LDS, and the queries' reads are kept apart: 104.4 -> 99.6
// there.  Measured and not better: eight waves with 32 columns each (121), sixteen waves (114), fragments read a step
// ahead by hand (121).
template <int DK, int CW>
constexpr size_t pair_lds_bytes(bool summary) {
    return (size_t)2 * C * (DK * (summary ? 1 : 2) + 16 * CW) * 2 + (summary ? 0 : (size_t)2 * C * PLD * 2 + (size_t)C * (16 * CW + 8) * 2);
}

// Whole portions that nothing comes in front of: the longest of them as two pieces of the same length in time.  The second one follows the state over the first one's tokens (keys and
// values only: kFollow of a chunk) and goes on from there with outputs: the same operations on the same numbers, no summary and no launch in front.  Both would read a state that the
// second one replaces: portions behind a state stay whole, and with them all of the launch.
// A workgroup a CU walks at its own pace, so the longest portion sets the time, 1.6 to 1.75 of the mean.  As many pieces are made as bring the longest one (a chunk to start, and those that
// it takes), the even load (times kUneven, what the order by length leaves on it) and the pairs below down together.
// A workgroup begins with a portion of its own, whole, while its first wave weighs the lengths, and learns behind the first chunk's images where to stop.  Second pieces go to workgroups
// without a portion where CUs are left, and in place of the shortest portions where not; those then go behind the next shortest ones, in the same workgroup.  (Chosen first, with a workgroup
// for every piece that there might be: 2.2 us in front of each, and 1 to 2 at the end of the launch for those that had none; lengths much alike 0.93 to 0.96 of the speed of whole portions,
// 31 portions of 8 heads 0.88.)
// Eight sets of lengths each, 16 heads of 128, against whole portions: 16384 tokens of 16 1.21 times as fast (128 -> 106 us), 9000 of 14 1.16, 12000 of 19 1.11; 8 heads, 14000 of 28 1.17.
// Lengths of 0.9 to 1.1 of their mean, which are not cut, and launches with a portion behind a state: 0.99 (0.9 us, half of it the choice).
constexpr int kSplitPortions = 32;
constexpr float kFollow = 0.5f, kUneven = 1.2f, kLate = 0.6f;                  // (a second piece starts behind the choice)
// of the portions that run at once, those cut at most (11)
__host__ __device__ __forceinline__ int lightning_most_cut(int places) { return places * 5 / 16; }
struct LightningWalk {
    int seg, from, to, next;                         // portion (-1: none), tokens followed, end in tokens; the portion behind it (-1: none)
    int row0, rows;                                  // of the portion
};
__device__ __forceinline__ float lane_value(float v, int lane) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane)); }
// sums of lanes 0 .. l in lanes l < 32
__device__ __forceinline__ float sum_to_here32(float v) {
    v += dpp_f32<0x111>(v);                          // row_shr:1, 2, 4, 8
    v += dpp_f32<0x112>(v);
    v += dpp_f32<0x114>(v);
    v += dpp_f32<0x118>(v);
    return v + (threadIdx.x & 16 ? lane_value(v, 15) : 0.f);
}
// (a wave) What workgroup y of a head walks; it has begun with portion `own`, the y-th longest where they are more than run at once.
__device__ __forceinline__ LightningWalk lightning_walk_of(const LightningArgs& a, int walks_each, int y, int own) {
    const int lane = threadIdx.x & 63, i = lane & 31, n = a.n_chunks, places = 256 / walks_each;
    const int32_t* ch = a.chunks + 4 * (i < n ? i : 0);
    const int first_row = ch[0], listed = ch[1], rows = i < n && listed > 0 ? listed : 0;
    const int64_t position = a.positions[rows ? first_row : 0];                // (looked at last)
    const int steps = (rows + 15) >> 4, key = (steps < 1023 ? steps : 1023) * 32 + 31 - i;      // as longest_first orders them
    int rank = 0;
#pragma unroll
    for (int k = 0; k < 32; ++k) rank += __builtin_amdgcn_readlane(key, k) > key ? 1 : 0;
    // lanes p and 32 + p: the p-th longest
    const int lane_of = 4 * (rank + (lane & 32)), seg = __builtin_amdgcn_ds_permute(lane_of, i), mine = __builtin_amdgcn_ds_permute(lane_of, (rows + C - 1) / C);
    int cut = (int)((mine + kLate) * (1.f / (2.f - kFollow)));
    if (mine + kLate - (1.f - kFollow) * cut > cut + 1.f) ++cut;               // (the piece that is longer then is shorter)
    const float first = cut + 1.f, second = kFollow * cut + (mine - cut) + 1.f + kLate, whole = mine + 1.f;
    // lane p: the longest p as two pieces (lengths fall with the lane, and with them whole and halves)
    const bool real = lane < 32 && lane < n;
    const float one = real ? first + second - whole : 0.f, added = sum_to_here32(one), all = lane_value(sum_to_here32(real ? whole : 0.f), 31);
    const float top = lane_value(fmaxf(first, second), 0);
    const float rest = real ? whole : 0.f, longest = lane ? fmaxf(top, rest) : rest;
    const int could = __builtin_popcountll(__builtin_amdgcn_ballot_w64(lane < 32 && mine >= 4)), most = could < lightning_most_cut(places) ? could : lightning_most_cut(places);
    const float even = (all + added - one) * kUneven / places;
    // more pieces than CUs for them: of the places, ranks up to places - lane - 1 have a portion of their own, and the longest of the others goes behind the last of those
    const auto portion = [&](int p) { return __uint_as_float(__builtin_amdgcn_ds_bpermute(4 * p, __float_as_uint(whole))); };
    const float pair = portion(places - lane) + portion(places - lane - 1);
    const int over = n + lane - places;              // portions that go behind others
    float cost = longest;
    if (over > 0) cost = fmaxf(fmaxf(longest, even), lane ? pair : 0.f);
    if (lane > most || (lane && over > 0 && n - 2 * over < lane)) cost = INFINITY;       // (none goes behind a piece)
    if (lane) cost = cost * (1.f / 0.97f);           // (not for little)
    float least = cost;                              // (of the first row of lanes: fewer are cut)
    least = fminf(least, dpp_f32<0x128>(least));     // row_ror:8, 4, 2, 1
    least = fminf(least, dpp_f32<0x124>(least));
    least = fminf(least, dpp_f32<0x122>(least));
    least = lane_value(fminf(least, dpp_f32<0x121>(least)), 0);
    const int split = __builtin_ctzll(__builtin_amdgcn_ballot_w64(cost == least));
    const int behind = n + split > places ? n + split - places : 0, holders = n - behind;     // portions behind others; workgroups with one of their own
    // (the other pairs: lane p, the p-th longest that goes behind)
    const float uncut = lane_value(cost, 0), pairs = portion(holders + lane) + portion(holders - 1 - lane);
    const bool worse = lane < behind && pairs > uncut;
    const LightningWalk as_begun{own, 0, 0x7FFFFFFF, -1, 0, 0};
    if (!split || __builtin_amdgcn_ballot_w64(worse || position > 0)) return as_begun;
    LightningWalk to{-1, 0, 0x7FFFFFFF, -1, 0, 0};
    const int r = y >= n ? 0 : n <= places ? __builtin_amdgcn_readlane(rank, y) : y;
    if (y < n && r < holders) {
        to.seg = __builtin_amdgcn_readlane(seg, r);
        if (r < split) to.to = C * __builtin_amdgcn_readlane(cut, r);
        if (holders - 1 - r < behind) to.next = __builtin_amdgcn_readlane(seg, 2 * holders - 1 - r);
    } else {
        const int piece = y < n ? r - holders : behind + y - n;
        if (piece < split) {
            to.seg = __builtin_amdgcn_readlane(seg, piece), to.from = C * __builtin_amdgcn_readlane(cut, piece);
            to.row0 = __builtin_amdgcn_readlane(first_row, to.seg), to.rows = __builtin_amdgcn_readlane(rows, to.seg);
        }
    }
    return to;
}

template <int DK, int CW, int PW, bool SUMMARY, bool PIECES>
__global__ __launch_bounds__(64 * (CW + PW), DK == 64 && CW == 4 ? 4 : 1) void lightning_pair_kernel(const LightningArgs a) {
    constexpr int T = 64 * PW, VW = 16 * CW, KP = DK / 8, KROW = DK * 2, VP = VW / 8, VROW = VW * 2, NQ = C * KP / T, NV = C * VP / T, DT = DK / 16, PT = PW / 4;
    constexpr int KIMG = C * KROW, VIMG = C * VROW;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char* kimg0 = smem;                                               // [2][C][DK] keys
    unsigned char* vimg0 = kimg0 + 2 * KIMG;                                   // [2][C][VW] values
    unsigned char* qimg0 = vimg0 + 2 * VIMG;                                   // [2][C][DK] queries
    uint16_t* p_lds = reinterpret_cast<uint16_t*>(qimg0 + 2 * KIMG);           // [hi | lo][C][PLD] weights
    constexpr int OLD = VW + 8;
    uint16_t* o_lds = p_lds + 2 * C * PLD;                                     // [C][OLD] outputs, on their way from columns of 16 tokens to rows
    __shared__ __attribute__((aligned(16))) float pw[C + 1], fall_s[C];        // decay^0 .. decay^C; decay^(C - 1 - key)
    auto swz = [](int r) { return KROW == 128 ? (r >> 1) & 7 : r & 15; };      // rows of 256 bytes span all banks: 16 of them apart, not 8
    auto swzv = [](int r) { return VROW == 128 ? (r >> 1) & 7 : (2 * r) & 14; };
    __shared__ int walk_s[6];
    const int slices = a.dv / VW, head = blockIdx.x / slices, v0 = (blockIdx.x - head * slices) * VW;
    // portion, tokens that are only followed, the portion behind it (PIECES: known behind the first barrier; none is begun with where workgroups are more than portions)
    int seg = PIECES && (int)blockIdx.y >= a.n_chunks ? -1 : longest_first(a, a.heads * slices), from = 0, next_seg = -1;
    int row0 = 0, n_rows = 0;
    int64_t slot = -1;
    bool last = true, known = !PIECES;
    auto open = [&]() __attribute__((always_inline)) {                         // the portion `seg`, whole
        const int32_t* ch = a.chunks + 4 * seg;
        row0 = ch[0], n_rows = ch[1], slot = a.state_slots[ch[2]];
        last = seg + 1 == a.n_chunks || a.chunks[4 * (seg + 1) + 3] == 0;
    };
    if (seg >= 0) open();
    if (SUMMARY && last) return;                     // (nothing follows it)
    int lane = threadIdx.x & 63, lq = lane & 15, lg = lane >> 4;
    const int wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool prepares = wave_id >= CW;
    const int wave = prepares ? wave_id - CW : wave_id;
    const int64_t head_state = (int64_t)a.dk * a.dv;
    if constexpr (!PIECES) {
        if (n_rows <= 0) {
            if (SUMMARY || (last && slot >= 0 && a.chunks[4 * seg + 3] > 0))
                pass_segment<SUMMARY>(a.seg_state + ((int64_t)seg * a.heads + head) * head_state + v0, a.state + (slot * a.heads + head) * head_state + v0, DK, VW, a.dv);
            return;
        }
        if (threadIdx.x <= C) {
            const float p = powf(a.decay[head], (float)threadIdx.x);
            pw[threadIdx.x] = p;
            if (threadIdx.x < C) fall_s[C - 1 - threadIdx.x] = p;
        }
        __syncthreads();
    }
    // PIECES: what was chosen (behind the first barrier): whether that is another portion than the one begun with
    auto look = [&]() __attribute__((always_inline)) {
        const int at = __builtin_amdgcn_readfirstlane(walk_s[0]), to = __builtin_amdgcn_readfirstlane(walk_s[2]);
        from = __builtin_amdgcn_readfirstlane(walk_s[1]), next_seg = __builtin_amdgcn_readfirstlane(walk_s[3]);
        const bool other = at != seg;
        seg = at;
        if (to < n_rows) n_rows = to, last = false;
        if (other) {                                 // (none, or a second piece)
            row0 = __builtin_amdgcn_readfirstlane(walk_s[4]), n_rows = __builtin_amdgcn_readfirstlane(walk_s[5]), last = true;
            if (seg >= 0) slot = a.state_slots[a.chunks[4 * seg + 2]];
        }
        return other;
    };
    auto take_next = [&]() __attribute__((always_inline)) {
        if (!PIECES || next_seg < 0) return false;
        seg = next_seg, next_seg = -1, from = 0;
        open();
        return true;
    };

    if (prepares) {
        int tid = threadIdx.x - 64 * CW;
        const uint16_t* qkv = reinterpret_cast<const uint16_t*>(a.qkv);
        const int64_t k_off = (int64_t)a.heads * a.dk + head * DK, v_off = 2 * (int64_t)a.heads * a.dk + (int64_t)head * a.dv + v0, q_off = (int64_t)head * DK;
        u32x4 qr[NQ], kr[NQ], vr[NV];
        const u32x4 zero = {0u, 0u, 0u, 0u};
        // Bytes from a chunk's first row: one scalar base per chunk, no address arithmetic in the lanes.  (64 bits: rows may be any distance apart.  32 bits
        // would save half a percent: one sequence of 1536 tokens 95.7 us against 96.3, 16 of them 129 against 131, which is not worth a second form)
        int64_t at[NQ], atv[NV];
        const int64_t row_bytes = a.qkv_stride * 2;
        auto place = [&](int rows) __attribute__((always_inline)) {            // rows past the portion's end read its last one
#pragma unroll
            for (int j = 0; j < NQ; ++j) {
                const int e = j * T + tid, r = e / KP;
                at[j] = (r < rows ? r : rows - 1) * row_bytes + (e - r * KP) * 16;
            }
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                const int e = j * T + tid, r = e / VP;
                atv[j] = (r < rows ? r : rows - 1) * row_bytes + (e - r * VP) * 16;
            }
        };
        auto base_of = [&](int t0) __attribute__((always_inline)) { return reinterpret_cast<const unsigned char*>(qkv + (int64_t)(row0 + t0) * a.qkv_stride); };
        // (every chunk asks for as many rows as any other, in straight line, the last one's again behind the end: behind a branch around loads the compiler waits
        // for all that are in flight instead of the ones it needs)
        int t_last = 0;
        constexpr std::bool_constant<!SUMMARY> with_q{};
        constexpr std::bool_constant<false> no_q{};
        auto fetch_qk = [&](int t, auto q) __attribute__((always_inline)) {
            const int t0 = t < t_last ? t : t_last;
            if (n_rows - t0 < C) place(n_rows - t0);
            const unsigned char* base = base_of(t0);
#pragma unroll
            for (int j = 0; j < NQ; ++j) {
                kr[j] = *reinterpret_cast<const u32x4*>(base + 2 * k_off + at[j]);
                if constexpr (decltype(q)::value) qr[j] = *reinterpret_cast<const u32x4*>(base + 2 * q_off + at[j]);
            }
        };
        auto fetch_v = [&](int t) __attribute__((always_inline)) {
            const unsigned char* base = base_of(t < t_last ? t : t_last);
#pragma unroll
            for (int j = 0; j < NV; ++j) vr[j] = *reinterpret_cast<const u32x4*>(base + 2 * v_off + atv[j]);
        };
        auto stage_qk = [&](int t0, int buf, auto q) __attribute__((always_inline)) {    // rows past the end are zero (as is silu of them)
            const int n = n_rows - t0;
            if (n < C) {
#pragma unroll
                for (int j = 0; j < NQ; ++j)
                    if ((j * T + tid) / KP >= n) {
                        kr[j] = zero;
                        if constexpr (decltype(q)::value) qr[j] = zero;
                    }
            }
#pragma unroll
            for (int j = 0; j < NQ; ++j) {
                const int e = j * T + tid, r = e / KP, pc = e - r * KP;
                *reinterpret_cast<u32x4*>(kimg0 + buf * KIMG + r * KROW + (pc ^ swz(r)) * 16) = silu8(kr[j]);
                if constexpr (decltype(q)::value) *reinterpret_cast<u32x4*>(qimg0 + buf * KIMG + r * KROW + (pc ^ swz(r)) * 16) = silu8(qr[j]);
            }
        };
        auto stage_v = [&](int t0, int buf) __attribute__((always_inline)) {
            const int n = n_rows - t0;
            if (n < C) {
#pragma unroll
                for (int j = 0; j < NV; ++j)
                    if ((j * T + tid) / VP >= n) vr[j] = zero;
            }
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                const int e = j * T + tid, r = e / VP, pc = e - r * VP;
                *reinterpret_cast<u32x4*>(vimg0 + buf * VIMG + r * VROW + (pc ^ swzv(r)) * 16) = silu8(vr[j]);
            }
        };
        // weights D[key 16 jt + 4 lg + r][query 16 tile + lq]: PT waves share a tile of queries, every PT-th tile of keys each; keys behind all queries stay zero
        const int tile = wave / PT;
        int Rq = 16 * tile + lq;
        constexpr int KT = 4 / PT;                   // key tiles a wave may have
        float fall[KT][4];
        auto falls = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < KT; ++i) {
                const int jt = PT * i + wave % PT;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int back = Rq - (16 * jt + 4 * lg + r);
                    fall[i][r] = pw[back >= 0 ? back : 0];
                }
                const int to = Rq * PLD + 32 * (jt >> 1) + 8 * lg + 4 * (jt & 1);
                if (jt > tile) *reinterpret_cast<u32x2*>(p_lds + to) = *reinterpret_cast<u32x2*>(p_lds + C * PLD + to) = u32x2{0u, 0u};
            }
        };
        if constexpr (!SUMMARY && !PIECES) falls();
        auto weights_of = [&](auto nc, int buf) __attribute__((always_inline)) {       // nc key tiles; only the last can be the queries' own
            constexpr int N = decltype(nc)::value;
            const unsigned char *kimg = kimg0 + buf * KIMG, *qimg = qimg0 + buf * KIMG;
            f32x4 s[N];
#pragma unroll
            for (int i = 0; i < N; ++i) s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < DK / 32; ++st) {
                const bf16x8 qf = *reinterpret_cast<const bf16x8*>(qimg + Rq * KROW + ((4 * st + lg) ^ swz(Rq)) * 16);
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    const int Rk = 16 * (PT * i + wave % PT) + lq;
                    const bf16x8 kf = *reinterpret_cast<const bf16x8*>(kimg + Rk * KROW + ((4 * st + lg) ^ swz(Rk)) * 16);
                    s[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf, s[i], 0, 0, 0);
                }
            }
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const int jt = PT * i + wave % PT;
                float p[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    p[r] = s[i][r] * fall[i][r];
                    if (i == N - 1 && 16 * jt + 4 * lg + r > Rq) p[r] = 0.f;
                }
                const u32x2 hi = {pack_bf16x2_once(p[0], p[1]), pack_bf16x2_once(p[2], p[3])};
                const u32x2 lo = {pack_bf16x2(p[0] - bf16_lo(hi[0]), p[1] - bf16_hi(hi[0])), pack_bf16x2(p[2] - bf16_lo(hi[1]), p[3] - bf16_hi(hi[1]))};
                const int to = Rq * PLD + 32 * (jt >> 1) + 8 * lg + 4 * (jt & 1);
                *reinterpret_cast<u32x2*>(p_lds + to) = hi;
                *reinterpret_cast<u32x2*>(p_lds + C * PLD + to) = lo;
            }
        };
        const int mine = (tile - wave % PT + PT) / PT;       // key tiles wave % PT, + PT, .. up to `tile`
        auto weights = [&](int buf) __attribute__((always_inline)) {
            if constexpr (!SUMMARY) {
                if (mine == 1) weights_of(std::integral_constant<int, 1>{}, buf);
                else if (mine == 2) weights_of(std::integral_constant<int, 2>{}, buf);
                if constexpr (PT == 1) {
                    if (mine == 3) weights_of(std::integral_constant<int, 3>{}, buf);
                    else if (mine == 4) weights_of(std::integral_constant<int, 4>{}, buf);
                }
            }
        };
        for (;;) {
            if constexpr (PIECES) lane = lane_now() & 63, tid = (64 * wave + lane) & (T - 1), lq = lane & 15, lg = lane >> 4, Rq = 16 * tile + lq;
            if (!PIECES || n_rows > 0) {
                t_last = (n_rows - 1) / C * C;
                place(C);
                fetch_qk(0, with_q);
                fetch_v(0);
                stage_qk(0, 0, with_q);
                fetch_qk(C, with_q);
                stage_v(0, 0);
                fetch_v(C);
            }
            if (!known || n_rows > 0) lds_only_barrier();
            if (!known) {
                known = true;
                if (look()) continue;
                t_last = (n_rows - 1) / C * C;
            }
            if (!PIECES || n_rows > 0) {
                int t0 = 0, buf = 0;
                if constexpr (PIECES) falls();
                if (PIECES && from) {                // (at least three chunks)
                    lds_only_barrier();
                    auto follow = [&](auto q) __attribute__((always_inline)) {
                        stage_qk(t0 + C, buf ^ 1, no_q);
                        fetch_qk(t0 + 2 * C, q);
                        lds_only_barrier();
                        stage_v(t0 + C, buf ^ 1);
                        fetch_v(t0 + 2 * C);
                        lds_only_barrier();
                        t0 += C;
                        buf ^= 1;
                    };
                    while (t0 < from - 2 * C) follow(no_q);
                    follow(with_q);                  // (asks for the first chunk that has outputs)
                } else {
                    weights(0);
                    lds_only_barrier();
                }
                for (; t0 < n_rows; t0 += C, buf ^= 1) {
                    const bool next = t0 + C < n_rows;
                    if (next) stage_qk(t0 + C, buf ^ 1, with_q);
                    fetch_qk(t0 + 2 * C, with_q);
                    lds_only_barrier();
                    if (next) {
                        weights(buf ^ 1);
                        stage_v(t0 + C, buf ^ 1);
                    }
                    fetch_v(t0 + 2 * C);
                    lds_only_barrier();
                }
            }
            if (!take_next()) return;
        }
    }

    // state: value column v0 + 16 wave + lq, key rows 16 t + 4 lg + r
    f32x4 S[DT];
    int sv = v0 + 16 * wave + lq;
    int tr = 4 * lg + (lq >> 2), tp = lq & 3;        // transposed reads: row and column quarter this lane addresses
    // what a followed chunk does to the state: the second half of the loop below.  (Shared with it as a function, that loop loses 1 % of its speed)
    auto values = [&](bf16x8 (&vf)[2], const unsigned char* vimg) __attribute__((always_inline)) {
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            const int ra = 32 * hh + tr, rb = ra + 16, pc = 2 * wave + (tp >> 1);
            const u32x2 lo = lds_tr16(vimg + ra * VROW + (pc ^ swzv(ra)) * 16 + (tp & 1) * 8), hi = lds_tr16(vimg + rb * VROW + (pc ^ swzv(rb)) * 16 + (tp & 1) * 8);
            const u32x4 raw = {lo[0], lo[1], hi[0], hi[1]};
            vf[hh] = *reinterpret_cast<const bf16x8*>(&raw);
        }
    };
    auto advance = [&](const bf16x8 (&vf)[2], int n, const unsigned char* kimg) __attribute__((always_inline)) {
        // ---- the state behind these tokens
        const float decayed = pw[n];
#pragma unroll
        for (int t = 0; t < DT; ++t) S[t] *= decayed;
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            const u32x4 raw = *reinterpret_cast<const u32x4*>(&vf[hh]);
            f32x4 fall[2];                           // what a value decays by until the chunk's end
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int key = 32 * hh + 16 * q + 4 * lg;
                if (n == C) {
                    fall[q] = *reinterpret_cast<const f32x4*>(fall_s + key);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) fall[q][r] = pw[key + r < n ? n - 1 - key - r : 0];
                }
            }
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = (j & 1 ? bf16_hi(raw[j >> 1]) : bf16_lo(raw[j >> 1])) * fall[j >> 2][j & 3];
            bf16x8 hi, lo;
            split_hi_lo(v, hi, lo);
            const int ra = 32 * hh + tr, rb = ra + 16;
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                const int pc = 2 * t + (tp >> 1);
                const u32x2 klo = lds_tr16(kimg + ra * KROW + (pc ^ swz(ra)) * 16 + (tp & 1) * 8), khi = lds_tr16(kimg + rb * KROW + (pc ^ swz(rb)) * 16 + (tp & 1) * 8);
                const u32x4 kraw = {klo[0], klo[1], khi[0], khi[1]};
                const bf16x8 kf = *reinterpret_cast<const bf16x8*>(&kraw);
                S[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, hi, S[t], 0, 0, 0);
                S[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, lo, S[t], 0, 0, 0);
            }
        }
    };
    for (;;) {
        // (what hangs on the lane is computed for each portion: held over them it would not fit the registers; the mask tells the compiler that lanes are 64)
        if constexpr (PIECES) lane = lane_now() & 63, lq = lane & 15, lg = lane >> 4, sv = v0 + 16 * wave + lq, tr = 4 * lg + (lq >> 2), tp = lq & 3;
        if (!known && wave_id == 0) {                // (before the state is asked for: loads are waited for in their order)
            const LightningWalk w = lightning_walk_of(a, a.heads * slices, blockIdx.y, seg);
            if (lane == 0) walk_s[0] = w.seg, walk_s[1] = w.from, walk_s[2] = w.to, walk_s[3] = w.next, walk_s[4] = w.row0, walk_s[5] = w.rows;
        }
#pragma unroll
        for (int t = 0; t < DT; ++t) S[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (!SUMMARY) {
            const float* src = nullptr;
            if (a.summaries) src = a.seg_state + ((int64_t)seg * a.heads + head) * head_state;
            else if (slot >= 0 && (!PIECES || (known ? false : n_rows > 0)) && a.positions[row0] > 0) src = a.state + (slot * a.heads + head) * head_state;
            if (src) {
#pragma unroll
                for (int t = 0; t < DT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) S[t][r] = src[(int64_t)(16 * t + 4 * lg + r) * a.dv + sv];
            }
        }
        if (!known && wave_id != 0) {
            const int t = 64 * wave_id - 64 + lane;
            if (t <= C) {
                const float p = powf(a.decay[head], (float)t);
                pw[t] = p;
                if (t < C) fall_s[C - 1 - t] = p;
            }
        }
        if (!known || n_rows > 0) lds_only_barrier();
        if (!known) {
            known = true;
            if (look()) continue;
        }
        if (!PIECES || n_rows > 0) {
            lds_only_barrier();
            int t0 = 0, buf = 0;
            if constexpr (PIECES) {
                for (; t0 < from; t0 += C, buf ^= 1) {
                    bf16x8 vf[2];
                    values(vf, vimg0 + buf * VIMG);
                    lds_only_barrier();
                    advance(vf, C, kimg0 + buf * KIMG);
                    lds_only_barrier();
                }
            }
            for (; t0 < n_rows; t0 += C, buf ^= 1) {
                const int n = n_rows - t0 < C ? n_rows - t0 : C;
                const unsigned char *kimg = kimg0 + buf * KIMG, *qimg = qimg0 + buf * KIMG, *vimg = vimg0 + buf * VIMG;
                // value fragments: lane = column 16 wave + lq, slots = keys 32 hh + 4 lg + 0..3 and the same + 16
                bf16x8 vf[2];
#pragma unroll
                for (int hh = 0; hh < 2; ++hh) {
                    const int ra = 32 * hh + tr, rb = ra + 16, pc = 2 * wave + (tp >> 1);
                    const u32x2 lo = lds_tr16(vimg + ra * VROW + (pc ^ swzv(ra)) * 16 + (tp & 1) * 8), hi = lds_tr16(vimg + rb * VROW + (pc ^ swzv(rb)) * 16 + (tp & 1) * 8);
                    const u32x4 raw = {lo[0], lo[1], hi[0], hi[1]};
                    vf[hh] = *reinterpret_cast<const bf16x8*>(&raw);
                }
                if constexpr (!SUMMARY) {
                    // what the state gives: slots of a 32-wide step are key rows 16 (2 st) + 4 lg + 0..3 and 16 (2 st + 1) + 4 lg + 0..3
                    f32x4 o[4];                              // o^T: value 16 wave + 4 lg + r, token 16 it + lq
#pragma unroll
                    for (int it = 0; it < 4; ++it) o[it] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int st = 0; st < DK / 32; ++st) {
                        const f32x4 s0 = S[2 * st], s1 = S[2 * st + 1];
                        const float v[8] = {s0[0], s0[1], s0[2], s0[3], s1[0], s1[1], s1[2], s1[3]};
                        bf16x8 hi, lo;
                        split_hi_lo(v, hi, lo);
#pragma unroll
                        for (int it = 0; it < 4; ++it) {
                            const int R = 16 * it + lq;
                            const unsigned char* qrow = qimg + R * KROW + (lg & 1) * 8;
                            const u32x2 qa = *reinterpret_cast<const u32x2*>(qrow + ((4 * st + (lg >> 1)) ^ swz(R)) * 16);
                            const u32x2 qb = *reinterpret_cast<const u32x2*>(qrow + ((4 * st + 2 + (lg >> 1)) ^ swz(R)) * 16);
                            asm volatile("" ::: "memory");   // (kept apart, or two rows' reads become one, whose halves have to be moved)
                            const u32x4 raw = {qa[0], qa[1], qb[0], qb[1]};
                            const bf16x8 qf = *reinterpret_cast<const bf16x8*>(&raw);
                            o[it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, qf, o[it], 0, 0, 0);
                            o[it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, qf, o[it], 0, 0, 0);
                        }
                    }
#pragma unroll
                    for (int it = 0; it < 4; ++it) o[it] *= pw[16 * it + lq + 1];
#pragma unroll
                    for (int it = 0; it < 4; ++it)
#pragma unroll
                        for (int hh = 0; hh <= it / 2; ++hh) {
                            const uint16_t* pr = p_lds + (16 * it + lq) * PLD + 32 * hh + 8 * lg;
                            o[it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[hh], *reinterpret_cast<const bf16x8*>(pr), o[it], 0, 0, 0);
                            o[it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[hh], *reinterpret_cast<const bf16x8*>(pr + C * PLD), o[it], 0, 0, 0);
                        }
#pragma unroll
                    for (int it = 0; it < 4; ++it) act_st4(o_lds + (16 * it + lq) * OLD + 16 * wave + 4 * lg, o[it]);
                }
                lds_only_barrier();                          // the weights may be replaced; outputs are there
                if constexpr (!SUMMARY) {
                    typedef u32x4 __attribute__((aligned(8))) u32x4_half;      // (rows of results may be 8 bytes off a multiple of 16)
                    const int row = (64 * wave + lane) / VP, col = (64 * wave + lane) % VP * 8;
                    uint16_t* out = reinterpret_cast<uint16_t*>(a.out) + (int64_t)(row0 + t0) * a.out_stride + (int64_t)head * a.dv + v0;
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const u32x4 v = *reinterpret_cast<const u32x4*>(o_lds + (row + 32 * j) * OLD + col);
                        if (row + 32 * j < n) *reinterpret_cast<u32x4_half*>(out + (row + 32 * j) * a.out_stride + col) = v;
                    }
                }
                // ---- the state behind these tokens
                const float decayed = pw[n];
#pragma unroll
                for (int t = 0; t < DT; ++t) S[t] *= decayed;
#pragma unroll
                for (int hh = 0; hh < 2; ++hh) {
                    const u32x4 raw = *reinterpret_cast<const u32x4*>(&vf[hh]);
                    f32x4 fall[2];                           // what a value decays by until the chunk's end
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const int key = 32 * hh + 16 * q + 4 * lg;
                        if (n == C) {
                            fall[q] = *reinterpret_cast<const f32x4*>(fall_s + key);
                        } else {
#pragma unroll
                            for (int r = 0; r < 4; ++r) fall[q][r] = pw[key + r < n ? n - 1 - key - r : 0];
                        }
                    }
                    float v[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) v[j] = (j & 1 ? bf16_hi(raw[j >> 1]) : bf16_lo(raw[j >> 1])) * fall[j >> 2][j & 3];
                    bf16x8 hi, lo;
                    split_hi_lo(v, hi, lo);
                    const int ra = 32 * hh + tr, rb = ra + 16;
#pragma unroll
                    for (int t = 0; t < DT; ++t) {
                        const int pc = 2 * t + (tp >> 1);
                        const u32x2 klo = lds_tr16(kimg + ra * KROW + (pc ^ swz(ra)) * 16 + (tp & 1) * 8), khi = lds_tr16(kimg + rb * KROW + (pc ^ swz(rb)) * 16 + (tp & 1) * 8);
                        const u32x4 kraw = {klo[0], klo[1], khi[0], khi[1]};
                        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(&kraw);
                        S[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, hi, S[t], 0, 0, 0);
                        S[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, lo, S[t], 0, 0, 0);
                    }
                }
                lds_only_barrier();                          // this chunk's images may be replaced
            }
            float* dst = nullptr;
            if constexpr (SUMMARY) dst = a.seg_state + ((int64_t)seg * a.heads + head) * head_state;
            else if (last && slot >= 0) dst = a.state + (slot * a.heads + head) * head_state;
            if (dst) {
#pragma unroll
                for (int t = 0; t < DT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) dst[(int64_t)(16 * t + 4 * lg + r) * a.dv + sv] = S[t][r];
            }
        }
        if (!take_next()) return;
    }
}

// contributions of the segments -> states at their starts, in place; a thread per four state elements of a portion, walking its segments
__global__ __launch_bounds__(256) void lightning_starts_kernel(const LightningArgs a) {
    const int64_t head_state = (int64_t)a.dk * a.dv, per = a.heads * head_state, e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    const int first = blockIdx.y;                    // only a portion's first segment starts a walk
    if (a.chunks[4 * first + 3] != 0) return;
    const int count = portion_segments(a.chunks, a.n_chunks, first);
    if (e >= per) return;
    const float d = a.decay[e / head_state];
    const int64_t slot = a.state_slots[a.chunks[4 * first + 2]];
    const f32x4 cur = slot >= 0 && portion_carries(a.chunks, a.n_chunks, first, a.positions) ? *reinterpret_cast<const f32x4*>(a.state + slot * per + e) : f32x4{};
    float of = 0.f, power = 1.f;                     // (segments but the last are of one length)
    segment_starts(a.seg_state + first * per + e, per, count, cur, [&](int k) { return (float)a.chunks[4 * (first + k) + 1]; },
                   [&](float tokens) {
                       if (tokens != of) {
                           of = tokens;
                           power = powf(d, tokens);
                       }
                       return power;
                   });
}

// ------------------------------------------------------------------------------------------------ token by token, any type and size
// one workgroup per (portion, head, 32 value columns); the state slice in LDS, 8 groups of key rows x 32 columns
template <typename T>
__global__ __launch_bounds__(256) void lightning_generic_kernel(const LightningArgs a) {
    extern __shared__ float lds_f[];                 // [dk][32] state, [2][dk] k and q, [8][32] sums
    float *S = lds_f, *kq = S + a.dk * 32, *red = kq + 2 * a.dk;
    const int first = blockIdx.x, head = blockIdx.y, tid = threadIdx.x, c = tid & 31, rg = tid >> 5, col = blockIdx.z * 32 + c;
    if (a.chunks[4 * first + 3] != 0) return;        // a portion is walked whole from its first segment
    const int row0 = a.chunks[4 * first];
    int n_rows = a.chunks[4 * first + 1];
    for (int k = first + 1; k < a.n_chunks && a.chunks[4 * k + 3] != 0; ++k) n_rows += a.chunks[4 * k + 1];
    const int64_t slot = a.state_slots[a.chunks[4 * first + 2]], head_state = (int64_t)a.dk * a.dv;
    const bool ok = col < a.dv;
    float* pool = slot >= 0 ? a.state + (slot * a.heads + head) * head_state : nullptr;
    const bool carry = pool && portion_carries(a.chunks, a.n_chunks, first, a.positions);
    for (int r = rg; r < a.dk; r += 8) S[r * 32 + c] = carry && ok ? pool[(int64_t)r * a.dv + col] : 0.f;
    const float d = a.decay[head];
    for (int t = 0; t < n_rows; ++t) {
        const T* x = reinterpret_cast<const T*>(a.qkv) + (int64_t)(row0 + t) * a.qkv_stride;
        for (int i = tid; i < a.dk; i += 256) {
            const float k = act_ld(x + (int64_t)a.heads * a.dk + head * a.dk + i), q = act_ld(x + head * a.dk + i);
            kq[i] = act_round(silu_f(k), (const T*)nullptr);
            kq[a.dk + i] = act_round(silu_f(q), (const T*)nullptr);
        }
        const float v = ok ? act_round(silu_f(act_ld(x + 2 * (int64_t)a.heads * a.dk + (int64_t)head * a.dv + col)), (const T*)nullptr) : 0.f;
        __syncthreads();
        float acc = 0.f;
        for (int r = rg; r < a.dk; r += 8) {
            const float s = d * S[r * 32 + c] + kq[r] * v;
            S[r * 32 + c] = s;
            acc += s * kq[a.dk + r];
        }
        red[rg * 32 + c] = acc;
        __syncthreads();
        if (rg == 0 && ok) {
            float s = 0.f;
#pragma unroll
            for (int k = 0; k < 8; ++k) s += red[k * 32 + c];
            act_st(reinterpret_cast<T*>(a.out) + (int64_t)(row0 + t) * a.out_stride + (int64_t)head * a.dv + col, s);
        }
    }
    if (pool && ok)
        for (int r = rg; r < a.dk; r += 8) pool[(int64_t)r * a.dv + col] = S[r * 32 + c];
}

// ------------------------------------------------------------------------------------------------ one token per sequence (bf16)
// grid (heads, rows, dv / VC): VC / 4 lanes hold a state row's slice, 1024 / VC rows at a time
template <int VC>
__global__ __launch_bounds__(256) void lightning_step_kernel(const LightningArgs a) {
    constexpr int LN = VC / 4, RG = 256 / LN, UN = 8;
    extern __shared__ float lds_s[];                 // [2][dk] k and q, then [RG][VC] sums
    float *kq = lds_s, *red = lds_s + 2 * a.dk;
    const int head = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, c = (tid % LN) * 4, rg = tid / LN, col = blockIdx.z * VC + c;
    const int64_t slot = a.state_slots[row], head_state = (int64_t)a.dk * a.dv;
    const bool carry = slot >= 0 && a.positions[row] > 0;
    float* pool = a.state + ((slot >= 0 ? slot : 0) * a.heads + head) * head_state + col;
    const uint16_t* x = reinterpret_cast<const uint16_t*>(a.qkv) + (int64_t)row * a.qkv_stride;
    f32x4 s[UN];
#pragma unroll
    for (int u = 0; u < UN; ++u) {                   // asked for before anything is computed
        const int r = rg + u * RG;
        s[u] = carry && r < a.dk ? *reinterpret_cast<const f32x4*>(pool + (int64_t)r * a.dv) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for (int i = tid; i < a.dk; i += 256) {
        kq[i] = act_round(silu_f(act_ld(x + (int64_t)a.heads * a.dk + head * a.dk + i)), (const uint16_t*)nullptr);
        kq[a.dk + i] = act_round(silu_f(act_ld(x + head * a.dk + i)), (const uint16_t*)nullptr);
    }
    f32x4 v = act_ld4(x + 2 * (int64_t)a.heads * a.dk + (int64_t)head * a.dv + col);
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = act_round(silu_f(v[k]), (const uint16_t*)nullptr);
    const float d = a.decay[head];
    __syncthreads();
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int r0 = 0; r0 < a.dk; r0 += UN * RG) {
        if (r0) {
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                const int r = r0 + rg + u * RG;
                s[u] = carry && r < a.dk ? *reinterpret_cast<const f32x4*>(pool + (int64_t)r * a.dv) : f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const int r = r0 + rg + u * RG;
            if (r >= a.dk) continue;
            const f32x4 n = s[u] * d + v * kq[r];
            acc += n * kq[a.dk + r];
            if (slot >= 0) *reinterpret_cast<f32x4*>(pool + (int64_t)r * a.dv) = n;
        }
    }
    *reinterpret_cast<f32x4*>(red + rg * VC + c) = acc;
    __syncthreads();
    if (rg == 0) {
        f32x4 o = acc;
        for (int k = 1; k < RG; ++k) o += *reinterpret_cast<const f32x4*>(red + k * VC + c);
        act_st4(reinterpret_cast<uint16_t*>(a.out) + (int64_t)row * a.out_stride + (int64_t)head * a.dv + col, o);
    }
}

// ------------------------------------------------------------------------------------------------ norm and gate behind the heads
template <typename T, int CH>
__global__ __launch_bounds__(256) void norm_gate_kernel(T* __restrict__ out, uint16_t* __restrict__ packed, const T* __restrict__ x, const T* __restrict__ gate,
                                                        const float* __restrict__ w, float eps, int cols, int n, int64_t x_stride, int64_t gate_stride, int64_t out_stride) {
    __shared__ float lds[4];
    const int64_t row = blockIdx.x;
    f32x8 v[CH], gt[CH];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int c = (threadIdx.x + i * 256) * 8;
        v[i] = gt[i] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
        if (c < cols) {
            v[i] = act_ld8(x + row * x_stride + c);
            gt[i] = act_ld8(gate + row * gate_stride + c);
        }
        ss += sum4(v[i].a * v[i].a) + sum4(v[i].b * v[i].b);
    }
    const float inv = 1.f / sqrtf(block_sum256(ss, lds) / n + eps);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int c = (threadIdx.x + i * 256) * 8;
        if (c >= cols) continue;
        f32x8 r = v[i];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            r.a[k] *= inv * w[c + k] * sigmoid_f(gt[i].a[k]);
            r.b[k] *= inv * w[c + 4 + k] * sigmoid_f(gt[i].b[k]);
        }
        if (packed) act_st8(packed + pack_index((int)row, c, cols), r);
        else act_st8(out + row * out_stride + c, r);
    }
}

int walk_wide(const LightningArgs& a, hipStream_t stream) {
    constexpr size_t sum_lds = (size_t)C * (kWide + VS) * 2, lds = sum_lds + (size_t)C * kWide * 2 + (size_t)2 * C * PLD * 2;
    if (lds > 64 * 1024)
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(lightning_walk_kernel<false>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    const dim3 grid(a.n_chunks, a.heads, a.dv / VS);
    if (a.summaries) {
        lightning_walk_kernel<true><<<grid, 256, sum_lds, stream>>>(a);
        int rc = check_launch("lightning summary");
        if (rc) return rc;
        const int64_t per = (int64_t)a.heads * a.dk * a.dv;
        lightning_starts_kernel<<<dim3((unsigned)((per + 1023) / 1024), a.n_chunks), 256, 0, stream>>>(a);
        rc = check_launch("lightning starts");
        if (rc) return rc;
    }
    lightning_walk_kernel<false><<<grid, 256, lds, stream>>>(a);
    return check_launch("lightning walk");
}

template <int DK, int CW, int PW>
int pair_dk(const LightningArgs& a, hipStream_t stream) {
    constexpr size_t sum_lds = pair_lds_bytes<DK, CW>(true), lds = pair_lds_bytes<DK, CW>(false);
    if (lds > 64 * 1024)
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(lightning_pair_kernel<DK, CW, PW, false, false>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (sum_lds > 64 * 1024)
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(lightning_pair_kernel<DK, CW, PW, true, false>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)sum_lds);
    // heads run fastest: workgroups are dealt round-robin over the 8 XCDs, and segments differ in length while the heads of one do not
    const int walks = a.heads * (a.dv / (16 * CW));
    dim3 grid(walks, a.n_chunks);
    if (a.summaries) {
        lightning_pair_kernel<DK, CW, PW, true, false><<<grid, 64 * (CW + PW), sum_lds, stream>>>(a);
        int rc = check_launch("lightning summary");
        if (rc) return rc;
        const int64_t per = (int64_t)a.heads * a.dk * a.dv;
        lightning_starts_kernel<<<dim3((unsigned)((per + 1023) / 1024), a.n_chunks), 256, 0, stream>>>(a);
        rc = check_launch("lightning starts");
        if (rc) return rc;
    }
    // The longest portions as two pieces, where whole ones come to 193 to 320 workgroups: fewer are better cut into segments, more fill the CUs more than once and even out.  Other launches
    // have a kernel without that, as have those of less than four chunks a portion.
    const int places = 256 / walks, most = lightning_most_cut(places);
    if (!a.summaries && most && a.n_chunks <= kSplitPortions && walks * a.n_chunks > 192 && walks * a.n_chunks <= 320 && a.rows >= 4 * C * a.n_chunks) {
        if (a.n_chunks < places) grid.y = a.n_chunks + most < places ? a.n_chunks + most : places;
        if (lds > 64 * 1024)
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(lightning_pair_kernel<DK, CW, PW, false, true>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        lightning_pair_kernel<DK, CW, PW, false, true><<<grid, 64 * (CW + PW), lds, stream>>>(a);
    } else {
        lightning_pair_kernel<DK, CW, PW, false, false><<<grid, 64 * (CW + PW), lds, stream>>>(a);
    }
    return check_launch("lightning walk");
}

template <typename T>
void norm_gate_t(void* out, void* packed, const void* x, const void* gate, const float* w, float eps, int rows, int cols, int n, int64_t xs, int64_t gs, int64_t os,
                 hipStream_t stream) {
    const int ch = (cols + 2047) / 2048;
    auto go = [&](auto k) {
        norm_gate_kernel<T, decltype(k)::value><<<rows, 256, 0, stream>>>((T*)out, (uint16_t*)packed, (const T*)x, (const T*)gate, w, eps, cols, n, xs, gs, os);
    };
    if (ch <= 1) go(std::integral_constant<int, 1>{});
    else if (ch <= 2) go(std::integral_constant<int, 2>{});
    else if (ch <= 4) go(std::integral_constant<int, 4>{});
    else if (ch <= 8) go(std::integral_constant<int, 8>{});
    else go(std::integral_constant<int, kRowPieces>{});
}

}  // namespace

bool lightning_supported(int dk, int dv) { return (dk == 64 || dk == 128 || dk == 256) && dv > 0 && dv % 64 == 0; }

int launch_lightning_chunks(const LightningArgs& a, int f32, int generic, hipStream_t stream) {
    if (!f32 && !generic && lightning_supported(a.dk, a.dv)) {
        switch (a.dk) {
            case 64: return a.dv % 128 == 0 ? pair_dk<64, 8, 4>(a, stream) : pair_dk<64, 4, 4>(a, stream);
            case 128: return a.dv % 128 == 0 ? pair_dk<128, 8, 4>(a, stream) : pair_dk<128, 4, 4>(a, stream);
            default: return walk_wide(a, stream);
        }
    }
    const size_t lds = ((size_t)a.dk * 34 + 256) * 4;
    const dim3 grid(a.n_chunks, a.heads, (a.dv + 31) / 32);
    const void* fn = f32 ? reinterpret_cast<const void*>(lightning_generic_kernel<float>) : reinterpret_cast<const void*>(lightning_generic_kernel<uint16_t>);
    if (lds > 64 * 1024) (void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (f32) lightning_generic_kernel<float><<<grid, 256, lds, stream>>>(a);
    else lightning_generic_kernel<uint16_t><<<grid, 256, lds, stream>>>(a);
    return check_launch("lightning generic");
}

int launch_lightning_step(const LightningArgs& a, hipStream_t stream) {
    const bool wide = (int64_t)a.rows * a.heads * (a.dv / 64) >= 512;
    const size_t lds = (size_t)2 * a.dk * 4 + 1024 * 4;
    if (wide) lightning_step_kernel<64><<<dim3(a.heads, a.rows, a.dv / 64), 256, lds, stream>>>(a);
    else lightning_step_kernel<32><<<dim3(a.heads, a.rows, a.dv / 32), 256, lds, stream>>>(a);
    return check_launch("lightning step");
}

int launch_norm_gate(void* out, void* packed, const void* x, const void* gate, const float* w, float eps, int rows, int cols, int n, int64_t x_stride,
                     int64_t gate_stride, int64_t out_stride, int f32, hipStream_t stream) {
    if (f32) norm_gate_t<float>(out, nullptr, x, gate, w, eps, rows, cols, n, x_stride, gate_stride, out_stride, stream);
    else norm_gate_t<uint16_t>(out, packed, x, gate, w, eps, rows, cols, n, x_stride, gate_stride, out_stride, stream);
    return check_launch("norm_gate");
}

}  // namespace nvh
