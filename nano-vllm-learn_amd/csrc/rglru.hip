// Real-gated linear recurrent unit with a causal depthwise convolution in front of it:
//   u = conv(x)           y-branch gate applied at the end
//   r = sigmoid(ra u), i = sigmoid(ri u)            block-diagonal maps (MFMA)
//   log a = -rate r ; S = a S + sqrt(1 - a^2) i u ; out = S gelu(y)
// The recurrence and everything that enters it besides u is fp32; u is rounded once to the activation type.
//
// Prompt portions (launch_rglru_chunks) come cut into segments by the host and are worked through 64 tokens at a time, by workgroups that own a diagonal block:
// convolution into LDS, both gates on MFMA tiles, and the scan of the 64 tokens IN the accumulator layout, then S gelu(y) back out through LDS.
// - Blocks of up to 256 channels (bf16) mostly: any workgroup of the block takes any step, and the state in front of a step comes from the ones before it
//   (rglru_chain_kernel; a lane holds 16 consecutive tokens).  Cut or whole portions, the steps are the same.
// - Otherwise a workgroup walks a segment with the state in registers (rglru_scan_kernel; larger blocks rglru_walk_kernel; a lane holds 4 consecutive tokens of one
//   channel, the 4 lane groups 16: compose 4 in the lane, two shuffles across the groups, a carry over the 16-token tiles).  A portion of one segment is one such walk.
//   Of a cut one a SUMMARY walk first leaves (product of decays, end value) of every segment but the last, and the second walk of a segment starts from the composition
//   of the ones before it.  Blocks of up to 256 channels come here where walks of whole portions are faster (whole_walks), and of cut ones from callers without `links`.
// State and convolution ring are read by the walks and written by a small launch behind them, by the steps in a portion's last one: nobody sees a half-updated one.
// Decode (launch_rglru_step): one workgroup per 16 channels and 32 sequences does all of it in one launch.  Convolution inputs live in a ring of
// `taps` entries (input of position p at entry p % taps): the entry a step writes is the one no workgroup of that step reads.
// A sequence's first token (position 0) takes state and earlier inputs as zero instead of reading them: slots need no clearing when reused.
// Bytes per (token, channel) of a walk: 2 (x) + 2 (y) + 2 (out); about 25 vector instructions and 8 transcendentals: issue-bound.
#include "hybrid.h"

namespace nvh {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
constexpr int CH = kRglruChunk;
constexpr int kGroup = 256;                          // channels one walking workgroup owns at most (16 waves x 16)

__device__ __forceinline__ float fast_sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ float fast_sigmoid(float x) { return fast_rcp(1.f + fast_exp2(-kLog2e * x)); }
__device__ __forceinline__ float fast_gelu(float z) {
    constexpr float c = 2.f * kLog2e * 0.7978845608028654f;
    const float t = z * (c + c * 0.044715f * (z * z));
    return z - z * fast_rcp(1.f + fast_exp2(t));
}
// decay a = exp(-rate r) and input sqrt(1 - a^2) i u; 1 - a^2 by its series where it would cancel
__device__ __forceinline__ void decay_and_input(float rate, float r, float ig, float u, float& a, float& b) {
    const float y = (2.f * rate) * r;
    a = fast_exp2((-kLog2e * rate) * r);
    const float series = y * (1.f + y * (-1.f / 2 + y * (1.f / 6 - y * (1.f / 24))));
    b = fast_sqrt(y < 0.06f ? series : 1.f - a * a) * ig * u;
}

// convolution input of the token `t` rows after the portion's first row (negative: before it, from the ring; before position 0: zero)
template <typename T>
__device__ __forceinline__ const T* conv_input(const RglruArgs& a, int seq_row0, int t, int64_t pos0, int slot, int ch) {
    if (t >= 0) return reinterpret_cast<const T*>(a.yx) + (int64_t)(seq_row0 + t) * a.yx_stride + a.width + ch;
    const int64_t p = pos0 + t;
    if (p < 0 || slot < 0) return nullptr;
    return reinterpret_cast<const T*>(a.conv_state) + ((int64_t)slot * a.taps + (int)(p % a.taps)) * a.width + ch;
}

__device__ __forceinline__ void fma8(float (&acc)[8], const u32x4 v, const float* w) {
    const f32x4 w0 = *reinterpret_cast<const f32x4*>(w), w1 = *reinterpret_cast<const f32x4*>(w + 4);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float wa = k < 2 ? w0[2 * k] : w1[2 * k - 4], wb = k < 2 ? w0[2 * k + 1] : w1[2 * k - 3];
        acc[2 * k] += wa * bf16_lo(v[k]);
        acc[2 * k + 1] += wb * bf16_hi(v[k]);
    }
}
__device__ __forceinline__ u32x4 pack8(const float (&v)[8]) {
    return u32x4{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
}

// 8 channels x CNT consecutive tokens of the convolution; row(t) -> pointer of token t's input (null: zero).  Every input row is unpacked once.
template <int TAPS, int CNT, typename Row>
__device__ __forceinline__ void conv_run(const RglruArgs& a, int ch, int taps_rt, float (&acc)[CNT][8], Row row) {
    const f32x4 b0 = *reinterpret_cast<const f32x4*>(a.conv_b + ch), b1 = *reinterpret_cast<const f32x4*>(a.conv_b + ch + 4);
#pragma unroll
    for (int i = 0; i < CNT; ++i)
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[i][k] = k < 4 ? b0[k] : b1[k - 4];
    if constexpr (TAPS > 0) {
        f32x4 w[TAPS][2];
#pragma unroll
        for (int j = 0; j < TAPS; ++j)
#pragma unroll
            for (int q = 0; q < 2; ++q) w[j][q] = *reinterpret_cast<const f32x4*>(a.conv_w + (int64_t)j * a.width + ch + 4 * q);
        u32x4 v[CNT + TAPS - 1];
#pragma unroll
        for (int s = 0; s < CNT + TAPS - 1; ++s) {
            const uint16_t* p = row(s - (TAPS - 1));
            v[s] = p ? *reinterpret_cast<const u32x4*>(p) : u32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int s = 0; s < CNT + TAPS - 1; ++s)
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float x = k & 1 ? bf16_hi(v[s][k >> 1]) : bf16_lo(v[s][k >> 1]);
#pragma unroll
                for (int i = 0; i < CNT; ++i)
                    if (s - i >= 0 && s - i < TAPS) acc[i][k] += w[s - i][k >> 2][k & 3] * x;
            }
    } else {
        for (int j = 0; j < taps_rt; ++j)
#pragma unroll
            for (int i = 0; i < CNT; ++i) {
                const uint16_t* p = row(i + j - (taps_rt - 1));
                if (p) fma8(acc[i], *reinterpret_cast<const u32x4*>(p), a.conv_w + (int64_t)j * a.width + ch);
            }
    }
}

// Only a portion's last segment may have no rows; where that is its only one, nothing is walked and the slot keeps what it holds.
__device__ __forceinline__ bool portion_without_rows(int n, int kth) { return n <= 0 && kth == 0; }

// what a segment starts from (segment table index `seg`, channel ch)
__device__ __forceinline__ float walk_start(const RglruArgs& a, bool summary, bool more, int seg, int kth, int slot, int64_t pos0, int ch) {
    float cs = 0.f;
    if (kth == 0) {
        if (!summary && more) return a.a_cum[(int64_t)seg * a.width + ch];     // left there by the summary walk: the state itself is being replaced
        if (pos0 > 0 && slot >= 0) cs = a.state[(int64_t)slot * a.width + ch];
    } else if (!summary) {
        const int64_t first = (int64_t)(seg - kth) * a.width + ch;
        cs = a.s_loc[first];
        for (int k = 1; k < kth; ++k) cs = a.a_cum[first + (int64_t)k * a.width] * cs + a.s_loc[first + (int64_t)k * a.width];
    }
    return cs;
}

// ------------------------------------------------------------------------------------------------ prompt portions, MFMA form (bf16)
// grid (segments, blocks x channel groups of at most 256); a wave owns 16 channels
template <bool SUMMARY>
__global__ __launch_bounds__(1024) void rglru_walk_kernel(const RglruArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint16_t u_lds[];           // [CH][block + 8] u; behind it [CH][group + 8] y, then out
    const int groups = (a.block + kGroup - 1) / kGroup, seg = blockIdx.x, blk = blockIdx.y / groups, g0 = (blockIdx.y - blk * groups) * kGroup;
    const int row0 = a.chunks[seg * 4], n = a.chunks[seg * 4 + 1], seq = a.chunks[seg * 4 + 2], kth = a.chunks[seg * 4 + 3];
    const bool more = seg + 1 < a.n_chunks && a.chunks[seg * 4 + 6] == seq;    // another segment of this sequence follows
    if ((SUMMARY && !more) || portion_without_rows(n, kth)) return;
    const int off0 = kth * a.segment, seq_row0 = row0 - off0;
    const int slot = a.state_slots[seq];
    const int64_t pos0 = a.positions[seq_row0];
    const int gcols = a.block - g0 < kGroup ? a.block - g0 : kGroup;           // this workgroup's channels of the block: g0 ..
    const int ld = a.block + 8, oct = a.block / 8, yld = gcols + 8, goct = gcols / 8;
    uint16_t* y_lds = u_lds + CH * ld;
    const int tid = threadIdx.x, threads = blockDim.x, lane = tid & 63, wave = tid >> 6, lq = lane & 15, lg = lane >> 4;
    const uint16_t* yx = reinterpret_cast<const uint16_t*>(a.yx);
    const uint16_t* ra = reinterpret_cast<const uint16_t*>(a.ra) + (int64_t)blk * a.block * a.block;
    const uint16_t* ri = reinterpret_cast<const uint16_t*>(a.ri) + (int64_t)blk * a.block * a.block;
    const bool mine = 16 * wave < gcols;             // (a narrower last group leaves waves to the row work only)
    const int cg = mine ? 16 * wave + lq : lq, cb = g0 + cg, ch = blk * a.block + cb;
    const float rb = a.ra_b[ch], ib = a.ri_b[ch], rate = a.rate[ch];
    float ca = 1.f, cs = walk_start(a, SUMMARY, more, seg, kth, slot, pos0, ch);
    if (SUMMARY && kth == 0 && mine && lg == 0) a.a_cum[(int64_t)seg * a.width + ch] = cs;
    const int pairs = CH / 2 * oct;
    for (int t0 = 0; t0 < n; t0 += CH) {
        const int cnt = n - t0 < CH ? n - t0 : CH;
        // ---- u into LDS, two tokens x 8 channels a time; y beside it
        const bool inside = off0 + t0 >= a.taps - 1;                           // no tap reaches in front of the portion
        for (int e = tid; e < pairs; e += threads) {
            const int tp = e / oct, o = e - tp * oct, t = 2 * tp, c8 = blk * a.block + o * 8;
            u32x4 r0 = {0, 0, 0, 0}, r1 = {0, 0, 0, 0};
            if (t < cnt) {
                float acc[2][8];
                const int at = off0 + t0 + t;
                const uint16_t* base = yx + (int64_t)(seq_row0 + at) * a.yx_stride + a.width + c8;
                const int last = t + 1 < cnt ? 1 : 0;                          // (an odd tail repeats its last row: not used)
                if (inside && a.taps == 4)
                    conv_run<4, 2>(a, c8, 4, acc, [&](int s) { return base + (int64_t)(s < last ? s : last) * a.yx_stride; });
                else
                    conv_run<0, 2>(a, c8, a.taps, acc, [&](int s) { return conv_input<uint16_t>(a, seq_row0, at + (s < last ? s : last), pos0, slot, c8); });
                r0 = pack8(acc[0]);
                if (last) r1 = pack8(acc[1]);
            }
            *reinterpret_cast<u32x4*>(u_lds + t * ld + o * 8) = r0;
            *reinterpret_cast<u32x4*>(u_lds + (t + 1) * ld + o * 8) = r1;
        }
        if (!SUMMARY)
            for (int e = tid; e < cnt * goct; e += threads) {
                const int t = e / goct, o = e - t * goct;
                *reinterpret_cast<u32x4*>(y_lds + t * yld + o * 8) =
                    *reinterpret_cast<const u32x4*>(yx + (int64_t)(row0 + t0 + t) * a.yx_stride + blk * a.block + g0 + o * 8);
            }
        __syncthreads();
        if (mine) {
            f32x4 gr[4], gi[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) gr[m] = gi[m] = f32x4{0.f, 0.f, 0.f, 0.f};
            const uint16_t* wr = ra + (int64_t)cb * a.block + 8 * lg;
            const uint16_t* wi = ri + (int64_t)cb * a.block + 8 * lg;
            bf16x8 br = *reinterpret_cast<const bf16x8*>(wr), bi = *reinterpret_cast<const bf16x8*>(wi);
            for (int k = 0; k < a.block; k += 32) {
                const int kn = k + 32 < a.block ? k + 32 : k;                  // the next step's weights travel under this one's products
                const bf16x8 nr = *reinterpret_cast<const bf16x8*>(wr + kn), ni = *reinterpret_cast<const bf16x8*>(wi + kn);
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const bf16x8 ua = *reinterpret_cast<const bf16x8*>(u_lds + (16 * m + lq) * ld + k + 8 * lg);
                    gr[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ua, br, gr[m], 0, 0, 0);
                    gi[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ua, bi, gi[m], 0, 0, 0);
                }
                br = nr;
                bi = ni;
            }
            // ---- decays, inputs and the scan: this lane holds tokens 16 m + 4 lg + i of one channel
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                if (16 * m >= cnt) break;
                float av[4], sv[4];
                float pa = 1.f, ps = 0.f;                                      // inclusive composition over the lane's 4 tokens
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int t = 16 * m + 4 * lg + i;
                    float dec, inp;
                    decay_and_input(rate, fast_sigmoid(gr[m][i] + rb), fast_sigmoid(gi[m][i] + ib), act_ld(u_lds + t * ld + cb), dec, inp);
                    if (t >= cnt) dec = 1.f, inp = 0.f;
                    ps = dec * ps + inp;
                    pa *= dec;
                    av[i] = pa;
                    sv[i] = ps;
                }
                float ga = pa, gs = ps;                                        // inclusive over the lane groups so far
                {
                    const float oa = __shfl_up(ga, 16), os = __shfl_up(gs, 16);
                    if (lg >= 1) { gs = ga * os + gs; ga *= oa; }
                }
                {
                    const float oa = __shfl_up(ga, 32), os = __shfl_up(gs, 32);
                    if (lg >= 2) { gs = ga * os + gs; ga *= oa; }
                }
                if (!SUMMARY) {
                    float xa = __shfl_up(ga, 16), xs = __shfl_up(gs, 16);
                    if (lg == 0) { xa = 1.f; xs = 0.f; }
                    const float before = xa * cs + xs;                      // the state in front of this lane's first token
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        uint16_t* p = y_lds + (16 * m + 4 * lg + i) * yld + cg;
                        act_st(p, (av[i] * before + sv[i]) * fast_gelu(act_ld(p)));
                    }
                }
                const float ta = __shfl(ga, 48 + lq), ts = __shfl(gs, 48 + lq);    // the whole tile
                cs = ta * cs + ts;
                ca *= ta;
            }
        }
        __syncthreads();
        if (!SUMMARY)
            for (int e = tid; e < cnt * goct; e += threads) {
                const int t = e / goct, o = e - t * goct;
                *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(a.out) + (int64_t)(row0 + t0 + t) * a.out_stride + blk * a.block + g0 + o * 8) =
                    *reinterpret_cast<const u32x4*>(y_lds + t * yld + o * 8);
            }
        // (the next tokens' y goes where these rows were read from: same threads, same places)
    }
    if (mine && lg == 0 && (SUMMARY || !more)) {
        a.s_loc[(int64_t)seg * a.width + ch] = cs;
        if (SUMMARY && kth) a.a_cum[(int64_t)seg * a.width + ch] = ca;
    }
}

// ------------------------------------------------------------------------------------------------ prompt portions, blocks of up to 256 channels
// The same walk with everything in flight early: x and y of the next 64 tokens travel by LDS-DMA under this step's arithmetic, both gates' weights of a wave's
// 16 channels stay in registers for the whole segment, and u and y come into the accumulator layout by single elements (through an MFMA with a 0/1 selection matrix
// a gate without a number took its 15 neighbours' with it).
// Eight transcendentals and about 25 vector instructions per (token, channel) bound it (the vector units issue three quarters of the time at a block of 256), so
// a block has a wave for every 16 channels, four on each SIMD at 256: 128 registers a lane, addresses computed again (fresh) instead of held.  Rows are
// reached by 32-bit offsets from a step's first one; the 16-token passes are unrolled and find everything at fixed distances.  One barrier behind the scan frees u and
// makes out whole, one behind the rows' way out and the next convolution frees x.
// Against the walk without LDS-DMA, four blocks of 256 channels, 16 sequences of 1024 tokens as whole portions: 200 -> 148 us (144 since elements are read singly); of
// 32 channels 66 -> 59 (56).  What runs in their place now (whole_walks says where not) takes 70 and 30 there.
constexpr int HALO = 8;                              // rows in front of a step's 64 in the x image: taps <= HALO + 1

__device__ __forceinline__ int fresh(int v) {         // computed again from here on instead of held in registers across the loop
    asm volatile("" : "+v"(v));
    return v;
}

__device__ __forceinline__ void lds_barrier() {      // (a __syncthreads() would drain the DMA in flight)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <int KS> constexpr size_t scan_x_bytes() { return (size_t)(CH + HALO) * KS * 64 + 1024; }     // (the last DMA instruction may run over)
template <int KS> constexpr int scan_y_dma() { return 512 + (KS & (KS - 1) ? 0 : 16); }                 // elements between the pieces of two DMA instructions
template <int KS> constexpr size_t scan_y_bytes() { return (size_t)4 * KS * scan_y_dma<KS>() * 2; }
template <int KS> constexpr size_t scan_lds_bytes(int taps) {
    return scan_x_bytes<KS>() + (size_t)CH * (KS * 32 + 8) * 2 + 2 * scan_y_bytes<KS>() + (size_t)(taps + 1) * KS * 128;
}

template <int KS, bool SUMMARY>                      // block = 32 KS; grid (blocks, segments)
__global__ __launch_bounds__(128 * KS, 4) void rglru_scan_kernel(const RglruArgs a) {
    constexpr int BLOCK = 32 * KS, OCT = 4 * KS, WAVES = 2 * KS, THREADS = 64 * WAVES, LD = BLOCK + 8;
    constexpr int XINS = ((CH + HALO) * OCT + 63) / 64;                        // DMA instructions; y has two a wave
    // y image: pieces of 8 channels in order, odd rows' swapped in pairs, 32 spare bytes behind 64 where a row is a power of two: 16 rows' pieces miss each
    // other's banks, and the four rows of a lane lie at fixed distances
    constexpr int YDMA = scan_y_dma<KS>(), YBUF = 4 * KS * YDMA;
    static_assert(XINS <= 3 * WAVES && CH * OCT == 2 * THREADS);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    uint16_t* x_lds = reinterpret_cast<uint16_t*>(smem);                       // [HALO + CH][BLOCK]
    uint16_t* u_lds = x_lds + scan_x_bytes<KS>() / 2;                          // [CH][LD]
    uint16_t* y_lds = u_lds + CH * LD;                                         // [2][YBUF]; out after the scan
    float* w_lds = reinterpret_cast<float*>(y_lds + 2 * YBUF);                 // [taps + 1][BLOCK]: taps, then the bias
    const int seg = blockIdx.y + blockIdx.z * gridDim.y, blk = blockIdx.x, c0 = blk * BLOCK;
    if (seg >= a.n_chunks) return;
    const int row0 = a.chunks[seg * 4], n = a.chunks[seg * 4 + 1], seq = a.chunks[seg * 4 + 2], kth = a.chunks[seg * 4 + 3];
    const bool more = seg + 1 < a.n_chunks && a.chunks[seg * 4 + 6] == seq;
    if ((SUMMARY && !more) || portion_without_rows(n, kth)) return;
    const int off0 = kth * a.segment, seq_row0 = row0 - off0;
    const int slot = a.state_slots[seq];
    const int64_t pos0 = a.positions[seq_row0];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lq = lane & 15, lg = lane >> 4;
    const uint16_t* yx = reinterpret_cast<const uint16_t*>(a.yx);
    auto dma = [&](const char* src, void* dst) __attribute__((always_inline)) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
    };
    const uint32_t stride = (uint32_t)a.yx_stride * 2;                         // bytes; a step's 72 rows are reached by 32-bit offsets from its first one
    auto stage_x = [&](int t0) __attribute__((always_inline)) {                // rows t0 - HALO .. t0 + CH - 1 of the segment, clamped to the portion's rows that exist
        const char* base = reinterpret_cast<const char*>(yx + (int64_t)(row0 + t0 - HALO) * a.yx_stride + a.width + c0);
        const int lo = HALO - off0 - t0, hi = n - 1 + HALO - t0;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int ins = wave + WAVES * j;
            if (ins < XINS) {
                const int s = ins * 64 + fresh(lane), r = s / OCT, d = r < lo ? lo : (r > hi ? hi : r);
                dma(base + ((uint32_t)d * stride + (uint32_t)(s % OCT) * 16), x_lds + ins * 512);
            }
        }
    };
    auto stage_y = [&](int t0, uint16_t* image) __attribute__((always_inline)) {
        const char* base = reinterpret_cast<const char*>(yx + (int64_t)(row0 + t0) * a.yx_stride + c0);
        const int hi = n - 1 - t0;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int ins = wave + WAVES * j, s = ins * 64 + fresh(lane), r = s / OCT, d = r < hi ? r : hi;
            dma(base + ((uint32_t)d * stride + (uint32_t)((s % OCT) ^ (r & 1)) * 16), image + ins * YDMA);
        }
    };
    stage_x(0);
    if (!SUMMARY && n > 0) stage_y(0, y_lds);        // (a last segment without rows has some of x in front of it, but none of y)
    for (int e = tid; e < (a.taps + 1) * BLOCK; e += THREADS)
        w_lds[e] = e < a.taps * BLOCK ? a.conv_w[(int64_t)(e / BLOCK) * a.width + c0 + e % BLOCK] : a.conv_b[c0 + e % BLOCK];

    // ---- this wave's 16 channels
    const int cb = 16 * wave + lq, ch = c0 + cb;
    bf16x8 wr[KS], wi[KS];
    {
        const uint16_t* pr = reinterpret_cast<const uint16_t*>(a.ra) + (int64_t)ch * BLOCK + 8 * lg;
        const uint16_t* pi = reinterpret_cast<const uint16_t*>(a.ri) + (int64_t)ch * BLOCK + 8 * lg;
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            wr[k] = *reinterpret_cast<const bf16x8*>(pr + 32 * k);
            wi[k] = *reinterpret_cast<const bf16x8*>(pi + 32 * k);
        }
    }
    const float rb = -kLog2e * a.ra_b[ch], ib = -kLog2e * a.ri_b[ch], rate = a.rate[ch];
    float ca = 1.f, cs = walk_start(a, SUMMARY, more, seg, kth, slot, pos0, ch);
    if (SUMMARY && kth == 0 && lg == 0) a.a_cum[(int64_t)seg * a.width + ch] = cs;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    if (off0 == 0)                                   // inputs in front of the portion: from the ring, zero in front of the sequence
        for (int e = tid; e < (a.taps - 1) * OCT; e += THREADS) {
            const int back = e / OCT + 1, o = e % OCT;
            const uint16_t* p = conv_input<uint16_t>(a, seq_row0, -back, pos0, slot, c0 + o * 8);
            *reinterpret_cast<u32x4*>(x_lds + (HALO - back) * BLOCK + o * 8) = p ? *reinterpret_cast<const u32x4*>(p) : u32x4{0, 0, 0, 0};
        }

    auto convolve = [&]() __attribute__((always_inline)) {                     // x -> u, eight tokens x 2 channels a thread
        const int id = fresh(tid), o = 2 * (id % (16 * KS)), t = 8 * (id / (16 * KS));
        const uint16_t* xp = x_lds + (HALO + t - (a.taps - 1)) * BLOCK + o;
        const float* wp = w_lds + o;
        const f32x2 bias = *reinterpret_cast<const f32x2*>(wp + a.taps * BLOCK);
        float acc[8][2];
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i][0] = bias[0], acc[i][1] = bias[1];
        if (a.taps == 4) {
            f32x2 w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = *reinterpret_cast<const f32x2*>(wp + j * BLOCK);
#pragma unroll
            for (int s = 0; s < 11; ++s) {
                const uint32_t v = *reinterpret_cast<const uint32_t*>(xp + s * BLOCK);
                const float lo = bf16_lo(v), hi = bf16_hi(v);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (s - j >= 0 && s - j < 8) {
                        acc[s - j][0] += w[j][0] * lo;
                        acc[s - j][1] += w[j][1] * hi;
                    }
            }
        } else {
            for (int j = 0; j < a.taps; ++j) {
                const f32x2 w = *reinterpret_cast<const f32x2*>(wp + j * BLOCK);
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const uint32_t v = *reinterpret_cast<const uint32_t*>(xp + (i + j) * BLOCK);
                    acc[i][0] += w[0] * bf16_lo(v);
                    acc[i][1] += w[1] * bf16_hi(v);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) *reinterpret_cast<uint32_t*>(u_lds + (t + i) * LD + o) = pack_bf16x2(acc[i][0], acc[i][1]);
    };
    lds_barrier();                                   // (what came out of the ring)
    convolve();
    lds_barrier();
    for (int t0 = 0; t0 < n; t0 += CH) {
        const int cnt = n - t0 < CH ? n - t0 : CH;
        uint16_t* y_now = y_lds + (t0 / CH & 1) * YBUF;
        if (t0 + CH < n) {                           // x has become u, and the other y image went out before the barrier
            stage_x(t0 + CH);
            if (!SUMMARY) stage_y(t0 + CH, y_lds + ((t0 / CH + 1) & 1) * YBUF);
        }
        const int ln = fresh(lane), lq = ln & 15, lg = ln >> 4, piece = 2 * wave + (lq >> 3);
        const auto at = [](int row, int p) { const int s = row * OCT + p; return s / 64 * YDMA + s % 64 * 8; };
        const uint16_t *u_row = u_lds + lq * LD + 8 * lg, *u_own = u_lds + 4 * lg * LD + cb;
        uint16_t* y_even = y_now + at(4 * lg, piece) + (lq & 7);               // this lane's channel in rows 4 lg and, by fixed distances, 4 lg + 2
        uint16_t* y_odd = y_now + at(4 * lg, piece ^ 1) + (lq & 7);            // ... and, likewise, in 4 lg + 1 and 4 lg + 3
#pragma unroll
        for (int tm = 0; tm < CH; tm += 16) {        // 16 tokens at a time
            if (tm > 0 && tm >= cnt) break;
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
            f32x4 gr = zero, gi = zero;
#pragma unroll
            for (int k = 0; k < KS; ++k) {
                const bf16x8 ua = *reinterpret_cast<const bf16x8*>(u_row + tm * LD + 32 * k);
                gr = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ua, wr[k], gr, 0, 0, 0);
                gi = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ua, wi[k], gi, 0, 0, 0);
            }
            float uu[4], yv[4], av[4], sv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) uu[i] = act_ld(u_own + (tm + i) * LD);
            if (!SUMMARY)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int off = tm / 16 * KS * YDMA + (KS == 8 ? i / 2 * YDMA : i / 2 * 2 * BLOCK);
                    yv[i] = act_ld(i & 1 ? y_odd + off + BLOCK : y_even + off);
                }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float rg = fast_rcp(1.f + fast_exp2(gr[i] * -kLog2e + rb)), ig = fast_rcp(1.f + fast_exp2(gi[i] * -kLog2e + ib));
                decay_and_input(rate, rg, ig, uu[i], av[i], sv[i]);
            }
            if (tm + 16 > cnt) {                     // (tokens past the end leave the state alone)
                asm volatile("");                    // (a branch: the comparisons are wanted in the last step only)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (tm + 4 * lg + i >= cnt) av[i] = 1.f, sv[i] = 0.f;
            }
#pragma unroll
            for (int i = 1; i < 4; ++i) {            // inclusive inside the lane
                sv[i] += av[i] * sv[i - 1];
                av[i] *= av[i - 1];
            }
            // across the four lane groups (4 tokens each): e = the even group of the pair, then both pairs' totals to everyone
            const auto swap16 = [](float v) { return __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false); };
            const auto swap32 = [](float v) { return __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false); };
            const bool odd = lg & 1;
            const float pa = av[3], ps = sv[3];
            const float ea = __uint_as_float(swap16(pa)[0]), es = __uint_as_float(swap16(ps)[0]);
            const float ia = odd ? pa * ea : pa, is = odd ? pa * es + ps : ps;                      // inclusive inside the pair
            const auto ha = swap32(__uint_as_float(swap16(ia)[1])), hs = swap32(__uint_as_float(swap16(is)[1]));
            const float la = __uint_as_float(ha[0]), ls = __uint_as_float(hs[0]), ua_ = __uint_as_float(ha[1]), us_ = __uint_as_float(hs[1]);
            if (!SUMMARY) {
                float before = lg >= 2 ? la * cs + ls : cs;
                before = odd ? ea * before + es : before;                                           // the state in front of this lane's first token
#pragma unroll
                for (int i = 0; i < 4; i += 2) {
                    const uint32_t two = pack_bf16x2((av[i] * before + sv[i]) * fast_gelu(yv[i]), (av[i + 1] * before + sv[i + 1]) * fast_gelu(yv[i + 1]));
                    const int off = tm / 16 * KS * YDMA + (KS == 8 ? i / 2 * YDMA : i * BLOCK);
                    y_even[off] = (uint16_t)two;
                    y_odd[off + BLOCK] = (uint16_t)(two >> 16);
                }
            }
            cs = ua_ * (la * cs + ls) + us_;
            if (SUMMARY) ca *= la * ua_;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // the next step's x and y, asked for a step ago
        lds_barrier();                               // they are in LDS for everyone; u is free and out is whole
        if (!SUMMARY) {
            char* out = reinterpret_cast<char*>(reinterpret_cast<uint16_t*>(a.out) + (int64_t)(row0 + t0) * a.out_stride + c0);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int e = fresh(tid) + j * THREADS, r = e / OCT, p = e % OCT;
                if (r < cnt)
                    *reinterpret_cast<u32x4*>(out + ((uint32_t)r * (uint32_t)(a.out_stride * 2) + (uint32_t)p * 16)) = *reinterpret_cast<const u32x4*>(y_now + at(r, p ^ (r & 1)));
            }
        }
        if (t0 + CH < n) convolve();
        lds_barrier();
    }
    if (lg == 0 && (SUMMARY || !more)) {
        a.s_loc[(int64_t)seg * a.width + ch] = cs;
        if (SUMMARY && kth) a.a_cum[(int64_t)seg * a.width + ch] = ca;
    }
}

// ------------------------------------------------------------------------------------------------ the same blocks, any workgroup any 64 tokens
// The same arithmetic, cut into steps of 64 tokens that any workgroup of the block can take: what enters the recurrence needs no state, so a step's decays and
// inputs are composed from its first token on, and only the state in front of it comes from elsewhere: out = (A h + S) gelu(y).  A workgroup keeps both gates'
// weights of its block in registers (a wave its 16 channels') and draws steps by ticket, in the order of rglru_steps_kernel's list.  The state in front is found by decoupled
// look-back (Merrill and Garland, single-pass parallel prefix scan, 2016).  Per step and wave: products, gates, scan -> (product of decays, end value) of its 16 channels published;
// then the state in front: the nearest step of the portion that has published the state behind it, and from there the published pairs one by one (always this order of sums,
// whoever was first); then the output, and the next step's convolution.
// A drawn step waits for steps drawn before it only, and those are in the hands of workgroups that run: no assumption on how many are resident or on their order.  The
// wait is bounded all the same (a state of NaN behind it).
// x travels by LDS-DMA under a step's products, y a step ahead; u and y come into the accumulator layout by single elements.  Rows lie so that a lane of the accumulators
// holds 16 consecutive tokens of a channel: one composition across lanes a step, not four.
// Both gates' products of all 64 tokens come first and decays and inputs take their place: 64 registers of weights and 32 of these leave room for rows asked for ahead.
// 128 registers a lane (four waves on each SIMD at 256 channels): addresses are computed again (fresh) instead of held.
// Bound by the issue of vector instructions (about 60 and 8 transcendentals per element, 80 % of the time) on 250 of 256 CUs; a step takes 11 us whoever takes it, of which the state
// in front costs 1.  16384 tokens of 16 uneven sequences, 10 blocks of 256: walks 224 us on 160 CUs, the longest 28 steps; steps by any workgroup 135.  5 sequences, 4 blocks: 106 -> 91 (in
// segments with a summary pass before).  One sequence of 2000 tokens, 4 blocks: 45 -> 38.
constexpr int kWaitLimit = 1 << 22;                  // polls of about a microsecond
constexpr int kAhead = 2;                            // rows of u asked for ahead of the products that take them
constexpr size_t kStepInfoBytes = 2 * 8 * 4;
template <int KS> constexpr size_t chain_lds_bytes(int taps) { return scan_lds_bytes<KS>(taps) + kStepInfoBytes; }

__device__ __forceinline__ void vm_drain() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// what workgroups hand each other: written through to memory and read past the caches
template <typename T> __device__ __forceinline__ void st_through(T* p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename T> __device__ __forceinline__ T ld_through(const T* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// decay a = exp(-rate r) and input sqrt(1 - a^2) i u; 1 - a^2 by its series where it would cancel
__device__ __forceinline__ void decay_and_input_both(float rate, float r, float ig, float u, float& a, float& b) {
    const float t = (-kLog2e * rate) * r, y = t * (-2.f / kLog2e);
    a = fast_exp2(t);
    float series = y * (1.f + y * (-1.f / 2 + y * ((y - 4.f) * (-1.f / 24))));
    asm volatile("" : "+v"(series));                 // (both, and a choice: branches around either cost more)
    b = fast_sqrt(y < 0.06f ? series : 1.f - a * a) * ig * u;
}

// the links of a launch (a.links): a ticket per block; a word per (channels of a wave, step): 0, 1 = its pair is there, 2 = the state behind it is; what the steps are; the pairs;
// the states
constexpr int kTicketWords = 16, kStepWords = 8;
struct Links {
    uint32_t* tickets;
    uint32_t* flags;                                 // [width / 16][steps]
    int* steps;                                      // [steps][8]: first row, rows (0: past the last step), tokens of the portion in front, slot, position of the portion's first token > 0, last of it
    uint64_t* pairs;                                 // [steps][width]: product of decays | end value << 32
    float* after;                                    // [steps][width]
};
__host__ __device__ __forceinline__ int64_t link_words(int blocks, int64_t width, int64_t steps) { return (blocks * (int64_t)kTicketWords + width / 16 * steps + 63) / 64 * 64; }
__device__ __forceinline__ Links links_of(const RglruArgs& a) {
    Links l;
    l.tickets = reinterpret_cast<uint32_t*>(a.links);
    l.flags = l.tickets + a.blocks * kTicketWords;
    l.steps = reinterpret_cast<int*>(l.tickets + link_words(a.blocks, a.width, a.max_steps));
    l.pairs = reinterpret_cast<uint64_t*>(l.steps + (int64_t)a.max_steps * kStepWords);
    l.after = reinterpret_cast<float*>(l.pairs + (int64_t)a.max_steps * a.width);
    return l;
}

// In front of the scan: tickets and flags are cleared and the steps listed.  Up to 256 segments: the first steps of all portions, then the second ones, and so on (the state in
// front of a step has then mostly been published when the step is drawn); more of them: in the table's order, by the first workgroup.
__global__ __launch_bounds__(256) void rglru_steps_kernel(const RglruArgs a) {
    const Links links = links_of(a);
    const int tid = threadIdx.x, few = a.n_chunks <= 256, id0 = blockIdx.x * 256 + tid, ids = few ? gridDim.x * 256 : 256;
    if (!few && blockIdx.x > 0) {
        if (id0 < link_words(a.blocks, a.width, a.max_steps) / 4) reinterpret_cast<u32x4*>(links.tickets)[id0] = u32x4{0, 0, 0, 0};
        return;
    }
    __shared__ int upto[256];                        // steps up to and with each of 256 segments
    __shared__ int2 part[256];                       // steps of its portion in front of each, its own
    __shared__ u32x4 what[256];                      // first row, rows, slot, 1: not the portion's start but the sequence's, 2: the portion's last
    int before = 0;
    for (int group = 0; group < a.n_chunks; group += 256) {
        const int seg = group + tid;
        const bool have = seg < a.n_chunks;
        const int* row = a.chunks + (int64_t)(have ? seg : group) * 4;
        const int first = row[0], n = have ? row[1] : 0, seq = row[2], kth = row[3], own = n > 0 ? (n + CH - 1) / CH : 0;
        const bool more = seg + 1 < a.n_chunks && row[6] == seq && row[5] > 0;
        const int slot = a.state_slots[seq];
        const bool old = n > 0 && kth == 0 && a.positions[first] > 0;
        int sum = own;
        for (int d = 1; d < 64; d *= 2) {
            const int o = __shfl_up(sum, d);
            if ((tid & 63) >= d) sum += o;
        }
        part[tid] = int2{kth * (a.segment / CH), own};
        upto[tid] = sum;
        __syncthreads();
        const int w0 = upto[63], w1 = w0 + upto[127], w2 = w1 + upto[191], all = w2 + upto[255];
        __syncthreads();
        upto[tid] = sum + (tid < 64 ? 0 : tid < 128 ? w0 : tid < 192 ? w1 : w2);
        what[tid] = u32x4{(uint32_t)first, (uint32_t)n, (uint32_t)slot, (uint32_t)old + 2 * !more};
        if (group == 0 && id0 < link_words(a.blocks, a.width, a.max_steps) / 4) reinterpret_cast<u32x4*>(links.tickets)[id0] = u32x4{0, 0, 0, 0};
        __syncthreads();
        for (int s = id0; s < all && before + s < a.max_steps; s += ids) {     // (more than max_steps: segments that share rows, which is no table)
            int k = 0;
            for (int d = 128; d > 0; d /= 2)
                if (upto[k + d - 1] <= s) k += d;
            const u32x4 w = what[k];
            const int t0 = (s - (k ? upto[k - 1] : 0)) * CH, left = (int)w[1] - t0, step = part[k].x + t0 / CH;
            int at = before + s;                     // its place among the steps
            if (few && all <= a.max_steps) {
                at = 0;
#pragma unroll 8
                for (int o = 0; o < a.n_chunks; ++o) {
                    const int d = step - part[o].x;
                    at += (d < 0 ? 0 : d < part[o].y ? d : part[o].y) + (o < k && d >= 0 && d < part[o].y);
                }
            }
            int* to = links.steps + (int64_t)at * kStepWords;
            *reinterpret_cast<u32x4*>(to) = u32x4{w[0] + t0, (uint32_t)(left < CH ? left : CH), (uint32_t)step * CH, w[2]};
            *reinterpret_cast<u32x4*>(to + 4) = u32x4{step == 0 && (w[3] & 1), left <= CH && (w[3] & 2), (uint32_t)(before + s), 0u};
        }
        before += all;
        __syncthreads();
    }
    for (int s = before + id0; s < a.max_steps; s += ids) links.steps[(int64_t)s * kStepWords + 1] = 0;
}

template <int KS>                                    // block = 32 KS; grid blocks x workgroups per block, blocks fastest
__global__ __launch_bounds__(128 * KS, 4) void rglru_chain_kernel(const RglruArgs a) {
    constexpr int BLOCK = 32 * KS, OCT = 4 * KS, WAVES = 2 * KS, THREADS = 64 * WAVES, LD = BLOCK + 8;
    constexpr int XINS = ((CH + HALO) * OCT + 63) / 64;                        // DMA instructions; y has two a wave
    // y image: pieces of 8 channels in order, odd rows' swapped in pairs, 32 spare bytes behind 64 where a row is a power of two: 16 rows' pieces miss each
    // other's banks, and the four rows of a lane lie at fixed distances
    constexpr int YDMA = scan_y_dma<KS>(), YBUF = 4 * KS * YDMA;
    static_assert(XINS <= 3 * WAVES && CH * OCT == 2 * THREADS);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    uint16_t* x_lds = reinterpret_cast<uint16_t*>(smem);                       // [HALO + CH][BLOCK]
    uint16_t* u_lds = x_lds + scan_x_bytes<KS>() / 2;                          // [CH][LD]
    uint16_t* y_lds = u_lds + CH * LD;                                         // [2][YBUF]; out behind the scan
    float* w_lds = reinterpret_cast<float*>(y_lds + 2 * YBUF);                 // [taps + 1][BLOCK]: taps, then the bias
    int* info_lds = reinterpret_cast<int*>(w_lds + (a.taps + 1) * BLOCK);      // [2][8]: a step as it is listed, its number behind it (< 0: none)
    const int blk = blockIdx.x % a.blocks, c0 = blk * BLOCK;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const auto lane_now = [&]() __attribute__((always_inline)) { return fresh(tid) & 63; };
    const Links links = links_of(a);
    const uint16_t* yx = reinterpret_cast<const uint16_t*>(a.yx);
    auto dma = [&](const char* src, void* dst) __attribute__((always_inline)) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
    };
    const uint32_t stride = (uint32_t)a.yx_stride * 2;                         // bytes; a step's 72 rows are reached by 32-bit offsets from its first one

    // rows of u and y (and out) in LDS: four tiles of 16, row 4 q + j of tile m holds token 16 q + 4 m + j, so that a lane of the accumulators holds 16 consecutive tokens
    const auto token = [](int r) { return 16 * (r >> 2 & 3) + 4 * (r >> 4) + (r & 3); };
    const auto place = [](int row, int p) { const int s = row * OCT + p; return s / 64 * YDMA + s % 64 * 8; };
    auto draw = [&]() __attribute__((always_inline)) {                         // (a wave)
        uint32_t t = 0;
        if (lane_now() == 0) t = __hip_atomic_fetch_add(links.tickets + blk * kTicketWords, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return (int)__builtin_amdgcn_readfirstlane(t);
    };
    auto look_up = [&](int number) __attribute__((always_inline)) {            // lanes 0..5: what the step is
        return links.steps[(int64_t)(number < a.max_steps ? number : a.max_steps - 1) * kStepWords + (lane_now() & 7)];
    };
    auto note = [&](int number, int word, int which) __attribute__((always_inline)) {
        const int ln = lane_now(), cnt = __builtin_amdgcn_readlane(word, 1);
        if (ln < 8) info_lds[8 * which + ln] = ln == 6 && (number >= a.max_steps || cnt <= 0) ? -1 : word;
    };
    struct Step { int row, cnt, off, slot, old, last, id; };
    auto read_info = [&](int which) __attribute__((always_inline)) {
        const int* p = info_lds + 8 * which;
        const auto get = [&](int i) { return __builtin_amdgcn_readfirstlane(p[i]); };
        return Step{get(0), get(1), get(2), get(3), get(4), get(5), get(6)};
    };

    auto stage_x = [&](const Step& s) __attribute__((always_inline)) {         // the step's rows and HALO in front of them, clamped to the portion's rows that exist
        const char* base = reinterpret_cast<const char*>(yx + (int64_t)(s.row - HALO) * a.yx_stride + a.width + c0);
        const int lo = HALO - s.off, hi = s.cnt - 1 + HALO;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int ins = wave + WAVES * j;
            if (ins < XINS) {
                const int e = ins * 64 + lane_now(), r = e / OCT, d = r < lo ? lo : (r > hi ? hi : r);
                dma(base + ((uint32_t)d * stride + (uint32_t)(e % OCT) * 16), x_lds + ins * 512);
            }
        }
    };
    auto stage_y = [&](const Step& s, uint16_t* image) __attribute__((always_inline)) {
        const char* base = reinterpret_cast<const char*>(yx + (int64_t)s.row * a.yx_stride + c0);
        const int hi = s.cnt - 1;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int ins = wave + WAVES * j, e = ins * 64 + lane_now(), r = e / OCT, t = token(r), d = t < hi ? t : hi;
            dma(base + ((uint32_t)d * stride + (uint32_t)((e % OCT) ^ (r & 1)) * 16), image + ins * YDMA);
        }
    };
    auto ring_rows = [&](const Step& s) __attribute__((always_inline)) {       // a portion's first step: inputs in front of it from the ring, zero in front of the sequence
        const int64_t pos0 = s.old ? a.positions[s.row] : 0;
        for (int e = fresh(tid); e < (a.taps - 1) * OCT; e += THREADS) {
            const int back = e / OCT + 1, o = e % OCT;
            const uint16_t* p = conv_input<uint16_t>(a, s.row, -back, pos0, s.slot, c0 + o * 8);
            *reinterpret_cast<u32x4*>(x_lds + (HALO - back) * BLOCK + o * 8) = p ? *reinterpret_cast<const u32x4*>(p) : u32x4{0, 0, 0, 0};
        }
        lds_barrier();
    };
    auto convolve = [&]() __attribute__((always_inline)) {                     // x -> u, eight tokens x 2 channels a thread
        const int id = fresh(tid), o = 2 * (id % (16 * KS)), t = 8 * (id / (16 * KS));
        const uint16_t* xp = x_lds + (HALO + t - (a.taps - 1)) * BLOCK + o;
        const float* wp = w_lds + o;
        const f32x2 bias = *reinterpret_cast<const f32x2*>(wp + a.taps * BLOCK);
        float acc[8][2];
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i][0] = bias[0], acc[i][1] = bias[1];
        if (a.taps == 4) {
            f32x2 w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = *reinterpret_cast<const f32x2*>(wp + j * BLOCK);
#pragma unroll
            for (int s = 0; s < 11; ++s) {
                const uint32_t v = *reinterpret_cast<const uint32_t*>(xp + s * BLOCK);
                const float lo = bf16_lo(v), hi = bf16_hi(v);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (s - j >= 0 && s - j < 8) {
                        acc[s - j][0] += w[j][0] * lo;
                        acc[s - j][1] += w[j][1] * hi;
                    }
            }
        } else {
            for (int j = 0; j < a.taps; ++j) {
                const f32x2 w = *reinterpret_cast<const f32x2*>(wp + j * BLOCK);
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const uint32_t v = *reinterpret_cast<const uint32_t*>(xp + (i + j) * BLOCK);
                    acc[i][0] += w[0] * bf16_lo(v);
                    acc[i][1] += w[1] * bf16_hi(v);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) *reinterpret_cast<uint32_t*>(u_lds + (4 * (t & 8) + t / 16 * 4 + 16 * (i / 4) + i % 4) * LD + o) = pack_bf16x2(acc[i][0], acc[i][1]);
    };

    if (wave == 0) {
        const int first = draw();
        note(first, look_up(first), 0);
    }
    // ---- this wave's 16 channels
    const int lq = tid & 15, lg = tid >> 4 & 3, ch = c0 + 16 * wave + lq;
    bf16x8 wr[KS], wi[KS];
    {
        const uint16_t* pr = reinterpret_cast<const uint16_t*>(a.ra) + (int64_t)ch * BLOCK + 8 * lg;
        const uint16_t* pi = reinterpret_cast<const uint16_t*>(a.ri) + (int64_t)ch * BLOCK + 8 * lg;
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            wr[k] = *reinterpret_cast<const bf16x8*>(pr + 32 * k);
            wi[k] = *reinterpret_cast<const bf16x8*>(pi + 32 * k);
        }
    }
    const float rb = -kLog2e * a.ra_b[ch], ib = -kLog2e * a.ri_b[ch], rate = a.rate[ch];
    for (int e = tid; e < (a.taps + 1) * BLOCK; e += THREADS)
        w_lds[e] = e < a.taps * BLOCK ? a.conv_w[(int64_t)(e / BLOCK) * a.width + c0 + e % BLOCK] : a.conv_b[c0 + e % BLOCK];
    lds_barrier();                                   // (the weights are on their way)
    Step now = read_info(0);
    if (now.id < 0) return;
    stage_x(now);
    stage_y(now, y_lds);
    if (wave == 0) {                                 // (a workgroup holds one step more than it works on)
        const int second = draw();
        note(second, look_up(second), 1);
    }
    uint32_t* flags = links.flags + (int64_t)(blk * WAVES + wave) * a.max_steps;
    vm_drain();
    lds_barrier();
    if (now.off == 0) ring_rows(now);
    convolve();
    lds_barrier();
    for (int which = 0;; which ^= 1) {
        const Step next = read_info(which ^ 1);
        if (next.id >= 0) {                          // (x has become u, and the rows that went out last are gone)
            stage_x(next);
            stage_y(next, y_lds + (which ^ 1) * YBUF);
        }
        uint16_t* y_now = y_lds + which * YBUF;
        // gates of all tokens first, then decays and inputs in their place: av, sv compose this lane's 16 tokens from its first one on
        f32x4 av[4], sv[4];
        {
            const int ln = lane_now();
            const uint16_t* u_row = u_lds + (ln & 15) * LD + 8 * (ln >> 4);
#pragma unroll
            for (int m = 0; m < 4; ++m) av[m] = sv[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < KS; ++k)
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const bf16x8 ua = *reinterpret_cast<const bf16x8*>(u_row + 16 * m * LD + 32 * k);
                    av[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ua, wr[k], av[m], 0, 0, 0);
                    sv[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ua, wi[k], sv[m], 0, 0, 0);
                }
            __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);             // (rows of u some products ahead)
#pragma unroll
            for (int k = 0; k < 4 * KS - kAhead; ++k) {
                __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, 2 * kAhead, 0);
        }
        float ca, cs, ba = 1.f, bs = 0.f;            // the whole step's pair, and what is in front of this lane's tokens
        {
            const int ln = lane_now(), lg = ln >> 4;
            const uint16_t* u_own = u_lds + 4 * lg * LD + 16 * wave + (ln & 15);
            float uu[4], un[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) uu[i] = act_ld(u_own + i * LD);
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                if (m < 3)
#pragma unroll
                    for (int i = 0; i < 4; ++i) un[i] = act_ld(u_own + (16 * m + 16 + i) * LD);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float rg = fast_rcp(1.f + fast_exp2(av[m][i] * -kLog2e + rb)), ig = fast_rcp(1.f + fast_exp2(sv[m][i] * -kLog2e + ib));
                    float dec, inp;
                    decay_and_input_both(rate, rg, ig, uu[i], dec, inp);
                    av[m][i] = dec;
                    sv[m][i] = inp;
                }
                if (now.cnt < CH) {                  // (tokens past the end leave the state alone)
                    asm volatile("");                // (a branch: the comparisons are wanted in the last step only)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (16 * lg + 4 * m + i >= now.cnt) av[m][i] = 1.f, sv[m][i] = 0.f;
                }
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (m + i > 0) {
                        const float fa = i ? av[m][i - 1] : av[m - 1][3], fs = i ? sv[m][i - 1] : sv[m - 1][3];
                        sv[m][i] += av[m][i] * fs;
                        av[m][i] *= fa;
                    }
#pragma unroll
                for (int i = 0; i < 4; ++i) uu[i] = un[i];
            }
            // across the four lane groups (16 tokens each): e = the even group of the pair, then both pairs' totals to everyone
            const auto swap16 = [](float v) { return __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false); };
            const auto swap32 = [](float v) { return __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false); };
            const bool odd = lg & 1;
            const float pa = av[3][3], ps = sv[3][3];
            const float ea = __uint_as_float(swap16(pa)[0]), es = __uint_as_float(swap16(ps)[0]);
            const float ia = odd ? pa * ea : pa, is = odd ? pa * es + ps : ps;                  // inclusive inside the pair
            const auto ha = swap32(__uint_as_float(swap16(ia)[1])), hs = swap32(__uint_as_float(swap16(is)[1]));
            const float la = __uint_as_float(ha[0]), ls = __uint_as_float(hs[0]), ua_ = __uint_as_float(ha[1]), us_ = __uint_as_float(hs[1]);
            if (lg >= 2) ba = la, bs = ls;
            bs = odd ? ea * bs + es : bs;
            ba = odd ? ea * ba : ba;
            cs = ua_ * ls + us_;
            ca = ua_ * la;
        }
        // ---- the step's pair, or the state behind it where the one in front is known
        constexpr float kLeast = 1.4e-45f;           // (a product that has vanished: not zero, an infinite state stays one)
        if (ca == 0.f) ca = kLeast;
        const int64_t at = (int64_t)now.id * a.width + c0 + 16 * wave;          // (the same in all lanes)
        float h = 0.f;                               // the state in front of the step
        int drawn = 0, drawn_word = 0;               // (wave 0) the step behind the next one
        {
            const int ln = lane_now();
            if (now.off == 0) {
                if (now.old && now.slot >= 0) h = a.state[(int64_t)now.slot * a.width + c0 + 16 * wave + (ln & 15)];
                if (ln < 16) st_through(links.after + at + ln, ca * h + cs);
            } else if (ln < 16) {
                st_through(links.pairs + at + ln, (uint64_t)__float_as_uint(ca) | (uint64_t)__float_as_uint(cs) << 32);
            }
            if (wave == 0 && next.id >= 0) drawn = draw();
            vm_drain();                              // it is there; so are the next step's x and this one's y
            if (ln == 0) st_through(flags + now.id, now.off == 0 ? 2u : 1u);
        }
        if (wave == 0 && next.id >= 0) drawn_word = look_up(drawn);
        if (now.off > 0) {
            const int ln = lane_now(), depth = now.off / CH < now.id ? now.off / CH : now.id;
            int p = 0;
            bool there = false;
            for (int tries = 0; tries < kWaitLimit && !there && depth; ++tries) {
                if (tries) __builtin_amdgcn_s_sleep(1);
                const uint32_t f = ln < depth ? ld_through(flags + now.id - 1 - ln) : 3u;
                const uint64_t whole = __ballot(f == 2u), none = __ballot(f == 0u);
                p = whole ? __builtin_ctzll(whole) : 0;
                there = whole && !(none & ((1ull << p) - 1));
            }
            asm volatile("" ::: "memory");
            h = ld_through(links.after + (at - (int64_t)(p + 1) * a.width) + (ln & 15));
            for (int k = p; k > 0; k -= 8) {
                uint64_t pair[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) pair[i] = ld_through(links.pairs + (at - (int64_t)(k > i ? k - i : 1) * a.width) + (ln & 15));
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (k > i) h = __uint_as_float((uint32_t)pair[i]) * h + __uint_as_float((uint32_t)(pair[i] >> 32));
            }
            if (!there) h = __uint_as_float(0x7FC00000u);
            if (ln < 16) st_through(links.after + at + ln, ca * h + cs);
        }
        if (__any(__builtin_isinf(h))) {
            if (ba == 0.f) ba = kLeast;
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (av[m][i] == 0.f) av[m][i] = kLeast;
        }
        {
            const int ln = lane_now(), lq = ln & 15, lg = ln >> 4, piece = 2 * wave + (lq >> 3);
            uint16_t* y_even = y_now + place(4 * lg, piece) + (lq & 7);        // this lane's channel in rows 4 lg and, by fixed distances, 4 lg + 2
            uint16_t* y_odd = y_now + place(4 * lg, piece ^ 1) + (lq & 7);     // ... and, likewise, in 4 lg + 1 and 4 lg + 3
            const auto off = [](int m, int i) { return m * KS * YDMA + (KS == 8 ? i / 2 * YDMA : i / 2 * 2 * BLOCK); };
            const float before = ba * h + bs;
            float yv[4], yn[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) yv[i] = act_ld(i & 1 ? y_odd + off(0, i) + BLOCK : y_even + off(0, i));
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                if (m < 3)
#pragma unroll
                    for (int i = 0; i < 4; ++i) yn[i] = act_ld(i & 1 ? y_odd + off(m + 1, i) + BLOCK : y_even + off(m + 1, i));
#pragma unroll
                for (int i = 0; i < 4; i += 2) {
                    const uint32_t two = pack_bf16x2((av[m][i] * before + sv[m][i]) * fast_gelu(yv[i]), (av[m][i + 1] * before + sv[m][i + 1]) * fast_gelu(yv[i + 1]));
                    y_even[off(m, i)] = (uint16_t)two;
                    y_odd[off(m, i) + BLOCK] = (uint16_t)(two >> 16);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) yv[i] = yn[i];
            }
        }
        if (now.last) {
            const int slot = now.slot, ln = lane_now();
            if (slot >= 0) {
                if (ln < 16) a.state[(int64_t)slot * a.width + c0 + 16 * wave + ln] = ca * h + cs;
                const int portion = now.off + now.cnt, keep = portion < a.taps ? portion : a.taps;
                for (int e = fresh(tid); e < keep * OCT; e += THREADS) {       // (its first step, which has read the ring, has published)
                    const int row = now.row + now.cnt - 1 - e / OCT, c = c0 + e % OCT * 8;
                    *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(a.conv_state) + ((int64_t)slot * a.taps + (int)(a.positions[row] % a.taps)) * a.width + c) =
                        *reinterpret_cast<const u32x4*>(yx + (int64_t)row * a.yx_stride + a.width + c);
                }
            }
        }
        if (wave == 0 && next.id >= 0) note(drawn, drawn_word, which);
        if (now.off > 0) {
            vm_drain();
            if (lane_now() == 0) st_through(flags + now.id, 2u);
        }
        lds_barrier();                               // out is whole, u is free, the next x and y are there for everyone
        {
            char* out = reinterpret_cast<char*>(reinterpret_cast<uint16_t*>(a.out) + (int64_t)now.row * a.out_stride + c0);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int e = fresh(tid) + j * THREADS, r = e / OCT, p = e % OCT, t = token(r);
                if (t < now.cnt)
                    *reinterpret_cast<u32x4*>(out + ((uint32_t)t * (uint32_t)(a.out_stride * 2) + (uint32_t)p * 16)) = *reinterpret_cast<const u32x4*>(y_now + place(r, p ^ (r & 1)));
            }
        }
        if (next.id < 0) break;
        if (next.off == 0) ring_rows(next);
        convolve();
        lds_barrier();
        now = next;
    }
}

// ------------------------------------------------------------------------------------------------ prompt portions, any type and size
// one workgroup per (segment, 64 channels of a diagonal block): gates by plain dot products over LDS tiles, scan by one thread per channel
template <typename T, bool SUMMARY>
__global__ __launch_bounds__(256) void rglru_walk_generic_kernel(const RglruArgs a) {
    constexpr int KT = 32;
    __shared__ float u_t[CH][KT + 1];
    __shared__ float wr_t[64][KT + 1], wi_t[64][KT + 1];
    __shared__ float dec[CH][65], inp[CH][65];
    const int seg = blockIdx.x;
    const int tiles = (a.block + 63) / 64, blk = blockIdx.y / tiles, n0 = (blockIdx.y % tiles) * 64;
    const int row0 = a.chunks[seg * 4], n = a.chunks[seg * 4 + 1], seq = a.chunks[seg * 4 + 2], kth = a.chunks[seg * 4 + 3];
    const bool more = seg + 1 < a.n_chunks && a.chunks[seg * 4 + 6] == seq;
    if ((SUMMARY && !more) || portion_without_rows(n, kth)) return;
    const int off0 = kth * a.segment, seq_row0 = row0 - off0;
    const int slot = a.state_slots[seq];
    const int64_t pos0 = a.positions[seq_row0];
    const T* ra = reinterpret_cast<const T*>(a.ra) + (int64_t)blk * a.block * a.block;
    const T* ri = reinterpret_cast<const T*>(a.ri) + (int64_t)blk * a.block * a.block;
    const int tid = threadIdx.x, c = tid & 63, tq = tid >> 6;
    const int ch = blk * a.block + n0 + c;
    const bool live = n0 + c < a.block;
    auto conv_at = [&](int t, int cc) {              // t: tokens behind the segment's first
        float s = a.conv_b[cc];
        for (int j = 0; j < a.taps; ++j) {
            const T* p = conv_input<T>(a, seq_row0, off0 + t - (a.taps - 1) + j, pos0, slot, cc);
            if (p) s += a.conv_w[(int64_t)j * a.width + cc] * act_ld(p);
        }
        return act_round(s, (const T*)nullptr);
    };
    float ca = 1.f, cs = live ? walk_start(a, SUMMARY, more, seg, kth, slot, pos0, ch) : 0.f;
    if (SUMMARY && kth == 0 && live && tid < 64) a.a_cum[(int64_t)seg * a.width + ch] = cs;
    for (int t0 = 0; t0 < n; t0 += CH) {
        const int cnt = n - t0 < CH ? n - t0 : CH;
        float gr[16], gi[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) gr[i] = gi[i] = 0.f;
        for (int k0 = 0; k0 < a.block; k0 += KT) {
            for (int e = tid; e < CH * KT; e += 256) {
                const int t = e / KT, k = e % KT;
                u_t[t][k] = t < cnt ? conv_at(t0 + t, blk * a.block + k0 + k) : 0.f;
            }
            for (int e = tid; e < 64 * KT; e += 256) {
                const int o = e / KT, k = e % KT;
                const bool ok = n0 + o < a.block;
                wr_t[o][k] = ok ? act_ld(ra + (int64_t)(n0 + o) * a.block + k0 + k) : 0.f;
                wi_t[o][k] = ok ? act_ld(ri + (int64_t)(n0 + o) * a.block + k0 + k) : 0.f;
            }
            __syncthreads();
            for (int k = 0; k < KT; ++k) {
                const float wr = wr_t[c][k], wi = wi_t[c][k];
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const float u = u_t[tq * 16 + i][k];
                    gr[i] += wr * u;
                    gi[i] += wi * u;
                }
            }
            __syncthreads();
        }
        if (live) {
            const float rb = a.ra_b[ch], ib = a.ri_b[ch], rate = a.rate[ch];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int t = tq * 16 + i;
                if (t < cnt) {
                    // (accurate exponentials: this form also serves the true fp32 model)
                    const float r = 1.f / (1.f + expf(-(gr[i] + rb))), ig = 1.f / (1.f + expf(-(gi[i] + ib)));
                    const float log_a = -rate * r;
                    dec[t][c] = expf(log_a);
                    inp[t][c] = sqrtf(-expm1f(2.f * log_a)) * ig * conv_at(t0 + t, ch);
                }
            }
        }
        __syncthreads();
        if (tid < 64 && live)
            for (int t = 0; t < cnt; ++t) {
                cs = dec[t][c] * cs + inp[t][c];
                ca *= dec[t][c];
                inp[t][c] = cs;
            }
        __syncthreads();
        if (!SUMMARY && live)
            for (int t = tq; t < cnt; t += 4) {
                const float y = act_ld(reinterpret_cast<const T*>(a.yx) + (int64_t)(row0 + t0 + t) * a.yx_stride + ch);
                act_st(reinterpret_cast<T*>(a.out) + (int64_t)(row0 + t0 + t) * a.out_stride + ch, inp[t][c] * gelu_tanh_f(y));
            }
        __syncthreads();
    }
    if (tid < 64 && live && (SUMMARY || !more)) {
        a.s_loc[(int64_t)seg * a.width + ch] = cs;
        if (SUMMARY && kth) a.a_cum[(int64_t)seg * a.width + ch] = ca;
    }
}

// behind the walks: every sequence's last segment hands its end value to the state and the portion's last inputs to the ring
template <typename T>
__global__ __launch_bounds__(256) void rglru_keep_kernel(const RglruArgs a) {
    const int seg = blockIdx.x, ch = (blockIdx.y * 256 + threadIdx.x) * 4;
    const int row0 = a.chunks[seg * 4], n = a.chunks[seg * 4 + 1], seq = a.chunks[seg * 4 + 2], kth = a.chunks[seg * 4 + 3];
    const int slot = a.state_slots[seq];
    if (ch >= a.width || slot < 0 || portion_without_rows(n, kth) || (seg + 1 < a.n_chunks && a.chunks[seg * 4 + 6] == seq)) return;
    *reinterpret_cast<f32x4*>(a.state + (int64_t)slot * a.width + ch) = *reinterpret_cast<const f32x4*>(a.s_loc + (int64_t)seg * a.width + ch);
    const int portion = kth * a.segment + n, keep = portion < a.taps ? portion : a.taps;
    for (int j = 0; j < keep; ++j) {
        const int row = row0 + n - 1 - j;
        act_st4(reinterpret_cast<T*>(a.conv_state) + ((int64_t)slot * a.taps + (int)(a.positions[row] % a.taps)) * a.width + ch,
                act_ld4(reinterpret_cast<const T*>(a.yx) + (int64_t)row * a.yx_stride + a.width + ch));
    }
}

// ------------------------------------------------------------------------------------------------ one token per sequence (bf16)
// grid (width / 16 channel tiles, 32-row tiles); the 4 waves split the contraction over the diagonal block and add up through LDS.
// Everything whose address needs no result of this launch (gate weights, states, y) is asked for before the convolution.
template <int KW>                                    // contraction steps of 32 per wave held in registers (0: a loop)
__global__ __launch_bounds__(256) void rglru_step_kernel(const RglruArgs a, const int rows) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int per = a.block / 16, blk = blockIdx.x / per, nt = blockIdx.x % per;
    const int r0 = blockIdx.y * 32, nr = rows - r0 < 32 ? rows - r0 : 32;
    const int ld = a.block + 8, oct = a.block / 8, ksteps = a.block / 32;
    uint16_t* u_lds = reinterpret_cast<uint16_t*>(smem);                        // [32][block + 8]
    f32x4* red = reinterpret_cast<f32x4*>(smem + 32 * ld * 2);                  // [wave][2 gates x 2 row tiles][64 lanes]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lq = lane & 15, lg = lane >> 4;
    const uint16_t* yx = reinterpret_cast<const uint16_t*>(a.yx);
    const uint16_t* wr = reinterpret_cast<const uint16_t*>(a.ra) + ((int64_t)blk * a.block + 16 * nt + lq) * a.block + 8 * lg;
    const uint16_t* wi = reinterpret_cast<const uint16_t*>(a.ri) + ((int64_t)blk * a.block + 16 * nt + lq) * a.block + 8 * lg;
    bf16x8 br[KW > 0 ? KW : 1], bi[KW > 0 ? KW : 1];
#pragma unroll
    for (int k = 0; k < KW; ++k) {
        const int ks = wave + 4 * k < ksteps ? wave + 4 * k : 0;
        br[k] = *reinterpret_cast<const bf16x8*>(wr + 32 * ks);
        bi[k] = *reinterpret_cast<const bf16x8*>(wi + 32 * ks);
    }
    // this thread's two outputs: (row tile m, lane of the C layout, half of its 4 rows)
    const int m = tid >> 7, cl = (tid >> 1) & 63, half = tid & 1;
    const int cb = 16 * nt + (cl & 15), ch0 = blk * a.block + cb;
    int slot[2];
    int64_t pos[2];
    float old[2], yv[2];
    uint16_t xin[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = 16 * m + 4 * (cl >> 4) + 2 * half + i, rc = r0 + (row < nr ? row : 0);
        slot[i] = a.state_slots[rc];
        pos[i] = a.positions[rc];
        yv[i] = act_ld(yx + (int64_t)rc * a.yx_stride + ch0);
        xin[i] = yx[(int64_t)rc * a.yx_stride + a.width + ch0];
        old[i] = slot[i] >= 0 ? a.state[(int64_t)slot[i] * a.width + ch0] : 0.f;
        if (pos[i] <= 0) old[i] = 0.f;
    }
    const float rb = a.ra_b[ch0], ib = a.ri_b[ch0], rate = a.rate[ch0];
    for (int e = tid; e < 32 * oct; e += 256) {
        const int row = e / oct, o = e - row * oct;
        u32x4 packed = {0, 0, 0, 0};
        if (row < nr) {
            const int sl = a.state_slots[r0 + row], ch = blk * a.block + o * 8;
            const int64_t ps = a.positions[r0 + row];
            float acc[1][8];
            auto in = [&](int s) { return conv_input<uint16_t>(a, r0 + row, s, ps, sl, ch); };
            if (a.taps == 4) conv_run<4, 1>(a, ch, 4, acc, in);
            else conv_run<0, 1>(a, ch, a.taps, acc, in);
            packed = pack8(acc[0]);
        }
        *reinterpret_cast<u32x4*>(u_lds + row * ld + o * 8) = packed;
    }
    __syncthreads();
    f32x4 g[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) g[q] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto product = [&](int ks, const bf16x8 wr_k, const bf16x8 wi_k) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const bf16x8 ua = *reinterpret_cast<const bf16x8*>(u_lds + (16 * q + lq) * ld + 32 * ks + 8 * lg);
            g[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ua, wr_k, g[q], 0, 0, 0);
            g[2 + q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ua, wi_k, g[2 + q], 0, 0, 0);
        }
    };
    if constexpr (KW > 0) {
#pragma unroll
        for (int k = 0; k < KW; ++k)
            if (wave + 4 * k < ksteps) product(wave + 4 * k, br[k], bi[k]);
    } else {
        for (int ks = wave; ks < ksteps; ks += 4) product(ks, *reinterpret_cast<const bf16x8*>(wr + 32 * ks), *reinterpret_cast<const bf16x8*>(wi + 32 * ks));
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) red[(wave * 4 + q) * 64 + lane] = g[q];
    __syncthreads();
    f32x4 sr = {0.f, 0.f, 0.f, 0.f}, si = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        sr += red[(w * 4 + m) * 64 + cl];
        si += red[(w * 4 + 2 + m) * 64 + cl];
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = 16 * m + 4 * (cl >> 4) + 2 * half + i;
        if (row >= nr) continue;
        float dec, inp;
        decay_and_input(rate, fast_sigmoid((half ? sr[2 + i] : sr[i]) + rb), fast_sigmoid((half ? si[2 + i] : si[i]) + ib), act_ld(u_lds + row * ld + cb), dec, inp);
        const float s = dec * old[i] + inp;
        if (slot[i] >= 0) {
            a.state[(int64_t)slot[i] * a.width + ch0] = s;
            reinterpret_cast<uint16_t*>(a.conv_state)[((int64_t)slot[i] * a.taps + (int)(pos[i] % a.taps)) * a.width + ch0] = xin[i];
        }
        const float o = s * fast_gelu(yv[i]);
        if (a.out) act_st(reinterpret_cast<uint16_t*>(a.out) + (int64_t)(r0 + row) * a.out_stride + ch0, o);
        if (a.out_packed) act_st(reinterpret_cast<uint16_t*>(a.out_packed) + pack_index(r0 + row, ch0, a.width), o);
    }
}

constexpr size_t kMaxLds = 160 * 1024;
size_t walk_lds(int block) { return (size_t)CH * ((block + 8) + ((block < kGroup ? block : kGroup) + 8)) * 2; }
size_t step_lds(int block) { return (size_t)32 * (block + 8) * 2 + 16 * 64 * sizeof(f32x4); }
template <bool SUMMARY, int KS>
bool scan_ks(const RglruArgs& a, hipStream_t stream) {
    const size_t lds = scan_lds_bytes<KS>(a.taps);
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(rglru_scan_kernel<KS, SUMMARY>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds);
    // blocks run fastest: workgroups are dealt round-robin over the 8 XCDs, and segments differ in length while the blocks of one do not
    const int deep = (a.n_chunks + 65534) / 65535;
    rglru_scan_kernel<KS, SUMMARY><<<dim3(a.blocks, (a.n_chunks + deep - 1) / deep, deep), 128 * KS, lds, stream>>>(a);
    return true;
}
bool scan_takes(int block, int taps) { return block <= 256 && block % 32 == 0 && taps <= HALO + 1 && chain_lds_bytes<8>(taps) <= kMaxLds; }
bool near_rows(const RglruArgs& a) { return a.yx_stride < 1 << 24 && a.out_stride < 1 << 24; }     // (32-bit row offsets: 72 rows of less than 2^25 bytes)
template <bool SUMMARY>
bool scan(const RglruArgs& a, hipStream_t stream) {
    if (!near_rows(a) || !scan_takes(a.block, a.taps)) return false;
    switch (a.block / 32) {
        case 1: return scan_ks<SUMMARY, 1>(a, stream);
        case 2: return scan_ks<SUMMARY, 2>(a, stream);
        case 3: return scan_ks<SUMMARY, 3>(a, stream);
        case 4: return scan_ks<SUMMARY, 4>(a, stream);
        case 5: return scan_ks<SUMMARY, 5>(a, stream);
        case 6: return scan_ks<SUMMARY, 6>(a, stream);
        case 7: return scan_ks<SUMMARY, 7>(a, stream);
        case 8: return scan_ks<SUMMARY, 8>(a, stream);
        default: return false;
    }
}

template <int KS>
void chain_ks(const RglruArgs& a, hipStream_t stream) {
    const size_t lds = chain_lds_bytes<KS>(a.taps);
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(rglru_chain_kernel<KS>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds);
    rglru_steps_kernel<<<(int)((link_words(a.blocks, a.width, a.max_steps) / 4 + 255) / 256), 256, 0, stream>>>(a);
    // as many workgroups as run at once, and no more than there can be steps
    const int fit = (int)(kMaxLds / lds), per_cu = fit < 8 / KS ? fit : 8 / KS, all = 256 * (per_cu < 1 ? 1 : per_cu) / a.blocks;
    const int each = all < 1 ? 1 : (all < a.max_steps ? all : a.max_steps);
    rglru_chain_kernel<KS><<<a.blocks * each, 128 * KS, lds, stream>>>(a);
}
bool chain(const RglruArgs& a, hipStream_t stream) {
    // (a segment of n rows is ceil(n / CH) steps; the device counts them, so there has to be room for as many as there can be)
    if (!a.links || a.max_steps <= 0 || a.max_steps < a.n_chunks + (int64_t)a.rows / CH || !near_rows(a) || !scan_takes(a.block, a.taps)) return false;
    switch (a.block / 32) {
        case 1: chain_ks<1>(a, stream); break;
        case 2: chain_ks<2>(a, stream); break;
        case 3: chain_ks<3>(a, stream); break;
        case 4: chain_ks<4>(a, stream); break;
        case 5: chain_ks<5>(a, stream); break;
        case 6: chain_ks<6>(a, stream); break;
        case 7: chain_ks<7>(a, stream); break;
        default: chain_ks<8>(a, stream);
    }
    return true;
}

template <bool SUMMARY>
int walk(const RglruArgs& a, int f32, int generic, hipStream_t stream) {
    const size_t lds = walk_lds(a.block);
    if (f32 || generic == 1 || lds > kMaxLds) {
        const dim3 grid(a.n_chunks, a.blocks * ((a.block + 63) / 64));
        if (f32) rglru_walk_generic_kernel<float, SUMMARY><<<grid, 256, 0, stream>>>(a);
        else rglru_walk_generic_kernel<uint16_t, SUMMARY><<<grid, 256, 0, stream>>>(a);
    } else if (generic == 2 || !scan<SUMMARY>(a, stream)) {
        const int waves = a.block < kGroup ? a.block / 16 : kGroup / 16;
        if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(rglru_walk_kernel<SUMMARY>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds);
        rglru_walk_kernel<SUMMARY><<<dim3(a.n_chunks, a.blocks * ((a.block + kGroup - 1) / kGroup)), waves * 64, lds, stream>>>(a);
    }
    return check_launch("rglru_walk");
}

template <int KW>
void step_kw(const RglruArgs& a, int rows, hipStream_t stream) {
    const size_t lds = step_lds(a.block);
    if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(rglru_step_kernel<KW>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds);
    rglru_step_kernel<KW><<<dim3(a.blocks * (a.block / 16), (rows + 31) / 32), 256, lds, stream>>>(a, rows);
}

}  // namespace

bool rglru_step_supported(int block) { return step_lds(block) <= kMaxLds; }
int64_t rglru_link_bytes(int block, int blocks, int taps, int max_steps, int f32) {
    if (f32 || !scan_takes(block, taps) || max_steps <= 0) return 0;
    const int64_t width = (int64_t)block * blocks;
    return 4 * (link_words(blocks, width, max_steps) + (int64_t)kStepWords * max_steps) + 12 * width * max_steps;
}

// Whole portions that one workgroup each walks better than any takes their steps, a walk has no list of steps and no tickets to wait for:
// - portions of a few steps.  In microseconds, at blocks of 256 channels, a walk of k steps takes 14 + 7.4 k while all have a CU of their own (28 of 40 portions of 50 tokens, 4
//   blocks; 42 of 20 of 100, 10 blocks), 16 + 17 k in two rounds; the chain 21 + 11 per round of steps (33 and 43 there).  From five steps on the chain is ahead (47 against 32 of
//   10 portions of 200 tokens, 4 blocks);
// - narrower blocks whose walks fill half of the GPU's waves (16 portions of 1024 tokens: 64 blocks of 32 channels 91 against 103, 16 of 128 93 against 98, 10 of 192, which
//   do not, 120 against 108).
bool whole_walks(const RglruArgs& a) {
    const int64_t k = a.segment / CH, walks = (int64_t)a.n_chunks * a.blocks, ks = a.block / 32;
    if (a.summaries) return false;
    if (ks < 8 && walks * ks >= 1024) return true;
    if (k > 4 || walks > 512) return false;
    const int64_t at_once = a.blocks < 256 ? 256 / a.blocks * a.blocks : a.blocks, steps = (a.max_steps - a.n_chunks / 2) * (int64_t)a.blocks, rounds = (steps + at_once - 1) / at_once;
    return (walks <= 256 ? 14 + 7.4 * k : 16 + 17.0 * k) < 21 + 11.0 * rounds;
}

int launch_rglru_chunks(const RglruArgs& a, int f32, int generic, hipStream_t stream) {
    if (a.n_chunks == 0) return 0;
    if (!f32 && generic == 0 && !whole_walks(a) && chain(a, stream)) return check_launch("rglru_chain");
    int rc = a.summaries ? walk<true>(a, f32, generic, stream) : 0;
    if (!rc) rc = walk<false>(a, f32, generic, stream);
    if (rc) return rc;
    const dim3 grid(a.n_chunks, (a.width / 4 + 255) / 256);
    if (f32) rglru_keep_kernel<float><<<grid, 256, 0, stream>>>(a);
    else rglru_keep_kernel<uint16_t><<<grid, 256, 0, stream>>>(a);
    return check_launch("rglru_keep");
}

int launch_rglru_step(const RglruArgs& a, int rows, hipStream_t stream) {
    if (a.block <= 128) step_kw<1>(a, rows, stream);
    else if (a.block <= 256) step_kw<2>(a, rows, stream);
    else if (a.block <= 512) step_kw<4>(a, rows, stream);
    else step_kw<0>(a, rows, stream);
    return check_launch("rglru_step");
}

}  // namespace nvh
