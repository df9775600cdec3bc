// Selective scan: per channel c and state n, with a step size per (token, channel) and input and output vectors per token,
//   S[c, n] <- exp(dt_c A[c, n]) S[c, n] + dt_c x_c B_n        y_c = sum_n S[c, n] C_n + D_c x_c        out = y silu(z)
// dt = softplus(projection + bias).  Everything but the projections and x is fp32.
//
// Prompt portions (launch_scan_chunks): a workgroup owns one (segment, CHN channels) and takes TT tokens at a time.  dt and dt x are computed once per (token,
// channel) on 16-byte pieces of the rows and left in LDS, next to B and C of the tokens; then NL lanes per channel walk the tokens with NS states each in
// registers; a last pass adds D x, gates and writes 16-byte pieces.  The next tile's rows are fetched while this one is scanned.
// A portion of several segments: a SUMMARY walk leaves every segment's own contribution and its sum of dt (the product of its decays is exp(A sum dt)), a small
// launch turns those into states at segment starts, and the second walk begins there.
// Decoding (launch_scan_step): four states per lane, dt from the projection's low-rank row on the spot, several rows per workgroup so that its weights are read
// once for all of them.
// Per (token, channel, state): one transcendental and four vector instructions: issue-bound, not HBM-bound.  So the walk is written for few instructions and no
// waits: every load is unconditional (rows past the end repeat the last one; a load behind a branch makes the compiler wait for all of them), dt comes without
// division and without a branch, and no branch parts the tokens of a tile, so that the operands of eight are read from LDS ahead of their arithmetic.
// Channels run fastest over the grid, or whole segments of different lengths fall on single XCDs.  16384 tokens of 16 sequences, 4096 channels of 16 states: 613 -> 316 us as whole portions.
// A sequence's first token (position 0) takes the state as zero instead of reading it: slots need no clearing when reused.
#include <type_traits>

#include "api_common.h"
#include "mixers.h"

namespace nvh {

namespace {

using ScanArgs = nvh_scan_desc;
constexpr int TILE = 2048;                           // (token, channel) pairs a workgroup stages at a time
constexpr int min3(int x, int y, int z) { return x < y ? (x < z ? x : z) : (y < z ? y : z); }

// log(1 + e^z) = max(z, 0) + log(1 + e), e = e^-|z|, without a branch or a selection: log(1 + e) / e on [0, 1] by a minimax polynomial of degree 8 (relative error of the coefficients as
// they stand 6.4e-8, -6e-8 of it at small e, where the first one is 1 - 2^-24; 1.7e-7 with 32-bit rounding)
__device__ __forceinline__ float softplus_f(float z) {
    const float e = fast_exp2(-kLog2e * __builtin_fabsf(z));
    float p = 0.005232693627476692f;
    p = p * e - 0.02950523979961872f;
    p = p * e + 0.07822596281766891f;
    p = p * e - 0.13663247227668762f;
    p = p * e + 0.19106008112430573f;
    p = p * e - 0.2484298199415207f;
    p = p * e + 0.3331909775733948f;
    p = p * e - 0.4999949336051941f;
    p = p * e + 0.9999999403953552f;
    return p * e + max2(z, 0.f);
}

__device__ __forceinline__ float gate_f(float z) { return z * fast_rcp(1.f + fast_exp2(-kLog2e * z)); }         // silu

template <int LANES>
__device__ __forceinline__ float sum_lanes(float v) {        // over aligned groups of LANES lanes
    if constexpr (LANES >= 2) v += pair_in_row<1>(v);
    if constexpr (LANES >= 4) v += pair_in_row<2>(v);
    if constexpr (LANES >= 8) v += pair_in_row<4>(v);
    if constexpr (LANES >= 16) v += pair_in_row<8>(v);
    if constexpr (LANES >= 32) v = sum_xor16(v);
    if constexpr (LANES >= 64) v = sum_xor32(v);
    return v;
}

// B and C of a token as a lane's NS states read them from LDS: [lane of the channel][B (NS) | C (NS)]
template <typename T, int NS>
struct StatePairs {
    float b[NS], c[NS];
    __device__ __forceinline__ void read(const T* p) {
        if constexpr (sizeof(T) == 2) {
            uint32_t raw[NS];
#pragma unroll
            for (int i = 0; i < NS; i += 4) {
                const u32x4 v = *reinterpret_cast<const u32x4*>(p + 2 * i);
#pragma unroll
                for (int k = 0; k < 4; ++k) raw[i + k] = v[k];
            }
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                b[i] = i & 1 ? bf16_hi(raw[i >> 1]) : bf16_lo(raw[i >> 1]);
                c[i] = i & 1 ? bf16_hi(raw[(NS + i) >> 1]) : bf16_lo(raw[(NS + i) >> 1]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < NS; i += 4) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(p + i), w = *reinterpret_cast<const f32x4*>(p + NS + i);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    b[i + k] = v[k];
                    c[i + k] = w[k];
                }
            }
        }
    }
};

template <typename T, int NS, int NL, bool SUMMARY>
__global__ __launch_bounds__(256) void scan_walk_kernel(const ScanArgs a) {
    constexpr int NP = NS * NL, CHN = 256 / NL, TT = min3(TILE / CHN, 64, 4096 / NP), PIECES = TT * CHN / 8;        // (PIECES <= 256)
    constexpr int BCP = (TT * 2 * NP / 8 + 255) / 256, U = NS < 8 ? NS : 8;    // pieces of B | C per thread; states of a lane a piece holds
    __shared__ __attribute__((aligned(16))) float dt_s[TT * CHN], dx_s[TT * CHN], y_s[SUMMARY ? 8 : TT * CHN];
    // B and C in LDS: widened once on the way in up to 64 states (16 sequences of 512 tokens, 4096 channels: 157 us against 177 at 16 states, 242 against 296 at 32,
    // 414 against 494 at 64); beyond that the wider rows' bank conflicts cost more than widening on every read (1021 against 928 at 128)
    using L = typename std::conditional<NP <= 64, float, T>::type;
    __shared__ __attribute__((aligned(16))) L bc_s[TT * 2 * NP];
    const int seg = longest_first(a, a.inner / CHN);        // channels run fastest: workgroups are dealt round-robin over the XCDs
    const int32_t* ch = a.chunks + 4 * seg;
    const int row0 = ch[0], n_rows = ch[1], seq = ch[2];
    const bool last = seg + 1 == a.n_chunks || a.chunks[4 * (seg + 1) + 3] == 0;
    if (SUMMARY && last) return;                     // (nothing follows it)
    const int tid = threadIdx.x, c0 = blockIdx.x * CHN, lane_ch = tid / NL, sl = tid % NL;
    const int64_t slot = a.state_slots[seq];
    if (n_rows <= 0) {
        const int mine = a.inner - c0 < CHN ? a.inner - c0 : CHN;
        if (SUMMARY || (last && slot >= 0 && ch[3] > 0))
            pass_segment<SUMMARY>(a.seg_state + ((int64_t)seg * a.inner + c0) * NP, a.state + (slot * a.inner + c0) * NP, mine, NP, NP);
        if (SUMMARY && tid < mine) a.seg_dt[(int64_t)seg * a.inner + c0 + tid] = 0.f;
        return;
    }
    const int my = c0 + lane_ch < a.inner ? c0 + lane_ch : a.inner - 1;          // the channel this lane scans (a last group may be short)
    float A[NS], S[NS], dt_sum = 0.f;
    const float* src = nullptr;
    if constexpr (!SUMMARY) {
        if (a.summaries) src = a.seg_state + ((int64_t)seg * a.inner + my) * NP;
        else if (slot >= 0 && a.positions[row0] > 0) src = a.state + (slot * a.inner + my) * NP;
    }
#pragma unroll
    for (int s = 0; s < NS; s += 4) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(a.a_log2 + (int64_t)my * NP + sl * NS + s);
        f32x4 w = {0.f, 0.f, 0.f, 0.f};
        if (src) w = *reinterpret_cast<const f32x4*>(src + sl * NS + s);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            A[s + k] = v[k];
            S[s + k] = w[k];
        }
    }
    // ---- this thread's piece of the tile: token pt, channels pc .. pc + 7
    const int pt = tid / (CHN / 8), pc = c0 + tid % (CHN / 8) * 8;
    const bool piece = tid < PIECES && pc < a.inner;
    const int pcc = pc < a.inner ? pc : a.inner - 8; // (channels come in eights)
    const f32x8 bias = act_ld8(a.dt_bias + pcc);
    f32x8 D = bias;
    if (!SUMMARY) D = act_ld8(a.d + pcc);
    using Raw = typename std::conditional<sizeof(T) == 2, u32x4, f32x8>::type;
    auto widen = [](const Raw& r) {
        if constexpr (sizeof(T) == 2) return unpack8(r);
        else return r;
    };
    Raw xr, dr, zr, bc[BCP];
    auto fetch = [&](int t0) __attribute__((always_inline)) {                  // rows past the end: the last one again
        const int top = n_rows - 1;
        const int64_t r = row0 + (t0 + pt < top ? t0 + pt : top);
        xr = *reinterpret_cast<const Raw*>(reinterpret_cast<const T*>(a.x) + r * a.x_stride + pcc);
        dr = *reinterpret_cast<const Raw*>(reinterpret_cast<const T*>(a.dt) + r * a.dt_stride + pcc);
        if constexpr (!SUMMARY) zr = *reinterpret_cast<const Raw*>(reinterpret_cast<const T*>(a.z) + r * a.z_stride + pcc);
#pragma unroll
        for (int j = 0; j < BCP; ++j) {
            const int e = j * 256 + tid, t = t0 + e / (2 * NP / 8), p = e % (2 * NP / 8);
            bc[j] = *reinterpret_cast<const Raw*>(reinterpret_cast<const T*>(a.bc) + (int64_t)(row0 + (t < top ? t : top)) * a.bc_stride + p * 8);
        }
    };
    fetch(0);
    for (int t0 = 0; t0 < n_rows; t0 += TT) {
        const int n = n_rows - t0 < TT ? n_rows - t0 : TT;
        const f32x8 xk = widen(xr);
        const Raw zk = SUMMARY ? xr : zr;
        if (tid < PIECES) {
            const f32x8 dk = widen(dr);
            f32x8 dt;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                dt.a[k] = pt < n ? softplus_f(dk.a[k] + bias.a[k]) : 0.f;      // (a token past the end leaves the state alone)
                dt.b[k] = pt < n ? softplus_f(dk.b[k] + bias.b[k]) : 0.f;
            }
            f32x8 dx = {dt.a * xk.a, dt.b * xk.b};
            if (pt >= n) dx = f32x8{f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
            act_st8(dt_s + tid * 8, dt);
            act_st8(dx_s + tid * 8, dx);
        }
        if (n < TT) {                                // rows past the end count nothing, not even infinite ones
#pragma unroll
            for (int j = 0; j < BCP; ++j)
                if ((j * 256 + tid) / (2 * NP / 8) >= n) bc[j] = Raw{};
        }
#pragma unroll
        for (int j = 0; j < BCP; ++j) {
            const int e = j * 256 + tid, t = e / (2 * NP / 8), p = e % (2 * NP / 8), half = p / (NP / 8), s0 = p % (NP / 8) * 8;       // states s0 .. s0 + 7 of B or C
            if (e < TT * 2 * NP / 8) {
                L* row = bc_s + t * 2 * NP + half * NS;
                if constexpr (sizeof(L) == sizeof(T)) {
                    const L* from = reinterpret_cast<const L*>(&bc[j]);
#pragma unroll
                    for (int u = 0; u < 8; u += U) {
                        L* dst = row + (s0 + u) / NS * 2 * NS + (s0 + u) % NS;
                        if constexpr (U * sizeof(L) == 8) *reinterpret_cast<u32x2*>(dst) = *reinterpret_cast<const u32x2*>(from + u);
                        else if constexpr (U * sizeof(L) == 16) *reinterpret_cast<u32x4*>(dst) = *reinterpret_cast<const u32x4*>(from + u);
                        else act_st8(dst, *reinterpret_cast<const f32x8*>(from + u));
                    }
                } else {
                    const f32x8 v = widen(bc[j]);
                    *reinterpret_cast<f32x4*>(row + s0 / NS * 2 * NS + s0 % NS) = v.a;
                    *reinterpret_cast<f32x4*>(row + (s0 + 4) / NS * 2 * NS + (s0 + 4) % NS) = v.b;
                }
            }
        }
        __syncthreads();
        fetch(t0 + TT);
        constexpr int UN = NS <= 4 ? 8 : 4;          // tokens whose operands are on their way from LDS together
        static_assert(TT % UN == 0);
        for (int tb = 0; tb < n; tb += UN) {
#pragma unroll
            for (int t = tb; t < tb + UN; ++t) {
                const float dt = dt_s[t * CHN + lane_ch], dx = dx_s[t * CHN + lane_ch];
                StatePairs<L, NS> v;
                v.read(bc_s + t * 2 * NP + sl * 2 * NS);
                float y = 0.f;
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    S[s] = fast_exp2(dt * A[s]) * S[s] + dx * v.b[s];
                    if constexpr (!SUMMARY) y += S[s] * v.c[s];
                }
                if constexpr (SUMMARY) {
                    dt_sum += dt;
                } else {
                    y = sum_lanes<NL>(y);
                    y_s[t * CHN + lane_ch] = y;      // (all the channel's lanes hold the sum: a branch here would end the block that reads ahead)
                }
            }
        }
        __syncthreads();
        if constexpr (!SUMMARY) {
            if (piece && pt < n) {
                f32x8 y = act_ld8(y_s + tid * 8);
                const f32x8 z = widen(zk);
                y.a += D.a * xk.a;
                y.b += D.b * xk.b;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    y.a[k] *= gate_f(z.a[k]);
                    y.b[k] *= gate_f(z.b[k]);
                }
                act_st8(reinterpret_cast<T*>(a.out) + (int64_t)(row0 + t0 + pt) * a.out_stride + pc, y);
            }
        }
        // (the next tile's y is written behind the barrier that follows its staging)
    }
    if (c0 + lane_ch >= a.inner) return;
    float* dst = nullptr;
    if constexpr (SUMMARY) {
        dst = a.seg_state + ((int64_t)seg * a.inner + my) * NP;
        if (sl == 0) a.seg_dt[(int64_t)seg * a.inner + my] = dt_sum;
    } else if (last && slot >= 0) {
        dst = a.state + (slot * a.inner + my) * NP;
    }
    if (!dst) return;
#pragma unroll
    for (int s = 0; s < NS; s += 4) *reinterpret_cast<f32x4*>(dst + sl * NS + s) = f32x4{S[s], S[s + 1], S[s + 2], S[s + 3]};
}

// ------------------------------------------------------------------------------------------------ whole portions, 16 states (bf16)
// Where the waves of whole portions, with four states a lane, would leave the GPU idle: a state per lane, four times as many waves and no pass over segments in front.
// A row of 16 lanes is a channel, a wave four of them.  dt and dt x of 16 tokens lie one per lane of the row and reach all of it as an operand's row broadcast; a
// token's 16 products with C are added up for 16 tokens at once, so that each lane ends with its token's y, and D x, gate and store follow there.
// Bound by vector issue (a lane-crossing addition takes as long as two plain ones, so that a filled GPU is 6 to 13 % slower with it than with four states a lane) and, for few
// portions, by a wave's own pace.  That: 35 ns a token with the step sizes computed in front of each 16 tokens and dt A multiplied by the lanes, 31 with the next 16 tokens' step sizes in
// between and dt A from the matrix cores, one product of a 4 x 1 and a 1 x 4 matrix a row and four tokens (four waves on a SIMD, issue: 85 -> 80 ns); no token past the end is
// told apart in the loop.  A layer of 16384 tokens of 5 sequences, 2048 channels: 195 -> 187 us.
// Against segments in two passes: 16384 tokens of 5 sequences, 2048 channels: 280 (segments, two passes) -> 230 us; of 16: 252 -> 198; 7000 tokens
// of 5, 4096 channels: 225 -> 161; 2400 of 9, 2048 channels: 52 -> 35.
constexpr int ROW_TT = 64, ROW_CHN = 16, ROW_LD = ROW_TT + 4;

template <int J>
__device__ __forceinline__ float row_lane(float v) { return dpp_f32<0x150 + J>(v); }           // lane J of the row

// lane i of each row: the sum over the row of p[i].  Two tokens share a register from the first addition on (banks of four lanes that an addition leaves alone keep the other
// token's sum); in front of the block and inside it two instructions or more lie between a register's write and its reading across lanes.
__device__ __forceinline__ float row_sums(float (&p)[16], int lane) {
    asm("s_nop 1\n"
        "v_add_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0x3\n v_add_f32_dpp %0, %8, %8 row_ror:8 row_mask:0xf bank_mask:0xc\n"
        "v_add_f32_dpp %1, %1, %1 row_ror:8 row_mask:0xf bank_mask:0x3\n v_add_f32_dpp %1, %9, %9 row_ror:8 row_mask:0xf bank_mask:0xc\n"
        "v_add_f32_dpp %2, %2, %2 row_ror:8 row_mask:0xf bank_mask:0x3\n v_add_f32_dpp %2, %10, %10 row_ror:8 row_mask:0xf bank_mask:0xc\n"
        "v_add_f32_dpp %3, %3, %3 row_ror:8 row_mask:0xf bank_mask:0x3\n v_add_f32_dpp %3, %11, %11 row_ror:8 row_mask:0xf bank_mask:0xc\n"
        "v_add_f32_dpp %4, %4, %4 row_ror:8 row_mask:0xf bank_mask:0x3\n v_add_f32_dpp %4, %12, %12 row_ror:8 row_mask:0xf bank_mask:0xc\n"
        "v_add_f32_dpp %5, %5, %5 row_ror:8 row_mask:0xf bank_mask:0x3\n v_add_f32_dpp %5, %13, %13 row_ror:8 row_mask:0xf bank_mask:0xc\n"
        "v_add_f32_dpp %6, %6, %6 row_ror:8 row_mask:0xf bank_mask:0x3\n v_add_f32_dpp %6, %14, %14 row_ror:8 row_mask:0xf bank_mask:0xc\n"
        "v_add_f32_dpp %7, %7, %7 row_ror:8 row_mask:0xf bank_mask:0x3\n v_add_f32_dpp %7, %15, %15 row_ror:8 row_mask:0xf bank_mask:0xc\n"
        "v_add_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0x5\n v_add_f32_dpp %0, %4, %4 row_half_mirror row_mask:0xf bank_mask:0xa\n"
        "v_add_f32_dpp %1, %1, %1 row_half_mirror row_mask:0xf bank_mask:0x5\n v_add_f32_dpp %1, %5, %5 row_half_mirror row_mask:0xf bank_mask:0xa\n"
        "v_add_f32_dpp %2, %2, %2 row_half_mirror row_mask:0xf bank_mask:0x5\n v_add_f32_dpp %2, %6, %6 row_half_mirror row_mask:0xf bank_mask:0xa\n"
        "v_add_f32_dpp %3, %3, %3 row_half_mirror row_mask:0xf bank_mask:0x5\n v_add_f32_dpp %3, %7, %7 row_half_mirror row_mask:0xf bank_mask:0xa\n"
        "s_nop 1"
        : "+&v"(p[0]), "+&v"(p[1]), "+&v"(p[2]), "+&v"(p[3]), "+&v"(p[4]), "+&v"(p[5]), "+&v"(p[6]), "+&v"(p[7])        // (written while the others are still to be read)
        : "v"(p[8]), "v"(p[9]), "v"(p[10]), "v"(p[11]), "v"(p[12]), "v"(p[13]), "v"(p[14]), "v"(p[15]));
    const bool b1 = lane & 1, b2 = lane & 2;
    float u[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const float lo = p[2 * t] + dpp_f32<0xB1>(p[2 * t]), hi = p[2 * t + 1] + dpp_f32<0xB1>(p[2 * t + 1]);    // quad_perm [1,0,3,2]
        u[t] = b1 ? hi : lo;
    }
    const float lo = u[0] + dpp_f32<0x4E>(u[0]), hi = u[1] + dpp_f32<0x4E>(u[1]);                                // quad_perm [2,3,0,1]
    return b2 ? hi : lo;
}

__global__ __launch_bounds__(256) void scan_rows_kernel(const ScanArgs a) {
    __shared__ __attribute__((aligned(16))) uint16_t x_s[ROW_TT * ROW_CHN], d_s[ROW_TT * ROW_CHN], z_s[ROW_TT * ROW_CHN];
    __shared__ __attribute__((aligned(16))) float bc_s[32 * ROW_LD];           // [B 0..15 | C 0..15][token]
    const int seg = longest_first(a, a.inner / ROW_CHN), groups = gridDim.x;
    const int32_t* chk = a.chunks + 4 * seg;
    const int row0 = chk[0], n_rows = chk[1];
    if (n_rows <= 0) return;
    const int64_t slot = a.state_slots[chk[2]];
    // neighbouring channels' 32-byte pieces of a row share lines: they go to one XCD (workgroups are dealt round-robin)
    const int g = groups % 8 ? blockIdx.x : blockIdx.x % 8 * (groups / 8) + blockIdx.x / 8, c0 = g * ROW_CHN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, st = lane & 15, lc = 4 * wave + (lane >> 4);
    const int my = c0 + lc < a.inner ? c0 + lc : a.inner - 1;
    const float A = a.a_log2[(int64_t)my * 16 + st], bias = a.dt_bias[my], D = a.d[my];
    float S = 0.f;
    if (slot >= 0 && a.positions[row0] > 0) S = a.state[(slot * a.inner + my) * 16 + st];
    // ---- this thread's pieces: x and z (tid < 128), dt; and 8 of a token's B | C
    const int pt = (tid & 127) >> 1, pc = c0 + (tid & 1) * 8, pcc = pc < a.inner ? pc : a.inner - 8, bt = tid >> 2, bp = tid & 3;
    const bool low = tid < 128;
    const uint16_t* from = reinterpret_cast<const uint16_t*>(low ? a.x : a.dt) + pcc;
    const int64_t from_stride = low ? a.x_stride : a.dt_stride;
    u32x4 r0, r1, rb;
    auto fetch = [&](int t0) __attribute__((always_inline)) {                  // rows past the end: the last one again
        const int top = n_rows - 1;
        const int64_t r = row0 + (t0 + pt < top ? t0 + pt : top);
        r0 = *reinterpret_cast<const u32x4*>(from + r * from_stride);
        r1 = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(a.z) + r * a.z_stride + pcc);
        rb = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(a.bc) + (int64_t)(row0 + (t0 + bt < top ? t0 + bt : top)) * a.bc_stride + bp * 8);
    };
    fetch(0);
    for (int t0 = 0; t0 < n_rows; t0 += ROW_TT) {
        const int n = n_rows - t0 < ROW_TT ? n_rows - t0 : ROW_TT;
        // rows past the end count nothing, not even infinite ones: a step of softplus(-inf) = 0 leaves the state alone
        if (pt >= n) r0 = low ? u32x4{0, 0, 0, 0} : u32x4{0xFF80FF80u, 0xFF80FF80u, 0xFF80FF80u, 0xFF80FF80u};
        if (bt >= n) rb = u32x4{0, 0, 0, 0};
        *reinterpret_cast<u32x4*>((low ? x_s : d_s) + (tid & 127) * 8) = r0;
        if (low) *reinterpret_cast<u32x4*>(z_s + tid * 8) = r1;
        {
            const f32x8 v = unpack8(rb);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                bc_s[(8 * bp + i) * ROW_LD + bt] = v.a[i];
                bc_s[(8 * bp + 4 + i) * ROW_LD + bt] = v.b[i];
            }
        }
        __syncthreads();
        fetch(t0 + ROW_TT);
        // token k + st of this lane's channel: its steps, and what the output needs
        float xv, zv, dt, dx;
        auto steps = [&](int k, float& xv, float& zv, float& dt, float& dx) __attribute__((always_inline)) {
            const int e = (k + st) * ROW_CHN + lc;
            xv = act_ld(x_s + e), zv = act_ld(z_s + e);
            dt = softplus_f(act_ld(d_s + e) + bias);
            dx = dt * xv;
        };
        steps(0, xv, zv, dt, dx);
#pragma unroll
        for (int k = 0; k < ROW_TT; k += 16) {
            if (k >= n) break;
            float xn = 0.f, zn = 0.f, dtn = 0.f, dxn = 0.f;      // the next 16 tokens', in between these ones' chain
            if (k + 16 < ROW_TT) steps(k + 16, xn, zn, dtn, dxn);
            const float* b_row = bc_s + st * ROW_LD + k;
            float p[16];
            auto token = [&](auto j, float at, float b, float c) __attribute__((always_inline)) {
                constexpr int J = decltype(j)::value;
                float in = row_lane<J>(dx) * b;      // (the broadcast is an operand of the multiplication, as long as that is not merged into the sum)
                asm("" : "+v"(in));
                S = fast_exp2(at) * S + in;
                p[J] = S * c;
            };
            f32x4 at[4], b[4], c[4];
            auto four = [&](auto q) __attribute__((always_inline)) {
                constexpr int Q = decltype(q)::value;
                token(std::integral_constant<int, 4 * Q>(), at[Q][0], b[Q][0], c[Q][0]);
                token(std::integral_constant<int, 4 * Q + 1>(), at[Q][1], b[Q][1], c[Q][1]);
                token(std::integral_constant<int, 4 * Q + 2>(), at[Q][2], b[Q][2], c[Q][2]);
                token(std::integral_constant<int, 4 * Q + 3>(), at[Q][3], b[Q][3], c[Q][3]);
            };
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                b[q] = *reinterpret_cast<const f32x4*>(b_row + 4 * q);
                c[q] = *reinterpret_cast<const f32x4*>(b_row + 16 * ROW_LD + 4 * q);
            }
            // dt of tokens 4 q .. times this lane's A: block q of the row's four holds those tokens and is every block's left operand
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
            at[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(dt, A, zero, 2, 0, 0);
            at[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(dt, A, zero, 2, 1, 0);
            at[2] = __builtin_amdgcn_mfma_f32_4x4x1f32(dt, A, zero, 2, 2, 0);
            at[3] = __builtin_amdgcn_mfma_f32_4x4x1f32(dt, A, zero, 2, 3, 0);
            four(std::integral_constant<int, 0>());
            four(std::integral_constant<int, 1>());
            four(std::integral_constant<int, 2>());
            four(std::integral_constant<int, 3>());
            __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);   // (everything asked for before the chain)
            __builtin_amdgcn_sched_group_barrier(0x8, 4, 0);
            act_st(z_s + (k + st) * ROW_CHN + lc, (row_sums(p, lane) + D * xv) * gate_f(zv));
            xv = xn, zv = zn, dt = dtn, dx = dxn;
        }
        __syncthreads();
        if (low && pt < n && pc < a.inner)
            *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(a.out) + (int64_t)(row0 + t0 + pt) * a.out_stride + pc) = *reinterpret_cast<const u32x4*>(z_s + tid * 8);
        // (this thread puts the next z where it has just read)
    }
    if (c0 + lc < a.inner && slot >= 0) a.state[(slot * a.inner + my) * 16 + st] = S;
}

// contributions of the segments -> states at their starts, in place; a thread per four states of a portion, walking its segments
__global__ __launch_bounds__(256) void scan_starts_kernel(const ScanArgs a) {
    const int64_t per = (int64_t)a.inner * a.n, e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    const int first = blockIdx.y;                    // only a portion's first segment starts a walk
    if (a.chunks[4 * first + 3] != 0) return;
    const int count = portion_segments(a.chunks, a.n_chunks, first);
    if (e >= per) return;
    const f32x4 A = *reinterpret_cast<const f32x4*>(a.a_log2 + e);
    const int64_t c = e / a.n, slot = a.state_slots[a.chunks[4 * first + 2]];
    const f32x4 cur = slot >= 0 && portion_carries(a.chunks, a.n_chunks, first, a.positions) ? *reinterpret_cast<const f32x4*>(a.state + slot * per + e) : f32x4{};
    segment_starts(a.seg_state + first * per + e, per, count, cur, [&](int k) { return a.seg_dt[(int64_t)(first + k) * a.inner + c]; },
                   [&](float dt) {
                       const f32x4 p = A * dt;
                       return f32x4{fast_exp2(p[0]), fast_exp2(p[1]), fast_exp2(p[2]), fast_exp2(p[3])};
                   });
}

// one new token per sequence (bf16): grid (channel groups, groups of R rows), LN = n / 4 lanes per channel
template <int LN, int R>
__global__ __launch_bounds__(256) void scan_step_kernel(const ScanArgs a) {
    constexpr int CHN = 256 / LN, NP = 4 * LN;
    const int tid = threadIdx.x, sl = tid % LN, c = blockIdx.x * CHN + tid / LN;
    const bool ok = c < a.inner;
    const int my = ok ? c : a.inner - 1;
    const uint16_t* w = reinterpret_cast<const uint16_t*>(a.w_dt) + (int64_t)my * a.rank;
    const int r0 = blockIdx.y * R;
    f32x4 s[R];
    float xv[R], zv[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {                    // asked for before anything is computed
        const int row = r0 + i < a.rows ? r0 + i : a.rows - 1;
        const int64_t slot = a.state_slots[row];
        s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (slot >= 0 && a.positions[row] > 0) s[i] = *reinterpret_cast<const f32x4*>(a.state + (slot * a.inner + my) * NP + 4 * sl);
        xv[i] = act_ld(reinterpret_cast<const uint16_t*>(a.x) + (int64_t)row * a.x_stride + my);
        zv[i] = act_ld(reinterpret_cast<const uint16_t*>(a.z) + (int64_t)row * a.z_stride + my);
    }
    const f32x4 A = *reinterpret_cast<const f32x4*>(a.a_log2 + (int64_t)my * NP + 4 * sl);
    float acc[R];
#pragma unroll
    for (int i = 0; i < R; ++i) acc[i] = 0.f;
    for (int p = sl * 8; p < a.rank; p += LN * 8) {
        const u32x4 wv = *reinterpret_cast<const u32x4*>(w + p);
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int row = r0 + i < a.rows ? r0 + i : a.rows - 1;
            const u32x4 v = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(a.dt) + (int64_t)row * a.dt_stride + p);
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[i] = dot2_bf16(wv[k], v[k], acc[i]);
        }
    }
    const float bias = a.dt_bias[my], D = a.d[my];
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const int row = r0 + i;
        if (row >= a.rows) continue;                 // (workgroup-uniform)
        const float dt = softplus_f(sum_lanes<LN>(acc[i]) + bias), dx = dt * xv[i];
        const uint16_t* bc = reinterpret_cast<const uint16_t*>(a.bc) + (int64_t)row * a.bc_stride + 4 * sl;
        const f32x4 b = act_ld4(bc), cv = act_ld4(bc + NP);
        f32x4 n;
        float y = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            n[k] = fast_exp2(dt * A[k]) * s[i][k] + dx * b[k];
            y += n[k] * cv[k];
        }
        const int64_t slot = a.state_slots[row];
        if (ok && slot >= 0) *reinterpret_cast<f32x4*>(a.state + (slot * a.inner + my) * NP + 4 * sl) = n;
        y = (sum_lanes<LN>(y) + D * xv[i]) * gate_f(zv[i]);
        if (ok && sl == 0) {
            if (a.out) act_st(reinterpret_cast<uint16_t*>(a.out) + (int64_t)row * a.out_stride + c, y);
            if (a.out_packed) act_st(reinterpret_cast<uint16_t*>(a.out_packed) + pack_index(row, c, a.inner), y);
        }
    }
}

template <typename T, int NS, int NL>
int walk_ns(const ScanArgs& a, hipStream_t stream) {
    constexpr int CHN = 256 / NL;
    const dim3 grid((a.inner + CHN - 1) / CHN, a.n_chunks);
    if (a.summaries) {
        scan_walk_kernel<T, NS, NL, true><<<grid, 256, 0, stream>>>(a);
        int rc = check_launch("scan summary");
        if (rc) return rc;
        const int64_t per = (int64_t)a.inner * a.n;
        scan_starts_kernel<<<dim3((unsigned)((per + 1023) / 1024), a.n_chunks), 256, 0, stream>>>(a);
        rc = check_launch("scan starts");
        if (rc) return rc;
    }
    scan_walk_kernel<T, NS, NL, false><<<grid, 256, 0, stream>>>(a);
    return check_launch("scan walk");
}

constexpr int kWholeChannels = 40960;                // (the host's choice of segments asks for it: nvh_scan_whole_channels)
template <typename T>
int walk_t(const ScanArgs& a, hipStream_t stream) {
    // Lanes per channel: more of them add up y over more lanes and read dt and dt x again, fewer make fewer waves, each with more registers.  16 sequences of 512
    // tokens, 4096 channels: 8 states 122 us with 2 lanes, 159 with 1; 16 states 153 with 4 lanes, 164 with 2; 32 states 244 with 4 lanes, 314 with 8;
    // 64 states 420 with 4 lanes, 506 with 8.
    switch (a.n) {
        case 8: return walk_ns<T, 4, 2>(a, stream);
        case 16:
            // Four states a lane fill the GPU from about four waves on every SIMD on (portions x channels / 16384), with long portions from two and a half.
            // Whole portions, one against four states a lane: 23 of 200 tokens, 2048 channels (2.9 waves) 59 to 64 us; 13 of 250, 4096 channels (3.25) 74 to 77; 31 of 100 (3.9) 41 to 40; 17
            // of 200, 4096 channels (4.25) 82 to 71; 8 of 600 (2.0) 108 to 116, 10 of 790 (2.5) 180 to 173.
            if constexpr (sizeof(T) == 2) {
                const int64_t fill = (int64_t)a.n_chunks * a.inner;
                if (!a.summaries && (fill < kWholeChannels || (fill < 65536 && a.rows / a.n_chunks < 512))) {
                    scan_rows_kernel<<<dim3((a.inner + 15) / 16, a.n_chunks), 256, 0, stream>>>(a);
                    return check_launch("scan rows");
                }
            }
            return walk_ns<T, 4, 4>(a, stream);
        case 32: return walk_ns<T, 8, 4>(a, stream);
        case 64: return walk_ns<T, 16, 4>(a, stream);
        case 128: return walk_ns<T, 16, 8>(a, stream);
        default: return walk_ns<T, 16, 16>(a, stream);
    }
}

template <int LN>
void step_ln(const ScanArgs& a, hipStream_t stream) {
    constexpr int CHN = 256 / LN;
    const unsigned groups = (a.inner + CHN - 1) / CHN;
    if ((int64_t)groups * a.rows >= 2048) scan_step_kernel<LN, 4><<<dim3(groups, (a.rows + 3) / 4), 256, 0, stream>>>(a);
    else scan_step_kernel<LN, 1><<<dim3(groups, a.rows), 256, 0, stream>>>(a);
}

int check_scan(const char* fn, const nvh_scan_desc* d, int dtype) {
    DTYPE(fn);
    REQUIRE(d->x && d->dt && d->dt_bias && d->bc && d->z && d->a_log2 && d->d && d->positions && d->state_slots && d->state && (d->out || d->out_packed), NVH_E_NULL, "%s: null pointer", fn);
    REQUIRE(d->rows > 0 && d->inner > 0 && d->inner % 8 == 0 && nvh_scan_states(d->n) == d->n, NVH_E_SHAPE, "%s: %d channels (%%8), %d states", fn, d->inner, d->n);
    REQUIRE(d->x_stride % 8 == 0 && d->x_stride >= d->inner && d->z_stride % 8 == 0 && d->z_stride >= d->inner && d->bc_stride % 8 == 0 && d->bc_stride >= 2 * d->n &&
            d->dt_stride % 8 == 0 && (!d->out || (d->out_stride % 8 == 0 && d->out_stride >= d->inner)), NVH_E_STRIDE, "%s: row strides", fn);
    REQUIRE(aligned16(d->x) && aligned16(d->dt) && aligned16(d->dt_bias) && aligned16(d->bc) && aligned16(d->z) && aligned16(d->a_log2) && aligned16(d->d) && aligned16(d->state) &&
            aligned16(d->seg_state) && aligned16(d->out) && aligned16(d->out_packed), NVH_E_ALIGN, "%s: pointers must be 16-byte aligned", fn);
    return 0;
}

}  // namespace

}  // namespace nvh

using namespace nvh;

extern "C" {

int nvh_scan_states(int n) {
    for (int p = 8; p <= 256; p *= 2)
        if (n > 0 && n <= p) return p;
    return 0;
}

int nvh_scan_whole_channels(void) { return kWholeChannels; }

int nvh_scan_chunks(const nvh_scan_desc* d, int dtype, void* stream) {
    REQUIRE(d, NVH_E_NULL, "scan_chunks: null descriptor");
    if (d->n_chunks == 0) return 0;
    const int rc = check_scan("scan_chunks", d, dtype);
    if (rc) return rc;
    REQUIRE(d->chunks && d->n_chunks > 0 && d->n_chunks <= 65535 && d->out && d->dt_stride >= d->inner && (!d->summaries || (d->seg_state && d->seg_dt)), NVH_E_NULL,
            "scan_chunks: %d segments or null pointer", d->n_chunks);
    return dtype == NVH_F32 ? walk_t<float>(*d, (hipStream_t)stream) : walk_t<uint16_t>(*d, (hipStream_t)stream);
}

int nvh_scan_step(const nvh_scan_desc* d, int dtype, void* stream) {
    REQUIRE(d, NVH_E_NULL, "scan_step: null descriptor");
    if (d->rows == 0) return 0;
    const int rc = check_scan("scan_step", d, dtype);
    if (rc) return rc;
    REQUIRE(dtype == NVH_BF16 && d->w_dt && aligned16(d->w_dt) && d->rank > 0 && d->rank % 8 == 0 && d->dt_stride >= d->rank && d->rows <= 65535 && (!d->out_packed || d->inner % 32 == 0),
            NVH_E_SHAPE, "scan_step: bf16, rank %d (%%8), rows %d", d->rank, d->rows);
    switch (d->n / 4) {
        case 2: step_ln<2>(*d, (hipStream_t)stream); break;
        case 4: step_ln<4>(*d, (hipStream_t)stream); break;
        case 8: step_ln<8>(*d, (hipStream_t)stream); break;
        case 16: step_ln<16>(*d, (hipStream_t)stream); break;
        case 32: step_ln<32>(*d, (hipStream_t)stream); break;
        default: step_ln<64>(*d, (hipStream_t)stream); break;
    }
    return check_launch("scan_step");
}

}  // extern "C"
