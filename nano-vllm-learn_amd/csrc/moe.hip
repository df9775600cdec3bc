// Mixture of experts; the router's scores are sigmoids with choice corrections and expert groups, or a softmax over the chosen logits.
//   route     32-bit logits of a row tile against every expert (MFMA for bf16), group and expert choice, weights: one launch
//   dispatch  pairs (row, chosen expert) sorted by expert and cut into tiles of one expert each: two launches, no host round trip
//   gemm      expert products: gate | up with the gated unit in the epilogue, and down.  Large batches: 128 x 128 or 256 x 256 MFMA tiles over the
//             sorted pairs, the rows gathered by the DMA that fills LDS; both products in one launch where that fills the CUs better.  At most 64 rows: every wave streams 16 weight rows once for all the rows that chose the expert.
// Outputs stay per pair; the weighted sum over a row's experts belongs to the residual add (hybrid_ops.hip).
#include "attend_tile.h"
#include "mixers.h"

namespace nvh {

namespace {

// ------------------------------------------------------------------------------------------------ choice (one wave per row)
__device__ __forceinline__ float wave_max64(float v) {
    v = fmaxf(v, pair_in_row<1>(v));
    v = fmaxf(v, pair_in_row<2>(v));
    v = fmaxf(v, pair_in_row<4>(v));
    v = fmaxf(v, pair_in_row<8>(v));
    v = max_xor16(v);
    return max_xor32(v);
}
// lane that holds the wave's largest value (the first of equal ones)
__device__ __forceinline__ int wave_winner(float v) {
    const uint64_t b = __builtin_amdgcn_ballot_w64(v == wave_max64(v));
    return b ? __builtin_ctzll(b) : 0;               // (0 only where a router delivers no number)
}
__device__ __forceinline__ float lane_value(float v, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane)); }

__device__ __forceinline__ float group_score(const float* choice, int size) {
    float b0 = -INFINITY, b1 = -INFINITY;            // the two largest
    for (int k = 0; k < size; ++k) {
        const float c = choice[k];
        b1 = fmaxf(b1, fminf(b0, c));
        b0 = fmaxf(b0, c);
    }
    return size > 1 ? b0 + b1 : b0;
}

__device__ __forceinline__ void store_choice(const MoeRouteArgs& a, int row, int lane, int id, float score, float total) {
    if (lane < a.top) {
        a.ids[(int64_t)row * a.top + lane] = id;
        a.weights[(int64_t)row * a.top + lane] = score / (total + 1e-20f) * a.scale;
    }
}

// score of an expert from its logit
__device__ __forceinline__ float expert_score(const MoeRouteArgs& a, float z, int e) { return a.softmax ? z + a.correction[e] : 1.f / (1.f + expf(-z)); }
// its part of the weights, with `top` the score of the first choice (a softmax is taken relative to its largest entry)
__device__ __forceinline__ float expert_part(const MoeRouteArgs& a, float score, float top) { return a.softmax ? expf(score - top) : score; }

// z [E]: logits in, scores out; choice [E], gs [groups]: scratch in LDS.  Up to 64 experts: one per lane, LDS for the group scores only.
__device__ __forceinline__ void choose_experts(const MoeRouteArgs& a, int row, int lane, float* z, float* choice, float* gs) {
    const int size = a.experts / a.groups;
    float total = 0.f, mine = 0.f, top = 0.f;
    int my_id = 0;
    if (a.experts <= 64) {
        const bool ok = lane < a.experts;
        const float s = ok ? expert_score(a, z[lane], lane) : 0.f;
        float c = ok ? (a.softmax ? s : s + a.correction[lane]) : -INFINITY;
        if (a.keep < a.groups) {
            choice[lane] = c;
            wave_lds_sync();
            float g = lane < a.groups ? group_score(choice + lane * size, size) : -INFINITY;
            uint64_t open = 0;
            for (int k = 0; k < a.keep; ++k) {
                const int w = wave_winner(g);
                open |= 1ull << w;
                if (lane == w) g = -INFINITY;
            }
            if (!((open >> (lane / size)) & 1)) c = -INFINITY;
        }
        for (int k = 0; k < a.top; ++k) {
            const int w = wave_winner(c);
            const float score = lane_value(s, w);
            if (k == 0) top = score;
            const float sw = expert_part(a, score, top);
            total += sw;
            if (lane == k) {
                mine = sw;
                my_id = w < a.experts ? w : 0;
            }
            if (lane == w) c = -INFINITY;
        }
        store_choice(a, row, lane, my_id, mine, total);
        return;
    }
    for (int e = lane; e < a.experts; e += 64) {
        const float s = expert_score(a, z[e], e);
        z[e] = s;
        choice[e] = a.softmax ? s : s + a.correction[e];
    }
    wave_lds_sync();
    auto best = [&](const float* list, int n) {      // index of the list's largest value
        float v = -INFINITY;
        int i = 0;
        for (int e = lane; e < n; e += 64) {
            const float c = list[e];
            if (c > v) {
                v = c;
                i = e;
            }
        }
        return __builtin_amdgcn_readlane(i, wave_winner(v));
    };
    if (a.keep < a.groups) {
        for (int g = lane; g < a.groups; g += 64) gs[g] = group_score(choice + g * size, size);
        wave_lds_sync();
        for (int k = 0; k < a.keep; ++k) {           // an open group is marked by NaN: it loses every comparison
            const int g = best(gs, a.groups);
            if (lane == 0) gs[g] = NAN;
            wave_lds_sync();
        }
        for (int e = lane; e < a.experts; e += 64)
            if (gs[e / size] == gs[e / size]) choice[e] = -INFINITY;
        wave_lds_sync();
    }
    for (int k = 0; k < a.top; ++k) {
        const int e = best(choice, a.experts);
        if (k == 0) top = z[e];
        const float s = expert_part(a, z[e], top);
        total += s;
        if (lane == k) {
            mine = s;
            my_id = e;
        }
        wave_lds_sync();
        if (lane == 0) choice[e] = -INFINITY;
        wave_lds_sync();
    }
    store_choice(a, row, lane, my_id, mine, total);
}

// live rows (at most 16) per workgroup, the contraction shared by 8 waves, 64 experts at a time
__global__ __launch_bounds__(512) void moe_route_kernel(const MoeRouteArgs a, const int live) {
    extern __shared__ __attribute__((aligned(16))) float lds_r[];
    const int ez = (a.experts + 63) / 64 * 64;
    float *part = lds_r, *z = part + 8 * 16 * 68, *choice = z + 16 * ez, *gs = choice + 8 * ez;     // [8][16][64 + 4], [16][ez], per wave [ez], [groups]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lq = lane & 15, lg = lane >> 4;
    const int r0 = blockIdx.x * live, rows = a.rows - r0 < live ? a.rows - r0 : live, row = r0 + (lq < rows ? lq : rows - 1);
    const int steps = a.cols / 32, per = (steps + 7) / 8, s0 = wave * per, s1 = s0 + per < steps ? s0 + per : steps;
    const uint16_t* x = reinterpret_cast<const uint16_t*>(a.x) + (int64_t)row * a.x_stride + 8 * lg;
    for (int e0 = 0; e0 < a.experts; e0 += 64) {
        const uint16_t* w[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int e = e0 + 16 * t + lq;
            w[t] = reinterpret_cast<const uint16_t*>(a.router) + (int64_t)(e < a.experts ? e : a.experts - 1) * a.cols + 8 * lg;
        }
        f32x4 acc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto walk = [&](auto ntc) {                  // (tiles that hold no expert are not read)
            constexpr int NT = decltype(ntc)::value;
            constexpr int UN = 4;
            int s = s0;
            for (; s + UN <= s1; s += UN) {
                bf16x8 xf[UN], wf[UN][NT];
#pragma unroll
                for (int i = 0; i < UN; ++i) {
                    xf[i] = *reinterpret_cast<const bf16x8*>(x + 32 * (s + i));
#pragma unroll
                    for (int t = 0; t < NT; ++t) wf[i][t] = *reinterpret_cast<const bf16x8*>(w[t] + 32 * (s + i));
                }
#pragma unroll
                for (int i = 0; i < UN; ++i)
#pragma unroll
                    for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i][t], xf[i], acc[t], 0, 0, 0);
            }
            for (; s < s1; ++s) {
                const bf16x8 xf = *reinterpret_cast<const bf16x8*>(x + 32 * s);
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(w[t] + 32 * s), xf, acc[t], 0, 0, 0);
            }
        };
        switch ((a.experts - e0 + 15) / 16) {
            case 1: walk(std::integral_constant<int, 1>{}); break;
            case 2: walk(std::integral_constant<int, 2>{}); break;
            case 3: walk(std::integral_constant<int, 3>{}); break;
            default: walk(std::integral_constant<int, 4>{}); break;
        }
        // D: lane = row lq, experts 16 t + 4 lg ..
#pragma unroll
        for (int t = 0; t < 4; ++t) *reinterpret_cast<f32x4*>(part + (wave * 16 + lq) * 68 + 16 * t + 4 * lg) = acc[t];
        __syncthreads();
        for (int i = tid; i < rows * 64; i += 512) {
            const int r = i >> 6, e = i & 63;
            float s = 0.f;
#pragma unroll
            for (int k = 0; k < 8; ++k) s += part[(k * 16 + r) * 68 + e];
            z[r * ez + e0 + e] = s;
        }
        __syncthreads();
    }
    for (int r = wave; r < rows; r += 8) choose_experts(a, r0 + r, lane, z + r * ez, choice + wave * ez, gs + wave * a.groups);
}

// any type and width: one workgroup per row, a wave per expert in turn
template <typename T>
__global__ __launch_bounds__(256) void moe_route_generic_kernel(const MoeRouteArgs a) {
    extern __shared__ __attribute__((aligned(16))) float lds_r[];
    float *z = lds_r, *choice = z + a.experts, *gs = choice + a.experts;
    const int row = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const T* x = reinterpret_cast<const T*>(a.x) + (int64_t)row * a.x_stride;
    for (int e = wave; e < a.experts; e += 4) {
        const T* w = reinterpret_cast<const T*>(a.router) + (int64_t)e * a.cols;
        float s = 0.f;
        for (int c = lane * 4; c < a.cols; c += 256) s += sum4(act_ld4(x + c) * act_ld4(w + c));
        s = wave_sum64(s);
        if (lane == 0) z[e] = s;
    }
    __syncthreads();
    if (wave == 0) choose_experts(a, row, lane, z, choice, gs);
}

// ------------------------------------------------------------------------------------------------ dispatch
constexpr int DP = 2048;                             // pairs per workgroup

__global__ __launch_bounds__(256) void moe_count_kernel(int32_t* __restrict__ counts, const int32_t* __restrict__ ids, int pairs, int experts) {
    __shared__ int hist[kMoeMaxExperts];
    for (int e = threadIdx.x; e < experts; e += 256) hist[e] = 0;
    __syncthreads();
    const int p0 = blockIdx.x * DP + threadIdx.x;
    int id[DP / 256];                                // (all asked for at once)
#pragma unroll
    for (int u = 0; u < DP / 256; ++u) id[u] = ids[p0 + 256 * u < pairs ? p0 + 256 * u : pairs - 1];
#pragma unroll
    for (int u = 0; u < DP / 256; ++u)
        if (p0 + 256 * u < pairs) atomicAdd(&hist[id[u]], 1);
    __syncthreads();
    for (int e = threadIdx.x; e < experts; e += 256) counts[(int64_t)blockIdx.x * experts + e] = hist[e];
}

// Every workgroup sums the counts in front of its own pairs; the first one also writes the tiles.  Up to kCountHere pairs each counts all of them itself: the launch that counts takes
// longer than that.  (Both bound by latency: every load of a thread is asked for at once, and all threads sum the counts.  One by one, 32 threads summing: dispatch of 65536 pairs of 32
// experts 13.2 -> 6.7 us, 12000 7.1 -> 6.4.)  300 tokens' 1200 pairs 1.9 + 3.1 us in two launches, 2.4 in one (1024 wide: the call 55 -> 52 us); 7200
// pairs 89 -> 86.
constexpr int kCountHere = 4 * DP;
template <bool COUNTED>
__global__ __launch_bounds__(256) void moe_scatter_kernel(int32_t* __restrict__ slot_pair, int32_t* __restrict__ tiles, const int32_t* __restrict__ counts,
                                                          const int32_t* __restrict__ ids, int pairs, int experts, int tile_rows, int max_tiles, uint32_t* __restrict__ clear, int clear_words) {
    __shared__ int at[kMoeMaxExperts], total[kMoeMaxExperts], start[kMoeMaxExperts], tile0[kMoeMaxExperts];
    __shared__ int n_tiles;
    constexpr int PER = DP / 256;
    const int p0 = blockIdx.x * DP;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < clear_words; i += gridDim.x * 256) clear[i] = 0;            // (for the launch behind this one)
    auto take = [&](int first, int (&id)[PER]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const int p = first + 256 * u + (int)threadIdx.x;
            id[u] = ids[p < pairs ? p : pairs - 1];
        }
    };
    int own[PER];                                    // the experts of this workgroup's pairs
    take(p0, own);
    for (int e = threadIdx.x; e < experts; e += 256) at[e] = total[e] = 0;
    __syncthreads();
    if constexpr (COUNTED) {                         // (every thread, as the counts lie)
        const int words = (int)gridDim.x * experts, mine = (int)blockIdx.x * experts;
        for (int i0 = 0; i0 < words; i0 += 4 * 256) {
            int c[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = i0 + 256 * u + (int)threadIdx.x;
                c[u] = counts[i < words ? i : 0];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = i0 + 256 * u + (int)threadIdx.x, e = i % experts;
                if (i < words && c[u]) {
                    atomicAdd(&total[e], c[u]);
                    if (i < mine) atomicAdd(&at[e], c[u]);
                }
            }
        }
    } else {
        auto count = [&](int first, const int (&id)[PER]) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < PER; ++u)
                if (first + 256 * u + (int)threadIdx.x < pairs) {
                    atomicAdd(&total[id[u]], 1);
                    if (first < p0) atomicAdd(&at[id[u]], 1);
                }
        };
        for (int first = 0; first < pairs; first += DP) {
            if (first == p0) continue;
            int id[PER];
            take(first, id);
            count(first, id);
        }
        count(p0, own);
    }
    __syncthreads();
    if (threadIdx.x < 64) {                          // exclusive scans over the experts, 64 at a time
        int base = 0, tbase = 0;
        for (int e0 = 0; e0 < experts; e0 += 64) {
            const int e = e0 + threadIdx.x, n = e < experts ? total[e] : 0, t = (n + tile_rows - 1) / tile_rows;
            int s = n, u = t;
            for (int d = 1; d < 64; d <<= 1) {
                const int ps = __shfl_up(s, d), pu = __shfl_up(u, d);
                if ((int)threadIdx.x >= d) {
                    s += ps;
                    u += pu;
                }
            }
            if (e < experts) {
                start[e] = base + s - n;
                tile0[e] = tbase + u - t;
            }
            base += __shfl(s, 63);
            tbase += __shfl(u, 63);
        }
        if (threadIdx.x == 0) n_tiles = tbase;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < experts; e += 256) at[e] += start[e];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int p = p0 + 256 * u + (int)threadIdx.x;
        if (p < pairs) slot_pair[atomicAdd(&at[own[u]], 1)] = p;
    }
    if (blockIdx.x == 0) {
        for (int e = threadIdx.x; e < experts; e += 256)
            for (int t = 0; t * tile_rows < total[e]; ++t) {
                const int left = total[e] - t * tile_rows;
                reinterpret_cast<int4*>(tiles)[tile0[e] + t] = int4{e, start[e] + t * tile_rows, left < tile_rows ? left : tile_rows, n_tiles};
            }
        for (int t = n_tiles + threadIdx.x; t < max_tiles; t += 256) reinterpret_cast<int4*>(tiles)[t] = int4{0, 0, 0, n_tiles};
    }
}

// ------------------------------------------------------------------------------------------------ products, large batches (bf16)
// MW x NW waves of MT x NT tiles of 16 x 16: TM pairs by TN weight rows per workgroup, 32 of the contraction at a time, both operands by LDS-DMA through a
// ring of four images: three are on their way while the fourth is read into registers, and the one before it is multiplied from there.
// GLU: weight rows alternate 16 of gate, 16 of up, so a lane holds both halves of its outputs.
constexpr int TK = 32, kRing = 4;
// SiLU(g) u, or the clamped unit where the launch names an alpha
__device__ __forceinline__ float expert_unit(const MoeGemmArgs& a, float g, float u) { return a.alpha != 0.f ? clamped_glu(g, u, a.limit, a.alpha) : silu_f(g) * u; }
template <int MW, int NW, int MT, int NT>
struct GemmShape {
    static constexpr int WAVES = MW * NW, TM = MW * MT * 16, TN = NW * NT * 16, ROWS = TM + TN, STEP = MT >= 4 ? MT / 4 : 1, UNIT = MW * STEP * 16, IMG = ROWS * TK * 2, DMA = IMG / 1024 / WAVES;
    static constexpr size_t LDS = (size_t)kRing * IMG;
    static_assert(IMG % (1024 * WAVES) == 0 && NT % 2 == 0, "DMA instructions and gate/up tiles divide evenly");
};

// A workgroup's part of a product: rows of tile mt (pairs first .. of an expert, `live` of them) and columns nt.
struct ExpertTile {
    int nt, mt, expert, first, live;
};
// The idx-th one of the row tiles lo .. hi - 1 times nx columns: an expert's, up to eight row tiles times the columns at a time, rows first.  What runs at once shares rows and weights
// in an XCD's L2.  (Eight row tiles whosever they are share less: 12000 tokens, 32 experts of 1536, 1000 -> 955 us, 3000 385 -> 371; 1500 at 1024 wide 74 -> 73)
// The tiles of an expert share its pairs evenly, in units of what the waves multiply at a time, instead of all but the last being full: workgroups of one length fill the rounds that the
// CUs take them in better.  (1024 wide, 3000 tokens 132 -> 129 us.  In units of a row of every wave's tiles a tile of 240 would multiply 256, eight times an expert: 16384 tokens at
// 2048 wide 1155 -> 1160)
// rows 0: eight row tiles at a time, whosever they are.  For launches of up to a workgroup a CU: an expert's tiles together would leave the experts with the most pairs to one XCD.  (8 experts
// of 1536, 2048 wide, 99 tokens of an uneven route, gate | up 24.8 -> 22.0 us; 16 of 512, 4096 wide, 322 tokens 40.8 -> 37.3)
constexpr int kAlone = 256;
// a / b of up to 2^20 (by 32 bits: half of the instructions in front of a workgroup's first load)
__device__ __forceinline__ int few_over(int a, int b) { return (int)(((float)a + 0.5f) * fast_rcp((float)b)); }
template <int TM, int UNIT>
__device__ __forceinline__ ExpertTile find_tile(const int32_t* table, int tiles, int nx, int idx, int lo, int hi, int rows, int lane) {
    ExpertTile to;
    int m, nt;
    if (rows) {
        m = lo + idx / nx;
        nt = idx - (m - lo) * nx;
    } else {
        const int g = few_over(idx, 8 * nx), in = idx - g * 8 * nx, gm = tiles - 8 * g < 8 ? tiles - 8 * g : 8;
        nt = few_over(in, gm);
        m = 8 * g + in - nt * gm;
    }
    const int at = m - 32 + lane;                    // a tile of the expert, and 63 around it
    const int4 t = reinterpret_cast<const int4*>(table)[at < 0 ? 0 : at < tiles ? at : tiles - 1];
    to.expert = __builtin_amdgcn_readlane(t.x, 32);
    const uint64_t same = __builtin_amdgcn_ballot_w64(at >= 0 && at < tiles && t.x == to.expert);
    // the only tile of its expert: nothing to order or share (100 tokens, 32 experts, a call 39.8 -> 39.4 us)
    if ((same >> 31 & 7) == 2) return ExpertTile{nt, m, to.expert, __builtin_amdgcn_readlane(t.y, 32), __builtin_amdgcn_readlane(t.z, 32)};
    const int back = __builtin_clz(~(uint32_t)same | 1), ahead = __builtin_ctz(~(uint32_t)(same >> 33));
    const bool all_seen = back + 1 + ahead < 32;     // (lane 0's and lane 63's are not of it then); otherwise the eight around this one that are
    int from = m - back, to_end = m + ahead + 1;
    const int n = to_end - from, t0 = from;
    to.nt = nt, to.mt = m;
    if (rows) {
        if (!all_seen) {
            from = from > (m & ~7) ? from : m & ~7;
            to_end = to_end < (m | 7) + 1 ? to_end : (m | 7) + 1;
        }
        from = from > lo ? from : lo;
        to_end = to_end < hi ? to_end : hi;
        int in = idx - (from - lo) * nx;
        const int span = to_end - from, groups = (span + rows - 1) / rows;
        rows = few_over(span + groups - 1, groups);    // nine tiles: five and four
        const int g = few_over(in, rows * nx), left = span - rows * g, gm = left < rows ? left : rows;
        in -= g * rows * nx;
        to.nt = few_over(in, gm);
        to.mt = from + rows * g + in - to.nt * gm;
    }
    to.first = __builtin_amdgcn_readlane(t.y, to.mt - m + 32);
    to.live = __builtin_amdgcn_readlane(t.z, to.mt - m + 32);
    if (all_seen && n > 1) {
        const int all = (n - 1) * TM + __builtin_amdgcn_readlane(t.z, t0 + n - 1 - m + 32), each = few_over(all + n * UNIT - 1, n * UNIT) * UNIT, nth = to.mt - t0;
        to.first += nth * (each - TM);
        to.live = all - nth * each < each ? all - nth * each : each;
    }
    return to;
}

// 16-byte pieces of an image's row are xor-ed with 0, 2, 3, 1 for rows 0-3, 4-7, 8-11, 12-15: a 16-byte read takes lanes 0-3, 12-15 and 20-27 of 32 in one cycle, the others
// in the next, and either set of 16 (8 rows at one column, the 8 other rows at the next one) then spreads over all banks
__device__ __forceinline__ int image_swizzle(int r) { return (0x78 >> ((r >> 1) & 6)) & 3; }

// What a lane asks for: its piece of each DMA instruction of an image, 16 rows of 64 bytes.  A wave whose pieces are of pairs that do not exist leaves them out (weights come first).
template <class G>
struct ExpertFeed {
    const uint16_t* src[G::DMA];
    bool feeds;
    __device__ __forceinline__ void aim(bool glu, const MoeGemmArgs& a, const ExpertTile& to, int wave, int lane) {
        const uint16_t* w = reinterpret_cast<const uint16_t*>(a.w) + (int64_t)to.expert * (glu ? 2 : 1) * a.n * a.k;
        const int col0 = to.nt * (glu ? G::TN / 2 : G::TN);
#pragma unroll
        for (int j = 0; j < G::DMA; ++j) {
            const int R = (wave * G::DMA + j) * 16 + (lane >> 2), piece = ((lane & 3) ^ image_swizzle(R)) * 8;
            if (R < G::TN) {
                int col = col0 + (glu ? (R >> 5) * 16 + (R & 15) : R);
                if (col >= a.n) col = a.n - 1;
                src[j] = w + (int64_t)(glu && (R & 16) ? a.n + col : col) * a.k + piece;
            } else {
                const int r = R - G::TN, pair = a.slot_pair[to.first + (r < to.live ? r : to.live - 1)];
                src[j] = reinterpret_cast<const uint16_t*>(a.x) + (glu ? (int64_t)(pair / a.top) * a.x_stride : (int64_t)pair * a.k) + piece;
            }
        }
        feeds = wave * G::DMA * 16 < G::TN + to.live;
    }
    __device__ __forceinline__ void stage(unsigned char* lds, int it, int buf, int wave) const {
        if (!feeds) return;
#pragma unroll
        for (int j = 0; j < G::DMA; ++j) dma16(src[j] + it * TK, lds + buf * G::IMG + (wave * G::DMA + j) * 1024);
    }
    // (images past the last one are asked for again: every iteration leaves the same number of loads in flight, without a branch)
    __device__ __forceinline__ void stage_next(unsigned char* lds, int it, int iters, int wave) const { stage(lds, it < iters ? it : iters - 1, it % kRing, wave); }
    __device__ __forceinline__ void begin(unsigned char* lds, int iters, int wave) const {
#pragma unroll
        for (int it = 0; it < kRing; ++it) stage_next(lds, it, iters, wave);
    }
};

// Rows of pairs that do not exist are not multiplied: the waves along the rows share the tiles of 16 that there are.  (100 tokens' pairs in tiles of 256: 207 -> 179 us; in tiles of
// 128: 167 -> 160; of 16384 tokens, 8 tiles of 256 an expert: 1367 -> 1340, when the first waves were full and the last ones did without; shared evenly, 25 pairs an expert in tiles of
// 128: 162 -> 155)
struct WaveRows {
    int row0, mine;                                  // pairs of a wave, from row0 on (none: <= 0)
    __device__ __forceinline__ WaveRows(int live, int wm, int waves) {
        const int part = ((live + 15) / 16 + waves - 1) / waves;
        row0 = 16 * wm * part;
        mine = live - row0 < 16 * part ? live - row0 : 16 * part;
    }
};

// D[weight row 16 i + 4 lg + r][pair 16 j + lq] of a wave, behind start (0); the images have been begun.
// landed(): behind the barrier after the first image.
template <int MW, int NW, int MT, int NT, class Landed>
__device__ __forceinline__ void expert_sums(f32x4 (&acc)[NT][MT], const ExpertFeed<GemmShape<MW, NW, MT, NT>>& feed, unsigned char* lds, int iters, const WaveRows& rows, int wave, int lane,
                                            float start, Landed landed) {
    using G = GemmShape<MW, NW, MT, NT>;
    constexpr int TN = G::TN, DMA = G::DMA;
    const int lq = lane & 15, lg = lane >> 4, wn = wave % NW, mine = rows.mine;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{start, start, start, start};
    // the oldest image in flight has landed (`younger` behind it), and everyone has read the one before it
    auto arrive = [&](auto younger) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(younger)::value * DMA) : "memory");
        lds_only_barrier();
    };
    constexpr std::integral_constant<int, kRing - 2> in_flight{};
    // the products of this wave's first MTU tiles of pairs
    auto run = [&](auto mtu) __attribute__((always_inline)) {
        constexpr int MTU = decltype(mtu)::value;
        struct Operands {
            bf16x8 w[NT], x[MTU];
        };
        Operands even, odd;                          // of the image being multiplied and of the next one, read meanwhile
        auto read = [&](int it, Operands& f) __attribute__((always_inline)) {
            const int at = (it % kRing) * G::IMG + lq * 64 + (lg ^ image_swizzle(lq)) * 16;
            const unsigned char* wimg = lds + at + wn * NT * 16 * 64;
            const unsigned char* ximg = lds + at + (TN + rows.row0) * 64;
#pragma unroll
            for (int t = 0; t < NT; ++t) f.w[t] = *reinterpret_cast<const bf16x8*>(wimg + t * 16 * 64);
#pragma unroll
            for (int t = 0; t < MTU; ++t) f.x[t] = *reinterpret_cast<const bf16x8*>(ximg + t * 16 * 64);
        };
        // reads and loads spread between the products
        auto spread = []() __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < NT + MTU; ++k) {
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);             // LDS read
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);             // MFMA
            }
#pragma unroll
            for (int k = 0; k < DMA; ++k) {
                __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);             // load
                __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
            }
        };
        auto multiply = [&](const Operands& f) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < MTU; ++j)
#pragma unroll
                for (int i = 0; i < NT; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[i], f.x[j], acc[i][j], 0, 0, 0);
        };
        read(0, even);
        for (int it = 0; it < iters; it += 2) {
            arrive(in_flight);
            read(it + 1, odd);
            feed.stage_next(lds, it + kRing, iters, wave);
            multiply(even);
            spread();
            arrive(in_flight);
            read(it + 2, even);                      // (behind the last image: read and not used)
            feed.stage_next(lds, it + 1 + kRing, iters, wave);
            multiply(odd);
            spread();
        }
    };
    arrive(std::integral_constant<int, kRing - 1>{});
    landed();
    constexpr int STEP = G::STEP;                    // (in quarters: a copy of the loop for each)
    if (mine > (MT - STEP) * 16) {
        run(std::integral_constant<int, MT>{});
    } else if (MT > 2 && mine > (MT - 2 * STEP) * 16) {
        run(std::integral_constant<int, MT - STEP>{});
    } else if (MT > 2 && mine > STEP * 16) {
        run(std::integral_constant<int, MT / 2>{});
    } else if (mine > 0) {
        run(std::integral_constant<int, STEP>{});
    } else {
        for (int it = 0; it < iters; ++it) {
            arrive(in_flight);
            feed.stage_next(lds, it + kRing, iters, wave);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_only_barrier();                              // the images are done with
}

// Results through LDS (2048 bytes a wave, room), 16 or 32 rows at a time, and whole rows of the wave's columns to memory.  THROUGH: past the caches.  (All rows at once, with what names
// their places loaded behind: 2048 wide, 16384 tokens 1182 -> 1167 us)
// between(h): before the first, the third and the fifth eighth of them.
template <bool GLU, bool THROUGH, int MW, int NW, int MT, int NT, class Between>
__device__ __forceinline__ void expert_results(const f32x4 (&acc)[NT][MT], const MoeGemmArgs& a, const ExpertTile& to, const WaveRows& rows, unsigned char* room, int wave, int lane,
                                               Between between) {
    using G = GemmShape<MW, NW, MT, NT>;
    constexpr int CW = GLU ? NT * 8 : NT * 16, CP = CW / 8, PR = 1024 / CW, PASSES = MT * 16 / PR;      // columns of a wave, 16-byte pieces of a row; rows of a pass
    static_assert(PR % 16 == 0 && PR * CP == 128 && PASSES >= 1, "two pieces a lane and pass");
    const int lq = lane & 15, lg = lane >> 4, wn = wave % NW, mine = rows.mine;
    const int col = to.nt * (GLU ? G::TN / 2 : G::TN) + wn * CW + (lane % CP) * 8;
    int pair[2 * PASSES];
#pragma unroll
    for (int k = 0; k < 2 * PASSES; ++k) {
        const int r = (k * 64 + lane) / CP;
        pair[k] = a.slot_pair[to.first + (mine > 0 ? rows.row0 + (r < mine ? r : mine - 1) : 0)];
    }
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
        if (8 * p % (2 * PASSES) == 0 && 8 * p / (2 * PASSES) < 3) between(8 * p / (2 * PASSES));
        if (mine <= p * PR) continue;
#pragma unroll
        for (int jj = 0; jj < PR / 16; ++jj) {
            const int j = p * (PR / 16) + jj, r = 16 * jj + lq;
            auto put = [&](int c, f32x4 v) {         // columns c .. + 3 of row r
                act_st4(reinterpret_cast<uint16_t*>(room + r * CW * 2 + (((c >> 3) ^ (r & (CP - 1))) * 16 + (c & 4) * 2)), v);
            };
            if constexpr (GLU) {
#pragma unroll
                for (int i = 0; i < NT / 2; ++i) {
                    f32x4 v;
#pragma unroll
                    for (int q = 0; q < 4; ++q) v[q] = expert_unit(a, acc[2 * i][j][q], acc[2 * i + 1][j][q]);
                    put(16 * i + 4 * lg, v);
                }
            } else {
#pragma unroll
                for (int i = 0; i < NT; ++i) put(16 * i + 4 * lg, acc[i][j]);
            }
        }
        wave_lds_sync();
        u32x4 v[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int r = (k * 64 + lane) / CP;
            v[k] = *reinterpret_cast<const u32x4*>(room + r * CW * 2 + ((lane % CP) ^ (r & (CP - 1))) * 16);
        }
        wave_lds_sync();
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            if (p * PR + (k * 64 + lane) / CP < mine && col < a.n) {           // (n is a multiple of 64: whole pieces)
                uint16_t* dst = reinterpret_cast<uint16_t*>(a.out) + (int64_t)pair[2 * p + k] * a.n + col;
                if (THROUGH) st16_global_sc1(dst, v[k]);
                else *reinterpret_cast<u32x4*>(dst) = v[k];
            }
        }
    }
}

template <bool GLU, int MW, int NW, int MT, int NT>
__global__ __launch_bounds__(64 * MW * NW) void moe_gemm_kernel(const MoeGemmArgs a) {
    using G = GemmShape<MW, NW, MT, NT>;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];        // [ring][TN weight rows | TM pairs][64 bytes]
    // one XCD takes a run of the parts
    const int nx = gridDim.x, tiles = a.tiles[3], total = nx * tiles, lin = (int)(blockIdx.x + gridDim.x * blockIdx.y), per = total >> 3;
    if (lin >= total) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const ExpertTile to = find_tile<G::TM, G::UNIT>(a.tiles, tiles, nx, lin < per * 8 ? (lin & 7) * per + (lin >> 3) : lin, 0, tiles, total <= kAlone ? 0 : 8, lane);
    const int iters = a.k / TK;                      // (k is a multiple of 64: even)
    ExpertFeed<G> feed;
    feed.aim(GLU, a, to, wave, lane);
    feed.begin(lds, iters, wave);
    const WaveRows rows(to.live, wave / NW, MW);
    f32x4 acc[NT][MT];
    expert_sums<MW, NW, MT, NT>(acc, feed, lds, iters, rows, wave, lane, 0.f, [] {});
    expert_results<GLU, false, MW, NW, MT, NT>(acc, a, to, rows, lds + wave * 2048, wave, lane, [](int) {});
}

// Both products in one launch of workgroups that stay: the parts of the second one fill the CUs that the last round of the first one leaves idle, and the other way round at its head.
// A row of tiles is split over eight lists, one for the workgroups of an XCD; a list is its tiles' parts of the first product and behind them those of the second one, drawn by ticket.
// Whose list is at an end draws from the next one's.  A part of the second product waits until all columns of its row tile are stored, and those were drawn before it
// from the same list: they are in the hands of workgroups that run, and never wait; who waits keeps no other part waiting.  (No assumption on how many are resident, on their order,
// or on who runs where; the wait is bounded all the same: behind one that ran out the part's outputs are NaN, and a word beside the tickets says so.)
// What the second product reads is stored through to memory, announced behind the stores' arrival, and lies in lines of its own (rows of whole 128 bytes): no cache holds an older copy.
// The next part is looked up, and its first images asked for if its rows are there, while this one's results leave: the ring is free by then, they have LDS of their own.
// A wave waits for its stores once all are out, beside those images; they are announced behind the next part's first barrier.
// Bound by the products while they run (0.95 us an image of 256 x 256, the rate of a large product at the clock the card keeps under it); a part of 64 images at 2048 wide is 60 us of those
// and, before, 4.5 of lookups and first images and 6 to 8 of results.  3000 tokens, 32 experts of 1536: 371 us in two launches, 313 with the parts one after the other, 308 overlapped;
// 12000 966, 935, 930; 1024 wide, of 768, 6000 176, 164, 160.  (Announced from the next part's loop without a wait of its own: 1 % slower, rows came later to those who waited)
// Few operations on shared words: 256 workgroups that look at eight lists when theirs is at an end took 25 us for it.
constexpr int kListWords = 32, kRanOut = 16;         // tickets a line each; in the first line, whether a wait ran out
constexpr uint32_t kWaitLimit = 1 << 22;             // polls of about a microsecond
struct MoeBothArgs {
    MoeGemmArgs up, down;
    uint32_t* tickets;                               // [8][kListWords], zero; then per row tile its stored columns, [tiles][kListWords], zero
    uint32_t wait_limit, missing;                    // columns waited for that nobody stores (tests: the wait that runs out)
};
template <int MW, int NW, int MT, int NT>
constexpr size_t both_lds_bytes() { return GemmShape<MW, NW, MT, NT>::LDS + MW * NW * 2048 + 16; }
template <int MW, int NW, int MT, int NT>
__global__ __launch_bounds__(64 * MW * NW) void moe_both_kernel(const MoeBothArgs a) {
    using G = GemmShape<MW, NW, MT, NT>;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    int* const next = reinterpret_cast<int*>(lds + G::LDS + G::WAVES * 2048);  // list (-1: at the end), number in it; whether the rows are there
    uint32_t* const stored = a.tickets + 8 * kListWords;
    const int tiles = a.up.tiles[3], nx = (a.up.n + G::TN / 2 - 1) / (G::TN / 2), ny = (a.down.n + G::TN - 1) / G::TN;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    unsigned char* const room = lds + G::LDS + wave * 2048;
    const auto begin = [&](int list) { return (int)((int64_t)tiles * list >> 3); };
    const auto parts = [&](int list) { return (begin(list + 1) - begin(list)) * (nx + ny); };
    const auto draw = [&](int list) {                // (a wave)
        uint32_t t = 0;
        if (lane_now() == 0) t = __hip_atomic_fetch_add(a.tickets + list * kListWords, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return t;
    };
    const auto settle = [&](int list, uint32_t ticket) {                       // (a wave) that ticket, or one of the first later list that has any
        int number = __builtin_amdgcn_readfirstlane(ticket);
        if (number >= parts(list)) {                 // (all lists' tickets at once, one per lane: what is at an end stays there)
            const int one = lane_now() & 7;
            const uint32_t seen = __hip_atomic_load(a.tickets + one * kListWords, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const uint32_t open = (uint32_t)__builtin_amdgcn_ballot_w64((int)seen < parts(one)) & 0xFF;
            uint32_t later = (open | open << 8) >> (list + 1) & 0x7F;          // list + 1, list + 2, ..
            const int was = list;
            list = -1;
            while (later) {
                const int next_one = (was + 1 + __builtin_ctz(later)) & 7;
                number = __builtin_amdgcn_readfirstlane(draw(next_one));
                if (number < parts(next_one)) {
                    list = next_one;
                    break;
                }
                later &= later - 1;
            }
        }
        if (lane_now() == 0) {
            next[0] = list;
            next[1] = number;
        }
    };
    const auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    struct Part {
        int list;                                    // -1: none
        bool glu;
        ExpertTile to;
    };
    Part now, then;
    ExpertFeed<G> feed;
    const auto take = [&](Part& part, int lane) {    // the one that was settled
        const int list = uniform(next[0]), number = uniform(next[1]);
        part.list = list;
        if (list < 0) return;
        const int lo = begin(list), hi = begin(list + 1), first = (hi - lo) * nx;
        part.glu = number < first;
        const ExpertTile to = find_tile<G::TM, G::UNIT>(a.up.tiles, tiles, part.glu ? nx : ny, part.glu ? number : number - first, lo, hi, tiles < 128 ? 4 : 8, lane);
        part.to = ExpertTile{uniform(to.nt), uniform(to.mt), uniform(to.expert), uniform(to.first), uniform(to.live)};
    };
    const uint32_t all_columns = (uint32_t)nx + a.missing;
    const auto columns = [&](int mt) { return __hip_atomic_load(stored + mt * kListWords, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    int announce = -1;                               // a row tile whose columns are on their way to memory
    const auto announce_it = [&]() {
        if (announce >= 0 && wave == 0 && lane_now() == 0) __hip_atomic_fetch_add(stored + announce * kListWords, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        announce = -1;
    };
    const auto arrived = [&]() {                     // all that the workgroup has stored
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_only_barrier();
        announce_it();
    };
    uint32_t drawn = 0;                              // the part behind the one that has begun
    const auto go = [&](const Part& part) {
        if (wave == 0) drawn = draw(part.list);
        feed.begin(lds, (part.glu ? a.up.k : a.down.k) / TK, wave);
    };
    if (wave == 0) settle(blockIdx.x & 7, draw(blockIdx.x & 7));
    lds_only_barrier();
    take(then, lane_now());
    bool begun = false;
    if (then.list >= 0) feed.aim(then.glu, then.glu ? a.up : a.down, then.to, wave, lane_now());
    while (then.list >= 0) {
        float start = 0.f;
        if (!begun) {
            arrived();                               // (before it waits for anyone)
            if (!then.glu) {
                if (wave == 0 && lane_now() == 0) {
                    uint32_t tries = 0;
                    while (columns(then.to.mt) < all_columns && ++tries < a.wait_limit) __builtin_amdgcn_s_sleep(8);
                    next[2] = tries < a.wait_limit;
                    if (tries >= a.wait_limit) __hip_atomic_store(a.tickets + kRanOut, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                lds_only_barrier();
                if (!uniform(next[2])) start = __uint_as_float(0x7FC00000u);
            }
            go(then);
        }
        now = then;
        const int lane = lane_now();                 // (what hangs on it is computed for each part: held over the loop it would take too many registers)
        const WaveRows rows(now.to.live, wave / NW, MW);
        f32x4 acc[NT][MT];
        expert_sums<MW, NW, MT, NT>(
            acc, feed, lds, (now.glu ? a.up.k : a.down.k) / TK, rows, wave, lane, start,
            [&] {
                announce_it();
                if (wave == 0) settle(now.list, drawn);
            });
        const auto between = [&](int h) __attribute__((always_inline)) {
            if (h == 0) {
                take(then, lane_now());
            } else if (h == 1) {
                if (then.list >= 0) feed.aim(then.glu, then.glu ? a.up : a.down, then.to, wave, lane_now());
                if (wave == 0 && lane_now() == 0) next[2] = then.list >= 0 && (then.glu || columns(then.to.mt) >= all_columns);
            } else {
                lds_only_barrier();
                begun = uniform(next[2]);
                if (begun) go(then);
            }
        };
        if (now.glu) {
            expert_results<true, true, MW, NW, MT, NT>(acc, a.up, now.to, rows, room, wave, lane_now(), between);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                   // (announced behind the next barrier)
            announce = now.to.mt;
        } else {
            expert_results<false, false, MW, NW, MT, NT>(acc, a.down, now.to, rows, room, wave, lane_now(), between);
        }
    }
    arrived();
}

template <bool GLU, int MW, int NW, int MT, int NT>
void gemm_shape(const MoeGemmArgs& a, hipStream_t stream) {
    using G = GemmShape<MW, NW, MT, NT>;
    const int outs = GLU ? G::TN / 2 : G::TN;
    if (G::LDS > 64 * 1024)
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(moe_gemm_kernel<GLU, MW, NW, MT, NT>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)G::LDS);
    moe_gemm_kernel<GLU, MW, NW, MT, NT><<<dim3((a.n + outs - 1) / outs, a.max_tiles), 64 * G::WAVES, G::LDS, stream>>>(a);
}

// ------------------------------------------------------------------------------------------------ products, at most 64 rows (bf16)
// grid (n / (16 x waves' tiles), experts): the pairs of the expert are found from the ids; an expert nobody chose costs one scan.
// SPLIT: the 4 waves share one 16-column tile and split the contraction; otherwise every wave owns a tile.
template <bool GLU, int MT, bool SPLIT>
__device__ __forceinline__ void moe_small_tile(const MoeGemmArgs& a, int expert, int n0, int s0, int s1, const int* list, int count, float* red, int wave, int lane) {
    const int lq = lane & 15, lg = lane >> 4;
    const uint16_t* w = reinterpret_cast<const uint16_t*>(a.w) + ((int64_t)expert * (GLU ? 2 : 1) * a.n + n0 + lq) * a.k + 8 * lg;
    const uint16_t* x[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int p = list[16 * m + lq < count ? 16 * m + lq : count - 1];
        x[m] = reinterpret_cast<const uint16_t*>(a.x) + (GLU ? (int64_t)(p / a.top) * a.x_stride : (int64_t)p * a.k) + 8 * lg;
    }
    f32x4 g[MT], u[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) g[m] = u[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int UN = GLU ? (MT > 2 ? 2 : 4) : (MT > 2 ? 4 : 8);
    const int64_t up = (int64_t)a.n * a.k;
    int s = s0;
    for (; s + UN <= s1; s += UN) {
        bf16x8 wg[UN], wu[UN], xf[UN][MT];
#pragma unroll
        for (int i = 0; i < UN; ++i) {
            wg[i] = *reinterpret_cast<const bf16x8*>(w + 32 * (s + i));    // (half of a 128-byte line: a streaming hint would drop the other half)
            if constexpr (GLU) wu[i] = *reinterpret_cast<const bf16x8*>(w + up + 32 * (s + i));
        }
#pragma unroll
        for (int i = 0; i < UN; ++i)
#pragma unroll
            for (int m = 0; m < MT; ++m) xf[i][m] = *reinterpret_cast<const bf16x8*>(x[m] + 32 * (s + i));
#pragma unroll
        for (int i = 0; i < UN; ++i)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                g[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wg[i], xf[i][m], g[m], 0, 0, 0);
                if constexpr (GLU) u[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wu[i], xf[i][m], u[m], 0, 0, 0);
            }
    }
    for (; s < s1; ++s) {
        const bf16x8 wg = *reinterpret_cast<const bf16x8*>(w + 32 * s);
        bf16x8 wu = wg;
        if constexpr (GLU) wu = *reinterpret_cast<const bf16x8*>(w + up + 32 * s);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const bf16x8 xf = *reinterpret_cast<const bf16x8*>(x[m] + 32 * s);
            g[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wg, xf, g[m], 0, 0, 0);
            if constexpr (GLU) u[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wu, xf, u[m], 0, 0, 0);
        }
    }
    if constexpr (SPLIT) {                           // red [4 waves][2][MT][64 lanes][4]
        constexpr int W = 2 * MT * 256;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            *reinterpret_cast<f32x4*>(red + wave * W + m * 256 + lane * 4) = g[m];
            if constexpr (GLU) *reinterpret_cast<f32x4*>(red + wave * W + (MT + m) * 256 + lane * 4) = u[m];
        }
        __syncthreads();
        if (wave) return;
#pragma unroll
        for (int k = 1; k < 4; ++k)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                g[m] += *reinterpret_cast<const f32x4*>(red + k * W + m * 256 + lane * 4);
                if constexpr (GLU) u[m] += *reinterpret_cast<const f32x4*>(red + k * W + (MT + m) * 256 + lane * 4);
            }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        if (16 * m + lq >= count) continue;
        f32x4 v = g[m];
        if constexpr (GLU) {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = expert_unit(a, g[m][r], u[m][r]);
        }
        act_st4(reinterpret_cast<uint16_t*>(a.out) + (int64_t)list[16 * m + lq] * a.n + n0 + 4 * lg, v);
    }
}

template <bool GLU, bool SPLIT>
__global__ __launch_bounds__(256) void moe_small_kernel(const MoeGemmArgs a) {
    __shared__ int list[64];
    __shared__ int count_s;
    __shared__ __attribute__((aligned(16))) float red[SPLIT ? 4 * 2 * 4 * 256 : 4];
    const int expert = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (wave == 0) {                                 // (an expert is chosen at most once per row: at most 64 pairs)
        int n = 0;
        for (int p0 = 0; p0 < a.pairs; p0 += 64) {
            const bool mine = p0 + lane < a.pairs && a.ids[p0 + lane] == expert;
            const uint64_t ball = __builtin_amdgcn_ballot_w64(mine);
            const int at = n + __popcll(ball & ((1ull << lane) - 1));
            if (mine && at < 64) list[at] = p0 + lane;
            n += __popcll(ball);
        }
        if (lane == 0) count_s = n < 64 ? n : 64;
    }
    __syncthreads();
    const int count = __builtin_amdgcn_readfirstlane(count_s);
    if (count == 0) return;
    const int tile = SPLIT ? blockIdx.x : blockIdx.x * 4 + wave, steps = a.k / 32;
    if (tile * 16 >= a.n) return;                    // (whole waves; only the form without a later barrier has such tiles)
    const int per = (steps + 3) / 4, s0 = SPLIT ? wave * per : 0, s1 = SPLIT ? (s0 + per < steps ? s0 + per : steps) : steps;
    if (count <= 16) moe_small_tile<GLU, 1, SPLIT>(a, expert, tile * 16, s0, s1, list, count, red, wave, lane);
    else if (count <= 32) moe_small_tile<GLU, 2, SPLIT>(a, expert, tile * 16, s0, s1, list, count, red, wave, lane);
    else moe_small_tile<GLU, 4, SPLIT>(a, expert, tile * 16, s0, s1, list, count, red, wave, lane);
}

// ------------------------------------------------------------------------------------------------ products in 32-bit
// 64 pairs x 64 outputs per workgroup, 16 of the contraction at a time through LDS, 4 x 4 outputs per thread
constexpr int FM = 64;

template <bool GLU>
__global__ __launch_bounds__(256) void moe_gemm_f32_kernel(const MoeGemmArgs a) {
    __shared__ __attribute__((aligned(16))) float xs[16][FM + 4], ws[2][16][64 + 4];
    const int mt = blockIdx.y, n0 = blockIdx.x * 64, tid = threadIdx.x;
    const int expert = a.tiles[4 * mt], first = a.tiles[4 * mt + 1], live = a.tiles[4 * mt + 2];
    if (live <= 0) return;
    const float* w = reinterpret_cast<const float*>(a.w) + (int64_t)expert * (GLU ? 2 : 1) * a.n * a.k;
    const int lr = tid >> 2, lc = (tid & 3) * 4;     // staging: row lr, 4 of the contraction
    const int pair = a.slot_pair[first + (lr < live ? lr : live - 1)];
    const float* x = reinterpret_cast<const float*>(a.x) + (GLU ? (int64_t)(pair / a.top) * a.x_stride : (int64_t)pair * a.k) + lc;
    const float* wr = w + (int64_t)(n0 + lr) * a.k + lc;
    const int tm = (tid >> 4) * 4, tn = (tid & 15) * 4;
    float g[4][4] = {}, u[4][4] = {};
    for (int k0 = 0; k0 < a.k; k0 += 16) {
        const f32x4 xv = *reinterpret_cast<const f32x4*>(x + k0), gv = *reinterpret_cast<const f32x4*>(wr + k0);
        f32x4 uv = gv;
        if constexpr (GLU) uv = *reinterpret_cast<const f32x4*>(wr + (int64_t)a.n * a.k + k0);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            xs[lc + i][lr] = xv[i];
            ws[0][lc + i][lr] = gv[i];
            if constexpr (GLU) ws[1][lc + i][lr] = uv[i];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const f32x4 m = *reinterpret_cast<const f32x4*>(&xs[k][tm]), n = *reinterpret_cast<const f32x4*>(&ws[0][k][tn]);
            f32x4 n2 = n;
            if constexpr (GLU) n2 = *reinterpret_cast<const f32x4*>(&ws[1][k][tn]);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    g[i][j] += m[i] * n[j];
                    if constexpr (GLU) u[i][j] += m[i] * n2[j];
                }
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (tm + i >= live) continue;
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[j] = g[i][j];
            if constexpr (GLU) {
                if (a.alpha != 0.f) {
                    const float gate = fminf(g[i][j], a.limit);
                    v[j] = gate / (1.f + expf(-a.alpha * gate)) * (fminf(fmaxf(u[i][j], -a.limit), a.limit) + 1.f);
                } else {
                    v[j] = g[i][j] / (1.f + expf(-g[i][j])) * u[i][j];
                }
            }
        }
        *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.out) + (int64_t)a.slot_pair[first + tm + i] * a.n + n0 + tn) = v;
    }
}

}  // namespace

int launch_moe_route(const MoeRouteArgs& a, int f32, hipStream_t stream) {
    if (!f32 && a.cols % 32 == 0) {
        const int ez = (a.experts + 63) / 64 * 64;
        const size_t lds = (size_t)(8 * 16 * 68 + 24 * ez + 8 * a.groups) * 4;
        if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(moe_route_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        const int live = a.rows <= 256 ? 2 : a.rows <= 2048 ? 8 : 16;           // few rows: more workgroups, shorter choice
        moe_route_kernel<<<(a.rows + live - 1) / live, 512, lds, stream>>>(a, live);
    } else {
        const size_t lds = (size_t)(2 * a.experts + a.groups) * 4;
        if (f32) moe_route_generic_kernel<float><<<a.rows, 256, lds, stream>>>(a);
        else moe_route_generic_kernel<uint16_t><<<a.rows, 256, lds, stream>>>(a);
    }
    return check_launch("moe_route");
}

int moe_dispatch_blocks(int pairs) { return (pairs + DP - 1) / DP; }

int launch_moe_dispatch(int32_t* slot_pair, int32_t* tiles, int32_t* counts, const int32_t* ids, int pairs, int experts, int tile_rows, int max_tiles,
                        uint32_t* clear, size_t clear_words, hipStream_t stream) {
    const int grid = moe_dispatch_blocks(pairs);
    if (pairs <= kCountHere) {
        moe_scatter_kernel<false><<<grid, 256, 0, stream>>>(slot_pair, tiles, counts, ids, pairs, experts, tile_rows, max_tiles, clear, (int)clear_words);
        return check_launch("moe_scatter");
    }
    moe_count_kernel<<<grid, 256, 0, stream>>>(counts, ids, pairs, experts);
    const int rc = check_launch("moe_count");
    if (rc) return rc;
    moe_scatter_kernel<true><<<grid, 256, 0, stream>>>(slot_pair, tiles, counts, ids, pairs, experts, tile_rows, max_tiles, clear, (int)clear_words);
    return check_launch("moe_scatter");
}

// Rows of a tile, by the pairs an expert has on average and by all columns of the experts (`wide`: how many workgroups a row of tiles is).  us at 2048 wide, experts of 1536, and
// at 1024, of 768; 8 to 128 experts, even and crowded (the k-th one k^-0.6 as often) routes:
// - few pairs: 64, whose images leave room for three workgroups on a CU, as the weight stream wants: 32 experts of 1536, 8 pairs 138 against 147 with 128 rows, 16 155 against 167.
//   From 17 to 25 pairs many wide experts lose with them where a route crowds some (0.92 to 0.95 of the speed); up to 36864 columns in all it is the same or better.
// - 256, twice the products per byte of weights and rows read, where an expert's pairs mostly fit one such tile or fill several, and there are tiles enough:
//   from 110 pairs on, 32 experts of 1536, 125 206 against 230, 150 212 against 244; with 98304 columns already from 100 on (64 experts of 1536 0.90 to 0.96 with 128);
//   193 to 240, below 24576 columns half the CUs and more would get none: 8 experts 1.28 to 2.1 times as fast with 128, 16 of 768 1.3 to 1.65;
//   256 to 287, where the second tile is mostly empty, 128 is 1.0 to 1.9 times as fast up to 36864 columns (24 of 1536, 48 of 768), 256 from 49152 on (128 experts 0.79 to 0.93 with 128);
//   more: 32 of 1536, 350 316 against 375, 500 418 against 485.
int moe_tile_rows(int pairs, int experts, int n, int f32) {
    if (f32) return FM;
    const int mean = pairs / experts;
    const int64_t wide = (int64_t)experts * n;
    if (mean <= 16 || (mean <= 25 && wide < 49152)) return 64;
    const bool large = mean >= 288 ? true : mean >= 256 ? wide >= 49152 : mean > 240 ? false : mean >= 193 ? wide >= 24576 : mean >= 110 || (mean >= 100 && wide >= 98304);
    return large ? 256 : 128;
}

// compute units of the current device (256 on MI355X), read once
static int device_cus() {
    static const int n = [] {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
        return v;
    }();
    return n;
}

// Whether both products go in one launch: tiles of 256 rows (a workgroup a CU) that are enough, as far as the pairs tell, for two and a half rounds of the CUs and some experts with two
// tiles, and a second product whose parts, which come last, are not the longer ones.  us of four routes each, two launches against one: 2048 wide, 32 experts of 1536, 170 pairs an expert
// 205 against 212, 190 223 against 220, 220 250 against 223, 290 279 against 272, 375 302 against 295, 430 383 against 339, 600 448 against 435, 1000 681 against 666; 1024 wide, of 768,
// 240 (1.8 rounds) 85 against 101, 330 (2.2) 105 against 109, 375 (2.4) 112 against 112, 400 (2.6) 126 against 113, 460 136 against 117, 1000 238 against 209; 4096 wide, of 512, 170
// 177 against 182, 190 193 against 185, 375 269 against 242, 550 362 against 308; 24 experts of 1536 at 2048, 220 202 against 206, 240 220 against 202.  768 wide, 16 experts of 2048,
// 500 to 600 142 to 150 against 144 to 152, around them up to 1.16 times as fast.  From 20 rounds on the idle ends are little against what each part's hand-over
// costs: 2048 wide, 16384 tokens by sigmoids 1106 against 1118, by a softmax 1256 against 1240.  Tiles of 128 rows, two workgroups a CU, fill their rounds better as they are:
// 32 experts of 1536, 2048 wide, 60 pairs 158 against 164.
bool moe_one_launch(int pairs, int experts, int n, int cols, int tile_rows) {
    if (tile_rows != 256 || pairs / experts < 180 || n > cols) return false;
    const int64_t tiles = pairs / 256 + experts / 2, parts = tiles * ((n + 127) / 128 + (cols + 255) / 256);
    return 2 * parts >= 5 * device_cus() && parts < 20 * device_cus();
}
size_t moe_links_words(int tile_rows, int max_tiles) { return tile_rows == 256 ? (size_t)(8 + max_tiles) * kListWords : 0; }

const uint32_t* moe_ran_out(const uint32_t* tickets) { return tickets + kRanOut; }

int launch_moe_both(const MoeGemmArgs& up, const MoeGemmArgs& down, uint32_t* tickets, uint32_t wait_limit, uint32_t missing, hipStream_t stream) {
    using G = GemmShape<2, 4, 8, 4>;
    const size_t lds = both_lds_bytes<2, 4, 8, 4>();
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(moe_both_kernel<2, 4, 8, 4>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    const int64_t parts = (int64_t)up.max_tiles * ((up.n + G::TN / 2 - 1) / (G::TN / 2) + (down.n + G::TN - 1) / G::TN);
    moe_both_kernel<2, 4, 8, 4><<<(int)(parts < device_cus() ? parts : device_cus()), 64 * G::WAVES, lds, stream>>>(
        MoeBothArgs{up, down, tickets, wait_limit ? wait_limit : kWaitLimit, missing});
    return check_launch("moe_both");
}

int launch_moe_gemm(const MoeGemmArgs& a, int f32, hipStream_t stream) {
    if (f32) {
        const dim3 grid(a.n / 64, a.max_tiles);
        if (a.glu) moe_gemm_f32_kernel<true><<<grid, 256, 0, stream>>>(a);
        else moe_gemm_f32_kernel<false><<<grid, 256, 0, stream>>>(a);
    } else if (!a.tiles) {
        const int tiles = a.n / 16, busy = a.pairs < a.experts ? a.pairs : a.experts;
        const bool split = a.k >= 2048 || (int64_t)busy * tiles < 4 * 512;     // a long contraction, or too few waves with a tile each: four share one
        const dim3 grid(split ? tiles : (tiles + 3) / 4, a.experts);
        if (a.glu && split) moe_small_kernel<true, true><<<grid, 256, 0, stream>>>(a);
        else if (a.glu) moe_small_kernel<true, false><<<grid, 256, 0, stream>>>(a);
        else if (split) moe_small_kernel<false, true><<<grid, 256, 0, stream>>>(a);
        else moe_small_kernel<false, false><<<grid, 256, 0, stream>>>(a);
    } else {
        if (a.tile_rows == 256) {
            if (a.glu) gemm_shape<true, 2, 4, 8, 4>(a, stream);
            else gemm_shape<false, 2, 4, 8, 4>(a, stream);
        } else if (a.tile_rows == 64) {
            if (a.glu) gemm_shape<true, 2, 2, 2, 4>(a, stream);
            else gemm_shape<false, 2, 2, 2, 4>(a, stream);
        } else {
            // eight waves of 32 x 64 (94 registers: four on a SIMD) against four of 64 x 64 (146): the rows of pairs that do not exist idle smaller parts, and more waves cover the
            // loads.  50 pairs an expert 189 -> 169 us, 75 196 -> 173, 100 217 -> 209 (1024 wide 64 -> 59, 67 -> 62, 80 -> 73)
            if (a.glu) gemm_shape<true, 4, 2, 2, 4>(a, stream);
            else gemm_shape<false, 4, 2, 2, 4>(a, stream);
        }
    }
    return check_launch("moe_gemm");
}

}  // namespace nvh
