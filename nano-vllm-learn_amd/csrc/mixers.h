// Launcher interface of the paged sink/window attention, lightning attention and mixture-of-experts kernels (the api_*.hip files validate), and the pieces
// their kernels share.
#pragma once
#include "hybrid.h"

namespace nvh {

using AttnPrepArgs = nvh_attn_prep_desc;
using PagedAttendArgs = nvh_paged_attend_desc;
using LightningArgs = nvh_lightning_desc;
using MoeRouteArgs = nvh_moe_route_desc;
using MoeGemmArgs = nvh_moe_gemm_desc;
using ResidualNormArgs = nvh_residual_norm_desc;

constexpr int kRowPieces = 16;                       // 8-element pieces a thread of a row kernel holds at most: rows of up to 256 * 16 * 8 elements
constexpr int kMaxRowCols = 256 * kRowPieces * 8;
constexpr int kAttendTicketWords = 32;               // one arrival ticket per 128-byte line
constexpr int kRowsHeads = 8;                        // query heads of one key/value head a pass over single rows holds at most
constexpr int kLightningChunk = 64;                  // tokens a workgroup takes at a time
constexpr int kMoeMaxExperts = 1024;

int launch_attn_prep(const AttnPrepArgs& a, int f32, hipStream_t stream);
bool paged_attend_supported(int dk, int dv, int block_size);
inline int paged_attend_groups(int heads, int kv_heads) { return (heads / kv_heads + kRowsHeads - 1) / kRowsHeads; }      // passes per key/value head
int launch_paged_attend_rows(const PagedAttendArgs& a, int f32, int generic, hipStream_t stream);
int launch_paged_attend_prompt(const PagedAttendArgs& a, hipStream_t stream);

__host__ __device__ constexpr int score_cols(int heads) { return (heads + 3) / 4 * 4; }          // row length of PagedAttendArgs::scores
bool talk_rows_supported(int heads, int dk, int dv, int block_size);
int launch_talk_rows(const PagedAttendArgs& a, int f32, int generic, hipStream_t stream);
bool talk_prompt_supported(int heads, int kv_heads, int dk, int dv, int block_size);
constexpr float kTalkPromptCap = 1e4f;               // it takes capped scores only
int launch_talk_prompt(const PagedAttendArgs& a, hipStream_t stream);

bool lightning_supported(int dk, int dv);
int launch_lightning_chunks(const LightningArgs& a, int f32, int generic, hipStream_t stream);
int launch_lightning_step(const LightningArgs& a, hipStream_t stream);
int launch_norm_gate(void* out, void* packed, const void* x, const void* gate, const float* w, float eps, int rows, int cols, int n, int64_t x_stride,
                     int64_t gate_stride, int64_t out_stride, int f32, hipStream_t stream);

int launch_moe_route(const MoeRouteArgs& a, int f32, hipStream_t stream);
int moe_dispatch_blocks(int pairs);
int launch_moe_dispatch(int32_t* slot_pair, int32_t* tiles, int32_t* counts, const int32_t* ids, int pairs, int experts, int tile_rows, int max_tiles,
                        uint32_t* clear, size_t clear_words, hipStream_t stream);      // (clear: words set to zero besides)
bool moe_one_launch(int pairs, int experts, int n, int cols, int tile_rows);
size_t moe_links_words(int tile_rows, int max_tiles);    // of that launch
int launch_moe_both(const MoeGemmArgs& up, const MoeGemmArgs& down, uint32_t* tickets, uint32_t wait_limit, uint32_t missing, hipStream_t stream);
const uint32_t* moe_ran_out(const uint32_t* tickets);    // its word: 1 after a wait that ran out
int moe_tile_rows(int pairs, int experts, int n, int f32);
int launch_moe_gemm(const MoeGemmArgs& a, int f32, hipStream_t stream);

int launch_residual_norm(const ResidualNormArgs& a, int f32, hipStream_t stream);
int launch_poly_norm(void* out, void* packed, const void* z, const float* coef, float eps, int rows, int cols, int n, int64_t z_stride, int64_t out_stride, int f32,
                     hipStream_t stream);
int launch_softcap(void* x, float cap, int rows, int cols, int64_t stride, int f32, hipStream_t stream);

// ---- 8 elements of an activation row
struct f32x8 {
    f32x4 a, b;
};
__device__ __forceinline__ f32x8 unpack8(u32x4 r) {
    return {f32x4{bf16_lo(r[0]), bf16_hi(r[0]), bf16_lo(r[1]), bf16_hi(r[1])}, f32x4{bf16_lo(r[2]), bf16_hi(r[2]), bf16_lo(r[3]), bf16_hi(r[3])}};
}
__device__ __forceinline__ f32x8 act_ld8(const uint16_t* p) { return unpack8(*reinterpret_cast<const u32x4*>(p)); }
__device__ __forceinline__ f32x8 act_ld8(const float* p) { return {*reinterpret_cast<const f32x4*>(p), *reinterpret_cast<const f32x4*>(p + 4)}; }
__device__ __forceinline__ void act_st8(uint16_t* p, const f32x8& v) {
    *reinterpret_cast<u32x4*>(p) = u32x4{pack_bf16x2(v.a[0], v.a[1]), pack_bf16x2(v.a[2], v.a[3]), pack_bf16x2(v.b[0], v.b[1]), pack_bf16x2(v.b[2], v.b[3])};
}
__device__ __forceinline__ void act_st8(float* p, const f32x8& v) {
    *reinterpret_cast<f32x4*>(p) = v.a;
    *reinterpret_cast<f32x4*>(p + 4) = v.b;
}
__device__ __forceinline__ float sum4(f32x4 v) { return (v[0] + v[1]) + (v[2] + v[3]); }

__device__ __forceinline__ float wave_sum64(float v) {
    v = group_sum<16>(v);
    v = sum_xor16(v);
    return sum_xor32(v);
}
// Segment that row blockIdx.y of a launch with `walks_each` workgroups per segment walks: the longest portions first (up to 64 of them, whole; segments of cut ones are much
// alike).  Workgroups start in the order of their numbers, all of them at once where they fit: the last ones share a compute unit with others, which should be short, and where some
// wait, the long ones should not.  Uneven portions: 11 of 1090 tokens on average, time mixing with 32 heads 160 -> 137 us; 24 of 670, lightning attention with 16 heads 120 -> 102;
// 30 of 300, scan of 4096 channels 170 -> 158; 5 of 3277, 2048 channels, a state per lane 223 -> 215.  With a compute unit each any order does.
// Two workgroups a compute unit (PAIRS) and fewer than two for each: the longest portions go to the units that get one, and of the others the longest starts beside the shortest (a
// unit takes another workgroup once each has one, in the same order; were it not so, the order would only be another one).  11 portions, 32 heads: 139 -> 130 us; 14 of 857, 120 -> 109;
// 16 of 1000, 146 -> 138.
template <bool PAIRS = false, typename Args>
__device__ __forceinline__ int longest_first(const Args& a, int walks_each) {
    int nth = blockIdx.y;
    if (a.n_chunks > 64 || a.summaries || a.n_chunks * walks_each <= 256) return nth;
    if constexpr (PAIRS) {
        const int each = 256 / walks_each, two = a.n_chunks - each;            // portions whose walks come first, and that share
        if (two <= each) nth = nth < two ? each - two + nth : nth < each ? nth - two : a.n_chunks - 1 - (nth - each);
    }
    const int lane = threadIdx.x & 63, n = a.chunks[4 * (lane < a.n_chunks ? lane : 0) + 1], steps = n > 0 ? (n + 15) >> 4 : 0;
    return nth_largest<10>(steps < 1023 ? steps : 1023, a.n_chunks, nth);
}

// sums of two values over a 256-thread workgroup; `lds` holds 8 floats and is free again after the next barrier
__device__ __forceinline__ void block_sum256x2(float& u, float& v, float* lds) {
    u = wave_sum64(u);
    v = wave_sum64(v);
    if ((threadIdx.x & 63) == 0) {
        lds[threadIdx.x >> 6] = u;
        lds[4 + (threadIdx.x >> 6)] = v;
    }
    __syncthreads();
    u = lds[0] + lds[1] + lds[2] + lds[3];
    v = lds[4] + lds[5] + lds[6] + lds[7];
}

// sums of N values over a 256-thread workgroup; `lds` holds 4 * N floats and is free again after the next barrier
template <int N>
__device__ __forceinline__ void block_sums256(float (&v)[N], float* lds) {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = wave_sum64(v[i]);
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int i = 0; i < N; ++i) lds[4 * i + (threadIdx.x >> 6)] = v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = lds[4 * i] + lds[4 * i + 1] + lds[4 * i + 2] + lds[4 * i + 3];
}

__device__ __forceinline__ void wave_lds_sync() {    // LDS written by other lanes of this wave is visible behind it
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ float silu_f(float z) { return z / (1.f + __expf(-z)); }

// ---- keys a query at position `pos` sees, as 64-key tiles: the tiles of the kept first tokens, then those of the window
struct VisibleTiles {
    int kept, first, count;                          // tiles [0, kept), then [first, first + count - kept)
    __device__ __forceinline__ int tile(int i) const { return i < kept ? i : first + i - kept; }
};
// the first key, kept ones aside, that a query at `pos` sees through a window (the last `window` tokens; 0: all) or in its chunk (chunk > 0)
__device__ __forceinline__ int first_seen(int pos, int window, int chunk) {
    if (chunk > 0) return pos - pos % chunk;
    return window > 0 && pos >= window ? pos - window + 1 : 0;
}
// lo: first_seen of the first query that walks along, last_pos: position of the last one
__device__ __forceinline__ VisibleTiles visible_from(int lo, int last_pos, int keep_first) {
    VisibleTiles v;
    v.first = lo >> 6;
    const int k = (keep_first + 63) >> 6;
    v.kept = k < v.first ? k : v.first;
    v.count = v.kept + ((last_pos + 64) >> 6) - v.first;
    return v;
}
// first_pos .. last_pos: positions of the queries that walk together
__device__ __forceinline__ VisibleTiles visible_tiles(int first_pos, int last_pos, int window, int keep_first) {
    return visible_from(first_seen(first_pos, window, 0), last_pos, keep_first);
}

// 4 columns of a head's output at `pos`, from dimension d on (a multiple of 4), turned back: interleaved pairs of the first `rot` dimensions, table rows cos | sin
__device__ __forceinline__ f32x4 turn_back(f32x4 v, const float* table, int64_t pos, int max_position, int rot, int d) {
    if (d >= rot) return v;
    const float* cs = table + (pos < max_position ? pos : max_position - 1) * rot;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        if (d + 2 * p >= rot) continue;
        const float c = cs[d / 2 + p], s = cs[rot / 2 + d / 2 + p], x = v[2 * p], y = v[2 * p + 1];
        v[2 * p] = x * c + y * s;
        v[2 * p + 1] = y * c - x * s;
    }
    return v;
}
// the same for columns COLS t + 4 lg .. of all t: where a lane's two pairs lie side by side in the table on 8 bytes (every usual width), everything
// is asked of the table before anything is turned, two pairs a load.  Tile by tile each turn waited for its own four loads, DT round trips to the
// cache one behind the other at the end of every block: paged_prompt_kernel over 16384 new tokens, chunk mask, 128 columns turned:
// 16 heads 79.7 -> 71.2 us (16 sequences) and 71.7 -> 64.7 (5), 32 heads 131.7 -> 116.5 (30).
template <int COLS = 16, int DT>
__device__ __forceinline__ void turn_back_tiles(f32x4 (&v)[DT], const float* table, int64_t pos, int max_position, int rot, int lg) {
    if (rot & 3 || reinterpret_cast<uintptr_t>(table) & 7) {
#pragma unroll
        for (int t = 0; t < DT; ++t) v[t] = turn_back(v[t], table, pos, max_position, rot, COLS * t + 4 * lg);
        return;
    }
    const float* cs = table + (pos < max_position ? pos : max_position - 1) * rot;
    f32x2 c[DT], s[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) {
        const int i = COLS / 2 * t + 2 * lg, at = 2 * i < rot ? i : 0;
        c[t] = *reinterpret_cast<const f32x2*>(cs + at);
        s[t] = *reinterpret_cast<const f32x2*>(cs + rot / 2 + at);
    }
#pragma unroll
    for (int t = 0; t < DT; ++t) {
        const bool turned = COLS * t + 4 * lg < rot;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const float x = v[t][2 * p], y = v[t][2 * p + 1];
            v[t][2 * p] = turned ? x * c[t][p] + y * s[t][p] : x;
            v[t][2 * p + 1] = turned ? y * c[t][p] - x * s[t][p] : y;
        }
    }
}

// ---- segment tables of the recurrent mechanisms: [first row, rows, sequence, index in its portion].  A segment may have no rows: it is left out of the
// walks (which ask for rows before they count them), and a portion of such segments leaves its state as it is.
// Whether a portion goes on from its slot's state: not where its first token is at position 0.
__device__ __forceinline__ bool portion_carries(const int32_t* chunks, int n_chunks, int first, const int64_t* positions) {
    for (int c = first; c < n_chunks && (c == first || chunks[4 * c + 3] != 0); ++c)
        if (chunks[4 * c + 1] > 0) return positions[chunks[4 * c]] > 0;
    return true;
}

// Segments of the portion whose first one is row `first` of the table (all lanes of a wave ask).
__device__ __forceinline__ int portion_segments(const int32_t* chunks, int n_chunks, int first) {
    int count = 1, run;
    do {
        const int c = first + count + (int)(threadIdx.x & 63);
        const uint64_t others = ~__builtin_amdgcn_ballot_w64(c < n_chunks && chunks[4 * c + 3] != 0);
        run = others ? __builtin_ctzll(others) : 64;
        count += run;
    } while (run == 64);
    return count;
}

// Contributions of a portion's `count` segments -> states at their starts, in place, of the four neighbouring state elements at own: own[k * per ..] of segment k, `cur` in front
// of the first (the last segment left no contribution).  ahead(k) is what the factor of segment k comes from, factor() of it the factor.
// Nothing a segment reads depends on the one before, but its store might be the next one's load for all the compiler knows: one at a time a segment cost a trip to
// memory.  Up to 16 of them are asked for together.  33 segments, 8 heads of 128 x 128 states: 25.8 -> 10.2 us (one element a thread 12.6); 16 of 64 x 64 16.4 -> 8.6; 2048 channels
// of 16 states 15.8 -> 6.6.  3 portions of 5 segments, 16 heads of 128 x 128: 18.6 -> 7.8.
template <int U, typename Ahead, typename Factor>
__device__ __forceinline__ void segment_starts_of(float* own, int64_t per, int k0, f32x4& cur, Ahead ahead, Factor factor) {
    f32x4 mine[U];
    float raw[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        mine[u] = *reinterpret_cast<const f32x4*>(own + (k0 + u) * per);
        raw[u] = ahead(k0 + u);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        *reinterpret_cast<f32x4*>(own + (k0 + u) * per) = cur;
        cur = factor(raw[u]) * cur + mine[u];
    }
}
template <typename Ahead, typename Factor>
__device__ __forceinline__ void segment_starts(float* own, int64_t per, int count, f32x4 cur, Ahead ahead, Factor factor) {
    int k = 0;
    for (; k + 16 < count; k += 16) segment_starts_of<16>(own, per, k, cur, ahead, factor);
    if (k + 8 < count) segment_starts_of<8>(own, per, k, cur, ahead, factor), k += 8;
    if (k + 4 < count) segment_starts_of<4>(own, per, k, cur, ahead, factor), k += 4;
    if (k + 2 < count) segment_starts_of<2>(own, per, k, cur, ahead, factor), k += 2;
    if (k + 1 < count) segment_starts_of<1>(own, per, k, cur, ahead, factor), k += 1;
    *reinterpret_cast<f32x4*>(own + k * per) = cur;
}
// What a workgroup leaves of `rows` x `cols` state elements behind a segment without rows: a summary of nothing, or the state at its start.
template <bool SUMMARY>
__device__ __forceinline__ void pass_segment(float* seg_state, float* state, int rows, int cols, int64_t stride) {
    for (int e = threadIdx.x; e < rows * cols; e += blockDim.x) {
        const int64_t at = e / cols * stride + e % cols;
        if constexpr (SUMMARY) seg_state[at] = 0.f;
        else state[at] = seg_state[at];
    }
}

}  // namespace nvh
