// Attention of prompt portions over the pages of one layer (gfx950 MFMA, tile schemes of attend_tile.h): keys and values come straight from the pages,
// 64 rows of one (page, key/value head) per tile by LDS-DMA, double-buffered.  A query tile walks the tiles of the kept first tokens, then the window's:
// what no query of the tile sees is not read.  A sink starts the running maximum and sum.
// Algorithmic flops per launch: sum over sequences of 2 (DK + DV) heads (visible pairs).
#include "attend_tile.h"
#include "mixers.h"

namespace nvh {

namespace {

template <int BM, bool ORDERED>
__device__ __forceinline__ bool prompt_tile(const PagedAttendArgs& a, int* words, PromptTile& t) {
    if constexpr (ORDERED) {
        if (!few_prompts_tile<BM>(a.cu_q, a.cu_k, a.batch, a.heads, a.kv_heads, a.chunk > 0 ? a.chunk : a.window, words, t)) return false;
    } else {
        attend_unit(a.heads, t.qt, t.head, t.b);
        prompt_rows(a.cu_q, a.cu_k, t);
    }
    return t.qt * BM < t.sq && t.sk >= t.sq;
}

// WIDE: 128 rows a workgroup on 32 x 32 tiles (attend_walk32); otherwise 64 rows on 16 x 16 tiles.  The same sums to the bit.  ORDERED: few_prompts_tile (of its own: the code in front
// of other launches was 0.2 us).
// (heads of 128 / 64: three workgroups a CU, as their images allow; without the bound 169 registers for 168, and 195 -> 212 us for 4 prompts of 12000 tokens, 16 heads)
template <int DK, int DV, bool WIDE, bool ORDERED>
__global__ __launch_bounds__(256, WIDE && DK == 128 && DV == 64 ? 3 : WIDE || DK + DV <= 320 ? 2 : 1) void paged_prompt_kernel(const PagedAttendArgs a) {
    using Images = TileImages<DK, DV>;
    constexpr int WR = WIDE ? 32 : 16, BM = 4 * WR, BN = Images::BN, KP = Images::KP, VP = Images::VP, NK = Images::NK, NV = Images::NV;
    extern __shared__ __attribute__((aligned(512))) unsigned char lds[];
    PromptTile tile;
    if (!prompt_tile<BM, ORDERED>(a, reinterpret_cast<int*>(lds), tile)) return;
    const int head = tile.head, b = tile.b, q_beg = tile.q_beg, sq = tile.sq, sk = tile.sk, q0 = tile.qt * BM;
    const int shift = sk - sq;                       // query row r has position r + shift
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lq = lane & (WR - 1), lg = lane / WR;
    const int g = head / (a.heads / a.kv_heads);
    const int rows = sq - q0 < BM ? sq - q0 : BM;
    const VisibleTiles vis = visible_from(first_seen(q0 + shift, a.window, a.chunk), q0 + rows - 1 + shift, a.keep_first);
    const int wave_first = q0 + wave * WR + shift, wave_last = wave_first + WR - 1;       // positions of this wave's rows
    const int lo_first = first_seen(wave_first, a.window, a.chunk), lo_last = first_seen(wave_last, a.window, a.chunk);

    // ---- staging: this lane's piece of each DMA instruction: row of the tile and offset inside it
    const uint16_t* cache = reinterpret_cast<const uint16_t*>(a.cache) + (int64_t)g * a.block_size * (DK + DV);
    const int64_t page_elems = (int64_t)a.kv_heads * a.block_size * (DK + DV);
    PageNumbers pages{a.block_tables + (int64_t)b * a.bt_stride, (sk - 1) / a.block_size};
    auto swz_of_v = [](int row) __attribute__((always_inline)) { return WIDE ? swz_v32<DV>(row) : swz_v<DV>(row); };
    uint32_t koff[NK], voff[NV];                     // of a full tile, in bytes from its first row
#pragma unroll
    for (int j = 0; j < NK; ++j) {
        const int s = (wave * NK + j) * 64 + lane, R = s / KP;
        koff[j] = (R * DK + ((s - R * KP) ^ swz_k<DK>(R)) * 8) * 2;
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int s = (wave * NV + j) * 64 + lane, R = s / VP;
        voff[j] = (R * DV + ((s - R * VP) ^ swz_of_v(R)) * 8) * 2;
    }
    auto dma = [](const char* base, uint32_t at, unsigned char* to) __attribute__((always_inline)) {
        if constexpr (WIDE) dma16_uncounted(base, at, to);
        else dma16(base + at, to);
    };
    auto stage = [&](int it, int buf) __attribute__((always_inline)) {
        unsigned char* kimg = Images::k(lds, buf);
        unsigned char* vimg = Images::v(lds, buf);
        const int kv0 = vis.tile(it) * BN, page = kv0 / a.block_size, off = kv0 - page * a.block_size, live = sk - kv0 < BN ? sk - kv0 : BN;
        const uint16_t* head = cache + pages.at(page, lane) * page_elems;
        const char* kb = reinterpret_cast<const char*>(head + (int64_t)off * DK);
        const char* vb = reinterpret_cast<const char*>(head + (int64_t)a.block_size * DK + (int64_t)off * DV);
#pragma unroll
        for (int j = 0; j < NK; ++j) {
            uint32_t at = koff[j];
            if (live < BN) {                         // rows past the end repeat the last key: masked
                const int s = (wave * NK + j) * 64 + lane, R = s / KP;
                at = ((R < live ? R : live - 1) * DK + ((s - R * KP) ^ swz_k<DK>(R)) * 8) * 2;
            }
            dma(kb, at, kimg + (wave * NK + j) * 1024);
        }
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            uint32_t at = voff[j];
            if (live < BN) {
                const int s = (wave * NV + j) * 64 + lane, R = s / VP;
                at = ((R < live ? R : live - 1) * DV + ((s - R * VP) ^ swz_of_v(R)) * 8) * 2;
            }
            dma(vb, at, vimg + (wave * NV + j) * 1024);
        }
    };
    const int my_q = q0 + wave * WR + lq, lo = first_seen(my_q + shift, a.window, a.chunk), pos = my_q + shift < sk - 1 ? my_q + shift : sk - 1;
    const bool q_ok = my_q < sq;
    const uint16_t* qp = reinterpret_cast<const uint16_t*>(a.q) + (int64_t)(q_beg + (q_ok ? my_q : sq - 1)) * a.q_stride + (int64_t)head * DK + lg * 8;
    // (computed when it is needed: held over the walk, heads of 256 / 256 took 3 % longer)
    auto out = [&]() __attribute__((always_inline)) { return reinterpret_cast<uint16_t*>(a.out) + (int64_t)(q_beg + my_q) * a.out_stride + head * DV; };
    const float start = a.sink ? a.sink[head] * kLog2e : -INFINITY;
    auto first_key = [&](int it) { return vis.tile(it) * BN; };
    if constexpr (WIDE) {
        stage(0, 0);
        u32x4 qf[DK / 16];
#pragma unroll
        for (int st = 0; st < DK / 16; ++st) qf[st] = *reinterpret_cast<const u32x4*>(qp + st * 16);
        attend_walk32<DK, DV, false, false>(
            lds, vis.count, a.scale * kLog2e, start, lane, qf, stage, first_key, [&](int key) { return key <= wave_last && key < sk && (key + 32 > lo_first || key < a.keep_first); },
            [&](int key, auto& s) {
                constexpr int N = 32 * (sizeof(s) / sizeof(s[0]));
                const int mine = key + 4 * lg;
                if (key + N - 1 > wave_first || key + N > sk) hide_scores(s, [&](int at) { return at <= pos - mine; });
                if (key < lo_last && key + N > a.keep_first) {
                    if (key >= a.keep_first) hide_scores(s, [&](int at) { return at >= lo - mine; });
                    else hide_scores(s, [&](int at) { return at >= lo - mine || at < a.keep_first - mine; });
                }
            },
            [&](f32x4 (&v)[DV / 8]) {
                if (a.o_cos_sin && q_ok) turn_back_tiles<8>(v, a.o_cos_sin, my_q + shift, a.max_position, a.o_rot, lg);
                uint16_t* const o_lds = reinterpret_cast<uint16_t*>(lds) + wave * WR * kRowOut<DV>;
                int out_lane = lane;                 // (not seen by the compiler yet: no address is held over the walk)
                asm volatile("" : "+v"(out_lane));
#pragma unroll
                for (int u = 0; u < DV / 8; ++u) act_st4(o_lds + (out_lane & (WR - 1)) * kRowOut<DV> + 8 * u + 4 * (out_lane / WR), v[u]);
                const int r0 = q0 + wave * WR;
                rows_out<DV, WR>(o_lds, out_lane, [&](int r) { return r0 + r < sq ? reinterpret_cast<uint16_t*>(a.out) + (int64_t)(q_beg + r0 + r) * a.out_stride + head * DV : nullptr; });
            });
    } else {
        attend_walk<DK, DV, 1>(
            lds, vis.count, a.scale * kLog2e, start, lane, stage, [&](int, int st) { return *reinterpret_cast<const bf16x8*>(qp + st * 32); }, first_key,
            [&](int kv0) { return kv0 <= wave_last && (kv0 + BN > lo_first || kv0 < a.keep_first); },
            [&](int kv0) { return kv0 + BN - 1 > wave_first || kv0 + BN > sk || (kv0 < lo_last && kv0 + BN > a.keep_first); },
            [&](int kv0, int, int off) {
                const int at = kv0 + 4 * lg + off;
                return at <= pos && (at >= lo || at < a.keep_first);
            },
            [&](int) { return q_ok ? out() : nullptr; },
            [&](int, f32x4 (&v)[DV / 16]) {
                if (a.o_cos_sin) turn_back_tiles(v, a.o_cos_sin, my_q + shift, a.max_position, a.o_rot, lg);
            });
    }
}

template <int DK, int DV, bool WIDE, bool ORDERED>
int launch_form(const PagedAttendArgs& a, hipStream_t stream) {
    constexpr size_t lds = TileImages<DK, DV>::BYTES;
    constexpr int BM = WIDE ? 128 : 64;
    if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(paged_prompt_kernel<DK, DV, WIDE, ORDERED>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    paged_prompt_kernel<DK, DV, WIDE, ORDERED><<<dim3(a.heads, a.batch, (a.max_q + BM - 1) / BM), 256, lds, stream>>>(a);
    return check_launch("paged_attend_prompt");
}
// Two or three portions in the order of their work, unless all workgroups run at once where the images leave room for two and more on a CU (64 rows): finding the tile is 0.7 us of 15 to 30,
// and nothing waits for a CU (32 sets of 2 and 3 portions: 0.93 to 1.0 of the speed with the order, six of them 1.06 to 1.18).
template <int DK, int DV, bool WIDE>
int launch_one(const PagedAttendArgs& a, hipStream_t stream) {
    constexpr int64_t room = 163840 / TileImages<DK, DV>::BYTES;
    const bool at_once = !WIDE && room > 1 && ((int64_t)a.rows + 63 * (int64_t)a.batch) * a.heads <= 64 * 256 * room;
    return few_prompts(a.batch) && !at_once ? launch_form<DK, DV, WIDE, true>(a, stream) : launch_form<DK, DV, WIDE, false>(a, stream);
}
template <int DK, int DV>
int launch_dims(const PagedAttendArgs& a, hipStream_t stream) {
    if constexpr (DV <= 128) {
        // Up to 2.2 workgroups of 64 rows a CU, those: a launch that leaves CUs idle takes as long as its longest walk over the keys.  8 heads of 128 / 128, us with 128 and with
        // 64 rows: one prompt of 2414 tokens 72 and 59, 12 later portions of 3013 with a window 41 and 34, 5 of 3648 with chunks 36 and 29; 16 heads, 4 of 2183 33 and 27; but
        // 2 later portions of 2415 (2.4 a CU, walks of equal length) 92 and 106, 2 of 4140 103 and 116.
        // But only where all of them run at once, ragged last ones included: wide images leave room for two on a CU (one of 256 / 128), and with 128 rows a second round is
        // shorter.  2 later portions of 1100 and 3 windowed ones of 730, 16 heads: 128 / 128 104 and 131, 37 and 40; 192 / 64 100 and 125, 35 and 43; 192 / 128 123 and 145; 256 / 128
        // at half as many rows 123 and 138; where all fit it is 0.98 to 1.6 times as fast, 1.2 in the mean.
        constexpr int64_t at_once = 163840 / TileImages<DK, DV>::BYTES * 256;
        const bool few = (int64_t)a.rows * a.heads <= 36044 && ((int64_t)a.rows + 63 * (int64_t)a.batch) * a.heads <= 64 * at_once;
        if (a.max_q > 256 && !few) return launch_one<DK, DV, true>(a, stream);
    }
    return launch_one<DK, DV, false>(a, stream);
}

}  // namespace

int launch_paged_attend_prompt(const PagedAttendArgs& a, hipStream_t stream) {
    switch (a.dk * 1000 + a.dv) {
        case 64064: return launch_dims<64, 64>(a, stream);
        case 64128: return launch_dims<64, 128>(a, stream);
        case 128064: return launch_dims<128, 64>(a, stream);
        case 128128: return launch_dims<128, 128>(a, stream);
        case 192064: return launch_dims<192, 64>(a, stream);
        case 192128: return launch_dims<192, 128>(a, stream);
        case 256064: return launch_dims<256, 64>(a, stream);
        case 256128: return launch_dims<256, 128>(a, stream);
        case 256256: return launch_dims<256, 256>(a, stream);
        default: set_error("paged_attend_prompt: key width %d / value width %d", a.dk, a.dv); return -2;
    }
}

}  // namespace nvh
