// The MFMA tile of the prompt-attention kernels that read keys and values from LDS images of 64 rows (unequal widths DK, DV):
// four waves x QT x 16 query rows, S^T = K Q^T and O^T = V^T P^T with the weights as bf16 hi + lo halves, online softmax in the log2 domain.
// A kernel stages the images (16-byte pieces swizzled by swz_k / swz_v), fills the query fragments and says which keys a query sees.
#pragma once
#include <type_traits>

#include "hybrid.h"

namespace nvh {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int OFF>
__device__ __forceinline__ u32x2 ds_read_tr16(uint32_t lds_addr) {
    static_assert(OFF >= 0 && OFF < 65536, "ds offset field is 16 bits");
    u32x2 r;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(lds_addr), "n"(OFF) : "memory");
    return r;
}
// the same read through the compiler's builtin: it places the wait itself and may move other work in between
__device__ __forceinline__ u32x2 lds_tr16(const void* p) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p));
}
__device__ __forceinline__ uint32_t lds_addr_of(const void* p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p; }
__device__ __forceinline__ float max3f(float x, float y, float z) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(y), "v"(z));
    return r;
}
// workgroup barrier behind this wave's LDS traffic only (a __syncthreads() would drain the loads in flight)
__device__ __forceinline__ void lds_only_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
// 16 bytes per lane from global memory to 1024 consecutive LDS bytes
__device__ __forceinline__ void dma16(const void* src, unsigned char* lds_wave_base) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)lds_wave_base, 16, 0, 0);
}
// the same behind the compiler's back: it would wait for all loads in flight before the first transposed read that follows (the kernel counts them itself).
// base: uniform; at: this lane's offset in bytes.
__device__ __forceinline__ void dma16_uncounted(const void* base, uint32_t at, const unsigned char* lds_wave_base) {
    asm volatile("s_mov_b32 m0, %0\n s_nop 0\n global_load_lds_dwordx4 %1, %2" ::"s"(lds_addr_of(lds_wave_base)), "v"(at), "s"(base) : "memory", "m0");
}
// 16-byte pieces of a row are xor-ed inside groups of 8 (rows of an odd number of 128-byte lines) or 16 (even)
template <int W>
__device__ __forceinline__ int swz_k(int row) { return (W / 64) & 1 ? ((row >> 1) & 7) : (row & 15); }
template <int W>
__device__ __forceinline__ int swz_v(int row) { return W == 64 ? (row & 6) : ((2 * row) & 14); }

// A wave's results, bf16, on their way out: rows of D columns, D + 8 apart in LDS that is the wave's own; lane l has written 4 columns of one of them.  As they lie there a store would be 16
// or 32 bytes of 16 or 32 rows; here it is whole rows.  row(r): where row r's columns go, or null (8 bytes off a multiple of 16, it may be).
// 24 prompts of 16384 tokens, 14 / 2 heads of 64, 68.4 -> 64.6 us; 8 of 8192 behind cached ones, 28 / 4 heads of 128, 288 -> 282; 2 of 7831, 16 / 8 heads, 172.6 -> 166.8.
template <int D>
constexpr int kRowOut = D + 8;
template <int D, int ROWS, typename Row>
__device__ __forceinline__ void rows_out(const uint16_t* o_lds, int lane, Row row) {
    typedef u32x4 __attribute__((aligned(8))) u32x4_half;
    constexpr int PER = D / 8, STEP = 64 / PER;
    asm volatile("" ::: "memory");                   // (a wave's LDS accesses are done in their order)
    __builtin_amdgcn_wave_barrier();
    const int r0 = lane / PER, col = lane % PER * 8;
#pragma unroll
    for (int j = 0; j < ROWS / STEP; ++j) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(o_lds + (r0 + STEP * j) * kRowOut<D> + col);
        uint16_t* const to = row(r0 + STEP * j);
        if (to) *reinterpret_cast<u32x4_half*>(to + col) = v;
    }
}

// LDS of a tile walk: V images of both buffers, then their K images (V offsets fit a DS immediate)
template <int DK, int DV>
struct TileImages {
    static constexpr int BN = 64, KROW = DK * 2, VROW = DV * 2, KIMG = BN * KROW, VIMG = BN * VROW;
    static constexpr int KP = DK / 8, VP = DV / 8;   // 16-byte pieces per row == DMA instructions per image
    static constexpr int NK = KP / 4, NV = VP / 4;   // ... per wave
    static constexpr size_t BYTES = (size_t)2 * (KIMG + VIMG);
    static __device__ __forceinline__ unsigned char* k(unsigned char* lds, int buf) { return lds + 2 * VIMG + buf * KIMG; }
    static __device__ __forceinline__ unsigned char* v(unsigned char* lds, int buf) { return lds + buf * VIMG; }
};

// One workgroup's attention over n_tiles tiles of 64 keys; wave w holds query rows 16 QT w .. of the workgroup's 64 QT.  The kernel says
//   stage(it, buf)       starts the NK + NV DMA instructions per wave that fill buffer `buf` with tile `it`
//   query(qs, st)        query fragment: row lq of sub-tile qs, columns 32 st + 8 lg .. (B operand of S^T)
//   first_key(it)        key of the tile's first row; covers(kv0): this wave sees something of that tile; masked(kv0): but not all of it:
//   sees(kv0, qs, off)   key kv0 + 4 lg + off counts for the lane's query of sub-tile qs
//   row(qs)              where the lane's query of sub-tile qs goes, or null; last(qs, v): changes its output columns 16 t + 4 lg .. of all t, v[t]
// start: score (log2 domain) of a softmax entry without key and value, -inf for none.
// (The sums, the fragments and the tile loop live in ONE function: split up, the same code takes 32 registers more.)
template <int DK, int DV, int QT, typename Stage, typename Query, typename FirstKey, typename Covers, typename Masked, typename Sees, typename Row, typename Last>
__device__ __forceinline__ void attend_walk(unsigned char* lds, int n_tiles, float scale_log2, float start, int lane, Stage stage, Query query, FirstKey first_key, Covers covers,
                                            Masked need_mask, Sees sees, Row row, Last last) {
    using Images = TileImages<DK, DV>;
    constexpr int BN = Images::BN, KROW = Images::KROW, VROW = Images::VROW, KIMG = Images::KIMG, VIMG = Images::VIMG, NK = Images::NK, NV = Images::NV;
    static_assert((DV & (DV - 1)) == 0 && VROW <= 512);
    constexpr int STEPS = DK / 32, DT = DV / 16, NT = BN / 16;
    const int lq = lane & 15, lg = lane >> 4;
    f32x4 o[QT][DT];
    float m[QT], l[QT];                              // running maximum (log2 domain) and this lane's share of the sum
#pragma unroll
    for (int qs = 0; qs < QT; ++qs) {
        m[qs] = start;
        l[qs] = start > -INFINITY && lg == 0 ? 1.f : 0.f;
#pragma unroll
        for (int t = 0; t < DT; ++t) o[qs][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    stage(0, 0);
    bf16x8 qf[QT][STEPS];
#pragma unroll
    for (int qs = 0; qs < QT; ++qs)
#pragma unroll
        for (int st = 0; st < STEPS; ++st) qf[qs][st] = query(qs, st);
    // waited for here: left to the loop, the wait for these loads would drain the DMA in flight in every tile
#pragma unroll
    for (int qs = 0; qs < QT; ++qs)
#pragma unroll
        for (int st = 0; st < STEPS; ++st) asm volatile("" : "+v"(qf[qs][st]));
    uint32_t vbase;                                  // of this lane's transposed reads; piece t of a row is an exclusive or away (swizzles are even)
    {
        const int R0 = 4 * lg + (lq >> 2), p = lq & 3;                         // rows R0, R0 + 16, R0 + 32 share a swizzle
        vbase = lds_addr_of(lds + R0 * VROW + (p & 1) * 8 + (((p >> 1) ^ swz_v<DV>(R0)) * 16));
    }
    auto tile_body = [&](auto bufc, const int it) {
        constexpr int buf = decltype(bufc)::value;
        if (it + 1 < n_tiles) {
            stage(it + 1, buf ^ 1);
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NK + NV) : "memory");     // tile `it` has landed, tile it + 1 is in flight
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const unsigned char* kimg = lds + 2 * VIMG + buf * KIMG;
        const int kv0 = first_key(it);
        if (covers(kv0)) {
            f32x4 sT[QT][NT];
#pragma unroll
            for (int tt = 0; tt < NT; ++tt) {
#pragma unroll
                for (int qs = 0; qs < QT; ++qs) sT[qs][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
                const int R = 16 * tt + lq;
#pragma unroll
                for (int st = 0; st < STEPS; ++st) {
                    const bf16x8 kf = *reinterpret_cast<const bf16x8*>(kimg + R * KROW + (((4 * st + lg) ^ swz_k<DK>(R)) * 16));
#pragma unroll
                    for (int qs = 0; qs < QT; ++qs) sT[qs][tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[qs][st], sT[qs][tt], 0, 0, 0);
                }
            }
            // the max chain reads the accumulators through inline asm: one statement that takes all of them carries the MFMA wait states
            if constexpr (QT == 1) asm volatile("s_nop 7" : "+v"(sT[0][0]), "+v"(sT[0][1]), "+v"(sT[0][2]), "+v"(sT[0][3]));
            else asm volatile("s_nop 7" : "+v"(sT[0][0]), "+v"(sT[0][1]), "+v"(sT[0][2]), "+v"(sT[0][3]), "+v"(sT[1][0]), "+v"(sT[1][1]), "+v"(sT[1][2]), "+v"(sT[1][3]));
            const bool masked = need_mask(kv0);
#pragma unroll
            for (int qs = 0; qs < QT; ++qs) {
                if (masked) {
#pragma unroll
                    for (int tt = 0; tt < NT; ++tt)
#pragma unroll
                        for (int r = 0; r < 4; ++r) sT[qs][tt][r] = sees(kv0, qs, 16 * tt + r) ? sT[qs][tt][r] : -INFINITY;
                }
                float mx = max3f(sT[qs][0][0], sT[qs][0][1], sT[qs][0][2]);
                mx = max3f(mx, sT[qs][0][3], sT[qs][1][0]);
                mx = max3f(mx, sT[qs][1][1], sT[qs][1][2]);
                mx = max3f(mx, sT[qs][1][3], sT[qs][2][0]);
                mx = max3f(mx, sT[qs][2][1], sT[qs][2][2]);
                mx = max3f(mx, sT[qs][2][3], sT[qs][3][0]);
                mx = max3f(mx, sT[qs][3][1], sT[qs][3][2]);
                mx = max2(mx, sT[qs][3][3]);
                mx = max_xor16(mx);
                mx = max_xor32(mx);
                mx *= scale_log2;                                                  // (the host admits positive scales only)
                const float m_new = moved_max(m[qs], mx);
                const float m_use = m_new == -INFINITY ? 0.f : m_new;
                float psum = 0.f;
#pragma unroll
                for (int tt = 0; tt < NT; ++tt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float e = fast_exp2(sT[qs][tt][r] * scale_log2 - m_use);
                        sT[qs][tt][r] = e;
                        psum += e;
                    }
                if (__builtin_amdgcn_ballot_w64(m_new != m[qs]) != 0) {
                    const float alpha = fast_exp2(m[qs] - m_use);
                    l[qs] *= alpha;
#pragma unroll
                    for (int t = 0; t < DT; ++t) o[qs][t] *= alpha;
                }
                l[qs] += psum;
                m[qs] = m_new;
            }
#pragma unroll
            for (int hh = 0; hh < BN / 32; ++hh) {
                bf16x8 p_hi[QT], p_lo[QT];
#pragma unroll
                for (int qs = 0; qs < QT; ++qs) {
                    u32x4 hraw, lraw;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float p0 = sT[qs][2 * hh + (j >> 1)][2 * (j & 1)], p1 = sT[qs][2 * hh + (j >> 1)][2 * (j & 1) + 1];
                        hraw[j] = pack_bf16x2_once(p0, p1);
                        lraw[j] = pack_bf16x2(p0 - bf16_lo(hraw[j]), p1 - bf16_hi(hraw[j]));
                    }
                    p_hi[qs] = *reinterpret_cast<const bf16x8*>(&hraw);
                    p_lo[qs] = *reinterpret_cast<const bf16x8*>(&lraw);
                }
                constexpr int VB = DT < 16 ? DT : 16;                              // pieces whose reads are in flight together
#pragma unroll
                for (int tb = 0; tb < DT; tb += VB) {
                    u32x2 vlo[VB], vhi[VB];
#pragma unroll
                    for (int t = 0; t < VB; ++t) {
                        const uint32_t at = vbase ^ ((tb + t) * 32);
                        if (hh == 0) {
                            vlo[t] = ds_read_tr16<buf * VIMG>(at);
                            vhi[t] = ds_read_tr16<buf * VIMG + 16 * VROW>(at);
                        } else {
                            vlo[t] = ds_read_tr16<buf * VIMG + 32 * VROW>(at);
                            vhi[t] = ds_read_tr16<buf * VIMG + 48 * VROW>(at);
                        }
                    }
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    __builtin_amdgcn_sched_barrier(0);
                    bf16x8 vf[VB];
#pragma unroll
                    for (int t = 0; t < VB; ++t) {
                        const u32x4 raw = {vlo[t][0], vlo[t][1], vhi[t][0], vhi[t][1]};
                        vf[t] = *reinterpret_cast<const bf16x8*>(&raw);
                    }
#pragma unroll
                    for (int t = 0; t < VB; ++t)
#pragma unroll
                        for (int qs = 0; qs < QT; ++qs) o[qs][tb + t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[t], p_hi[qs], o[qs][tb + t], 0, 0, 0);
#pragma unroll
                    for (int t = 0; t < VB; ++t)
#pragma unroll
                        for (int qs = 0; qs < QT; ++qs) o[qs][tb + t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[t], p_lo[qs], o[qs][tb + t], 0, 0, 0);
                }
            }
        }
        lds_only_barrier();                                                    // everyone's reads of this buffer are done
    };
    for (int it = 0; it < n_tiles; it += 2) {
        tile_body(std::integral_constant<int, 0>{}, it);
        if (it + 1 < n_tiles) tile_body(std::integral_constant<int, 1>{}, it + 1);
    }
    // (what lies behind comes from a lane number that the compiler has not seen: addresses found in front of the walk would be held over it.  192 / 128 with two sub-tiles would spill 18
    // registers: 17 prompts of 7131 tokens, 4 heads, 41.5 us and with them 54.9)
    asm volatile("" : "+v"(lane));
    const int out_row = lane & 15, out_group = lane >> 4;
#pragma unroll
    for (int qs = 0; qs < QT; ++qs) {
        float sum = sum_xor16(l[qs]);
        sum = sum_xor32(sum);
        uint16_t* out = row(qs);
        const float inv = sum > 0.f ? 1.f / sum : 0.f;
#pragma unroll
        for (int t = 0; t < DT; ++t) o[qs][t] *= inv;
        if (out) last(qs, o[qs]);
        // (nobody reads the images any more)
        unsigned char* const mine = lds + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * (16 * kRowOut<DV> * 2 + 128);
        uint16_t** const to = reinterpret_cast<uint16_t**>(mine);
        uint16_t* const o_lds = reinterpret_cast<uint16_t*>(mine + 128);
        if (out_group == 0) to[out_row] = out;
#pragma unroll
        for (int t = 0; t < DT; ++t) act_st4(o_lds + out_row * kRowOut<DV> + 16 * t + 4 * out_group, o[qs][t]);
        rows_out<DV, 16>(o_lds, lane, [&](int r) { return to[r]; });
        asm volatile("" ::: "memory");               // (the next rows go to the same words)
    }
}

__device__ __forceinline__ uint32_t pack_f16x2(float lo, float hi) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));      // (round to nearest even)
}

// ---- the same walk on 32 x 32 tiles: four waves of 32 query rows
// What binds a walk is vector issue (softmax, hi + lo halves) and the matrix pipe, whose product keeps other vector instructions from issuing for 10 to 12 cycles, be it 16 x 16 x 32
// (16 cycles of the pipe) or 32 x 32 x 16 (32 cycles, twice the work): half the issue per flop here, half the fragments read from LDS, one lane-crossing step of a row's maximum instead of
// two.  Blocks of 32 keys that a wave sees nothing of are left out.  16384 tokens of 4 sequences over pages, 16 heads of 128: 387 -> 375 us, 1.1 PFLOP/s with both halves of P (a large
// bf16 product: 1.2); 14 sequences with a window of 512: 131 -> 124.  Vector issue is then 79 % of the time, the matrix pipe 58 %; the clock is at what power leaves (1.7 GHz), so
// that waves kept busier and a priority for the workgroups with the longest walks gave nothing.
// 16-byte pieces of a V row are xor-ed so that the four rows of a transposed read (and both 16-column blocks that half a wave reads) lie in different banks
template <int W>
__device__ __forceinline__ int swz_v32(int row) { return W == 64 ? (row & 2) * 2 : (row & 3) * 4; }

template <bool F16>
__device__ __forceinline__ f32x16 mfma32(const u32x4& a, const u32x4& b, const f32x16& c) {
    if constexpr (F16) return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// scores of NB blocks of 32 keys: s[k][r] is `at` = 32 k + 8 (r / 4) + r % 4 past the lane's first key; those that keep() does not want become -inf
template <int NB, typename Keep>
__device__ __forceinline__ void hide_scores(f32x16 (&s)[NB], Keep keep) {
#pragma unroll
    for (int k = 0; k < NB; ++k)
#pragma unroll
        for (int r = 0; r < 16; ++r) s[k][r] = keep(32 * k + 8 * (r >> 2) + (r & 3)) ? s[k][r] : -INFINITY;
}

// One workgroup's attention over n_tiles tiles of 64 keys; wave w holds query rows 32 w .. of the workgroup's 128, lane l row l % 32.  The kernel has started the DMA of
// tile 0 into buffer 0 and the loads of the queries (qf[st]: columns 16 st + 8 (l / 32) .. of the lane's) and says
//   stage(it, buf)   starts the NK + NV DMA instructions per wave that fill buffer `buf` with tile `it` (dma16_uncounted, pieces swizzled by swz_k / swz_v32)
//   first_key(it)    key of the tile's first row; covers(key): this wave sees something of the 32 keys from there on
//   hide(key, s)     sets scores of the keys from there on that do not count to -inf: s[k][r] is key + 4 (l / 32) + 32 k + 8 (r / 4) + r % 4 (hide_scores)
//   finish(v)        takes the lane's output columns 8 u + 4 (l / 32) .. of all u, v[u]
// F16: V holds fp16 and P is rounded to it, one product instead of two.  PAIRS: a lane's weights are added up in even and odd ones.
// Sums come out to the bit as attend_walk has them: a 16 x 16 x 32 product adds up like two 32 x 32 x 16 ones behind each other, its lane groups g in the order of their keys
// (step i takes groups 2 i and 2 i + 1: keys 8 i + 4 lh + j and 16 further), and the shares of the softmax's sum are those of the lane groups.
template <int DK, int DV, bool F16, bool PAIRS, typename Stage, typename FirstKey, typename Covers, typename Hide, typename Finish>
__device__ __forceinline__ void attend_walk32(unsigned char* lds, int n_tiles, float scale_log2, float start, int lane, u32x4 (&qf)[DK / 16], Stage stage, FirstKey first_key,
                                              Covers covers, Hide hide, Finish finish) {
    using Images = TileImages<DK, DV>;
    constexpr int KROW = Images::KROW, VROW = Images::VROW, KIMG = Images::KIMG, VIMG = Images::VIMG, NK = Images::NK, NV = Images::NV;
    constexpr int STEPS = DK / 16, DT = DV / 32, KG = (DK / 64) & 1 ? 4 : 8;     // KG: steps inside a group of swizzled pieces
    const int lq = lane & 31, lh = lane >> 5;
    f32x16 o[DT];
    float m = start, l[2] = {start > -INFINITY && lh == 0 ? 1.f : 0.f, 0.f};     // running maximum (log2 domain); this lane's shares of the sum, lane groups lh and lh + 2
#pragma unroll
    for (int t = 0; t < DT; ++t) o[t] = f32x16{};
#pragma unroll
    for (int st = 0; st < STEPS; ++st) asm volatile("" : "+v"(qf[st]));          // (waited for here, not in every tile)
    const int kb = lq * KROW + ((lh ^ swz_k<DK>(lq)) * 16);                      // step st: an exclusive or away (32 (st % KG)), and 32 KG (st / KG) further
    int vb;                                                                      // columns 32 t ..: an exclusive or away (64 t)
    {
        const int q = (lane & 15) >> 2, p = lane & 3;                            // lane 4 q + p of 16 addresses key row q, columns 4 p ..
        vb = (4 * lh + q) * VROW + (((2 * (lane >> 4 & 1) + (p >> 1)) ^ swz_v32<DV>(q)) * 16) + (p & 1) * 8;
    }
    // NB blocks of 32 keys from `key` on, whose rows start at kimg and vimg
    auto blocks = [&](auto nb, const int key, const unsigned char* kimg, const unsigned char* vimg) __attribute__((always_inline)) {
        constexpr int NB = decltype(nb)::value;
        f32x16 s[NB];
#pragma unroll
        for (int k = 0; k < NB; ++k) s[k] = f32x16{};
#pragma unroll
        for (int st = 0; st < STEPS; ++st)
#pragma unroll
            for (int k = 0; k < NB; ++k)
                s[k] = mfma32<false>(*reinterpret_cast<const u32x4*>(kimg + (kb ^ (32 * (st % KG))) + 32 * KG * (st / KG) + 32 * KROW * k), qf[st], s[k]);
        __builtin_amdgcn_sched_group_barrier(0x100, 3 * NB, 0);                  // fragments three steps ahead of their products
#pragma unroll
        for (int st = 0; st < STEPS - 3; ++st) {
            __builtin_amdgcn_sched_group_barrier(0x8, NB, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, NB, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x8, 3 * NB, 0);
        // the max chain reads the accumulators through inline asm: one statement that takes all of them carries the MFMA wait states
        if constexpr (NB == 2) asm volatile("s_nop 15\n s_nop 3" : "+v"(s[0]), "+v"(s[1]));
        else asm volatile("s_nop 15\n s_nop 3" : "+v"(s[0]));
        hide(key, s);
        float top[NB];
#pragma unroll
        for (int k = 0; k < NB; ++k) top[k] = max3f(s[k][0], s[k][1], s[k][2]);
#pragma unroll
        for (int r = 3; r < 15; r += 2)
#pragma unroll
            for (int k = 0; k < NB; ++k) top[k] = max3f(top[k], s[k][r], s[k][r + 1]);
        float mx = NB == 2 ? max2(max3f(top[0], s[0][15], s[NB - 1][15]), top[NB - 1]) : max2(top[0], s[0][15]);
        mx = max_xor32(mx) * scale_log2;                                         // (the host admits positive scales only)
        const float m_new = moved_max(m, mx);
        const float m_use = m_new == -INFINITY ? 0.f : m_new;
        float psum[2][2] = {{0.f, 0.f}, {0.f, 0.f}};
#pragma unroll
        for (int k = 0; k < NB; ++k)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float e = fast_exp2(s[k][r] * scale_log2 - m_use);
                s[k][r] = e;
                psum[r >> 2 & 1][PAIRS ? r & 1 : 0] += e;
            }
        if (__builtin_amdgcn_ballot_w64(m_new != m) != 0) {
            const float alpha = fast_exp2(m - m_use);
            l[0] *= alpha;
            l[1] *= alpha;
#pragma unroll
            for (int t = 0; t < DT; ++t) o[t] *= alpha;
        }
        l[0] += PAIRS ? psum[0][0] + psum[0][1] : psum[0][0];
        l[1] += PAIRS ? psum[1][0] + psum[1][1] : psum[1][0];
        m = m_new;
#pragma unroll
        for (int k = 0; k < NB; ++k) {
            u32x2 v[4][DT];                                                      // rows 8 i + 4 lh .. of the 32 keys
#pragma unroll
            for (int t = 0; t < DT; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i][t] = lds_tr16(vimg + (vb ^ (64 * t)) + (32 * k + 8 * i) * VROW);
            u32x4 hi[2], lo[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int r = 4 * i + 8 * (j >> 1) + 2 * (j & 1);
                    const float p0 = s[k][r], p1 = s[k][r + 1];
                    if constexpr (F16) {
                        hi[i][j] = pack_f16x2(p0, p1);
                    } else {
                        hi[i][j] = pack_bf16x2_once(p0, p1);
                        lo[i][j] = pack_bf16x2(p0 - bf16_lo(hi[i][j]), p1 - bf16_hi(hi[i][j]));
                    }
                }
            u32x4 vf[2][DT];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int t = 0; t < DT; ++t) vf[i][t] = u32x4{v[i][t][0], v[i][t][1], v[i + 2][t][0], v[i + 2][t][1]};
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int t = 0; t < DT; ++t) o[t] = mfma32<F16>(vf[i][t], hi[i], o[t]);
            if constexpr (!F16) {
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int t = 0; t < DT; ++t) o[t] = mfma32<false>(vf[i][t], lo[i], o[t]);
            }
        }
    };
    for (int it = 0, buf = 0; it < n_tiles; ++it, buf ^= 1) {
        if (it + 1 < n_tiles) {
            stage(it + 1, buf ^ 1);
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NK + NV) : "memory");       // tile `it` has landed, tile it + 1 is in flight
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const unsigned char *kimg = Images::k(lds, buf), *vimg = Images::v(lds, buf);
        const int key = first_key(it);
        const bool a = covers(key), b = covers(key + 32);
        if (a != b) blocks(std::integral_constant<int, 1>{}, key + (b ? 32 : 0), kimg + (b ? 32 * KROW : 0), vimg + (b ? 32 * VROW : 0));
        if (a && b) blocks(std::integral_constant<int, 2>{}, key, kimg, vimg);
        lds_only_barrier();                                                      // everyone's reads of this buffer are done
    }
    const float sum = sum_xor32(l[0]) + sum_xor32(l[1]), inv = sum > 0.f ? 1.f / sum : 0.f;
    f32x4 v[DV / 8];
#pragma unroll
    for (int u = 0; u < DV / 8; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[u][r] = o[u >> 2][4 * (u & 3) + r] * inv;
    finish(v);
}

// What a workgroup of a prompt launch works on: query tile qt (BM rows) of one head of one sequence, and where that sequence's rows lie
struct PromptTile {
    int qt, head, b, q_beg, sq, k_beg, sk;
};

constexpr int kFewPrompts = 3;
__host__ __device__ __forceinline__ bool few_prompts(int batch) { return batch > 1 && batch <= kFewPrompts; }

// Two or three sequences (grid: heads x sequences x query tiles of the longest prompt): the tiles that see the most keys start first, whichever sequence they are of and however many
// keys it has cached, and a workgroup number that no tile is left for comes after all others.  Workgroups are dealt round-robin over the 8 XCDs, each with an L2 of its own: from 16
// pairs (sequence, key head) on, a multiple of 8, the tiles of a pair go to one XCD, the pairs with the most work dealt first, back and forth; fewer make one list for all XCDs.
// Against the order of the grid: 2 prompts of 2834 tokens, 512 of them cached, 16 / 8 heads of 128, 88.6 -> 72.9 us; 2 of 2703, 1280 cached, 14 / 2 of 64, 57.9 -> 53.9; over pages, 3 of
// 4792, 16 heads, 74.2 -> 70.9.  With more sequences finding the tile takes longer (1.5 us for 24) than the order gives: 9 of 11522, 28 / 4 heads of 128, 200 -> 208; 30 of 2294 27.0 -> 30.2.
// One alone has its heaviest tiles first in the order of the grid, and finding them is 0.7 us: over pages, 61 of 300 to 5000 tokens, 0.92 to 0.99 of the speed.
// Lane i of the first wave holds sequence i.  span > 0: keys a query sees at most.  words: 8 of the workgroup's LDS, free again behind it.
template <int BM>
__device__ __forceinline__ bool few_prompts_tile(const int32_t* cu_q, const int32_t* cu_k, int batch, int heads, int kv_heads, int span, int* words, PromptTile& t) {
    if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == 0) {
        const int lin = (int)blockIdx.x + (int)gridDim.x * ((int)blockIdx.y + (int)gridDim.y * (int)blockIdx.z);
        const int lane = threadIdx.x & 63, i = lane < batch ? lane : batch - 1;
        const int q_beg = cu_q[i], sq = cu_q[i + 1] - q_beg, k_beg = cu_k[i], sk = cu_k[i + 1] - k_beg;
        // sequences by their work: queries times the keys they see, in blocks of 64
        const uint32_t seen = (uint32_t)(sk > sq ? 2 * sk - sq : sk) >> 1, part = span > 0 && (uint32_t)span < seen ? (uint32_t)span : seen;
        const uint32_t work = (uint32_t)((sq + 63) >> 6) * ((part + 63) >> 6);
        const int key = lane < batch ? (int)(work < (1u << 24) ? work : 1u << 24) * 64 + 63 - lane : -1;
        int rank = 0;
#pragma unroll
        for (int j = 0; j < kFewPrompts; ++j) rank += __builtin_amdgcn_readlane(key, j) > key ? 1 : 0;
        const int order = __builtin_amdgcn_ds_permute(rank * 4, lane);           // lane r: the sequence of rank r
        // lane j: stream j of this workgroup's list, a (sequence, key head) or a sequence, its tiles on levels first .. first + n - 1
        const int G = heads / kv_heads, units = batch * kv_heads;
        const bool split = (units & 7) == 0 && units >= 16 && units <= 512;      // (then the grid is a multiple of 8 too)
        const int x = lin & 7, u = split ? 8 * lane + (lane & 1 ? 7 - x : x) : lane;
        const int of = split ? (int)(((float)u + 0.5f) * fast_rcp((float)kv_heads)) : lane;      // u / kv_heads (of at most 512)
        const int seq = __builtin_amdgcn_ds_bpermute(of * 4, order);
        const int my_tiles = (sq + BM - 1) / BM < (int)gridDim.z ? (sq + BM - 1) / BM : (int)gridDim.z, ahead = sk > sq ? (sk - sq) / BM : 0;
        const int its_tiles = __builtin_amdgcn_ds_bpermute(seq * 4, my_tiles), first = __builtin_amdgcn_ds_bpermute(seq * 4, ahead);     // (by all lanes)
        const int streams = split ? units >> 3 : batch, n = lane < streams ? its_tiles : 0, end = n > 0 ? first + n : 0;
        const int idx = split ? lin >> 3 : lin, heads_in = split ? G : heads, r0 = (int)((uint32_t)idx / (uint32_t)heads_in), g = idx - r0 * heads_in;
        // the level of tile r0 of the list: 64 levels at once, lane l counts the tiles from level top - 64 + l on
        float high = (float)end;
        high = max2(high, pair_in_row<1>(high));
        high = max2(high, pair_in_row<2>(high));
        high = max2(high, pair_in_row<4>(high));
        high = max2(high, pair_in_row<8>(high));
        high = max_xor32(max_xor16(high));
        int level = -1, r = 0;
        for (int top = __builtin_amdgcn_readfirstlane((int)high), above = 0; top > 0; top -= 64) {
            const int v = top - 64 + lane;
            int from = 0;
            for (int j = 0; j < streams; j += 4)
#pragma unroll
                for (int k = 0; k < 4; ++k) {        // (streams past the last one have no tiles)
                    const int e = __builtin_amdgcn_readlane(end, j + k), c = __builtin_amdgcn_readlane(n, j + k), left = e - v;
                    from += left < 0 ? 0 : left < c ? left : c;
                }
            const uint64_t hit = __builtin_amdgcn_ballot_w64(from > r0 && v >= 0);
            if (hit) {
                const int at = 63 - __builtin_clzll(hit);
                level = top - 64 + at;
                r = r0 - (at < 63 ? __builtin_amdgcn_readlane(from, (at + 1) & 63) : above);
                break;
            }
            above = __builtin_amdgcn_readlane(from, 0);
        }
        const uint64_t on = __builtin_amdgcn_ballot_w64(first <= level && level < end);
        const int below = __builtin_amdgcn_mbcnt_hi((uint32_t)(on >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)on, 0));
        const uint64_t mine = __builtin_amdgcn_ballot_w64(below == r) & on;
        const int j = mine ? __builtin_ctzll(mine) : 0, b = __builtin_amdgcn_readlane(seq, j);
        const int qt = level < 0 ? -1 : level - __builtin_amdgcn_readlane(first, j);
        const int head = split ? __builtin_amdgcn_readlane(u - of * kv_heads, j) * G + g : g;
        const int out[7] = {qt, head, b, __builtin_amdgcn_readlane(q_beg, b), __builtin_amdgcn_readlane(sq, b), __builtin_amdgcn_readlane(k_beg, b), __builtin_amdgcn_readlane(sk, b)};
        if (lane == 0) {
#pragma unroll
            for (int k = 0; k < 7; ++k) words[k] = out[k];
        }
    }
    __syncthreads();
    t.qt = __builtin_amdgcn_readfirstlane(words[0]), t.head = __builtin_amdgcn_readfirstlane(words[1]), t.b = __builtin_amdgcn_readfirstlane(words[2]);
    t.q_beg = __builtin_amdgcn_readfirstlane(words[3]), t.sq = __builtin_amdgcn_readfirstlane(words[4]);
    t.k_beg = __builtin_amdgcn_readfirstlane(words[5]), t.sk = __builtin_amdgcn_readfirstlane(words[6]);
    __syncthreads();
    return t.qt >= 0;
}

// rows of sequence t.b
__device__ __forceinline__ void prompt_rows(const int32_t* cu_q, const int32_t* cu_k, PromptTile& t) {
    t.q_beg = cu_q[t.b], t.sq = cu_q[t.b + 1] - t.q_beg, t.k_beg = cu_k[t.b], t.sk = cu_k[t.b + 1] - t.k_beg;
}

// (sequence, head, query tile) of this workgroup: the query tiles of one (sequence, head) share one XCD's L2, heaviest tiles first (workgroups are
// dealt round-robin over the 8 XCDs).  Grid: heads x sequences x query tiles.
__device__ __forceinline__ void attend_unit(int heads, int& qt, int& head, int& b) {
    qt = gridDim.z - 1 - blockIdx.z;
    head = blockIdx.x;
    b = blockIdx.y;
    const int units = (int)(gridDim.x * gridDim.y);
    if ((units & 7) == 0) {
        const int lin = (int)blockIdx.x + (int)gridDim.x * ((int)blockIdx.y + (int)gridDim.y * (int)blockIdx.z);
        const int idx = lin >> 3, per = units >> 3, u = (lin & 7) + 8 * (idx % per);
        b = u / heads;
        head = u - b * heads;
        qt = (int)gridDim.z - 1 - idx / per;
    }
}

}  // namespace nvh
