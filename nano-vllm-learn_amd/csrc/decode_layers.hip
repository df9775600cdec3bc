// A decode step's layers in one launch, for up to three sequences: (folded RMSNorm ->) qkv projection -> (q/k norm ->) RoPE, K/V store and attention over pages ->
// output projection + residual -> (folded RMSNorm ->) gate_up, SiLU -> down projection + residual, for every layer of a decoder whose layers fit the registers of
// the chip (Qwen2-0.5B: 30 MB a layer, 128 MB of registers).  Replaces five launches a layer (nanovllm/models/qwen3.py:179-193).
//
// What bounds such a step is latency.  A launch that depends on the one before costs 1.5 us of boundary, 0.5 of dispatch and 1.9 until its first weights arrive,
// five times a layer (Qwen2-0.5B, one sequence: 22 us a layer, whose weights stream in 6).  Here:
//   * The workgroups, one a CU, stay.  `nf` of them (the front) hold rows of the qkv and output projections and attend, the others hold rows of gate_up and
//     down.  A wave keeps its rows of the weights in registers and asks for the next layer's as soon as the workgroup is done with this layer's: the front's
//     weights and keys travel while the others work, theirs while the front works.  (Weights asked for while a workgroup itself waits would cost it their time: a
//     wave's loads, and those of a CU, return in order, and a poll waits behind them.  The others ask for two pieces at a time: 200 CUs with all of theirs under way
//     keep the front's polls waiting; four at a time 362 -> 366 us a step.)
//   * Results go from workgroup to workgroup through memory, marked: an activation is a 4-byte word (bf16 value, low half of the launch's number), a share of
//     an attention output an 8-byte word (fp32 value, number of the launch).  Both are written and read whole, so a reader that finds the mark has the value:
//     no flag, no fence, no second trip.  A hop between all workgroups takes 1.2 to 1.6 us, with a flag for each workgroup 2.4 to 3.2.  Stores are written
//     through, loads pass the caches (sc1).  Every layer has words of its own, so no word is written twice by a launch, and every launch writes all that it
//     reads: what such a word holds before is the mark of an earlier launch (or 0, as it was allocated).
//   * A wait that lasts too long (`spin_limit` polls, 3 ms: workgroups that have not been placed yet, because another stream's kernels hold their CUs) is ended
//     by work: the workgroup goes through the phases since its last one and does every share of which no results have come, whose ever it is.  A share's inputs
//     are complete when it is done; done twice it writes the same bits; and nothing is overwritten that a share reads.  So the step ends however few workgroups
//     run at a time.
// A column of a product is a wave's: its lanes hold 16-byte pieces of the weight row, 64 apart, and add up products with the same pieces of the activations
// (16 x 16 matrix tiles would read 64 lanes' worth of LDS for the few columns a workgroup has: 2.1 us for the down projection where this takes 0.5).  Eight waves of
// three columns rather than twelve of two: sums and epilogues are issued by fewer waves.  Up to three rows; four would take as long as launches of their own.
// Whole step with the LM head, contexts of 513 to 1024 tokens, launches -> this: Qwen2-0.5B one sequence 598 -> 354 us (layers with LDS for the weights and twelve
// waves 387), two 606 -> 443, three 606 -> 527; Qwen3-0.6B 730 -> 502, 733 -> 598, 761 -> 720.  For which sizes and contexts: decode_layers_tokens.
// Beside another stream (Qwen2-0.5B, one sequence; launches in brackets): copies of 256 MB 600 us (1130), small kernels 360 (603), attention over prompts 385 (602, at times 2770),
// products of 2048 400 (602), two such sessions 673 each (728): other streams' kernels get no CU while the step runs.  On a stream that may not use every CU workgroups start behind
// others' ends, and each part waits for that: 16 ms with 248 CUs, 53 with 128 (launches 0.63, 0.73).
// Arithmetic and rounding points are those of linear_stream.hip, rope_store.hip and decode_chunked.h (P as hi + lo); sums have another order.
#include "decode_layers.h"

#include "decode_chunked.h"

// RoPE's products and sums round separately (this file is built without contraction)
#pragma clang fp contract(off)

namespace nvh {

namespace {

constexpr int kWavesWg = 8, kThreads = kWavesWg * 64;
constexpr int kColumns = 3;                      // of a projection that a wave takes at a time (down: one)
constexpr int kPhases = 5;
constexpr int kMostColumns = kDecodeLayersColumns;
constexpr int kHeld = 24;                        // 16-byte registers of weights
constexpr int kRounds = 2;                       // rounds of the waves over the columns of a share, at most (plan_decode_layers)
constexpr int kFlightFront = 8, kFlightRest = 2;               // loads of weights a wave has under way
enum { PH_QKV, PH_ATTEND, PH_O, PH_GATE_UP, PH_DOWN };

__device__ __forceinline__ void barrier_lds() {  // orders LDS traffic only: loads into LDS stay in flight
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ void drain_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// words of the exchange: in global memory, at an address that is the same for the wave and in scalar registers (an access that the compiler takes for a flat one
// counts as LDS traffic too: the next barrier would wait for its acknowledgement)
typedef __attribute__((address_space(1))) uint32_t Word;
__device__ __forceinline__ Word* uniform(const Word* p) {
    const uint64_t v = (uint64_t)p;
    return (Word*)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(v >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)v));
}
// N 16-byte loads past the caches, waited for: base + off[i]
template <int N>
__device__ __forceinline__ void load_through(u32x4 (&v)[N], const Word* base, const uint32_t (&off)[N]) {
    static_assert(N == 1 || N == 2 || N == 4 || N == 8, "");
    if constexpr (N == 1) {
        asm volatile("global_load_dwordx4 %0, %1, %2 sc1\n s_waitcnt vmcnt(0)" : "=&v"(v[0]) : "v"(off[0]), "s"(base) : "memory");
    } else if constexpr (N == 2) {
        asm volatile("global_load_dwordx4 %0, %2, %4 sc1\n global_load_dwordx4 %1, %3, %4 sc1\n s_waitcnt vmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]) : "v"(off[0]), "v"(off[1]), "s"(base) : "memory");
    } else if constexpr (N == 4) {
        asm volatile("global_load_dwordx4 %0, %4, %8 sc1\n global_load_dwordx4 %1, %5, %8 sc1\n global_load_dwordx4 %2, %6, %8 sc1\n"
                     "global_load_dwordx4 %3, %7, %8 sc1\n s_waitcnt vmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]) : "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(base) : "memory");
    } else {
        asm volatile("global_load_dwordx4 %0, %8, %16 sc1\n global_load_dwordx4 %1, %9, %16 sc1\n global_load_dwordx4 %2, %10, %16 sc1\n"
                     "global_load_dwordx4 %3, %11, %16 sc1\n global_load_dwordx4 %4, %12, %16 sc1\n global_load_dwordx4 %5, %13, %16 sc1\n"
                     "global_load_dwordx4 %6, %14, %16 sc1\n global_load_dwordx4 %7, %15, %16 sc1\n s_waitcnt vmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
                     : "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "v"(off[4]), "v"(off[5]), "v"(off[6]), "v"(off[7]), "s"(base) : "memory");
    }
}
__device__ __forceinline__ void store_word(Word* p, uint32_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ uint32_t load_word(const Word* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ uint32_t bf16_bits(float v) { return __builtin_bit_cast(uint16_t, (__bf16)v); }
__device__ __forceinline__ int div_by(int x, uint32_t d, uint32_t magic) { return d == 1 ? x : (int)__umulhi((uint32_t)x, magic); }

// two activations' words -> their values as packed bf16
__device__ __forceinline__ uint32_t pair_of(uint32_t w0, uint32_t w1) { return __builtin_amdgcn_perm(w1, w0, 0x07060302u); }
__device__ __forceinline__ bool marked(const u32x4& v, uint32_t mark16) {
    const uint32_t d = ((v[0] ^ mark16) | (v[1] ^ mark16) | (v[2] ^ mark16) | (v[3] ^ mark16)) & 0xffffu;
    return d == 0;
}

// The arguments, read where they are used: left to itself the compiler reads all of them (and everything that hangs on them) in front of the loop over the layers
// and spills 330 scalar and 70 vector registers.
typedef const __attribute__((address_space(4))) DecodeLayersArgs Args;
__device__ __forceinline__ Args& fresh_args() {
    Args* p = (Args*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *p;
}

// wait until at most N of this wave's loads are under way
template <int N>
__device__ __forceinline__ void loads_left() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// Sums over the wave of four values: a row of 16 lanes each, in the order 0, 2, 1, 3 (column_of)
__device__ __forceinline__ float sum_four(float v0, float v1, float v2, float v3) { return group_sum<16>(fold16(fold32(v0, v1), fold32(v2, v3))); }
__device__ __forceinline__ int column_of(int lane) { return (lane >> 5) | ((lane >> 3) & 2); }
__device__ __forceinline__ float sum_wave(float v) {
    v = sum_xor16(v);
    v = sum_xor32(v);
    return group_sum<16>(v);
}

template <int D>
struct Walk {                                    // attention: waves that take 16-token tiles, and tiles of a wave in LDS
    static constexpr int kWaves = kDecodeLayersWalkers, kBufs = kDecodeLayersBuffers;
    static constexpr int kRow = D * 2, kImage = 16 * kRow, kBuf = 2 * kImage, kWave = kBufs * kBuf;
};

template <int D, bool QK_NORM, int M>
__global__ __launch_bounds__(kThreads) void decode_layers_kernel(const DecodeLayersArgs) {
    using W = Walk<D>;
    constexpr int LPT = D / 8, TPI = 64 / LPT, NI = 16 / TPI, STEPS = D / 32, DT = D / 16;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool front = (int)blockIdx.x < fresh_args().nf;
    const int own = front ? (int)blockIdx.x : (int)blockIdx.x - fresh_args().nf;

    typedef volatile __attribute__((address_space(3))) uint32_t LdsWord;         // (typed: the compiler takes a volatile access through lds for a flat one)
    LdsWord* const say = (LdsWord*)(lds + kLdsSay);                              // [0] launch number, [1] results are missing, [2], [3] a wait of this share ran out
    if (threadIdx.x == 0) {
        Args& a = fresh_args();
        // Launches so far and, in the high half, workgroups of this one that have started: the last of them puts the next launch's number there, when all others hold
        // this one's.  (A load, a counter and a wait of one workgroup for all to have started would need an end for that wait, and a number for whoever starts behind it.)
        typedef __attribute__((address_space(1))) uint64_t Start;
        Start* const start = (Start*)a.sync;
        const uint64_t was = __hip_atomic_fetch_add(start, 1ull << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((uint32_t)(was >> 32) == (uint32_t)a.grid - 1) __hip_atomic_store(start, (uint64_t)((uint32_t)was + 1u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        say[0] = (uint32_t)was;
        say[1] = say[2] = say[3] = 0;
        if ((int)blockIdx.x >= a.late_from)
            for (int i = 0; i < a.late_for; ++i) __builtin_amdgcn_s_sleep(8);    // (tests: workgroups that start late)
    }
    // what every layer needs of the step's rows: context, slot, cos and sin of the position
    LdsWord* const row_ctx = say + 8, * const row_slot = say + 16;
    float* const rope = reinterpret_cast<float*>(lds + kLdsRope);
    {
        Args& a = fresh_args();
        if (threadIdx.x < M) {
            row_ctx[threadIdx.x] = a.context_lens[threadIdx.x];
            row_slot[threadIdx.x] = a.slots[threadIdx.x];
        }
        for (int i = threadIdx.x; i < M * D; i += kThreads) rope[i] = a.cos_sin[a.positions[i / D] * D + i % D];
    }
    __syncthreads();
    uint32_t* const results = reinterpret_cast<uint32_t*>(lds + kLdsResults);   // [row of the batch][column of the share]
    const uint32_t launch = __builtin_amdgcn_readfirstlane(say[0]);
    const uint32_t mark32 = launch + 1, mark16 = mark32 & 0xffffu;
    auto layer_words = [&](Args& a, int l) { return uniform((const Word*)a.ws + (int64_t)l * a.layer_words); };

    // ---- a share of a projection: n columns from c0 on (gate_up: n of gate and the same n of up), contraction k
    struct Share { int c0, n, k, x; };
    auto share = [&](Args& a, int ph, int role) {
        Share s;
        const int N = ph == PH_QKV ? a.nqkv : ph == PH_GATE_UP ? a.inter : a.hidden;
        const int R = ph <= PH_O ? a.nf : a.nm;
        const uint32_t magic = ph <= PH_O ? a.nf_magic : a.nm_magic;
        s.c0 = div_by(N * role, R, magic);
        s.n = div_by(N * (role + 1), R, magic) - s.c0;
        s.k = ph == PH_O ? a.qsize : ph == PH_DOWN ? a.inter : a.hidden;
        s.x = a.l_x[ph];
        return s;
    };
    // ---- the weights of this wave's columns, in registers: a row's 16-byte pieces lie 64 apart in a lane (zeros past its end: the buffer says where that is).
    // Front: qkv, two rounds of three columns of two pieces, then the output projection, three of four; the others: gate, up, three columns of two each, then down, one of ten
    u32x4 held[kHeld];
    auto row_buffer = [&](const uint16_t* w, int row, int rows, int k, int skip) {         // (no such row, or none left behind `skip` bytes: zeros, and no traffic)
        const int bytes = row < rows && 2 * k > skip ? 2 * k - skip : 0;
        return __builtin_amdgcn_make_buffer_rsrc((void*)(w + (int64_t)(row < rows ? row : 0) * k + skip / 2), 0, bytes, 0x00020000);
    };
    auto ask_weights = [&](Args& a, int l, int role) {
        const Share s = share(a, front ? PH_QKV : PH_GATE_UP, role), t = share(a, front ? PH_O : PH_DOWN, role);
        const uint16_t* const w = reinterpret_cast<const uint16_t*>(front ? a.layer[l].qkv_w : a.layer[l].gate_up_w) + (int64_t)s.c0 * s.k;
        const uint16_t* const v = reinterpret_cast<const uint16_t*>(front ? a.layer[l].o_w : a.layer[l].down_w) + (int64_t)t.c0 * t.k;
        const int c = kColumns * wave, d = front ? c + kColumns * kWavesWg : c;
        const uint16_t* const w2 = front ? w : w + (int64_t)a.inter * s.k;
        const __amdgpu_buffer_rsrc_t row[9] = {
            row_buffer(w, c, s.n, s.k, 0), row_buffer(w, c + 1, s.n, s.k, 0), row_buffer(w, c + 2, s.n, s.k, 0),
            row_buffer(w2, d, s.n, s.k, 0), row_buffer(w2, d + 1, s.n, s.k, 0), row_buffer(w2, d + 2, s.n, s.k, 0),
            row_buffer(v, front ? c : wave, t.n, t.k, 0), row_buffer(v, front ? c + 1 : wave, t.n, t.k, front ? 0 : 4096), row_buffer(v, front ? c + 2 : wave, t.n, t.k, front ? 0 : 8192)};
        const int at = 16 * lane_now();
#pragma unroll
        for (int i = 0; i < kHeld; ++i) {
            held[i] = __builtin_amdgcn_raw_buffer_load_b128(row[i < 12 ? i >> 1 : i / 4 + 3], at + 1024 * (i < 12 ? i & 1 : i & 3), 0, NVH_DMA_AUX);       // (what the check of the end sees: not the scalar offset)
            if (front) loads_left<kFlightFront - 1>();
            else loads_left<kFlightRest - 1>();
        }
    };

    // ---- attention: what a share is
    struct Chunk { int b, g, c, pair, ctx, tiles, used; };
    auto used_of = [&](Args& a, int tiles) {                                     // shares that hold tokens: as many as keep all tiles in LDS, where there are so many
        return min((tiles + W::kWaves * W::kBufs - 1) / (W::kWaves * W::kBufs), a.chunks);
    };
    auto chunk_of = [&](Args& a, int role) {
        Chunk ck;
        ck.pair = div_by(role, a.chunks, a.chunks_magic);
        ck.c = role - ck.pair * a.chunks;
        ck.b = div_by(ck.pair, a.kvh, a.kvh_magic);
        ck.g = ck.pair - ck.b * a.kvh;
        ck.ctx = __builtin_amdgcn_readfirstlane(row_ctx[ck.b]);
        ck.tiles = (ck.ctx + 15) >> 4;
        ck.used = used_of(a, ck.tiles);
        return ck;
    };
    auto slot_of = [&](Args& a, const Chunk& ck, int t0) {                       // a tile of 16 tokens lies inside a page
        const int page = t0 / a.block_size;
        return a.block_tables[(int64_t)ck.b * a.bt_stride + min(page, a.max_blocks - 1)] * (int64_t)a.block_size + (t0 - page * a.block_size);
    };
    auto ask_tile = [&](Args& a, int l, const Chunk& ck, int tile, int64_t slot0, int buf) {
        const int lane = lane_now(), dp = lane % LPT, dr = lane / LPT;
        const int t0 = 16 * tile, last = ck.ctx - t0 - 1;
        const int64_t row = (int64_t)a.kvh * D, base = slot0 * row + (int64_t)ck.g * D;
        const uint16_t* const kc = reinterpret_cast<const uint16_t*>(a.layer[l].k_cache), * const vc = reinterpret_cast<const uint16_t*>(a.layer[l].v_cache);
        unsigned char* const img = lds + a.l_kv + wave * W::kWave + buf * W::kBuf;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int T = i * TPI + dr, Tc = min(T, last);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(kc + base + Tc * row + (dp ^ chunk_swizzle<LPT>(T)) * 8),
                                             (__attribute__((address_space(3))) void*)(img + i * 1024), 16, 0, NVH_DMA_AUX);
        }
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int T = i * TPI + dr, Tc = min(T, last);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(vc + base + Tc * row + (dp ^ chunk_swizzle_v<LPT>(T)) * 8),
                                             (__attribute__((address_space(3))) void*)(img + W::kImage + i * 1024), 16, 0, NVH_DMA_AUX);
        }
    };
    auto first_tile = [&](const Chunk& ck) { return ck.c < ck.used ? ck.c * W::kWaves + wave : ck.tiles; };
    // which token of this lane's row of a tile is one of this step's rows: their keys and values are not read from the cache (which this launch writes)
    auto new_row = [&](const Chunk& ck, int tile, int64_t slot0) {
        const int lq = lane_now() & 15, n_live = ck.ctx - 16 * tile;
        int from = -1;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int slot = row_slot[m];
            if (slot >= 0 && (int64_t)slot - slot0 == lq && lq < n_live) from = m;
        }
        return from;
    };
    // the first tiles of this wave in this workgroup's own share: the same in every layer
    int64_t tile_slot[W::kBufs];
    int tile_from[W::kBufs];
    auto find_tiles = [&](Args& a, int role) {
        if (wave >= W::kWaves || role >= a.shares) return;
        const Chunk ck = chunk_of(a, role);
        int t = first_tile(ck);
#pragma unroll
        for (int i = 0; i < W::kBufs; ++i, t += ck.used * W::kWaves) {
            tile_slot[i] = 0;
            tile_from[i] = -1;
            if (t < ck.tiles) {
                tile_slot[i] = slot_of(a, ck, 16 * t);
                tile_from[i] = new_row(ck, t, tile_slot[i]);
            }
        }
    };
    auto ask_tiles = [&](Args& a, int l, int role) {
        if (wave >= W::kWaves || role >= a.shares) return;
        const Chunk ck = chunk_of(a, role);
        int t = first_tile(ck);
#pragma unroll
        for (int i = 0; i < W::kBufs; ++i, t += ck.used * W::kWaves)
            if (t < ck.tiles) ask_tile(a, l, ck, t, tile_slot[i], i);
    };
    auto ask_layer = [&](int l) {                                                // everything of the next layer that waits for nothing
        l = __builtin_amdgcn_readfirstlane(l);
        Args& a = fresh_args();
        ask_weights(a, l, own);
        if (front) ask_tiles(a, l, own);
    };

    // ---- gathering.  quads: 16-byte pieces, thread t takes t, t + kThreads, ...; use(piece, words) for each.  Marks are checked piece by piece
    uint32_t limit = fresh_args().spin_limit;
    int flag = 2;                                                                // a word for every other share that passes barriers: a wave may wait for the next one while another still
                                                                                 // looks at this one's (attention that a workgroup has no share of passes none, and leaves the word as it is)
    auto ran_out = [&](uint32_t& spins) {
        if (++spins < limit) return false;
        say[flag] = 1;
        return true;
    };
    auto gather_words = [&](const Word* src, int quads, int t, auto use) {
        auto batch = [&](int q0, auto count) {
            constexpr int N = decltype(count)::value;
            u32x4 v[N];
            uint32_t off[N];
#pragma unroll
            for (int i = 0; i < N; ++i) off[i] = 16u * (uint32_t)min(q0 + i * kThreads, quads - 1);
            for (uint32_t spins = 0;;) {
                load_through(v, src, off);
                bool ok = true;
#pragma unroll
                for (int i = 0; i < N; ++i) ok = ok && marked(v[i], mark16);
                if (ok || ran_out(spins)) break;
            }
#pragma unroll
            for (int i = 0; i < N; ++i)
                if (q0 + i * kThreads < quads) use(q0 + i * kThreads, v[i]);
        };
        for (int q = t; q < quads;) {
            const int left = (quads - q + kThreads - 1) / kThreads;
            if (left == 1) batch(q, std::integral_constant<int, 1>{}), q += kThreads;
            else if (left == 2) batch(q, std::integral_constant<int, 2>{}), q += 2 * kThreads;
            else batch(q, std::integral_constant<int, 4>{}), q += 4 * kThreads;
        }
    };
    // M rows of k words into LDS as bf16 rows
    auto gather_rows = [&](int tid, const Word* src, int k, int x) {
        gather_words(src, M * (k >> 2), tid, [&](int q, const u32x4& v) { *reinterpret_cast<u32x2*>(lds + x + 8 * q) = u32x2{pair_of(v[0], v[1]), pair_of(v[2], v[3])}; });
    };
    auto gather_input = [&](Args& a, int tid, int l, int x) {                    // the stream in front of layer l
        if (l > 0) return gather_rows(tid, layer_words(a, l - 1) + a.o_down, a.hidden, x);
        const int per = a.hidden >> 3;
#pragma unroll
        for (int m = 0; m < M; ++m)
            for (int c = tid; c < per; c += kThreads) *reinterpret_cast<u32x4*>(lds + x + m * 2 * a.hidden + 16 * c) = *reinterpret_cast<const u32x4*>(a.x + m * a.x_stride + 8 * c);
    };

    // ---- products of R rows of P pieces with the M rows of activations: this lane's share of each sum.  piece(row, i): a piece of the row's weights
    auto dots = [&](const unsigned char* x, int k, auto rows_tag, auto pieces_tag, auto norm_tag, float (&acc)[6][M], float (&ss)[M], auto piece) {
        constexpr int R = decltype(rows_tag)::value, P = decltype(pieces_tag)::value;
        const int lane = lane_now(), last = (k >> 3) - 1;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            if (m > 0) asm volatile("" ::: "memory");                            // (a row's pieces at a time: registers)
            u32x4 xv[P];
#pragma unroll
            for (int i = 0; i < P; ++i) xv[i] = *reinterpret_cast<const u32x4*>(x + m * 2 * k + 16 * min(64 * i + lane, last));
#pragma unroll
            for (int i = 0; i < P; ++i) {
                if (64 * i + lane > last) xv[i] = u32x4{0, 0, 0, 0};
                u32x4 wv[R];
#pragma unroll
                for (int r = 0; r < R; ++r) wv[r] = piece(r, i);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if constexpr (decltype(norm_tag)::value) ss[m] = dot2_bf16(xv[i][j], xv[i][j], ss[m]);
#pragma unroll
                    for (int r = 0; r < R; ++r) acc[r][m] = dot2_bf16(xv[i][j], wv[r][j], acc[r][m]);
                }
            }
        }
    };

    bool have_x = false;                                                         // the stream that the residual sums need is in LDS
    // ---- one share of a projection: a wave takes three columns (gate_up: three of gate and the three of up that belong to them; down: one) of every 24
    // help: another workgroup's, whose weights are not held but read.  Returns whether a wait ran out
    auto project = [&](auto phase, auto help, int l, int role) -> bool {
        constexpr int ph = decltype(phase)::value;
        constexpr bool norm = ph == PH_QKV || ph == PH_GATE_UP;
        constexpr int C = ph == PH_DOWN ? 1 : kColumns;
        Args& a = fresh_args();
        const int G = a.group, lane = lane_now(), tid = wave * 64 + lane;
        Word* const words = layer_words(a, l);
        const Share s = share(a, ph, role);
        const int column = C > 1 ? column_of(lane) : 0, row = C * wave + column;
        const unsigned char* const xs = lds + s.x;
        const int hidden = a.hidden;
        const float eps = ph == PH_QKV ? a.norm_eps : a.post_eps;
        const bool at_end = ph == PH_DOWN && l == a.layers - 1;
        const float inv_k = 1.f / (float)s.k;
        Word* const to = uniform(words + (ph == PH_QKV ? a.o_qkv : ph == PH_O ? a.o_o : ph == PH_GATE_UP ? a.o_act : a.o_down) + s.c0);
        const int width = ph == PH_QKV ? a.nqkv : ph == PH_GATE_UP ? a.inter : hidden;
        const unsigned char* const res = lds + (ph == PH_O ? a.l_x[PH_QKV] : a.l_x[PH_GATE_UP]) + 2 * s.c0;
        float bias[kRounds];
#pragma unroll
        for (int i = 0; i < kRounds; ++i) bias[i] = 0.f;
        if (ph == PH_QKV && a.layer[l].qkv_bias) {
#pragma unroll
            for (int i = 0; i < kRounds; ++i) bias[i] = (float)reinterpret_cast<const __bf16*>(a.layer[l].qkv_bias)[s.c0 + min(row + C * kWavesWg * i, s.n - 1)];
        }
        asm volatile("" ::"s"(s.c0), "s"(s.n), "s"(s.k), "s"(hidden), "s"(eps), "s"(to), "s"(width), "s"((int)at_end), "s"(inv_k));      // read in front of the wait
        if (ph == PH_QKV || (ph == PH_O && !have_x)) gather_input(a, tid, l, a.l_x[PH_QKV]);
        if (ph == PH_GATE_UP || (ph == PH_DOWN && !have_x)) gather_rows(tid, words + a.o_o, hidden, a.l_x[PH_GATE_UP]);
        if (ph == PH_DOWN) gather_rows(tid, words + a.o_act, s.k, s.x);
        if (ph == PH_O) {
            // the shares of the attention outputs, merged (a thread: two dims of one head)
            const Word* const recs = uniform(words + a.o_rec);
            const int total = M * a.h * (D / 2);
            for (int it = tid; it < total; it += kThreads) {
                const int bh = it / (D / 2), d2 = it % (D / 2);                  // row of the batch * heads + head
                const int pair = div_by(bh, G, a.group_magic), g = bh - pair * G;   // (heads = kv heads * group: pairs are numbered alike)
                const int m = M == 1 ? 0 : div_by(bh, a.h, a.h_magic);
                const uint32_t base = 8u * (uint32_t)((pair * a.chunks * G + g) * (D + 2)), step = 8u * (uint32_t)(G * (D + 2));
                const int used = max(used_of(a, ((int)row_ctx[m] + 15) >> 4), 1);
                float mx = -INFINITY, sum = 0.f, o0 = 0.f, o1 = 0.f;
                auto merge = [&](int c0, auto count) {
                    constexpr int N = decltype(count)::value;
                    u32x4 v[2 * N];
                    uint32_t off[2 * N];
#pragma unroll
                    for (int i = 0; i < N; ++i) {
                        off[2 * i] = base + (uint32_t)min(c0 + i, used - 1) * step + 16 * d2;
                        off[2 * i + 1] = off[2 * i] - 16 * d2 + 8 * D;
                    }
                    for (uint32_t spins = 0;;) {
                        load_through(v, recs, off);
                        bool ok = true;
#pragma unroll
                        for (int i = 0; i < 2 * N; ++i) ok = ok && v[i][1] == mark32 && v[i][3] == mark32;
                        if (ok || ran_out(spins)) break;
                    }
                    float top = mx;
#pragma unroll
                    for (int i = 0; i < N; ++i) top = fmaxf(top, __uint_as_float(v[2 * i + 1][0]));
                    const float keep = mx == -INFINITY ? 0.f : fast_exp2(mx - top);
                    o0 *= keep; o1 *= keep; sum *= keep;
#pragma unroll
                    for (int i = 0; i < N; ++i) {
                        const float mi = __uint_as_float(v[2 * i + 1][0]);
                        const float f = c0 + i < used && mi != -INFINITY ? fast_exp2(mi - top) : 0.f;
                        o0 = fmaf(__uint_as_float(v[2 * i][0]), f, o0);
                        o1 = fmaf(__uint_as_float(v[2 * i][2]), f, o1);
                        sum = fmaf(__uint_as_float(v[2 * i + 1][2]), f, sum);
                    }
                    mx = top;
                };
                if (used == 1) merge(0, std::integral_constant<int, 1>{});
                else if (used == 2) merge(0, std::integral_constant<int, 2>{});
                else
                    for (int c0 = 0; c0 < used; c0 += 4) merge(c0, std::integral_constant<int, 4>{});
                const float inv = mx == -INFINITY ? 0.f : fast_rcp(sum);         // (no tokens: zeros)
                *reinterpret_cast<uint32_t*>(lds + s.x + 2 * (bh * D + 2 * d2)) = pack_bf16x2(o0 * inv, o1 * inv);
            }
        }
        barrier_lds();
#pragma unroll
        for (int i = 0; i < (ph == PH_QKV ? kRounds : 1); ++i) {
            if (C * (wave + kWavesWg * i) >= s.n) continue;
            const int r = C * (wave + kWavesWg * i) + column;
            float acc[6][M], ss[M];
#pragma unroll
            for (int m = 0; m < M; ++m) acc[0][m] = acc[1][m] = acc[2][m] = acc[3][m] = acc[4][m] = acc[5][m] = ss[m] = 0.f;
            constexpr int R = ph == PH_GATE_UP ? 6 : C, P = ph == PH_DOWN ? 10 : ph == PH_O ? 4 : 2, from = ph == PH_O || ph == PH_DOWN ? 12 : 0;
            using std::integral_constant;
            if constexpr (decltype(help)::value) {
                const uint16_t* const w = reinterpret_cast<const uint16_t*>(ph == PH_QKV ? a.layer[l].qkv_w : ph == PH_O ? a.layer[l].o_w : ph == PH_GATE_UP ? a.layer[l].gate_up_w
                                                                                                                                                          : a.layer[l].down_w) + (int64_t)s.c0 * s.k;
                const int c = C * (wave + kWavesWg * i);
                __amdgpu_buffer_rsrc_t rows[R];
#pragma unroll
                for (int q = 0; q < R; ++q) rows[q] = row_buffer(w + (q >= 3 ? (int64_t)a.inter * s.k : 0), c + q % 3, s.n, s.k, 0);
#pragma unroll 1
                for (int p = lane; p < (s.k >> 3) + lane; p += 64) {             // (the same sums in the same order, few registers)
                    u32x4 wv[R];
#pragma unroll
                    for (int q = 0; q < R; ++q) wv[q] = __builtin_amdgcn_raw_buffer_load_b128(rows[q], 16 * p, 0, 0);
#pragma unroll
                    for (int m = 0; m < M; ++m) {
                        u32x4 xv = *reinterpret_cast<const u32x4*>(xs + m * 2 * s.k + 16 * min(p, (s.k >> 3) - 1));
                        if (p >= s.k >> 3) xv = u32x4{0, 0, 0, 0};
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            if constexpr (norm) ss[m] = dot2_bf16(xv[j], xv[j], ss[m]);
#pragma unroll
                            for (int q = 0; q < R; ++q) acc[q][m] = dot2_bf16(xv[j], wv[q][j], acc[q][m]);
                        }
                    }
                }
            } else if (i == 0) {
                dots(xs, s.k, integral_constant<int, R>{}, integral_constant<int, P>{}, std::bool_constant<norm>{}, acc, ss, [&](int r, int p) { return held[from + r * P + p]; });
            } else {
                dots(xs, s.k, integral_constant<int, R>{}, integral_constant<int, P>{}, std::bool_constant<norm>{}, acc, ss, [&](int r, int p) { return held[6 + r * 2 + p]; });
            }
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const float y = C > 1 ? sum_four(acc[0][m], acc[1][m], acc[2][m], 0.f) : sum_wave(acc[0][m]);
                float u = 0.f, scale = 1.f;
                if (ph == PH_GATE_UP) u = sum_four(acc[3][m], acc[4][m], acc[5][m], 0.f);
                if (norm) scale = rsqrtf(sum_wave(ss[m]) * inv_k + eps);
                if ((C > 1 ? lane & 15 : lane) || column >= C || r >= s.n) continue;
                uint32_t v;
                if (ph == PH_QKV) {
                    v = bf16_bits(y * scale + (i == 0 ? bias[0] : bias[1]));
                } else if (ph == PH_GATE_UP) {
                    const float gt = (float)(__bf16)(y * scale), ut = (float)(__bf16)(u * scale);
                    v = bf16_bits((float)(__bf16)(gt / (1.f + __expf(-gt))) * ut);
                } else {
                    v = bf16_bits(y + (float)*reinterpret_cast<const __bf16*>(res + 2 * (m * hidden + r)));
                }
                results[m * kMostColumns + r] = v << 16 | mark16;
            }
        }
        barrier_lds();
        const bool late = __builtin_amdgcn_readfirstlane(say[flag]) != 0;
        // one wave stores a row's results: words of a line that come from several waves are so many writes one behind the other at the memory side, with polls
        // between them (hop 2.8 us instead of 1.3)
        if (wave < M && lane < s.n && !late) {
            const uint32_t v = results[wave * kMostColumns + lane];
            if (!at_end) {
                store_word(to + wave * width + lane, v);
            } else {
                a.out[wave * a.out_stride + s.c0 + lane] = (uint16_t)(v >> 16);
                if (a.out_packed) a.out_packed[pack_index(wave, s.c0 + lane, hidden)] = (uint16_t)(v >> 16);
            }
        }
        return late;
    };

    // ---- one share of the attention
    auto attend = [&](auto help, int l, int role) -> bool {
        Args& a = fresh_args();
        const int G = a.group, lane = lane_now(), tid = wave * 64 + lane, lq = lane & 15, lg = lane >> 4;
        Word* const words = layer_words(a, l);
        if (role >= a.shares) return false;
        const Chunk ck = chunk_of(a, role);
        if (ck.c >= max(ck.used, 1)) return false;                           // (without tokens the first share says so)
        flag ^= 1;
        unsigned char* const qs = lds + a.l_q;                               // [head][D + 8]
        unsigned char* const news = lds + a.l_news;                          // [row of the batch][k, v][D]
        float* const ml = reinterpret_cast<float*>(lds + a.l_ml);            // [wave][max, sum][16]
        const int live_waves = min(max(ck.tiles - ck.c * W::kWaves, 0), W::kWaves);
        const int tile0 = first_tile(ck), tile_step = ck.used * W::kWaves;
        unsigned char* const kv0 = lds + a.l_kv;
        unsigned char* const kv_wave = kv0 + wave * W::kWave;
        Word* const rec = uniform(words + a.o_rec + (int64_t)(ck.pair * a.chunks + ck.c) * G * (2 * (D + 2)));
        const float scale_log2 = a.scale_log2;
        if constexpr (decltype(help)::value) {                                   // (another workgroup's share: the own tiles are found again behind it)
            find_tiles(a, role);
            ask_tiles(a, l, role);
        }
        // addresses of the operands, found in front of the wait
        constexpr int B = W::kBufs;
        typedef const __attribute__((address_space(3))) bf16x8 LdsFrag;
        const int dp = lane % LPT, dr = lane / LPT;
        const int vq = lq >> 2, vp = lq & 3, vR = 4 * lg + vq;                   // lane 4q + p of its group addresses key row q, dims 4p..
        uint32_t q_at = lds_offset(qs + min(lq, G - 1) * (2 * D + 16) + lg * 16), k_at[STEPS], v_at[DT], fin_at = lds_offset(kv_wave) + lq * 4 * D + 16 * lg;
#pragma unroll
        for (int st = 0; st < STEPS; ++st) {
            k_at[st] = lds_offset(kv_wave) + lq * W::kRow + (((4 * st + lg) ^ chunk_swizzle<LPT>(lq)) * 16);
            asm volatile("" : "+v"(k_at[st]));
        }
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            v_at[t] = lds_offset(kv_wave) + W::kImage + vR * W::kRow + (vp & 1) * 8 + ((2 * t + (vp >> 1)) ^ chunk_swizzle_v<LPT>(vR)) * 16;
            asm volatile("" : "+v"(v_at[t]));
        }
        asm volatile("" : "+v"(q_at), "+v"(fin_at));
        int mg = tid / (D / 2), md = tid % (D / 2);                              // what this thread merges first: head, pair of dims
        uint32_t ml_at = lds_offset(ml) + 4 * mg, ow_at = lds_offset(kv0) + 8 * tid;
        asm volatile("" : "+v"(ml_at), "+v"(ow_at), "+v"(mg), "+v"(md));
        asm volatile("" ::"s"(rec), "s"(scale_log2), "s"(live_waves));
        drain_loads();                                                           // the first tiles (in front of the rows this share stores, whose acknowledgement nobody needs)
        // q heads of the group; k and v of every row (a row's earlier tokens may be rows of this batch): four dims of each half of a head to a thread
        const int items = (G + 2 * M) * LPT;
        const Word* const src = words + a.o_qkv;
        for (int it = tid; it < items; it += kThreads) {
            const int hh = it / LPT, c8 = it % LPT;
            const bool is_q = hh < G, is_v = hh >= G + M;
            const int m = is_q ? ck.b : is_v ? hh - G - M : hh - G;
            const int head = is_q ? ck.g * G + hh : (is_v ? a.h + a.kvh : a.h) + ck.g;
            f32x4 co = {1.f, 1.f, 1.f, 1.f}, si = {0.f, 0.f, 0.f, 0.f};
            if (!is_v) {
                const float* const cs = rope + m * D + 4 * c8;
                co = *reinterpret_cast<const f32x4*>(cs);
                si = *reinterpret_cast<const f32x4*>(cs + D / 2);
            }
            u32x2 w1 = {}, w2 = {};
            if constexpr (QK_NORM) {
                if (!is_v) {
                    const uint16_t* const nw = reinterpret_cast<const uint16_t*>(is_q ? a.layer[l].q_norm_w : a.layer[l].k_norm_w) + 4 * c8;
                    w1 = *reinterpret_cast<const u32x2*>(nw);
                    w2 = *reinterpret_cast<const u32x2*>(nw + D / 2);
                }
            }
            uint16_t* row = nullptr;
            if (!is_q && m == ck.b && ck.c == 0) {
                const int slot = row_slot[m];
                if (slot >= 0) row = reinterpret_cast<uint16_t*>(is_v ? a.layer[l].v_cache : a.layer[l].k_cache) + ((int64_t)slot * a.kvh + ck.g) * D + 4 * c8;
            }
            u32x4 v[2];
            const uint32_t o = 4u * (uint32_t)(m * a.nqkv + head * D + 4 * c8);
            const uint32_t off[2] = {o, o + 2 * D};
            bool there = false;
            for (uint32_t spins = 0; !there;) {
                load_through(v, src, off);
                there = marked(v[0], mark16) && marked(v[1], mark16);
                if (!there && ran_out(spins)) break;
            }
            float x1[4], x2[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) { x1[e] = bf16_hi(v[0][e]); x2[e] = bf16_hi(v[1][e]); }
            if constexpr (QK_NORM) {
                float ss = 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e) ss += x1[e] * x1[e] + x2[e] * x2[e];
                ss = group_sum<LPT>(ss);                                     // the LPT lanes of a head
                if (!is_v) {
                    const float inv = rsqrtf(ss * (1.f / D) + a.qk_eps);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        x1[e] = (float)(__bf16)((float)(__bf16)(x1[e] * inv) * (e & 1 ? bf16_hi(w1[e >> 1]) : bf16_lo(w1[e >> 1])));
                        x2[e] = (float)(__bf16)((float)(__bf16)(x2[e] * inv) * (e & 1 ? bf16_hi(w2[e >> 1]) : bf16_lo(w2[e >> 1])));
                    }
                }
            }
            float y1[4], y2[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float a1 = x1[e] * co[e], b1 = x2[e] * si[e], a2 = x2[e] * co[e], b2 = x1[e] * si[e];
                y1[e] = is_v ? x1[e] : a1 - b1;
                y2[e] = is_v ? x2[e] : a2 + b2;
            }
            const u32x2 p1 = {pack_bf16x2(y1[0], y1[1]), pack_bf16x2(y1[2], y1[3])}, p2 = {pack_bf16x2(y2[0], y2[1]), pack_bf16x2(y2[2], y2[3])};
            unsigned char* const dst = (is_q ? qs + hh * (2 * D + 16) : news + (2 * m + (is_v ? 1 : 0)) * 2 * D) + 8 * c8;
            *reinterpret_cast<u32x2*>(dst) = p1;
            *reinterpret_cast<u32x2*>(dst + D) = p2;
            if (row && there) {
                *reinterpret_cast<u32x2*>(row) = p1;
                *reinterpret_cast<u32x2*>(row + D / 2) = p2;
            }
        }
        barrier_lds();
        if (wave < live_waves) {
            bf16x8 qf[STEPS];
#pragma unroll
            for (int st = 0; st < STEPS; ++st) qf[st] = *(LdsFrag*)(q_at + 64 * st);
            float m_run = -INFINITY, l_run = 0.f;
            f32x4 o[DT];
#pragma unroll
            for (int t = 0; t < DT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
            auto tiles = [&](int tile, auto first_tag) {                         // the tiles of both buffers together
                constexpr bool first = decltype(first_tag)::value;
                f32x4 sT[B];
                u32x2 vt[B][DT];
#pragma unroll
                for (int b = 0; b < B; ++b) {
                    const int at = tile + b * tile_step, n_live = ck.ctx - 16 * at;
                    sT[b] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
                    if (n_live <= 0) continue;                                   // (the same for the wave)
                    unsigned char* const lds_k = kv_wave + b * W::kBuf;
                    unsigned char* const lds_v = lds_k + W::kImage;
                    const int from = first ? tile_from[b] : new_row(ck, at, slot_of(a, ck, 16 * at));
                    for (uint64_t hits = __builtin_amdgcn_ballot_w64(from >= 0 && lg == 0); hits; hits &= hits - 1) {
                        const int T = __builtin_ctzll(hits), m = __builtin_amdgcn_readlane(from, T);
                        const int which = lane / LPT, p = lane % LPT;
                        if (which < 2) {
                            const u32x4 v = *reinterpret_cast<const u32x4*>(news + (2 * m + which) * 2 * D + 16 * p);
                            *reinterpret_cast<u32x4*>(which ? lds_v + T * W::kRow + (p ^ chunk_swizzle_v<LPT>(T)) * 16 : lds_k + T * W::kRow + (p ^ chunk_swizzle<LPT>(T)) * 16) = v;
                        }
                    }
                    if (n_live < 16) {                                           // rows past the context: P = 0 must not meet a value that is not finite
#pragma unroll
                        for (int i = 0; i < NI; ++i) {
                            const int T = i * TPI + dr;
                            if (T >= n_live) *reinterpret_cast<u32x4*>(lds_v + T * W::kRow + dp * 16) = u32x4{0, 0, 0, 0};
                        }
                    }
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    sT[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int st = 0; st < STEPS; ++st) {
                        const bf16x8 kf = *(LdsFrag*)(k_at[st] + b * W::kBuf);
                        sT[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[st], sT[b], 0, 0, 0);
                    }
#pragma unroll
                    for (int t = 0; t < DT; ++t) vt[b][t] = ds_read_tr16_b64_asm(v_at[t] + b * W::kBuf);
                    if (n_live < 16) {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (4 * lg + r >= n_live) sT[b][r] = -INFINITY;
                    }
                }
                static_assert(B == 2, "");
                asm volatile("s_nop 7\n\ts_nop 7" : "+v"(sT[0]), "+v"(sT[1]));   // the maxima below are asm statements: the compiler does not pad them behind the products
                float mx = max2(max2(max2(sT[0][0], sT[0][1]), max2(sT[0][2], sT[0][3])), max2(max2(sT[1][0], sT[1][1]), max2(sT[1][2], sT[1][3])));
                mx = max_xor16(mx);
                mx = max_xor32(mx);
                const float m_new = max2(m_run, mx * scale_log2), alpha = fast_exp2(m_run - m_new);
                bf16x4 p_hi[B], p_lo[B];
                float lsum = 0.f;
#pragma unroll
                for (int b = 0; b < B; ++b)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float pv = fast_exp2(fmaf(sT[b][r], scale_log2, -m_new));
                        lsum += pv;
                        p_hi[b][r] = (__bf16)pv;
                        p_lo[b][r] = (__bf16)(pv - (float)p_hi[b][r]);
                    }
                l_run = l_run * alpha + lsum;
                m_run = m_new;
                if (!first) {
#pragma unroll
                    for (int t = 0; t < DT; ++t) o[t] = o[t] * alpha;
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
                typedef short s16x4 __attribute__((ext_vector_type(4)));
#pragma unroll
                for (int b = 0; b < B; ++b) {
                    if (ck.ctx <= 16 * (tile + b * tile_step)) continue;
#pragma unroll
                    for (int t = 0; t < DT; ++t)
                        o[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, vt[b][t]), __builtin_bit_cast(s16x4, p_hi[b]), o[t], 0, 0, 0);
#pragma unroll
                    for (int t = 0; t < DT; ++t)
                        o[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, vt[b][t]), __builtin_bit_cast(s16x4, p_lo[b]), o[t], 0, 0, 0);
                }
#pragma unroll
                for (int b = 0; b < B; ++b) {
                    const int next = tile + (B + b) * tile_step;
                    if (next < ck.tiles) ask_tile(a, l, ck, next, slot_of(a, ck, 16 * next), b);
                }
            };
            tiles(tile0, std::true_type{});
            for (int tile = tile0 + B * tile_step; tile < ck.tiles; tile += B * tile_step) {
                drain_loads();
                tiles(tile, std::false_type{});
            }
            l_run = sum_xor16(l_run);
            l_run = sum_xor32(l_run);
            if (lq < G) {                                                    // over this wave's own images, all read by now
#pragma unroll
                for (int t = 0; t < DT; ++t) *(__attribute__((address_space(3))) f32x4*)(fin_at + 64 * t) = o[t];
                if (lg == 0) {
                    ml[(wave * 2 + 0) * 16 + lq] = m_run;
                    ml[(wave * 2 + 1) * 16 + lq] = l_run;
                }
            }
        }
        barrier_lds();
        const bool late = __builtin_amdgcn_readfirstlane(say[flag]) != 0;
        for (int it = tid; it < G * D / 2; it += kThreads) {                     // two dims of a head to a thread
            typedef const __attribute__((address_space(3))) float LdsFloat;
            typedef const __attribute__((address_space(3))) f32x2 LdsPair;
            float mw[W::kWaves], lw[W::kWaves];
            f32x2 ow[W::kWaves];
#pragma unroll
            for (int w = 0; w < W::kWaves; ++w) {                                // (waves without tiles hold what they held: not counted)
                mw[w] = w < live_waves ? *(LdsFloat*)(ml_at + 128 * w) : -INFINITY;
                lw[w] = *(LdsFloat*)(ml_at + 128 * w + 64);
                ow[w] = *(LdsPair*)(ow_at + w * W::kWave);
            }
            float mx = -INFINITY, sum = 0.f;
            f32x2 ov = {0.f, 0.f};
            if (live_waves > 0) {
                mx = mw[0];
#pragma unroll
                for (int w = 1; w < W::kWaves; ++w) mx = fmaxf(mx, mw[w]);
#pragma unroll
                for (int w = 0; w < W::kWaves; ++w) {
                    if (w < live_waves) {
                        const float f = fast_exp2(mw[w] - mx);
                        ov[0] = fmaf(ow[w][0], f, ov[0]);
                        ov[1] = fmaf(ow[w][1], f, ov[1]);
                        sum = fmaf(lw[w], f, sum);
                    }
                }
            }
            if (!late) {
                Word* const p = rec + mg * (2 * (D + 2));
                st16_global_sc1((void*)(p + 4 * md), u32x4{__float_as_uint(ov[0]), mark32, __float_as_uint(ov[1]), mark32});
                if (md == 0) st16_global_sc1((void*)(p + 2 * D), u32x4{__float_as_uint(mx), mark32, __float_as_uint(sum), mark32});
            }
            ml_at += 4 * (kThreads / (D / 2));
            ow_at += 8 * kThreads;
            mg += kThreads / (D / 2);
        }
        return late;
    };
    auto run = [&](auto help, int l, int ph, int role) -> bool {
        if (ph != PH_ATTEND) flag ^= 1;                                          // (there behind the early ends)
        l = __builtin_amdgcn_readfirstlane(l);                                   // (what the compiler does not see: else it reads the layer's pointers by vector loads)
        role = __builtin_amdgcn_readfirstlane(role);
        switch (__builtin_amdgcn_readfirstlane(ph)) {
            case PH_QKV: return project(std::integral_constant<int, PH_QKV>{}, help, l, role);
            case PH_ATTEND: return attend(help, l, role);
            case PH_O: return project(std::integral_constant<int, PH_O>{}, help, l, role);
            case PH_GATE_UP: return project(std::integral_constant<int, PH_GATE_UP>{}, help, l, role);
            default: return project(std::integral_constant<int, PH_DOWN>{}, help, l, role);
        }
    };

    // ---- are the results of a share there?  (the same for the workgroup)
    auto complete = [&](int l, int ph, int role) -> bool {
        Args& a = fresh_args();
        const int G = a.group, tid = wave * 64 + lane_now();
        const Word* const words = layer_words(a, l);
        if (ph == PH_ATTEND) {
            if (role >= a.shares) return true;
            const Chunk ck = chunk_of(a, role);
            if (ck.c >= max(ck.used, 1)) return true;
            const int n = G * (D + 2);
            const Word* const rec = words + a.o_rec + (int64_t)role * n * 2;
            for (int i = tid; i < n; i += kThreads)
                if (load_word(rec + 2 * i + 1) != mark32) say[1] = 1;
        } else if (ph == PH_DOWN && l == a.layers - 1) {
            return true;                                                         // (no phase waits for these)
        } else {
            const Share s = share(a, ph, role);
            const int N = ph == PH_QKV ? a.nqkv : ph == PH_GATE_UP ? a.inter : a.hidden;
            const Word* const p = words + (ph == PH_QKV ? a.o_qkv : ph == PH_O ? a.o_o : ph == PH_GATE_UP ? a.o_act : a.o_down) + s.c0;
            for (int m = 0; m < M; ++m)
                if (tid < s.n && (load_word(p + m * N + tid) & 0xffffu) != mark16) say[1] = 1;
        }
        __syncthreads();
        const bool missing = __builtin_amdgcn_readfirstlane(say[1]) != 0;
        __syncthreads();
        if (threadIdx.x == 0) say[1] = 0;
        __syncthreads();
        return !missing;
    };

    // One loop over own shares and, after a wait that ran out, the shares it waits for: phase by phase from this workgroup's last one, those without results
    const int layers = fresh_args().layers;
    int l = 0, ph = front ? PH_QKV : PH_GATE_UP, last = 0, rescues = 0;
    int help_t = -1, help_role = 0;                                              // phase (of all layers) and share to look at next, while helping
    bool lost = false;
    bool find = true, ask = true;                                                // the first tiles, and what the layer reads, are to be asked for (again)
    while (l < layers && !lost) {
        if (help_t >= 0) {
            const int rl = help_t / kPhases, rp = help_t - rl * kPhases;
            if (help_role >= (rp <= PH_O ? fresh_args().nf : fresh_args().nm)) {
                help_role = 0;
                if (++help_t < l * kPhases + ph) continue;
                help_t = -1;                                                     // what this workgroup waited for is there
                limit = min(fresh_args().spin_limit, 64u);
                lost = ++rescues > 2 * kPhases * layers;
                find = ask = true;
                continue;
            }
            const int role = help_role++;
            if (complete(rl, rp, role)) continue;
            lost = run(std::true_type{}, rl, rp, role);                          // (the inputs of a share that is done here are complete)
            __syncthreads();
            continue;
        }
        if (ask) {
            if (front && find) find_tiles(fresh_args(), own);
            ask_layer(l);
            find = ask = false;
        }
        if (run(std::false_type{}, l, ph, own)) {
            __syncthreads();                                                     // (waits for this wave's loads into LDS, too)
            if (threadIdx.x == 0) say[2] = say[3] = 0;
            __syncthreads();
            have_x = false;
            limit = 1u << 20;
            help_t = last;
            help_role = 0;
            continue;
        }
        last = l * kPhases + ph;
        have_x = ph == PH_QKV || ph == PH_GATE_UP || (ph == PH_ATTEND && have_x);
        if (ph == (front ? PH_O : PH_DOWN)) {
            ph = front ? PH_QKV : PH_GATE_UP;
            ++l;
            barrier_lds();                                                       // the images of this layer have been read
            ask = l < layers;
        } else {
            ++ph;
        }
    }
    drain_loads();
    if (lost && threadIdx.x == 0) {                                              // (never seen.  A workgroup that gave up leaves no plausible results, and says so)
        Args& a = fresh_args();
        store_word((Word*)a.sync + kDecodeLayersGaveUp, 1u);
        for (int i = 0; i < M * a.hidden; ++i) {
            a.out[i / a.hidden * a.out_stride + i % a.hidden] = 0x7fff;
            if (a.out_packed) a.out_packed[pack_index(i / a.hidden, i % a.hidden, a.hidden)] = 0x7fff;
        }
    }
}

}  // namespace

int launch_decode_layers(const DecodeLayersArgs& a, int hd, bool qk_norm, int lds, hipStream_t stream) {
    auto go = [&](auto kernel) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kDecodeLayersLds);
        if (e != hipSuccess) { set_error("decode_layers: %s", hipGetErrorString(e)); return (int)e; }
        hipLaunchKernelGGL(kernel, dim3(a.grid), dim3(kThreads), lds, stream, a);
        return check_launch("decode_layers");
    };
    auto rows = [&](auto d, auto norm) {
        constexpr int D = decltype(d)::value;
        constexpr bool N = decltype(norm)::value;
        return a.m == 1 ? go(decode_layers_kernel<D, N, 1>) : a.m == 2 ? go(decode_layers_kernel<D, N, 2>) : go(decode_layers_kernel<D, N, 3>);
    };
    auto heads = [&](auto d) { return qk_norm ? rows(d, std::true_type{}) : rows(d, std::false_type{}); };
    return hd == 64 ? heads(std::integral_constant<int, 64>{}) : heads(std::integral_constant<int, 128>{});
}

}  // namespace nvh
