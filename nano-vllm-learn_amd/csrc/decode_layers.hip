// A decode step's layers in one launch, for one or two sequences: (folded RMSNorm ->) qkv projection -> (q/k norm ->) RoPE, K/V store and attention over pages ->
// output projection + residual -> (folded RMSNorm ->) gate_up, SiLU -> down projection + residual, for every layer of a decoder whose layers fit the LDS of the
// chip (Qwen2-0.5B: 30 MB a layer, 40 MB of LDS).  Replaces five launches a layer (nanovllm/models/qwen3.py:179-193).
//
// What bounds such a step is latency.  A launch that depends on the one before costs 1.5 us of boundary, 0.5 of dispatch and 1.9 until its first weights arrive,
// five times a layer (Qwen2-0.5B, one sequence: 22 us a layer, whose weights stream in 6).  Here:
//   * The workgroups, one a CU, stay.  `nf` of them (the front) hold rows of the qkv and output projections and attend, the others hold rows of gate_up and
//     down.  A workgroup keeps its rows of the weights in LDS and asks for the next layer's as soon as it is done with this layer's: the front's weights and
//     keys travel while the others work, theirs while the front works.  (Weights asked for while a workgroup itself waits would cost it their time: a wave's
//     loads, and those of a CU, return in order, and a poll waits behind them.)
//   * Results go from workgroup to workgroup through memory, marked: an activation is a 4-byte word (bf16 value, low half of the launch's number), a share of
//     an attention output an 8-byte word (fp32 value, number of the launch).  Both are written and read whole, so a reader that finds the mark has the value:
//     no flag, no fence, no second trip.  A hop between all workgroups takes 1.5 to 1.8 us, with a flag for each workgroup 2.4 to 3.2.  Stores are written
//     through, loads pass the caches (sc1).  Every layer has words of its own, so no word is written twice by a launch, and every launch writes all that it
//     reads: what such a word holds before is the mark of an earlier launch (or 0, as it was allocated).
//   * A wait that lasts too long (`spin_limit` polls, 3 ms: workgroups that have not been placed yet, because another stream's kernels hold their CUs) is ended
//     by work: the workgroup goes through the phases since its last one and does every share of which no results have come, whose ever it is.  A share's inputs
//     are complete when it is done; done twice it writes the same bits; and nothing is overwritten that a share reads.  So the step ends however few workgroups
//     run at a time.
// A column of a product is a wave's: its lanes take 16-byte pieces of the weight row and of the activations and add up (reads of 1 KB from LDS without conflicts;
// 16 x 16 matrix tiles would read 64 lanes' worth for the few columns a workgroup has: 2.1 us for the down projection where this takes 0.7).
// One sequence of 513 to 1024 tokens, Qwen2-0.5B, whole step with the LM head: 603 -> 387 us; two sequences 604 -> 459; Qwen3-0.6B 733 -> 556 and 737 -> 666.
// Arithmetic and rounding points are those of linear_stream.hip, rope_store.hip and decode_chunked.h (P as hi + lo); sums have another order.
#include "decode_layers.h"

#include "decode_chunked.h"

// RoPE's products and sums round separately (this file is built without contraction)
#pragma clang fp contract(off)

namespace nvh {

namespace {

constexpr int kWavesWg = 12, kThreads = kWavesWg * 64;
constexpr int kPhases = 5;
constexpr int kMostColumns = kDecodeLayersColumns;
constexpr int kRounds = 2;                       // rounds of the waves over the columns of a share, at most (plan_decode_layers)
constexpr int kFlightFront = 4, kFlightRest = 2;               // loads of weights a wave has under way
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
    static_assert(N == 1 || N == 2 || N == 4 || N == 8 || N == 16, "");
    if constexpr (N == 1) {
        asm volatile("global_load_dwordx4 %0, %1, %2 sc1\n s_waitcnt vmcnt(0)" : "=&v"(v[0]) : "v"(off[0]), "s"(base) : "memory");
    } else if constexpr (N == 2) {
        asm volatile("global_load_dwordx4 %0, %2, %4 sc1\n global_load_dwordx4 %1, %3, %4 sc1\n s_waitcnt vmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]) : "v"(off[0]), "v"(off[1]), "s"(base) : "memory");
    } else if constexpr (N == 4) {
        asm volatile("global_load_dwordx4 %0, %4, %8 sc1\n global_load_dwordx4 %1, %5, %8 sc1\n global_load_dwordx4 %2, %6, %8 sc1\n"
                     "global_load_dwordx4 %3, %7, %8 sc1\n s_waitcnt vmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]) : "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(base) : "memory");
    } else if constexpr (N == 16) {
        asm volatile("global_load_dwordx4 %0, %16, %32 sc1\n"
                     "global_load_dwordx4 %1, %17, %32 sc1\n"
                     "global_load_dwordx4 %2, %18, %32 sc1\n"
                     "global_load_dwordx4 %3, %19, %32 sc1\n"
                     "global_load_dwordx4 %4, %20, %32 sc1\n"
                     "global_load_dwordx4 %5, %21, %32 sc1\n"
                     "global_load_dwordx4 %6, %22, %32 sc1\n"
                     "global_load_dwordx4 %7, %23, %32 sc1\n"
                     "global_load_dwordx4 %8, %24, %32 sc1\n"
                     "global_load_dwordx4 %9, %25, %32 sc1\n"
                     "global_load_dwordx4 %10, %26, %32 sc1\n"
                     "global_load_dwordx4 %11, %27, %32 sc1\n"
                     "global_load_dwordx4 %12, %28, %32 sc1\n"
                     "global_load_dwordx4 %13, %29, %32 sc1\n"
                     "global_load_dwordx4 %14, %30, %32 sc1\n"
                     "global_load_dwordx4 %15, %31, %32 sc1\n s_waitcnt vmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7]), "=&v"(v[8]), "=&v"(v[9]), "=&v"(v[10]), "=&v"(v[11]), "=&v"(v[12]), "=&v"(v[13]), "=&v"(v[14]), "=&v"(v[15])
                     : "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "v"(off[4]), "v"(off[5]), "v"(off[6]), "v"(off[7]), "v"(off[8]), "v"(off[9]), "v"(off[10]), "v"(off[11]), "v"(off[12]), "v"(off[13]), "v"(off[14]), "v"(off[15]), "s"(base) : "memory");
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

// sums over the wave of two values: of the first in the lower 32 lanes, of the second in the upper ones
__device__ __forceinline__ float sum_two(float x, float y) {
    float t = fold32(x, y);
    t = sum_xor16(t);
    return group_sum<16>(t);
}

template <int D>
struct Walk {                                    // attention: waves that take 16-token tiles, and tiles of a wave in LDS
    static constexpr int kWaves = kDecodeLayersWalkers(D), kBufs = kDecodeLayersBuffers(D);
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
        say[0] = load_word((const Word*)a.sync);
        say[1] = say[2] = say[3] = 0;
        __hip_atomic_fetch_add(a.sync + 32, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((int)blockIdx.x >= a.late_from)
            for (int i = 0; i < a.late_for; ++i) __builtin_amdgcn_s_sleep(8);    // (tests: workgroups that start late)
    }
    // what every layer needs of the step's rows: context, slot, cos and sin of the position
    LdsWord* const row_ctx = say + 8, * const row_slot = say + 8 + M;
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
    struct Share { int c0, n, k, region, x; };
    auto share = [&](Args& a, int ph, int role) {
        Share s;
        const int N = ph == PH_QKV ? a.nqkv : ph == PH_GATE_UP ? a.inter : a.hidden;
        const int R = ph <= PH_O ? a.nf : a.nm;
        const uint32_t magic = ph <= PH_O ? a.nf_magic : a.nm_magic;
        s.c0 = div_by(N * role, R, magic);
        s.n = div_by(N * (role + 1), R, magic) - s.c0;
        s.k = ph == PH_O ? a.qsize : ph == PH_DOWN ? a.inter : a.hidden;
        s.region = a.l_region[ph];
        s.x = a.l_x[ph];
        return s;
    };
    // ---- this wave's part of a share's weights into LDS, as they lie in memory
    auto ask_rows = [&](const uint16_t* w, int bytes, int to) {
        const int lane = lane_now();
        const char* const src = reinterpret_cast<const char*>(w);
        for (int i = wave * 1024; i < bytes; i += kWavesWg * 1024) {
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + min(i + 16 * lane, bytes - 16)),
                                             (__attribute__((address_space(3))) void*)(lds + to + i), 16, 0, NVH_DMA_AUX);
            if (front) loads_left<kFlightFront - 1>();
            else loads_left<kFlightRest - 1>();
        }
    };
    auto ask_weights = [&](Args& a, int l, int ph, int role) {
        const Share s = share(a, ph, role);
        const uint16_t* const w = reinterpret_cast<const uint16_t*>(ph == PH_QKV ? a.layer[l].qkv_w : ph == PH_O ? a.layer[l].o_w : ph == PH_GATE_UP ? a.layer[l].gate_up_w : a.layer[l].down_w);
        ask_rows(w + (int64_t)s.c0 * s.k, s.n * s.k * 2, s.region);
        if (ph == PH_GATE_UP) ask_rows(w + (int64_t)(a.inter + s.c0) * s.k, s.n * s.k * 2, s.region + a.l_up);
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
        if (front) {
            ask_weights(a, l, PH_QKV, own);
            ask_tiles(a, l, own);
            ask_weights(a, l, PH_O, own);
        } else {
            ask_weights(a, l, PH_GATE_UP, own);
            ask_weights(a, l, PH_DOWN, own);
        }
    };

    // ---- gathering.  quads: 16-byte pieces, thread t takes t, t + kThreads, ...; use(piece, words) for each.  Marks are checked piece by piece
    uint32_t limit = fresh_args().spin_limit;
    int flag = 2;                                                                // a word for every other share: a wave may wait for the next while another still looks at this one's
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

    // ---- products of R rows of weights with the M rows of activations: this lane's share of each sum.  A lane takes every 64th piece of 16 bytes; U pieces of
    // each row are asked for at once
    auto dots = [&](const unsigned char* x, int k, const unsigned char* const (&w)[4], auto rows_tag, auto unroll_tag, auto norm_tag, float (&acc)[4][M], float (&ss)[M]) {
        constexpr int R = decltype(rows_tag)::value, U = decltype(unroll_tag)::value;
        constexpr bool norm = decltype(norm_tag)::value;
        const int lane = lane_now(), pieces = k >> 3;
        for (int p0 = 0; p0 < pieces; p0 += 64 * U) {
            u32x4 xv[U][M], wv[U][R];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int p = p0 + 64 * u + lane;
#pragma unroll
                for (int m = 0; m < M; ++m) xv[u][m] = u32x4{0, 0, 0, 0};
#pragma unroll
                for (int r = 0; r < R; ++r) wv[u][r] = u32x4{0, 0, 0, 0};
                if (p < pieces) {
#pragma unroll
                    for (int m = 0; m < M; ++m) xv[u][m] = *reinterpret_cast<const u32x4*>(x + m * 2 * k + 16 * p);
#pragma unroll
                    for (int r = 0; r < R; ++r) wv[u][r] = *reinterpret_cast<const u32x4*>(w[r] + 16 * p);
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int m = 0; m < M; ++m)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if (norm) ss[m] = dot2_bf16(xv[u][m][i], xv[u][m][i], ss[m]);
#pragma unroll
                        for (int r = 0; r < R; ++r) acc[r][m] = dot2_bf16(xv[u][m][i], wv[u][r][i], acc[r][m]);
                    }
        }
    };

    bool have_x = false;                                                         // the stream that the residual sums need is in LDS
    // ---- one share of a projection: a wave takes two columns (gate_up: two of gate and the two of up that belong to them) of every 24
    // ready: its weights have been asked for.  Returns whether a wait ran out
    auto project = [&](auto phase, int l, int role, bool ready) -> bool {
        constexpr int ph = decltype(phase)::value;
        constexpr bool norm = ph == PH_QKV || ph == PH_GATE_UP;
        constexpr int C = ph == PH_DOWN ? 1 : 2;                                 // columns a wave takes at a time
        Args& a = fresh_args();
        const int G = a.group, lane = lane_now(), tid = wave * 64 + lane;
        Word* const words = layer_words(a, l);
        const Share s = share(a, ph, role);
        const int half = C == 2 ? lane >> 5 : 0, row = C * wave + half;
        const unsigned char* const xs = lds + s.x;
        const unsigned char* const ws = lds + s.region;
        const int up = a.l_up, hidden = a.hidden;
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
            for (int i = 0; i < kRounds; ++i) bias[i] = (float)reinterpret_cast<const __bf16*>(a.layer[l].qkv_bias)[s.c0 + min(row + 2 * kWavesWg * i, s.n - 1)];
        }
        asm volatile("" ::"s"(s.c0), "s"(s.n), "s"(s.k), "s"(up), "s"(hidden), "s"(eps), "s"(to), "s"(width), "s"((int)at_end), "s"(inv_k));      // read in front of the wait
        if (!ready) ask_weights(a, l, ph, role);
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
                else if (used <= 4) merge(0, std::integral_constant<int, 4>{});
                else
                    for (int c0 = 0; c0 < used; c0 += 8) merge(c0, std::integral_constant<int, 8>{});
                const float inv = mx == -INFINITY ? 0.f : fast_rcp(sum);         // (no tokens: zeros)
                *reinterpret_cast<uint32_t*>(lds + s.x + 2 * (bh * D + 2 * d2)) = pack_bf16x2(o0 * inv, o1 * inv);
            }
        }
        drain_loads();                                                           // this wave's part of the weights
        barrier_lds();
        const bool late = __builtin_amdgcn_readfirstlane(say[flag]) != 0;
        for (int i = 0; C * (wave + kWavesWg * i) < s.n; ++i) {
            const int r0 = C * (wave + kWavesWg * i), r1 = min(r0 + 1, s.n - 1), r = r0 + half;
            float acc[4][M], ss[M];
#pragma unroll
            for (int m = 0; m < M; ++m) acc[0][m] = acc[1][m] = acc[2][m] = acc[3][m] = ss[m] = 0.f;
            const unsigned char* const rows[4] = {ws + r0 * 2 * s.k, ws + r1 * 2 * s.k, ws + up + r0 * 2 * s.k, ws + up + r1 * 2 * s.k};
            dots(xs, s.k, rows, std::integral_constant<int, ph == PH_GATE_UP ? 4 : C>{}, std::integral_constant<int, ph == PH_DOWN ? (M == 1 ? 10 : 5) : 2>{}, std::bool_constant<norm>{}, acc, ss);
#pragma unroll
            for (int m = 0; m < M; ++m) {
                float y = sum_two(acc[0][m], acc[C - 1][m]), u = 0.f;
                if (ph == PH_GATE_UP) u = sum_two(acc[2][m], acc[3][m]);
                float scale = 1.f;
                if (norm) scale = rsqrtf(sum_two(ss[m], ss[m]) * inv_k + eps);
                if ((C == 2 ? lane & 31 : lane) || r >= s.n) continue;
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
    auto attend = [&](int l, int role, bool ready) -> bool {
        Args& a = fresh_args();
        const int G = a.group, lane = lane_now(), tid = wave * 64 + lane, lq = lane & 15, lg = lane >> 4;
        Word* const words = layer_words(a, l);
        if (role >= a.shares) return false;
        const Chunk ck = chunk_of(a, role);
        if (ck.c >= max(ck.used, 1)) return false;                           // (without tokens the first share says so)
        unsigned char* const qs = lds + a.l_q;                               // [head][D + 8]
        unsigned char* const news = lds + a.l_news;                          // [row of the batch][k, v][D]
        float* const ml = reinterpret_cast<float*>(lds + a.l_ml);            // [wave][max, sum][16]
        const int live_waves = min(max(ck.tiles - ck.c * W::kWaves, 0), W::kWaves);
        const int tile0 = first_tile(ck), tile_step = ck.used * W::kWaves;
        unsigned char* const kv0 = lds + a.l_kv;
        unsigned char* const kv_wave = kv0 + wave * W::kWave;
        Word* const rec = uniform(words + a.o_rec + (int64_t)(ck.pair * a.chunks + ck.c) * G * (2 * (D + 2)));
        const float scale_log2 = a.scale_log2;
        if (!ready) {                                                            // (another workgroup's share: the own tiles are found again behind it)
            find_tiles(a, role);
            ask_tiles(a, l, role);
        }
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
            for (uint32_t spins = 0;;) {
                load_through(v, src, off);
                if ((marked(v[0], mark16) && marked(v[1], mark16)) || ran_out(spins)) break;
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
            if (row) {
                *reinterpret_cast<u32x2*>(row) = p1;
                *reinterpret_cast<u32x2*>(row + D / 2) = p2;
            }
        }
        barrier_lds();
        const bool late = __builtin_amdgcn_readfirstlane(say[flag]) != 0;
        if (late) return true;
        if (wave < live_waves) {
            bf16x8 qf[STEPS];
#pragma unroll
            for (int st = 0; st < STEPS; ++st) qf[st] = *reinterpret_cast<const bf16x8*>(qs + min(lq, G - 1) * (2 * D + 16) + (4 * st + lg) * 16);
            const int dp = lane % LPT, dr = lane / LPT;
            float m_run = -INFINITY, l_run = 0.f;
            f32x4 o[DT];
#pragma unroll
            for (int t = 0; t < DT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
            int buf = 0;
            for (int tile = tile0; tile < ck.tiles; tile += tile_step) {
                if (tile >= tile0 + W::kBufs * tile_step) drain_loads();
                const int t0 = 16 * tile, n_live = ck.ctx - t0;
                unsigned char* const lds_k = kv_wave + buf * W::kBuf;
                unsigned char* const lds_v = lds_k + W::kImage;
                int from = tile_from[0];
                if (W::kBufs > 1 && tile == tile0 + tile_step) from = tile_from[W::kBufs - 1];
                else if (tile != tile0) from = new_row(ck, tile, slot_of(a, ck, t0));
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
                f32x4 sT = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int st = 0; st < STEPS; ++st) {
                    const bf16x8 kf = *reinterpret_cast<const bf16x8*>(lds_k + lq * W::kRow + (((4 * st + lg) ^ chunk_swizzle<LPT>(lq)) * 16));
                    sT = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[st], sT, 0, 0, 0);
                }
                const int vq = lq >> 2, vp = lq & 3, R = 4 * lg + vq;        // lane 4q + p of its group addresses key row q, dims 4p..
                const uint32_t vrow = lds_offset(lds_v + R * W::kRow + (vp & 1) * 8);
                const int swz = chunk_swizzle_v<LPT>(R);
                u32x2 vt[DT];
#pragma unroll
                for (int t = 0; t < DT; ++t) vt[t] = ds_read_tr16_b64_asm(vrow + ((2 * t + (vp >> 1)) ^ swz) * 16);
                if (n_live < 16) {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (4 * lg + r >= n_live) sT[r] = -INFINITY;
                }
                asm volatile("s_nop 7\n\ts_nop 7" : "+v"(sT));               // the maxima below are asm statements: the compiler does not pad them behind the products
                float mx = max2(max2(sT[0], sT[1]), max2(sT[2], sT[3]));
                mx = max_xor16(mx);
                mx = max_xor32(mx);
                const float m_new = max2(m_run, mx * scale_log2), alpha = fast_exp2(m_run - m_new);
                bf16x4 p_hi, p_lo;
                float lsum = 0.f;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float pv = fast_exp2(fmaf(sT[r], scale_log2, -m_new));
                    lsum += pv;
                    p_hi[r] = (__bf16)pv;
                    p_lo[r] = (__bf16)(pv - (float)p_hi[r]);
                }
                l_run = l_run * alpha + lsum;
                m_run = m_new;
#pragma unroll
                for (int t = 0; t < DT; ++t) o[t] = o[t] * alpha;
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
                typedef short s16x4 __attribute__((ext_vector_type(4)));
                const s16x4 hi = __builtin_bit_cast(s16x4, p_hi), lo = __builtin_bit_cast(s16x4, p_lo);
#pragma unroll
                for (int t = 0; t < DT; ++t) o[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, vt[t]), hi, o[t], 0, 0, 0);
#pragma unroll
                for (int t = 0; t < DT; ++t) o[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, vt[t]), lo, o[t], 0, 0, 0);
                if (tile + W::kBufs * tile_step < ck.tiles) ask_tile(a, l, ck, tile + W::kBufs * tile_step, slot_of(a, ck, 16 * (tile + W::kBufs * tile_step)), buf);
                buf = buf + 1 == W::kBufs ? 0 : buf + 1;
            }
            l_run = sum_xor16(l_run);
            l_run = sum_xor32(l_run);
            if (lq < G) {                                                    // over this wave's own images, all read by now
                float* const fin = reinterpret_cast<float*>(kv_wave) + lq * D + 4 * lg;
#pragma unroll
                for (int t = 0; t < DT; ++t) *reinterpret_cast<f32x4*>(fin + 16 * t) = o[t];
                if (lg == 0) {
                    ml[(wave * 2 + 0) * 16 + lq] = m_run;
                    ml[(wave * 2 + 1) * 16 + lq] = l_run;
                }
            }
        }
        barrier_lds();
        for (int it = tid; it < G * D / 2; it += kThreads) {                 // two dims of a head to a thread
            const int g = it / (D / 2), d2 = it % (D / 2);
            float mw[W::kWaves], lw[W::kWaves];
            f32x2 ow[W::kWaves];
#pragma unroll
            for (int w = 0; w < W::kWaves; ++w) {                            // (waves without tiles repeat the last one that has some, and do not count)
                const int wc = min(w, max(live_waves - 1, 0));
                mw[w] = ml[(wc * 2 + 0) * 16 + g];
                lw[w] = ml[(wc * 2 + 1) * 16 + g];
                ow[w] = reinterpret_cast<const f32x2*>(kv0 + wc * W::kWave)[it];
            }
            float mx = -INFINITY, sum = 0.f;
            f32x2 ov = {0.f, 0.f};
            if (live_waves > 0) {
                mx = mw[0];
#pragma unroll
                for (int w = 1; w < W::kWaves; ++w) mx = fmaxf(mx, mw[w]);
#pragma unroll
                for (int w = 0; w < W::kWaves; ++w) {
                    const float f = w < live_waves ? fast_exp2(mw[w] - mx) : 0.f;
                    ov[0] = fmaf(ow[w][0], f, ov[0]);
                    ov[1] = fmaf(ow[w][1], f, ov[1]);
                    sum = fmaf(lw[w], f, sum);
                }
            }
            Word* const p = rec + g * (2 * (D + 2));
            st16_global_sc1((void*)(p + 4 * d2), u32x4{__float_as_uint(ov[0]), mark32, __float_as_uint(ov[1]), mark32});
            if (d2 == 0) st16_global_sc1((void*)(p + 2 * D), u32x4{__float_as_uint(mx), mark32, __float_as_uint(sum), mark32});
        }
        return false;
    };
    auto run = [&](int l, int ph, int role, bool ready) -> bool {
        flag ^= 1;
        l = __builtin_amdgcn_readfirstlane(l);                                   // (what the compiler does not see: else it reads the layer's pointers by vector loads)
        role = __builtin_amdgcn_readfirstlane(role);
        switch (__builtin_amdgcn_readfirstlane(ph)) {
            case PH_QKV: return project(std::integral_constant<int, PH_QKV>{}, l, role, ready);
            case PH_ATTEND: return attend(l, role, ready);
            case PH_O: return project(std::integral_constant<int, PH_O>{}, l, role, ready);
            case PH_GATE_UP: return project(std::integral_constant<int, PH_GATE_UP>{}, l, role, ready);
            default: return project(std::integral_constant<int, PH_DOWN>{}, l, role, ready);
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
    if (front) find_tiles(fresh_args(), own);
    ask_layer(0);
    while (l < layers && !lost) {
        int rl = l, rp = ph, rr = own;
        if (help_t >= 0) {
            rl = help_t / kPhases;
            rp = help_t - rl * kPhases;
            if (help_role >= (rp <= PH_O ? fresh_args().nf : fresh_args().nm)) {
                help_role = 0;
                if (++help_t < l * kPhases + ph) continue;
                help_t = -1;                                                     // what this workgroup waited for is there
                limit = min(fresh_args().spin_limit, 64u);
                lost = ++rescues > 2 * kPhases * layers;
                if (front) find_tiles(fresh_args(), own);
                ask_layer(l);
                continue;
            }
            rr = help_role++;
            if (complete(rl, rp, rr)) continue;
        }
        const bool out = run(rl, rp, rr, help_t < 0);
        if (help_t >= 0) {
            lost = out;                                                          // (the inputs of a share that is done here are complete)
            __syncthreads();
        } else if (out) {
            __syncthreads();                                                     // (waits for this wave's loads into LDS, too)
            if (threadIdx.x == 0) say[2] = say[3] = 0;
            __syncthreads();
            have_x = false;
            limit = 1u << 20;
            help_t = last;
            help_role = 0;
        } else {
            last = l * kPhases + ph;
            have_x = ph == PH_QKV || ph == PH_GATE_UP || (ph == PH_ATTEND && have_x);
            const bool layer_done = ph == (front ? PH_O : PH_DOWN);
            ph = layer_done ? (front ? PH_QKV : PH_GATE_UP) : ph + 1;
            if (layer_done && ++l < layers) {
                barrier_lds();                                                   // the weights of this layer have been read
                ask_layer(l);
            }
        }
    }
    drain_loads();
    if (threadIdx.x == 0) {
        Args& a = fresh_args();
        if (lost) {                                                              // (never seen.  A workgroup that gave up leaves no plausible results, and says so)
            store_word((Word*)a.sync + 64, 1u);
            for (int i = 0; i < M * a.hidden; ++i) {
                a.out[i / a.hidden * a.out_stride + i % a.hidden] = 0x7fff;
                if (a.out_packed) a.out_packed[pack_index(i / a.hidden, i % a.hidden, a.hidden)] = 0x7fff;
            }
        }
        if (blockIdx.x == 0) {                                                   // the number of the next launch, once every workgroup of this one has read its own
            for (int i = 0; i < 1 << 24 && load_word((const Word*)a.sync + 32) != (uint32_t)a.grid; ++i) __builtin_amdgcn_s_sleep(8);
            store_word((Word*)a.sync + 32, 0u);
            store_word((Word*)a.sync, launch + 1);
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
        return a.m == 1 ? go(decode_layers_kernel<D, N, 1>) : go(decode_layers_kernel<D, N, 2>);
    };
    auto heads = [&](auto d) { return qk_norm ? rows(d, std::true_type{}) : rows(d, std::false_type{}); };
    return hd == 64 ? heads(std::integral_constant<int, 64>{}) : heads(std::integral_constant<int, 128>{});
}

}  // namespace nvh
