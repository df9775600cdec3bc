// C ABI of a decode step's layers in one launch.
#include <cmath>
#include <cstring>

#include "api_common.h"
#include "decode_layers.h"

namespace nvh {

static uint32_t magic_of(uint32_t d) { return (uint32_t)((1ull << 32) / d + 1); }

int plan_decode_layers(DecodeLayersArgs& a, int cus, int m, int hidden, int h, int kvh, int hd, int inter, int layers) {
    if (m < 1 || m > kDecodeLayersRows || (hd != 64 && hd != 128) || h <= 0 || kvh <= 0 || h % kvh || h / kvh > 16 || layers < 1 || layers > kDecodeLayersMost) return 0;
    const int qsize = h * hd, nqkv = (h + 2 * kvh) * hd;
    // what a wave holds of the weights: rows of up to 2, 4 and 10 times 64 pieces of 16 bytes
    if (hidden % 8 || inter % 8 || hidden <= 0 || inter <= 0 || hidden > 1024 || qsize > 2048 || inter > 5120 || cus < 64) return 0;
    const int kv = kDecodeLayersWalkers * kDecodeLayersBuffers * 64 * hd;
    const int front_lds = kLdsCommon + kv + 2 * m * (hidden + qsize) + 16 * (2 * hd + 16) + 2 * m * 2 * hd + kDecodeLayersWalkers * 2 * 16 * 4, rest_lds = kLdsCommon + 2 * m * (hidden + inter);
    const int lds = front_lds > rest_lds ? front_lds : rest_lds;
    if (lds > kDecodeLayersLds) return 0;
    auto per = [](int n, int parts) { return (n + parts - 1) / parts; };
    int best = 0, best_rounds = 0, best_load = 0;
    for (int nf = 16; nf <= cus - 16; nf += 4) {
        const int nm = cus - nf;
        const int rq = per(nqkv, nf), ro = per(hidden, nf), rg = per(inter, nm), rd = per(hidden, nm);
        if (nf < m * kvh || rq > 48 || ro > 24 || rg > 24 || rd > 8) continue;             // eight waves with three columns each, one of down; two rounds of qkv
        const int f = rq * hidden + ro * qsize, g = 2 * rg * hidden + rd * inter, load = f > g ? f : g, rounds = per(rq, 24);
        if (!best || rounds < best_rounds || (rounds == best_rounds && load < best_load)) { best = nf; best_rounds = rounds; best_load = load; }
    }
    if (!best) return 0;
    const int nf = best, nm = cus - nf;
    a.m = m; a.hidden = hidden; a.h = h; a.kvh = kvh; a.group = h / kvh; a.inter = inter; a.nqkv = nqkv; a.qsize = qsize; a.layers = layers;
    a.grid = cus; a.nf = nf; a.nm = nm;
    a.chunks = nf / (m * kvh) < 16 ? nf / (m * kvh) : 16;
    a.shares = m * kvh * a.chunks;
    a.nf_magic = magic_of(nf); a.nm_magic = magic_of(nm); a.chunks_magic = magic_of(a.chunks); a.kvh_magic = magic_of(kvh); a.group_magic = magic_of(a.group); a.h_magic = magic_of(h);
    a.o_qkv = 0; a.o_o = m * nqkv; a.o_act = a.o_o + m * hidden; a.o_down = a.o_act + m * inter; a.o_rec = a.o_down + m * hidden;
    a.layer_words = a.o_rec + (int64_t)a.shares * a.group * 2 * (hd + 2);
    int at = kLdsCommon;
    auto take = [&](int bytes) { const int x = at; at += bytes; return x; };
    a.l_kv = take(kv);
    a.l_x[0] = take(2 * m * hidden);
    a.l_x[2] = take(2 * m * qsize);
    a.l_q = take(16 * (2 * hd + 16));
    a.l_news = take(2 * m * 2 * hd);
    a.l_ml = take(kDecodeLayersWalkers * 2 * 16 * 4);
    a.l_x[1] = 0;
    at = kLdsCommon;
    a.l_x[3] = take(2 * m * hidden);
    a.l_x[4] = take(2 * m * inter);
    return lds;
}

// Contexts up to which this beats launches of their own, a multiple of 128, 0 for none.  Us a layer, from 3800 timed steps of 730 random shapes (1 to 32 layers; contexts of 1 to 12288): a
// launch saves 5.9 where one row is served and 1.2 less for each further one, 0.21 - 0.03 m a MB of weights, 1.5 with a q/k norm (a launch of its own there), and the split attention of a
// launch costs 0.5 up to 1024 tokens and 0.3 for every 1024.  It costs here, one behind the other: reading the shares of the attention (the output projection's workgroups read all of
// them, 1024 values and four shares a trip; 0.35 a trip alone, 0.6 in traffic of several rows), and 2.5 for every further round of tiles.  Starting all CUs is 8.  What is left has to be 0.85
// a layer, for all contexts up to that one.  Of 2480 of those steps that it then takes the slowest has 0.95 of the launches' speed and three others less than 0.99; by tokens a share
// alone, the second bound here, 349 of 3100 were slower, up to 0.63: three rows of 768 / 16 / 2 heads of 128, 5120 tokens, 476 us by launches and 629; one layer 31 and 41.
int decode_layers_tokens(int cus, int m, int hidden, int h, int kvh, int hd, int inter, int layers, bool qk_norm) {
    DecodeLayersArgs a{};
    if (!plan_decode_layers(a, cus, m, hidden, h, kvh, hd, inter, layers)) return 0;
    const float mb = 2e-6f * ((float)hidden * (a.nqkv + a.qsize) + 3.f * (float)hidden * inter);
    // Attention is the front's alone, its tokens come a round (two tiles of 16 of each of eight waves) behind the other, where a launch of its own has the whole chip: up to six times
    // 128 tokens a share of one sequence, three and a half of two, two and a half of three.  Whole steps, this against launches: Qwen3-0.6B one sequence of 4096 tokens (2.8 times 128 a
    // share) 654 us against 823; two of 1500 / 2500 / 3500 (2.1 / 3.6 / 5 times) 682 / 806 / 888 against 776 / 828 / 845; three of 1500 (3.2) 807 against 837; Qwen2-0.5B two of 4096
    // (2.7) 564 against 628, three of 2048 / 4096 (2 / 4) 579 / 671 against 619 / 639
    const int most = a.chunks * kDecodeLayersWalkers * 16 * (m == 1 ? 12 : m == 2 ? 7 : 5) / 2;
    int tokens = 0;
    for (int ctx = 128; ctx <= most; ctx += 128) {
        const int used = (ctx + 255) / 256 < a.chunks ? (ctx + 255) / 256 : a.chunks, rounds = (ctx + 256 * used - 1) / (256 * used);
        const int trips = (m * a.qsize + 1023) / 1024 * (used <= 2 ? 1 : (used + 3) / 4);
        const float gain = 5.9f - 1.2f * m + (0.21f - 0.03f * m) * mb + (qk_norm ? 1.5f : 0.f) - (a.qsize > 1024 ? 0.5f : 0.f) + 0.5f * (ctx < 1024 ? ctx : 1024) / 1024 + 0.3f * ctx / 1024 -
                           (m == 1 ? 0.35f : 0.6f) * trips - 2.5f * (rounds - 1);
        if (layers * (gain - 0.85f) < 8.f) break;
        tokens = ctx;
    }
    return tokens;
}

static int device_cus() {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    return v;
}

}  // namespace nvh

using namespace nvh;

extern "C" {

size_t nvh_decode_layers_workspace(int m, int hidden, int h, int kvh, int hd, int inter, int n_layers) {
    DecodeLayersArgs a{};
    if (!plan_decode_layers(a, device_cus(), m, hidden, h, kvh, hd, inter, n_layers)) return 0;
    return kDecodeLayersSync + (size_t)a.layer_words * 4 * n_layers;
}

int nvh_decode_layers_tokens(int m, int hidden, int h, int kvh, int hd, int inter, int n_layers) {
    return decode_layers_tokens(device_cus(), m, hidden, h, kvh, hd, inter, n_layers, false);
}

int nvh_decode_layers_tokens_for(int m, int hidden, int h, int kvh, int hd, int inter, int n_layers, int qk_norm) {
    return decode_layers_tokens(device_cus(), m, hidden, h, kvh, hd, inter, n_layers, qk_norm != 0);
}

int nvh_decode_layers_variant(uint32_t spin_limit, int late_from, int late_for, const nvh_decode_layers_desc* d, int dtype, void* stream) {
    REQUIRE(d, NVH_E_NULL, "decode_layers: null descriptor");
    if (d->m == 0) return 0;
    REQUIRE(dtype == NVH_BF16, NVH_E_DTYPE, "decode_layers: dtype %d unsupported (bf16 only)", dtype);
    REQUIRE(d->x && d->out && d->layers && d->positions && d->cos_sin && d->slot_mapping && d->context_lens && d->block_tables && d->workspace, NVH_E_NULL, "decode_layers: null pointer");
    REQUIRE(d->block_size > 0 && d->block_size % 64 == 0 && d->max_blocks > 0, NVH_E_SHAPE, "decode_layers: block_size %d must be a positive multiple of 64, max_blocks %d > 0",
            d->block_size, d->max_blocks);
    REQUIRE(d->x != d->out, NVH_E_SHAPE, "decode_layers: out may not be x");
    REQUIRE(!d->out_packed || d->hidden % 32 == 0, NVH_E_SHAPE, "decode_layers: out_packed needs hidden %% 32 == 0");
    DecodeLayersArgs a{};
    const int lds = plan_decode_layers(a, device_cus(), d->m, d->hidden, d->h, d->kvh, d->hd, d->inter, d->n_layers);
    REQUIRE(lds, NVH_E_SHAPE, "decode_layers: m %d hidden %d heads %d/%d of %d inter %d layers %d not served", d->m, d->hidden, d->h, d->kvh, d->hd, d->inter, d->n_layers);
    const size_t need = kDecodeLayersSync + (size_t)a.layer_words * 4 * d->n_layers;
    REQUIRE(d->workspace_bytes >= need, NVH_E_WORKSPACE, "decode_layers: workspace %zu B < required %zu B", d->workspace_bytes, need);
    REQUIRE(d->x_row_stride % 8 == 0 && d->x_row_stride >= d->hidden && d->out_row_stride >= d->hidden && d->bt_row_stride >= d->max_blocks, NVH_E_STRIDE, "decode_layers: row strides");
    REQUIRE(aligned16(d->x) && aligned16(d->cos_sin) && aligned16(d->workspace), NVH_E_ALIGN, "decode_layers: pointers must be 16-byte aligned");
    const bool qk_norm = d->layers[0].q_norm_w != nullptr;
    for (int i = 0; i < d->n_layers; ++i) {
        const nvh_decode_layer& l = d->layers[i];
        REQUIRE(l.qkv_w && l.o_w && l.gate_up_w && l.down_w && l.k_cache && l.v_cache && (l.q_norm_w != nullptr) == qk_norm && (l.k_norm_w != nullptr) == qk_norm, NVH_E_NULL,
                "decode_layers: null pointer in layer %d", i);
        REQUIRE(aligned16(l.qkv_w) && aligned16(l.o_w) && aligned16(l.gate_up_w) && aligned16(l.down_w) && aligned16(l.k_cache) && aligned16(l.v_cache) && aligned16(l.q_norm_w) &&
                aligned16(l.k_norm_w), NVH_E_ALIGN, "decode_layers: pointers must be 16-byte aligned (layer %d)", i);
        a.layer[i] = l;
    }
    a.x = (const uint16_t*)d->x; a.x_stride = d->x_row_stride; a.out = (uint16_t*)d->out; a.out_stride = d->out_row_stride; a.out_packed = (uint16_t*)d->out_packed;
    a.positions = d->positions; a.cos_sin = d->cos_sin; a.slots = d->slot_mapping; a.context_lens = d->context_lens; a.block_tables = d->block_tables; a.bt_stride = d->bt_row_stride;
    a.block_size = d->block_size; a.max_blocks = d->max_blocks;
    a.norm_eps = d->norm_eps; a.post_eps = d->post_eps; a.qk_eps = d->qk_eps; a.scale_log2 = d->scale * kLog2e;
    a.sync = (uint32_t*)d->workspace; a.ws = a.sync + kDecodeLayersSync / 4;
    a.spin_limit = spin_limit ? spin_limit : 4096; a.late_from = late_for > 0 ? late_from : 0x7fffffff; a.late_for = late_for;
    return launch_decode_layers(a, d->hd, qk_norm, lds, (hipStream_t)stream);
}

int nvh_decode_layers_stream(void* stream) {
    constexpr int kWords = 32;
    uint32_t mask[kWords] = {};
    const int cus = device_cus(), words = (cus + 31) / 32;
    if (cus <= 0 || words > kWords || hipExtStreamGetCUMask((hipStream_t)stream, words, mask) != hipSuccess) {
        (void)hipGetLastError();
        return cus > 0;                                                          // (no answer: a stream like others)
    }
    int n = 0;
    for (int i = 0; i < words; ++i) n += __builtin_popcount(mask[i]);
    return n >= cus;
}

int nvh_decode_layers_status(const void* workspace, uint32_t* gave_up) {
    REQUIRE(workspace && gave_up, NVH_E_NULL, "decode_layers_status: null pointer");
    const hipError_t e = hipMemcpy(gave_up, (const uint32_t*)workspace + kDecodeLayersGaveUp, sizeof(uint32_t), hipMemcpyDeviceToHost);
    REQUIRE(e == hipSuccess, (int)e, "decode_layers_status: %s", hipGetErrorString(e));
    return 0;
}

int nvh_decode_layers(const nvh_decode_layers_desc* d, int dtype, void* stream) { return nvh_decode_layers_variant(0, 0, 0, d, dtype, stream); }

}  // extern "C"
