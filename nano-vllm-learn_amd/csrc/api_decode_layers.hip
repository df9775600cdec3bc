// C ABI of a decode step's layers in one launch.
#include <cmath>
#include <cstring>

#include "api_common.h"
#include "decode_layers.h"

namespace nvh {

static int up(int x, int to) { return (x + to - 1) / to * to; }
static uint32_t magic_of(uint32_t d) { return (uint32_t)((1ull << 32) / d + 1); }

int plan_decode_layers(DecodeLayersArgs& a, int cus, int m, int hidden, int h, int kvh, int hd, int inter, int layers) {
    if (m < 1 || m > kDecodeLayersRows || (hd != 64 && hd != 128) || kvh <= 0 || h % kvh || h / kvh > 16 || layers < 1 || layers > kDecodeLayersMost) return 0;
    if (hidden % 8 || inter % 8 || hidden <= 0 || inter <= 0 || hidden > 8192 || inter > 16384 || cus < 64) return 0;
    const int qsize = h * hd, nqkv = (h + 2 * kvh) * hd;
    const int kv = kDecodeLayersWalkers(hd) * kDecodeLayersBuffers(hd) * 64 * hd;
    auto per = [](int n, int parts) { return (n + parts - 1) / parts; };
    int best = 0, best_rounds = 0, best_load = 0, best_lds = 0;
    for (int nf = 16; nf <= cus - 16; nf += 4) {
        const int nm = cus - nf;
        const int rq = per(nqkv, nf), ro = per(hidden, nf), rg = per(inter, nm), rd = per(hidden, nm);
        if (nf < m * kvh || rq > kDecodeLayersColumns || ro > kDecodeLayersColumns || rg > kDecodeLayersColumns || rd > kDecodeLayersColumns) continue;
        const int f = up(rq * hidden * 2, 1024) + up(ro * qsize * 2, 1024) + kv + 2 * m * (hidden + qsize) + 16 * (2 * hd + 16) + 2 * m * 2 * hd + kDecodeLayersWalkers(hd) * 2 * 16 * 4;
        const int g = 2 * up(rg * hidden * 2, 1024) + up(rd * inter * 2, 1024) + 2 * m * (hidden + inter);
        if (kLdsCommon + f > kDecodeLayersLds || kLdsCommon + g > kDecodeLayersLds) continue;
        const int rounds = per(rq, 24) + per(ro, 24) + 2 * per(rg, 24) + per(rd, 24), load = f > g ? f : g;
        if (!best || rounds < best_rounds || (rounds == best_rounds && load < best_load)) { best = nf; best_rounds = rounds; best_load = load; best_lds = kLdsCommon + load; }
    }
    if (!best) return 0;
    const int nf = best, nm = cus - nf;
    a.m = m; a.hidden = hidden; a.h = h; a.kvh = kvh; a.group = h / kvh; a.inter = inter; a.nqkv = nqkv; a.qsize = qsize; a.layers = layers;
    a.grid = cus; a.nf = nf; a.nm = nm;
    a.chunks = nf / (m * kvh) < 16 ? nf / (m * kvh) : 16;
    a.shares = m * kvh * a.chunks;
    // Attention is the front's alone, its tiles of 16 tokens come a round of the waves at a time (1.3 us), where a launch of its own has the whole chip: five rounds of one
    // sequence are worth what the rest gains, three of two.  Whole steps, one launch against five a layer: Qwen3-0.6B one sequence of 2000 / 4096 tokens (3 / 5 rounds) 652 / 755 us
    // against 768 / 817; two of 768 / 1500 / 2500 (2 / 4 / 6 rounds) 666 / 765 / 867 against 737 / 771 / 834; Qwen2-0.5B two of 4096 (3 rounds) 572 against 639
    a.most_tokens = a.chunks * kDecodeLayersWalkers(hd) * 16 * (m == 1 ? 5 : 3);
    a.nf_magic = magic_of(nf); a.nm_magic = magic_of(nm); a.chunks_magic = magic_of(a.chunks); a.kvh_magic = magic_of(kvh); a.group_magic = magic_of(a.group); a.h_magic = magic_of(h);
    a.o_qkv = 0; a.o_o = m * nqkv; a.o_act = a.o_o + m * hidden; a.o_down = a.o_act + m * inter; a.o_rec = a.o_down + m * hidden;
    a.layer_words = a.o_rec + (int64_t)a.shares * a.group * 2 * (hd + 2);
    int at = kLdsCommon;
    auto take = [&](int bytes) { const int x = at; at += bytes; return x; };
    a.l_region[0] = take(up(per(nqkv, nf) * hidden * 2, 1024));
    a.l_region[2] = take(up(per(hidden, nf) * qsize * 2, 1024));
    a.l_kv = take(kv);
    a.l_x[0] = take(2 * m * hidden);
    a.l_x[2] = take(2 * m * qsize);
    a.l_q = take(16 * (2 * hd + 16));
    a.l_news = take(2 * m * 2 * hd);
    a.l_ml = take(kDecodeLayersWalkers(hd) * 2 * 16 * 4);
    a.l_region[1] = a.l_x[1] = 0;
    at = kLdsCommon;
    a.l_up = up(per(inter, nm) * hidden * 2, 1024);
    a.l_region[3] = take(2 * a.l_up);
    a.l_region[4] = take(up(per(hidden, nm) * inter * 2, 1024));
    a.l_x[3] = take(2 * m * hidden);
    a.l_x[4] = take(2 * m * inter);
    return best_lds;
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
    DecodeLayersArgs a{};
    return plan_decode_layers(a, device_cus(), m, hidden, h, kvh, hd, inter, n_layers) ? a.most_tokens : 0;
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

int nvh_decode_layers(const nvh_decode_layers_desc* d, int dtype, void* stream) { return nvh_decode_layers_variant(0, 0, 0, d, dtype, stream); }

}  // extern "C"
