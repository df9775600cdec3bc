// A decode step's layers in one launch (decode_layers.hip): arguments, and how shares, LDS and scratch are laid out.
#pragma once
#include <stdint.h>

#include "../../include/nvh_attn.h"
#include "common.h"

namespace nvh {

constexpr int kDecodeLayersMost = 32;            // layers of a launch: their pointers are kernel arguments (4 KB)
constexpr int kDecodeLayersRows = 3;             // sequences of a step
constexpr int kDecodeLayersLds = 160 * 1024;
constexpr int kDecodeLayersSync = 1024;          // bytes in front of the words: [0] launches so far, [1] workgroups of this one that have started,
constexpr int kDecodeLayersGaveUp = 64;          // [64] a workgroup gave up
constexpr int kDecodeLayersColumns = 48;            // of a workgroup's share of a projection (of gate and of up each)
constexpr int kLdsSay = 0, kLdsResults = 128, kLdsRope = kLdsResults + kDecodeLayersRows * kDecodeLayersColumns * 4, kLdsCommon = kLdsRope + kDecodeLayersRows * 128 * 4;     // bytes of LDS both kinds of workgroup lay out alike
constexpr int kDecodeLayersWalkers = 8, kDecodeLayersBuffers = 2;      // attention: waves that take tiles of 16 tokens, and tiles of a wave in LDS

struct DecodeLayersArgs {
    const uint16_t* x;                           // [m, hidden], the stream in front of the first layer
    int64_t x_stride;
    uint16_t* out;                               // [m, hidden] behind the last one; not x
    int64_t out_stride;
    uint16_t* out_packed;                        // nullable: also in fragment order
    const int64_t* positions;
    const float* cos_sin;
    const int32_t* slots;
    const int32_t* context_lens;
    const int32_t* block_tables;
    int64_t bt_stride;
    uint32_t* sync;
    uint32_t* ws;
    int64_t layer_words;
    int m, hidden, h, kvh, group, inter, nqkv, qsize, layers, block_size, max_blocks;
    int grid, nf, nm;                            // workgroups; of the front; of the feed-forward
    int chunks, shares;                          // attention: shares of a (sequence, key head); of all
    float norm_eps, post_eps, qk_eps, scale_log2;
    uint32_t spin_limit;
    int late_from, late_for;
    uint32_t nf_magic, nm_magic, chunks_magic, kvh_magic, group_magic, h_magic;
    int o_qkv, o_o, o_act, o_down, o_rec;        // words of a layer
    int l_kv, l_q, l_news, l_ml;      // bytes of LDS
    int l_x[5];                                  // inputs of the phases
    nvh_decode_layer layer[kDecodeLayersMost];
};

static_assert(sizeof(DecodeLayersArgs) <= 4096, "kernel arguments");

// Fills everything but pointers; returns the bytes of LDS, 0 if these sizes are not served.
int plan_decode_layers(DecodeLayersArgs& a, int cus, int m, int hidden, int h, int kvh, int hd, int inter, int layers);
// Longest context up to which it pays (0: never): of any step whose table is no wider.
int decode_layers_tokens(int cus, int m, int hidden, int h, int kvh, int hd, int inter, int layers, bool qk_norm);
int launch_decode_layers(const DecodeLayersArgs& a, int hd, bool qk_norm, int lds, hipStream_t stream);

}  // namespace nvh
