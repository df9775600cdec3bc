// C ABI of the mixture of experts (declared in include/nvh_attn.h): argument validation, dispatch.
// Nothing here allocates, synchronises or reads device memory, nvh_moe_experts_status aside: every other entry point is capture-safe.
#include "api_common.h"
#include "mixers.h"

using namespace nvh;

extern "C" {

int nvh_moe_route(const nvh_moe_route_desc* d, int dtype, void* stream) {
    REQUIRE(d, NVH_E_NULL, "moe_route: null descriptor");
    if (d->rows == 0) return 0;
    DTYPE("moe_route");
    REQUIRE(d->x && d->router && d->correction && d->ids && d->weights, NVH_E_NULL, "moe_route: null pointer");
    REQUIRE(d->rows > 0 && d->cols > 0 && d->cols % 8 == 0 && d->experts > 0 && d->experts <= kMoeMaxExperts && d->groups > 0 && d->experts % d->groups == 0 && d->keep > 0 &&
            d->keep <= d->groups && (!d->softmax || d->groups == 1) && d->top > 0 && d->top <= 64 && d->top <= d->keep * (d->experts / d->groups), NVH_E_SHAPE,
            "moe_route: %d experts (<= %d) in %d groups, %d kept, top %d (<= 64)", d->experts, kMoeMaxExperts, d->groups, d->keep, d->top);
    REQUIRE(d->x_stride % 8 == 0 && d->x_stride >= d->cols, NVH_E_STRIDE, "moe_route: row stride");
    REQUIRE(aligned16(d->x) && aligned16(d->router), NVH_E_ALIGN, "moe_route: pointers must be 16-byte aligned");
    return launch_moe_route(*d, dtype == NVH_F32, (hipStream_t)stream);
}

int nvh_moe_dispatch_blocks(int pairs) { return pairs > 0 ? moe_dispatch_blocks(pairs) : 0; }

int nvh_moe_dispatch(int32_t* slot_pair, int32_t* tiles, int32_t* counts, const int32_t* ids, int pairs, int experts, int tile_rows, int max_tiles, void* stream) {
    if (pairs == 0) return 0;
    REQUIRE(slot_pair && tiles && counts && ids, NVH_E_NULL, "moe_dispatch: null pointer");
    REQUIRE(pairs > 0 && experts > 0 && experts <= kMoeMaxExperts && tile_rows > 0 && max_tiles >= pairs / tile_rows + experts, NVH_E_SHAPE,
            "moe_dispatch: %d pairs %d experts: room for %d tiles of %d", pairs, experts, max_tiles, tile_rows);
    REQUIRE(aligned16(tiles), NVH_E_ALIGN, "moe_dispatch: tiles must be 16-byte aligned");
    return launch_moe_dispatch(slot_pair, tiles, counts, ids, pairs, experts, tile_rows, max_tiles, nullptr, 0, (hipStream_t)stream);
}

int nvh_moe_tile_rows(int pairs, int experts, int dtype) { return pairs > 0 && experts > 0 ? moe_tile_rows(pairs, experts, 1024, dtype == NVH_F32) : 0; }

static int moe_gemm_ok(const nvh_moe_gemm_desc* d, int dtype) {
    DTYPE("moe_gemm");
    REQUIRE(d->out && d->x && d->w && (d->tiles ? d->slot_pair != nullptr : d->ids != nullptr), NVH_E_NULL, "moe_gemm: null pointer");
    REQUIRE(d->pairs > 0 && d->top > 0 && d->pairs % d->top == 0 && d->experts > 0 && d->experts <= kMoeMaxExperts && d->n > 0 && d->n % 64 == 0 && d->k > 0 && d->k % 64 == 0,
            NVH_E_SHAPE, "moe_gemm: %d pairs of top %d, n %d k %d (%%64)", d->pairs, d->top, d->n, d->k);
    REQUIRE(!d->tiles || d->tile_rows == (dtype == NVH_F32 ? 64 : 128) || (dtype == NVH_BF16 && (d->tile_rows == 64 || d->tile_rows == 256)), NVH_E_SHAPE, "moe_gemm: tiles of %d rows", d->tile_rows);
    REQUIRE(d->tiles ? d->max_tiles > 0 && d->max_tiles <= 65535 : dtype == NVH_BF16 && d->pairs / d->top <= 64, NVH_E_SHAPE,
            "moe_gemm: %d tiles, or the small form with more than 64 rows", d->max_tiles);
    REQUIRE(!d->glu || (d->x_stride % 8 == 0 && d->x_stride >= d->k), NVH_E_STRIDE, "moe_gemm: row stride");
    REQUIRE(aligned16(d->out) && aligned16(d->x) && aligned16(d->w) && aligned16(d->tiles), NVH_E_ALIGN, "moe_gemm: pointers must be 16-byte aligned");
    return 0;
}

int nvh_moe_gemm(const nvh_moe_gemm_desc* d, int dtype, void* stream) {
    REQUIRE(d, NVH_E_NULL, "moe_gemm: null descriptor");
    if (d->pairs == 0) return 0;
    const int rc = moe_gemm_ok(d, dtype);
    return rc ? rc : launch_moe_gemm(*d, dtype == NVH_F32, (hipStream_t)stream);
}

// scratch of nvh_moe_experts in 32-bit words: units of the experts | chosen experts | pairs by expert | tiles | counts | links of the launch of both products
struct MoeScratch {
    int rows, max_tiles;                             // of a tile; tiles at most (rows 0: the small form, no tiles)
    size_t ids, slots, tiles, counts, links, link_words, words;
    MoeScratch(int tokens, int top, int experts, int n, int dtype) {
        const size_t pairs = (size_t)tokens * top, part = (pairs + 3) / 4 * 4;
        const bool small = dtype == NVH_BF16 && tokens <= 64;
        rows = small ? 0 : moe_tile_rows((int)pairs, experts, n, dtype == NVH_F32);
        max_tiles = small ? 0 : (int)pairs / rows + experts;
        ids = pairs * n / (dtype == NVH_F32 ? 1 : 2);
        slots = ids + part;
        tiles = slots + (small ? 0 : part);
        counts = tiles + 4 * (size_t)max_tiles;
        links = counts + (small ? 0 : (size_t)moe_dispatch_blocks((int)pairs) * experts);
        link_words = small || dtype != NVH_BF16 ? 0 : moe_links_words(rows, max_tiles);
        words = links + link_words;
    }
};
static bool moe_sizes_ok(int rows, int top, int experts, int n) {
    return rows > 0 && top > 0 && experts > 0 && experts <= kMoeMaxExperts && (int64_t)rows * top <= 0x7fffffff && n > 0 && n % 64 == 0;
}

// Both products in one launch: the rule of sizes, scratch with room for its links and what the second one reads in lines of its own, and outputs, which are stored while the first product still
// runs, apart from what that reads (two launches let `out` hold x).
static bool experts_in_one(const nvh_moe_experts_desc* d, const MoeScratch& s) {
    const auto apart = [&](const void* p, int64_t elems) {
        const uintptr_t a = reinterpret_cast<uintptr_t>(p), b = reinterpret_cast<uintptr_t>(d->out);
        return a + 2 * (uintptr_t)elems <= b || b + 2 * (uintptr_t)d->rows * d->top * d->cols <= a;
    };
    return s.link_words && d->scratch_bytes >= 4 * s.words && (reinterpret_cast<uintptr_t>(d->scratch) & 127) == 0 && moe_one_launch(d->rows * d->top, d->experts, d->n, d->cols, s.rows) &&
           apart(d->x, (d->rows - 1) * d->x_stride + d->cols) && apart(d->gate_up, (int64_t)d->experts * 2 * d->n * d->cols);
}

size_t nvh_moe_experts_scratch_bytes(int rows, int top, int experts, int n, int dtype) {
    return moe_sizes_ok(rows, top, experts, n) ? 4 * MoeScratch(rows, top, experts, n, dtype).words : 0;
}

int nvh_moe_experts_one_launch(const nvh_moe_experts_desc* d, int dtype) {
    REQUIRE(d, NVH_E_NULL, "moe_experts_one_launch: null descriptor");
    if (d->rows == 0) return 0;
    DTYPE("moe_experts_one_launch");
    REQUIRE(moe_sizes_ok(d->rows, d->top, d->experts, d->n) && d->cols > 0, NVH_E_SHAPE, "moe_experts_one_launch: sizes");
    return experts_in_one(d, MoeScratch(d->rows, d->top, d->experts, d->n, dtype));
}

static int moe_experts(const nvh_moe_experts_desc* d, int dtype, uint32_t wait_limit, uint32_t missing, void* stream) {
    REQUIRE(d, NVH_E_NULL, "moe_experts: null descriptor");
    if (d->rows == 0) return 0;
    DTYPE("moe_experts");
    REQUIRE(moe_sizes_ok(d->rows, d->top, d->experts, d->n), NVH_E_SHAPE, "moe_experts: %d rows, top %d of %d experts (<= %d), n %d (%%64)", d->rows, d->top, d->experts, kMoeMaxExperts,
            d->n);
    const MoeScratch s(d->rows, d->top, d->experts, d->n, dtype);
    REQUIRE(d->scratch, NVH_E_NULL, "moe_experts: null pointer");
    REQUIRE(aligned16(d->scratch), NVH_E_ALIGN, "moe_experts: scratch must be 16-byte aligned");
    REQUIRE(d->scratch_bytes >= 4 * s.links, NVH_E_WORKSPACE, "moe_experts: scratch %zu B < required %zu B", d->scratch_bytes, 4 * s.links);
    int32_t* at = reinterpret_cast<int32_t*>(d->scratch);
    int32_t* const ids = at + s.ids;
    const int pairs = d->rows * d->top;
    nvh_moe_route_desc route{};
    route.x = d->x; route.x_stride = d->x_stride; route.router = d->router; route.correction = d->correction;
    route.rows = d->rows; route.cols = d->cols; route.experts = d->experts; route.top = d->top; route.groups = d->groups; route.keep = d->keep;
    route.scale = d->scale; route.ids = ids; route.weights = d->weights; route.softmax = d->softmax;
    int rc = nvh_moe_route(&route, dtype, stream);
    if (rc) return rc;
    nvh_moe_gemm_desc g{};
    g.out = at; g.x = d->x; g.x_stride = d->x_stride; g.w = d->gate_up;
    g.pairs = pairs; g.top = d->top; g.experts = d->experts; g.n = d->n; g.k = d->cols; g.glu = 1; g.limit = d->limit; g.alpha = d->alpha;
    g.ids = ids;
    const bool both = experts_in_one(d, s);
    uint32_t* const links = reinterpret_cast<uint32_t*>(at + s.links);
    if (s.rows) {
        rc = launch_moe_dispatch(at + s.slots, at + s.tiles, at + s.counts, ids, pairs, d->experts, s.rows, s.max_tiles, both ? links : nullptr, both ? s.link_words : 0, (hipStream_t)stream);
        if (rc) return rc;
        g.slot_pair = at + s.slots; g.tiles = at + s.tiles; g.tile_rows = s.rows;
        g.max_tiles = s.max_tiles - d->experts + (d->experts < pairs ? d->experts : pairs);
    }
    nvh_moe_gemm_desc down = g;
    down.out = d->out; down.x = at; down.w = d->down; down.n = d->cols; down.k = d->n; down.glu = 0; down.limit = down.alpha = 0.f;
    if (both) {
        if ((rc = moe_gemm_ok(&g, dtype)) || (rc = moe_gemm_ok(&down, dtype))) return rc;
        return launch_moe_both(g, down, links, wait_limit, missing, (hipStream_t)stream);
    }
    rc = nvh_moe_gemm(&g, dtype, stream);
    return rc ? rc : nvh_moe_gemm(&down, dtype, stream);
}

int nvh_moe_experts(const nvh_moe_experts_desc* d, int dtype, void* stream) { return moe_experts(d, dtype, 0, 0, stream); }

int nvh_moe_experts_variant(uint32_t wait_limit, uint32_t missing, const nvh_moe_experts_desc* d, int dtype, void* stream) { return moe_experts(d, dtype, wait_limit, missing, stream); }

int nvh_moe_experts_status(const nvh_moe_experts_desc* d, int dtype, uint32_t* ran_out) {
    REQUIRE(ran_out, NVH_E_NULL, "moe_experts_status: null pointer");
    *ran_out = 0;
    const int one = nvh_moe_experts_one_launch(d, dtype);
    if (one <= 0) return one;
    const MoeScratch s(d->rows, d->top, d->experts, d->n, dtype);
    hipError_t e = hipDeviceSynchronize();
    if (e == hipSuccess) e = hipMemcpy(ran_out, moe_ran_out(reinterpret_cast<const uint32_t*>(d->scratch) + s.links), sizeof(uint32_t), hipMemcpyDeviceToHost);
    REQUIRE(e == hipSuccess, (int)e, "moe_experts_status: %s", hipGetErrorString(e));
    return 0;
}

}  // extern "C"
