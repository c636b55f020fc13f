/* Prefill-shaped EXACT_F32 requests over keys and values split into 16-bit parts beforehand: the plan of a
 * request, the bytes it wants attached, and its launches.
 *
 * One launch splits the visible key and value rows (kernels/gqa_f32_halve_rows.h), the second walks them
 * with the query heads of a kv head packed into the rows of its tiles and, where the launch would leave
 * units idle, in runs of keys (the plan of the bf16 prefill, rocm_prefill.c, with steps of 32 keys), and
 * a third merges the runs.  Parts and partials live in the attached workspace; without one
 * that holds them a request runs in one launch with fp32 products (kernels/gqa_f32_walk.h).
 * Everything here is a function of the request's geometry only, so that the planner's
 * workspace_required and the execution agree. */
#include "rocm_state.h"

#include <math.h>
#include <string.h>

enum {
    HALVED_STEP_KEYS = 32,
    HALVED_KEYS_MIN = 64,
    HALVED_GROUP_MAX = 16 /* query heads packed into the rows of a tile */
};
/* Bytes of parts a request may ask for: a quarter more than the F32 rows that they are made from.  The offsets of a
 * kv head's tiles are 32-bit ones; 2 GiB, 209715 keys of 8 kv heads of 128, keeps them below 2^31.  A request past it
 * runs in one launch, which takes 6 (300 tokens behind 60000: 8.5 ms, with the workspace 1.4) to 17 times
 * as long (64 tokens: 8.4 ms, 0.50). */
#define HALVED_TILES_MAX (2ull << 30)

typedef struct {
    yvex_rocm_walk_plan walk;
    unsigned long long kv_tiles, tile_bytes; /* of all kv heads */
    unsigned long long total;
} halved_plan;

static unsigned long long visible_keys(const yvex_transformer_attention_requirement *r)
{
    return r->mask == YVEX_TRANSFORMER_ATTENTION_MASK_CAUSAL ? r->query_start + r->query_tokens
                                                             : r->key_value_tokens;
}

/* Returns 0 when the request is not for these kernels.  Walks of fewer than 64 keys stay with the one launch: the
 * launch that splits, and a workgroup's longer start, cost more than they save.  With the workspace / without,
 * us: 40/8 heads of 128, 32 tokens 13.2 / 10.9, 64 15.1 / 16.1, 32 behind 32 14.8 / 15.5, 100 17.7 / 25.7, 200 22.3 /
 * 39.4, 330 28.8 / 58.0, 1777 142 / 310, 4096 596 / 1418, 32 behind 200 23.1 / 42.7, 32 behind 4000 42 / 573, 300
 * behind 5000 146 / 764; 16/4 of 64, 32 9.1 / 7.4, 64 10.4 / 10.3, 32 behind 32 10.2 / 9.9, 32 behind 64 11.1 / 12.4,
 * 200 13.9 / 23.3, 1000 37.0 / 88.3; 24/4 of 256, 32 22.0 / 16.4, 64 25.3 / 25.9, 32 behind 32 25.2 / 25.1, 32 behind
 * 64 28.0 / 33.6, 200 38 / 69, 1000 120 / 289, 64 behind 20000 206 / 5288. */
static int halved_plan_make(const yvex_transformer_attention_requirement *r, halved_plan *plan)
{
    const unsigned long long d = r->head_dimension, group = r->query_heads / r->key_value_heads;
    memset(plan, 0, sizeof(*plan));
    /* token_of (prefill_rows.h) is exact for row counts below 2^27 and at most 16 heads to a kv head (with 71 it is
     * first wrong at token 975685, with 127 at 304672); 32-bit offsets into a tile and into the tiles of a kv head */
    if (group > HALVED_GROUP_MAX || r->query_tokens > (1ull << 27) / group || r->query_heads > 65535ull ||
        r->key_value_tokens > (1ull << 30) || ((r->key_token_stride | r->value_token_stride) >> 24) != 0ull ||
        (r->key_value_heads * d >> 24) != 0ull)
        return 0;
    if (visible_keys(r) < HALVED_KEYS_MIN) return 0;
    plan->kv_tiles = (visible_keys(r) + HALVED_STEP_KEYS - 1ull) / HALVED_STEP_KEYS;
    plan->tile_bytes = r->key_value_heads * plan->kv_tiles * 320ull * d;
    if (plan->tile_bytes > HALVED_TILES_MAX) return 0;
    yvex_rocm_walk_plan_whole(r, group, HALVED_STEP_KEYS, &plan->walk);
    if (plan->walk.whole_items > 0x7fffffffull) return 0;
    yvex_rocm_walk_plan_cut(r, &plan->walk);
    plan->total = plan->tile_bytes + plan->walk.acc_bytes + plan->walk.ml_bytes;
    return 1;
}

unsigned long long yvex_rocm_halved_workspace(const yvex_transformer_attention_requirement *r)
{
    halved_plan plan;
    return halved_plan_make(r, &plan) ? plan.total : 0ull;
}

static yvex_rocm_function_id by_head_dimension(unsigned long long d, yvex_rocm_function_id at_64)
{
    return d == 64ull ? at_64 : (yvex_rocm_function_id)(at_64 + (d == 128ull ? 1 : 2));
}

int yvex_rocm_halved_launch(yvex_backend *backend, const yvex_transformer_attention_request *request,
                            const yvex_rocm_gqa_f32_params *f, yvex_backend_operation_facts *facts, int *taken,
                            yvex_error *err)
{
    static const char where[] = "rocm.transformer.gqa";
    const yvex_backend_operation_variant variant = YVEX_BACKEND_VARIANT_ROCM_ATTENTION_GQA_F32;
    const yvex_transformer_attention_requirement *r = &request->requirement;
    const yvex_rocm_backend_state *state = yvex_rocm_state(backend);
    yvex_rocm_gqa_f32_halved_params params;
    yvex_rocm_prefill_params *w = &params.walk;
    unsigned long long work = 0ull;
    halved_plan plan;
    int rc;
    *taken = 0;
    if (!halved_plan_make(r, &plan) ||
        yvex_backend_workspace_acquire(backend, plan.total, 256ull, &work) != YVEX_BACKEND_RESIDENT_HIT)
        return YVEX_OK;
    *taken = 1;
    memset(&params, 0, sizeof(params));
    w->q = (const uint16_t *)(const void *)f->q;
    w->k = (const uint16_t *)(const void *)f->k;
    w->v = (const uint16_t *)(const void *)f->v;
    w->out = (uint16_t *)(void *)f->out;
    w->lse = f->lse;
    w->status = f->status;
    w->q_stride = f->q_stride;
    w->k_stride = f->k_stride;
    w->v_stride = f->v_stride;
    w->query_tokens = (uint32_t)f->query_tokens;
    w->kv_tokens = (uint32_t)f->kv_tokens;
    w->query_start = (uint32_t)f->query_start;
    w->query_heads = (uint32_t)f->query_heads;
    w->kv_heads = (uint32_t)f->kv_heads;
    w->pack = (uint32_t)plan.walk.pack;
    w->row_heads = (uint32_t)plan.walk.row_heads;
    w->pack_inverse = (uint32_t)((0xffffffffull + plan.walk.pack) / plan.walk.pack);
    w->causal = (uint32_t)f->causal;
    w->rows = (uint32_t)plan.walk.rows;
    w->query_tiles = (uint32_t)plan.walk.query_tiles;
    w->whole_items = (uint32_t)plan.walk.whole_items;
    w->tail_items = (uint32_t)plan.walk.tail_items;
    w->splits = (uint32_t)plan.walk.splits;
    w->merge_groups = plan.walk.splits > 8ull ? 4u : 1u;
    params.tiles = (unsigned char *)(uintptr_t)work;
    w->part_acc = (float *)(uintptr_t)(work + plan.tile_bytes);
    w->part_ml = (float *)(uintptr_t)(work + plan.tile_bytes + plan.walk.acc_bytes);
    params.scale = f->scale;
    params.kv_tiles = (uint32_t)plan.kv_tiles;
    /* two workgroups of a unit: the second tier of items in reverse, equal sums for causal walks */
    if (f->causal && r->head_dimension != 256ull && state->compute_units > 0 &&
        plan.walk.whole_items >= 2ull * (unsigned long long)state->compute_units)
        params.pair_units = (uint32_t)state->compute_units;
    rc = yvex_rocm_launch(backend, by_head_dimension(r->head_dimension, YVEX_ROCM_FN_GQA_F32_HALVE_64), variant,
                          (unsigned int)plan.kv_tiles, (unsigned int)r->key_value_heads, 1u, 256u, 0u, &params,
                          where, err);
    if (rc == YVEX_OK)
        rc = yvex_rocm_launch(backend, by_head_dimension(r->head_dimension, YVEX_ROCM_FN_GQA_F32_HALVED_64), variant,
                              (unsigned int)(plan.walk.whole_items + plan.walk.tail_items * plan.walk.splits), 1u,
                              1u, 256u, 0u, &params, where, err);
    if (rc == YVEX_OK && plan.walk.splits > 1ull)
        rc = yvex_rocm_launch(backend, by_head_dimension(r->head_dimension, YVEX_ROCM_FN_GQA_F32_MERGE_64), variant,
                              (unsigned int)(plan.walk.tail_items * YVEX_ROCM_PREFILL_ROWS * r->head_dimension *
                                             w->merge_groups / 1024ull),
                              1u, 1u, 256u, 0u, &params, where, err);
    if (rc == YVEX_OK) {
        facts->kernel_launches = plan.walk.splits > 1ull ? 3ull : 2ull;
        facts->temporary_bytes = plan.total;
    }
    return rc;
}
