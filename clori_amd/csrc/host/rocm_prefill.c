/* Multi-token bf16 attention of the ROCm arm: how the work of a launch is cut, and the launch.
 *
 * The query heads of a kv head are packed into the rows of its query tiles (kernel_params.h), so
 * the number of items is kv_heads * ceil(query_tokens * group / 128), and an item walks the keys
 * its last token sees in steps of 64.  (A single query token is not packed and not cut: one item
 * per query head.)  Up to a multiple of the compute units the items are walked
 * whole, one workgroup each, the longest first; when what is left over would keep a fraction of
 * the units busy for long, its walks are cut into runs of keys, one workgroup each, and a second
 * launch merges the runs.  Nine tokens of 40/8 heads of 128 behind 12001: one tile per query head
 * walked 188 steps on 40 units, 160 us; packed and cut into 256 runs, 17.4 us. 2000 tokens of 24/4
 * heads of 256 behind 13333: 376 items took two turns of 256 units with half of the second empty,
 * 1182 us; with its tail cut, 873 (both with one wave per 32 rows; prefill_pair.hip has 634).  A
 * prompt of 2048 tokens without a history is not cut and gains from the packing only that a tile
 * spans 26 tokens instead of 128 (50.6 -> 50.2 us).  Walks that are not cut and all start at once are
 * packed only where that does not put them into fewer workgroups: packed / one query head to a tile,
 * us, 40 tokens of 40/8 heads of 128 7.5 / 6.5, 300 11.4 / 10.7, 20 behind 200 9.7 / 8.9, 21 of 24/4 of
 * 256 11.6 / 9.7; with as many workgroups either way 500 behind 500 of 16/4 of 64 15.9 / 16.1.
 * The cut is a function of the request's geometry only (256 units, never the device), so that the
 * planner's workspace_required and the execution agree. */
#include "rocm_state.h"

#include <math.h>
#include <string.h>

enum {
    PREFILL_UNITS = 256,
    PREFILL_SPLITS_MAX = 64,
    PREFILL_RUN_STEPS_MIN = 2,
    /* Bytes of partial rows a request may ask for.  Runs past it are many runs of many items, whose
     * predicted gain is small and whose partials cost more than predicted (24/4 heads of 256, before
     * with 32, 16 and 7 runs / now: 1316 tokens behind 803329 21.8 / 20.9 ms, 2631 behind 342689 18.4 /
     * 18.1, 736 behind 25193 476 / 461 us; 686 behind 346068, 23 runs in 401 MB, 5.2 / 5.6 ms).  A
     * threshold on the predicted gain would be wrong: 17 tokens of 16/4 heads of 64 behind 867 are to
     * gain 1.4 % and take 8.9 us instead of 13.1. */
    PREFILL_PARTIALS_MAX = 96 << 20
};

/* Steps of an item of query tile `q_tile`. */
static unsigned long long item_steps(const yvex_transformer_attention_requirement *r,
                                     const yvex_rocm_walk_plan *plan, unsigned long long q_tile)
{
    unsigned long long last = (q_tile + 1ull) * YVEX_ROCM_PREFILL_ROWS, keys = r->key_value_tokens;
    if (last > plan->rows) last = plan->rows;
    if (r->mask == YVEX_TRANSFORMER_ATTENTION_MASK_CAUSAL) keys = r->query_start + (last - 1ull) / plan->pack + 1ull;
    return (keys + plan->step_keys - 1ull) / plan->step_keys;
}

/* What the tail costs in nanoseconds when each of its walks is cut into `splits` runs: every unit
 * takes its share of the runs one after the other, each with the start and end of a workgroup;
 * a cut tail also writes its partials, reads them back and pays a launch. */
static unsigned long long tail_cost(const yvex_transformer_attention_requirement *r, const yvex_rocm_walk_plan *plan,
                                    unsigned long long steps, unsigned long long splits)
{
    /* 0.9 us for a 128-row step of 64 keys at 128 in bf16; walks over F32 parts (32 keys) are cut alike */
    const unsigned long long step_ns = 7ull * r->head_dimension;
    const unsigned long long turns = (plan->tail_items * splits + PREFILL_UNITS - 1ull) / PREFILL_UNITS;
    const unsigned long long live = plan->rows < YVEX_ROCM_PREFILL_ROWS ? plan->rows : YVEX_ROCM_PREFILL_ROWS;
    unsigned long long cost = turns * ((steps + splits - 1ull) / splits * step_ns + 3500ull);
    if (splits > 1ull) /* F32 rows written and read at about 4 TB/s, and the second launch */
        cost += 5000ull + plan->tail_items * splits * live * r->head_dimension * 8ull / 4000ull;
    return cost;
}

/* Every walk whole, `pack` query heads to a row head. */
void yvex_rocm_walk_plan_whole(const yvex_transformer_attention_requirement *r, unsigned long long pack,
                               unsigned long long step_keys, yvex_rocm_walk_plan *plan)
{
    memset(plan, 0, sizeof(*plan));
    plan->step_keys = step_keys;
    plan->pack = pack;
    plan->row_heads = r->query_heads / pack;
    plan->rows = r->query_tokens * pack;
    plan->query_tiles = (plan->rows + YVEX_ROCM_PREFILL_ROWS - 1ull) / YVEX_ROCM_PREFILL_ROWS;
    plan->whole_items = plan->query_tiles * plan->row_heads;
    plan->splits = 1ull;
}

/* Cuts the walks of the items past a multiple of the units where that is predicted to take less time. */
void yvex_rocm_walk_plan_cut(const yvex_transformer_attention_requirement *r, yvex_rocm_walk_plan *plan)
{
    const unsigned long long items = plan->whole_items;
    unsigned long long steps, splits, best, slots, run_bytes;
    if (items % PREFILL_UNITS == 0ull) return;
    plan->whole_items = items / PREFILL_UNITS * PREFILL_UNITS;
    plan->tail_items = items - plan->whole_items;
    steps = item_steps(r, plan, plan->query_tiles - 1ull - plan->whole_items / plan->row_heads);
    run_bytes = plan->tail_items * YVEX_ROCM_PREFILL_ROWS * r->head_dimension * sizeof(float);
    best = tail_cost(r, plan, steps, 1ull);
    for (splits = 2ull; splits <= PREFILL_SPLITS_MAX && splits * PREFILL_RUN_STEPS_MIN <= steps &&
                        splits * run_bytes <= PREFILL_PARTIALS_MAX; ++splits) {
        const unsigned long long cost = tail_cost(r, plan, steps, splits);
        if (cost < best) {
            best = cost;
            plan->splits = splits;
        }
    }
    if (plan->splits == 1ull) {
        plan->whole_items = items;
        plan->tail_items = 0ull;
        return;
    }
    slots = plan->tail_items * plan->splits * YVEX_ROCM_PREFILL_ROWS;
    plan->acc_bytes = slots * r->head_dimension * sizeof(float);
    plan->ml_bytes = slots * 2ull * sizeof(float);
}

/* Whole walks of so few steps, at head dimension 256, that the pairs of prefill_pair.hip cost more to
 * start and end than they save per step: up to seven steps, four where few tokens leave the other
 * kernel's waves without rows.  One wave per 32 rows / pairs, us, 24/4 heads: 128 tokens 15.0 / 19.2,
 * 256 19.7 / 22.7, 448 24.7 / 26.8, 513 (nine steps) 29.3 / 29.8, 700 36.5 / 33.6; 60 behind 150 18.1 /
 * 22.2, 120 behind 260 23.8 / 25.1, 128 behind 380 (eight) 28.5 / 28.0, 10 behind 200 17.4 / 17.1. */
static int walks_are_short(const yvex_transformer_attention_requirement *r, const yvex_rocm_walk_plan *plan)
{
    return item_steps(r, plan, plan->query_tiles - 1ull) <= (r->query_tokens >= 64ull ? 7ull : 4ull);
}

/* Returns 0 when the request is past the launch range: 65535 query heads or tiles of 128 tokens,
 * 2^31 - 1 (head, tile) pairs (so that rows stay below 2^27). */
static int prefill_plan_make(const yvex_transformer_attention_requirement *r, int may_split, yvex_rocm_walk_plan *plan)
{
    const unsigned long long token_tiles = (r->query_tokens + YVEX_ROCM_PREFILL_ROWS - 1ull) / YVEX_ROCM_PREFILL_ROWS;
    if (r->query_heads > 65535ull || token_tiles > 65535ull || r->query_heads * token_tiles > 0x7fffffffull) return 0;
    yvex_rocm_walk_plan_whole(r, r->query_tokens == 1ull ? 1ull : r->query_heads / r->key_value_heads, 64ull, plan);
    if (may_split && r->query_tokens > 1ull) yvex_rocm_walk_plan_cut(r, plan);
    if (plan->splits == 1ull && r->query_tokens > 1ull && r->query_heads * token_tiles <= PREFILL_UNITS) {
        const int short_walks = r->head_dimension == 256ull && walks_are_short(r, plan);
        /* Every walk has a unit of its own either way; one query head to a tile then means as many
         * steps in more workgroups of fewer live waves. */
        if ((r->head_dimension != 256ull || short_walks) && r->query_heads * token_tiles > plan->whole_items)
            yvex_rocm_walk_plan_whole(r, 1ull, 64ull, plan);
        plan->short_walks = short_walks;
    }
    return 1;
}

/* Bytes of the partials of a request (0: its walks are not cut, or the execution will refuse it). */
unsigned long long yvex_rocm_prefill_workspace(const yvex_transformer_attention_requirement *r)
{
    yvex_rocm_walk_plan plan;
    /* both multiples of the 1 KB that 128 rows take */
    return prefill_plan_make(r, 1, &plan) ? plan.acc_bytes + plan.ml_bytes : 0ull;
}

static yvex_rocm_function_id by_head_dimension(unsigned long long d, yvex_rocm_function_id at_64,
                                               yvex_rocm_function_id at_128, yvex_rocm_function_id at_256)
{
    return d == 64ull ? at_64 : d == 256ull ? at_256 : at_128;
}

int yvex_rocm_prefill_execute(yvex_backend *backend, const yvex_transformer_attention_request *request,
                              yvex_device_tensor *lse, const yvex_device_tensor *gate,
                              const yvex_rocm_attention_geometry *g, yvex_backend_operation_facts *facts,
                              yvex_error *err)
{
    static const char where[] = "rocm.transformer.gqa.prefill";
    const yvex_backend_operation_variant variant = YVEX_BACKEND_VARIANT_ROCM_ATTENTION_GQA_BF16;
    yvex_rocm_backend_state *state = yvex_rocm_state(backend);
    const yvex_transformer_attention_requirement *r = &request->requirement;
    unsigned long long work = 0ull;
    yvex_rocm_prefill_params params;
    yvex_rocm_walk_plan plan;
    int rc;
    /* the kernel addresses K and V through 32-bit buffer offsets */
    if (r->key_value_tokens * g->k_stride * 2ull >= 0xffffffffull ||
        r->key_value_tokens * g->v_stride * 2ull >= 0xffffffffull || !prefill_plan_make(r, 1, &plan)) {
        yvex_error_set(err, YVEX_ERR_BOUNDS, "rocm.transformer.attention",
                       "prefill geometry exceeds admitted launch range");
        return YVEX_ERR_BOUNDS;
    }
    backend_workspace_reset(backend);
    /* Without an attached workspace that holds the partials the walks stay whole: allocating and
     * freeing them around the call costs more than the cut saves, and waits for the stream. */
    if (plan.splits > 1ull &&
        yvex_backend_workspace_acquire(backend, plan.acc_bytes + plan.ml_bytes, 256ull, &work) !=
            YVEX_BACKEND_RESIDENT_HIT) {
        work = 0ull;
        (void)prefill_plan_make(r, 0, &plan);
    }
    memset(&params, 0, sizeof(params));
    params.q = (const uint16_t *)request->query->data;
    params.k = (const uint16_t *)request->key->data;
    params.v = (const uint16_t *)request->value->data;
    params.out = (uint16_t *)request->output->data;
    params.lse = lse ? (float *)lse->data : NULL;
    params.gate = gate ? (const uint16_t *)gate->data : NULL;
    params.status = state->device_status;
    params.q_stride = g->q_stride;
    params.k_stride = g->k_stride;
    params.v_stride = g->v_stride;
    params.query_tokens = (uint32_t)r->query_tokens;
    params.kv_tokens = (uint32_t)r->key_value_tokens;
    params.query_start = (uint32_t)r->query_start;
    params.query_heads = (uint32_t)r->query_heads;
    params.kv_heads = (uint32_t)r->key_value_heads;
    params.pack = (uint32_t)plan.pack;
    params.row_heads = (uint32_t)plan.row_heads;
    params.pack_inverse = (uint32_t)((0xffffffffull + plan.pack) / plan.pack);
    params.causal = (uint32_t)g->causal;
    params.rows = (uint32_t)plan.rows;
    params.query_tiles = (uint32_t)plan.query_tiles;
    params.scale_log2 = (1.0f / sqrtf((float)r->head_dimension)) * 1.4426950408889634f;
    params.whole_items = (uint32_t)plan.whole_items;
    params.tail_items = (uint32_t)plan.tail_items;
    params.splits = (uint32_t)plan.splits;
    /* one trip of the merge takes eight runs; more go to four groups of threads side by side */
    params.merge_groups = plan.splits > 8ull ? 4u : 1u;
    params.part_acc = (float *)(uintptr_t)work;
    params.part_ml = (float *)(uintptr_t)(work + plan.acc_bytes);
    rc = yvex_rocm_launch(backend,
                          by_head_dimension(r->head_dimension, YVEX_ROCM_FN_PREFILL_BF16_64, YVEX_ROCM_FN_PREFILL_BF16,
                                            plan.short_walks ? YVEX_ROCM_FN_PREFILL_BF16_256_SHORT
                                                             : YVEX_ROCM_FN_PREFILL_BF16_256),
                          variant, (unsigned int)(plan.whole_items + plan.tail_items * plan.splits), 1u, 1u, 256u,
                          0u, &params, where, err);
    if (rc == YVEX_OK && plan.splits > 1ull)
        rc = yvex_rocm_launch(backend,
                              by_head_dimension(r->head_dimension, YVEX_ROCM_FN_PREFILL_MERGE_64,
                                                YVEX_ROCM_FN_PREFILL_MERGE, YVEX_ROCM_FN_PREFILL_MERGE_256),
                              variant,
                              (unsigned int)(plan.tail_items * YVEX_ROCM_PREFILL_ROWS * r->head_dimension *
                                             params.merge_groups / 1024ull),
                              1u, 1u, 256u, 0u, &params, where, err);
    if (rc == YVEX_OK) {
        facts->kernel_launches = plan.splits > 1ull ? 2ull : 1ull;
        facts->accelerated_matrix_launches = 1ull;
        facts->temporary_bytes = plan.acc_bytes + plan.ml_bytes;
        facts->compulsory_memory_facts_available = 1;
        rc = yvex_rocm_complete(backend, variant, where, facts, err);
    }
    backend_workspace_reset(backend);
    return rc;
}
