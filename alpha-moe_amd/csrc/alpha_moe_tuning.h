/*
 * Internal hook of libalpha_moe_hip.so for experiments and tests; not part of the operator's C ABI
 * (include/alpha_moe_hip.h) and free to change between versions.
 *
 * alpha_moe_set_tunable installs (set != 0) or clears (set == 0) a tuning override.  `name` is one of
 * ALPHA_MOE_PATH (1 direct, 2 stream, 3 or 4 group, 5 small, each where it takes the call), ALPHA_MOE_STRICT_QUEUE, ALPHA_MOE_KBPI, ALPHA_MOE_TPI,
 * ALPHA_MOE_LAG, ALPHA_MOE_GRID, ALPHA_MOE_TILE_GPS, ALPHA_MOE_TILE_NT, ALPHA_MOE_GROUP_PIECES; ALPHA_MOE_TILE_LAG,
 * ALPHA_MOE_TILE_GRID and ALPHA_MOE_WIDE_PP belonged to kernels that are gone: accepted, without effect.
 * The environment variables of the same names are read once, when the library is first used; no launch reads the
 * environment.  Not thread-safe against concurrent launches.  Results stay within the parity bar whatever is set.
 * Returns ALPHA_MOE_ERR_SHAPE for an unknown name.
 *
 * alpha_moe_group_plan tells how the group kernel would serve a call: plan = {tiles of 16 rows its variant takes in a row block,
 * 64-column groups of a down-projection item, items' column slabs, w2 block scales an item's table holds}.  Returns
 * ALPHA_MOE_ERR_SHAPE for a call that another kernel serves.  Host only.
 */
#ifndef ALPHA_MOE_TUNING_H
#define ALPHA_MOE_TUNING_H
#ifdef __cplusplus
extern "C" {
#endif
int alpha_moe_set_tunable(const char *name, int value, int set);
int alpha_moe_group_plan(int top_k, int M, int K, int N, int num_experts, int sorted_num, int block_m, int stages, int plan[4]);
#ifdef __cplusplus
}
#endif
#endif
