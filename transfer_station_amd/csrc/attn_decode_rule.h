/* attn_decode_rule.h -- how many 16-row blocks of a kv head one decode workgroup serves: the host
 * layer sizes the key split with it, the launcher takes the kernel by it. */
#ifndef ATTN_DECODE_RULE_H
#define ATTN_DECODE_RULE_H

#define ATTN_DECODE_TARGET_WG 512
#define ATTN_DECODE_MIN_KEYS 128 /* keys per split: one 32-key tile per wave, 4 waves */

/* Two, where a kv head has three or four blocks, the head dim leaves registers for two (D <= 128) and
 * the grid of one block per workgroup has its full number of workgroups: K and V are then read half
 * as often (64 rows over 4001 keys, 32 kv heads 28.6 -> 23.2 us). Grids that the key count keeps
 * smaller lose by halving (16 heads x 3 rows over 500 keys 8.2 -> 8.45 us). */
static inline int attn_decode_blocks(int nrb, int dp, int Hkv, int Sk) {
    const long by_len = ((long)Sk + ATTN_DECODE_MIN_KEYS - 1) / ATTN_DECODE_MIN_KEYS;
    return nrb > 2 && dp <= 128 && (long)Hkv * nrb * by_len >= ATTN_DECODE_TARGET_WG ? 2 : 1;
}

#endif
