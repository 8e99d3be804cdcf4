/* attn_decode_rule.h -- how a decode call is cut: 16-row blocks of a kv head per workgroup, parts of
 * the key range and keys per part. The host layer sizes the launch with it, the launcher takes the
 * kernel by it. */
#ifndef ATTN_DECODE_RULE_H
#define ATTN_DECODE_RULE_H

#define ATTN_SLOTS 65536 /* split-K partial slots of a scratch, one per (query row, part) */
#define ATTN_DECODE_TARGET_WG 512
#define ATTN_DECODE_MIN_KEYS 128 /* keys per part: one 32-key tile per wave, 4 waves */

struct attn_decode_cut {
    int blocks, nsplit, kps; /* row blocks per workgroup, parts, keys per part */
};

/* The cut with `blocks` row blocks per workgroup: one workgroup per (kv head, part, group of
 * blocks), parts up to the target grid, no more than the key count and the slots allow. */
static inline struct attn_decode_cut attn_decode_cut_for(int Hq, int Hkv, int Sq, int Sk, int nrb,
                                                         int blocks) {
    const long rows = (long)Hq * Sq;
    const long cap = ATTN_SLOTS / (rows > 0 ? rows : 1);
    const long wgs = (long)Hkv * ((nrb + blocks - 1) / blocks);
    const long by_len = ((long)Sk + ATTN_DECODE_MIN_KEYS - 1) / ATTN_DECODE_MIN_KEYS;
    long ns = (ATTN_DECODE_TARGET_WG + wgs - 1) / wgs;
    /* Grouped blocks: no more than the 64 parts that one merge wave covers. */
    if (blocks > 1 && ns > 64)
        ns = 64;
    if (ns > by_len)
        ns = by_len;
    if (ns > cap)
        ns = cap;
    if (ns < 2)
        ns = 1;
    /* keys per part: a multiple of 128 covering Sk in ns pieces */
    long kps = ((long)Sk + ns - 1) / ns;
    kps = (kps + ATTN_DECODE_MIN_KEYS - 1) / ATTN_DECODE_MIN_KEYS * ATTN_DECODE_MIN_KEYS;
    struct attn_decode_cut c = {blocks, (int)(((long)Sk + kps - 1) / kps), (int)kps};
    return c;
}

/* Two blocks per workgroup read K and V half as often. They are taken where a kv head has three or
 * four blocks, the head dim leaves registers for two (D <= 128), and the grid they are launched with
 * still has a workgroup per CU (256 of them) with at least 96 KB of K and V each, or 256 KB where one
 * block per workgroup would need no parts and no merge. Measured over 33 to 64 rows, 1 to 200 kv
 * heads, 500 to 65536 keys, D = 64, 100 and 128, one block -> two, us at D = 128 unless said:
 *   32 kv heads x 64 rows over 4001 keys 32.7 -> 26.4, 128 kv heads x 2000 at D = 64 26.8 -> 21.9;
 *   2 kv heads x 64 rows over 32768 keys (256 workgroups) 19.0 -> 18.0;
 * and where the rule keeps one:
 *   1 kv head x 64 rows over 65536 keys at D = 64 (128 workgroups) 14.7 -> 18.3;
 *   64 kv heads x 64 rows over 500 keys (one 128-key step each) 13.7 -> 17.7;
 *   200 kv heads x 48 rows over 500 keys at D = 64 (no parts with one block) 11.1 -> 16.1. */
static inline struct attn_decode_cut attn_decode_cut_of(int Hq, int Hkv, int Sq, int Sk, int nrb,
                                                        int dp) {
    if (nrb > 2 && dp <= 128) {
        const struct attn_decode_cut two = attn_decode_cut_for(Hq, Hkv, Sq, Sk, nrb, 2);
        const long grid = (long)Hkv * ((nrb + 1) / 2) * two.nsplit;
        const long kb = (long)two.kps * dp * 4 / 1024; /* of K and V per workgroup */
        if (2 * grid >= ATTN_DECODE_TARGET_WG &&
            kb >= ((long)Hkv * nrb < ATTN_DECODE_TARGET_WG ? 96 : 256))
            return two;
    }
    return attn_decode_cut_for(Hq, Hkv, Sq, Sk, nrb, 1);
}

#endif
