// Which kernel, tile or split a call takes, from its sizes and form alone: host code without the GPU
// runtime, so that the lines can be tested on any machine. cus: compute units of the device.
#pragma once

#include <stdint.h>

namespace tsfm {
namespace rules {

// Whether f32 attention whose rows fit the kernel with resident keys (attn_f32.hip) runs faster on the bf16x3
// kernel (attn_x3.hip). Launch times in us, resident / bf16x3, at 12 heads; "rows" are (series, head) pairs.
// A row of 32k + 1 queries (lone) costs the bf16x3 kernel a pass of its own for the last one.
struct AttnForm {
    int64_t rows;
    int n_q, n_k;
    bool causal;     // CAUSAL, CAUSAL_KEYS
    bool decoder;    // DECODER
    bool keys_hard;  // FULL_KEYS: invalid keys at -inf, so every chunk with one goes through the mask rule
    bool keys_soft;  // KEYS_ADDITIVE (neither of the four: FULL)
    bool dense;      // a dense bias, read per score in either kernel
    bool rel;        // the T5 table
    bool rope;
};
inline bool attn_x3_pays(const AttnForm& f, int64_t cus) {
    const bool lone = f.n_q % 32 == 1;
    // The causal masks: the resident kernel skips half its tiles. Past two rows per CU and 96 queries the
    // bf16x3 kernel wins (516 rows of 96 queries: 29.4 / 20.9).
    const bool many = f.rows >= 2 * cus && f.n_q >= 96;
    if (f.causal) return many;
    if (f.rows <= cus) {
        // One row per CU or fewer: the resident kernel's nine waves of 16 queries finish a row sooner up to 64
        // queries (12 rows with RoPE, key-masked: 64: 8.4 / 8.6, 66: 11.2 / 10.3, 109: 14.8 / 12.9), and
        // without RoPE, where it stages by DMA, up to 68 (plain 66: 9.3 / 9.7, 69: 10.4 / 10.0; T5 66: 9.4 /
        // 10.1 with all keys valid). Scores that need work of their own there cost the bf16x3 kernel more:
        // a dense bias (128: 16.3 / 19.5, 252 rows of 144: 25.4 / 34.8), hard key masks (80 with RoPE:
        // 11.8 / 14.0, plain 66: 9.4 / 12.1; from 130 on it wins while two workgroups a row fit the
        // CUs, 144: 22.6 / 19.8) and decoder rows with RoPE (72 over 144: 1.04).
        if (lone || f.dense || (f.decoder && f.rope)) return false;
        if (f.keys_hard) return !f.rel && f.n_q > 128 && 2 * f.rows <= cus;
        return f.n_q > (f.rope ? 64 : 68);
    }
    // More rows than CUs: the resident kernel holds one per CU and takes them in rounds; the bf16x3 kernel has
    // three workgroups a CU in flight (264 rows, key-masked with RoPE: 37: 12.6 / 10.9, 109: 27.8 / 19.5; decoder
    // rows of 32 queries over 94 keys: 16.0 / 10.8). Not for a handful of queries (one over 129 keys: 11.6 /
    // 13.1), nor 33 and 65 (11.8 / 12.8, 16.8 / 18.4).
    if (f.n_q < 8) return false;
    const bool heavy = f.dense || f.keys_hard || (f.decoder && f.rope);
    if (lone) return f.n_q > 65 && (many || !heavy);
    // Just under a whole number of rows per CU the resident kernel's last round is full: heavy scores lose there
    // (504 rows of 144, dense: 1.30, hard masks 1.1-1.23; of 72, hard masks: 1.08), except from 96 to 128
    // queries.
    const bool slack = f.rows % cus <= cus * 3 / 4;
    if (f.keys_hard) {
        // 8-16: 6.5 / 7.4, 17-32: 0.82-1.0, 33-64: 10.7 / 11.7 at 264 rows and 1.25 at 768.
        if (f.n_q <= 16 || (f.n_q > 32 && f.n_q <= 64)) return false;
        if (f.n_q >= 96 && f.dense) return many;
        return slack || (f.n_q >= 96 && f.n_q <= 128) || many;
    }
    if (f.dense) return slack || f.n_q <= 128 || many;
    if (!f.rope && !f.decoder && f.rows < 2 * cus && f.n_k <= 64) {
        // Short rows by DMA: 34 queries (1.06; with all keys valid 1.13, and up to 48 1.0-1.04), and, without
        // the T5 table either, up to 16 (6.3 / 6.6, 6.4 / 7.0).
        if (f.n_q > 32 && f.n_q <= (f.keys_soft || f.rel ? 34 : 48)) return false;
        if (!f.rel && f.n_q <= 16 && f.n_k <= 16) return false;
    }
    return true;
}

// Tiles of 128 x 128 from which a product runs on them (BIG), and on 64 x 64 ones (SMALL, a quarter of the
// work) below. BIG tiles pay from where the SMALL ones would start another round, not from a tile for every
// CU. Launch times in us, SMALL / BIG, at 256 CUs:
//  - Split inside the product: three SMALL workgroups a CU, one BIG: past 192 tiles (768 indices: 180 tiles 41.5 /
//    41.8, 198 56.1 / 42.5, 216 56.1 / 43.8).
//  - Pre-split operands: two SMALL workgroups a CU, so past 128, with room for the sharing that SMALL tiles lose
//    late (1024 indices, 2048 columns: 162 tiles of 768 indices 49.6 / 46.3; Chronos-2 layers of 4820 rows 1505 /
//    1432). Short reductions keep SMALL ones up to a round of the others (512 indices, 162 tiles 37.6 / 38.5,
//    192 38.2 / 39.5, 216 43.1 / 39.9).
//  - The f32 instruction (reductions not of whole 32s): four SMALL workgroups a CU, two BIG, so a round of SMALL
//    ones lasts to 256 tiles; from 512 indices on BIG ones read their operands less often (528: 204 tiles
//    45.4 / 42.9, 1040: 216 82.8 / 76.6; 176: 19.6 / 19.7, with RoPE 20.7 / 21.5; 48: 9.9 / 11.0).
inline int64_t big_tiles_min(int64_t d_in, bool presplit, int64_t cus) {
    const int64_t thin = cus * 25 / 32, round = cus;  // 200 and 256 tiles
    if (d_in % 32 != 0) return d_in >= 512 ? thin : round;
    return presplit && d_in >= 768 ? cus * 5 / 8 : thin;  // (160 tiles)
}

// How many workgroups share a tile's reduction of `steps` 16-wide steps, and how many steps each takes, for a
// product of `blocks` tiles of 64 x 64. pairs: shares of an even number of steps (32-wide ones).
//
// Each share costs its start, its partial sums' trip through memory and the longer sum afterwards (half of an
// 18 us launch of 576 workgroups), so a product is shared out only while the CUs have fewer than about one and
// a half workgroups each: aiming at 360 / 420 / 470 / 512 workgroups, Chronos-2 layers of 545 rows take 434 /
// 432 / 454 / 466 us, the Chronos-Bolt-small forecast 971 / 936 / 940 / 948, Chronos-Bolt-base layers of 528
// rows 467 / 464 / 490 / 492. Where 512 deals the CUs their workgroups evenly and 420 does not (32 or 64 tiles:
// 16 or 8 shares against 13 or 7), the fullest CU has less to do with 512: four outputs of 2048 indices, 1024
// columns each, 33 rows 18.8 / 17.1 us; 4096 indices, 512 columns, 8 rows 18.3 / 17.1.
struct Split {
    int shares, steps;  // shares: 1 = unsplit
};
constexpr int64_t kSplitBlocks = 420;  // tiles from which the reduction is never shared out
inline Split split_aiming_at(int64_t workgroups, int64_t blocks, int steps, bool pairs) {
    const Split whole = {1, steps};
    if (steps < 16) return whole;
    int64_t s = (workgroups + blocks - 1) / blocks;
    if (s > steps / 8) s = steps / 8;
    if (s > 16) s = 16;
    if (s < 2) return whole;
    int per = (int)((steps + s - 1) / s);
    if (pairs) per += per & 1;
    s = (steps + per - 1) / per;
    return s < 2 ? whole : Split{(int)s, per};
}
// device_cus: asked only where the two differ (it takes 0.3 us of the host).
template <class Cus>
inline Split reduction_split(int64_t blocks, int steps, bool pairs, Cus&& device_cus) {
    if (blocks <= 0 || blocks >= kSplitBlocks) return {1, steps};
    const Split a = split_aiming_at(kSplitBlocks, blocks, steps, pairs), b = split_aiming_at(512, blocks, steps, pairs);
    if (a.shares == b.shares) return a;
    const int64_t cus = device_cus();
    // Steps the fullest CU walks.
    auto longest = [&](const Split& s) { return (s.shares * blocks + cus - 1) / cus * s.steps; };
    return cus > 0 && longest(b) < longest(a) ? b : a;
}

// Whether a product runs on pre-split operands when a workspace is lent, instead of splitting inside. Splitting
// the weights costs the same at any row count and saves each row tile its own split, so it pays by rows and by
// the work of the product. Pre-split / split inside, over some 1300 products of 64 to 2600 rows and 512 to 4096
// indices (whole calls in us: Chronos-2 layers of 484 rows 500 / 457, 1205 rows 675 / 634, 4820 rows 1513 /
// 1707; Timestral q/k/v/gate, 4096 columns: 999 rows 62 / 57, 1332 rows 87 / 93):
//  - From 2048 rows or 5 2^30 multiply-adds on: 0.83-1.0 (reductions of 512 up to 1.3).
//  - With less work, a product that shares its reduction out loses (200 rows of 4096 indices, 1536 columns: 1.19).
//    One that cannot (whole: RoPE, half-precision outputs; or tiles enough without) walks all of it in each
//    tile, and its own split with it. There pre-split wins for long reductions at any size (4096 indices, 1536
//    columns: 200 rows 81 / 97, 768 rows 99 / 124; 1536 from 1.5 2^30 on: 900 rows 0.92), for others at 4.5
//    2^30, at 1200 rows and more 3.75 2^30 (1024 indices, 3072 columns: 1205 rows 1.02, 1332 0.95, 1500 80 /
//    84). Not for more than 4096 columns, whose weights take longer to split (2048 indices, 6144 columns: 128
//    rows 1.13), nor where its tiles, two a CU, start a second round that three a CU do not (1500 rows of
//    1536 indices, 1536 columns: 77 / 69).
// whole: the product's form keeps it from sharing its reduction out.
inline bool planes_pay(int64_t tokens, int64_t d_in, int64_t n_cols, bool whole, int64_t cus) {
    const int64_t macs = tokens * n_cols * d_in, quarter = (int64_t)1 << 28;  // (quarters of 2^30)
    if (d_in % 32 != 0 || macs < 4 * quarter) return false;
    if (tokens >= 2048 || macs >= 20 * quarter) return true;
    const int64_t blocks = (tokens + 63) / 64 * ((n_cols + 63) / 64);
    if ((!whole && blocks < kSplitBlocks) || n_cols > 4096) return false;
    if (blocks > 2 * cus && blocks < 4 * big_tiles_min(d_in, true, cus)) return false;
    if (d_in >= 2048 || (d_in >= 1536 && macs >= 6 * quarter)) return true;
    return macs >= (tokens < 1200 ? 18 : 15) * quarter;
}

// Whether a Timestral forecast splits its layers' weights once for all its decode blocks (a copy of 1.5x the
// weights) instead of once per block and product. Only blocks of at least kKeptBlock tokens read the copy: shorter
// ones split inside their products, whose reductions are shared out over more workgroups. It takes two such
// blocks, of kKeptTokens together, to repay it. Whole forecasts, with the copy / without, four layers of 1024, by
// the tokens of their blocks: 1520 and 752: 1.02, 1008, 512, 512 and 288: 1.02, 504 and 188: 1.10; three of
// 768 and 432: 1.00; 1140, 768, 768 and 432: 0.98, 1900 and 940: 0.99, three of 1024 and 576: 0.97, 3024 and
// 1128: 0.97.
constexpr int64_t kKeptBlock = 768, kKeptTokens = 2048;
struct KeptWeights {
    int blocks = 0;
    int64_t tokens = 0;
    void add(int64_t block_tokens) {
        if (block_tokens < kKeptBlock) return;
        blocks++;
        tokens += block_tokens;
    }
    bool pay() const { return blocks >= 2 && tokens >= kKeptTokens; }
};

}  // namespace rules
}  // namespace tsfm
