// kxw4_route.hpp — which kernel a decode launch (at most 16 tokens) runs on:
// the strip kernel (kxw4_strip.hip), the row-wave kernel (kxw4_rowwave.hip)
// or the K-parallel kernel (kxw4_decode.hip); and, last, which packed prompts
// run on the general GEMM kernel (kxw4_gemm.hip). Plain C++, so that the rules
// can be checked without a GPU.
//
// Every kernel gives the same bits; the lines lie where the times cross. They
// were measured over 256-73,728 rows (W8: 262,144) of 1,024-17,408 columns
// and 1-16 tokens, launches of a graph replay over 620 MB of weights in turn,
// so that the weights come from HBM (figures: us a launch, MI355X, 256 CUs).
// A shape that the row-wave kernel has no LDS for goes on to the strip kernel.
#pragma once

namespace kxw4 {

enum DecodeRoute { kRouteStrip = 0, kRouteRowwave = 1, kRouteKParallel = 2 };

struct DecodeShape {
    int cus;                          // compute units of the device
    int rgs;                          // 16-row groups over all weights
    int T, K, group;
    int S;                            // split count of every token and weight, 0 if they differ
    bool blocks;                      // activation scales per K32 block, else per token
    bool w8;
};

// The K-parallel kernel's LDS words for slices of `tl` tokens: partials
// [nu][tl][16] int32, scales [g][16] uint16, split partials [smax][tl][16]
// float, in the general mode the activation scale and code sum [nu][tl], then
// 64 dummy words.
constexpr int decode_lds_words(int nu, int g, int tl, int smax, bool side) {
    return nu * tl * 16 + g * 8 + smax * tl * 16 + (side ? 2 * nu * tl : 0) + 64;
}

// Its tokens per slice: the most (at most 64) whose LDS fits in 64 KB, 0 if
// one token's does not.
inline int kparallel_slice(int nu, int g, int T, int smax, bool side) {
    int ts = T < 64 ? T : 64;
    while (ts > 1 && 4ll * decode_lds_words(nu, g, ts, smax, side) > 64 * 1024) ts = (ts + 1) / 2;
    return 4ll * decode_lds_words(nu, g, ts, smax, side) > 64 * 1024 ? 0 : ts;
}

// W8: a row-wave work-group takes 16 row-groups, so the rows are good for it
// where they fill the CUs and are long: from four rounds on (245,760 rows, K
// = 5120: strip 240 against 235 us at T = 8; 248,320: 239 / 233; 393,216: 381
// / 372; rounds that are 15/16 full or more: 294,912 rows take 291 / 292),
// from two at K = 8192 (122,880 rows, T = 4: 196 / 187), and in one round past
// eight tokens (57,344 rows, K = 5120, T = 12: 67 / 60; 65,536: 76 / 71). Two
// and three rounds of shorter rows tie, emptier ones lose (200,000 rows, T =
// 1: 189 / 210), still shorter rows too (65,536 rows, K = 4096, T = 8: 54 /
// 61).
inline DecodeRoute route_w8(const DecodeShape &s) {
    if (s.S != 1 || s.K < 4608) return kRouteStrip;
    const long long per = 16ll * s.cus, rounds = (s.rgs + per - 1) / per;
    if (rounds >= 4 || (rounds >= 2 && s.K >= 8192))
        return 16ll * s.rgs >= 15 * rounds * per ? kRouteRowwave : kRouteStrip;
    return rounds == 1 && s.T > 8 && 8ll * s.rgs >= 7 * per ? kRouteRowwave : kRouteStrip;
}

// Reference mode: many rows in one split, group 64 (34,816 rows, K = 5120, T
// = 4: 32.4 / 29.8; 65,536 rows, T = 8: 45.9 / 43.0; at group 32 both take the
// same), and two splits where the rows fill six row-groups per CU and no more
// (24,576 rows, K = 8192, T = 4: 31.9 / 28.6 at group 64, 32.4 / 30.3 at 32;
// 26,624 rows tie or lose). One or two tokens stay on the strips, whose
// chains run on the real tokens alone.
inline DecodeRoute route_blocks(const DecodeShape &s) {
    if (s.T <= 2 || s.group == 16) return kRouteStrip;
    if (s.S == 1) return s.group == 64 && s.rgs >= 8 * s.cus ? kRouteRowwave : kRouteStrip;
    return s.S == 2 && s.K >= 4096 && s.rgs > 5 * s.cus && s.rgs <= 6 * s.cus ? kRouteRowwave : kRouteStrip;
}

// Per token. The row-wave kernel cuts the rows evenly over the CUs and keeps
// four tiles of weights in flight per wave, which long streams reward; the
// strips run more splits of more rows side by side.
inline DecodeRoute route_token(const DecodeShape &s) {
    const int T = s.T, K = s.K, cus = s.cus;
    const bool g64 = s.group == 64;
    auto rowwave = [](bool yes) { return yes ? kRouteRowwave : kRouteStrip; };
    // one or two splits: enough rows to stream (34,816 rows, K = 5120, T = 1:
    // strip 22.6 against row-wave 18.4 us; 17,408 rows, T = 2 14.6 / 11.6, T =
    // 16 16.6 / 14.5). (Short rows in two splits of one or two tokens at
    // group 128: 28,480 rows, K = 2432 9.7 / 10.8.)
    if (s.S <= 2) return rowwave(!(s.S == 2 && T <= 2 && !g64 && K < 2560 && s.rgs > 5 * cus));
    if (s.rgs <= cus) {
        // At most one row-group per CU: the K-parallel kernel reads a
        // row-group in consecutive kilobytes by one work-group. It is ahead
        // while its token slices are short (past five tokens the chains of a
        // slice take over: 640 rows, K = 6144, T = 8, one slice of eight:
        // strip 7.7 against 9.2 us; K = 7936, two of four: 9.0 / 7.5) and all
        // resident at once (3,072 rows, K = 17408, T = 4: 12.4 / 15.9).
        // Sixteen splits (the GEMM plan): 1,024 rows, group 128, K = 12288, T =
        // 1 8.5 / 6.8; K = 17408, T = 16 12.6 / 10.3; group 64, K = 3840, T = 1
        // 6.4 / 5.4.
        const int nu = K / s.group, ts = kparallel_slice(nu, nu, T, s.S, false);
        const bool kpar = ts > 0 && ts <= 5 && (long long)s.rgs * ((T + ts - 1) / ts) <= cus;
        if (s.S == 16) return kpar && K > (T <= 4 ? 1024 : 2048) ? kRouteKParallel : kRouteStrip;
        if (s.S != 8 || T > 4) return kRouteStrip;
        // eight splits (the GEMV plan): 2,048 rows, K = 8192, group 64, T = 1
        // strip 6.8 against row-wave 5.6 us; K = 17408, T = 3 10.9 / 10.0;
        // group 128, K = 12288, T = 4 8.7 / K-parallel 8.0
        if (T <= 2) return rowwave(K > (g64 ? 2048 : 4096));
        if (g64) return rowwave(K > 8192);
        return kpar && K > 4096 ? kRouteKParallel : kRouteStrip;
    }
    // More rows, four splits and up.
    const bool two = s.rgs <= 2 * cus;
    const int kmin = g64 ? 6144 : 8192;
    // 8,192 rows in four splits, group 64: K = 4096, T = 1 7.6 / 6.8 us; 6,144
    // rows in eight: K = 8192, T = 2 9.0 / 8.4
    if (T <= 2) return rowwave(s.S == 4 ? K >= (two ? 4096 : 6144) : two && K >= kmin);
    // 14,336 rows in four splits, K = 8192, T = 8: 17.4 / 15.3; 6,144 rows in
    // eight, group 64, K = 12288: 14.6 / 12.6 (17,408 rows in eight, K = 5120,
    // T = 4: 19.5 / 27.8)
    if (T <= 8) return rowwave(s.S == 4 ? K >= 6144 : T > 4 && two && K >= kmin);
    // 6,144 rows, K = 12288, T = 12: 15.6 / 13.3; 16,384 rows in eight, K =
    // 8192: 25.6 / 21.4 (10,240 rows: 15.2 / 19.5)
    return rowwave(K >= (g64 ? 4608 : 6144) && (two || (s.rgs > 3 * cus && s.rgs <= 4 * cus)));
}

// The launch's kernel among those built for its mode (strip_takes).
inline DecodeRoute decode_route(const DecodeShape &s) {
    if (s.T > 16 || s.S == 0) return kRouteStrip;
    if (s.w8) return route_w8(s);
    return s.blocks ? route_blocks(s) : route_token(s);
}

// One-split projections of up to this many 16-row x 32-token strips run on
// the strip kernel, whose grid still fills the chip where the large tiles
// leave CUs idle (us on strips / on tiles). Per token, group 128: N = 5120, K =
// 17408, T = 256, 2,560 strips: 58 / 81; up to 4,000 strips 10-30 % ahead. Group
// 64, whose tiles share more of the unpack: up to 3,100 strips 9 % ahead, from
// there to 4,000 2 % behind (17,408 rows, K = 5120, T = 96, 3,264 strips: 33.1 /
// 29.8; 14,336 rows, K = 4096, T = 128: 27.0 / 24.9). Reference mode: N = 5120,
// K = 17408, T = 512, 5,120 strips: 227 / 234; 17,408 rows, K = 5120, T = 256,
// 8,704 strips: 113 / 109.
inline long long one_split_strips(int block, int group) {
    if (block == 32) return 5500;
    return group == 64 ? 3100 : 4000;
}

// Reference-mode GEMM tiles of 128 rows: 64 tokens wide, or 32. The wider one
// takes a CU 1.65 times as long for twice the work (swept at 484 points: 1.56
// to 1.84), so what counts is how many of each the busiest CU gets. 34,816
// rows, K = 5120, T = 90: 3 wide against 4 narrow per CU, 111 against 92 us; T =
// 128: 3 against 5, 112 / 116; 17,408 rows, T = 300: 3 against 6, 111 / 131;
// 10,240 rows, T = 300: 2 against 4, 83 / 90. `rows`: 128-row tiles over all
// weights.
inline bool gemmr_wide(int cus, long long rows, int T) {
    const long long wide = (rows * ((T + 63) / 64) + cus - 1) / cus, narrow = (rows * ((T + 31) / 32) + cus - 1) / cus;
    return 165 * wide < 100 * narrow;
}

// W4A4 GEMM tiles of 64 rows: 64 tokens, or 128. At K = 17408 a 64 x 64 tile
// takes a CU 46-51 us and a 128 x 64 tile, whose two token blocks share the
// weight unpack, 88-95 us: 1.87 times as long for twice the work, so the
// smaller one wins where its finer grid saves more than that, and where two of
// them run side by side in place of a single large one (swept at 284 points;
// 64 x 64 against 128 x 64, N = 5120, K = 17408: T = 64 98 against 134 us, T = 512
// 154.7 / 179.8, T = 1024 252 / 284, T = 2048 463 / 441; N = 17408, K = 5120, T =
// 512 128.5 / 134.2; N = 2048, K = 5120, T = 1024, two for one: 40.2 / 42.7).
// `rows`: 64-row tiles.
inline bool w4a4_small(int cus, long long rows, int T) {
    const long long large = (rows * ((T + 127) / 128) + cus - 1) / cus, small = (rows * ((T + 63) / 64) + cus - 1) / cus;
    return large == 1 || 100 * small < 187 * large;
}

// A packed prompt in per-token mode whose segments have one split and several:
// strips and large tiles in a launch each, or the general GEMM kernel in one.
struct PackedShape {
    int cus, K, group;
    int launches;                     // of the strip and large-tile kernels
    int tile_runs;                    // of the large tiles
    long long few, lots;              // split strips of at most 8 tokens, of 16
    long long strips;                 // one-split strips of 32 tokens
    long long tile_work;              // row-groups x tokens on the large tiles
    long long general;                // work-groups (64 tokens x 128 rows) of the general kernel
};

// The general kernel's tiles reach over segments, so segments of a few tokens
// cost it nothing, and it walks all of K in one pass whatever the split
// counts: about 8 us per 1,000 columns while its work-groups are resident
// (two per CU), more rows and tokens on top. The other launches cost their
// strips and about 6 us each. Both sides fitted over 1,581 random packings of
// 2-7 segments of 1-600 tokens, 512-17,408 rows, 1,024-17,408 columns (mean
// error 9 %); us a projection, in thousands of columns. (123 + 48 + 119 + 33 +
// 6 + 39 tokens of two weights of 5,344 rows, K = 1920, group 64: 54.8 against
// 37.3 us on the general kernel; 16 + 32 + 64 + 128 + 256 tokens of two of
// 5,120, K = 17408: 234 against 296.)
inline bool packed_general(const PackedShape &s) {
    const bool g64 = s.group == 64;
    const double k = s.K / 1000.0, full = 2.0 * s.cus;
    double general = 18 + k * (g64 ? 7.2 : 6.4);
    if (s.general > s.cus) general += 2 * k;
    if (s.general > full) general += k * (4.7 + (g64 ? 10.5 : 9.0) * (s.general / full - 1));
    const double others = 5.6 * s.launches +
                          k * ((1.0 * s.few + 1.5 * s.lots + 1.0 * s.strips) / 1000 + (s.strips ? 1.0 : 0.0) +
                               2.5 * s.tile_runs + (g64 ? 3.0 : 2.0) * s.tile_work / 1e5);
    return others > general;
}

}  // namespace kxw4
