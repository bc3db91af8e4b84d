// kxw4_strip.hip — projections of one to a few hundred tokens under any split
// plan: the GEMV (kernels_dpas.cpp:586-675, K16 683-760, W8 771-844), the
// fan-out GEMV (945-1102) and the GEMM (1334-1490, W8 1578-1629).
//
// A wave owns a strip of 16 weight rows x one tile of TT tokens and one split
// of K at a time, and runs its outputs' reference chains in registers: the
// 16x16 int8 MFMA leaves row n = l%16 of tokens 4*(l/16)+r in register r of
// lane l for each unit, in unit order. A work-group is SW streams x RW waves:
// the RW waves of a stream take neighbouring row-groups and share the
// stream's activation tiles, the streams are the splits of the same rows,
// whose partials meet in LDS for the ordered sum (S = 1: one stream).
//
// What bounds it. With tens of tokens in reference mode the chain (VALU: 3
// operations per output and K32 unit, about 1.1 ns each per SIMD, beside ~14
// per unit for the zero-point fold; 66 % busy at 27 tokens, 83 % at 512). At one
// token, and per token where few strips leave one wave per SIMD, latency: the
// VALU is 23-40 % busy, LDS 10 %, HBM at 2.9-3.9 TB/s, and the waves wait 38-47 %
// of their time. Neither a memory round trip nor a barrier is paid per 128-K
// tile (the figures of this list: four weights in turn, partly in the
// last-level cache):
//   * every operand of a stage (packed weights, activations, both scales)
//     reaches LDS by direct global->LDS loads, and a stage holds U = 2 or 4
//     tiles, double-buffered: one wait and one barrier per U tiles (one tile
//     per stage: N = 5120, K = 17408, T = 64 per-token 57 against 42 us);
//     deeper rings measured worse at tens of tokens, since they cost
//     work-groups per CU (block mode N = 17408, K = 5120, T = 64: 53 against 43
//     us); at a few tokens only with weights partly in the last-level cache,
//     so whether a deeper ring helps a stream from HBM there is open;
//   * the pointers of a stage's loads move by constants, so an issue is a
//     handful of scalar operations (recomputed from the tile index they were
//     ~70 per stage: 42 -> 37.6 us for the shape above);
//   * in block mode a unit's MFMAs are issued before the previous unit's
//     chain (left to the compiler each chain waits for its own MFMA: block
//     mode N = 17408, T = 64: 55 -> 48 us);
//   * the activation scales of a lane's four tokens are read once per tile,
//     four units at a time, in the [token][unit] order they arrive in.
// Measured against the kernels it replaced (launches of a graph replay, weights
// from HBM): reference mode, group 64, N = 5120, K = 17408: GEMV T = 1 20.9 ->
// 17.0 us, GEMM T = 16 272 -> 24.7, T = 64 3145 -> 72.7; fan-out over 34,816
// rows, K = 5120, T = 1 67.5 -> 25.3; per token, group 64, N = 5120, K = 17408,
// T = 64 333 -> 36.6; K16 N = 5120, K = 17408: T = 1 36.2 -> 20.0, T = 16 325 ->
// 32.2; W8 N = 17408, K = 5120: T = 8 30.5 -> 22.2, T = 64 140 -> 43.2, T = 256 402
// -> 107. Launches of up to 16 tokens that another kernel runs faster stay
// there (kxw4_route.hpp).
#include "kxw4_device.hpp"
#include "kxw4_internal.hpp"

#include <algorithm>
#include <type_traits>

namespace kxw4 {


enum { kStW4 = 0, kStW8 = 1, kStK16 = 2 };

#define KXW4_ST_LDS(p) ((__attribute__((address_space(3))) void *)(p))

// Sizes of one stream's stage (U 128-K tiles) in LDS: weights [U][RW][tile],
// activations [U][TT tokens][128 B] (16-byte pieces XOR-swizzled by the
// token), weight scales [RW][groups of U tiles][16] u16, activation scales
// [U][TT tokens][4]. TT: tokens per tile, 1, 2, 8, 16 or 32 (up to 8 tokens
// the MFMA's other rows repeat them; with 1 or 2 the chains run on the real
// tokens' registers alone).
template <int TT, int RW, int U, bool BLK, int WF>
struct StShape {
    static constexpr int NT = TT == 32 ? 2 : 1;              // 16-token MFMA rows
    static constexpr int NR = TT < 4 ? TT : 4;               // result registers that hold tokens
    static constexpr int TB = WF == kStW8 ? 2 : 1;
    static constexpr int W_TILE = RW * TB * kTileBytes, W_BYTES = U * W_TILE;
    static constexpr int A_TILE = TT * kTileK, A_BYTES = U * A_TILE;
    static constexpr int S_ROW = U * (WF == kStK16 ? 256 : 128);   // most scale bytes of a row-group and stage
    static constexpr int S_BYTES = RW * S_ROW;
    static constexpr int AS_TILE = BLK ? TT * 16 : 0, AS_BYTES = U * AS_TILE;
    static constexpr int A_OFF = W_BYTES, S_OFF = A_OFF + A_BYTES, AS_OFF = S_OFF + S_BYTES;
    static constexpr int STAGE = AS_OFF + AS_BYTES;
    // 16-byte pieces of activations and of activation scales, 64 to a load,
    // dealt to the row waves
    static constexpr int PA = U * 8 * TT, A_LOADS = ((PA + 63) / 64 + RW - 1) / RW;
    static constexpr int PS = U * TT, S_LOADS = ((PS + 63) / 64 + RW - 1) / RW;
    // loads a wave issues per stage when it issues all of them (RW = 1)
    static constexpr int LOADS = U * TB + A_LOADS + 1 + (BLK ? S_LOADS : 0);
    static_assert(LOADS <= 63, "vmcnt field");
    static_assert(STAGE % 16 == 0, "16-byte stages");
};

// int8 bytes w - z of one packed dword (a K32 unit's eight nibbles of a
// lane): each nibble becomes 0x80 | (w ^ 8) = 136 + w, minus z + 8 (zz, in
// every byte) leaves 128 + w - z in [113, 143], so no borrow crosses a byte,
// and the XOR makes it two's complement.
__device__ __forceinline__ long st_fold(uint32_t d, uint32_t zz) {
    const uint32_t lo = ((((d ^ 0x08080808u) & 0x0F0F0F0Fu) | 0x80808080u) - zz) ^ 0x80808080u;
    const uint32_t hi = (((((d >> 4) ^ 0x08080808u) & 0x0F0F0F0Fu) | 0x80808080u) - zz) ^ 0x80808080u;
    return (long)((uint64_t)lo | ((uint64_t)hi << 32));
}

// BLK: activation scales per (token, K32 block), units of 32 (reference
// mode; W4 weights have FP16|zp scales); else one scale per token, plain FP16
// weight scales, units of one weight group. VAR: GEMV (two accumulators),
// fan-out or GEMM (x * (ws * as)).
template <int TT, int RW, int U, int UNIT, bool BLK, int VAR, int WF>
__global__ __launch_bounds__(512) void strip_kernel(const StripArgs a) {
    using S = StShape<TT, RW, U, BLK, WF>;
    constexpr int UPS = kTileK / UNIT, TB = S::TB, NT = S::NT, NR = S::NR;
    constexpr bool ALT2 = VAR == kVarGemv && WF != kStK16;
    constexpr bool ZP = BLK && WF != kStW8;
    static_assert(U % 2 == 0, "the GEMV accumulator of a whole tile is its place in the stage");
    static_assert(!BLK || UNIT == 32, "K32 activation blocks");
    static_assert(BLK || WF == kStW4, "per-token mode: W4");
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];

    // ---- block -> (entry, token tile, row-groups): the work-groups of one
    // XCD (blockIdx % 8) take consecutive tiles, token tiles fastest, so the
    // token tiles of the same rows read the weights from that XCD's L2 ----
    const int nblk = gridDim.x, id = blockIdx.x;
    const int q8 = nblk / 8, r8 = nblk % 8, xcd = id % 8, j8 = id / 8;
    const int L = xcd < r8 ? xcd * (q8 + 1) + j8 : r8 * (q8 + 1) + (xcd - r8) * q8 + j8;
    // (the first entry and all four weights are read with constant indices,
    // so their scalar loads go out together; an indexed read of the kernel
    // arguments would add a dependent round trip each to the start)
    StripEntry e = a.e[0];
    for (int i = 1; i < a.entries; ++i)
        if (L >= a.e[i].blk) e = a.e[i];
    StripWeight w = a.w[0];
#pragma unroll
    for (int i = 1; i < kMaxWeights; ++i) {
        StripWeight o = a.w[i];
        asm volatile("" : "+s"(o.codes), "+s"(o.scales), "+s"(o.y), "+s"(o.M));
        if (e.w == i) w = o;
    }
    const int t1 = e.t1;
    const int within = L - e.blk, ntt = (t1 - e.t0 + TT - 1) / TT;
    const int rgi = ntt == 1 ? within : within / ntt;        // (one token tile: no division)
    const int t0 = e.t0 + (within - rgi * ntt) * TT;
    const uint8_t *codes = w.codes;
    const uint8_t *scales = reinterpret_cast<const uint8_t *>(w.scales);
    const int M = w.M, RG = M / 16;
    const int K = a.K, NTK = K / kTileK, Nu = K / UNIT;
    // streams of this block's entry: its splits, a.waves / RW at most (then
    // each takes two in turn); with one row wave the waves left over take
    // further row-groups (`item`), so entries of different split counts share
    // a launch
    const int SP = e.S, SW = min(SP, a.waves / RW);          // (powers of two)
    const int ls = __builtin_ctz(SP), lsw = __builtin_ctz(SW);

    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g4 = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rw = wave % RW, sw = RW == 1 ? wave & (SW - 1) : wave / RW;   // row wave, stream
    const int item = RW == 1 ? wave >> lsw : 0;
    const int rg = RW == 1 ? rgi * (a.waves >> lsw) + item : rgi * RW + rw;
    const int rgc = min(rg, RG - 1);                         // (row-groups past M load the last one, store nothing)
    const int gpt = kTileK / a.group;                        // scale groups per tile
    const int gsh = BLK && WF != kStK16 ? __builtin_ctz(a.group / 32) : 0;

    // ---- load issue: wave-uniform pointers that move one stage per issue
    // and 32-bit lane offsets that do not change ----
    // (piece p of token t of a tile is stored at slot p ^ (t & 7); ptile:
    // the tile of the stage a lane's piece belongs to)
    uint32_t woff[U][TB], aoff[S::A_LOADS], soff[S::S_LOADS];
    int atile[S::A_LOADS], stile[S::S_LOADS];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int h = 0; h < TB; ++h) woff[u][h] = (u * TB + h) * kTileBytes + lane * 16;
#pragma unroll
    for (int i = 0; i < S::A_LOADS; ++i) {
        const int g = min((rw + RW * i) * 64 + lane, S::PA - 1);
        const int t = (g >> 3) % TT;
        atile[i] = g / (8 * TT);
        aoff[i] = (uint32_t)min(t0 + t, t1 - 1) * K + atile[i] * kTileK + ((g & 7) ^ (t & 7)) * 16;
    }
#pragma unroll
    for (int i = 0; i < S::S_LOADS; ++i) {
        const int g = min((RW - 1 - rw + RW * i) * 64 + lane, S::PS - 1);
        stile[i] = g / TT;
        soff[i] = (uint32_t)min(t0 + g % TT, t1 - 1) * (K / 32) * 4 + stile[i] * 16;
    }
    const int sgr = gpt * 2;                                 // 16-byte pieces of scales per tile
    const uint8_t *const wrow = codes + (size_t)rgc * NTK * (kTileBytes * TB);
    const uint8_t *const srow = scales + (size_t)rgc * NTK * gpt * 32;
    uint8_t *const ring = smem + (RW == 1 ? wave : sw) * 2 * S::STAGE;
    const uint8_t *wp = nullptr, *sp_ = nullptr, *qp = nullptr, *ap = nullptr;
    int islot = 0;                                           // stage the next issue fills
    auto seek = [&](int kt) {
        wp = wrow + (size_t)kt * (kTileBytes * TB);
        sp_ = srow + (size_t)kt * gpt * 32;
        qp = reinterpret_cast<const uint8_t *>(a.q) + (size_t)kt * kTileK;
        ap = reinterpret_cast<const uint8_t *>(a.ascale) + (size_t)kt * 16;
        islot = 0;
    };
    // the next U tiles, of which `have` are inside K (the others repeat the
    // last one and are never used)
    auto issue = [&](int have) {
        uint8_t *b = ring + islot * S::STAGE;
        asm volatile("" : "+s"(wp), "+s"(sp_), "+s"(qp), "+s"(ap));
        auto load = [&](auto full) {
            constexpr bool FULL = decltype(full)::value;
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int h = 0; h < TB; ++h)
                    __builtin_amdgcn_global_load_lds(
                        (const void *)(wp + (FULL ? woff[u][h] : woff[u][h] - max(u + 1 - have, 0) * kTileBytes * TB)),
                        KXW4_ST_LDS(b + u * S::W_TILE + (rw * TB + h) * 1024), 16, 0, 0);
#pragma unroll
            for (int i = 0; i < S::A_LOADS; ++i) {
                const int c = rw + RW * i;
                if (c * 64 < S::PA && (S::PA % 64 == 0 || c * 64 + lane < S::PA))
                    __builtin_amdgcn_global_load_lds(
                        (const void *)(qp + (FULL ? aoff[i] : aoff[i] - max(atile[i] + 1 - have, 0) * kTileK)),
                        KXW4_ST_LDS(b + S::A_OFF + c * 1024), 16, 0, 0);
            }
            if (lane < sgr * (FULL ? U : have))
                __builtin_amdgcn_global_load_lds((const void *)(sp_ + lane * 16),
                                                 KXW4_ST_LDS(b + S::S_OFF + rw * S::S_ROW), 16, 0, 0);
            if constexpr (BLK) {
#pragma unroll
                for (int i = 0; i < S::S_LOADS; ++i) {
                    const int c = RW - 1 - rw + RW * i;
                    if (c * 64 < S::PS && (S::PS % 64 == 0 || c * 64 + lane < S::PS))
                        __builtin_amdgcn_global_load_lds(
                            (const void *)(ap + (FULL ? soff[i] : soff[i] - max(stile[i] + 1 - have, 0) * 16)),
                            KXW4_ST_LDS(b + S::AS_OFF + c * 1024), 16, 0, 0);
                }
            }
        };
        if (have >= U) load(std::true_type{});
        else load(std::false_type{});
        wp += U * kTileBytes * TB;
        sp_ += (size_t)U * gpt * 32;
        qp += U * kTileK;
        ap += U * 16;
        islot ^= 1;
    };

    // ---- per-lane read offsets inside a stage ----
    const int w_rd = rw * TB * 1024 + lane * 16;
    const int ta = TT >= 16 ? n : n & (TT - 1);              // this lane's operand row (up to 8 tokens repeat)
    const int a_rd0 = S::A_OFF + ta * 128 + ((g4 ^ (ta & 7)) * 16);
    const int a_rd1 = S::A_OFF + ta * 128 + (((4 + g4) ^ (ta & 7)) * 16);
    const int s_rd = S::S_OFF + rw * S::S_ROW + n * 2;
    const int as_rd = S::AS_OFF + (TT >= 16 ? 4 * g4 : TT == 8 ? 4 * (g4 & 1) : 0) * 16;   // tokens of register 0

    // The output's token scales and residuals, loaded where their latency
    // hides: behind the first stage's loads (one row wave), else after the
    // stream, before the split sum. (Two loops: with the residual's test
    // between the registers of one loop the compiler keeps `tsc` in private
    // memory, and the store there waits for the first stage before the second
    // is requested. Weights from HBM, 4096 x 4096: T = 2 5.93 -> 5.83 us, T
    // = 8 6.34 -> 6.10 at group 64; 2 to 16 tokens 4 % faster over 512-65,536
    // rows of 1,024-17,408 columns.)
    const int row = rg * 16 + n;
    float tsc[NT][4], rsd[NT][4];
    auto load_epilogue = [&]() {
        if (sw != 0) return;
        if constexpr (!BLK) {
#pragma unroll
            for (int b = 0; b < NT; ++b)
#pragma unroll
                for (int r = 0; r < NR; ++r) tsc[b][r] = a.ascale[min(t0 + 16 * b + 4 * g4 + r, t1 - 1)];
        }
        if (!a.residual) return;
#pragma unroll
        for (int b = 0; b < NT; ++b)
#pragma unroll
            for (int r = 0; r < NR; ++r)
                rsd[b][r] = a.residual[(size_t)min(t0 + 16 * b + 4 * g4 + r, t1 - 1) * M + min(row, M - 1)];
    };

    float res[NT][4] = {}, res_prev[NT][4];                  // this turn's chains and the turn before's
    const int turns = SP >> lsw;                             // splits a stream runs in turn (1 or 2)
#pragma unroll 1
    for (int turn = 0; turn < turns; ++turn) {
        const int sp = sw * turns + turn;
        const int u0 = (int)(((long long)Nu * sp) >> ls), u1 = (int)(((long long)Nu * (sp + 1)) >> ls);
        const int kt0 = u0 / UPS, ntl = u1 > u0 ? (u1 + UPS - 1) / UPS - kt0 : 0;
        const int nst = (ntl + U - 1) / U;
        // stages of the longest stream: the barriers are the work-group's
        int nmax = nst;
        if constexpr (RW > 1) {
            for (int o = 0; o < SW; ++o) {
                const int so = o * turns + turn;
                const int v0 = (int)(((long long)Nu * so) >> ls), v1 = (int)(((long long)Nu * (so + 1)) >> ls);
                nmax = max(nmax, v1 > v0 ? ((v1 + UPS - 1) / UPS - v0 / UPS + U - 1) / U : 0);
            }
        }
        float f0[NT][4], f1[NT][4];
#pragma unroll
        for (int b = 0; b < NT; ++b)
#pragma unroll
            for (int r = 0; r < NR; ++r) f0[b][r] = f1[b][r] = 0.0f;

        // (the stages of the turn before may still be read by other waves)
        if (turn > 0) lds_sync();
        seek(kt0);
        const int room = NTK - kt0;                          // tiles from the split's start to the end of K
        if (nst > 0) issue(room);
        if (NT == 1 && RW == 1 && turn == 0) load_epilogue();           // (behind the first stage's loads)
        // (a stream of two stages has both in flight from the start; longer
        // ones keep one ahead: two took 12.3 against 10.8 us at T = 1, N = 5120,
        // K = 17408 per token, weights partly in the last-level cache)
        const bool both = RW == 1 && nst == 2;
        if (both) issue(room - U);
        // stages whose tiles lie wholly inside the split
        const int nfull = u0 % UPS == 0 && u1 % UPS == 0 ? ntl / U : 0;

        int slot = 0;
        auto step = [&](int kt, auto uc, auto edge) {
            constexpr bool EDGE = decltype(edge)::value;     // a tile with units outside the split
            constexpr int UI = decltype(uc)::value;          // the tile's place in its stage
            const uint8_t *sb = ring + slot * S::STAGE;
            const uint8_t *ss = sb + UI * gpt * 32;          // (scale rows follow the tiles closely)
            v4u wd[TB];
#pragma unroll
            for (int h = 0; h < TB; ++h) wd[h] = *reinterpret_cast<const v4u *>(sb + w_rd + UI * S::W_TILE + h * 1024);
            v4i A[NT][2];
#pragma unroll
            for (int b = 0; b < NT; ++b) {
                A[b][0] = *reinterpret_cast<const v4i *>(sb + a_rd0 + UI * S::A_TILE + b * 2048);
                A[b][1] = *reinterpret_cast<const v4i *>(sb + a_rd1 + UI * S::A_TILE + b * 2048);
            }
            const v4i zero = {0, 0, 0, 0};
            if constexpr (!BLK) {
#pragma unroll
                for (int j = 0; j < UPS; ++j) {
                    if (EDGE && (kt * UPS + j < u0 || kt * UPS + j >= u1)) continue;
                    const float ws = half_bits_to_float(*reinterpret_cast<const uint16_t *>(ss + s_rd + j * 32));
                    v4i b0 = {}, b1 = {};
                    if constexpr (UNIT == 128) {
                        b0 = unpack_k64(wd[0].x, wd[0].y);
                        b1 = unpack_k64(wd[0].z, wd[0].w);
                    } else {
                        b0 = j == 0 ? unpack_k64(wd[0].x, wd[0].y) : unpack_k64(wd[0].z, wd[0].w);
                    }
#pragma unroll
                    for (int b = 0; b < NT; ++b) {
                        v4i acc;
                        if constexpr (UNIT == 128) {
                            acc = mfma_k64(A[b][0], b0, zero);
                            acc = mfma_k64(A[b][1], b1, acc);
                        } else {
                            acc = mfma_k64(A[b][j], b0, zero);
                        }
                        // GEMV: units at odd offsets from the split's start
                        // feed the second accumulator. Stages hold an even
                        // number of tiles, so a whole tile's parity is its
                        // place in the stage; a split that starts on an odd
                        // half tile swaps the two, and their sum commutes.
                        constexpr bool kOddTile = UNIT == 128 && (UI & 1);
#pragma unroll
                        for (int r = 0; r < NR; ++r) {
                            float &F = ALT2 && (kOddTile || (UNIT == 64 && j == 1)) ? f1[b][r] : f0[b][r];
                            F = __builtin_fmaf((float)acc[r], ws, F);
                        }
                    }
                }
            } else {
                // activation scales of tokens 4*g4 + r, the step's four units
                v4f as[NT][4];
#pragma unroll
                for (int b = 0; b < NT; ++b)
#pragma unroll
                    for (int r = 0; r < NR; ++r)
                        as[b][r] = *reinterpret_cast<const v4f *>(sb + as_rd + UI * S::AS_TILE + b * 256 + r * 16);
                // A unit's scale words, weight operand and MFMAs; then, once
                // the next unit's MFMAs are issued, its chain updates (the
                // scheduling barriers keep that order: left alone, each
                // unit's updates follow its own MFMAs and wait for them).
                uint32_t sw0[4], sw1[WF == kStK16 ? 4 : 1];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if constexpr (WF == kStK16) {
                        sw0[j] = *reinterpret_cast<const uint16_t *>(ss + s_rd + 2 * j * 32);
                        sw1[j] = *reinterpret_cast<const uint16_t *>(ss + s_rd + (2 * j + 1) * 32);
                    } else {
                        sw0[j] = *reinterpret_cast<const uint16_t *>(ss + s_rd + (j >> gsh) * 32);
                    }
                }
                constexpr int H = WF == kStK16 ? 2 : 1;      // MFMAs per unit and token block
                v4i acc[2][NT][H];
                auto front = [&](int j) {
                    long bv;
                    if constexpr (WF == kStW8) {
                        const v4u hh = wd[j >> 1];
                        bv = (j & 1) ? (long)(((uint64_t)hh.w << 32) | hh.z) : (long)(((uint64_t)hh.y << 32) | hh.x);
                    } else {
                        // (K16: lane groups 0-1 carry the unit's first half)
                        uint32_t sz = sw0[j];
                        if constexpr (WF == kStK16) sz = g4 < 2 ? sw0[j] : sw1[j];
                        const uint32_t d = j == 0 ? wd[0].x : j == 1 ? wd[0].y : j == 2 ? wd[0].z : wd[0].w;
                        bv = st_fold(d, __builtin_amdgcn_perm(0u, (sz & 0xFu) ^ 8u, 0u));
                    }
#pragma unroll
                    for (int b = 0; b < NT; ++b) {
                        const v4i c = A[b][j >> 1];
                        const long av = (j & 1) ? (long)(((uint64_t)(uint32_t)c.w << 32) | (uint32_t)c.z)
                                                : (long)(((uint64_t)(uint32_t)c.y << 32) | (uint32_t)c.x);
                        if constexpr (WF == kStK16) {
                            acc[j & 1][b][0] = mfma_k32(av, g4 < 2 ? bv : 0l, zero);
                            acc[j & 1][b][H - 1] = mfma_k32(av, g4 < 2 ? 0l : bv, zero);
                        } else {
                            acc[j & 1][b][0] = mfma_k32(av, bv, zero);
                        }
                    }
                };
                auto chain = [&](int j) {
                    if (EDGE && (kt * 4 + j < u0 || kt * 4 + j >= u1)) return;
#pragma unroll
                    for (int h = 0; h < H; ++h) {
                        uint32_t s = sw0[j];
                        if constexpr (WF == kStK16) s = h ? sw1[j] : sw0[j];
                        const float ws = half_bits_to_float((uint16_t)(ZP ? s & 0xFFF0u : s));
#pragma unroll
                        for (int b = 0; b < NT; ++b)
#pragma unroll
                            for (int r = 0; r < NR; ++r) {
                                const float asv = as[b][r][j], x = (float)acc[j & 1][b][h][r];
                                float &F = (ALT2 && (j & 1)) ? f1[b][r] : f0[b][r];
                                if constexpr (VAR == kVarGemm) F = __builtin_fmaf(x, ws * asv, F);
                                else F = __builtin_fmaf(x * ws, asv, F);
                            }
                    }
                };
                front(0);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (j < 3) front(j + 1);
                    __builtin_amdgcn_sched_barrier(0);
                    chain(j);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        for (int i = 0; i < nmax; ++i) {
            // This wave's loads of stage i. Several row waves: the barrier
            // publishes every wave's and frees the other stage; one: a
            // stream's stages are its own.
            if (both && i == 0) KXW4_WAIT_VMCNT(S::LOADS);
            else KXW4_WAIT_VMCNT(0);
            if constexpr (RW > 1) {
                lds_sync_after_dma();
            } else {
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_waitcnt(0xC07F);          // lgkmcnt(0): the reads of the stage refilled next
                asm volatile("" ::: "memory");
            }
            if (!both && i + 1 < nst) issue(room - (i + 1) * U);
            auto tiles = [&](auto edge) {
                constexpr bool EDGE = decltype(edge)::value;
                auto one = [&](auto uc) {
                    constexpr int UI = decltype(uc)::value;
                    if (!EDGE || i * U + UI < ntl) step(kt0 + i * U + UI, uc, edge);
                };
                one(std::integral_constant<int, 0>{});
                one(std::integral_constant<int, 1>{});
                if constexpr (U > 2) {
                    one(std::integral_constant<int, 2>{});
                    one(std::integral_constant<int, 3>{});
                }
            };
            if (i < nfull) tiles(std::false_type{});
            else if (i < nst) tiles(std::true_type{});
            slot ^= 1;
        }
#pragma unroll
        for (int b = 0; b < NT; ++b)
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                res_prev[b][r] = res[b][r];
                res[b][r] = ALT2 ? f0[b][r] + f1[b][r] : f0[b][r];
            }
    }

    if constexpr (NT > 1 || RW > 1) load_epilogue();

    // ---- ordered split sum (from 0.0f), then the output ----
    if (SP > 1) {
        float *part = reinterpret_cast<float *>(smem);
        lds_sync();                                          // every wave is past its last step
        const int last = item * SP + sw * turns + turns - 1; // the wave's last split, in res
        constexpr int PITCH = RW * NT * 256;                 // floats of one split
#pragma unroll
        for (int b = 0; b < NT; ++b)
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                float *p = part + last * PITCH + (rw * NT + b) * 256 + r * 64 + lane;
                *p = res[b][r];
                if (turns > 1) p[-PITCH] = res_prev[b][r];
            }
        lds_sync();
        if (sw != 0) return;
        // (all of a token block's partials are read before the ordered adds:
        // a loop over the splits would wait for each read in turn)
        auto split_sum = [&](auto sc) {
            constexpr int SC = decltype(sc)::value;
#pragma unroll
            for (int b = 0; b < NT; ++b) {
                float v[SC][4];
                const float *p = part + item * SC * PITCH + (rw * NT + b) * 256 + lane;
#pragma unroll
                for (int q = 0; q < SC; ++q)
#pragma unroll
                    for (int r = 0; r < NR; ++r) v[q][r] = p[q * PITCH + r * 64];
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    float sum = 0.0f;
#pragma unroll
                    for (int q = 0; q < SC; ++q) sum = sum + v[q][r];
                    res[b][r] = sum;
                }
            }
        };
        switch (SP) {
        case 2: split_sum(std::integral_constant<int, 2>{}); break;
        case 4: split_sum(std::integral_constant<int, 4>{}); break;
        case 8: split_sum(std::integral_constant<int, 8>{}); break;
        default: split_sum(std::integral_constant<int, 16>{}); break;
        }
    }
    if (rg >= RG) return;
    constexpr float kInv16 = !BLK ? 0.0625f : 1.0f;          // the 16 w unpack's factor (per-token mode)
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int tl = 16 * b + 4 * g4 + r, t = t0 + tl;
            if (t >= t1 || (TT < 16 && tl >= TT)) continue;
            const float v = BLK ? res[b][r] : res[b][r] * (tsc[b][r] * kInv16);
            float out;
            if (a.residual) out = v + rsd[b][r];
            else if (VAR == kVarGemv && SP > 1) out = v + 0.0f;
            else out = v;
            if (a.y_bf16) static_cast<uint16_t *>(w.y)[(size_t)t * M + row] = float_to_bf16(out);
            else static_cast<float *>(w.y)[(size_t)t * M + row] = out;
        }
}

template <int TT, int RW, int U, int UNIT, bool BLK, int VAR, int WF>
static int st_launch(StripArgs &a, hipStream_t st) {
    using S = StShape<TT, RW, U, BLK, WF>;
    int smax = 1;
    for (int i = 0; i < a.entries; ++i) smax = std::max(smax, a.e[i].S);
    a.waves = RW > 1 ? smax * RW : a.same_s ? std::min(smax, 8) : smax >= 8 ? 8 : 4;
    auto blocks = [&]() {
        int blk = 0;
        for (int i = 0; i < a.entries; ++i) {
            a.e[i].blk = blk;
            const int rows = RW == 1 ? a.waves / std::min(a.e[i].S, a.waves) : RW;   // row-groups per block
            blk += ((a.e[i].t1 - a.e[i].t0 + TT - 1) / TT) * ((a.w[a.e[i].w].M / 16 + rows - 1) / rows);
        }
        return blk;
    };
    int blk = blocks();
    // Eight streams while every work-group is resident at once, else four
    // that take their splits in turn.
    if (RW == 1 && smax == 8 && blk > device_cus() * (160 * 1024 / (16 * S::STAGE))) {
        a.waves = 4;
        blk = blocks();
    }
    const size_t lds = std::max((size_t)2 * (RW == 1 ? a.waves : smax) * S::STAGE, (size_t)std::max(2 * a.waves, RW) * S::NT * 1024);
    if (lds > 160 * 1024 || a.waves > 8) return -2;          // (the rules below never ask for it)
    auto k = strip_kernel<TT, RW, U, UNIT, BLK, VAR, WF>;
    static bool attr[64] = {};                               // (the attribute is per device)
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return -6;
    if (!attr[dev]) {
        if (hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                160 * 1024) != hipSuccess)
            return -6;
        attr[dev] = true;
    }
    hipLaunchKernelGGL(k, dim3(blk), dim3(64 * a.waves), lds, st, a);
    return hipGetLastError() == hipSuccess ? 0 : -6;
}

// Row waves per work-group and tiles per stage. S = 1: four row waves share
// the activations; with 16-token tiles and a grid of at most one and a half
// work-groups per CU, four tiles per stage, since nothing else hides a
// stage's barrier and LDS latency (per-token N = 5120, K = 17408, T = 64:
// 37.6 -> 32.6 us; with more work-groups the LDS they take costs more than
// that: block mode N = 17408, K = 5120, T = 32: 31.7 -> 37.4 us). S > 1: one
// row wave per stream (T = 16, N = 5120, K = 17408, S = 4: 14.2 against 17.5
// us per-token and 22.2 against 24.4 us in block mode for two), two for W8
// past 16 tokens, whose tiles are twice as large (T = 48: 37.0 against 46 us).
template <int TT, int UNIT, bool BLK, int VAR, int WF>
static int st_rw(StripArgs &a, int T, int smax, hipStream_t st) {
    if constexpr (TT == 32 && VAR == kVarFanout) {          // (planned with 1, 8 or 16 splits)
        return st_launch<TT, 4, 2, UNIT, BLK, VAR, WF>(a, st);
    } else if constexpr (TT == 32) {
        return smax <= 2 ? st_launch<TT, 4, 2, UNIT, BLK, VAR, WF>(a, st) : st_launch<TT, 2, 2, UNIT, BLK, VAR, WF>(a, st);
    } else {
        if (smax == 1) {
            if constexpr (TT == 16) {
                long long blks = 0;
                for (int i = 0; i < a.entries; ++i)
                    blks += (long long)((a.e[i].t1 - a.e[i].t0 + 15) / 16) * ((a.w[a.e[i].w].M / 16 + 3) / 4);
                if (2 * blks <= 3LL * device_cus()) return st_launch<TT, 4, 4, UNIT, BLK, VAR, WF>(a, st);
            }
            return st_launch<TT, 4, 2, UNIT, BLK, VAR, WF>(a, st);
        }
        if constexpr (TT == 16 && WF == kStW8 && VAR == kVarGemm) {
            if (smax <= 4 && a.same_s && T > 16) return st_launch<TT, 2, 2, UNIT, BLK, VAR, WF>(a, st);
        }
        return st_launch<TT, 1, 2, UNIT, BLK, VAR, WF>(a, st);
    }
}

// Whether the entries of split count SC fill 32-token tiles: these share a
// row-group's unpack and scales between two blocks and
// pay once the 16-token ones fill the SIMDs four times over (W8, with no
// unpack but twice the weight bytes: twice) and their padding costs less than
// that (a 32-token strip takes 1.6 times a 16-token one).
static bool st_fills_32(const StripArgs &a, int SC, int per_simd) {
    long long strips16 = 0, strips32 = 0;
    for (int i = 0; i < a.entries; ++i) {
        if (a.e[i].S != SC) continue;
        const long long t = a.e[i].t1 - a.e[i].t0, rgs = a.w[a.e[i].w].M / 16;
        strips16 += rgs * ((t + 15) / 16);
        strips32 += rgs * ((t + 31) / 32);
    }
    return strips16 * SC > per_simd && 5 * strips16 > 8 * strips32;
}

// The entries of `a` that `pick` names, taken out of it.
template <class F>
static StripArgs st_take(StripArgs &a, F pick) {
    StripArgs own = a;
    int left = 0;
    own.entries = 0;
    for (int i = 0; i < a.entries; ++i) {
        if (pick(a.e[i])) own.e[own.entries++] = a.e[i];
        else a.e[left++] = a.e[i];
    }
    a.entries = left;
    return own;
}

template <int UNIT, bool BLK, int VAR, int WF>
static int st_shape(StripArgs &a, hipStream_t st) {
    constexpr int kFill = WF == kStW8 ? 2000 : 4400;
    constexpr bool k32 = WF == kStW4 || (WF == kStW8 && VAR == kVarGemm);   // (K16 and the W8 GEMV: 16 tokens at most)
    int T = 0, smax = 1;
    a.same_s = 1;
    for (int i = 0; i < a.entries; ++i) {
        T = std::max(T, a.e[i].t1 - a.e[i].t0);
        smax = std::max(smax, a.e[i].S);
        a.same_s &= a.e[i].S == a.e[0].S;
    }
    if constexpr (k32) {
        if (a.same_s && smax <= 4 && st_fills_32(a, smax, kFill)) return st_rw<32, UNIT, BLK, VAR, WF>(a, T, smax, st);
    }
    if (!a.same_s) {
        // entries of one split count that fill the 32-token tiles by
        // themselves: a launch of their own
        for (int SC = 1; k32 && SC <= 4; SC *= 2) {
            if (!st_fills_32(a, SC, kFill)) continue;
            StripArgs rest = a;
            StripArgs own = st_take(rest, [&](const StripEntry &e) { return e.S == SC; });
            const int r = st_shape<UNIT, BLK, VAR, WF>(own, st);
            return r ? r : st_shape<UNIT, BLK, VAR, WF>(rest, st);
        }
        // few-token entries apart from the others, once the grid is several
        // rounds deep: a 16-token tile of theirs costs as much as a full one
        // (1 + 1 + 14 + 19 + 34 tokens of two weights of 3,568 rows, K = 3712,
        // beside 371 tokens in one split: 103 -> 80 us; a shallower grid only
        // pays the second launch)
        StripArgs rest = a;
        StripArgs few = st_take(rest, [](const StripEntry &e) { return e.t1 - e.t0 <= 8; });
        long long strips16 = 0;
        for (int i = 0; i < a.entries; ++i)
            strips16 += (long long)(a.w[a.e[i].w].M / 16) * ((a.e[i].t1 - a.e[i].t0 + 15) / 16);
        if (few.entries && rest.entries && strips16 > 6ll * device_cus()) {
            const int r = st_shape<UNIT, BLK, VAR, WF>(few, st);
            return r ? r : st_shape<UNIT, BLK, VAR, WF>(rest, st);
        }
    }
    if (T == 1) return st_rw<1, UNIT, BLK, VAR, WF>(a, T, smax, st);
    if (T == 2) return st_rw<2, UNIT, BLK, VAR, WF>(a, T, smax, st);
    if (T <= 8) return st_rw<8, UNIT, BLK, VAR, WF>(a, T, smax, st);
    return st_rw<16, UNIT, BLK, VAR, WF>(a, T, smax, st);
}

bool strip_takes(int group, int block, int scale_enc, long long T, int K) {
    if (T * K >= (1ll << 31)) return false;                  // 32-bit activation offsets
    return block == 32 ? scale_enc != 0 && group != 128 : scale_enc == 0 && (group == 64 || group == 128);
}

int launch_strip(StripArgs &a, hipStream_t st) {
    if (a.scale_enc == 2)
        return a.variant == kVarGemv ? st_shape<32, true, kVarGemv, kStW8>(a, st) : st_shape<32, true, kVarGemm, kStW8>(a, st);
    if (a.group == 16) return st_shape<32, true, kVarGemv, kStK16>(a, st);
    if (a.block == 32) {
        if (a.variant == kVarGemv) return st_shape<32, true, kVarGemv, kStW4>(a, st);
        if (a.variant == kVarFanout) return st_shape<32, true, kVarFanout, kStW4>(a, st);
        return st_shape<32, true, kVarGemm, kStW4>(a, st);
    }
    // (per-token: the fan-out and GEMM arithmetic are the same)
    if (a.group == 128)
        return a.variant == kVarGemv ? st_shape<128, false, kVarGemv, kStW4>(a, st) : st_shape<128, false, kVarGemm, kStW4>(a, st);
    return a.variant == kVarGemv ? st_shape<64, false, kVarGemv, kStW4>(a, st) : st_shape<64, false, kVarGemm, kStW4>(a, st);
}

}  // namespace kxw4
