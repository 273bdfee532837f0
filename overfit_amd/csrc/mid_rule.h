// mid_rule.h — which kernel takes a K-quant batch whose activation the library quantises itself. Host code without any HIP
// type, so that it can be compiled and checked anywhere.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

namespace ovfq {

enum class MidKernel { kNone, kSplit, kPanel };  // kNone: the kernels of gemv.hip, mfma.hip and project.hip

// 16-row activation tiles of a panel workgroup, and the launch's time by that choice in units of a Q4_K CU's time for one
// tile over the inputs (3.0 us at 4096). By the busiest XCD: up to one workgroup a CU, whose waits nothing hides, takes
// 3.9 / 4.8 / 6.1 / 7.6 at T = 2 .. 5; the two that run at once take T + 0.8 each, less where not every CU has the second; so do
// further ones (q/k/v of 4096, us at T = 2 / 3 / 4 / 5: 96 rows 21.9 / 20.0 / 22.8 / 26.4, 160 rows 23.3 / 27.0 / 30.8 / 27.5,
// 331 rows 44.8 / 41.1 / 46.6 / 39.4, 512 rows 54.7 / 59.4 / 50.6 / 56.4; gate/up of 14336 at 65 rows 50.1 / 48.1 / 55.1 / 39.6;
// 2304x2304 at 512 rows 21.6 / 20.7 / 22.3 / 25.3, 3072x1024 17.6 / 19.8 / 22.0 / 25.0; over 1600 random shapes of 1024 to 6400 inputs
// and 300 to 1100 rows where it differs from even shares of at most four tiles, its choice took 0.90 of their time and 1.002 of
// the best height's). Even shares for Q6_K, whose operand build leaves a step of five units before its first tile.
inline double panel_cost(int type, long o_tiles, long subs, int* T) {
    const auto cost = [&](int t) {
        const double w = (double)((o_tiles + 7) / 8 * ((subs + t - 1) / t)) / 32.0;
        if (w <= 1.0) return 2.6 + 0.38 * t + 0.122 * t * t;
        return (t + 0.8) * (w <= 2.0 ? 1.6 + 0.2 * w : std::ceil(w)) + (w > 2.0 ? 0.5 : 0.0);
    };
    *T = (int)((subs + (subs + 3) / 4 - 1) / ((subs + 3) / 4));
    if (type == 12)
        for (int t = (int)std::min(5l, subs); t >= 2; t--)
            if (cost(t) < cost(*T)) *T = t;
    return cost(*T);
}

// Whether the split or panel kernel takes a batch of a few rows that the multi-row decode kernel would take. That one works
// through a row in items of 16 super-blocks; where the last item is mostly empty (17 to 21 super-blocks, two items) it is
// overtaken at 2 rows by three or more weights and from 3 rows by any, given outputs enough for the split kernel to fill the
// chip with (us, multi-row / split, Q4_K: q/k/v of 5120 at 2 rows 13.9 / 12.6, of 5376 12.6 / 13.5; 2432x4352 at 3 rows 9.2 / 9.6,
// 3168x5120 11.5 / 10.1; 1552x4352 at 4 rows 9.3 / 9.3, 2352x4608 11.4 / 9.7; Q6_K 4128x5120 at 3 rows 13.8 / 14.4, 5168x4352 15.8 / 14.3;
// 1584x4352 at 4 rows 10.7 / 11.0, 3520x4352 14.3 / 11.8). It also loses on one very tall matrix (128256x2048 at 3 rows 64.9,
// panel kernel 39.1).
inline bool mid_over_decode(int type, int in, int rows, long tiles, int count) {
    const int spr = in / 256;
    const bool short_item = spr > 16 && 2 * ((spr + 15) / 16 * 16) >= 3 * spr;
    const long fills = rows == 2 ? 448 : type == 14 ? (rows == 3 ? 320 : 192) : (rows == 3 ? 192 : 96);
    return (short_item && tiles >= fills && (rows >= 3 || count >= 3)) || (rows >= 3 && count == 1 && tiles >= 1536);
}

// Measured on MI355X (graph replay with the quantise launch, us: the kernel chosen otherwise / split / panel):
//   Q4_K 4096x4096     16 rows 10.4 /  9.5 / 14.7   64 rows 23.5 / 14.1 / 17.3  128 rows 24.1 / 18.9 / 18.2  192 rows 24.6 / 25.3 / 21.8
//   Q4_K 1024x14336    64 rows 60.6 / 25.0 / 43.1  512 rows 69.0 / 49.4 / 51.8
//   Q4_K q/k/v of 4096 16 rows 23.5 / 10.9 / 14.9   64 rows 23.7 / 17.3 / 17.4   96 rows 24.3 / 21.2 / 20.7  192 rows 32.7 / 35.1 / 27.0
//   Q4_K 8192x8192     16 rows 22.0 / 17.5 / 23.6   64 rows 41.5 / 29.8 / 28.1   96 rows 42.0 / 41.6 / 34.0  256 rows 60.7 / 86.4 / 56.6
//   Q4_K 14336x4096     8 rows 17.6 / 16.0 / 15.6   32 rows 23.8 / 21.3 / 18.1   64 rows 25.3 / 29.4 / 23.2  192 rows 49.5 / 68.5 / 47.2
//   gate/up of 14336   16 rows 24.9 / 28.8 / 22.6   32 rows 33.8 / 35.7 / 26.0   64 rows 36.8 / 50.1 / 34.3  128 rows 51.9 / 89.9 / 59.0
//   Q6_K 4096x14336    24 rows 41.4 / 25.1 / 63.8   64 rows 76.8 / 31.9 / 78.8  192 rows 91.7 / 69.8 / 82.5  384 rows  107 /  121 /  121
//   Q6_K 14336x4096     8 rows 23.9 / 22.6 / 22.2   64 rows 37.9 / 34.8 / 30.0  160 rows 65.9 / 72.3 / 59.6  512 rows  129 /  172 /  124
//   Q4_K, short inputs   9136x1280 at 59 rows 13.2 / 17.7 / 12.1   7008x2816 at 18 rows 17.6 / 12.2 / 13.7   720x1024 at 529 rows 11.9 / 10.1 / 12.3
//   Q6_K, short inputs   5408x256 at 143 rows 9.6 / 15.5 / 8.8   912x3584 at 481 rows 30.5 / 22.3 / 28.5   4096x1536 at 251 rows 17.8 / 23.7 / 16.8
// From 4096 inputs on: the panel kernel on tall matrices (768 16-row tiles: it then has a workgroup for nearly every CU at any
// row count) up to 64 rows; on others the split kernel, while its work (weight tiles x activation tiles) is small. Shorter
// inputs give the split kernel's four waves a few rounds each, the last one partly empty, beside its fixed share, so its limit
// there is in the time of its workgroups, T + 2 units each for T activation tiles: 1536 units (256 workgroups of four tiles, one
// a CU), 2560 where all rounds are full; for Q6_K, whose operands cost the panel kernel as much again, 3072 and 4608 (not at one
// super-block a row). Past that the panel kernel (Q6_K 3735x3072 at 171 rows and Q4_K at 96 rows, panel / split, 24.4 / 22.0, 15.0 /
// 14.2 within the limit; the shapes above past it). The panel kernel
// in turn loses to the tiled one on Q6_K once that fills the chip (33216x512 at 327 rows 42.8 / 49.1, 13392x256 at 459 rows 20.9 /
// 24.0, 26064x1024 at 302 rows 45.7 / 48.4) and on Q4_K of 32768 or more outputs of under 2048 inputs (33696x256 at 39 rows 10.3 / 12.1).
// Up to 16 rows one or two short weights stay on the small-M kernel, one pass for any of these row counts, except where a row
// is one full round or, Q6_K, nearly three (us, small-M / split: Q4_K 4304x512 at 8 rows 6.3 / 6.7, 4368x1536 at 16 rows 8.5 / 9.0,
// 4336x2560 at 10 rows 9.7 / 9.8; Q6_K 4448x1536 at 11 rows 9.5 / 10.2, 4256x1024 at 10 rows 8.9 / 7.6, 4416x768 at 9 rows 8.1 / 7.6);
// three weights take it one by one (864x2560 in all at 15 rows 16.1 / 8.3). Up to 8 rows Q4_K weights of 6400 and more outputs
// stay there too (8016x4352 at 8 rows 11.6 / 12.6, 8752x8448 at 5 rows 21.1 / 23.0, 6784x8448 16.0 / 16.4).
// Past 64 rows, where the split kernel starts to read the weights twice, Q4_K takes the least of three estimates in
// panel_cost's units: the panel kernel's; 0.55 (0.48 from 8192 inputs) for 256 of the split kernel's 16 x 16 tiles (4096x4096 at
// 96 / 192 rows 14.9 / 24.3, 1024x14336 at 400 rows 42.0); and those of mfma.hip, 4.5 + 6.3 for 256 workgroups of the wide
// kernel (gate/up of 14336 at 128 / 256 / 512 rows 52.6 / 88.7 / 154) or 6.8 + 2.5 for 256 of the 64-row kernel, which has more
// than two for each CU (q/k/v of 4096 at 331 / 512 rows 42.8 / 47.7, of 5120 at 331 rows 52.4; with fewer it lost to the panel
// kernel at every size). us, otherwise / so: q/k/v of 4096 at 160 / 200 / 331 rows 32.3 / 31.4 / 43.4, 23.9 / 27.3 / 39.1; 4096x4096 at
// 300 rows 33.0 / 28.0; gate/up of 14336 at 65 / 160 rows 49.2 / 78.7, 39.7 / 70.7. Q6_K takes the
// panel kernel where it has a workgroup for every CU and the split kernel's work has grown, except where the pair-wide kernel
// builds each operand once for 128 rows. Past the small-M kernel's input size (16384), and below the tiled kernel's rows (32),
// the alternative is the general kernel (8192x28672, that / split, at 2 rows 36.9 / 41.5, 3 rows 43.7 / 41.5, 16 rows 141 / 43.1). Very tall matrices at 5
// to 8 rows stay on the expert-stream kernel (128256x2048 at 6 rows 39.4, panel 42.4), and at 3 and 4 rows, where the multi-row
// decode kernel takes 64 (3 rows, panel 41.8), only a pair does.
// Weights that all carry their MFMA-ready copy (`prepared`, Q6_K): the tiled kernel that reads it has no operands to build. Up
// to 128 rows the split and panel kernels are the faster all the same (us, prepared / split / panel: 4096x14336 at 64 and 128
// rows 77.4 / 32.2 / -, 87.8 / 49.3 / -, 14336x4096 at 64 rows 39.0 / - / 30.8, 28672x8192 at 128 rows 147 / - / 134); past that the
// panel kernel loses (14336x4096 at 160 / 512 rows 54.2 / - / 59.5, 101 / - / 128, 8192x8192 at 512 rows 116 / - / 145) and the split
// kernel wins as long as it has one pass (1024x14336 at 512 rows 88.0 / 53.8 / -, 4096x4096 at 160 / 200 rows 31.3 / 27.6 / -,
// 31.6 / 32.6 / -, 2048x2048 at 256 / 400 rows 18.7 / 15.0 / -, 19.1 / 22.9 / -).
// `in` % 256 == 0; `tiles`: 16-row weight tiles of the `count` weights.
inline MidKernel mid_choice(int type, int in, int rows, long tiles, int count, bool prepared = false) {
    constexpr int kSmallMaxIn = 16384, kTiledMinRows = 32;
    if (rows < 2 || (int64_t)in * 64 >= (int64_t)1 << 32) return MidKernel::kNone;  // 32-bit offsets into a workgroup's rows
    const bool q6 = type == 14, tall = tiles >= 768;
    if (in > kSmallMaxIn && rows < kTiledMinRows)
        return rows == 2 ? MidKernel::kNone : tall ? MidKernel::kPanel : MidKernel::kSplit;
    const int spr = in / 256;
    if (rows <= 16) {
        if (tall) {
            if (rows <= 4) return rows >= 3 && tiles >= 1536 && count == 1 ? MidKernel::kPanel : MidKernel::kNone;
            return rows <= 8 && tiles >= 1536 ? MidKernel::kNone : MidKernel::kPanel;
        }
        if (count < 3) {
            const bool rounds_full = spr == 4 || (q6 && (spr == 3 || (spr > 10 && rows > 8)));
            if (spr < 16 && !rounds_full) return MidKernel::kNone;
            if (!q6 && rows > 4 && rows <= 8 && tiles >= 400) return MidKernel::kNone;
        }
        return MidKernel::kSplit;
    }
    const long subs = (rows + 15) / 16, work = tiles * subs, o_tiles = (tiles + 3) / 4;
    const long split_n = (subs + 3) / 4, split_t = (subs + split_n - 1) / split_n, wide_wgs = o_tiles * ((rows + 127) / 128);
    const bool is_short = spr < 16;
    const bool rounds_full = spr % 4 == 0;
    const long units = q6 && spr > 1 ? (rounds_full ? 4608 : 3072) : rounds_full ? 2560 : 1536;
    const bool split_fits = !tall && (is_short ? tiles * split_n * (split_t + 2) <= units : work <= (q6 ? 4096 : 2880));
    if (prepared && rows > 128)
        return split_fits && work <= (spr < 8 ? 1536 : is_short ? 2048 : 2560) ? MidKernel::kSplit : MidKernel::kNone;
    if (!q6 && rows > 64) {
        if (is_short && split_fits) return MidKernel::kSplit;
        int T;
        const double panel = rows <= 512 || work <= 8192 ? panel_cost(type, o_tiles, subs, &T) : 1e30;
        const double split = split_fits ? (in < 8192 ? 0.55 : 0.48) / 256 * (double)(tiles * split_n * split_t) : 1e30;
        const long grid64 = o_tiles * ((rows + 63) / 64);
        const double other = wide_wgs >= 448 ? 4.5 + 6.3 / 256 * (double)wide_wgs : grid64 > 512 ? 6.8 + 2.5 / 256 * (double)grid64 : 1e30;
        if (panel < split && panel < 0.97 * other) return MidKernel::kPanel;
        return split < other ? MidKernel::kSplit : MidKernel::kNone;
    }
    const bool pairwide = q6 && rows > 64 && wide_wgs >= 192 && wide_wgs <= 256;
    if (q6 && !is_short && rows > 64 && rows <= 512 && o_tiles * split_n >= 256 && work > 3584 && !pairwide)
        return MidKernel::kPanel;
    if (split_fits) return MidKernel::kSplit;
    if (!q6) return (tall || is_short) && !(spr < 8 && tiles >= 2048 && rows > 32) ? MidKernel::kPanel : MidKernel::kNone;
    if (pairwide) return MidKernel::kNone;
    if (is_short) return work <= (spr <= 2 || rows > 512 ? 8192 : 32768) ? MidKernel::kPanel : MidKernel::kNone;
    return tall && rows <= 512 ? MidKernel::kPanel : MidKernel::kNone;
}

// Whether the operand-ordered Q8_0 kernels (q8_mid.hip) take a batch that they support and the decode GEMV does not (rows * in <=
// 32768, up to 8 rows; at 8 rows, us, GEMV / these: 4096x4096 10.4 / 11.5, 14336x4096 19.7 / 20.7, 2048x2048 6.9 / 7.9; 4096x14336,
// which it does not take, at 4 rows 22.2 against the row kernel's 51.6). `out`: the outputs of the largest weight. Up to 16 rows
// of fewer than 512 inputs (32 rows of one block) the MFMA kernel's one-wave workgroups are done before a split has paid (320x96
// at 16 rows 4.5 / 5.0, 512x512 5.9 / 5.4, 502x32 at 17 rows 5.4 / 6.0). Rows of few blocks leave the panel kernel little to walk for its fixed share: with many outputs the 64 x 64
// tile kernel is faster (us, that / these: 14146x32 at 146 rows 8.4 / 9.4, 4736x64 at 473 rows 8.5 / 9.4, 32729x320 at 214 rows 24.1 /
// 27.2; 24718x672 at 179 rows 26.9 / 29.2, 18313x1216 at 375 rows 52.2 / 54.8; from 2048 inputs on
// these won at every size).
inline bool q8_mid_choice(int in, long out, int rows) {
    if (in < 512 && rows <= (in < 64 ? 32 : 16)) return false;
    const long outs = out * rows;
    return in < 512 ? outs <= 1l << 20 : in < 2048 ? outs <= 3l << 20 : true;
}

}  // namespace ovfq
