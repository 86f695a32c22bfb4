// Kernel-variant selection for the convolution entry points: a table of measured choices for
// known layer shapes (the analogue of the reference's tuned-schedule tables, python/tensorizer/
// tune.py:20-48, which map (ashape, bshape, strides) to a schedule index read from cpu-tune.log /
// gpu-tune.log), a heuristic for every other shape, and a per-process override.
#pragma once
#include "host.hpp"
#include "loaders.hpp"

namespace unit {

struct TileShape {
  int bx, by, bkb, waves, pf;  // waves per workgroup; pf: stages of global loads in flight
  bool ff;                     // all fragments of a stage read at once (small wave tiles)
  int kg;                      // k-groups sharing the output tile
  bool direct;                 // operands straight from global memory to registers (int8 NCHW16c)
  bool lds;                    // operand tiles shared through LDS by direct loads (prepared int8 NCHW16c weights only)
};

// index = variant id used by the tuning table and UNIT_AMD_CONV_VARIANT (1-based there)
constexpr TileShape kConvTiles[] = {
#define UNIT_CONV_VARIANT(ID, BX, BY, BKB, WX, WY, PF, FF, KG) {BX, BY, BKB, (WX) * (WY) * (KG), PF, FF, KG, false, false},
#define UNIT_CONV_DIRECT(ID, TX, TY, KG, D) {(TX) * 32, (TY) * 32, 32, KG, (D) % 16, false, KG, true, false},
#define UNIT_CONV_LDS(ID, TX, TY, WX, WY, KG, KS, NST) \
  {(TX) * (WX) * 32, (TY) * (WY) * 32, 32 * (KS), (WX) * (WY) * (KG), NST, false, KG, false, true},
#include "conv_variants.def"
#undef UNIT_CONV_LDS
#undef UNIT_CONV_DIRECT
#undef UNIT_CONV_VARIANT
};
constexpr int kNumConvTiles = sizeof(kConvTiles) / sizeof(kConvTiles[0]);

struct ConvPlan {
  int variant;
  int splits;
  // Channel tiles per panel of the workgroup -> tile walk (0: all of them).  An XCD's workgroups
  // cover whole panels, so 0 makes every XCD read all weights and a slice of the pixels, while
  // a small panel gives each XCD a slice of the weights and all pixels: the better choice is the
  // one that pulls fewer bytes into the 8 L2s, which start cold at every kernel.
  int panel;
  bool halves = false;  // variant 68 of the fp16 operator on blocked weights: DirectShape's HALVES
};

struct TunedConv {
  int npix, K, C, KH, KW, sh;  // key
  int variant, splits, panel;
};

// Heuristic for shapes the table does not hold, distilled from the tuning runs: output-bound
// layers (few input channels, many pixels) want 64..128-pixel tiles of 64 channels with many
// workgroups in flight; long reductions want the 128-channel tiles with two stages of loads in
// flight; the 256 x 256 tiles only pay when they still give every CU several workgroups.
inline ConvPlan heuristic_plan(const unit_conv_desc *d, int npix, int kbytes, bool allow_split, bool direct_ok,
                               bool staged_too = false) {
  const int K = d->K;
  const bool strided = d->sh * d->sw > 1;
  const bool k128 = kbytes % 128 == 0;
  const auto tiles = [&](int bx, int by) { return (long)ceil_div(K, bx) * ceil_div(npix, by); };
  if (direct_ok) {
    // NCHW16c: the direct kernels won every tuned layer but the widest outputs.  One wave per
    // 64 x 64 tile when the tiles alone fill the SIMDs, else k-groups (4, 8) to put about a
    // thousand waves on the chip; the smallest problems use 64 x 32 (fp16: 32 x 64) tiles.
    const long t64 = tiles(64, 64);
    int v, panel = 0;
    // Long reductions on few output pixels: eight waves share a tile of one 32-channel block, which gives such a layer
    // twice the workgroups of 64 x 32 tiles and each wave half the k-steps in a row (its time is a chain of load
    // latencies, not a rate).  While 32 x 32 tiles are at most one per CU: u8 1536 -> 720, 3 x 3 on 17 x 14, 19.7 -> 10.6
    // us; fp16 1168 -> 32, 5 x 5 on 27 x 17, 85 -> 43; the 137 such rows of the tables 901 -> 751 in all.  Below 20
    // k-steps the sum of eight partial tiles costs what it gains (18: 4.36 against 4.34 us), in fp16 up to 24, all of
    // which the four six-deep waves of the tiles below have in flight at once (on 20 - 24 steps eight waves took 1.03 -
    // 1.14 times as long, prepared 352 -> 560, 1 x 1 stride 2 on 16 x 33, 3.51 -> 3.94; on 25 - 60 0.81 - 1.07 and
    // prepared 0.90 - 1.04 but for 1 x 1 at stride 2, up to 1.14; int8 0.92 - 1.05 up to 24, 0.79 - 0.99 past them).  16
    // fp16 channels at stride 1, where it was 1.03 - 1.06, keep 20: the shortest rings are tested there.  Above 256 tiles
    // the second round does (342 of them: 10.6 -> 8.0, 555: 22.0 -> 21.0, 720: 49.2 -> 51.1).  Up to 32 channels a
    // 64-channel tile is half padding: 32 x 64 tiles there (480 -> 32 on 76 x 72: 10.6 -> 7.0).  The eight waves' scratch
    // and tile leave the tap table less of the LDS than the four-wave tiles below do (with 4-channel blocks, a k-step per
    // window row, 7352 rows against 8528): up to 4096 steps, 64 KiB of table, all of them fit.
    const int ksteps = kbytes / 32, table_steps = d->cb == 4 ? kbytes / (4 * d->KW) : ksteps;
    const int least = allow_split || (K <= 16 && !strided) ? 20 : 25;
    if (ksteps >= 20 && table_steps <= 4096) {
      if (tiles(32, 32) <= 256) {
        if (ksteps >= least) return ConvPlan{82, 1, 4};
      } else if (K <= 32 && tiles(32, 64) <= 384) {
        return ConvPlan{83, 1, 0};
      }
    }
    if (allow_split) {  // the int8 operator; distilled from the tuner's choices on cold operands (batch 1 .. 256)
      const int nsteps = kbytes / 32;
      const bool wide = K % 128 == 0;  // 128-channel tiles
      if (t64 < 196)
        v = 60;  // 64 x 32 tiles, four k-groups, six deep
      else if (t64 < 392)
        v = nsteps >= 36 ? 63 : 52;  // 64 x 64, four k-groups: six deep for long reductions, else four
      else if (t64 < 784)
        v = nsteps <= 4 ? 70 : (nsteps <= 8 ? 50 : (nsteps < 72 || !wide ? 52 : 56));
      else if (t64 < 1568)
        v = nsteps <= 4 ? 70 : (nsteps <= 16 ? 71 : 68);  // one wave per tile: 2 / 3 deep at four waves per SIMD, then 6 deep
      else if (t64 < 3136)
        v = nsteps <= 8 ? 70 : (wide ? 54 : 71);  // 128-channel tiles while they still give every SIMD a wave
      else
        v = nsteps <= 36 ? 70 : 68;
      // Eight or more channel tiles: panels of four, so that an XCD's L2 holds a slice of the weights for all its
      // pixels; not when the stride skips input pixels (the data is then the sparse operand), nor when a long
      // reduction already keeps a large problem's weights hot.
      if (K >= 512 && !strided && (nsteps <= 16 || t64 < 784)) panel = 4;
    } else {  // the fp16 operator (a k-step is one tap of 16 channels), same source
      const int nsteps = kbytes / 32;
      const bool wide = K % 128 == 0;
      // Weights in the reference's layout (staged_too), whose fragments cost the direct kernels twenty instructions of
      // transposition each: a wave alone on its SIMD waits for them.  The lines lie where the waves of a tile size leave
      // SIMDs without a second wave; us of the tiles for prepared weights / of these:
      //   long reductions, from 196 tiles of 256 x 256 up: staged, both operands shared through LDS (at 192 46.4 / 42.0; 160,
      //   3 x 3 192 -> 128 on 56 x 56, batch 14, the direct kernel takes 32.2 where staged tiles take 41.7);
      //   up to one 64 x 128 tile per CU: four k-groups on them (64 -> 352, 5 x 5 on 36 x 38, batch 4, 22.6 / 11.6; 112 ->
      //   368, 3 x 3 on 76 x 64 15.4 / 9.2; 432 -> 224, 3 x 3 on 74 x 61 29.1 / 20.3), with 9 - 24 k-steps and no more than
      //   392 tiles of 64 x 64 rather on 64 x 32 (32 -> 608, 3 x 3 on 20 x 26, batch 4, 7.9 / 5.4);
      //   then two k-groups, six deep, to three tiles per CU (144 -> 2048, 3 x 3 on 22 x 30, batch 2, 21.4 / 15.3; 208 -> 400, 3 x 3 on
      //   36 x 57, batch 3, 25.5 / 19.0; 32 channels, half of the tile padding, 10.6 / 12.1: not these; 780 tiles 25.2 / 27.9);
      //   up to 1568 tiles, where 128-channel tiles or staged ones ran, one wave per tile or, past 90 k-steps and with two of them per CU, 64 x 128 (512 ->
      //   128, 1 x 1 on 28 x 28, batch 32, 14.5 / 9.8; 128 -> 1312, 5 x 5 on 14 x 20, batch 15, 38.2 / 35.4);
      //   from 1568 tiles on four deep (64 -> 32, 3 x 3 on 65 x 83, batch 27, 19.9 / 16.9; 512 -> 608, 1 x 1 on 86 x 60, batch 3,
      //   23.5 / 20.8), but from 10000 tiles and up to 18 k-steps three (32 -> 1648, 3 x 3 stride 2 on 80 x 112, batch 12, four deep
      //   64.3, three 60.7, six 61.1; 16 -> 1328, 3 x 3 on 80 x 111, batch 5 48.9 and 45.7).
      // Where these tiles are slower than with eight 16-bit loads per fragment, us then / these tiles / now:
      //   up to 32 channels, half of a 64-channel tile padding: 32 x 64 tiles of four groups (144 -> 32, 3 x 3 on 105 x 66, batch 5
      //   16.7 / 18.4 / 9.9; 496 -> 16, 5 x 5 on 30 x 41, batch 37 141 / 151 / 60; 512 -> 32 on 74 x 97, batch 11 71.7 / 77.3 / 41.6);
      //   few tiles, but more than 256 of 64 x 128: two groups there too (160 -> 1264, 3 x 3 stride 2 on 26 x 22, batch 13 18.3 /
      //   20.0 / 16.8);
      //   1025 to 1280 tiles, hardly more than one wave per SIMD, and 48 steps or more: the eight loads (128 -> 1904, 3 x 3 on
      //   16 x 15, batch 13 22.5 / 23.8; 448 -> 112, 3 x 3 on 55 x 54, batch 12 62.4 / 66.1; 40 - 45 steps 0.98 - 1.01 of them, 1287
      //   tiles 0.96);
      //   9 - 16 k-steps on 784 to 1568 tiles: one wave per tile there too (256 -> 1792 on 12 x 8, batch 24 9.5 / 9.8 / 7.8);
      //   up to 8 k-steps the stores decide: three deep at four waves per SIMD below 4000 tiles (64 -> 912 on 18 x 17, batch 45 12.0 /
      //   12.7 / 12.0; 80 -> 1520 on 20 x 16, batch 26 12.8 / 13.2 / 12.2; on 25 others 0.76 - 0.98 of then), six deep from 7000
      //   tiles and up to 4 steps (16 -> 240 on 99 x 112, batch 17 32.2 / 34.4 / 32.9; 64 -> 1088 on 81 x 112, batch 3 24.3 / 25.4 /
      //   24.1).  Left: 128 -> 1040 on 34 x 50, batch 6 11.8 / 12.3 / 12.1.
      if (staged_too) {
        if (nsteps >= 32 && K % 256 == 0 && tiles(256, 256) >= 196) return ConvPlan{0, 1, 0};
        if (nsteps <= 8 && t64 >= 1568) {
          if (t64 < 4000 && nsteps < 8) return ConvPlan{71, 1, 0};
          if (t64 >= 7000 && nsteps <= 4) return ConvPlan{68, 1, 0};
        }
        if (t64 > 256 && nsteps > 8) {
          if (t64 < 392 && nsteps <= 24) return ConvPlan{60, 1, 0};
          if (tiles(64, 128) <= 256 && nsteps > 24) return ConvPlan{59, 1, 0};
          if (K <= 32 && nsteps > 24 && t64 < 1568) return ConvPlan{61, 1, 0};
          if (t64 >= 392 && t64 <= 768 && nsteps > 24) return ConvPlan{67, 1, 0};
          if (t64 > 1024 && t64 <= 1280 && nsteps >= 48) return ConvPlan{68, 1, 0, true};
          if (t64 >= 784 && t64 < 1568) {
            if (nsteps >= 90 && tiles(64, 128) <= 512) return ConvPlan{59, 1, 0};
            return ConvPlan{nsteps > 36 ? 68 : 50, 1, 0};
          }
          if (t64 >= 10000 && nsteps <= 18) return ConvPlan{65, 1, 0};
          if (t64 >= 1568 && (!wide || nsteps > 36)) return ConvPlan{50, 1, 0};
        }
      }
      if (t64 < 196)
        v = 60;
      else if (t64 < 392)
        v = nsteps <= 8 ? 50 : 52;
      else if (t64 < 784)
        v = nsteps <= 8 ? 50 : (nsteps <= 36 || !wide ? 68 : 56);
      else if (t64 < 1568)
        v = nsteps <= 8 ? 65 : (!wide ? 68 : (nsteps <= 36 ? 54 : 55));
      else
        v = nsteps <= 8 ? 50 : (wide ? 54 : 68);
    }
    return ConvPlan{v, 1, panel};
  }
  int v;
  if (K % 128 != 0) {  // 64-channel tiles
    if (kbytes <= 64 || !k128)
      v = tiles(64, 256) >= 1024 ? 20 : (tiles(64, 128) >= 512 ? 10 : 19);
    else
      v = tiles(64, 256) >= 1024 ? 4 : (tiles(64, 128) >= 512 ? 17 : 19);
  } else if (!k128) {  // reduction is an odd number of 64-byte stages
    v = (K % 256 == 0 && tiles(256, 256) >= 512) ? 1 : (tiles(128, 256) >= 512 ? 3 : (tiles(128, 128) >= 256 ? 24 : 19));
  } else {
    v = (K % 256 == 0 && tiles(256, 256) >= 512) ? 0 : (tiles(128, 256) >= 512 ? 2 : (tiles(128, 128) >= 384 ? 18 : 23));
  }
  // k-splits accumulate with device-scope atomics, which this part executes at the memory side
  // (each XCD has its own L2): they only pay when the output is tiny and the reduction long
  // (batch-1 layers with a handful of tiles)
  int splits = 1;
  if (allow_split) {
    const TileShape &t = kConvTiles[v];
    const long nt = tiles(t.bx, t.by);
    const int nk = ceil_div(kbytes, t.bkb);
    while (nt * splits < 96 && nk / (splits * 2) >= 4 && splits < 8) splits *= 2;
  }
  return ConvPlan{v, splits, 0};
}

// The measured choice for this shape, or null.
inline const TunedConv *tuned_row(const unit_conv_desc *d, int npix, const TunedConv *table, int ntable, bool direct_ok, bool lds_ok) {
  // UNIT_AMD_CONV_NOTABLE=1: heuristic only (the tuner measures it as the baseline)
  if (tuning_override("UNIT_AMD_CONV_NOTABLE") > 0) return nullptr;
  for (int i = 0; i < ntable; ++i) {
    const TunedConv &e = table[i];
    // the tables were tuned on square strides without dilation; a direct choice needs a window the direct
    // kernels can run, otherwise the heuristic's (staged) choice stands
    if (e.npix == npix && e.K == d->K && e.C == d->C && e.KH == d->KH && e.KW == d->KW && e.sh == d->sh &&
        d->sw == d->sh && d->dh == 1 && d->dw == 1 && (direct_ok || !kConvTiles[e.variant].direct) &&
        (lds_ok || !kConvTiles[e.variant].lds))
      return &e;
  }
  return nullptr;
}

inline ConvPlan plan_conv(const unit_conv_desc *d, int npix, int kbytes, const TunedConv *table, int ntable,
                          bool allow_split, bool direct_ok, bool staged_too = false, bool lds_ok = false) {
  ConvPlan p = heuristic_plan(d, npix, kbytes, allow_split, direct_ok, staged_too);
  if (const TunedConv *e = tuned_row(d, npix, table, ntable, direct_ok, lds_ok)) p = ConvPlan{e->variant, e->splits, e->panel};
  // A direct variant whose k-groups park one float tile each can outgrow the LDS on very deep reductions (the tap
  // table follows the tiles): the one-wave six-deep kernel of the same family always fits.
  if (!allow_split && kConvTiles[p.variant].direct && kConvTiles[p.variant].kg > 1) {
    const TileShape &t = kConvTiles[p.variant];
    const long tile = (long)t.bx * t.by * 4 + t.bx * 4, scratch = 32 * 144 + 128;  // DirectShape: TILE + WSUM, kScratch
    if (t.kg * (scratch + tile) + (long)(kbytes / 32) * 8 > kMaxLds) p = ConvPlan{68, 1, p.panel};
  }
  const int ov = tuning_override("UNIT_AMD_CONV_VARIANT"), os = tuning_override("UNIT_AMD_CONV_SPLITK");
  if (ov > 0 && ov <= kNumConvTiles) p.variant = ov - 1, p.halves = false;
  if (os > 0) p.splits = os;
  const int op = tuning_override("UNIT_AMD_CONV_PANEL");
  if (op > 0) p.panel = op;
  if (!allow_split) p.splits = 1;
  // the LDS-shared variants exist for prepared weights with 16-channel blocks only: elsewhere their ids run the heuristic's choice
  if (kConvTiles[p.variant].lds && !lds_ok) {
    const ConvPlan h = heuristic_plan(d, npix, kbytes, allow_split, direct_ok, staged_too);
    p.variant = h.variant, p.halves = h.halves;
    if (!allow_split) p.splits = 1;
  }
  return p;
}

}  // namespace unit
