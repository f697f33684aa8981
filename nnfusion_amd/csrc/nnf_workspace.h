// Scratch-memory sizes of the launcher entry points and the tile plan they follow: pure host
// arithmetic, shared by the library (nnf_*_workspace_bytes, the GEMM dispatcher) and by the emitters,
// which reserve the scratch tensor at compile time.  Nothing here may depend on the device at hand.
#pragma once

#include <math.h>
#include <stddef.h>
#include <stdint.h>

#include <initializer_list>

namespace nnf
{
    namespace workspace
    {
        inline size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

        // ---- tile plan of the W8A8 MFMA GEMM (w8a8_gemm_dl.hip) ----------------------------------------
        enum GemmTile
        {
            GEMM_TILE_BIG = 0,   // 256 x 256 outputs
            GEMM_TILE_MID = 1,   // 128 x 128
            GEMM_TILE_SMALL = 2, //  64 x 256
            GEMM_TILE_TINY = 3,  //  32 x 256 (not built for W8A8)
            GEMM_TILE_TALL = 4,  // 256 x 128 (W8A8 only: fills the chip where 256 x 256 tiles leave CUs idle)
            // whole tiles of W8A8 that only the launch chooses (w8a8_whole_tile)
            GEMM_TILE_256_192 = 5,
            GEMM_TILE_192_256 = 6,
            GEMM_TILE_128_256 = 7,
            GEMM_TILE_192_128 = 8,
            GEMM_TILE_128_192 = 9,
        };
        struct GemmPlan
        {
            int tile = GEMM_TILE_BIG;
            int splits = 1; // K ranges; > 1 (and always for the small and tiny tiles): partial sums + a reduction pass
            bool reduce_pass = false;
        };
        constexpr int PLAN_CUS = 256; // the plan is made for the CU count of an MI355X

        inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

        // Estimated run time (seconds) of one tile shape and split count, from rates measured on an MI355X with
        // N(0,1) activations (the GEMMs are power bound: ~950 / 700 / 450 TFLOP/s for the three tile shapes when
        // every CU has a workgroup, and a CU runs faster when fewer are busy: hence the square root), ~6 TB/s for
        // the partial sums (written, then read by the reduction pass) and ~3 us for the second launch.
        // w8a8: the same tiles on the int8 matrix cores (~1870 / 1450 / 900 TOP/s, 1700 for 256 x 128; its weight bytes
        // differ too, but a memory-bound W8A8 shape is decided by the partial-sum term either way)
        inline double estimate_gemm(int M, int N, int K, bool gate, int tile, int splits, bool w8a8)
        {
            const int bm = tile == GEMM_TILE_BIG || tile == GEMM_TILE_TALL ? 256 : tile == GEMM_TILE_MID ? 128 : tile == GEMM_TILE_SMALL ? 64 : 32;
            const int bn = tile == GEMM_TILE_BIG ? (gate ? 128 : 256) : tile == GEMM_TILE_MID || tile == GEMM_TILE_TALL ? 128 : 256;
            static const double rates[2][5] = {{950e12, 700e12, 450e12, 300e12, 800e12}, {1870e12, 1450e12, 900e12, 600e12, 1700e12}};
            const double rate = rates[w8a8 ? 1 : 0][tile];
            const int tiles_m = ceil_div(M, bm), tiles_n = ceil_div(N, bn);
            const double blocks = (double)tiles_m * tiles_n * splits;
            const double rounds = (double)(((long long)blocks + PLAN_CUS - 1) / PLAN_CUS);
            const double util = blocks / (rounds * PLAN_CUS);
            const double n_total = (gate ? 2.0 : 1.0) * N;
            const double flops = 2.0 * tiles_m * bm * n_total * K; // whole tile rows are computed
            double t = flops / (rate * sqrt(util));
            const double weight_time = n_total * K / 2.0 / 4e12;
            if (t < weight_time)
                t = weight_time;
            if (splits > 1 || tile == GEMM_TILE_SMALL || tile == GEMM_TILE_TINY)
                t += 2.0 * splits * M * n_total * 4.0 / 6e12 + 3e-6;
            return t;
        }

        // N: output columns.  forced_tile >= 0 / forced_splits > 0 override the choice (a caller's plan argument).
        inline GemmPlan plan_gemm(int M, int N, int K, bool gate, bool w8a8, int forced_tile, int forced_splits)
        {
            static const int split_options[] = {1, 2, 3, 4, 6, 8, 12, 16};
            const int G = K / 128;
            GemmPlan best;
            double best_t = -1.0;
            for (int tile = GEMM_TILE_BIG; tile <= GEMM_TILE_TALL; ++tile)
            {
                // (forced_tile -2: 256-row tiles, their width left to the plan)
                if (tile == GEMM_TILE_TALL && !w8a8)
                    continue;
                if (forced_tile >= 0 ? tile != forced_tile
                    : forced_tile == -2 ? (tile != GEMM_TILE_BIG && tile != GEMM_TILE_TALL)
                                     : (((tile == GEMM_TILE_BIG || tile == GEMM_TILE_TALL) && M <= 128) ||
                                        (tile == GEMM_TILE_SMALL && M > 64) || (tile == GEMM_TILE_MID && M <= 64) ||
                                        (tile == GEMM_TILE_TINY && (M > 32 || w8a8))))
                    continue;
                for (int s : split_options)
                {
                    // every split keeps at least four groups (eight K steps)
                    if (forced_splits > 0 ? s != 1 : (s > 1 && G / s < 4))
                        continue;
                    const int splits = forced_splits > 0 ? (forced_splits < G ? forced_splits : G) : s;
                    const double t = estimate_gemm(M, N, K, gate, tile, splits, w8a8);
                    if (best_t < 0.0 || t < best_t)
                    {
                        best_t = t;
                        best.tile = tile;
                        best.splits = splits;
                    }
                }
            }
            best.reduce_pass = best.splits > 1 || best.tile == GEMM_TILE_SMALL || best.tile == GEMM_TILE_TINY;
            return best;
        }
        inline GemmPlan plan_w8a8_gemm(int M, int N, int K, int forced_tile = -1, int forced_splits = 0)
        {
            return plan_gemm(M, N, K, false, true, forced_tile, forced_splits);
        }
        // More than 128 rows of W8A8: whole tiles of another shape in place of `planned`, where the estimates say they are more than 2 %
        // faster.  Tiles of 256 x 128 and 128 x 128 alone leave up to half of the CUs idle in the last round: 3000 x 6144 x 5504 is 576 of
        // 256 x 128, 2.25 rounds in the time of three, and 768 of 128 x 192, three rounds of half the work.  Microseconds, fitted to 520
        // products of 129 .. 4096 rows (N = 256 .. 16384, K = 512 .. 16384, weights from memory, every shape timed; 10 % rms): rounds of
        // tiles x start, and per 128 of K a step a round and up to `load` with the CUs busy.  Over ranges of K: the plan's own estimate, which is
        // a tenth too long.  161 of the 520 are on another tile by it, 1.16 x in the geometric mean, the slowest of them 0.98; the fastest shape of
        // each would gain all of them 1.048, this gains 1.046.  (192 x 192, on
        // four wavefronts, is the fastest for three.)
        // The row of 128 x 128 is of stages of 128, one workgroup a CU; below K = 2560 the launch takes stages of 64 and two a CU, whose short
        // loops cover for each other.  There 128 x 256 tiles are estimated ahead a little too soon: 300 products whose columns are a multiple of
        // eight: in one round of them 0.98 at K = 512, 1.00 - 1.02 at 640, 1.05 at 768, 1.04 at 896, 1.06 - 1.11 above; in two 0.92 at 512, 0.95,
        // 0.98, 0.97 and 0.96 at 640 .. 1024, 1.00 at 1152, 1.03 at 1280 and up to 1.06 above (2143 x 7352 x 512 19.2 / 20.6 us, 1549 x 9984 x
        // 1152 31.3 / 31.8).  Other columns are stored an element at a time, with which fewer, larger tiles get along better: 1.11 - 1.17 at every K.
        inline int w8a8_whole_tile(int M, int N, int K, const GemmPlan& planned)
        {
            struct Cost
            {
                int tile, rows, cols;
                double start, step, load;
            };
            static const Cost costs[] = {
                {GEMM_TILE_BIG, 256, 256, 9.77, 1.109, 0.749},     {GEMM_TILE_TALL, 256, 128, 6.50, 0.738, 0.303},
                {GEMM_TILE_MID, 128, 128, 4.48, 0.359, 0.186},     {GEMM_TILE_256_192, 256, 192, 7.72, 1.036, 0.493},
                {GEMM_TILE_192_256, 192, 256, 7.80, 1.036, 0.438}, {GEMM_TILE_128_256, 128, 256, 6.61, 0.737, 0.299},
                {GEMM_TILE_192_128, 192, 128, 5.62, 0.595, 0.207}, {GEMM_TILE_128_192, 128, 192, 7.99, 0.459, 0.247},
            };
            if (M <= 128 || K < 512 || planned.tile == GEMM_TILE_SMALL || planned.tile == GEMM_TILE_TINY)
                return planned.tile;
            const long long mids = (long long)ceil_div(M, 128) * ceil_div(N, 128);
            if (planned.tile == GEMM_TILE_MID && planned.splits == 1 && (N & 7) == 0 && K < (mids > 2 * PLAN_CUS ? 1152 : 768))
                return planned.tile;
            const double steps = K / 128;
            double best = planned.splits > 1 ? 0.9e6 * estimate_gemm(M, N, K, false, planned.tile, planned.splits, true) : -1.0;
            const auto estimate = [&](const Cost& c) {
                const long long tiles = (long long)ceil_div(M, c.rows) * ceil_div(N, c.cols), rounds = (tiles + PLAN_CUS - 1) / PLAN_CUS;
                const double last = (double)(tiles - (rounds - 1) * PLAN_CUS) / PLAN_CUS;
                return rounds * (c.start + steps * c.step) + (rounds - 1 + last) * steps * c.load;
            };
            for (const Cost& c : costs)
                if (best < 0.0 && c.tile == planned.tile)
                    best = estimate(c);
            best *= 0.98;
            int tile = planned.tile;
            for (const Cost& c : costs)
                if (c.tile >= GEMM_TILE_256_192)
                {
                    const double t = estimate(c);
                    if (t < best)
                        best = t, tile = c.tile;
                }
            return tile;
        }
        // What the launch runs: that plan, but for other whole tiles (above) where the caller fixed nothing, and for 64 x 256 tiles, which write their results themselves where K is in one range
        // and whose ranges (never more than the plan's, whose scratch memory is what callers bring) follow a fit of measured
        // times: per round of tiles 3.6 us, per 128 of K 0.47 and up to 0.64 with the CUs busy; ranges 2 us, 0.28 each and their
        // sums at 10 TB/s (1482 timings, 17 .. 64 rows, 64 %: within 3 %).  33 .. 64 rows: 7 % faster in the geometric mean of
        // 66 products, 58 x 12672 x 512 10.1 -> 7.9 us.
        inline GemmPlan plan_w8a8_launch(int M, int N, int K, int forced_tile, int forced_splits)
        {
            GemmPlan p = plan_w8a8_gemm(M, N, K, forced_tile, forced_splits);
            if (p.tile != GEMM_TILE_SMALL)
            {
                const int tile = forced_tile == -1 && forced_splits <= 0 ? w8a8_whole_tile(M, N, K, p) : p.tile;
                if (tile != p.tile)
                    p.tile = tile, p.splits = 1, p.reduce_pass = false;
                return p;
            }
            static const int split_options[] = {1, 2, 3, 4, 6, 8, 12, 16};
            double best = -1.0;
            const int planned = p.splits;
            for (int s : split_options)
            {
                if (forced_splits > 0 || s > planned)
                    break;
                const long long grid = (long long)ceil_div(M, 64) * ceil_div(N, 256) * s, rounds = (grid + PLAN_CUS - 1) / PLAN_CUS;
                const double last = (double)(grid - (rounds - 1) * PLAN_CUS) / PLAN_CUS, steps = ceil_div(K / 128, s);
                const double t = 3.6 * rounds + steps * (0.47 * rounds + 0.64 * (rounds - 1 + last)) +
                                 (s > 1 ? 2.0 + 0.28 * s + (double)s * M * N * 8.0 / 1e7 : 0.0);
                if (best < 0.0 || t < best)
                    best = t, p.splits = s;
            }
            p.reduce_pass = p.splits > 1;
            return p;
        }
        // a caller's tile_rows / tile_cols as a forced tile of plan_w8a8_gemm (-1: none; -2: 256-row tiles of the
        // plan's own width)
        inline int w8a8_forced_tile(int tile_rows, int tile_cols)
        {
            if (tile_rows == 256)
                return tile_cols == 256 ? GEMM_TILE_BIG : tile_cols == 128 ? GEMM_TILE_TALL : -2;
            return tile_rows == 128 ? GEMM_TILE_MID : tile_rows == 64 ? GEMM_TILE_SMALL : -1;
        }
        inline size_t gemm_partial_bytes(int M, int N, bool gate, const GemmPlan& p)
        {
            return p.reduce_pass ? align256((size_t)p.splits * M * (gate ? 2 : 1) * N * sizeof(float)) : 0;
        }

        // ---- plan of the fp16 x int4 tile GEMM (w4a16_gemm_sk.h) ----------------------------------------------
        // Tiles of tile_rows x 256 weight rows (SiLU-gate: 128 gate + 128 up rows, i.e. 128 output columns) or, for
        // the products without SiLU-gate, tile_rows x 128; the
        // (tile, superstep of 256 k) units of the whole product are split evenly over `grid` workgroups, at most one per CU (or
        // one per tile: plan_w4a16_tiles chooses between numbers of workgroups and tile shapes).
        // A tile whose units belong to more than one workgroup is summed through the workspace: slots of
        // tile_rows x 256 fp32; workgroup v parks the first segment of its range in slot v and a later one in slot
        // grid + v; a second launch adds them up.
        struct SkPlan
        {
            int tile_rows = 0; // 32, 64, 128 or 256
            int tile_weight_rows = 256; // weight rows of a tile: 256, 128 (narrow tiles: plain product only) or 192 (whole tiles of 128 rows: plan_w4a16_192)
            int tiles_m = 0, tiles_n = 0;
            int supersteps = 0; // per tile: ceil(K / 256)
            long long units = 0;
            int grid = 0;
            int slots = 0;     // 0: every tile belongs to one workgroup (no workspace, no second launch)
            size_t bytes() const { return (size_t)slots * tile_rows * tile_weight_rows * sizeof(float); }
            // Synchronisation words for the one-launch form: two for RMSNorm's rstd[] computed inside the launch, then
            // two per tile (workgroups that share a tile add its parts up themselves).  0: no tile is shared and (rms)
            // there is no RMSNorm
            size_t sync_bytes(bool rms = false) const { return (slots || rms) ? ((size_t)tiles_m * tiles_n + 1) * 2 * sizeof(unsigned) : 0; }
        };
        // Tile shape.  What the caller fixes (forced_rows 32 / 64 / 128 / 256, forced_cols 128 / 256) is kept, the rest
        // is chosen by M and N (measured at N = K = 8192 and on the Llama shapes, the candidates in turns in one process):
        // 256 x 256 tiles touch every weight once per 256 rows and are the fastest from about 1500 rows on.  Below, every
        // output tile is shared by several workgroups and what a workgroup parks counts: up to 128 rows 128 x 128 tiles
        // (64 x 128 up to 64); above, 256 x 128 where M fills the 256-row tiles (an even number of 128-row blocks, or
        // less than a seventh of the rows wasted: M = 144 .. 256 40.8 - 42.2 us against 42.8 - 44.3 on 128 x 128 tiles,
        // M = 896 116 against 144) and 128 x 256 where it does not (an odd number of blocks: M = 288 .. 384 61.3 - 62.7
        // against 63.9 - 66.1, M = 576 .. 640 96 against 104); 128 x 128 again where 256-row tiles would leave fewer
        // than 64 tiles (N = 4096 at M = 192 .. 256).  SiLU-gate needs the gate | up halves of a 256-row weight tile;
        // 32-row tiles exist 256 wide only.
        inline void sk_tile_shape(int M, int N, bool gate, int forced_rows, int forced_cols, int& rows, int& cols)
        {
            const bool rows_forced = forced_rows == 32 || forced_rows == 64 || forced_rows == 128 || forced_rows == 256;
            if (rows_forced)
            {
                rows = forced_rows;
                cols = (forced_cols == 128 && !gate && rows != 32) ? 128 : 256;
                return;
            }
            cols = 256;
            if (gate || M <= 32 || M > 1536)
            {
                rows = M <= 32 ? 32 : M <= 64 ? 64 : M <= 1536 ? 128 : 256;
                return;
            }
            if (forced_cols == 256)
            {
                const int padded = ceil_div(M, 256) * 256;
                rows = M <= 64 ? 64 : M <= 128 ? 128 : ((padded - M) * 8 <= M ? 256 : 128);
                return;
            }
            cols = 128;
            rows = M <= 64 ? 64 : 128;
            if (M <= 128)
                return;
            const int blocks = ceil_div(M, 128), padded = ceil_div(M, 256) * 256;
            if ((blocks & 1) == 0 || (padded - M) * 7 <= padded)
            {
                if ((padded / 256) * ceil_div(N, 128) >= 64)
                    rows = 256;
            }
            else if (forced_cols != 128)
                cols = 256;
        }
        // tiles_n column tiles, `per_tile` units of K per tile, at least `min_units` units per workgroup (unless forced);
        // forced_grid: 0 = the plan's own choice
        inline SkPlan plan_sk(int M, int tiles_n, int per_tile, int min_units, int num_cu, int forced_tile_rows, long long forced_grid)
        {
            SkPlan p;
            const int rows = forced_tile_rows;
            p.tile_rows = rows;
            p.tiles_m = ceil_div(M, rows);
            p.tiles_n = tiles_n;
            const int G = per_tile;
            p.supersteps = G;
            p.units = (long long)p.tiles_m * p.tiles_n * G;
            long long grid = p.units / min_units < 1 ? 1 : p.units / min_units;
            if (grid > num_cu)
                grid = num_cu;
            // Whole tiles, one workgroup each, where the tiles fill at least half of the CUs and the CUs left idle cost
            // less than what sharing tiles costs (parts parked and added up, a second start of the pipeline in the
            // middle of the launch: about 30 us, some seven to eleven units of 256 k).  Measured against the even split
            // on 172 tiles of 128 x 256 (gate | up, M = 256, K = 4096) 76 -> 71 us, on 172 of 256 x 128 (M = 256,
            // N = 22016) 65 -> 55, 160 tiles (M = 640, N = 8192, K = 4096) 64 -> 52, 128 (M = 512, K = 2048) 33 -> 26,
            // 192 at K = 8192 111 -> 105; with 86 or 112 tiles (a third, 44 % of the CUs) the even split stays 4-10 %
            // faster.
            const long long tiles = (long long)p.tiles_m * p.tiles_n;
            if (tiles <= num_cu && 2 * tiles >= num_cu && (long long)G * (num_cu - tiles) <= 11ll * num_cu)
                grid = tiles;
            if (forced_grid > 0)
                grid = forced_grid < p.units ? forced_grid : p.units;
            p.grid = (int)grid;
            // Share v is the units [v * units / grid, (v + 1) * units / grid), rounded down.  In lowest terms a share is T / W tiles (W:
            // grid, T: tiles, over their common factor).  Share boundaries that are not tile boundaries exist unless W = 1 (or a
            // tile is one unit): then the first segment of some share is a part of a tile.  The first boundary behind a tile's
            // begin lies G * j / W units from it, j = 0 .. T - 1 all occurring; a share reaches over that begin and stops short of
            // the tile's end where 1 <= G * j / W < G for some j, and the largest j below W (and T) comes closest to that.  (No
            // walk over the shares: this is made on the host for every call, and again for every size query; 256 shares took 2 us.)
            long long common = p.grid, rest = tiles;
            while (rest)
            {
                const long long r = common % rest;
                common = rest, rest = r;
            }
            const long long W = p.grid / common, T = tiles / common;
            const bool first_used = W > 1 && G > 1, later_used = G * ((W < T ? W : T) - 1) >= W;
            p.slots = later_used ? 2 * p.grid : first_used ? p.grid : 0;
            return p;
        }
        // fp16 x int4: units of 256 k (supersteps), a workgroup keeps at least two (eight K steps of 64)
        // forced_tile_rows / forced_cols: 0 = the plan's own choice (sk_tile_shape)
        inline SkPlan plan_w4a16_sk(int M, int N, int K, bool gate, int num_cu, int forced_tile_rows = 0, long long forced_grid = 0,
                                    int forced_cols = 0)
        {
            if (M <= 0 || N <= 0 || K < 128 || num_cu < 1)
                return SkPlan();
            int rows, cols;
            sk_tile_shape(M, N, gate, forced_tile_rows, forced_cols, rows, cols);
            SkPlan p = plan_sk(M, ceil_div(N, (gate || cols == 128) ? 128 : 256), (K / 128 + 1) / 2, 2, num_cu, rows, forced_grid);
            p.tile_weight_rows = cols;
            return p;
        }

        // the plan with a forced tile height (0 = the plan's own) and a forced number of workgroups per tile (0 = the
        // plan's own grid)
        inline SkPlan plan_w4a16_sk_with(int M, int N, int K, bool gate, int num_cu, int tile_rows, int workgroups_per_tile,
                                         int tile_cols = 0)
        {
            if (workgroups_per_tile <= 0)
                return plan_w4a16_sk(M, N, K, gate, num_cu, tile_rows, 0, tile_cols);
            // (at most one workgroup per unit of 256 k: plan_sk limits the grid to the number of units)
            const SkPlan t = plan_w4a16_sk(M, N, K, gate, num_cu, tile_rows, 0, tile_cols);
            return plan_w4a16_sk(M, N, K, gate, num_cu, tile_rows, (long long)t.tiles_m * t.tiles_n * workgroups_per_tile, tile_cols);
        }

        // The library's own plan of a tile GEMM: every tile cut into the same number of parts, one workgroup each, or (plan_w4a16_sk)
        // an even split whose shares straddle tiles, whichever a fit of measured times says is faster.  A share that straddles a
        // tile boundary starts its pipeline twice and parks two parts; with equal parts it does neither, and a small product is
        // often fastest on whole tiles of few CUs.  Fitted to 4000 products (M = 18 .. 4096, N = 256 .. 16384, K = 512 .. 16384, a
        // quarter of them SiLU-gate; some 50 000 timed plans, weights from memory, 256 CUs): the estimates are within 10 % of the
        // measured time for nine in ten plans, and the plans they pick 15 % (SiLU-gate: 9 %) faster than the even split in the
        // geometric mean, within 1 - 2 % of the fastest one tried.  450 x 448 x 640: 17.1 -> 8.8 us; 110 x 12288 x 1536: 20.8 -> 13.4;
        // 128 x 9216 x 2304: 23.0 -> 16.0; 250 x 16384 x 4096: 47.0 -> 38.9; 450 x 9216 x 11008: 140 -> 106.
        // One in fifty of the plans picked is more than 1 % slower than the even split, by up to 13 % (77 x 5824 x 10624: 28.6 -> 29.2 us);
        // a wider margin than 3 % gives up more than it saves (the plans estimated 3 - 5 % ahead are 7 % faster in the geometric mean).
        // Microseconds: rounds of workgroups x start; the longest share's supersteps (256 k) x (step + load x busy CUs);
        // parts that meet: share + load, more of it from five and nine parts a tile on.
        struct SkCost
        {
            int rows, cols;
            double start, step, step_load, share, share_load, share_load_5, share_load_9; // equal parts
            double even_start, even_step, even_step_load, even_load;                      // the even split
        };
        inline double sk_cost_parts(const SkCost& c, long long tiles, int supersteps, int parts, int num_cu)
        {
            const long long grid = tiles * parts, rounds = (grid + num_cu - 1) / num_cu;
            const double last = (double)(grid - (rounds - 1) * num_cu) / num_cu, longest = ceil_div(supersteps, parts);
            double t = rounds * c.start + longest * (rounds * c.step + (rounds - 1 + last) * c.step_load);
            if (parts > 1)
                t += c.share + last * (c.share_load + (parts > 4 ? c.share_load_5 : 0.0) + (parts > 8 ? c.share_load_9 : 0.0));
            return t;
        }
        // N: output columns (gate: from 2 N weight rows).  rms: with the RMSNorm prologue, which a launch of more workgroups
        // than CUs leaves to a pass of its own.  Never parks more than the even split does: scratch memory sized for that
        // is enough, and is what the *_workspace_bytes queries keep asking for.  sync_bytes: of synchronisation words the caller
        // has (a generated program: what it reserved); tiles that need more are not shared.  0: none, parts are added up by a second launch.
        // even: plan_w4a16_sk of the same product.  blocks: other block parameters than groups of 128 and a scalar zero point
        inline SkPlan plan_w4a16_tiles(const SkPlan& even, int M, int N, int K, bool gate, bool rms, int num_cu, size_t sync_bytes,
                                       bool blocks = false)
        {
            static const SkCost costs[] = {
                {32, 256, 4.26, 1.70, 0.33, 4.65, 0.46, 2.98, 4.69, 8.0, 2.13, 0.0, 5.5},
                {64, 128, 3.58, 1.15, 0.28, 3.81, 1.07, 1.84, 2.61, 6.6, 1.64, 0.0, 3.8},
                {64, 256, 5.22, 1.85, 0.49, 4.56, 1.03, 2.61, 4.72, 9.0, 2.49, 0.0, 6.8},
                {128, 128, 3.94, 1.55, 0.38, 4.36, 3.20, 0.87, 2.40, 7.8, 1.72, 0.76, 4.9},
                {128, 256, 7.07, 2.29, 1.12, 4.44, 3.77, 1.28, 5.13, 10.8, 2.61, 1.37, 8.5},
                {256, 128, 6.43, 1.98, 1.33, 3.84, 6.48, 1.99, 1.31, 8.8, 0.0, 3.88, 10.0},
                {256, 256, 13.40, 3.67, 2.07, 2.60, 9.29, 1.77, 3.53, 20.8, 0.0, 7.17, 10.7},
            };
            static const int parts_tried[] = {1, 2, 3, 4, 6, 8, 12, 16};
            if (even.grid < 1)
                return even;
            const int weight_rows = gate ? 2 * N : N, G = even.supersteps;
            const long long even_tiles = (long long)even.tiles_m * even.tiles_n;
            // Where the fit is off by more than its spread, and a plan picked by it was slower than the even split (even split, the plan
            // without and with the correction timed in turns, the 160 of 60 000 drawn products whose plan they change):
            // whole 128 x 128 tiles on more than half of the CUs over K from 8192 on take 12 % longer than fitted (700 x 4096 x 8192
            // 67.4 us in the even split, 74.5 on them; 315 x 8192 x 11008 97.8 / 106.9): parts of larger tiles instead are 8 % faster in
            // the geometric mean, 2 % with the weights in the last-level cache; without synchronisation words (a second launch adds
            // the parts up) 3 % faster and 2 % slower: left on whole tiles, than which the even split is 10 % slower there;
            // SiLU-gate products of four supersteps on few whole tiles 3 % (1300 rows, 128 outputs, K = 896: halves of tiles 14.9 us in two
            // launches, whole ones 17.1): 3.5 % and 12 %.
            // (neither with other block parameters: 1000 x 4096 x 11008, groups of 32 with zero points, is faster on whole tiles)
            const auto estimate = [&](const SkCost& c, long long tiles, int parts) {
                const double t = sk_cost_parts(c, tiles, G, parts, num_cu);
                if (blocks || parts > 1 || c.rows != 128)
                    return t;
                return c.cols == 128 ? (sync_bytes && G >= 32 && tiles <= num_cu && 2 * tiles > num_cu ? 1.12 * t : t)
                                     : (gate && G == 4 && 16 * tiles <= num_cu ? 1.03 * t : t);
            };
            double best = -1.0;
            for (const SkCost& c : costs)
                if (c.rows == even.tile_rows && c.cols == even.tile_weight_rows)
                {
                    const double busy = (double)even.grid / num_cu, longest = (double)((even.units + even.grid - 1) / even.grid);
                    best = even.slots ? c.even_start + longest * (c.even_step + busy * c.even_step_load) + busy * c.even_load
                                      : estimate(c, even_tiles, 1);
                }
            best *= 0.97; // (another plan for a gain the estimates can tell from nothing)
            int rows = 0, cols = 0;
            long long best_grid = 0;
            for (const SkCost& c : costs)
            {
                // (64 x 256 is the SiLU-gate products' small tile; the others pad M to more than twice itself, or would
                // read the weights once per 64 / 128 rows of many)
                if ((gate ? c.cols == 128 : c.rows == 64 && c.cols == 256) || (c.rows > 64 && M <= c.rows / 2) || (c.rows == 32 && M > 64) ||
                    (c.rows == 64 && M > 256) || (c.rows == 128 && M > 2048))
                    continue;
                const long long tiles = (long long)ceil_div(M, c.rows) * ceil_div(weight_rows, c.cols);
                // (whole tiles that a workgroup walks one behind the other start their pipeline once, where the estimate has a start a
                // round: K = 384 .. 1280 on one round of 256 x 256 tiles is 7 - 18 % slower, 1000 x 16384 x 512 27.0 / 29.2 us;
                // level at 2048, 7 % faster above 4096; level for SiLU-gate)
                if (!gate && c.rows == 256 && c.cols == 256 && even.slots == 0 && even_tiles > num_cu && tiles <= num_cu && G >= 2 && G <= 6)
                    continue;
                for (int n : parts_tried)
                {
                    const long long grid = tiles * n;
                    if (n == 1 ? tiles > 4ll * num_cu : (n > G || grid > num_cu))
                        continue;
                    if (n > 1 && ((size_t)grid * c.rows * c.cols * sizeof(float) > even.bytes() ||
                                  (sync_bytes && (size_t)(tiles + 1) * 2 * sizeof(unsigned) > sync_bytes)))
                        continue;
                    const double t = estimate(c, tiles, n) + (rms && grid > num_cu ? 4.0 : 0.0);
                    if (t < best)
                        best = t, rows = c.rows, cols = c.cols, best_grid = grid;
                }
            }
            return best_grid ? plan_w4a16_sk(M, N, K, gate, num_cu, rows, best_grid, cols) : even;
        }
        // Eight wavefronts on a tile of 64 or 128 rows instead of four (gemm_sk::TileOf).  A wavefront's own share of the work is
        // halved, what comes before and behind the K loop is not, so it takes a long enough share; a second workgroup on the CU,
        // which hides the waits as well, has no room beside the two rings of the 128-wide tiles; and near the full chip the
        // activations' way out of LDS, read twice as often by the 256-wide ones, costs more than it hides.  3000 products on
        // every tile and number of parts, start / this in the geometric mean: 128 x 128 tiles, one a CU, shares of 2 / 4 / 8 / 16
        // / 32 supersteps 0.93 / 1.02 / 1.11 / 1.17 / 1.23 (with RMSNorm 1.31 on few CUs, where rstd[] of many rows a workgroup
        // takes half as long), more tiles than CUs 0.75 - 0.94; parts of 1 / 2 / 4 / 8 / 16: 0.92 / 0.95 / 1.02 / 1.09 / 1.16 up
        // to half of the CUs, 0.92 / 0.89 / 0.90 / 0.98 / 1.05 above three quarters; the even split of more tiles than workgroups
        // 0.94 / 0.97 / 1.02 / 1.03 / 1.03 (of fewer tiles 0.87 - 1.0, left on four); 128 x 256 one a CU 1.2 (few, short) .. 0.99
        // (220 and more, from 32 on), parts 1.10 .. 1.02, from three quarters of the CUs on 0.96 - 1.0.
        // The faster kernel takes power from its neighbours.  70 products of 128 x 128 tiles on 193 .. 255 CUs from eight
        // supersteps on, by themselves 1.047, with pauses 1.039, behind 64 x 4096 x 4096 1.039, behind the product that leads
        // back to their K 1.035, each for the whole sequence; behind two of M x 11008 x 4096 0.997 (0.93 .. 1.05).
        // ragged: columns that are no multiple of eight, whose rows are written an element at a time: from strips of 32 columns that takes
        // longer than from strips of 64 (tiles 256 wide on more than half of the CUs, K = 1024 .. 4096: 0.84 - 1.0, 1029 x 16190 x 1024 in
        // groups of 64 0.84, 300 x 16190 x 4096 0.93).
        inline bool sk_eight_wavefronts(const SkPlan& p, bool gate, bool rms, int num_cu, bool ragged = false)
        {
            if ((p.tile_rows != 64 && p.tile_rows != 128) || p.grid < 1)
                return false;
            if (ragged && !gate && p.tile_weight_rows == 256 && 2ll * p.grid > num_cu)
                return false;
            const long long tiles = (long long)p.tiles_m * p.tiles_n, share = p.units / p.grid;
            const bool one_each = p.grid == tiles, parts = p.grid > tiles && p.grid % tiles == 0;
            if (rms && p.grid <= num_cu && (long long)p.tiles_m * p.tile_rows >= 4ll * p.grid && (one_each || parts))
                return true;
            if (p.tile_weight_rows == 128)
            {
                if (one_each)
                    return p.grid <= num_cu && (share >= 8 || (share >= 4 && 8ll * p.grid <= 5ll * num_cu));
                if (parts)
                    return share >= 16 || (rms ? share >= 4 && 4ll * p.grid <= 3ll * num_cu : share >= 8 && 8ll * p.grid <= 5ll * num_cu);
                return tiles > p.grid && p.supersteps >= 8;
            }
            if (one_each)
                return share <= 16 || (share < 32 && p.grid <= num_cu && !gate) || 2ll * p.grid <= num_cu;
            if (parts)
                return 8ll * p.grid <= 5ll * num_cu && share < 32;
            return (!gate && p.supersteps < 8) || (rms && share < 16);
        }
        // Whole tiles of 128 x 192 (gemm_sk::TileOf<128, 192>: half of what a K step reads from LDS a weight, every wavefront three strips of
        // 32 columns over half of K) in place of the plan `other`, where they fill more than two thirds of the CUs and no more than all:
        // tiles of 128 x 256 leave a third idle there, those of 128 x 128 are too many for one round.  450 products of 100 .. 1600
        // rows: 1.05 - 1.17 x from there to the full chip (256 x 22016 x 4096 with RMSNorm and SiLU-gate 59.6 -> 54.4 us on 230 tiles), 0.6 - 0.9 on
        // fewer tiles and 0.6 - 0.8 on a few more than CUs; two rounds of them 0.93 - 1.04.  Below ten supersteps the sums that the halves of
        // K trade behind the loop cost more (0.91 - 1.06); above 40 and below three quarters of the CUs ranges of K are
        // ahead (0.96); and so are 64-row tiles where they are the plan's, of 129 .. 192 rows (0.91 - 0.98), and 32-row ones of up to
        // 64 rows, of which these tiles pad three quarters and half (16 SiLU-gate products 0.90 - 0.98: 41 x 16356 x 3328 40.8 us, 45.4 on them).
        // One round of whole 128 x 128 tiles, two thirds of the work a workgroup, is ahead as well: 37 products 0.72 - 0.93
        // (1024 x 4096 x 4096 39.1 us, 52.7 on 176 of these tiles; 148 x 16365 x 7936 with RMSNorm 78.7 / 92.5).
        // The rest is a matter of `work`, tiles x their size x supersteps, padding included, against the plan's.  The two rows of wavefronts of
        // these tiles take the supersteps in turn, so an odd number of them costs one more: whole tiles, no RMSNorm, columns a multiple of eight,
        // 1.00 x with ten supersteps, 0.97 with eleven, 1.02 with twelve, 0.99 with thirteen.  Of such products with up to 1.07 times the work
        // 948 gain 1.046, one is more than 3 % slower; above that 196 0.973 (4965 x 1024 x 3840 43.9 us, 47.2 on these tiles; 30827 x 128 x 2816
        // 32.2 / 38.9).  Columns that are no multiple of eight are stored an element at a time, with which fewer, larger tiles are behind: 121
        // products with up to 1.25 times the work 1.08, none below 1.02.  With RMSNorm more workgroups share the sums of squares: 777 products
        // 1.19, 0.98 .. 2.9.
        // Equal parts of tiles have less work a workgroup, and lose their lead with K, as their sums cost less of it:
        //  - halves of 256 x 128 and 128 x 256 and quarters of 256 x 256, two thirds of it, stay: 103 halves 0.95 on these tiles (4085 x 1024 x
        //    6656 60.6 us, 65.9; 1111 x 1792 x 9472 with SiLU-gate 79.5 / 85.0), 21 quarters from 20 supersteps on 0.91, below it 16 1.13.  With
        //    RMSNorm 77 1.33, but from 32 supersteps on and up to 4096 rows five 0.93;
        //  - thirds of 256 x 256, eight ninths of it, up to 35 supersteps: 261 1.12, but 20 of a little more work the shorter K is 1.00; up to 47:
        //    115 with up to 1.03 times the work 1.04, 26 others 0.97, with RMSNorm 270 1.17; above: 63 with less work 1.035, others 73 0.97,
        //    but with RMSNorm and more than 2048 rows 1.17.  Up to 256 rows, one row of tiles there and two here, 23 1.04 up to 41 supersteps,
        //    15 above 0.97.
        // (Without synchronisation words RMSNorm's sums of squares are a pass of their own and nothing is shared: 362 products 1.08, 12 of them more
        // than 3 % slower, 2291 x 1792 x 9728 0.88.  The tiles are the same all the same: words don't change a product's bits here.)
        // 4477 products of 65 .. 34000 rows that the rule without these exceptions takes: 1.10 x in the geometric mean, 331 of them more than 3 %
        // slower; 3886 are on these tiles, 1.12 x, 16 of them more than 3 % slower (662 x 6912 x 12032 0.95), and of the 591 others 13 would
        // gain more than 6 %.
        inline SkPlan plan_w4a16_192(const SkPlan& other, int M, int N, int K, bool gate, int num_cu, bool rms = true)
        {
            SkPlan p;
            p.tile_rows = 128;
            p.tile_weight_rows = 192;
            p.tiles_m = ceil_div(M, 128);
            p.tiles_n = ceil_div(N, gate ? 96 : 192);
            p.supersteps = K / 256;
            p.units = (long long)p.tiles_m * p.tiles_n * p.supersteps;
            const long long tiles = (long long)p.tiles_m * p.tiles_n;
            const bool one_round = other.tile_rows == 128 && other.tile_weight_rows == 128 && !other.slots && other.grid <= num_cu;
            if (other.grid < 1 || one_round || (K & 255) || other.tile_rows <= 64 || p.supersteps < 10 || tiles > num_cu || 3 * tiles <= 2ll * num_cu ||
                (p.supersteps > 40 && 4 * tiles < 3ll * num_cu))
                return other;
            const long long other_tiles = (long long)other.tiles_m * other.tiles_n, area = (long long)other.tile_rows * other.tile_weight_rows;
            const long long work = tiles * 128 * 192 * (p.supersteps + (p.supersteps & 1)), others = other_tiles * area * p.supersteps;
            if (!rms && !other.slots && 100 * work > ((N & 7) ? 125 : 107) * others)
                return other;
            if (other.slots && other.grid % other_tiles == 0)
            {
                const long long of_a_workgroup = area * other_tiles / other.grid;
                bool stays = false;
                if (of_a_workgroup <= 128 * 128)
                    stays = rms ? p.supersteps >= 32 && M <= 4096 : area < 256 * 256 || p.supersteps >= 20;
                else if (of_a_workgroup < 128 * 192)
                    stays = M <= 256             ? p.supersteps >= 42
                            : p.supersteps >= 48 ? work >= others && !(rms && M > 2048)
                                                 : !rms && 100 * work > (p.supersteps >= 36 ? 103 : 139 - p.supersteps) * others;
                if (stays)
                    return other;
            }
            p.grid = (int)tiles;
            return p;
        }
        inline SkPlan plan_w4a16_tiles(int M, int N, int K, bool gate, bool rms, int num_cu, size_t sync_bytes = SIZE_MAX)
        {
            return plan_w4a16_tiles(plan_w4a16_sk(M, N, K, gate, num_cu), M, N, K, gate, rms, num_cu, sync_bytes);
        }
        // ... of the plain product with other block parameters
        inline SkPlan plan_w4a16_tiles_q(int M, int N, int K, int num_cu, size_t sync_bytes = SIZE_MAX)
        {
            return plan_w4a16_tiles(plan_w4a16_sk(M, N, K, false, num_cu), M, N, K, false, false, num_cu, sync_bytes, true);
        }

        // ---- plan of the skinny (M <= 16) MFMA GEMV kernel ---------------------------------------------
        constexpr size_t LDS_BYTES_PER_CU = 160 * 1024; // gfx950
        struct SkinnyPlan
        {
            int cps = 0, ks = 0, h = 0; // groups per wavefront and pass, wavefronts per workgroup, passes over K
            bool a_regs = false;        // activations kept in registers
            // LDS bytes: staged activations; correction constants + scales; partial sums.  With a_regs the
            // activations are only staged until every wavefront has copied its share, and the partial sums and the
            // output parking area then reuse that space.
            size_t a_bytes = 0, fixed_bytes = 0, red_bytes = 0;
            size_t lds(size_t parking_bytes) const
            {
                const size_t tail = red_bytes + parking_bytes;
                return fixed_bytes + (a_regs ? (a_bytes > tail ? a_bytes : tail) : a_bytes + tail);
            }
        };
        // one workgroup spans all of K: fewest groups per wavefront first (more wavefronts in flight), two
        // passes beyond 16 * 3 groups
        inline SkinnyPlan plan_w4a16_skinny(int M, int K, int forced_cps = 0)
        {
            SkinnyPlan p;
            const int G = K >> 7;
            // (four groups per wavefront in one pass spill registers and measured 30 % slower than three in two passes)
            static const int options[6][2] = {{1, 1}, {2, 1}, {3, 1}, {3, 2}, {4, 2}, {4, 1}};
            for (const auto& o : options)
            {
                const int ks = (G + o[0] * o[1] - 1) / (o[0] * o[1]);
                if (forced_cps != 0 && o[0] != forced_cps)
                    continue;
                if (ks <= 16)
                {
                    p.cps = o[0];
                    p.h = o[1];
                    p.ks = ks;
                    break;
                }
            }
            if (p.cps == 0)
                return p;
            // the A operand fits in registers up to two groups per wavefront (32 VGPRs)
            p.a_regs = p.cps <= 2 && p.h == 1;
            p.a_bytes = ((size_t)G * 16 + 1) * M * 16;
            p.fixed_bytes = (size_t)G * 64 + 2 * (((size_t)16 * G * 2 + 15) & ~(size_t)15);
            p.red_bytes = (size_t)2 * M * 16 * 16 * 4;
            return p;
        }
        // true when one workgroup can hold the activations (M <= 16 rows of K) in LDS
        inline bool w4a16_skinny_fits(int M, int N, int K, int forced_cps = 0)
        {
            if (M < 1 || M > 16 || K < 128 || (K & 127) || N < 16)
                return false;
            // the scale block of a tile (16 rows x K/128 fp16) is fetched in whole, aligned 16-byte pieces
            if (((size_t)N * (K >> 7) * 2) % 16 != 0)
                return false;
            // the kernel addresses weights and scales with 32-bit offsets from their base
            if ((size_t)N * (size_t)(K >> 1) >= ((size_t)1 << 32))
                return false;
            const SkinnyPlan p = plan_w4a16_skinny(M, K, forced_cps);
            // leave room for the output parking area (a few tiles of M x 16 floats)
            return p.cps != 0 && p.cps <= (K >> 7) && p.lds(16 * 1024) <= LDS_BYTES_PER_CU;
        }

        // M <= 16 shapes whose activations do not fit at once are run over ranges of K whose activations do fit:
        // equal ranges (multiples of 1024 columns, at most 4096) when K divides that way, otherwise ranges of a
        // multiple of 1024 and a shorter last one of at least 1024.  Returns the length of the ranges (of all but
        // the last), or 0 when this does not apply.
        inline int w4a16_skinny_split_range(int M, int N, int K)
        {
            if (M < 1 || M > 16 || N < 16 || K < 2048 || (K & 127) || w4a16_skinny_fits(M, N, K))
                return 0;
            if ((size_t)N * (size_t)(K >> 1) >= ((size_t)1 << 32)) // 32-bit offsets over whole rows
                return 0;
            static const int equal[] = {2, 4, 8, 16};
            for (int s : equal)
            {
                const int r = K / s;
                if (K % s == 0 && (r & 1023) == 0 && r <= 4096 && w4a16_skinny_fits(M, N, r))
                    return r;
            }
            static const int lengths[] = {4096, 3072, 2048, 1024};
            for (int r : lengths)
            {
                const int s = (K + r - 1) / r;
                if (w4a16_skinny_fits(M, N, r) && s <= 16 && K - (s - 1) * r >= 1024)
                    return r;
            }
            return 0;
        }
        // the number of those ranges (0: does not apply)
        inline int w4a16_skinny_ksplits(int M, int N, int K)
        {
            const int r = w4a16_skinny_split_range(M, N, K);
            return r ? (K + r - 1) / r : 0;
        }
        inline size_t skinny_split_bytes(int M, int N_total, int K)
        {
            const int s = w4a16_skinny_ksplits(M, N_total, K);
            return s ? align256((size_t)s * M * N_total * sizeof(float)) : 0;
        }

        // ---- the VALU GEMV (w4a16_gemv.hip): up to four activation rows of K staged in LDS ----
        inline bool w4a16_gemv_valu_fits(int M, int K)
        {
            if (M < 1 || M > 16 || K < 32 || (K % 32) != 0)
                return false;
            const int mb = M >= 4 ? 4 : M;
            return (size_t)mb * ((K + 2047) >> 11) * 4 * 64 * 16 <= LDS_BYTES_PER_CU;
        }
        // ---- which kernel variants of the fp16 x int4 product can serve a shape (values of nnf_w4a16_variant) ----
        inline bool w4a16_variant_fits(int M, int N, int K, int variant, int num_cu = PLAN_CUS);

        // ---- one activation row: the row-streaming GEMV (w4a16_gemv_rows.hip) ----
        // Eight wavefronts per workgroup (one workgroup per CU) measured fastest: sixteen pay the per-wavefront
        // parts of the kernel twice as often, four leave the vector units idle between dependent instructions.
        constexpr int ROWS_WAVES = 8;
        inline int rows_grid(int N, int num_cu) { return N < num_cu ? N : num_cu; } // one workgroup per CU
        struct RowsPlan
        {
            int seg = 0;    // wavefront-wide loads (1 KiB of a weight row) per row and wavefront; 0: not applicable
            int kshift = 0; // log2 of the wavefronts that share a row
            int depth = 0;  // rows in flight per wavefront
            // ring + activations (+ zeros) + their constants + the workgroup's scales + parked outputs + row counters (32 bytes) + the wavefronts' sums of squares for RMSNorm (32 bytes)
            // (gate: N outputs from 2 N weight rows; a workgroup holds the scales of its gate rows and of its up rows as
            // two blocks, each rounded up to whole KiB)
            // group_shift: log2 of the group size; zero_points: a zero point per (row, group): 256 bytes more per ring slot
            // and 64 groups, and a second constant per unit of activations
            size_t lds_bytes(int N, int K, int grid, bool gate = false, int group_shift = 7, bool zero_points = false) const
            {
                const size_t rows = (size_t)(N / grid + 1);                       // outputs of a workgroup, at most
                const size_t a_pad = (((size_t)(K >> 3) + 63) & ~(size_t)63) + 4; // 16-byte units of activations
                const size_t halves = gate ? 2 : 1;
                const size_t slot = (size_t)seg * 1024 + (zero_points ? (size_t)((seg + 1) / 2) * 256 : 0);
                return (size_t)ROWS_WAVES * depth * slot + a_pad * 16 + a_pad * 4 * (zero_points ? 2 : 1) +
                       halves * ((rows * (size_t)(K >> group_shift) * 2 + 1023) & ~(size_t)1023) +
                       ((halves * rows) << kshift) * sizeof(float) + 64;
            }
        };
        // N: outputs (gate: from 2 N weight rows).  forced_depth: 0 = the plan's own choice
        inline RowsPlan plan_w4a16_rows(int M, int N, int K, int num_cu, int forced_depth = 0, bool gate = false,
                                        int group_shift = 7, bool zero_points = false, int bits = 4)
        {
            RowsPlan p;
            // whole 16-byte pieces of scales per segment, 4-byte aligned: K a multiple of 256
            // (the activations are fetched as at most 2048 16-byte units: K <= 16384)
            if (M != 1 || N < 1 || K < 1024 || K > 16384 || (K & 255) || num_cu < 1 || group_shift < 5 || group_shift > 7 ||
                (gate && (group_shift != 7 || zero_points)) || (bits != 4 && (bits != 8 || gate)))
                return p;
            const int loads_per_row = ((bits == 8 ? K : K >> 1) + 1023) >> 10;
            int kshift = 0;
            while ((1 << kshift) <= ROWS_WAVES && (loads_per_row + (1 << kshift) - 1) >> kshift > 3)
                ++kshift;
            if ((1 << kshift) > ROWS_WAVES)
                return p;
            p.kshift = kshift;
            p.seg = (loads_per_row + (1 << kshift) - 1) >> kshift;
            const int grid = rows_grid(N, num_cu);
            // rows per wavefront of a K segment: the first `depth` of them are fixed
            const int rows_q = ((gate ? 2 : 1) * (N / grid)) / (ROWS_WAVES >> kshift);
            // Two rows in flight per wavefront (a CU takes about 64 wavefront-wide loads in flight; more and the
            // wavefronts stall at issue), a little deeper when a wavefront has many rows to walk (measured).
            const int depth_max = p.seg == 3 ? 2 : 4;
            p.depth = forced_depth > 0 ? forced_depth : (rows_q >= 16 ? (p.seg == 1 ? 4 : 3) : 2);
            if (p.depth > depth_max)
                p.depth = depth_max;
            if (p.depth > rows_q)
                p.depth = rows_q < 1 ? 1 : rows_q;
            while (p.depth > 1 && p.lds_bytes(N, K, grid, gate, group_shift, zero_points) > LDS_BYTES_PER_CU)
                --p.depth;
            if (p.lds_bytes(N, K, grid, gate, group_shift, zero_points) > LDS_BYTES_PER_CU)
                p.seg = 0;
            return p;
        }

        // ---- W8A8 ---------------------------------------------------------------------------------------
        constexpr int Q8_SKINNY_CPS = 2; // preferred chunks per wavefront and pass (more in flight measured slower)
        struct Q8SkinnyPlan
        {
            int cps = 0, kh = 0, ks = 0; // 64-byte chunks of K per wavefront and pass, passes, wavefronts
            size_t lds = 0;              // LDS bytes without the output parking area
        };
        inline Q8SkinnyPlan plan_w8a8_skinny(int M, int K, int forced_cps = 0)
        {
            Q8SkinnyPlan pl;
            const int C = K >> 6;
            // chunks per wavefront and tile: the smallest power of two that needs at most 16 wavefronts
            int per_wave = 1;
            while (per_wave <= 16 && (C + per_wave - 1) / per_wave > 16)
                per_wave *= 2;
            if (per_wave > 16)
                return pl;
            int cps = forced_cps > 0 ? forced_cps : Q8_SKINNY_CPS;
            if (cps > per_wave)
                cps = per_wave;
            while (per_wave / cps > 8)
                cps *= 2;
            pl.cps = cps;
            pl.kh = per_wave / cps;
            pl.ks = (C + per_wave - 1) / per_wave;
            pl.lds = (size_t)pl.ks * per_wave * 4 * M * 16 + (size_t)2 * pl.ks * 256 * 4;
            return pl;
        }
        inline bool w8a8_skinny_fits(int M, int K)
        {
            if (M < 1 || M > 16 || (K & 63))
                return false;
            const Q8SkinnyPlan pl = plan_w8a8_skinny(M, K);
            return pl.cps != 0 && pl.lds + 16 * 1024 <= LDS_BYTES_PER_CU;
        }
        // ---- W8A8, 2 .. 32 activation rows: the row-streaming MFMA kernel (w8a8_mrows.hip) ----
        // K a multiple of 256 up to 16384 (12288 for 17 .. 32 rows).
        // One workgroup per CU, eight wavefronts that each own an eighth of K (256 bytes of every 2 KiB) and keep
        // their share of the activations in registers.  LDS: per wavefront a ring of 4-KiB slots, two sets of eight
        // partial tiles (one or two blocks of 16 rows), the workgroup's finished tiles parked until the end.
        // Two slots (64 KiB in flight per CU) measured 2-9 % faster than three.
        constexpr int W8A8_MROWS_SLOTS = 2;
        inline size_t w8a8_mrows_lds_bytes(int M, int slots, int tiles)
        {
            // ring; partial tiles and parked sums -- or, while the kernel starts, two blocks of 16 rows x 256 bytes of
            // activations per wavefront
            const size_t tail = (size_t)2 * 8 * (M <= 16 ? 1 : 2) * 1024 + (size_t)tiles * M * 64;
            const size_t staging = M > 16 ? (size_t)8 * 2 * 4096 : 0;
            return (size_t)8 * slots * 4096 + (tail > staging ? tail : staging);
        }
        inline bool w8a8_mrows_fits(int M, int N, int K, int num_cu)
        {
            if (M < 2 || M > 32 || N < 16 || num_cu < 1)
                return false;
            // ceil(K / 2048) steps per tile (a template parameter): 16 VGPRs of activations per step and block of rows
            if (K < 1024 || K > (M <= 16 ? 16384 : 12288) || (K & 255))
                return false;
            const int n_tiles = (N + 15) / 16;
            const int grid = n_tiles < num_cu ? n_tiles : num_cu;
            return w8a8_mrows_lds_bytes(M, W8A8_MROWS_SLOTS, (n_tiles + grid - 1) / grid) <= LDS_BYTES_PER_CU;
        }
        // Where the library picks it by itself.  Measured alternately on cold weights against the split-K M <= 16 kernel
        // it is level to 10 % faster up to M = 14 (6 % slower at M = 2, N = K = 8192: not taken below eight rows there),
        // 5-30 % faster at M = 16, and 4-38 % faster than the MFMA tile GEMM at M = 17 .. 32.
        // (Where K does not fill the last step, wavefronts fetch bytes that do not count: at least three quarters of what
        // is fetched must count.)
        inline bool w8a8_mrows_preferred(int M, int N, int K, int num_cu)
        {
            if (((K + 2047) >> 11) == 4 && M < 8) // N = K = 8192: 16.2 us at M = 2 against 15.3 (level from M = 8 on)
                return false;
            return w8a8_mrows_fits(M, N, K, num_cu) && 4 * K >= 3 * 2048 * ((K + 2047) >> 11);
        }
        // Two ranges of K, added up inside the launch (given synchronisation words: one per workgroup of a range, and room for
        // the int32 sums of the ranges): every workgroup fetches all M x K activations ahead of its first MFMA, over two ranges
        // half of them.  Measured (8 .. 32 rows, N = 4096 .. 8192, K = 8192 and 14336) 0.8 - 1.3 us faster than one pass;
        // slower at K = 4096, with more than four tiles per workgroup (N = 16384: +3 us) and over four ranges.
        // (A caller who names the row-streaming kernel; by itself the library runs these products on the K-streaming kernel: w8a8_kstream_choice.)
        inline int w8a8_mrows_ranges(int M, int N, int K, int num_cu)
        {
            const int per_range = num_cu / 2;
            if (M < 8 || K < 8192 || (K & 511) || per_range < 1 || (N + 15) / 16 > 4 * per_range)
                return 1;
            // (17 .. 32 rows, whose activations arrive as whole lines: only where a workgroup has more than one tile
            // anyway -- N = 4096 at 32 rows: 12.3 us in one pass, 13.0 over two ranges; N = 8192: 20.9 / 19.6)
            if (M > 16 && (N + 15) / 16 <= num_cu)
                return 1;
            return w8a8_mrows_fits(M, N, K / 2, per_range) ? 2 : 1;
        }
        inline size_t w8a8_mrows_ranges_bytes(int M, int N, int K, int num_cu)
        {
            const int ranges = w8a8_mrows_ranges(M, N, K, num_cu);
            return ranges > 1 ? align256((size_t)ranges * M * N * sizeof(int)) : 0;
        }
        // ---- 2 .. 16 activation rows (.. 32 up to K = 4096): the row-streaming MFMA kernel (w4a16_mrows.hip) ----
        // One workgroup per CU, eight wavefronts that each own an eighth of K (GW groups of every step of a tile) and
        // keep their share of the activations in registers.  LDS: per wavefront two slots of GW KiB of weights and of
        // their scales, two sets of eight partial tiles (one or two blocks of 16 rows), and the workgroup's finished
        // tiles parked until the end.
        // Two forms.  K / 1024 = 1, 2, 3, 4, 6, 8: K is a compile-time constant of the kernel.  Any other multiple of
        // 128 up to 8192 (M <= 16): K is a run-time value, two steps of 8 * GW groups with the smallest GW (1 .. 4)
        // that covers K; wavefronts past the end of K fetch groups that another one already covers and discard them.
        inline bool w4a16_mrows_fixed_k(int M, int K)
        {
            const int kw = K >> 10;
            return !(K & 1023) && kw >= 1 && kw <= 8 && kw != 5 && kw != 7 && (M <= 16 || kw <= 4) && M <= 32;
        }
        inline int w4a16_mrows_step_groups(int M, int K) // GW
        {
            const int kw = K >> 10, G = K >> 7;
            if (w4a16_mrows_fixed_k(M, K))
                return (kw & 1) ? kw : kw / 2; // even K / 1024: two steps per tile
            return G <= 16 ? 1 : G <= 32 ? 2 : G <= 48 ? 3 : 4;
        }
        // Whether the kernels of 8-bit weights and of a run-time K with other block parameters, which ask for their activations
        // behind the weights and in blocks of 16 rows, bring them in through LDS as whole lines or straight into the registers.
        // (The others always go through LDS, in blocks of 4, 8 or 16 rows ahead of the weights.)  Straight in, a load touches two
        // lines of every row for 32 bytes each, four times over; through LDS every line is touched once, but the blocks come one
        // behind the other (0.3 - 0.5 us).  Measured with 4-bit weights in groups of 128 loaded that way, K = 4096: 2 / 4 / 6 rows
        // 4.84 / 5.07 / 5.20 us straight against 5.19 / 5.27 / 5.29, 8 / 12 / 16 rows 5.63 / 6.52 / 7.3 against 5.30 / 5.40 /
        // 5.55; K = 8192: 4 / 6 rows 12.05 / 12.45 against 11.58 / 11.70; 32 rows at N = K = 4096: 10.8 against 7.1.
        constexpr bool mrows_stages_activations(int M, int K) { return (long long)M * K >= 32768; }
        // the room for that: two blocks of 16 rows x 256 bytes per wavefront, where the partial tiles and parked sums go later
        constexpr size_t mrows_tail_bytes(size_t tail) { return tail > (size_t)8 * 2 * 4096 ? tail : (size_t)8 * 2 * 4096; }
        inline size_t w4a16_mrows_lds_bytes_gw(int gw, int M, int tiles)
        {
            const size_t mb = M <= 16 ? 1 : M <= 32 ? 2 : 4; // blocks of 16 rows
            // ring, scales; partial tiles, the wavefronts' sums of squares per row (RMSNorm inside the kernel), parked sums --
            // or, while the kernel starts, 8 KiB of activations per wavefront (blocks of 16, 8 or 4 rows x 256 bytes) and up to
            // 2 KiB of the RMSNorm weight
            const size_t tail = (size_t)2 * 8 * mb * 1024 + 8 * mb * 64 + (size_t)tiles * M * 64;
            const size_t staging = (size_t)8 * (2 * 4096 + 2048);
            return (size_t)8 * 2 * gw * 1024 + 8 * 512 + (tail > staging ? tail : staging);
        }
        inline size_t w4a16_mrows_lds_bytes(int K, int M, int tiles)
        {
            return w4a16_mrows_lds_bytes_gw(w4a16_mrows_step_groups(M, K), M, tiles);
        }
        // N: output columns; gate: from 2 N weight rows (a workgroup walks the gate and the up tile of each output tile)
        // odd_groups: K may be an odd multiple of 128 (the run-time-K form fetches the scales of each row from its own word;
        // an even number of weight rows, so that the scales are whole words)
        inline bool w4a16_mrows_fits(int M, int N, int K, int num_cu, bool gate = false, bool odd_groups = false)
        {
            if (M < 2 || M > (odd_groups && K <= 2048 ? 64 : 32) || N < 16 || num_cu < 1 || K < 1024 || K > 8192 || (K & 127) ||
                ((K & 128) && (!odd_groups || (!gate && (N & 1)) || (size_t)(gate ? 2 : 1) * N * (K >> 7) >= ((size_t)1 << 30))))
                return false;
            if (!w4a16_mrows_fixed_k(M, K) && M > 16 && K > 4096) // two blocks of rows: at most four groups per wavefront
                return false;
            const int n_tiles = (N + 15) / 16;
            const int grid = n_tiles < num_cu ? n_tiles : num_cu;
            return w4a16_mrows_lds_bytes(K, M, (gate ? 2 : 1) * ((n_tiles + grid - 1) / grid)) <= LDS_BYTES_PER_CU;
        }
        // The same kernel for groups of 32 / 64 / 128 and zero points per (row, group) (w4a16_mrows_q_kernel): 2 .. 16 rows
        // (.. 32 up to K = 4096), K = 2048, 4096, 8192 (GW = K / 2048 groups of 128 per wavefront and step); per wavefront and ring slot 256 bytes
        // per 64 4-byte words of scales (GW x 128 / group scales for each of 16 rows) and as much again for zero points.
        // RMSNorm in front of such a product: inside the kernel, or a pass of its own ahead of it.  Inside, every workgroup
        // normalises all the rows for itself before its first product, twice over once a second block of rows is there; the
        // pass takes 2 us and a launch.  Measured (N = 2304 .. 11008, groups of 32 / 64 / 128, with and without zero points,
        // time with the pass / time inside; alone, with SiLU-gate behind): K = 2048, 2 .. 16 rows 1.01 - 1.16, 1.03 - 1.17;
        // 17 .. 32 rows 0.93 - 0.98, 0.97 - 1.02; K = 4096, 2 .. 7 rows 0.87 - 0.93, 0.92 - 0.99 (8 rows and up bring their
        // activations in as whole lines), 8 .. 16 rows 0.95 - 1.02, 0.97 - 1.03, 17 .. 32 rows 0.82 - 0.89, 0.83 - 0.93;
        // K = 3072 / 3584 0.88 - 1.00, 0.92 - 1.01; K = 4608 / 5120 0.76 - 0.96, 0.80 - 0.97; K = 8192 0.70 - 0.91, 0.78 - 0.95.
        // Those are times with the activations behind the weights.  Ahead of them, K = 4096 and 2 .. 7 rows (with the pass / inside):
        // alone 1.05 - 1.13 at 2304 and 4096 columns, 0.92 - 1.01 at 11008; with SiLU-gate 0.93 - 1.06.  The pass stays there: the
        // tests hold these products to the bits of the nodes one after the other.
        constexpr bool mrows_q_norm_inside(int M, int K) { return M <= 16 && (K == 2048 || (K == 4096 && mrows_stages_activations(M, K))); }
        // (fused: with room for the wavefronts' sums of squares per row, at the sizes that may have RMSNorm inside)
        // norm: with RMSNorm inside, 1 KiB of its weight per wavefront behind the activations while the kernel starts (at most
        // 72 KiB beside 41: always room)
        inline size_t w4a16_mrows_q_lds_bytes(int K, int M, int tiles, int group_shift, bool zero_points, bool fused = false, bool norm = false)
        {
            const int gw = K >> 11;
            const int words = (gw << (7 - group_shift)) / 2; // of scales per row, step and wavefront
            const int loads = (16 * words + 63) / 64;
            const size_t aux = (size_t)(zero_points ? 2 : 1) * loads * 256;
            const size_t mb = M <= 16 ? 1 : 2; // blocks of 16 rows
            const size_t tail = mrows_tail_bytes((size_t)2 * 8 * mb * 1024 + (size_t)tiles * M * 64), staging = (size_t)8 * (2 * 4096 + 1024);
            return (size_t)8 * 2 * gw * 1024 + 8 * 2 * aux + (fused && M <= 16 && K <= 4096 ? 8 * 64 : 0) + (norm && tail < staging ? staging : tail);
        }
        // (17 .. 32 rows: two blocks of rows in registers, up to K = 4096)
        // fused, gate: with the nodes around the product inside the kernel, N outputs from 2 N weight rows
        inline bool w4a16_mrows_q_fits(int M, int N, int K, int group_shift, bool zero_points, int num_cu, bool fused = false, bool gate = false)
        {
            if (M < 2 || M > 32 || (M > 16 && K > 4096) || N < 16 || num_cu < 1 || (K != 2048 && K != 4096 && K != 8192) ||
                group_shift < 5 || group_shift > 7)
                return false;
            if (((K >> 11) << (7 - group_shift)) & 1) // K = 2048 with groups of 128: half a word of scales per step
                return false;
            const int n_tiles = (N + 15) / 16;
            const int grid = n_tiles < num_cu ? n_tiles : num_cu;
            return w4a16_mrows_q_lds_bytes(K, M, (gate ? 2 : 1) * ((n_tiles + grid - 1) / grid), group_shift, zero_points, fused) <= LDS_BYTES_PER_CU;
        }
        // 8-bit weights, 2 .. 16 rows, up to 32 at K <= 4096 (w8a16_mrows_q_kernel): K = 4096 / 8192 (four 64-byte pieces of a weight row per
        // wavefront and step, two / four steps), K = 2048 with groups of 32 / 64 (two pieces, two steps)
        inline size_t w8a16_mrows_q_lds_bytes(int K, int M, int tiles, int group_shift, bool zero_points)
        {
            const int gw = K == 2048 ? 2 : 4;
            const int spr = (gw * 64) >> group_shift; // scales per row, step and wavefront
            const int loads = (16 * (spr / 2) + 63) / 64 + (zero_points ? (16 * spr + 63) / 64 : 0);
            const size_t mb = M <= 16 ? 1 : 2; // blocks of 16 rows
            return (size_t)8 * 2 * gw * 1024 + (size_t)8 * 2 * loads * 256 + mrows_tail_bytes((size_t)2 * 8 * mb * 1024 + (size_t)tiles * M * 64);
        }
        // (17 .. 32 rows: two blocks of rows in registers, up to K = 4096)
        inline bool w8a16_mrows_q_fits(int M, int N, int K, int group_shift, bool zero_points, int num_cu)
        {
            if (M < 2 || M > 32 || (M > 16 && K > 4096) || N < 16 || num_cu < 1 || (K != 2048 && K != 4096 && K != 8192) || group_shift < 5 ||
                group_shift > 7 || (K == 2048 && group_shift == 7))
                return false;
            const int n_tiles = (N + 15) / 16;
            const int grid = n_tiles < num_cu ? n_tiles : num_cu;
            return w8a16_mrows_q_lds_bytes(K, M, (n_tiles + grid - 1) / grid, group_shift, zero_points) <= LDS_BYTES_PER_CU;
        }
        // ... and with K as a run-time value (w4a16_mrows_q_any_kernel): 2 .. 16 rows, any other multiple of 256.  Up to
        // K = 8192 in one piece (two steps of 8 x gw blocks of 128 weights, when at least three quarters of what the
        // wavefronts fetch counts), above over ranges of at most 32 blocks with fp32 sums per range and the reduction pass
        // (as w4a16_mrows_split does it for groups of 128 with a scalar zero point).
        struct MrowsQAny
        {
            int ranges = 0, range_blocks = 0, gw = 0; // ranges 0: not applicable; 1: no workspace
        };
        inline size_t w4a16_mrows_q_any_lds_bytes(int gw, int M, int tiles, int group_shift, bool zero_points)
        {
            const int spc = 1 << (7 - group_shift);
            const int words = spc == 1 ? gw / 2 + 1 : gw * spc / 2;
            const int loads = (16 * words + 63) / 64;
            const size_t aux = (size_t)(zero_points ? 2 : 1) * loads * 256;
            return (size_t)8 * 2 * gw * 1024 + 8 * 2 * aux + mrows_tail_bytes((size_t)2 * 8 * 1024 + (size_t)tiles * M * 64);
        }
        inline MrowsQAny w4a16_mrows_q_any_plan(int M, int N, int K, int group_shift, bool zero_points, int num_cu, bool gate = false)
        {
            MrowsQAny p;
            if (M < 2 || M > 16 || N < 16 || K < 1024 || K > 65536 || (K & 255) || num_cu < 16 || group_shift < 5 || group_shift > 7)
                return p;
            const int B = K >> 7;
            int ranges = 1, rb = B, gw;
            if (K <= 8192)
            {
                gw = B <= 32 ? 2 : B <= 48 ? 3 : 4;
                if (4 * B < 3 * 16 * gw)
                    return p;
            }
            else
            {
                ranges = (B + 31) / 32;
                rb = (((B + ranges - 1) / ranges) + 1) & ~1;
                gw = 2;
                if (B - (ranges - 1) * rb < gw)
                    return p;
            }
            const int n_tiles = (N + 15) / 16, per_range = num_cu / ranges;
            const int grid = n_tiles < per_range ? n_tiles : per_range;
            if (w4a16_mrows_q_any_lds_bytes(gw, M, (gate ? 2 : 1) * ((n_tiles + grid - 1) / grid), group_shift, zero_points) > LDS_BYTES_PER_CU)
                return p;
            p.ranges = ranges;
            p.range_blocks = rb;
            p.gw = gw;
            return p;
        }
        // The tile GEMM with other block parameters (groups of 32 / 64 / 128, zero points per (row, group)): above 16 rows,
        // K a multiple of 256 (the kernel addresses its operands with 32-bit byte offsets); the plain product, same plan
        inline bool w4a16_gemm_q_addressable(int M, int N, int K, int group_shift)
        {
            return M > 16 && N >= 1 && K >= 256 && group_shift >= 5 && group_shift <= 7 && (size_t)M * K * 2 + 8192 < ((size_t)1 << 32) &&
                   (size_t)N * (K >> 1) < ((size_t)1 << 32);
        }
        inline bool w4a16_gemm_q_fits(int M, int N, int K, int group_shift)
        {
            return !(K & 255) && w4a16_gemm_q_addressable(M, N, K, group_shift);
        }
        // ... and on odd multiples of 128, whose last superstep of 256 is half work for nothing, given scratch memory that is preferred and not needed
        // (plan_w4a16_sk: what parked tiles may take), where it is ahead of the plain tile kernel.  900 products, time there /
        // here: K = 384 0.87, 640 0.95, 896 1.04, from 1152 on 1.1 - 1.5 (1000 x 4096 x 4224 in groups of 32 56.2 -> 41 us, 2000
        // rows 92.5 -> 68), but above 1600 rows 0.92 at 1152 / 1408, 1.03 up to 1920; few columns 0.8 - 0.97 at short K, and with
        // few rows too at long (185 x 320 x 15232).
        // Below 512 columns, where a few dozen tiles or their parts are all there is (192 .. 448 columns, 258 .. 2048 rows): K = 2176 / 2688
        // 0.76 - 0.97 up to 300 000 outputs, 1.0 - 1.57 from 320 000 on; K = 6272 0.90 - 0.96 up to 102 000, 0.99 - 1.6 above, from 8576
        // on 0.96 - 1.17 there as well.  Up to 128 rows and 1024 columns, where the plan is an even split whose shares of two
        // supersteps straddle tiles: 153 products 0.93 (0.80 .. 1.18); with equal parts of tiles 165 products 1.08 (0.94 .. 1.34).
        // Columns that are no multiple of eight, which this kernel writes an element at a time (2050 .. 16190 columns, 300 .. 1500 rows):
        // K = 1152 0.67 - 0.88, 1408 0.71 - 0.93, 2176 0.82 - 1.15 (0.95 in the mean), 2688 0.89 - 1.33 (1.03), 4224 1.0 - 1.4.
        inline bool w4a16_gemm_q_odd_fits(int M, int N, int K, int group_shift)
        {
            if ((K & 255) != 128 || ((N & 7) && K < 2688) || !w4a16_gemm_q_addressable(M, N, K, group_shift))
                return false;
            if (M <= 128 && N <= 1024)
            {
                const SkPlan p = plan_w4a16_tiles_q(M, N, K, PLAN_CUS);
                if (p.grid % (p.tiles_m * p.tiles_n))
                    return false;
            }
            if (N >= 512)
                return K >= (M > 1600 || N < 768 ? 2176 : 1152);
            return M > 256 && K >= 2176 && (long long)M * N >= (K < 3456 ? 320000 : K < 8192 ? 110000 : 0);
        }
        // ---- the plain tile kernel (wna16_generic.hip): tile shape and ranges of K ------------------------------------------
        // One range: the tile shape with the lowest time of a K step of 64 on a busy chip: 256 x 256 (0) 2.0 us a round of
        // tiles over the CUs, 256 x 128 (1) 1.2, 192 x 128 (4) 0.95, 128 x 128 (2) 0.9 while every tile has a CU to itself and 1.46 per round of
        // two tiles per CU, 64 x 64 (3) 0.27 + 0.286 per tile and CU (measured at K = 8192 and 4096, 256 CUs; twelve products
        // between 200 and 4096 rows: it picks the fastest of the four).
        // Ranges of K: steps are faster while CUs are idle (busy: their share that works; 64 x 64 tiles 0.3 us), every round of
        // workgroups costs 2.5 us, the reduction pass 3 us, 0.3 a range and its sums at 2.5 TB/s; taken where the estimate is 7 % lower and
        // ws_bytes hold the sums.  Sixty products of 17 .. 2500 rows, one range -> the plan's: 21 x 512 x 16256 81 -> 16 us,
        // 249 x 256 x 15232 80 -> 20, 126 x 1472 x 11648 86 -> 25, 1707 x 896 x 15872 156 -> 82, 261 x 3840 x 8320 88 -> 53.
        enum Wna16Tile
        {
            WNA16_256_256 = 0,
            WNA16_256_128 = 1,
            WNA16_128_128 = 2,
            WNA16_64_64 = 3,
            WNA16_192_128 = 4,
            // on pairs of wavefronts: all of K in one range
            WNA16_PAIRS_160_96 = 5,
            WNA16_PAIRS_128_128 = 6,
            WNA16_PAIRS_128_96 = 7,
        };
        struct Wna16TilePlan
        {
            int tile = WNA16_64_64, ranges = 1, range_k = 0;
            size_t bytes = 0; // of fp32 sums [ranges][M][N]
        };
        inline Wna16TilePlan plan_wna16_tile(int M, int N, int K, int num_cu, size_t ws_bytes, int bits = 8)
        {
            static const int rows[] = {256, 256, 128, 64, 192}, cols[] = {256, 128, 128, 64, 128};
            static const int ranges_tried[] = {2, 3, 4, 6, 8, 12, 16, 24};
            static const double step_idle[] = {0.9, 0.5, 0.35, 0.3, 0.42}, step_busy[] = {2.0, 1.2, 0.9, 0.44, 0.95};
            const auto tiles = [&](int tile) { return (long long)ceil_div(M, rows[tile]) * ceil_div(N, cols[tile]); };
            const auto rounds = [&](long long grid, int per_cu) { return (grid + (long long)num_cu * per_cu - 1) / ((long long)num_cu * per_cu); };
            const auto step_full = [&](int tile, long long grid) {
                const long long r = rounds(grid, 1);
                return tile == 0 ? 2.0 * r : tile == 1 ? 1.2 * r : tile == 4 ? 0.95 * r : tile == 2 ? (r == 1 ? 0.9 : 1.46 * rounds(grid, 2)) : 0.27 + 0.286 * r;
            };
            const auto estimate = [&](int tile, int ranges, int range_k) {
                const long long grid = tiles(tile) * ranges, r = rounds(grid, 1);
                const double busy = (double)grid / num_cu;
                // (64 x 64 tiles of one range: up to four a CU at once, no rounds)
                const bool together = tile == 3 && (r == 1 || ranges == 1);
                const double step = tile == 3 && together ? (busy <= 2.0 ? 0.30 + 0.14 * busy : 0.27 + 0.286 * busy)
                                    : r > 1              ? step_full(tile, grid)
                                                         : step_idle[tile] + busy * (step_busy[tile] - step_idle[tile]);
                return (together ? 4.5 : 2.0 + 2.5 * r) + step * ceil_div(range_k, 64) +
                       (ranges > 1 ? 3.0 + 0.3 * ranges + (double)ranges * M * N * sizeof(float) / 2.5e6 : 0.0);
            };
            Wna16TilePlan best;
            best.range_k = K;
            for (int tile : {2, 4, 1, 0}) // (ties: the larger tile)
                if (step_full(tile, tiles(tile)) <= step_full(best.tile, tiles(best.tile)))
                    best.tile = tile;
            double best_t = 0.93 * estimate(best.tile, 1, K);
            for (int tile = 0; tile < 5; ++tile)
                for (int want : ranges_tried)
                {
                    // (a range: whole groups and bytes of zero points, at least eight steps)
                    const int range_k = (K / want + 255) / 256 * 256, ranges = ceil_div(K, range_k);
                    const size_t bytes = (size_t)ranges * M * N * sizeof(float);
                    if (range_k < 512 || ranges < 2 || bytes > ws_bytes)
                        break;
                    const double t = estimate(tile, ranges, range_k);
                    if (t < best_t)
                        best_t = t, best.tile = tile, best.ranges = ranges, best.range_k = range_k, best.bytes = bytes;
                }
            // Pairs of wavefronts, all of K in one round of 160 x 96 (5), 128 x 128 (6) or 128 x 96 (7) tiles: 3.7 us and 0.68 / 0.66 / 0.59
            // a step, walked in fours, where that is 5 % below the estimate of the others.  Of 2568 products of 18 .. 4000 rows, 8 bits and
            // 4, it moves 116 (before the exception below): 1.11 x in the geometric mean (613 x 6272 x 10752 194 -> 137 us, 249 x 10368 x 4864 71 -> 56).  Two rounds and more 0.85 -
            // 1.08, K below 1024 0.87 - 0.98 with 4 bits and 1.04 with 8.  Ranges of K whose workgroups have no more work than a 128 x 128
            // tile, halves of 256 x 128 and quarters of 256 x 256 tiles, pay for their sums, less and less of it with K: 8 bits, 216 products with
            // such a plan 1.035 on 128 x 128 tiles up to K = 7500, above that 103 halves 0.99 and 31 quarters 0.96 (898 x 4032 x 9600 105 us, 112
            // on them).  Not so with 4 bits, whose steps take longer on the 256-row tiles: 284 halves 1.12, 1.10 above K = 7500, 31 quarters 1.02,
            // 0.97 from 10000 on; nor with columns that are no multiple of eight: 72 1.11.  (160 x 96 tiles, next in the estimate where they fit
            // as well, are 2 - 8 % behind 128 x 128: 423 x 8128 x 9344 104 us over ranges, 114 on them.  128 x 96, three quarters of the work:
            // 44 products of 8 bits from K = 7500 on 1.055.)
            double other = 0.95 * estimate(best.tile, best.ranges, best.range_k);
            const bool same_work = !(N & 7) && best.tile <= WNA16_256_128 && rows[best.tile] * cols[best.tile] <= 128 * 128 * best.ranges &&
                                   (bits == 8 ? K >= 7500 : K >= 10000 && best.tile == WNA16_256_256);
            if (K >= 1024)
                for (int pair = WNA16_PAIRS_160_96; pair <= WNA16_PAIRS_128_96; ++pair)
                {
                    if (pair != WNA16_PAIRS_128_96 && same_work)
                        continue;
                    const long long grid = (long long)ceil_div(M, pair == WNA16_PAIRS_160_96 ? 160 : 128) * ceil_div(N, pair == WNA16_PAIRS_128_128 ? 128 : 96);
                    const double step = pair == WNA16_PAIRS_160_96 ? 0.68 : pair == WNA16_PAIRS_128_128 ? 0.66 : 0.59;
                    const double t = 3.7 + step * 4 * ceil_div(K, 256);
                    if (grid <= num_cu && t < other)
                    {
                        other = t;
                        best = Wna16TilePlan();
                        best.tile = pair;
                        best.range_k = K;
                    }
                }
            return best;
        }
        // whether launch_wna16_generic runs a product on that kernel
        inline bool wna16_on_tile_kernel(int M, int N, int K, int bits, int group_shift, int num_cu)
        {
            if (M <= 16)
                return false;
            if (bits == 4)
                return !w4a16_mrows_q_fits(M, N, K, group_shift, true, num_cu);
            const int block = K == 8192 ? 16 : 32, blocks = ceil_div(M, block);
            return !w8a16_mrows_q_fits(M, N, K, group_shift, true, num_cu) &&
                   !(blocks <= (N <= 8192 ? 3 : 2) && w8a16_mrows_q_fits(block, N, K, group_shift, true, num_cu));
        }
        // nnf_wna16_gemm with parameters other than 4 bits / groups of 128 / scalar zero point, 4-bit weights: [ parked tiles ]
        // on the tile GEMM, [ fp32 sums per range of K ] for 2 .. 16 rows with K above 8192; nothing otherwise
        inline size_t wna16_gemm(int M, int N, int K, int bits, int group, int num_cu = PLAN_CUS)
        {
            const int gs = group == 32 ? 5 : group == 64 ? 6 : group == 128 ? 7 : 0;
            if (bits != 4 || gs == 0)
                return 0;
            if (w4a16_mrows_q_fits(M, N, K, gs, true, num_cu)) // up to 32 rows: the row-streaming kernel
                return 0;
            const MrowsQAny any = w4a16_mrows_q_any_plan(M, N, K, gs, true, num_cu); // ... over ranges of K: their fp32 sums
            if (any.ranges > 0)
                return any.ranges > 1 ? align256((size_t)any.ranges * M * N * sizeof(float)) : 0;
            if (!w4a16_gemm_q_fits(M, N, K, gs))
                return 0;
            return plan_w4a16_sk(M, N, K, false, num_cu).bytes();
        }
        // ... and what the plain tile kernel can use for ranges of K (it runs without)
        inline size_t wna16_gemm_preferred(int M, int N, int K, int bits, int group, int num_cu = PLAN_CUS)
        {
            const size_t needed = wna16_gemm(M, N, K, bits, group, num_cu);
            const int gs = group == 32 ? 5 : group == 64 ? 6 : group == 128 ? 7 : 0;
            if (bits == 4 && w4a16_gemm_q_odd_fits(M, N, K, gs))
            {
                const size_t parked = plan_w4a16_sk(M, N, K, false, num_cu).bytes();
                return parked > needed ? parked : needed;
            }
            if (gs == 0 || (bits != 4 && bits != 8) || (bits == 4 && w4a16_gemm_q_fits(M, N, K, gs)) ||
                !wna16_on_tile_kernel(M, N, K, bits, gs, num_cu))
                return needed;
            return align256(plan_wna16_tile(M, N, K, num_cu, (size_t)64 << 20, bits).bytes);
        }
        // ---- the fused product / MLP block for block parameters that run the nodes one after the other ----------------------
        inline size_t w4a16_gemm(int M, int N, int K, int, int num_cu = PLAN_CUS);
        // nnf_wna16_gemm's own scratch memory, whichever form the zero point takes
        // (needed: without what it can use but runs without)
        inline size_t wna16_gemm_any(int M, int N, int K, int bits, int group, bool needed, int num_cu = PLAN_CUS)
        {
            size_t a = needed ? wna16_gemm(M, N, K, bits, group, num_cu) : wna16_gemm_preferred(M, N, K, bits, group, num_cu);
            if (bits == 4 && group == 128)
            {
                const size_t b = w4a16_gemm(M, N, K, group, num_cu);
                a = b > a ? b : a;
            }
            return align256(a);
        }
        // nnf_wna16_gemm_fused: [ RMSNorm(A): M x K fp16 ][ the product, where the epilogue cannot read it from Y: M x rows fp16 ]
        //                       [ the product's own ]
        struct QFusedLayout
        {
            size_t xn = 0, product = 0, gemm = 0;
            size_t total() const { return xn + product + gemm; }
        };
        inline QFusedLayout wna16_fused_layout(int M, int N, int K, int bits, int group, bool rms, bool gate, bool through_scratch,
                                               bool needed = true)
        {
            QFusedLayout l;
            const int rows = gate ? 2 * N : N;
            l.xn = rms ? align256((size_t)M * K * 2) : 0;
            l.product = (gate || through_scratch) ? align256((size_t)M * rows * 2) : 0;
            l.gemm = wna16_gemm_any(M, rows, K, bits, group, needed);
            return l;
        }
        // nnf_fused_mlp_wna16: [ RMSNorm(x): M x H fp16 ][ gate | up products M x 2I fp16, then the down product M x H fp16 ]
        //                      [ h: M x I fp16 ][ the products' own ]
        inline size_t fused_mlp_wna16(int M, int H, int I, int bits, int group, bool needed = true)
        {
            const size_t a = wna16_gemm_any(M, 2 * I, H, bits, group, needed), b = wna16_gemm_any(M, H, I, bits, group, needed);
            const size_t wide = (size_t)(2 * I > H ? 2 * I : H);
            return align256((size_t)M * H * 2) + align256((size_t)M * wide * 2) + align256((size_t)M * I * 2) + (a > b ? a : b);
        }

        // K above 8192 (above 4096 for 17 .. 32 rows, above 2048 for 33 .. 64; a multiple of 256): the run-time-K form over equal ranges of K (in whole pairs of
        // groups; the last range may be shorter), each on its share of the CUs; fp32 sums per range, added by the
        // reduction pass.  Every workgroup fetches the activations of its range, so shorter ranges mean less of that
        // traffic (CUs x M x K / ranges x 2 bytes): ranges of at most 32 groups (GW = 2) measured fastest (K = 11008:
        // 3 ranges, 14336: 4, 28672: 7-8; 10-25 % faster than the fewest ranges that fit the registers).
        struct MrowsSplit
        {
            int ranges = 0, range_groups = 0, gw = 0;
        };
        inline MrowsSplit w4a16_mrows_split(int M, int N, int K, int num_cu)
        {
            MrowsSplit sp;
            // (What follows decides scratch sizes and the forms without the K-streaming kernel, which serves most of these products:
            // kstream_choice.)  (33 .. 64 rows run on the kernel, but against the tile GEMM, measured alternately: 33 / 40 rows take 25.9 / 27.4 us
            // against 29.1 / 29.3 at N = 22016, K = 4096 and 12.2 / 12.9 against 14.8 / 15.3 at N = K = 4096, are level at K = 8192 and
            // 11008, 8-10 % slower at K = 5120, and slower everywhere from about 48 rows on: taken up to 40 rows and K = 4096)
            // (8 .. 16 rows at K = 8192, up to 8192 weight rows: in one launch every workgroup fetches all M x 8192 activations
            // ahead of its first MFMA; over two ranges it fetches half of them.  With the activations fetched as whole lines
            // that is worth 5 % at 8 rows and nothing at 12 .. 16 (it was 10-18 % before); at 16384 weight rows one range is
            // 6 % faster, and it was slower at K = 5120 / 6144)
            const int longest_single = M <= 16 ? ((M >= 8 && K == 8192 && N <= 8192) ? 8191 : 8192) : M <= 32 ? 4096 : 2048;
            if (M < 2 || M > 40 || N < 16 || K <= longest_single || K > (M <= 32 ? 65536 : 4096) || (K & 255) || num_cu < 16)
                return sp;
            const int G = K >> 7;
            // 33 .. 64 rows: four blocks of rows leave registers for two groups per wavefront: ranges of 16 groups
            int ranges = M <= 32 ? (G + 31) / 32 : (G + 15) / 16;
            const int rg = (((G + ranges - 1) / ranges) + 1) & ~1;
            const int gw = rg <= 16 ? (M <= 32 ? 2 : 1) : rg <= 32 ? 2 : rg <= 48 ? 3 : 4;
            if ((M > 32 && gw > 1) || (M > 16 && gw > 2)) // (only with a forced number of ranges)
                return sp;
            if (G - (ranges - 1) * rg < gw) // the last range holds at least one wavefront's groups
                return sp;
            const int n_tiles = (N + 15) / 16, per_range = num_cu / ranges;
            const int grid = n_tiles < per_range ? n_tiles : per_range;
            if (w4a16_mrows_lds_bytes_gw(gw, M, (n_tiles + grid - 1) / grid) > LDS_BYTES_PER_CU)
                return sp;
            sp.ranges = ranges;
            sp.range_groups = rg;
            sp.gw = gw;
            return sp;
        }
        // synchronisation words for adding the ranges up inside the launch: one per workgroup of a range
        inline size_t mrows_split_sync_bytes(int num_cu) { return (size_t)num_cu * sizeof(unsigned); }
        // Adding the ranges up inside the launch pays while a workgroup has few output tiles: the last arriver adds its
        // tiles up one after the other, the reduction pass works on all of them at once (N = 28672 at 16 rows: 32 us
        // against 30.7 with the pass; N <= 14336: level or up to 8 % faster in the launch).
        inline bool mrows_split_adds_in_launch(int N, int ranges, int num_cu)
        {
            const int per_range = num_cu / ranges > 0 ? num_cu / ranges : 1;
            return ((N + 15) / 16 + per_range - 1) / per_range <= 8;
        }
        inline size_t mrows_split_bytes(int M, int N_total, int K)
        {
            const int r = w4a16_mrows_split(M, N_total, K, PLAN_CUS).ranges;
            return r ? align256((size_t)r * M * N_total * sizeof(float)) : 0;
        }
        // Where the library picks it by itself, from measurements against the split-K MFMA GEMV on cold weights
        // (M = 2 / 16): K = 2048, 4096, 6144, 8192: 0-15 % / 15-30 % faster;  K = 1024, 3072: 5-35 % faster;
        // run-time K from eight rows on: 15-35 % faster at K = 3584, 5120, 7168, level at K = 2560, slower at K = 1536 and 2304,
        // where most of what the wavefronts fetch is discarded: taken when at least three quarters of the fetched groups count.
        inline bool w4a16_mrows_preferred(int M, int N, int K, int num_cu, bool gate = false)
        {
            if (!w4a16_mrows_fits(M, N, K, num_cu, gate, true))
                return false;
            if (w4a16_mrows_fixed_k(M, K))
                return true;
            // Up to seven rows, even numbers of groups, against the MFMA GEMV, whatever part of what is fetched counts (N = 1024
            // / 4096 / 12288): K = 1280 .. 1920 1.0 - 1.2 x, 2304 .. 5888 1.0 - 1.1, 6144 .. 7936 1.04 - 1.4 (4096 x 7168 9.7 ->
            // 7.7 us at seven rows), 1024 and 1152 0.86 - 1.0.
            // (Before the activations came first, in blocks of four or eight rows, these were level or slower.)  Odd numbers of
            // groups keep the GEMV: 4 and 7 rows 1.0 - 1.3 x here from K = 1408 on, 2 and 6 rows 0.95 - 1.25 (K = 1152, 4224
            // and 6272 0.92 - 1.13); RMSNorm, whose pass goes ahead either way, level.
            if (M < 8)
                return !(K & 128) && K >= 1280;
            const int gw = w4a16_mrows_step_groups(M, K);
            // 8 .. 16 rows (K = 3200 1.15 - 1.4 x, 5504 1.6 - 1.75, 8064 1.2 - 1.45, 1920 1.1 - 1.25); 17 .. 32 rows, whose other
            // kernel is the tile GEMM, whatever part of what is fetched counts (K = 1664 .. 1920 1.8 - 2.9 x, 3200 1.7 - 2.5,
            // 3968 1.8 - 2.2).
            // 33 .. 64 rows (the library's own choice is the K-streaming kernel there, 1.2 - 1.9 x; scratch sizes follow this
            // rule), up to sixteen groups: four blocks of rows against the tile GEMM, 1152 / 4096 / 12288 / 22016 weight rows:
            // K = 1280 1.45 / 1.3 / 0.9 - 1.0 / 0.7 x, 1664 .. 2048 1.5 / 1.4 / 1.1 - 1.3 / 0.8 - 1.0; RMSNorm and SiLU-gate
            // 1.5 / 1.5 / 1.2 - 1.4 / 1.0 - 1.3
            if (M > 32)
                return gate ? 2 * N <= (K >= 1280 ? 22016 : 12288) : N <= (K >= 1408 ? 12288 : 8192);
            // (up to 16 rows K = 1536 on one group per wavefront is level: left where it was)
            return M > 16 || 4 * (K >> 7) >= (gw == 1 ? 52 : 3 * 16 * gw);
        }
        // ... except where the MFMA GEMV, which needs no scratch memory but RMSNorm's either, is faster: odd numbers of groups and up
        // to sixteen of them, of which less than seven eighths of what is fetched counts, at eight rows (up to sixteen groups) or
        // until the activations arrive as whole lines (eight to ten).  Time on the MFMA GEMV / here, N = 512 .. 4096, plain and with
        // RMSNorm: K = 3200, 8 .. 10 rows 0.94 - 0.98 (4096 columns at 8 rows 5.7 / 6.0 us), 3456, 8 and 9 rows 0.96 - 1.01, 1664, 8 rows
        // 0.94 - 0.97; with 9152 columns 0.98 - 1.06; K = 3712, 3968, 1792, and 1664 at nine rows: 0.98 - 1.2.
        // (Not with SiLU-gate, 1.05 - 1.2 x here, nor with the residual in place, for which that route asks for scratch memory.)
        // What the library runs by itself is the K-streaming kernel at these sizes (4096 columns at 8 rows of K = 3200 4.8 us);
        // scratch sizes, and devices that kernel does not fit, follow this rule.
        inline bool w4a16_skinny_ahead_of_mrows(int M, int N, int K)
        {
            const int gw = w4a16_mrows_step_groups(M, K);
            if (M < 8 || M > 16 || N > 8192 || w4a16_mrows_fixed_k(M, K) || 8 * (K >> 7) >= 7 * 16 * gw || !w4a16_skinny_fits(M, N, K))
                return false;
            return gw == 1 ? M == 8 && 4 * (K >> 7) >= 52 : (K & 128) && !mrows_stages_activations(M, K);
        }
        // ---- 2 .. 1024 activation rows in blocks of up to 64: the K-streaming kernel (w4a16_kstream.h) ----
        // One workgroup per CU with up to KSTREAM_MAX_TILES 16-row weight tiles, their sums in registers; K in chunks of eight groups.
        constexpr int KSTREAM_WAVES = 8, KSTREAM_MAX_TILES = 6, KSTREAM_MAX_GROUPS = 64;
        // chunks asked for ahead; blocks of 16 rows x 256 bytes of activations in a slot of a wavefront's ring; its bytes of LDS
        constexpr int kstream_depth(int tiles, int mb) { return tiles == 1 && mb == 1 ? 2 : 1; }
        constexpr int kstream_ring(int mb) { return mb < 4 ? mb : 3; }
        // qg: 0, or log2 of the group of other block parameters, whose scales and zero points come chunk by chunk: words of 16 rows, two of
        // them a group of 128 for groups of 32, 64 a load; of zero points as many bytes, a lane each
        constexpr int kstream_scale_loads(int tiles, int qg) { return (tiles * 16 * (qg == 5 ? 2 : 1) + 63) / 64; }
        constexpr int kstream_zero_loads(int tiles, int qg, int bits)
        {
            return (tiles * 16 * (bits == 8 ? 1 << (7 - qg) : qg == 5 ? 2 : 1) + 63) / 64;
        }
        constexpr int kstream_wave_bytes(int tiles, int mb, bool rms, int qg = 0, int bits = 4)
        {
            return kstream_depth(tiles, mb) * (kstream_ring(mb) * 4096 + tiles * 256 * bits + (rms ? 256 : 0) +
                                               (qg ? (kstream_scale_loads(tiles, qg) + kstream_zero_loads(tiles, qg, bits)) * 256 : 0));
        }
        // tiles whose eight partial sums are in LDS at a time (an even number where there is more than one round)
        constexpr int kstream_round(int tiles, int mb) { return mb == 4 && tiles > 4 ? 4 : tiles; }
        constexpr size_t kstream_lds_bytes(int tiles, int mb, bool rms, int qg = 0, int bits = 4)
        {
            const size_t stream = (size_t)KSTREAM_WAVES * kstream_wave_bytes(tiles, mb, rms, qg, bits) + (qg ? 0 : (size_t)tiles * 2048);
            const size_t sums = (size_t)4096 + (size_t)KSTREAM_WAVES * kstream_round(tiles, mb) * mb * 1024;
            return stream > sums ? stream : sums;
        }
        // built and used: what the LDS holds.  qg with RMSNorm needs registers for a group's own sums beside the accumulators: four blocks
        // of rows and five or six tiles spill 14 - 47 of 256
        constexpr bool kstream_built(int tiles, int mb, bool rms, int qg, int bits)
        {
            return kstream_lds_bytes(tiles, mb, rms, qg, bits) <= LDS_BYTES_PER_CU && !(qg && rms && tiles * mb >= 20);
        }
        // CUs of a block of rows: a multiple of eight, so that the workgroups of all blocks that read the same weights are on one XCD (they
        // are dealt out to the eight XCDs in turn)
        constexpr int kstream_cus(int share, int row_blocks) { return row_blocks > 1 && share >= 8 ? share & ~7 : share; }
        struct KstreamPlan
        {
            int tiles = 0; // weight tiles of a workgroup, at most; 0: does not apply
            int row_tiles = 0, row_blocks = 0; // blocks of row_tiles x 16 activation rows
            int tiles_q = 0, tiles_r = 0, grid = 0, ranges = 0, range_groups = 0;
            size_t partial_bytes = 0; // more than one range of K: their fp32 sums
        };
        // N: output columns (gate: from 2 N weight rows); more than one range of K: not with RMSNorm or SiLU-gate
        inline KstreamPlan kstream_plan(int M, int N, int K, int num_cu, bool gate, bool rms, int ranges, int row_blocks = 1, int qg = 0,
                                        int bits = 4)
        {
            KstreamPlan p;
            const int mb = ((M + row_blocks - 1) / row_blocks + 15) / 16, G = K >> 7;
            if (M < 2 || M > 4096 || mb > 4 || N < 16 || K < 1024 || (K & 127) || ranges < 1 || num_cu < ranges * row_blocks ||
                (ranges > 1 && (gate || rms)) || (row_blocks - 1) * mb * 16 >= M)
                return p;
            const int rg = (G + ranges - 1) / ranges, n_tiles = (N + 15) / 16, per_range = kstream_cus(num_cu / (ranges * row_blocks), row_blocks);
            const int grid = n_tiles < per_range ? n_tiles : per_range;
            const int tiles = (gate ? 2 : 1) * ((n_tiles + grid - 1) / grid);
            // (a range's scales: rows of 32 words, from a half word where rows or ranges start in the middle of one)
            if (qg ? ranges > 1 || G > 1023 || (size_t)(gate ? 2 : 1) * N * (K >> qg) >= ((size_t)1 << 31)
                   : rg > ((G & 1) || ranges > 1 ? KSTREAM_MAX_GROUPS - 2 : KSTREAM_MAX_GROUPS))
                return p;
            if ((ranges - 1) * rg >= G ||
                ((G & 1) && (qg == 0 || qg == 7) && ((N & 1) || (size_t)(gate ? 2 : 1) * N * G >= ((size_t)1 << 31))) || tiles > KSTREAM_MAX_TILES ||
                !kstream_built(tiles, mb, rms, qg, bits))
                return p;
            p.tiles = tiles;
            p.row_tiles = mb;
            p.row_blocks = row_blocks;
            p.grid = grid;
            p.tiles_q = n_tiles / grid;
            p.tiles_r = n_tiles % grid;
            p.ranges = ranges;
            p.range_groups = rg;
            p.partial_bytes =
                ranges > 1 ? (size_t)row_blocks * ranges * n_tiles * 16 * (row_blocks > 1 ? mb * 16 : (M + 3) & ~3) * sizeof(float) : 0;
            return p;
        }
        // Microseconds x 100 of a launch, a fit of 841 measured products (20 .. 512 rows, N = 512 .. 16384, K = 1152 .. 11008, with all numbers of ranges
        // and blocks of rows that apply; 11 % rms, and what it picks is within 4 % of the fastest but for 15 of them, 19 % at most): a chunk of eight
        // groups takes what its loads and its unpacking take, a little less where fewer CUs fetch the activations; ranges of K pay for
        // the sums' way through memory.
        inline int kstream_estimate(const KstreamPlan& p, int bits = 4)
        {
            const int chunks = (p.range_groups + KSTREAM_WAVES - 1) / KSTREAM_WAVES, workgroups = p.grid * p.ranges * p.row_blocks;
            const int mb = p.row_tiles, t = p.tiles;
            return chunks * (17 + 27 * mb + (bits == 8 ? 24 : 16) * t + 9 * mb * t) * (358 + (workgroups < 256 ? workgroups : 256)) / 614 + 200 + 6 * t + 15 * mb * t +
                   (p.ranges > 1 ? 84 + 20 * p.ranges + 60 * t : 0);
        }
        // 17 .. 32 rows, K = 2048 in fewer than 112 tiles, without RMSNorm and SiLU-gate: the row-streaming kernels, which have K as a compile-time
        // constant, are 2 - 6 % faster (17 x 512 x 2048 4.0 us there, 4.25 here; groups of 32 / 64 up to 8 %; at
        // 1920 columns level, at 2560 1 - 7 % slower; K = 4096 level at all widths)
        constexpr bool kstream_behind_mrows(int M, int N, int K, bool gate, bool rms)
        {
            return M > 16 && M <= 32 && K == 2048 && N < 1792 && !gate && !rms;
        }
        // What the library runs on it by itself, from measurements against the kernels that served these products before.  33 .. 64 rows:
        // everything that fits (against the tile GEMM: N = K = 4096 at 48 rows 13.8 -> 9.0 us, 12288 x 4096 21.0 -> 15.0, 4096 x 11008 20.5 -> 16.6,
        // RMSNorm and SiLU-gate at 11008 x 4096 35.2 -> 22.4; against the row-streaming kernel up to K = 2048 1.2 - 1.9 x).  17 .. 32 rows: all but more
        // than four tiles a workgroup where the row-streaming kernel runs K as a compile-time constant (11008 x 4096 with both: 18.6 us
        // there, 19.9 here) or over ranges (12288 x 11008: 25.1 us there, 26.8 here); with up to four 1.02 - 1.3 x, K = 5504 2.0 - 2.4 x.
        // More than 64 rows (blocks of at most 64 rows, each on its share of the CUs): the tile GEMM leaves CUs idle or shares tiles through
        // memory where a product has few tiles.  72 .. 512 rows, N = 1024 .. 12288: 1.05 - 2.3 x, with RMSNorm and SiLU-gate 1.1 - 3.0 (128 rows of N = K = 4096
        // 14.9 -> 11.0 us, 256 of 4096 x 6144 28.2 -> 22.9); not at six tiles of four blocks of 16 rows with RMSNorm or SiLU-gate beyond K = 2560
        // (0.84 - 1.1), five or six below K = 2048 (0.89 - 0.98), nor over ranges of K above 256 rows (0.87 - 1.1).
        inline bool kstream_ahead_of_tiles(const KstreamPlan& p, int M, int N, int K, bool gate, bool rms)
        {
            // (the longer K, the less there is to gain, down to nothing where the last tile of many workgroups is missing: 116 x 3200 x 8064 at 78 %
            // of the workgroups' tiles 0.91 x, 117 x 2240 x 8064 at 73 % 0.96, 804 x 1280 x 3456 at 84 % 0.95)
            // (256 x 1600 x 7424 0.92, 218 x 5376 x 7936 0.93, 921 x 256 x 5504 0.84)
            if ((M > 192 && K > 6144) || (M > 512 && K > 4096))
                return false;
            const int used = 100 * (gate ? 2 : 1) * ((N + 15) / 16) / (p.tiles * p.grid);
            if (used < (K > 6144 || (M > 512 && K > 2048) ? 86 : K > 3072 ? 60 : 0))
                return false;
            return p.tiles * p.row_tiles < 20 || (K >= 2048 && (p.tiles * p.row_tiles < 24 || K <= 2560 || (!gate && !rms)));
        }
        // partial_bytes, sync_bytes: of scratch memory and synchronisation words (one per workgroup of a range) at hand
        inline KstreamPlan kstream_choice(int M, int N, int K, int num_cu, bool gate, bool rms, size_t partial_bytes, size_t sync_bytes)
        {
            KstreamPlan best;
            const bool fixed_k = w4a16_mrows_fixed_k(M, K);
            // (17 .. 32 rows: N = 320 .. 600 at K = 1024 takes 3.3 us there, 3.5 here; N = 256 .. 2400 at K = 11776 .. 12288 0.92 - 0.97 x, 4480 and more
            // 1.06 - 1.16)
            if (M < 2 || M > 1024 || (M > 16 && M <= 32 && (K <= 1024 || (K > 11264 && N < 4096))) || kstream_behind_mrows(M, N, K, gate, rms))
                return best;
            // 2 .. 16 rows, against the row-streaming kernel and the MFMA GEMV (time there / here, 1320 products).  K that is a compile-time constant
            // of the row-streaming kernel stays there (SiLU-gate 0.85 - 1.08, others 0.91 - 1.25, most within 8 %); with any other K RMSNorm and SiLU-gate,
            // which cost passes of their own there, 1.03 - 2.4; plain products from eight rows on 1.0 - 1.6 (0.94 - 1.0 for K = 1152 .. 1536 at 8 and 9 rows in
            // one tile a workgroup), of fewer rows 0.94 - 1.3: left where they are, like K above 8192, 0.9 - 1.1 over ranges.
            if (M <= 16 && (fixed_k || K > 8192 || (!gate && !rms && (M < 8 || (K < 1664 && M <= 9 && N <= 4096)))))
                return best;
            const int fewest = (M + 63) / 64, most = M <= 32 ? 1 : fewest + 2;
            for (int row_blocks = fewest; row_blocks <= most; ++row_blocks)
                for (int ranges = 1; ranges <= (gate || rms || M <= 16 || M > 256 ? 1 : 4); ++ranges)
                {
                    const KstreamPlan p = kstream_plan(M, N, K, num_cu, gate, rms, ranges, row_blocks);
                    if (p.tiles == 0 || (ranges > 1 && (p.partial_bytes > partial_bytes || (size_t)p.grid * row_blocks * sizeof(unsigned) > sync_bytes)) ||
                        (M <= 32 && p.tiles > 4 && (ranges > 1 || fixed_k)) ||
                        (M > 64 && !kstream_ahead_of_tiles(p, M, N, K, gate, rms)))
                        continue;
                    if (best.tiles == 0 || kstream_estimate(p) < kstream_estimate(best))
                        best = p;
                }
            return best;
        }
        // The same kernel for 4-bit weights in groups of 2^qg with a scalar zero point or one per (row, group): what the library runs on it, from
        // measurements of 1050 products against the row-streaming kernels of these parameters and the tile GEMM (time there / here).  Up to 16 rows:
        // K = 2048 / 4096 / 8192 0.85 - 1.1, with RMSNorm 1.01 - 1.9 (SiLU-gate beyond four tiles a workgroup 0.84 - 1.07); other K 1.05 - 2.2, above 8192 from
        // 4096 columns on 1.06 - 1.28 up to two tiles (0.89 - 1.1 outside).  17 .. 32 rows 0.98 - 2.7, 33 .. 64 1.02 - 2.4 (two tiles and more of
        // four blocks of rows beyond K = 8192 0.91 - 1.0), more rows up to K = 6144 1.02 - 2.2 (0.85 - 1.3 beyond).
        inline KstreamPlan kstream_choice_q(int M, int N, int K, int qg, int num_cu, bool gate, bool rms)
        {
            KstreamPlan best;
            if (M < 2 || M > 512 || qg < 5 || qg > 7 || (M > 64 && K > 6144) ||
                (kstream_behind_mrows(M, N, K, gate, rms) && w4a16_mrows_q_fits(M, N, K, qg, true, num_cu)))
                return best;
            const int fewest = (M + 63) / 64, most = M <= 32 ? 1 : fewest + 2;
            for (int row_blocks = fewest; row_blocks <= most; ++row_blocks)
            {
                const KstreamPlan p = kstream_plan(M, N, K, num_cu, gate, rms, 1, row_blocks, qg);
                if (p.tiles == 0)
                    continue;
                if (M <= 16)
                {
                    const bool fixed_k = K == 2048 || K == 4096 || K == 8192;
                    // (K = 2048: where the row-streaming kernel takes these parameters, five and six tiles take 8 - 16 % less
                    // time there; up to four level or more)
                    const bool few = K != 2048 || w4a16_mrows_q_fits(M, N, K, qg, true, num_cu, true, gate);
                    if (fixed_k ? !rms || (gate && p.tiles > (few ? 4 : 6)) : K > 8192 && (N < 4096 || p.tiles > 2))
                        continue;
                }
                else if (M <= 64)
                {
                    if (K > 8192 && p.tiles * p.row_tiles >= 8)
                        continue;
                }
                else if (!kstream_ahead_of_tiles(p, M, N, K, gate, rms))
                    continue;
                if (best.tiles == 0 || kstream_estimate(p) < kstream_estimate(best))
                    best = p;
            }
            return best;
        }
        // The same kernel for 8-bit weights in groups of 2^qg (fused: nodes around the product, which take passes of their own elsewhere), from
        // measurements of 1140 products against the row-streaming kernel and the tile kernel (time there / here): 2 .. 16 rows 0.96 - 2.9, but
        // plain products that the row-streaming kernel takes with a compile-time K 0.85 - 1.1: left there; 17 .. 64 rows 0.98 - 2.6
        // (45 x 12288 x 4096 28.3 -> 18.2 us, with RMSNorm 31.5 -> 19.4), more rows 0.97 - 2.3 up to K = 8192 (0.82 - 1.1 beyond).
        inline KstreamPlan kstream_choice_b8(int M, int N, int K, int qg, int num_cu, bool gate, bool rms, bool fused, bool zero_points)
        {
            KstreamPlan best;
            if (M < 2 || M > 512 || qg < 5 || qg > 7 || (M > 64 && K > 8192) || (M <= 16 && !fused && w8a16_mrows_q_fits(M, N, K, qg, zero_points, num_cu)))
                return best;
            const int fewest = (M + 63) / 64, most = M <= 32 ? 1 : fewest + 2;
            for (int row_blocks = fewest; row_blocks <= most; ++row_blocks)
            {
                const KstreamPlan p = kstream_plan(M, N, K, num_cu, gate, rms, 1, row_blocks, qg, 8);
                if (p.tiles == 0)
                    continue;
                if (best.tiles == 0 || kstream_estimate(p, 8) < kstream_estimate(best, 8))
                    best = p;
            }
            return best;
        }
        // ---- W8A8: the K-streaming kernel (w8a8_kstream.hip) ----
        // bytes of K of a wavefront's part of a chunk: two lines of a row where the LDS has room for them and K is a multiple of that
        constexpr size_t w8a8_kstream_lds_bytes(int tiles, int mb, int unit)
        {
            const size_t stream = (size_t)KSTREAM_WAVES * (tiles + mb) * 16 * unit, sums = (size_t)KSTREAM_WAVES * kstream_round(tiles, mb) * mb * 1024;
            return stream > sums ? stream : sums;
        }
        constexpr int w8a8_kstream_unit(int tiles, int mb, int K)
        {
            return !(K & 255) && w8a8_kstream_lds_bytes(tiles, mb, 256) <= LDS_BYTES_PER_CU ? 256 : 128;
        }
        inline KstreamPlan w8a8_kstream_plan(int M, int N, int K, int num_cu, int row_blocks)
        {
            KstreamPlan p;
            const int mb = ((M + row_blocks - 1) / row_blocks + 15) / 16;
            if (M < 2 || mb > 4 || N < 16 || K < 1024 || (K & 127) || num_cu < row_blocks || (row_blocks - 1) * mb * 16 >= M ||
                (size_t)16 * K >= ((size_t)1 << 31))
                return p;
            const int n_tiles = (N + 15) / 16, per_block = kstream_cus(num_cu / row_blocks, row_blocks);
            const int grid = n_tiles < per_block ? n_tiles : per_block, tiles = (n_tiles + grid - 1) / grid;
            if (tiles > KSTREAM_MAX_TILES || w8a8_kstream_lds_bytes(tiles, mb, w8a8_kstream_unit(tiles, mb, K)) > LDS_BYTES_PER_CU)
                return p;
            p.tiles = tiles;
            p.row_tiles = mb;
            p.row_blocks = row_blocks;
            p.grid = grid;
            p.tiles_q = n_tiles / grid;
            p.tiles_r = n_tiles % grid;
            p.ranges = 1;
            return p;
        }
        // Microseconds x 100, a fit of 471 measured launches (2 .. 1000 rows, N = 512 .. 16384, K = 1152 .. 14336; 23 % rms, and the number of blocks of rows it
        // picks is within 6 % of the fastest everywhere)
        inline int w8a8_kstream_estimate(const KstreamPlan& p, int K)
        {
            const int unit = w8a8_kstream_unit(p.tiles, p.row_tiles, K), chunks = (K / unit + KSTREAM_WAVES - 1) / KSTREAM_WAVES;
            const int workgroups = p.grid * p.row_blocks;
            return chunks * (3 + unit / 128 * (23 * p.row_tiles + 40 * p.tiles)) * (363 + (workgroups < 256 ? workgroups : 256)) / 619 + 190 +
                   10 * p.tiles + 3 * p.row_tiles * p.tiles;
        }
        // What the library runs on it by itself (against the row-streaming kernel up to 32 rows and the tile GEMM, time there / here): 2 .. 32 rows
        // 1.0 - 2.8, but four tiles a workgroup of rows of 8 KiB up to 16 rows 0.81 - 0.85 (all workgroups in the same memory channels); 33 .. 64 rows
        // 1.04 - 2.9 (K = 14336 from 8192 columns on 0.96 - 1.03); more rows up to K = 8192 1.1 - 3.8 (14336: 0.9 - 1.7).
        inline KstreamPlan w8a8_kstream_choice(int M, int N, int K, int num_cu)
        {
            KstreamPlan best;
            if (M < 2 || M > 1024 || num_cu < 8 || (M > 32 && M <= 64 && K > 12288 && N >= 8192) || (M > 64 && K > 8192))
                return best;
            const int fewest = (M + 63) / 64, most = M <= 32 ? 1 : fewest + 2;
            for (int row_blocks = fewest; row_blocks <= most; ++row_blocks)
            {
                const KstreamPlan p = w8a8_kstream_plan(M, N, K, num_cu, row_blocks);
                if (p.tiles == 0 || (M <= 16 && p.tiles == 4 && K % 8192 == 0))
                    continue;
                if (best.tiles == 0 || w8a8_kstream_estimate(p, K) < w8a8_kstream_estimate(best, K))
                    best = p;
            }
            return best;
        }
        // ---- W8A8, one activation row: the row-streaming GEMV (w8a8_gemv_rows.hip) ----
        struct Q8RowsPlan
        {
            int seg = 0;    // wavefront-wide loads (1 KiB of a weight row) per row and wavefront; 0: not applicable
            int kshift = 0; // log2 of the wavefronts that share a row
            int depth = 0;  // rows in flight per wavefront
            // ring + activations (+ zeros) + parked sums + row counters
            size_t lds_bytes(int N, int K, int grid) const
            {
                const size_t rows = (size_t)(N / grid + 1); // of a workgroup, at most
                return (size_t)ROWS_WAVES * depth * seg * 1024 + (((size_t)K + 1023) & ~(size_t)1023) + 16 +
                       (rows << kshift) * sizeof(int) + 64;
            }
        };
        // forced_depth: for experiments (0: the plan's own choice)
        inline Q8RowsPlan plan_w8a8_rows(int M, int N, int K, int num_cu, int forced_depth = 0)
        {
            Q8RowsPlan p;
            if (M != 1 || N < 1 || K < 1024 || (K & 127) || num_cu < 1)
                return p;
            const int loads_per_row = (K + 1023) >> 10;
            int kshift = 0;
            while ((1 << kshift) <= ROWS_WAVES && (loads_per_row + (1 << kshift) - 1) >> kshift > 3)
                ++kshift;
            if ((1 << kshift) > ROWS_WAVES)
                return p; // K > 24576
            p.kshift = kshift;
            p.seg = (loads_per_row + (1 << kshift) - 1) >> kshift;
            const int grid = rows_grid(N, num_cu);
            const int rows_q = (N / grid) / (ROWS_WAVES >> kshift); // rows per wavefront of a K segment
            const int depth_max = p.seg == 3 ? 2 : 4;
            p.depth = forced_depth > 0 ? forced_depth : (rows_q >= 16 ? (p.seg == 1 ? 4 : 3) : 2);
            if (p.depth > depth_max)
                p.depth = depth_max;
            if (p.depth > rows_q)
                p.depth = rows_q < 1 ? 1 : rows_q;
            while (p.depth > 1 && p.lds_bytes(N, K, grid) > LDS_BYTES_PER_CU)
                --p.depth;
            if (p.lds_bytes(N, K, grid) > LDS_BYTES_PER_CU)
                p.seg = 0;
            return p;
        }
        // nnf_w8a8_gemm / nnf_w8a8_gemm_acc: [ int32 partial sums ] (same tile plan as the fp16 x int4 GEMM)
        inline size_t w8a8_gemm(int M, int N, int K)
        {
            if (M <= 0 || N <= 0 || K < 128)
                return 0;
            // (the row-streaming kernel over two ranges of K: the ranges' int32 sums)
            const size_t ranges = w8a8_mrows_preferred(M, N, K, PLAN_CUS) ? w8a8_mrows_ranges_bytes(M, N, K, PLAN_CUS) : 0;
            if (w8a8_skinny_fits(M, K))
                return ranges;
            const size_t tiles = gemm_partial_bytes(M, N, false, plan_w8a8_gemm(M, N, K));
            return tiles > ranges ? tiles : ranges;
        }
        // ---- which kernel serves an fp16 x int4 product, and the scratch memory that launch uses --------------------
        // Decided from the shape, the fused parts asked for and the device's CU count alone: the launcher, the entry
        // points' workspace checks and the *_workspace_bytes queries (for PLAN_CUS) all ask this one function.
        struct W4A16Route
        {
            // NONE: the kernel family asked for cannot serve the shape
            enum Kind { NONE, ROWS, MROWS, SKINNY, MROWS_SPLIT, SKINNY_SPLIT, TILE } kind = NONE;
            // the caller fixed nothing: the launch may run on the K-streaming kernel instead, within the scratch memory that `kind` asks for
            // (w4a16_launch_kstream; the size queries and checks stay those of `kind`)
            bool free_choice = false;
            int ksplits = 0;          // *_SPLIT: ranges of K (fp32 partial sums, then the reduction pass)
            bool normalised_copy = false; // RMSNorm as a pass that writes the normalised activations (MFMA GEMV kernels, and what
                                          // the row-streaming kernel took over from other kernels)
            // SKINNY with SiLU-gate: the products go to scratch memory, where the element-wise kernel reads them.  Also set for a
            // residual in place, which the kernel adds itself now: the scratch memory is still asked for, not written.
            bool via_scratch = false;
            SkPlan plan;              // TILE: what the caller fixed, or (own_plan) the even split, in whose scratch memory the launch fits
            bool own_plan = false;    // TILE: the launch follows plan_w4a16_tiles and plan_w4a16_192 (w4a16_launch_tiles)
            size_t partial_bytes = 0; // partial sums / parked tiles / the products ahead of SiLU-gate
            size_t rms_bytes = 0;     // RMSNorm prologue: rstd, fp32 [M] (the kernels multiply the RMSNorm weight in
                                      // themselves), or for the MFMA GEMV kernel the normalised activations, fp16 [M, K]
        };
        // N: output columns (gate: from 2 N weight rows); rms: with the RMSNorm prologue; in_place_residual: the residual
        // is the output buffer itself.  path: 0 the library's order of preference, 2 / 4 one family of GEMV kernels only
        // (values of nnf_w4a16_variant), 3 the tile GEMM with tile_rows / k_parts (0: its own plan).
        // room_for_copy = false: the caller's scratch memory does not hold the normalised activations of the products that the
        // row-streaming kernel took over from others: they run where they ran (see route_w4a16_within).
        inline W4A16Route route_w4a16_other(int M, int N, int K, bool gate, bool rms, bool in_place_residual, int num_cu, int path,
                                            int tile_rows, int k_parts, int tile_cols, bool room_for_copy)
        {
            W4A16Route r;
            if (M <= 0 || N <= 0 || K < 128 || (K & 127) || num_cu < 1)
                return r;
            const int n_rows = gate ? 2 * N : N; // weight rows
            const bool any = path == 0, rows_family = any || path == 4, skinny_family = any || path == 2;
            const size_t rstd_bytes = rms ? align256((size_t)M * sizeof(float)) : 0;
            const size_t xn_bytes = rms ? align256((size_t)M * K * 2) : 0;
            if (path != 3)
            {
                // the row-streaming kernels apply prologue and epilogue themselves: one launch, no scratch memory
                if (rows_family && plan_w4a16_rows(M, N, K, num_cu, 0, gate).seg != 0)
                    return r.kind = W4A16Route::ROWS, r.rms_bytes = rstd_bytes, r;
                // (K = 8192 at 8 .. 16 rows: over two ranges of K, see w4a16_mrows_split -- not with SiLU-gate, whose two halves
                // the reduction would have to pair, nor with RMSNorm, which the single launch folds in without a pre-pass)
                const bool two_ranges = !gate && !rms && K == 8192 && M >= 8 && M <= 16 && w4a16_mrows_split(M, n_rows, K, num_cu).ranges > 1;
                // (the products that once ran elsewhere: gamma times the activations alone may leave the range of fp16)
                const bool taken_over = rms && !w4a16_mrows_fixed_k(M, K) && ((K & 128) || M > 32 || 4 * (K >> 7) < 3 * 16 * (K <= 4096 ? 2 : 3) || (M < 8 && K > 6144));
                const bool gemv_ahead = any && !gate && !in_place_residual && w4a16_skinny_ahead_of_mrows(M, n_rows, K);
                if (rows_family && M > 1 && !two_ranges && !gemv_ahead && !(any && taken_over && !room_for_copy) &&
                    (any ? w4a16_mrows_preferred(M, N, K, num_cu, gate) : w4a16_mrows_fits(M, N, K, num_cu, gate)))
                {
                    r.kind = W4A16Route::MROWS;
                    r.normalised_copy = taken_over && room_for_copy;
                    r.rms_bytes = r.normalised_copy ? xn_bytes : rstd_bytes;
                    return r;
                }
                // the MFMA GEMV kernel writes the [M, 2N] gate | up pair to scratch memory (and once wrote the products ahead of a
                // residual in place there: what callers reserve for them stays what it was)
                if (skinny_family && M <= 16 && w4a16_skinny_fits(M, n_rows, K))
                {
                    r.kind = W4A16Route::SKINNY;
                    r.normalised_copy = true;
                    r.via_scratch = gate || in_place_residual;
                    r.partial_bytes = r.via_scratch ? align256((size_t)M * n_rows * 2) : 0;
                    r.rms_bytes = xn_bytes;
                    return r;
                }
                // more activations than one workgroup holds: ranges of K, fp32 sums per range, and the reduction pass
                // (K above 8192 in multiples of 256: the row-streaming MFMA kernel, otherwise the split-K one)
                if (rows_family && (r.ksplits = w4a16_mrows_split(M, n_rows, K, num_cu).ranges) > 0)
                {
                    r.kind = W4A16Route::MROWS_SPLIT;
                    r.partial_bytes = align256((size_t)r.ksplits * M * n_rows * sizeof(float));
                    r.rms_bytes = rstd_bytes;
                    return r;
                }
                if (skinny_family && (r.ksplits = w4a16_skinny_ksplits(M, n_rows, K)) > 0)
                {
                    r.kind = W4A16Route::SKINNY_SPLIT;
                    r.normalised_copy = true;
                    r.partial_bytes = align256((size_t)r.ksplits * M * n_rows * sizeof(float));
                    r.rms_bytes = xn_bytes;
                    return r;
                }
                r.ksplits = 0;
                if (!any)
                    return r;
            }
            r.kind = W4A16Route::TILE;
            // (the workspace: for the even split, of which the library's own plan never needs more)
            r.plan = plan_w4a16_sk_with(M, N, K, gate, num_cu, tile_rows, k_parts, tile_cols);
            r.own_plan = tile_rows == 0 && k_parts == 0 && tile_cols == 0;
            r.partial_bytes = r.plan.bytes();
            r.rms_bytes = rstd_bytes;
            return r;
        }

        inline W4A16Route route_w4a16(int M, int N, int K, bool gate, bool rms, bool in_place_residual, int num_cu, int path = 0,
                                      int tile_rows = 0, int k_parts = 0, int tile_cols = 0, bool room_for_copy = true)
        {
            W4A16Route r =
                route_w4a16_other(M, N, K, gate, rms, in_place_residual, num_cu, path, tile_rows, k_parts, tile_cols, room_for_copy);
            r.free_choice = path == 0 && tile_rows == 0 && k_parts == 0 && tile_cols == 0;
            return r;
        }
        // the plan of the launch on the K-streaming kernel, or one of no tiles: not there.  sync_bytes: of synchronisation words (0: none)
        inline KstreamPlan w4a16_launch_kstream(const W4A16Route& r, int M, int N, int K, bool gate, bool rms, int num_cu, size_t sync_bytes)
        {
            return r.free_choice && r.kind != W4A16Route::NONE ? kstream_choice(M, N, K, num_cu, gate, rms, r.partial_bytes, sync_bytes) : KstreamPlan();
        }

        // The route of a call that brings `bytes` of scratch memory.  What the size queries ask for covers the normalised activations
        // (M x K x 2 bytes) of the products that the row-streaming kernel took over, most of them from the tile GEMM, which asks for
        // rstd [M] and its parked tiles.  A caller that sized its scratch memory for those -- a generated program carries the
        // byte count as a literal -- keeps the kernel it had.
        inline W4A16Route route_w4a16_within(size_t bytes, int M, int N, int K, bool gate, bool rms, bool in_place_residual, int num_cu,
                                             int path = 0, int tile_rows = 0, int k_parts = 0, int tile_cols = 0)
        {
            const W4A16Route r = route_w4a16(M, N, K, gate, rms, in_place_residual, num_cu, path, tile_rows, k_parts, tile_cols);
            if (r.kind != W4A16Route::MROWS || !r.normalised_copy || r.rms_bytes + r.partial_bytes <= bytes)
                return r;
            return route_w4a16(M, N, K, gate, rms, in_place_residual, num_cu, path, tile_rows, k_parts, tile_cols, false);
        }

        // The plan of a TILE route's launch by the estimates, which are compared once, there, and not by the size queries and checks.  Its
        // synchronisation words are what a generated program reserves.  sync_bytes: of synchronisation words (0: none)
        inline SkPlan w4a16_launch_plan(const W4A16Route& r, int M, int N, int K, bool gate, bool rms, int num_cu, size_t sync_bytes = SIZE_MAX)
        {
            return r.own_plan ? plan_w4a16_tiles(r.plan, M, N, K, gate, rms, num_cu, sync_bytes) : r.plan;
        }
        // ... and the tiles it runs: that plan, or whole tiles of 128 x 192, which need no scratch memory and no words but RMSNorm's two
        inline SkPlan w4a16_launch_tiles(const W4A16Route& r, int M, int N, int K, bool gate, bool rms, int num_cu, size_t sync_bytes)
        {
            const SkPlan p = w4a16_launch_plan(r, M, N, K, gate, rms, num_cu, sync_bytes);
            return r.own_plan ? plan_w4a16_192(p, M, N, K, gate, num_cu, rms) : p;
        }

        inline bool w4a16_variant_fits(int M, int N, int K, int variant, int num_cu)
        {
            if (M <= 0 || N <= 0 || K < 128 || (K & 127))
                return false;
            if (variant == 1)
                return w4a16_gemv_valu_fits(M, K);
            return variant >= 0 && variant <= 4 && route_w4a16(M, N, K, false, false, false, num_cu, variant).kind != W4A16Route::NONE;
        }
        // nnf_w4a16_gemm: [ partial sums ]
        inline size_t w4a16_gemm(int M, int N, int K, int, int num_cu)
        {
            return route_w4a16(M, N, K, false, false, false, num_cu).partial_bytes;
        }
        // nnf_w4a16_gemm_fused: [ RMSNorm scratch ][ partial sums ], whichever of the optional parts the call uses
        inline size_t w4a16_gemm_fused(int M, int N, int K, int, int act, int num_cu = PLAN_CUS)
        {
            // (with and without the RMSNorm prologue, with the residual in place or not: the routes differ -- 8 .. 16 rows
            // at K = 8192 run over two ranges of K only without the prologue)
            const bool gate = act == 1;
            size_t most = 0;
            for (int rms = 0; rms < 2; ++rms)
                for (int in_place = 0; in_place < (gate ? 1 : 2); ++in_place)
                {
                    const W4A16Route r = route_w4a16(M, N, K, gate, rms != 0, in_place != 0, num_cu);
                    const size_t bytes = r.rms_bytes + r.partial_bytes;
                    most = bytes > most ? bytes : most;
                }
            return most;
        }
        // nnf_fused_mlp_w4a16: [ RMSNorm scratch of the first product ][ h: M x I fp16 ][ partial sums of either product ].
        // Of either product what a caller may fix (path: 0, or 3 with a plan's tiles); the down projection's residual is x, in
        // place where the caller passes it as the output too.  bytes: of scratch memory at hand (see route_w4a16_within)
        struct W4A16Choice
        {
            int path = 0, tile_rows = 0, k_parts = 0, tile_cols = 0;
        };
        struct FusedMlpRoutes
        {
            W4A16Route gate_up, down;
            size_t h_offset = 0, partial_offset = 0, total = 0;
        };
        inline FusedMlpRoutes fused_mlp_routes(int M, int H, int I, bool in_place, int num_cu, size_t bytes = SIZE_MAX,
                                               const W4A16Choice& gate_up = W4A16Choice(), const W4A16Choice& down = W4A16Choice())
        {
            FusedMlpRoutes f;
            f.down = route_w4a16(M, H, I, false, false, in_place, num_cu, down.path, down.tile_rows, down.k_parts, down.tile_cols);
            for (int room_for_copy = 1; room_for_copy >= 0; --room_for_copy)
            {
                f.gate_up = route_w4a16(M, I, H, true, true, false, num_cu, gate_up.path, gate_up.tile_rows, gate_up.k_parts,
                                        gate_up.tile_cols, room_for_copy != 0);
                f.h_offset = f.gate_up.rms_bytes;
                f.partial_offset = f.h_offset + align256((size_t)M * I * 2);
                f.total = f.partial_offset +
                          (f.gate_up.partial_bytes > f.down.partial_bytes ? f.gate_up.partial_bytes : f.down.partial_bytes);
                if (f.total <= bytes || f.gate_up.kind != W4A16Route::MROWS || !f.gate_up.normalised_copy)
                    break;
            }
            return f;
        }
        inline size_t fused_mlp_w4a16(int M, int H, int I, int, int num_cu = PLAN_CUS)
        {
            if (M <= 0 || I <= 0 || H < 128 || I < 128)
                return 0;
            const size_t a = fused_mlp_routes(M, H, I, false, num_cu).total, b = fused_mlp_routes(M, H, I, true, num_cu).total;
            return a > b ? a : b;
        }
    } // namespace workspace
} // namespace nnf
