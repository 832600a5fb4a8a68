// Index arithmetic of the kernels, as functions that compile for the device AND for the host.
//
// The kernels compute every global-memory offset (and the LDS offsets that depend on the launch
// geometry) through these functions; a host program can therefore walk (workgroup, wave, lane,
// iteration) tuples of a launch and check each access against the size of the buffer it goes to,
// without a GPU (tests/kernel_bounds/).  Offsets are in ELEMENTS of the tensor they index unless a
// name says bytes.  No HIP types here: the file is also compiled by g++.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define TI8_HD __host__ __device__ __forceinline__
#else
#define TI8_HD inline
#endif

namespace ti8 {
namespace idx {

TI8_HD int imin(int a, int b) { return a < b ? a : b; }
TI8_HD int imax(int a, int b) { return a > b ? a : b; }

// ---- LDS-tiled GEMM (gemm.hip) -------------------------------------------------------------

// workgroup id -> (tile_m, tile_n): mostly one contiguous range of tiles per XCD (ids 8 apart share an
// XCD; the first ones have a tile more where 8 does not divide their number), then groups of `group` tile rows walked column by
// column inside a group.  A number of tiles that 8 divides is in ranges whatever the launch.  Others, us in their own order, which spreads neighbours
// over all XCDs / in ranges: three GEMMs of a step in one launch, int32, 512 tokens 2176 -> 4992 40.3 / 34.6; 640, 8320 -> 1408 55.9 / 48.3; 1152,
// 8832 -> 3584 135 / 127; 3712, 7168 -> 8320 588 / 570; 13056, 7168 -> 11648 2680 / 2637.  A GEMM alone on fewer than 512 tiles of 128 rows, about
// two per CU, keeps its own order, in which the XCDs read the same panel of B at the same time: 1144 tokens 3456 -> 1152 (81 tiles) 24.0 / 25.8;
// 4143, 1024 -> 1280 (330) 17.1 / 18.4; 2300, 1664 -> 3456 (486) 27.4 / 28.9; from there on ranges: 5000, 1024 -> 2688 (840) 31.1 / 30.6.
struct TileCoord {
    int tile_m, tile_n;
};
TI8_HD TileCoord gemm_tile_of(int block_id, int tiles_m, int tiles_n, int group, bool several) {
    const int ntiles = tiles_m * tiles_n;
    const bool ranges = (ntiles & 7) == 0 || several || group < 8 || ntiles >= 512;      // (several GEMMs in the launch; 8: tiles of 128 rows)
    const int xcd = block_id & 7, pid = ranges ? xcd * (ntiles >> 3) + imin(xcd, ntiles & 7) + (block_id >> 3) : block_id;
    const int per_group = group * tiles_n;
    const int group_id = pid / per_group;
    const int first_m = group_id * group;
    const int gsz = imin(tiles_m - first_m, group);
    TileCoord t;
    t.tile_m = first_m + (pid % per_group) % gsz;
    t.tile_n = (pid % per_group) / gsz;
    return t;
}

// GEMM of a several-GEMM launch that workgroup `block` works for: GEMM i owns the workgroups
// [first[i], first[i + 1]), first[0] = 0; only first[1] and first[2] are needed for up to 3 GEMMs
TI8_HD int gemm_multi_pick(int block, int first1, int first2, int count) {
    int i = 0;
    if (count > 1 && block >= first1) i = 1;
    if (count > 2 && block >= first2) i = 2;
    return i;
}

// tile rows per group of the map above for tiles of bm rows
constexpr int gemm_group_rows(int bm) { return bm >= 256 ? 4 : 8; }

// index of the scale of operand row `row` at K block `kb` for a scale descriptor (mode = ti8_scale_mode:
// 0 per row, 1 per 128 x 128 block, 2 per (row, K block), 3 per 128 rows x 256 columns)
TI8_HD int64_t scale_index(int mode, int64_t bs, int64_t rs, int64_t ks, int64_t batch, int row, int kb) {
    switch (mode) {
        case 0: return batch * bs + (int64_t)row * rs;
        case 1: return batch * bs + (int64_t)(row >> 7) * rs + (int64_t)kb * ks;
        case 2: return batch * bs + (int64_t)row * rs + (int64_t)kb * ks;
        default: return batch * bs + (int64_t)(row >> 7) * rs + (int64_t)(kb >> 1) * ks;
    }
}

// first operand row of the rows that `wave` copies into LDS: its n_instr instructions cover
// n_instr * 8 consecutive rows of the tile starting at tile_row0; a span that starts past the
// operand's last row (rows is a multiple of 128, and so is the span's distance to the valid
// half) re-reads the 128 rows before it, whose results nobody stores
TI8_HD int gemm_wave_first_row(int tile_row0, int wave, int n_instr, int rows) {
    const int r = tile_row0 + wave * n_instr * 8;
    return r >= rows ? r - 128 : r;
}

// the same for the 16 rows that each wave (of eight) of the medium-size kernel copies; rows is a multiple of 32, and rows past
// the operand's last re-read its last 16
TI8_HD int gemm_mid_first_row(int tile_row0, int wave, int rows) { return imin(tile_row0 + wave * 16, rows - 16); }

// per-lane byte offset inside the 8-row slab one global->LDS instruction copies: lane l lands at
// byte 16 l of the 1 KiB LDS slab = (row l/8, physical chunk l%8), and fetches the logical chunk
// that the XOR swizzle puts there; `parity` = (index of the instruction within the tile) & 1
TI8_HD uint32_t gemm_lane_offset_bytes(int lane, int parity, int ld) {
    const int ld_row = lane >> 3;
    const int ch = (lane & 7) ^ ld_row ^ parity;
    return (uint32_t)(ld_row * ld + ch * 16);
}

// K offset (bytes = elements) of the tile fetched for K tile `kt`: tiles past the last one fetch
// the last one again (into a buffer nobody reads) so that the loop has no branch
TI8_HD int gemm_k_offset(int kt, int klast) { return imin(kt * 128, klast); }

// byte offset, from the operand's batch base, of the 16 bytes that `lane` fetches in instruction
// `i` (of the wave's n_instr) of a tile: the composition issue_tile_loads performs
TI8_HD int64_t gemm_load_offset_bytes(int first_row, int64_t ld, int koff, int i, uint32_t lane_off) {
    return (int64_t)first_row * ld + koff + (int64_t)i * (8 * ld) + lane_off;
}

// index into a block-scale grid for the per-K-tile factor that lane `lane` keeps in register c
// (K tile 64 c + lane, clamped): (row block) * rs + (kt >> shift) * ks, with ks = 0 for an operand
// whose factor is not applied inside the loop
TI8_HD int gemm_factor_kt(int c, int lane, int nkt) { return imin(c * 64 + lane, nkt - 1); }
TI8_HD int gemm_factor_block(int first_row_of_wave_tile, int rows) { return imin(first_row_of_wave_tile, rows - 1) >> 7; }
TI8_HD int64_t gemm_factor_index(int64_t batch, int64_t bs, int block, int64_t rs, int kt, int shift, int64_t ks) {
    return batch * bs + (int64_t)block * rs + (int64_t)(kt >> shift) * ks;
}

// epilogue: a wave stores its tile 32 rows at a time through an LDS slab; with wcols columns per
// wave tile a row of the tile takes lpr = wcols / 8 lanes (8 columns each) and one instruction
// covers rpi = 64 / lpr rows.  Slab rows are padded by 4 words.
constexpr int EPI_SLAB_LD(int wcols) { return wcols + 4; }
TI8_HD int epi_col_of_lane(int lane, int wcols) { return (lane % (wcols / 8)) * 8; }
TI8_HD int epi_row_of_lane(int lane, int wcols) { return lane / (wcols / 8); }
// the column scales are fetched before the main loop, 4 per lane: lane l those of the wave tile's
// columns 4 (l % 16) .. + 3; in the epilogue the lane that stores columns 8 q .. 8 q + 7 (q = lane % 8)
// takes scale c of them from lane 2 q + c / 4 (register c % 4 there)
TI8_HD int epi_scale_col_of_lane(int lane) { return (lane % 16) * 4; }
TI8_HD int epi_scale_lane(int lane, int c) { return 2 * (lane % 8) + (c >> 2); }
// persistent chained kernel (gemm_chain.hip): its slab holds 16 tile rows of 64 words per wave; accumulator
// register 8 h + e (e < 8) of a 32 x 32 block is row 16 h + epi_chain_slab_row(e, lane / 32) of the block, and
// word (row, col) sits at row * 64 + (col ^ 4 (row & 1))
// first column whose per-row scale of B a wave of the persistent kernel fetches: its tile's first column, or, for a
// tile outside the operand (N is a multiple of 128, the wave tile has 64 columns), the operand's last 64 columns
TI8_HD int chain_col_scale_first(int first_col_of_wave_tile, int ncols) { return imin(first_col_of_wave_tile, ncols - 64); }
// whether the persistent kernel takes a GEMM over so many K tiles.  It walks them in pairs: an odd number as one more, the last one again
// with a factor of 0, which changes no sum (x + 0 d = x).  us, this way / one workgroup per tile, 8192 x 4096: 9 K tiles 53.2 / 51.6,
// 13 68.8 / 69.4, 17 85.8 / 85.3, 25 115.5 / 118.2, 57 242 / 253, 91 378 / 400; 2048 x 2048, 64 tiles: 17 33.1 / 33.9, 91 130 / 146.
// Beside others in a launch, which it would keep on one workgroup per tile, a GEMM goes there from 13 on (the three of a step: 15360 tokens,
// 10112 -> 2176, one over 17 K tiles, 1147 us with one workgroup per tile, 1093; 9856, 1664 -> 1792, 13 K tiles 131, 133).
TI8_HD bool chain_takes(int nk, bool several) { return nk >= 2 && nk <= 256 && ((nk & 1) == 0 || nk >= (several ? 13 : 19)); }
// Which GEMMs of a call that chain their promotion go there, in one launch, the others staying on one workgroup per tile (same bits on either).
// among[i], alone[i]: whether it takes GEMM i beside others of its launch, and by itself; tiles[i] of 256 x 256, 0 for GEMMs of other kernels.  Apart, the
// persistent kernel's last round is paid for in full, so they go apart only where it fills its rounds (8576 tokens, 2944 -> 12800,
// H_128, dX alone 408 tiles on 256 CUs: apart 1450 us, together 1406)
TI8_HD void chains_of_call(const bool* among, const bool* alone, const int64_t* tiles, int count, int num_cu, bool* chains) {
    int together = 0, others = 0;
    int64_t chain_tiles = 0;
    for (int i = 0; i < count; ++i) together += chains[i] = tiles[i] && among[i];
    for (int i = 0; i < count; ++i) {
        if (together == 1) chains[i] = chains[i] && alone[i];
        if (chains[i]) chain_tiles += tiles[i];
        else others += tiles[i] != 0;
    }
    const int64_t rounds = (chain_tiles + num_cu - 1) / num_cu;
    if (others && chain_tiles * 20 < rounds * num_cu * 19)
        for (int i = 0; i < count; ++i) chains[i] = false;
}
// K tiles that it walks
TI8_HD int chain_walked(int nk) { return (nk + 1) & ~1; }
// tile that workgroup `w` of `grid` takes in the round that starts at tile `base`: its own number, in a partly filled last round of a
// launch of several GEMMs counted from the other end -- the longest K comes first there, so that round goes to the workgroups
// whose tiles before it were short.  Past the last tile: no tile (>= total), and none in any later round.
TI8_HD int chain_tile_of_round(int base, int grid, int total, int w, bool several) {
    return several && base + grid > total ? base + grid - 1 - w : base + w;
}
// cost of a tile: its K tiles, and about two and a half more for its end
TI8_HD int chain_tile_cost(int nk) { return 2 * chain_walked(nk) + 5; }
// cost of the busiest of `grid` workgroups that take tiles by rounds (chain_tile_of_round), a tile of GEMM i costing cost[i]: the load changes
// only where a GEMM begins, so those workgroups are looked at
TI8_HD int64_t chain_rounds_busiest(const int64_t* tiles, const int64_t* cost, int count, int grid) {
    int64_t first[4] = {0, 0, 0, 0};
    for (int i = 0; i < count; ++i) first[i + 1] = first[i] + tiles[i];
    const int64_t total = first[count], rounds = (total + grid - 1) / grid;
    int64_t busiest = 0;
    for (int q = 0; q < 4 * (count + 1); ++q) {
        int64_t w = (first[q >> 2] + grid - 1 + (q & 1)) % grid;   // the last workgroup in front of GEMM q / 4, or its first
        if (q & 2) w = grid - 1 - w;
        int64_t load = 0;
        for (int64_t r = 0; r < rounds; ++r) {
            const int64_t t = r * grid + (r == rounds - 1 && count > 1 ? grid - 1 - w : w);
            if (t < total) load += cost[t < first[1] ? 0 : (t < first[2] || count < 3 ? 1 : 2)];
        }
        if (load > busiest) busiest = load;
    }
    return busiest;
}
// The same for GEMMs over different numbers of K tiles, from a list: tiles in order, the longest K first, each to the workgroup that is
// free first.  A list serves the workgroups of one XCD (`slots` of them): XCD x takes tiles x, x + 8, ... of every GEMM, whose
// neighbours in its L2 they then stay, and entry v is tile 8 v + x of the launch, GEMM i having the tiles from 8 (n[0] + .. + n[i - 1]) on.
// cost[i] descending.  tile[first[s]] .. tile[first[s + 1] - 1]: what workgroup s takes.  Returns the cost of the busiest.
constexpr int CHAIN_LIST_SLOTS = 32, CHAIN_LIST_MAX = 480;
TI8_HD int chain_list(const int* n, const int* cost, int count, int slots, int* first, uint16_t* tile) {
    int free_at[CHAIN_LIST_SLOTS] = {}, slot_of[CHAIN_LIST_SLOTS];      // workgroups by the time at which they are free
    for (int s = 0; s < slots; ++s) slot_of[s] = s;
    uint8_t taken_by[CHAIN_LIST_MAX];
    int v = 0, busiest = 0;
    for (int i = 0; i < count; ++i) {
        // those that have not taken a tile of this GEMM yet, from `head` on, and those that have, in the order in which they are free again
        int head = 0, again_at[CHAIN_LIST_SLOTS], again[CHAIN_LIST_SLOTS], begin = 0, held = 0;
        for (int k = 0; k < n[i]; ++k) {
            int at, s;
            if (head < slots && (held == 0 || free_at[head] <= again_at[begin])) {
                at = free_at[head];
                s = slot_of[head++];
            } else {
                at = again_at[begin];
                s = again[begin];
                begin = (begin + 1) % CHAIN_LIST_SLOTS;
                --held;
            }
            const int to = (begin + held++) % CHAIN_LIST_SLOTS;
            again_at[to] = at + cost[i];
            again[to] = s;
            taken_by[v++] = (uint8_t)s;
        }
        int merged_at[CHAIN_LIST_SLOTS], merged[CHAIN_LIST_SLOTS];
        for (int q = 0; q < slots; ++q) {
            const bool old = head < slots && (held == 0 || free_at[head] <= again_at[begin]);
            merged_at[q] = old ? free_at[head] : again_at[begin];
            merged[q] = old ? slot_of[head] : again[begin];
            if (old) ++head;
            else {
                begin = (begin + 1) % CHAIN_LIST_SLOTS;
                --held;
            }
        }
        for (int q = 0; q < slots; ++q) {
            free_at[q] = merged_at[q];
            slot_of[q] = merged[q];
        }
        busiest = free_at[slots - 1];
    }
    int at[CHAIN_LIST_SLOTS + 1] = {};
    for (int k = 0; k < v; ++k) ++at[taken_by[k] + 1];
    for (int s = 0; s < slots; ++s) at[s + 1] += at[s];
    for (int s = 0; s <= slots; ++s) first[s] = at[s];
    for (int k = 0; k < v; ++k) tile[at[taken_by[k]]++] = (uint16_t)k;
    return busiest;
}
TI8_HD int epi_chain_slab_row(int e, int fr_half) { return 8 * (e >> 2) + 4 * fr_half + (e & 3); }
TI8_HD int epi_chain_slab_word(int row, int col) { return row * 64 + (col ^ (4 * (row & 1))); }
// index of the column scale of column `col` (clamped to the last column; stride 0 when absent)
TI8_HD int64_t epi_col_scale_index(int64_t batch, int64_t bs, int col, int ncols, int64_t cs) {
    return batch * bs + (int64_t)imin(col, ncols - 1) * cs;
}
// per-row scale of A of this lane's first output row (only waves whose tile lies inside the output get here)
TI8_HD int64_t epi_row_scale_base(int64_t batch, int64_t bs, int row0, int64_t rs) {
    return batch * bs + (int64_t)row0 * rs;
}
// output element offset of (batch, row0, col0) and the step between the rows one lane stores
TI8_HD int64_t epi_out_offset(int64_t batch, int64_t bsc, int row0, int64_t ldc, int col0) {
    return batch * bsc + (int64_t)row0 * ldc + col0;
}

// ---- Walsh-Hadamard transform (fwht.hip) ----------------------------------------------------
TI8_HD int fwht_padded(int i) { return i + (i >> 4); }
// element offset of segment `seg` (of L elements) of row `row`
TI8_HD int64_t fwht_segment_offset(int64_t block, int segs_per_row, int64_t ld, int L) {
    const int64_t row = block / segs_per_row;
    const int seg = (int)(block % segs_per_row);
    return row * ld + (int64_t)seg * L;
}
// whether the `len` elements from `first` of a segment exist in memory (`valid` elements do; the rest of a zero-extended
// row reads as zero and is not stored); valid is a multiple of len
TI8_HD bool fwht_chunk_valid(int first, int len, int valid) { return first + len <= valid; }
// LDS words a workgroup needs for L elements
TI8_HD int64_t fwht_lds_words(int64_t L) { return L + L / 16; }
// fwht_row_kernel (segments of 4096 * CH elements on 4 waves): first element of the 16-element chunk that the lane at chunk
// position `lp` of wave `w` takes from slice `k`; the word of its value `e` in the exchange buffer; and the first of the 4
// consecutive elements of (slice k, wave ws, chunk position lp) that wave `w` ends up with
TI8_HD int fwht_row_chunk_first(int k, int w, int lp) { return ((k * 4 + w) * 64 + lp) * 16; }
// (laid out so that a lane's elements 4j .. 4j + 3 are one aligned 16-byte unit and consecutive chunk positions are
// consecutive units: both the writes -- four units per lane -- and the reads -- unit j = w of all four waves -- are
// 16-byte LDS accesses without bank conflicts)
TI8_HD int fwht_row_lds(int w, int lp, int e) { return (((e >> 2) * 4 + w) * 64 + lp) * 4 + (e & 3); }
TI8_HD int fwht_row_out(int k, int ws, int lp, int w) { return ((k * 4 + ws) * 64 + lp) * 16 + 4 * w; }
// base LDS index of the radix-2^rb group `vt` in the pass over index bits [p, p + rb)
TI8_HD int fwht_group_base(int vt, int p, int rb) {
    const int lo = vt & ((1 << p) - 1);
    const int hi = vt >> p;
    return (hi << (p + rb)) | lo;
}

// transposed-input transform (y = FWHT of x^T along its rows = along the ROWS of x, length R):
// columns of x per workgroup (as many as fit the LDS budget of 32768 fp32 elements, at most the 8
// that one 16-byte load brings) and the column block of workgroup `id`: the G = 64 / W workgroups
// whose columns share one 128-byte line of every row get consecutive places on ONE XCD (workgroup
// ids 8 apart share an XCD), so that the line is fetched from HBM once; identity when the number of
// such groups is not a multiple of 8
TI8_HD int fwht_t_cols_per_wg(int64_t R) { return R <= 4096 ? 8 : (int)(32768 / R); }
// whether the one-kernel transposed transform is used: up to 2048 rows; longer columns go through a
// transposing copy into the output and an in-place transform there (lengths from 4096 on have the
// faster row kernel: 8192 x 4096 in 58 instead of 78 us, 8192 x 8192 in 105 instead of 146 us,
// 4096 x 4096 the same either way), which needs whole 64 x 64 tiles
TI8_HD bool fwht_t_direct(int64_t R, int64_t C) { return R <= 2048 || (C % 64) != 0; }
TI8_HD int64_t fwht_t_colblock(int64_t id, int64_t nblocks, int W) {
    const int G = 64 / W;
    if (nblocks % (8 * (int64_t)G) != 0) return id;
    const int64_t xcd = id & 7, j = id >> 3;
    return ((j / G) * 8 + xcd) * G + (j % G);
}

// ---- per-row quantiser (quant.hip) -----------------------------------------------------------
// row handled by (workgroup, wave): one workgroup per row, or one wave per row (4 rows per workgroup)
TI8_HD int64_t qrow_row(int64_t block, int wave, bool wg_row) { return wg_row ? block : block * 4 + wave; }
// 16-byte chunk index of load i of thread t (T threads per row)
TI8_HD int qrow_chunk(int t, int i, int T) { return t + i * T; }
// The quantisers that rotate 128-element segments first (H128 across 16 lanes x 8 elements) give chunk
// c ^ (c & 4 ? 3 : 0) of a segment to the lane that would otherwise hold chunk c: a permutation within
// every aligned group of 16 chunks (its own inverse), under which the partners of all four cross-lane
// stages are one DPP pattern away.
TI8_HD int had_chunk(int c) { return c ^ ((c & 4) ? 3 : 0); }

// ---- 128 x 128 tile quantisers (quant.hip) ---------------------------------------------------
struct TileId {
    int b, rb, cb;
};
TI8_HD TileId qblock_tile(int block, int nrb, int ncb) {
    TileId t;
    t.cb = block % ncb;
    block /= ncb;
    t.rb = block % nrb;
    t.b = block / nrb;
    return t;
}
// element offset of a tile's origin in a [B][R][C] tensor with tiles of 128 x tile_c
TI8_HD int64_t qblock_origin(int b, int64_t bs, int rb, int64_t ld, int cb, int tile_c) {
    return b * bs + (int64_t)rb * 128 * ld + (int64_t)cb * tile_c;
}
// thread t of 256 owns rows {64 h + 4 (t / 16) + j : h < 2, j < 4} x columns [8 (t % 16), + 8)
TI8_HD int qblock_row(int t, int h, int j) { return h * 64 + (t >> 4) * 4 + j; }
TI8_HD int qblock_col(int t) { return (t & 15) * 8; }
// the transposed tile leaves LDS as 128-byte rows: pass p of thread t writes row p * 32 + t / 8
// (= column of x), bytes 16 (t % 8) .. + 15 (= rows of x)
TI8_HD int qblock_t_row(int t, int p) { return p * 32 + (t >> 3); }
TI8_HD int qblock_t_col(int t) { return (t & 7) * 16; }

// ---- quantisers of a layer call in two launches (quant.hip) -------------------------------------
// Maxima of an operand [R][C]: a workgroup takes a part of tr x tc tiles of 128 x 128, the last ones in either direction shorter, and stores
// 16 bits per row of it and per column: rows [nct][R], cols [nrt][C], one array behind the other.  About 32 parts in either
// direction; a part keeps the maxima of its rows in LDS, so beyond 262144 rows there is one for every 8192.
constexpr int MAXIMA_ROW_TILES = 64;
struct MaximaParts {
    int tr, tc, nrt, nct;
};
TI8_HD MaximaParts maxima_parts(int64_t R, int64_t C) {
    MaximaParts m;
    const int64_t a = (R / 128 + 31) / 32;
    m.tr = (int)(a < MAXIMA_ROW_TILES ? a : MAXIMA_ROW_TILES);
    m.tc = (int)((C / 128 + 31) / 32);
    m.nrt = (int)((R / 128 + m.tr - 1) / m.tr);
    m.nct = (int)((C / 128 + m.tc - 1) / m.tc);
    return m;
}
TI8_HD int64_t maxima_rows_at(int ct, int64_t R, int row) { return (int64_t)ct * R + row; }
TI8_HD int64_t maxima_cols_at(int rt, int64_t C, int col) { return (int64_t)rt * C + col; }
// 32-bit words of both arrays (R and C are multiples of 128)
TI8_HD int64_t maxima_words(int64_t R, int64_t C) {
    const MaximaParts m = maxima_parts(R, C);
    return (m.nct * R + m.nrt * C) / 2;
}
// operands start at multiples of 8 workgroups: ids 8 apart are workgroups of one XCD
TI8_HD int64_t round8(int64_t n) { return (n + 7) / 8 * 8; }
// which of up to three operands `at` belongs to, operand i having [first[i], first[i + 1])
TI8_HD int operand_of(int at, const int* first, int count) {
    int i = 0;
    for (int k = 1; k < 3; ++k)
        if (k < count && at >= first[k]) i = k;
    return i;
}
// the conversion's tile of workgroup `block` of `grid` (a multiple of 8): from the end of the last operand to the beginning of the first, and
// every tile on the XCD that took its maxima where a part is one tile
TI8_HD int rowcol_multi_tile(int block, int grid) { return ((grid >> 3) - 1 - (block >> 3)) * 8 + (block & 7); }

// ---- GEMM with few rows (gemm_skinny.hip) ------------------------------------------------------
// Workgroup -> strip of B and rows of A, in blocks of the workgroup's size: those that share a strip on one XCD (ids 8 apart)
struct FewPlace {
    int strip, mt;
};
TI8_HD FewPlace few_place(int block, int mtiles, int nstrips) {
    FewPlace p;
    if ((nstrips & 7) == 0) {
        const int xcd = block & 7, idx = block >> 3;
        p.strip = (idx / mtiles) * 8 + xcd;
        p.mt = idx % mtiles;
    } else {
        p.strip = block / mtiles;
        p.mt = block % mtiles;
    }
    return p;
}
TI8_HD int64_t few_blocks(int64_t M, int64_t N, bool wide) { return wide ? (N / 64) * ((M + 63) / 64) : (N / 32) * (M / 32); }
// K tiles of a wave: [few_k_first(wave, nk), few_k_first(wave + 1, nk))
TI8_HD int few_k_first(int wave, int nk) { return (wave * nk) >> 2; }
// K tile of step i of a wave's walk over nq of nk, which starts at its tile `rot`; past the end: the last one again
TI8_HD int few_k_tile(int i, int rot, int kbeg, int nq, int nk) {
    int j = imin(i, imax(nq - 1, 0)) + rot;
    if (j >= nq) j -= nq;
    return imin(kbeg + imax(j, 0), nk - 1);
}
// ---- Y of up to 8 rows by 16 rows of the weight per workgroup (gemm_decode.hip) --------------------------------------
constexpr int DECODE_BATCH = 8;       // K tiles whose codes a wave makes together
// first step of a wave's walk over nq K tiles: that of the 32 x 32 block around these columns
TI8_HD int decode_rot(int n0, int nq) { return nq > 0 ? (int)((((unsigned)n0 >> 8) * 3u) % (unsigned)nq) : 0; }
// the lane's 16 columns of a row's K tile, and its 16 bytes of the weight's (the second half of the K tile: 64 bytes on)
TI8_HD int64_t decode_x_offset(int row, int64_t ldx, int kt, int lane) { return row * ldx + kt * 128 + (lane & 7) * 16; }
TI8_HD int64_t decode_w_offset(int n0, int64_t ldb, int kt, int lane) { return (int64_t)(n0 + (lane & 15)) * ldb + kt * 128 + (lane >> 4) * 16; }
// ---- Y and dX of a step on few tokens, the weight quantised in the kernel (gemm_skinny.hip: raw_block) ---------------
// Elements of the weight [R][C] that a lane loads for a K tile.  Y: piece i (of 4) of 8 columns of its row; the 64 columns of a matrix
// instruction are two pieces of four lanes each, and the codes of the tokens are read the same way.  dX: 2 columns of row j (of 16) of half h.
constexpr int RAW_STRIP_Y = 16, RAW_STRIP_DX = 32;
// part of the maxima that a lane looks at as its i-th: every fourth, past the last one that one again.  Up to 32 parts (maxima_parts, up to
// 32 * 128 * MAXIMA_ROW_TILES rows)
constexpr int RAW_PARTS = 32;
TI8_HD int raw_part(int i, int lane, int count) { return imin((lane >> 4) + 4 * i, count - 1); }
// Whether such a step takes them.  A workgroup walks the whole contraction, so a side much longer than the other leaves few of them with long
// walks; and for a second block of 16 tokens the codes are read twice as often, which costs what the saved launch gains, but on a small weight and
// on one whose codes both ways no longer fit the Infinity Cache (256 MiB) beside it and what the GEMMs write: 4 bytes per element of the weight
// and 2 of dW, 336 MiB at 14336 x 4096; at 8960 x 4864, 249 MiB, the gain (89.6 / 87.1) is what neighbours lose (5632 x 4736 60.8 / 63.7).
// The step, us, its weight quantised in memory / so: 16 tokens, 4096 -> 4096 37.7 / 32.5, 2048 -> 2048 22.3 / 17.3, 7936 -> 8960 177 / 132,
// 13440 -> 3200 89.8 / 76.1, 3200 -> 13440 88.6 / 75.0, 10240 -> 1024 37.1 / 34.5, 14336 -> 1024 44.8 / 45.9, 2048 -> 14336 62.7 / 62.4, 1536
// -> 8960 37.3 / 39.5, 1024 -> 14336 41.5 / 49.1; 32 tokens, 2048 -> 2048 22.3 / 17.2, 2560 -> 2560 26.8 / 22.4, 3072 -> 3072 29.3 / 29.0,
// 5632 -> 4736 60.8 / 63.7, 4864 -> 8960 89.6 / 87.1, 14336 -> 4096 123 / 111, 6144 -> 10240 137 / 124, 5120 -> 13312 170 / 133, 11008 ->
// 11008 291 / 262.  (The double-channel step converts X and dY between the maxima and the GEMMs: 17 tokens, 5632 -> 4736 66 / 77.)
TI8_HD bool raw_weight_takes(int64_t tokens, int64_t K, int64_t N) {
    return tokens <= 32 && (tokens <= 16 || N * K <= 2560 * 2560 || N * K >= 14336 * 4096) && N <= 5 * K && K <= 10 * N && K <= 32768 && N <= 32768;
}
TI8_HD int64_t raw_row_offset(int n0, int64_t ldw, int kt, int i, int lane) { return (int64_t)(n0 + (lane & 15)) * ldw + kt * 128 + i * 32 + (lane >> 4) * 8; }
TI8_HD int64_t raw_row_codes_offset(int token, int64_t lda, int kt, int i, int lane) { return (int64_t)token * lda + kt * 128 + i * 32 + (lane >> 4) * 8; }
TI8_HD int64_t raw_col_base(int n0, int64_t ldw, int kt, int h, int j) { return (int64_t)(kt * 128 + h * 64 + j) * ldw + n0; }
TI8_HD uint32_t raw_col_lane_bytes(int64_t ldw, int lane) { return (uint32_t)((lane >> 4) * 16 * (int)ldw + (lane & 15) * 2) * 2u; }
TI8_HD int64_t raw_col_codes_offset(int token, int64_t lda, int kt, int h, int lane) { return (int64_t)token * lda + kt * 128 + h * 64 + (lane >> 4) * 16; }
// dW beside them: workgroups for its 128 x 128 tiles, worker w taking w, w + workers, ...
TI8_HD int64_t thin_workers(int64_t M, int64_t N, int64_t num_cu) {
    const int64_t tiles = (M / 128) * (N / 128);
    return tiles < num_cu ? tiles : num_cu;
}

// ---- column sums (bias.hip) -----------------------------------------------------------------------
// Workgroup -> strip of 32 columns of column_sum_narrow_kernel: two neighbours, which share cache lines, on one XCD
TI8_HD int column_strip(int block, int strips) {
    const int group = block & ~15;
    return group + 16 <= strips ? group + (block & 7) * 2 + ((block >> 3) & 1) : block;
}
// Whether that kernel makes the sums in its one launch.  us in a graph, two launches / one: 16 x 4096 4.5 / 3.3, 512 x 14336 6.1 / 5.6,
// 1500 x 5632 6.2 / 4.7, 3000 x 5632 8.4 / 7.4, 3000 x 1024 5.2 / 5.0; 4096 x 5632 11.3 / 12.0, 1500 x 14336 11.0 / 11.5, 16384 x 4096 25.5 / 35.1.
TI8_HD bool column_sum_narrow(int64_t rows, int64_t cols) { return rows <= (cols <= 8192 ? 3072 : 1024); }

// ---- attention's backward (attention.hip) ---------------------------------------------------------
// Workgroup -> (batch, head) pair and block of its rows: the blocks of a pair on one XCD, whose L2 then serves the rows that they all
// stream.  The grid has round8(pairs) * blocks workgroups; those of a pair beyond the last do nothing.
struct AttentionPlace {
    int pair, block;
};
TI8_HD AttentionPlace attention_place(uint32_t workgroup, int blocks) {
    const int idx = (int)(workgroup >> 3);
    return AttentionPlace{(idx / blocks) * 8 + (int)(workgroup & 7), idx % blocks};
}
// bytes from the first row of a pair to the last one's end: what lies behind reads as zeros
TI8_HD int64_t attention_bytes(int seq, int64_t stride, int head_dim) { return ((int64_t)(seq - 1) * stride + head_dim) * 2; }
TI8_HD bool attention_stride_ok(int64_t stride, int64_t seq, int64_t head_dim) {
    // (offsets are 32 bits and run up to 352 rows past the last one)
    return stride >= head_dim && stride <= 0x3fffffff / (seq + 512);
}

// ---- which kernel an entry point launches (decided on the host) ------------------------------

// per-row quantiser: NLOAD 16-byte chunks per thread, one wave (4 rows per workgroup) or one
// 256-thread workgroup per row, by the number of 16-byte chunks in a row.  Up to a row per CU (256) the time is that of
// one row, and a whole workgroup takes it (37 rows of 4096 3.4 us, a wave per row 3.9; the call with its GEMM, 4096 ->
// 14336, 15.9 and 16.4).  `plain`: no rotation, and the arithmetic of the reference's kernels (the others have no such form).
struct QRowConfig {
    int nload;
    bool wg_row;
};
TI8_HD QRowConfig qrow_config(int nchunk, bool group128, int64_t rows, bool plain) {
    QRowConfig c;
    if (!group128 && plain && rows <= 256 && nchunk <= 256 * 2 && nchunk > 64) {
        c.nload = 2;
        c.wg_row = true;
    } else if (group128) {
        c.nload = nchunk <= 256 * 8 ? 8 : 16;
        c.wg_row = nchunk > 64 * 8;
    } else if (nchunk <= 64 * 8) {
        c.nload = nchunk <= 64 * 2 ? 2 : (nchunk <= 64 * 4 ? 4 : 8);
        c.wg_row = false;
    } else {
        c.nload = nchunk <= 256 * 4 ? 4 : (nchunk <= 256 * 8 ? 8 : 16);
        c.wg_row = true;
    }
    return c;
}

// Walsh-Hadamard transform: elements per workgroup (a whole group of n when n >= 2048, else as
// many groups as divide both the row and 2048) and threads per workgroup
TI8_HD int64_t fwht_segment_len(int64_t cols, int64_t n) {
    if (n >= 2048 || cols < n) return n;    // cols < n: a zero-extended row of n elements per workgroup
    int64_t a = cols, b = 2048;
    while (b) {
        const int64_t t = a % b;
        a = b;
        b = t;
    }
    return a;  // gcd(cols, 2048), a multiple of n because n divides both
}
TI8_HD int fwht_threads(int64_t) { return 256; }   // fwht_kernel: segments of up to 2048 elements (longer ones: fwht_row_kernel)

// LDS-tiled GEMM: tile shape, waves and epilogue kind by shape and scale modes.  `epi` values are
// the EPI_* constants of gemm_args.h; `mid`: the 128 x 128 tiles run on the medium-size kernel (gemm_mid.hip).
struct GemmConfig {
    int bm, bn, wm, wn, epi, mid;
};
TI8_HD GemmConfig gemm_config(int64_t M, int64_t N, int64_t K, int64_t batch, bool acc_i32_full, bool strict, int modeA,
                              int modeB, bool large, int num_cu) {
    const int64_t tiles_256x256 = ((M + 255) / 256) * ((N + 255) / 256) * batch;
    const int64_t tiles_256x128 = ((M + 255) / 256) * (N / 128) * batch;
    const int64_t tiles_128x128 = ((M + 127) / 128) * (N / 128) * batch;
    // the fast promotion keeps at most 256 per-K-tile factors on chip and cannot apply a factor that varies per row of A
    // inside the loop: those cases take the literal kernel
    if (!acc_i32_full && (strict || modeA == 2 || K > 256 * 128)) return GemmConfig{128, 128, 2, 2, 3, 0};
    // operand B scaled per (row, K block): 256 x 256 tiles with the chained promotion where they fill the machine
    if (!acc_i32_full && modeB == 2) return (large || tiles_256x256 >= num_cu) ? GemmConfig{256, 256, 2, 4, 6, 0} : GemmConfig{256, 128, 4, 2, 4, 0};
    const GemmConfig big = acc_i32_full ? GemmConfig{256, 256, 2, 4, 1, 0} : GemmConfig{256, 256, 2, 4, 5, 0};
    const GemmConfig small = acc_i32_full ? GemmConfig{128, 128, 2, 2, 1, 0} : GemmConfig{128, 128, 2, 2, 2, 0};
    if (large) return big;
    // Measured at N = 4096, promotion / int32, us.  One 128 x 128 tile per CU at most: the medium-size kernel (1024 rows, K =
    // 14336: 75.5 / 63.9, four waves 109 / 73.8, 256 x 256 tiles 159 / 121; 384 rows, K = 4096: 24 / 20, 32 / 19, 50 / 39).
    if (tiles_128x128 <= num_cu) {
        GemmConfig c = small;
        c.mid = 1;
        return c;
    }
    // More than half a round of 256 x 256 tiles: idle CUs leave the others a higher clock, and the large tile moves half the
    // bytes per product (3072 rows, K = 4096, 192 tiles: 61 / 50, 256 x 128 tiles 80, 128 x 128 on four waves - / 55; 768
    // rows, N = 14336, 168 tiles: 57 / 46 against 79 / 53).
    if (2 * tiles_256x256 > num_cu) return big;
    // Exactly one round of 256 x 128 tiles (2048 rows, K = 4096: 46, against 54 on 256 x 256 and 55 on the medium-size kernel)
    if (!acc_i32_full && tiles_256x128 >= num_cu) return GemmConfig{256, 128, 4, 2, 2, 0};
    // In between, 128 x 128 tiles on four waves, two workgroups per CU (1536 rows, K = 4096, 384 tiles: 42 / 33, against 52 /
    // 41 on 256 x 256 tiles and 51 / 42 on the medium-size kernel, whose 129 KiB of LDS leave room for one).
    return small;
}

// ---- several GEMMs in one launch: the kernel for all of them ----------------------------------------------------------------
// A GEMM of its own pays for the last round of its tiles in full, so GEMMs that choose by their own shape and end up on different
// kernels leave CUs idle several times (640 tokens, 2048 -> 5632, three GEMMs of a step: 63 us, on one kernel together 48; 1280
// tokens, 1280 -> 1280: 25.6 / 18.3; 2560 tokens, 2048 -> 8192: 187 / 158).  The times below are fits, in us on 256 CUs, to 40
// launches of 2 and 3 GEMMs of 384 .. 7040 tokens and 1024 .. 14336 features: a constant, the K tiles of the busiest CU, the mean
// over the CUs, and what a tile or a round costs besides; off by 4 % in the mean and 11 % at most (int32: 21 %, on tiles that
// leave most CUs idle).  Against the choice by shape alone the launches take 0.93 of the time in the mean and 1.01 at worst.
// With another number of CUs the shares per CU follow it and the constants do not: the order of the kernels is then a guess, the
// results are the same (all of these kernels give the same bits).
struct GemmSet {
    int64_t M[3], N[3], nk[3];   // nk (K tiles) descending: the order of the launch
    int count;
};
TI8_HD int64_t gemm_set_tiles(const GemmSet& s, int i, int bm) { return ((s.M[i] + bm - 1) / bm) * ((s.N[i] + bm - 1) / bm); }
// 128 x 128 tiles on four waves, two workgroups per CU
TI8_HD double gemm_set_time_small(const GemmSet& s, bool i32, int num_cu) {
    const double slots = 2.0 * num_cu;
    double tiles = 0, work = 0;
    for (int i = 0; i < s.count; ++i) {
        tiles += (double)gemm_set_tiles(s, i, 128);
        work += (double)(gemm_set_tiles(s, i, 128) * s.nk[i]);
    }
    const double mean = work / slots, over = tiles <= slots ? mean : mean + 0.5 * (double)s.nk[s.count - 1];
    const double longest = over > (double)s.nk[0] ? over : (double)s.nk[0];
    // (a tile alone on its CU waits through its K loop, however little the others have to do)
    const double alone = i32 ? 5.0 + 0.62 * (double)s.nk[0] : 6.0 + 0.87 * (double)s.nk[0];
    const double t = i32 ? 5.0 + 0.28 * longest + 0.71 * mean + 2.9 * tiles / slots : 6.3 + 0.37 * longest + 0.96 * mean + 1.84 * tiles / slots;
    return t > alone ? t : alone;
}
// 256 x 256 tiles, by rounds; the persistent kernel by lists where that is less (measured / predicted, us: the GEMMs of a step, 1024 tokens,
// 4096 -> 11008 156 / 161, 1280, 3200 -> 6528 101 / 101, 1536, 2048 -> 5632 81 / 79; on four waves 165, 112, 90).  `lists`: whether a GEMM over 13, 15 or
// 17 K tiles, which that kernel takes beside others only, may be in one.  It may where the whole call is priced (whole steps, us, on four
// waves / so: 1664 tokens, 2560 -> 9216 213 / 183; 1920, 4096 -> 9216 346 / 313; 2176, 2048 -> 7680 187 / 156); by rounds it is no faster there (the backward
// of 2780 tokens, 3712 -> 1664 79 / 85), and two GEMMs of a call beside a launch of the medium-size kernel lose by going apart with it (1664
// tokens, 1024 -> 12288 0.955 of the speed, 1920, 12800 -> 1024 0.926, 2176, 1024 -> 11776 0.930).
TI8_HD double gemm_set_time_large(const GemmSet& s, bool i32, int num_cu, bool lists) {
    int64_t tiles[3], total = 0;
    double work = 0;
    for (int i = 0; i < s.count; ++i) {
        total += tiles[i] = gemm_set_tiles(s, i, 256);
        work += (double)(tiles[i] * s.nk[i]);
    }
    const int64_t rounds = (total + num_cu - 1) / num_cu;
    const double mean = work / num_cu, longest = (double)chain_rounds_busiest(tiles, s.nk, s.count, num_cu);
    if (i32) return 8.6 + 0.71 * longest + 0.95 * mean + 1.2 * (double)rounds;
    // a GEMM over few K tiles of an odd number keeps the launch off the persistent kernel
    bool odd = false, listed = s.count > 1;
    for (int i = 0; i < s.count; ++i) {
        odd = odd || !chain_takes((int)s.nk[i], false);
        listed = listed && chain_takes((int)s.nk[i], lists);
    }
    const double by_rounds = (7.7 + 1.15 * longest + 0.9 * mean + 0.4 * (double)rounds) * (odd ? 1.04 : 1.0);
    if (!listed || num_cu % 8 || num_cu / 8 > CHAIN_LIST_SLOTS || total > 8 * (CHAIN_LIST_MAX - s.count)) return by_rounds;
    int n[3], cost[3], first[CHAIN_LIST_SLOTS + 1];
    uint16_t order[CHAIN_LIST_MAX];
    double walked = 0;
    for (int i = 0; i < s.count; ++i) {
        n[i] = (int)((tiles[i] + 7) / 8);
        cost[i] = chain_tile_cost((int)s.nk[i]);
        walked += (double)(tiles[i] * chain_walked((int)s.nk[i])) / num_cu;
    }
    const double by_list = 7.7 + 0.546 * (double)(chain_list(n, cost, s.count, num_cu / 8, first, order) - 3) + 0.9 * walked;
    return by_list < by_rounds ? by_list : by_rounds;
}
// the medium-size kernel, one workgroup per CU: past one round a workgroup's turn-over is not hidden
TI8_HD double gemm_set_time_mid(const GemmSet& s, bool i32, int num_cu) {
    double tiles = 0, work = 0;
    for (int i = 0; i < s.count; ++i) {
        tiles += (double)gemm_set_tiles(s, i, 128) / num_cu;
        work += (double)(gemm_set_tiles(s, i, 128) * s.nk[i]) / num_cu;
    }
    if (tiles > 1.0) work += (double)s.nk[s.count - 1] + 10.0;   // the last tiles, and 6 us of turn-over
    const double longest = work > (double)s.nk[0] ? work : (double)s.nk[0];
    return 7.0 + 0.5 * longest * (0.85 + 0.3 * (tiles < 1.0 ? tiles : 1.0)) * (i32 ? 0.85 : 1.0);
}

// 256 x 128 tiles, one workgroup per CU
TI8_HD double gemm_set_time_half(const GemmSet& s, int num_cu) {
    double work = 0;
    for (int i = 0; i < s.count; ++i) work += (double)(((s.M[i] + 255) / 256) * (s.N[i] / 128) * s.nk[i]) / num_cu;
    return 6.0 + 1.25 * (work > (double)s.nk[0] ? work : (double)s.nk[0]);
}

// `c` holds what gemm_config selects for each shape {M, N, K}, and becomes what the launch is to use
TI8_HD void gemm_configs_together(const int64_t (*shape)[3], int count, bool large, int num_cu, GemmConfig* c) {
    if (large || count < 2) return;
    const bool i32 = c[0].epi == 1;
    GemmSet all = {}, mids = {}, bigs = {}, halves = {}, smalls = {};
    int order[3] = {0, 1, 2};
    for (int i = 1; i < count; ++i)
        for (int j = i; j > 0 && shape[order[j]][2] > shape[order[j - 1]][2]; --j) {
            const int t = order[j];
            order[j] = order[j - 1];
            order[j - 1] = t;
        }
    int64_t mid_tiles = 0;
    for (int q = 0; q < count; ++q) {
        const int i = order[q];
        // EPI_ROWS, or EPI_PROMOTE / EPI_PROMOTE_CHAIN: kernels that take each other's GEMMs
        if (i32 ? c[i].epi != 1 : (c[i].epi != 2 && c[i].epi != 5)) return;
        GemmSet* const sets[2] = {&all, c[i].mid ? &mids : (c[i].bn == 256 ? &bigs : (c[i].bm == 256 ? &halves : &smalls))};
        for (int k = 0; k < 2; ++k) {
            GemmSet& s = *sets[k];
            s.M[s.count] = shape[i][0];
            s.N[s.count] = shape[i][1];
            s.nk[s.count++] = shape[i][2] >> 7;
        }
        if (c[i].mid) mid_tiles += gemm_set_tiles(all, q, 128);
    }
    if (bigs.count == count || (mids.count == count && mid_tiles <= num_cu)) return;
    const double small = gemm_set_time_small(all, i32, num_cu), big = gemm_set_time_large(all, i32, num_cu, true);
    // A launch for each kernel chosen; not for several rounds of medium-size tiles, and with 15 % on top where the four-wave kernel is
    // among them (measured over predicted: 369 / 336 us, 193 / 168, 185 / 160 at 3200, 6016 and 2176 tokens)
    double apart = mids.count == count && 4 * mid_tiles >= 5 * (int64_t)num_cu ? 1e30 : 0.0;
    if (mids.count) apart += gemm_set_time_mid(mids, i32, num_cu);
    if (bigs.count) apart += gemm_set_time_large(bigs, i32, num_cu, false);
    if (halves.count) apart += gemm_set_time_half(halves, num_cu);
    if (smalls.count) apart = 1.15 * (apart + gemm_set_time_small(smalls, i32, num_cu));
    const double margin = 1.04;   // what the fits are off by
    if (apart <= margin * small && apart <= margin * big) return;
    for (int i = 0; i < count; ++i)
        c[i] = big < small ? GemmConfig{256, 256, 2, 4, i32 ? 1 : 5, 0} : GemmConfig{128, 128, 2, 2, i32 ? 1 : 2, 0};
}

// Up to 256 rows: us that the few-rows kernel takes with workgroups of one 32 x 32 block or of four.  Bound by the bytes of both
// operands that pass into a CU's LDS, 55 per ns; workgroups of one block are two to a CU and leave no last round to wait for, those of
// four are alone on theirs (and a further round costs 6 us more: waiting for its first loads, and the sums of the four waves).
TI8_HD double few_rows_time(int64_t M, int64_t N, int64_t K, int64_t batch, int num_cu, bool wide) {
    const int64_t groups = (wide ? ((M + 63) / 64) * (N / 64) : ((M + 31) / 32) * (N / 32)) * batch;
    const double rounds = wide ? (double)((groups + num_cu - 1) / num_cu) : groups > num_cu ? (double)groups / num_cu : 1.0;
    return 2.0 + rounds * (wide ? 128.0 : 64.0) * (double)K / 55000.0 + (wide ? 6.0 * (rounds - 1.0) : 0.0);
}
// Whether four blocks are the faster ones; over 9 weights and 32 to 256 rows the choice is 0.5 % behind the better of both, and 8 % ahead
// of one block everywhere.  Equal times go to four: training launches Y and dX together, where one block's two to a CU are taken.
TI8_HD bool few_rows_wide(int64_t M, int64_t N, int64_t K, int64_t batch, int num_cu) {
    return M > 32 && few_rows_time(M, N, K, batch, num_cu, true) <= few_rows_time(M, N, K, batch, num_cu, false);
}

// Up to 256 rows: whether the medium-size kernel beats the few-rows kernel.  Its time grows with the K tiles a workgroup walks (0.85 us
// per two of them alone, 1.15 with all CUs busy; N = 14336, K = 4096: 25 us at 128 rows, 26 at 256, where the few-rows kernel takes 27
// and 46).
TI8_HD bool gemm_few_rows_prefers_mid(int64_t M, int64_t N, int64_t K, int64_t batch, int num_cu) {
    const double nk = (double)(K >> 7), tiles = (double)(((M + 127) / 128) * (N / 128) * batch) / num_cu;
    if (tiles > 1.0 || K > 256 * 128) return false;
    return 7.0 + 0.5 * nk * (0.85 + 0.3 * tiles) < few_rows_time(M, N, K, batch, num_cu, few_rows_wide(M, N, K, batch, num_cu));
}

// Whether the few-rows kernel quantises up to 8 rows of bf16 itself.  A wave then spends about as long on a K tile's codes as on waiting for
// the weight's next one: over many K tiles on few CUs that adds up to more than the launch that it saves.  us, apart / in the kernel,
// 8 rows, calls one after another: K -> N 2048 -> 1024 12.7 / 10.5, 4096 -> 4096 13.3 / 10.3, 4096 -> 14336 15.6 / 11.9, 8192 -> 8192
// 16.8 / 14.1, 12288 -> 4096 18.4 / 18.2, 14336 -> 1024 18.0 / 18.6, 14336 -> 5120 20.4 / 20.9, 14336 -> 7168 22.1 / 20.8,
// 14336 -> 14336 35.4 / 31.3.  By rows, which are read twice: 2048 -> 1024 14.1 / 11.1, 4096 -> 4096 14.0 / 10.8, 4096 -> 14336 14.5 / 12.1,
// 8192 -> 8192 14.7 / 14.1, 10240 -> 4096 15.4 / 15.1, 11008 -> 1152 13.5 / 13.8, 12288 -> 4096 16.8 / 17.3, 14336 -> 8192 21.9 / 22.0,
// 14336 -> 10240 30.4 / 27.1, 14336 -> 14336 33.7 / 33.3.
TI8_HD bool decode_quantises(int64_t N, int64_t K, bool by_rows, int num_cu) {
    return by_rows ? K / 128 <= 80 || N / 32 > num_cu : K / 128 <= 96 || N / 32 * 4 >= (int64_t)num_cu * 3;
}

// Whether up to 8 rows go to the kernel that takes 16 rows of the weight per workgroup (gemm_decode.hip).  Every workgroup makes the codes of
// all rows: beyond one workgroup per CU that is what it spends its time on.  us, this one / gemm_i8_decode_kernel, at 1 row, 4 and 8:
// 1024 -> 1024 3.0 3.7 4.7 / 4.0, 2048 -> 1024 3.6 4.3 5.2 / 5.1, 4096 -> 4096 4.9 5.6 6.6 / 7.5, 12288 -> 4096 11.5 13.1 15.6 / 18.3,
// 14336 -> 5120 18.5 21.4 32.1 / 20.6, 8192 -> 8192 14.2 16.0 21.9 / 13.9, 4096 -> 14336 11.9 14.6 24.5 / 11.0.  By rows: 2048 -> 1024
// 3.9 4.9 6.3 / 5.7, 4096 -> 4096 5.4 6.6 7.8 / 8.5, 12288 -> 4096 12.2 14.2 17.2 / 17.6; apart, 14336 -> 1024 10.4 12.9 17.9 / 16.6.
TI8_HD bool decode_narrow(int64_t N, int64_t K, int64_t rows, bool by_rows, int num_cu) {
    const int64_t nk = K / 128;
    return N / 16 <= num_cu && (rows <= 4 || (nk >= 24 && (!by_rows || nk <= 96)));
}

}  // namespace idx
}  // namespace ti8
