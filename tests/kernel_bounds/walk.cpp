// Host-side walk over the launches of libti8's kernels: for the geometry an entry point would
// launch, visit every (workgroup, wave, lane, iteration) and check each global-memory access
// against the number of elements that lie between the pointer the caller passed and the end of
// its allocation.  The offsets come from triton-int8_amd/csrc/index_math.h, the same functions the
// kernels call; what is mirrored by hand here is only the order in which a kernel combines them
// (each such place cites the kernel's lines).  Built with g++ by tests/test_kernel_bounds.py: no
// GPU, no HIP.
//
// Every walk_* function returns 0 when all accesses are in bounds (and, for the GEMM, when every
// element of C is stored exactly once), else 1 with a description of the first violation in msg.
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>

#include "index_math.h"

using namespace ti8::idx;

namespace {

struct Report {
    char* msg;
    int len;
    bool bad = false;
    int64_t checked = 0;
    void fail(const char* fmt, ...) {
        if (bad) return;
        bad = true;
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(msg, len, fmt, ap);
        va_end(ap);
    }
    // access of `n` elements at element offset `off` of a buffer with `size` elements
    bool access(const char* what, int64_t off, int64_t n, int64_t size, int64_t a = -1, int64_t b = -1, int64_t c = -1, int64_t d = -1) {
        ++checked;
        if (off < 0 || off + n > size) {
            fail("%s: elements [%lld, %lld) outside the buffer of %lld (at %lld, %lld, %lld, %lld)", what, (long long)off,
                 (long long)(off + n), (long long)size, (long long)a, (long long)b, (long long)c, (long long)d);
            return false;
        }
        return true;
    }
};

}  // namespace

extern "C" {

// ti8_fwht -> fwht_kernel<NT, false> (fwht.hip): bf16 x [rows][cols] (ldx) -> y (ldy).
// quant: ti8_fwht_quant_row -> fwht_kernel<NT, true>: one workgroup per row (L = n), int8 q [rows][cols] (ldy = ldq, y_elems
// = bytes of q) and one fp32 scale per row (s_elems) instead of y
static int walk_fwht_impl(bool quant, int64_t ldx, int64_t ldy, int64_t rows, int64_t cols, int64_t n, int64_t x_elems, int64_t y_elems,
                          int64_t s_elems, int64_t lds_bytes_limit, int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    const int64_t L = quant ? n : fwht_segment_len(cols, n);
    if (quant && cols > n) r.fail("fwht_quant_row: %lld columns exceed the transform length %lld", (long long)cols, (long long)n);
    if (n >= 4096) {
        // fwht_row_kernel<CH, QUANT>: 4 waves, slice by slice through a 2 x 4096-word exchange buffer, results stored from registers
        const int CH = (int)(n / 4096);
        const bool extended = cols < L;
        const int valid = (int)(extended ? cols : L);
        const int segs_per_row = extended ? 1 : (int)(cols / L);
        const int64_t nblocks = rows * segs_per_row;
        const int64_t lds_words = (CH > 1 ? 2 : 1) * 4 * 64 * 16;
        if (lds_words * 4 > 65536) r.fail("fwht rows: %lld bytes of static LDS", (long long)(lds_words * 4));
        if (quant && segs_per_row != 1) r.fail("fwht_quant_row: %d segments per row", segs_per_row);
        std::vector<uint8_t> taken((size_t)L / 4, 0);   // every group of 4 output elements belongs to exactly one thread
        for (int tid = 0; tid < 256 && !r.bad; ++tid) {
            const int lane = tid & 63, w = tid >> 6, lp = (lane & ~15) | had_chunk(lane & 15);
            for (int k = 0; k < CH; ++k) {
                const int64_t base = (int64_t)(k & 1) * 4 * 64 * 16;
                for (int e = 0; e < 16; ++e) r.access("fwht rows lds write", base + fwht_row_lds(w, lp, e), 1, lds_words, tid, k, e);
                for (int ws = 0; ws < 4; ++ws) {
                    for (int e = 0; e < 4; ++e) r.access("fwht rows lds read", base + fwht_row_lds(ws, lp, 4 * w + e), 1, lds_words, tid, k, ws, e);
                    const int first = fwht_row_out(k, ws, lp, w);
                    if (first < 0 || first + 4 > L || first % 4) { r.fail("fwht rows: thread %d owns elements from %d of %lld", tid, first, (long long)L); break; }
                    ++taken[(size_t)first / 4];
                }
            }
            if (quant) r.access("fwht rows lds wave maxima", w, 1, lds_words, tid);
        }
        for (size_t i = 0; i < taken.size() && !r.bad; ++i)
            if (taken[i] != 1) r.fail("fwht rows: elements %lld.. are stored by %d threads", (long long)(i * 4), (int)taken[i]);
        for (int64_t block = 0; block < nblocks && !r.bad; ++block) {
            const int64_t xo = fwht_segment_offset(block, segs_per_row, ldx, (int)L);
            const int64_t yo = fwht_segment_offset(block, segs_per_row, ldy, (int)L);
            for (int tid = 0; tid < 256; ++tid) {
                const int lane = tid & 63, w = tid >> 6, lp = (lane & ~15) | had_chunk(lane & 15);
                for (int k = 0; k < CH; ++k) {
                    const int first = fwht_row_chunk_first(k, w, lp);
                    const int from = fwht_chunk_valid(first, 16, valid) ? first : 0;   // a chunk past the end re-reads the first one
                    r.access("fwht x", xo + from, 8, x_elems, block, tid, k);
                    r.access("fwht x", xo + from + 8, 8, x_elems, block, tid, k);
                    for (int ws = 0; ws < 4; ++ws) {
                        const int out = fwht_row_out(k, ws, lp, w);
                        if (fwht_chunk_valid(out, 4, valid)) r.access(quant ? "fwht q" : "fwht y", yo + out, 4, y_elems, block, tid, k, ws);
                    }
                }
                if (quant && tid == 0) r.access("fwht s", block, 1, s_elems, block);
            }
        }
        *n_checked = r.checked;
        return r.bad;
    }
    const int NT = fwht_threads(L);
    const bool extended = cols < L;             // a zero-extended row per workgroup
    const int valid = (int)(extended ? cols : L);
    const int64_t nblocks = rows * (extended ? 1 : cols / L);
    const int64_t lds_words = fwht_lds_words(L);
    if (lds_words * 4 > lds_bytes_limit) r.fail("fwht: %lld bytes of LDS requested, limit %lld", (long long)(lds_words * 4), (long long)lds_bytes_limit);
    int logn = 0;
    while ((1LL << logn) < n) ++logn;
    const int segs_per_row = extended ? 1 : (int)(cols / L);
    // LDS indices do not depend on the workgroup: walk them once
    // segments of 1024 elements and more run bits 4..9 across the lanes of a wave (lane l of a row of 16 takes chunk
    // had_chunk(l)); that needs whole waves of chunks
    const bool by_lanes = L >= 1024;
    if (by_lanes && ((L >> 4) % 64)) r.fail("fwht: %lld chunks are not whole waves", (long long)(L >> 4));
    for (int tid = 0; tid < NT && !r.bad; ++tid) {
        for (int v0 = tid; v0 < (L >> 4); v0 += NT) {
            const int vt = by_lanes ? ((v0 & ~15) | had_chunk(v0 & 15)) : v0;
            for (int e = 0; e < 16; ++e) r.access("fwht lds first pass", vt * 17 + e, 1, lds_words, tid, vt, e);
        }
        auto pass = [&](int p, int rb) {   // pass_in_lds<RB, NT>
            const int ngroups = (int)(L >> rb);
            for (int vt = tid; vt < ngroups; vt += NT) {
                const int base = fwht_group_base(vt, p, rb);
                for (int e = 0; e < (1 << rb); ++e) r.access("fwht lds pass", fwht_padded(base + (e << p)), 1, lds_words, tid, vt, e, p);
            }
        };
        if (by_lanes) {
            if (logn - 10 > 0) pass(10, logn - 10);
        } else {
            const int rb1 = imin(4, logn - 4);
            pass(4, rb1);
            int rem = logn - 8;
            if (rem > 0) {
                const int rb2 = rem <= 5 ? rem : (rem + 1) / 2;
                pass(8, rb2);
                rem -= rb2;
                if (rem > 0) pass(8 + rb2, rem);
            }
        }
        if (quant) {   // one chunk per thread is kept in registers; the first words of LDS then hold one maximum per wave
            if (tid < (L >> 3)) r.access("fwht lds read-back", fwht_padded(tid * 8), 8, lds_words, tid);
            r.access("fwht lds wave maxima", tid >> 6, 1, lds_words, tid);
        } else {
            for (int c = tid; c < (L >> 3); c += NT) r.access("fwht lds read-back", fwht_padded(c * 8), 8, lds_words, tid, c);
        }
    }
    if (quant && (L >> 3) > NT) r.fail("fwht_quant_row: %lld chunks do not fit one per thread on %d threads", (long long)(L >> 3), NT);
    for (int64_t block = 0; block < nblocks && !r.bad; ++block) {
        const int64_t xo = fwht_segment_offset(block, segs_per_row, ldx, (int)L);
        const int64_t yo = fwht_segment_offset(block, segs_per_row, ldy, (int)L);
        for (int tid = 0; tid < NT; ++tid) {
            for (int v0 = tid; v0 < (L >> 4); v0 += NT) {   // two 16-byte loads: elements vt*16 .. +16
                const int vt = by_lanes ? ((v0 & ~15) | had_chunk(v0 & 15)) : v0;
                if (!fwht_chunk_valid(vt * 16, 16, valid)) continue;
                r.access("fwht x", xo + vt * 16, 8, x_elems, block, tid, vt);
                r.access("fwht x", xo + vt * 16 + 8, 8, x_elems, block, tid, vt);
            }
            for (int c = tid; c < (L >> 3); c += NT)
                if (fwht_chunk_valid(c * 8, 8, valid)) r.access(quant ? "fwht q" : "fwht y", yo + c * 8, 8, y_elems, block, tid, c);
            if (quant && tid == 0) r.access("fwht s", block, 1, s_elems, block);
        }
    }
    *n_checked = r.checked;
    return r.bad;
}
int walk_fwht(int64_t ldx, int64_t ldy, int64_t rows, int64_t cols, int64_t n, int64_t x_elems, int64_t y_elems,
              int64_t lds_bytes_limit, int64_t* n_checked, char* msg, int msglen) {
    return walk_fwht_impl(false, ldx, ldy, rows, cols, n, x_elems, y_elems, 0, lds_bytes_limit, n_checked, msg, msglen);
}
int walk_fwht_quant_row(int64_t ldx, int64_t ldq, int64_t rows, int64_t cols, int64_t n, int64_t x_elems, int64_t q_elems, int64_t s_elems,
                        int64_t lds_bytes_limit, int64_t* n_checked, char* msg, int msglen) {
    return walk_fwht_impl(true, ldx, ldq, rows, cols, n, x_elems, q_elems, s_elems, lds_bytes_limit, n_checked, msg, msglen);
}

// transpose_bf16_kernel (fwht.hip): x bf16 [R][C] (ldx) -> y bf16 [C][R] (ldy), 64 x 64 tiles
static void walk_transpose_tiles(Report& r, int64_t ldx, int64_t ldy, int64_t R, int64_t C, int64_t x_elems, int64_t y_elems) {
    if (R % 64 || C % 64) { r.fail("transpose: %lld x %lld is not made of 64 x 64 tiles", (long long)R, (long long)C); return; }
    const int tiles_c = (int)(C / 64);
    for (int64_t block = 0; block < (R / 64) * (C / 64) && !r.bad; ++block) {
        const int64_t tc = block % tiles_c, tr = block / tiles_c;
        for (int tid = 0; tid < 256; ++tid)
            for (int h = 0; h < 2; ++h) {
                const int a = (tid >> 3) + 32 * h, b = (tid & 7) * 8;
                r.access("fwht_t transpose x", (tr * 64 + a) * ldx + tc * 64 + b, 8, x_elems, block, tid, h);
                r.access("fwht_t transpose y", (tc * 64 + a) * ldy + tr * 64 + b, 8, y_elems, block, tid, h);
            }
    }
}
int walk_transpose_bf16(int64_t ldx, int64_t ldy, int64_t R, int64_t C, int64_t x_elems, int64_t y_elems, int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    walk_transpose_tiles(r, ldx, ldy, R, C, x_elems, y_elems);
    *n_checked = r.checked;
    return r.bad;
}

// ti8_fwht_t -> fwht_t_kernel<NT, W> (fwht.hip): x bf16 [R][C] (ldx) -> y bf16 [C][R] (ldy)
int walk_fwht_t(int64_t ldx, int64_t ldy, int64_t R, int64_t C, int64_t x_elems, int64_t y_elems, int64_t lds_bytes_limit,
                int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    if (!fwht_t_direct(R, C)) {
        // transpose_bf16_kernel: 64 x 64 tiles, thread t reads 8 columns of rows t/8 and t/8 + 32 and writes 8 rows
        // of columns t/8 and t/8 + 32; then fwht_kernel in place on y [C][R]
        walk_transpose_tiles(r, ldx, ldy, R, C, x_elems, y_elems);
        int64_t n2 = 0;
        const int bad = r.bad ? 1 : walk_fwht(ldy, ldy, C, R, R, y_elems, y_elems, lds_bytes_limit, &n2, msg, msglen);
        *n_checked = r.checked + n2;
        return bad;
    }
    const int W = fwht_t_cols_per_wg(R);
    const int NT = (int64_t)W * R >= 16384 ? 1024 : 256;
    const int64_t nblocks = C / W;
    const int64_t Lp = fwht_lds_words(R), lds_words = (int64_t)W * Lp;
    if (C % W) r.fail("fwht_t: %lld columns are not a multiple of %d per workgroup", (long long)C, W);
    if (lds_words * 4 > lds_bytes_limit) r.fail("fwht_t: %lld bytes of LDS requested, limit %lld", (long long)(lds_words * 4), (long long)lds_bytes_limit);
    int logn = 0;
    while ((1LL << logn) < R) ++logn;
    // LDS indices (the same for every workgroup)
    for (int tid = 0; tid < NT && !r.bad; ++tid) {
        for (int row = tid; row < R; row += NT)
            for (int w = 0; w < W; ++w) r.access("fwht_t lds fill", w * Lp + fwht_padded(row), 1, lds_words, tid, row, w);
        auto pass = [&](int p, int rb) {   // pass_in_lds_segments<RB, NT>
            const int per_seg = (int)(R >> rb);
            for (int vt = tid; vt < W * per_seg; vt += NT) {
                const int base = fwht_group_base(vt % per_seg, p, rb);
                for (int e = 0; e < (1 << rb); ++e)
                    r.access("fwht_t lds pass", (vt / per_seg) * Lp + fwht_padded(base + (e << p)), 1, lds_words, tid, vt, e, p);
            }
        };
        pass(0, 4);
        pass(4, imin(4, logn - 4));
        int rem = logn - 8;
        if (rem > 0) {
            const int rb2 = rem <= 5 ? rem : (rem + 1) / 2;
            pass(8, rb2);
            rem -= rb2;
            if (rem > 0) pass(8 + rb2, rem);
        }
        const int per_seg = (int)(R >> 3);
        for (int i = tid; i < W * per_seg; i += NT) r.access("fwht_t lds read-back", (i / per_seg) * Lp + fwht_padded((i % per_seg) * 8), 8, lds_words, tid, i);
    }
    std::vector<uint8_t> seen((size_t)nblocks, 0);
    for (int64_t block = 0; block < nblocks && !r.bad; ++block) {
        const int64_t cb = fwht_t_colblock(block, nblocks, W);
        if (cb < 0 || cb >= nblocks) { r.fail("fwht_t: workgroup %lld maps to column block %lld of %lld", (long long)block, (long long)cb, (long long)nblocks); break; }
        ++seen[(size_t)cb];
        const int64_t c0 = cb * W;
        for (int tid = 0; tid < NT; ++tid) {
            for (int row = tid; row < R; row += NT) r.access("fwht_t x", (int64_t)row * ldx + c0, W, x_elems, block, tid, row);
            const int per_seg = (int)(R >> 3);
            for (int i = tid; i < W * per_seg; i += NT) r.access("fwht_t y", (c0 + i / per_seg) * ldy + (int64_t)(i % per_seg) * 8, 8, y_elems, block, tid, i);
        }
    }
    for (int64_t cb = 0; cb < nblocks && !r.bad; ++cb)
        if (seen[(size_t)cb] != 1) r.fail("fwht_t: column block %lld is transformed %d times", (long long)cb, (int)seen[(size_t)cb]);
    *n_checked = r.checked;
    return r.bad;
}

// ti8_quant_row -> quant_row_kernel<NLOAD, WG_ROW, GROUP16, HAD> (quant.hip)
int walk_quant_row_form(int64_t ldx, int64_t ldq, int64_t rows, int64_t cols, int group, int plain, int64_t x_elems, int64_t q_elems,
                        int64_t s_elems, int* form, int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    const int nchunk = (int)(cols / 8);
    const QRowConfig cfg = qrow_config(nchunk, group == 128, rows, plain != 0);
    if (form) { form[0] = cfg.nload; form[1] = cfg.wg_row; }
    const int64_t grid = cfg.wg_row ? rows : (rows + 3) / 4;
    const int T = cfg.wg_row ? 256 : 64;
    const int ngrp = (int)(cols >> 7);
    std::vector<uint8_t> seen((size_t)rows, 0);
    for (int64_t block = 0; block < grid && !r.bad; ++block)
        for (int tid = 0; tid < 256; ++tid) {
            const int t = cfg.wg_row ? tid : (tid & 63);
            const int64_t row = qrow_row(block, tid >> 6, cfg.wg_row);
            if (row >= rows) continue;
            if (t == 0) ++seen[(size_t)row];
            for (int i = 0; i < cfg.nload; ++i) {
                const int c = qrow_chunk(t, i, T);
                if (c >= nchunk) continue;
                r.access("quant_row x", row * ldx + c * 8, 8, x_elems, block, tid, i);
                r.access("quant_row q", row * ldq + c * 8, 8, q_elems, block, tid, i);
                if (group == 128 && (c & 15) == 0) r.access("quant_row s", row * ngrp + (c >> 4), 1, s_elems, block, tid, i);
            }
            if (group != 128 && t == 0) r.access("quant_row s", row, 1, s_elems, block, tid);
        }
    // every chunk of a row is taken by exactly one (thread, load): T * NLOAD covers the row
    if ((int64_t)T * cfg.nload < nchunk) r.fail("quant_row: %d threads x %d loads do not cover %d chunks", T, cfg.nload, nchunk);
    for (int64_t row = 0; row < rows && !r.bad; ++row)
        if (seen[(size_t)row] != 1) r.fail("quant_row: row %lld handled %d times", (long long)row, (int)seen[(size_t)row]);
    *n_checked = r.checked;
    return r.bad;
}
int walk_quant_row(int64_t ldx, int64_t ldq, int64_t rows, int64_t cols, int group, int64_t x_elems, int64_t q_elems,
                   int64_t s_elems, int64_t* n_checked, char* msg, int msglen) {
    return walk_quant_row_form(ldx, ldq, rows, cols, group, 1, x_elems, q_elems, s_elems, nullptr, n_checked, msg, msglen);
}

// ti8_quant_block -> quant_block_kernel<NSUB, WRITE_Q, WRITE_QT> (quant.hip)
int walk_quant_block(int64_t bsx, int64_t ldx, int has_q, int64_t bsq, int64_t ldq, int has_qt, int64_t bsqt, int64_t ldqt,
                     int64_t ssb, int64_t ssr, int64_t ssc, int64_t B, int64_t R, int64_t C, int group_c, int64_t x_elems,
                     int64_t q_elems, int64_t qt_elems, int64_t s_elems, int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    const int nsub = group_c / 128;
    const int nrb = (int)(R / 128), ncb = (int)(C / group_c);
    const int64_t ntiles = B * nrb * ncb;
    for (int64_t block = 0; block < ntiles && !r.bad; ++block) {
        const TileId t = qblock_tile((int)block, nrb, ncb);
        const int64_t xo = qblock_origin(t.b, bsx, t.rb, ldx, t.cb, 128 * nsub);
        r.access("quant_block s", t.b * ssb + t.rb * ssr + t.cb * ssc, 1, s_elems, block);
        for (int tid = 0; tid < 256; ++tid) {
            for (int u = 0; u < nsub; ++u)
                for (int h = 0; h < 2; ++h)
                    for (int j = 0; j < 4; ++j) {
                        const int row = qblock_row(tid, h, j);
                        r.access("quant_block x", xo + (int64_t)row * ldx + u * 128 + qblock_col(tid), 8, x_elems, block, tid, h, j);
                        if (has_q)
                            r.access("quant_block q", qblock_origin(t.b, bsq, t.rb, ldq, t.cb, 128 * nsub) + u * 128 + qblock_col(tid) + (int64_t)row * ldq,
                                     8, q_elems, block, tid, h, j);
                    }
            if (has_qt) {
                const int64_t qo = qblock_origin(t.b, bsqt, t.cb, ldqt, t.rb, 128);
                for (int p = 0; p < 4; ++p) r.access("quant_block qT", qo + (int64_t)qblock_t_row(tid, p) * ldqt + qblock_t_col(tid), 16, qt_elems, block, tid, p);
            }
        }
    }
    *n_checked = r.checked;
    return r.bad;
}

// Partial maxima of an operand [R][C] (quant.hip: maxima_part, quant_rowcol_multi_kernel): every element that exists read once, every word of
// both arrays stored once, row maxima inside their LDS, 16-byte accesses on 16-byte boundaries; the conversion of every tile
// reads all parts' maxima of its own rows and columns.  x_elems elements of x, `words` 32-bit words of scratch.
int walk_maxima(int64_t R, int64_t C, int64_t valid, int64_t ldx, int64_t x_elems, int64_t words, int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    const MaximaParts m = maxima_parts(R, C);
    const int64_t cols0 = (int64_t)m.nct * R, halves = 2 * words;
    std::vector<uint8_t> stored((size_t)halves, 0), read((size_t)((R / 128) * (C / 128)), 0);
    for (int part = 0; part < m.nrt * m.nct && !r.bad; ++part) {
        const int ct = part % m.nct, rt = part / m.nct;
        const int rtiles = imin(m.tr, (int)(R >> 7) - rt * m.tr), ctiles = imin(m.tc, (int)(C >> 7) - ct * m.tc);
        if (rtiles < 1 || ctiles < 1) { r.fail("maxima: part %d has %d x %d tiles", part, rtiles, ctiles); break; }
        auto store = [&](const char* what, int64_t at, int n) {
            if (at % n) r.fail("%s: %lld is not a multiple of %d", what, (long long)at, n);
            if (r.access(what, at, n, halves, part))
                for (int e = 0; e < n; ++e) ++stored[(size_t)(at + e)];
        };
        for (int a = 0; a < rtiles; ++a)
            for (int b = 0; b < ctiles; ++b) {
                ++read[(size_t)((rt * m.tr + a) * (C / 128) + ct * m.tc + b)];
                for (int tid = 0; tid < 256; ++tid)
                    for (int i = 0; i < 8; ++i) {
                        const int64_t row = (rt * m.tr + a) * 128 + (tid >> 4) * 8 + i;
                        if (row < valid) r.access("maxima x", row * ldx + (ct * m.tc + b) * 128 + (tid & 15) * 8, 8, x_elems, part, tid, i);
                    }
            }
        for (int rg = 0; rg < 16; ++rg)
            for (int a = 0; a < rtiles; ++a) {
                r.access("maxima LDS", a * 128 + rg * 8, 8, MAXIMA_ROW_TILES * 128, part, rg, a);
                store("maxima rows", maxima_rows_at(ct, R, (rt * m.tr + a) * 128 + rg * 8), 8);
            }
        for (int b = 0; b < ctiles; ++b)
            for (int tid = 0; tid < 64; ++tid) store("maxima columns", cols0 + maxima_cols_at(rt, C, (ct * m.tc + b) * 128) + 2 * tid, 2);
    }
    for (size_t i = 0; i < read.size() && !r.bad; ++i)
        if (read[i] != 1) r.fail("maxima: tile %zu is read %d times", i, (int)read[i]);
    for (size_t i = 0; i < stored.size() && !r.bad; ++i)
        if (stored[i] != 1) r.fail("maxima: half word %zu is stored %d times", i, (int)stored[i]);
    for (int64_t tile = 0; tile < (R / 128) * (C / 128) && !r.bad; ++tile) {
        const int64_t cb = tile % (C / 128), rb = tile / (C / 128);
        for (int chunk = 0; chunk < 16; ++chunk) {
            for (int p = 0; p < m.nrt; ++p) r.access("conversion: columns", cols0 + cb * 128 + chunk * 8 + p * C, 8, halves, tile, p);
            for (int p = 0; p < m.nct; ++p) r.access("conversion: rows", rb * 128 + chunk * 8 + p * R, 8, cols0, tile, p);
        }
    }
    if (cols0 % 8 || C % 8) r.fail("conversion: columns' maxima off 16-byte boundaries");
    *n_checked = r.checked;
    return r.bad;
}

int64_t maxima_scratch_words(int64_t R, int64_t C) { return maxima_words(R, C); }

// Workgroups of the two launches (quant_call, quant_first_kernel, quant_rowcol_multi_kernel) for `count` operands quantised both ways, beside
// `block_tiles` tiles of block-quantised ones and `row_groups` workgroups of rows: each part and each tile belongs to one workgroup.
int walk_quant_call(const int64_t* R, const int64_t* C, int count, int block_tiles, int row_groups, int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    int first_part[4] = {0, 0, 0, 0}, first_tile[4] = {0, 0, 0, 0}, parts = 0, tiles = 0;
    std::vector<std::vector<int>> part_seen(count), tile_seen(count);
    for (int i = 0; i < 3; ++i) {
        first_part[i] = parts; first_tile[i] = tiles;
        if (i >= count) continue;
        const MaximaParts m = maxima_parts(R[i], C[i]);
        part_seen[i].assign(m.nrt * m.nct, 0);
        tile_seen[i].assign((R[i] / 128) * (C[i] / 128), 0);
        parts += (int)round8(m.nrt * m.nct);
        tiles += (int)round8((R[i] / 128) * (C[i] / 128));
    }
    const int blocks_end = (int)round8(block_tiles), rows_end = (int)round8(row_groups);
    int blocks = 0;
    for (int w = 0; w < rows_end + blocks_end + parts && !r.bad; ++w) {
        const int tile = w - rows_end, part = tile - blocks_end;
        ++r.checked;
        if (tile < 0) continue;
        if (part < 0) { blocks += tile < block_tiles; continue; }
        const int i = operand_of(part, first_part, count), at = part - first_part[i];
        if (at < 0 || at >= (int)round8((int64_t)part_seen[i].size())) r.fail("first launch: workgroup %d takes part %d of operand %d", w, at, i);
        else if (at < (int)part_seen[i].size()) ++part_seen[i][at];
        if (at == 0 && w % 8) r.fail("first launch: operand %d starts at workgroup %d", i, w);
    }
    if (blocks != block_tiles) r.fail("first launch: %d of %d block tiles", blocks, block_tiles);
    for (int w = 0; w < tiles && !r.bad; ++w) {
        const int tile = rowcol_multi_tile(w, tiles);
        ++r.checked;
        if (tile < 0 || tile >= tiles || tile % 8 != w % 8) { r.fail("conversion: workgroup %d takes tile %d", w, tile); break; }
        const int i = operand_of(tile, first_tile, count), at = tile - first_tile[i];
        if (at / (int)(C[i] / 128) < R[i] / 128) ++tile_seen[i][at];
    }
    for (int i = 0; i < count && !r.bad; ++i) {
        for (size_t k = 0; k < part_seen[i].size(); ++k)
            if (part_seen[i][k] != 1) r.fail("first launch: part %zu of operand %d is taken %d times", k, i, part_seen[i][k]);
        for (size_t k = 0; k < tile_seen[i].size(); ++k)
            if (tile_seen[i][k] != 1) r.fail("conversion: tile %zu of operand %d is taken %d times", k, i, tile_seen[i][k]);
    }
    *n_checked = r.checked;
    return r.bad;
}

// GEMM with few rows (gemm_skinny.hip: wavering_block), workgroups of one 32 x 32 block or of four (`wide`); scales by rows.  rows > 0: up to 8
// rows of bf16 that it quantises itself (a_elems in bf16).  Every element of C that exists is stored once, every K tile is walked once.
int walk_few_rows(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int wide, int rows, int64_t a_elems, int64_t b_elems, int64_t c_elems,
                  int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    const int MB = wide ? 2 : 1, NB = MB, nk = (int)(K >> 7);
    const int64_t b_at = rows ? 0 : MB * 4096, stage_bytes = b_at + NB * 4096, per_wave = 2 * stage_bytes + (rows ? 1024 : 0);
    const int64_t lds = rows ? 4 * per_wave + 4 * 8 * 4 : wide ? 131072 : 65536;
    const int mtiles = (int)((M + 32 * MB - 1) / (32 * MB)), nstrips = (int)(N / (32 * NB));
    std::vector<uint8_t> stored((size_t)(M * N), 0);
    const int64_t blocks = few_blocks(M, N, wide != 0);
    if (rows && M != 32) r.fail("decode: %lld rows of C", (long long)M);
    for (int64_t block = 0; block < blocks && !r.bad; ++block) {
        const FewPlace p = few_place((int)block, mtiles, nstrips);
        const int n0 = p.strip * 32 * NB, m0 = p.mt * 32 * MB, mblocks = imin(MB, ((int)M - m0) >> 5);
        if (mblocks < 1 || n0 >= N) { r.fail("few rows: workgroup %lld has no block (%d, %d)", (long long)block, m0, n0); break; }
        std::vector<uint8_t> walked((size_t)nk, 0);
        for (int wave = 0; wave < 4; ++wave) {
            const int kbeg = few_k_first(wave, nk), nq = few_k_first(wave + 1, nk) - kbeg;
            const int rot = nq > 0 && !wide ? (int)((((unsigned)block >> 3) * 3u) % (unsigned)nq) : 0;
            for (int i = 0; i <= nq; ++i) {         // one stage is fetched ahead
                const int kt = few_k_tile(i, rot, kbeg, nq, nk);
                if (kt < 0 || kt >= nk) { r.fail("few rows: K tile %d of %d", kt, nk); break; }
                if (i < nq) ++walked[(size_t)kt];
                const int64_t stage = wave * per_wave + (i & 1) * stage_bytes;
                for (int lane = 0; lane < 64; ++lane) {
                    const int ld_row = lane >> 3;
                    if (rows) {
                        const int64_t at = imin(ld_row, rows - 1) * lda + (lane & 7) * 16 + kt * 128;
                        r.access("few rows X", at, 8, a_elems, block, wave, lane, kt);
                        r.access("few rows X", at + 8, 8, a_elems, block, wave, lane, kt);
                        r.access("few rows LDS codes", wave * per_wave + 2 * stage_bytes + ld_row * 128 + ((lane & 7) ^ ld_row) * 16, 16, lds, block, wave, lane);
                    }
                    for (int b = 0; b < MB; ++b)
                        for (int q = 0; q < 4; ++q) {
                            const int64_t chunk = ((lane & 7) ^ ld_row ^ (q & 1)) * 16;
                            if (!rows) {
                                r.access("few rows A", (m0 + imin(b, mblocks - 1) * 32 + 8 * q + ld_row) * lda + kt * 128 + chunk, 16, a_elems, block, wave, lane, kt);
                                r.access("few rows LDS A", stage + b * 4096 + q * 1024 + lane * 16, 16, stage + b_at, block, wave, lane, q);
                            }
                            r.access("few rows B", (n0 + b * 32 + 8 * q + ld_row) * ldb + kt * 128 + chunk, 16, b_elems, block, wave, lane, kt);
                            r.access("few rows LDS B", stage + b_at + b * 4096 + q * 1024 + lane * 16, 16, stage + stage_bytes, block, wave, lane, q);
                        }
                }
            }
            r.access("few rows LDS", wave * per_wave, per_wave, lds, block, wave);
        }
        for (int kt = 0; kt < nk && !r.bad; ++kt)
            if (walked[(size_t)kt] != 1) r.fail("few rows: workgroup %lld walks K tile %d %d times", (long long)block, kt, (int)walked[(size_t)kt]);
        r.access("few rows LDS sums", 0, (int64_t)MB * NB * 4 * 32 * 32 * 4, lds, block);
        for (int t = 0; t < 256; ++t)
            for (int i = 0; i < mblocks; ++i)
                for (int j = 0; j < NB; ++j) {
                    const int row = m0 + i * 32 + (t >> 3), col = n0 + j * 32 + (t & 7) * 4;
                    if (!r.access("few rows C", row * ldc + col, 4, c_elems, block, t, i, j) || row >= M || col + 4 > N) { r.fail("few rows: C(%d, %d)", row, col); continue; }
                    for (int c = 0; c < 4; ++c) ++stored[(size_t)(row * N + col + c)];
                }
    }
    for (size_t i = 0; i < stored.size() && !r.bad; ++i)
        if (stored[i] != 1) r.fail("few rows: C(%lld, %lld) is stored %d times", (long long)(i / N), (long long)(i % N), (int)stored[i]);
    *n_checked = r.checked;
    return r.bad;
}

// Y of up to 8 rows, 16 columns per workgroup (gemm_decode.hip): every K tile of the rows and of the weight is read where it is and used once by
// one of the waves, every element of C stored once
int walk_decode_narrow(int rows, int64_t N, int64_t K, int64_t ldx, int64_t ldb, int64_t ldc, int64_t x_elems, int64_t b_elems, int64_t c_elems,
                       int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    const int nk = (int)(K >> 7);
    std::vector<uint8_t> stored((size_t)(rows * N), 0);
    for (int64_t block = 0; block < N / 16 && !r.bad; ++block) {
        const int n0 = (int)block * 16;
        std::vector<uint8_t> used((size_t)nk, 0);
        for (int wave = 0; wave < 4; ++wave) {
            const int kbeg = few_k_first(wave, nk), nq = few_k_first(wave + 1, nk) - kbeg, rot = decode_rot(n0, nq);
            if (rot != (nq > 0 ? (int)((((unsigned)(n0 / 32) >> 3) * 3u) % (unsigned)nq) : 0)) r.fail("decode narrow: another walk than that of the block of 32 columns");
            for (int batch = 0; batch == 0 || batch * DECODE_BATCH < nq; ++batch)
                for (int lane = 0; lane < 64; ++lane) {
                    for (int row = 0; row < rows; ++row) {
                        const int64_t at = decode_x_offset(row, ldx, few_k_tile(batch * DECODE_BATCH + (lane >> 3), rot, kbeg, nq, nk), lane);
                        r.access("decode narrow X", at, 8, x_elems, block, wave, lane, batch);
                        r.access("decode narrow X", at + 8, 8, x_elems, block, wave, lane, batch);
                    }
                    for (int t = batch * DECODE_BATCH; t < nq && t < (batch + 1) * DECODE_BATCH; ++t)
                        for (int h = 0; h < 2; ++h) r.access("decode narrow W", decode_w_offset(n0, ldb, few_k_tile(t, rot, kbeg, nq, nk), lane) + 64 * h, 16, b_elems, block, wave, lane, t);
                }
            for (int t = 0; t < nq; ++t) ++used[(size_t)few_k_tile(t, rot, kbeg, nq, nk)];
        }
        for (int kt = 0; kt < nk && !r.bad; ++kt)
            if (used[(size_t)kt] != 1) r.fail("decode narrow: workgroup %lld uses K tile %d %d times", (long long)block, kt, (int)used[(size_t)kt]);
        for (int lane = 0; lane < 64; ++lane) {
            const int row = lane & 15, col = n0 + (lane >> 4) * 4;
            if (row >= rows) continue;
            if (!r.access("decode narrow C", row * ldc + col, 4, c_elems, block, 0, lane) || col + 4 > N) continue;
            for (int c = 0; c < 4; ++c) ++stored[(size_t)(row * N + col + c)];
        }
    }
    for (size_t i = 0; i < stored.size() && !r.bad; ++i)
        if (stored[i] != 1) r.fail("decode narrow: C(%lld, %lld) is stored %d times", (long long)(i / N), (long long)(i % N), (int)stored[i]);
    *n_checked = r.checked;
    return r.bad;
}

// parts of a weight's maxima, the larger number of either direction
int raw_weight_parts(int64_t R, int64_t C) {
    const MaximaParts p = maxima_parts(R, C);
    return p.nrt > p.nct ? p.nrt : p.nct;
}

// Y (cols = 0) or dX of a step on few tokens from the weight itself, W [R][C] (gemm_skinny.hip: raw_block): every element of the weight is read by one
// lane, every K tile used by one wave of a workgroup against the codes of the same places, every element of the output's first 32 rows stored once
int walk_raw_weight(int cols, int tokens, int64_t R, int64_t C, int64_t ldw, int64_t lda, int64_t ldc, int64_t w_elems, int64_t a_elems, int64_t c_elems,
                    int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    const int width = cols ? RAW_STRIP_DX : RAW_STRIP_Y, strips = (int)((cols ? C : R) / width), nk = (int)((cols ? R : C) >> 7), blocks = tokens > 16 ? 2 : 1;
    const int64_t n = cols ? C : R;
    std::vector<uint8_t> read((size_t)(R * C), 0), stored((size_t)(32 * n), 0);
    for (int block = 0; block < strips && !r.bad; ++block) {
        const int n0 = (cols ? column_strip(block, strips) : block) * width;
        for (int wave = 0; wave < 4; ++wave) {
            const int kbeg = few_k_first(wave, nk), nq = few_k_first(wave + 1, nk) - kbeg, rot = decode_rot(n0, nq);
            if (nq > 64) r.fail("raw weight: %d K tiles of a wave", nq);
            for (int step = 0; step < nq; ++step) {
                const int kt = few_k_tile(step, rot, kbeg, nq, nk);
                for (int lane = 0; lane < 64; ++lane)
                    for (int h = 0; h < 2; ++h)
                        for (int j = 0; j < 16; ++j) {
                            // byte j of the lane's operand of half h: element of the weight, and of a token's codes
                            int64_t at, code;
                            if (cols) {
                                at = raw_col_base(n0, ldw, kt, h, j) + raw_col_lane_bytes(ldw, lane) / 2;
                                code = raw_col_codes_offset(0, lda, kt, h, lane) + j;
                                if (!r.access("raw weight W", at, 2, w_elems, block, wave, lane, kt)) continue;
                            } else {
                                const int i = 2 * h + (j >> 3);
                                at = raw_row_offset(n0, ldw, kt, i, lane) + (j & 7);
                                code = raw_row_codes_offset(0, lda, kt, i, lane) + (j & 7);
                                if (!r.access("raw weight W", at, 1, w_elems, block, wave, lane, kt)) continue;
                            }
                            for (int b = 0; b < blocks; ++b)
                                r.access("raw weight codes", code + (b * 16 + (lane & 15)) * lda, 1, a_elems, block, wave, lane, kt);
                            const int64_t row = at / ldw, col = at % ldw;
                            if (row >= R || col >= C || code != (cols ? row : col)) { r.fail("raw weight: element (%lld, %lld) meets code %lld", (long long)row, (long long)col, (long long)code); continue; }
                            for (int e = 0; e < (cols ? 2 : 1); ++e) ++read[(size_t)(row * C + col + e)];
                        }
            }
        }
        for (int wave = 0; wave < 2; ++wave)
            for (int lane = 0; lane < 64; ++lane) {
                const int token = wave * 16 + (lane & 15), count = cols ? 8 : 4;
                const int64_t col = n0 + (lane >> 4) * count;
                if (!r.access("raw weight C", token * ldc + col, count, c_elems, block, wave, lane) || col + count > n) continue;
                for (int e = 0; e < count; ++e) ++stored[(size_t)(token * n + col + e)];
            }
    }
    for (size_t i = 0; i < read.size() && !r.bad; ++i)
        if (read[i] != 1) r.fail("raw weight: W(%lld, %lld) is read %d times", (long long)(i / C), (long long)(i % C), (int)read[i]);
    for (size_t i = 0; i < stored.size() && !r.bad; ++i)
        if (stored[i] != 1) r.fail("raw weight: C(%lld, %lld) is stored %d times", (long long)(i / n), (long long)(i % n), (int)stored[i]);
    *n_checked = r.checked;
    return r.bad;
}

// dW of a step on few tokens (gemm_skinny.hip: thin_walk): every tile belongs to one worker, its rows and K tiles are read, every element stored once
int walk_thin(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int num_cu, int64_t a_elems, int64_t b_elems, int64_t c_elems,
              int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    const int tiles_n = (int)(N >> 7), tiles = (int)(M >> 7) * tiles_n, nk = (int)(K >> 7), workers = (int)thin_workers(M, N, num_cu);
    std::vector<uint8_t> seen((size_t)tiles, 0);
    for (int worker = 0; worker < workers && !r.bad; ++worker) {
        if (worker >= tiles) r.fail("thin: worker %d of %d has no tile, and fetches one all the same", worker, workers);
        for (int tile = worker; tile < tiles && !r.bad; tile += workers) {
            ++seen[(size_t)tile];
            const int m0 = (tile / tiles_n) * 128, n0 = (tile % tiles_n) * 128;
            std::vector<uint8_t> stored(128 * 16, 0), slab(32768 / 16, 0);
            for (int wave = 0; wave < 4; ++wave)
                for (int lane = 0; lane < 64; ++lane) {
                    for (int kt = 0; kt < nk; ++kt)
                        for (int i = 0; i < 4; ++i) {
                            const int64_t row = wave * 32 + 8 * i + (lane >> 3), at = kt * 128 + ((lane & 7) ^ (lane >> 3) ^ (i & 1)) * 16;
                            r.access("thin A", (m0 + row) * lda + at, 16, a_elems, tile, wave, lane, kt);
                            r.access("thin B", (n0 + row) * ldb + at, 16, b_elems, tile, wave, lane, kt);
                        }
                    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64, fr_row = lane & 31, fr_half = lane >> 5;
                    for (int i = 0; i < 2; ++i)
                        for (int j = 0; j < 2; ++j)
                            for (int q = 0; q < 4; ++q) {
                                const int row = wm + i * 32 + fr_row, col = wn + j * 32 + 8 * q + 4 * fr_half, at = row * 256 + ((col * 2) ^ ((row & 15) << 4));
                                if (r.access("thin LDS write", at, 8, 32768, tile, wave, lane)) slab[(size_t)at / 16] += 1;
                            }
                    for (int p = 0; p < 8; ++p) {
                        const int row = p * 16 + wave * 4 + (lane >> 4), chunk = lane & 15;
                        r.access("thin LDS read", row * 256 + ((chunk ^ (row & 15)) << 4), 16, 32768, tile, wave, lane, p);
                        r.access("thin C", (m0 + row) * ldc + n0 + chunk * 8, 8, c_elems, tile, wave, lane, p);
                        ++stored[(size_t)(row * 16 + chunk)];
                    }
                }
            for (size_t i = 0; i < stored.size() && !r.bad; ++i)
                if (stored[i] != 1 || slab[i] != 2) r.fail("thin: chunk %zu of tile %d is stored %d times, its halves written %d times", i, tile, (int)stored[i], (int)slab[i]);
        }
    }
    for (int t = 0; t < tiles && !r.bad; ++t)
        if (seen[(size_t)t] != 1) r.fail("thin: tile %d is taken %d times", t, (int)seen[(size_t)t]);
    *n_checked = r.checked;
    return r.bad;
}

// Attention's backward (attention.hip) on tensors of element strides sb, sh, ss: every load lies in its tensor or behind the rows of its pair
// (where it reads zeros), every tile of scores at or under the diagonal is computed once per kernel, those without a mask lie under it, every
// row of the results and every word of the workspace is stored once.  *past = rows behind the last that an offset reaches.
int walk_attention(int64_t batch, int64_t heads, int64_t seq, int D, int64_t sb, int64_t sh, int64_t ss, int waves_dq, int waves_dkdv, int64_t elems,
                   int64_t words, int64_t* past, int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    const int chunks = D / 8, slabs = 32 * 2 * D / 1024, rows_per_slab = 1024 / (2 * D), pairs = (int)(batch * heads);
    const int64_t padded = (seq + 31) / 32 * 32, bytes = attention_bytes((int)seq, ss, D);
    *past = 0;
    auto load = [&](const char* what, int pair, int64_t row, int at) {
        if (row - seq > *past) *past = row - seq;
        const int64_t offset = row * ss * 2 + at;
        ++r.checked;
        if (offset >= bytes) return;
        if (row >= seq || offset + 16 > bytes) r.fail("%s: row %lld, byte %d reaches into the buffer's end", what, (long long)row, at);
        r.access(what, (pair / heads) * sb + (pair % heads) * sh + offset / 2, 8, elems, pair, row, at);
    };
    for (int keys = 0; keys < 2; ++keys) {      // 0: a workgroup owns queries (dQ), 1: keys (dK and dV)
        const int waves = keys ? waves_dkdv : waves_dq, per_tile = slabs / waves, blocks = (int)((seq + waves * 32 - 1) / (waves * 32));
        const int all = (int)((seq + 31) / 32);
        std::vector<uint8_t> done((size_t)pairs * all * all, 0), row_stored((size_t)pairs * seq, 0), word_stored((size_t)(pairs * 2 * padded), 0);
        for (int w = 0; w < (int)round8(pairs) * blocks && !r.bad; ++w) {
            const AttentionPlace p = attention_place((uint32_t)w, blocks);
            if (p.pair >= pairs) continue;
            const int block = keys ? p.block : blocks - 1 - p.block, row0 = block * waves * 32;
            if (block < 0 || block >= blocks) { r.fail("attention: workgroup %d takes block %d", w, block); break; }
            const int first = keys ? row0 / 32 : 0;
            const int tiles = keys ? all : (int)(((row0 + waves * 32 < seq ? row0 + waves * 32 : seq) + 31) / 32);
            const int clear = keys ? imin(tiles, first + waves) : row0 / 32;
            for (int tile = first; tile < tiles + 2; ++tile) {      // two are fetched ahead
                std::vector<uint8_t> filled((size_t)32 * chunks, 0);
                for (int wave = 0; wave < waves; ++wave)
                    for (int lane = 0; lane < 64; ++lane) {
                        for (int i = 0; i < per_tile; ++i) {
                            const int row = wave * rows_per_slab + lane / chunks + i * 16;
                            load("attention tile", p.pair, (int64_t)tile * 32 + row, (lane % chunks) * 16);
                            const int lds = (wave + i * waves) * 1024 + lane * 16;
                            if (r.access("attention LDS tile", lds, 16, 64 * D, w, wave, lane)) ++filled[(size_t)lds / 16];
                            if (lds / (2 * D) != row) r.fail("attention: row %d of a tile lands in row %d", row, lds / (2 * D));
                        }
                        if (keys && tile < tiles) r.access("attention rows", p.pair * 2 * padded + (lane & 31) + (lane >> 5) * padded + tile * 32, 1, words, w, tile, lane);
                    }
                for (size_t i = 0; i < filled.size() && !r.bad; ++i)
                    if (filled[i] != 1) r.fail("attention: chunk %zu of a tile is loaded %d times", i, (int)filled[i]);
            }
            for (int wave = 0; wave < waves; ++wave) {
                const int own = row0 + wave * 32;
                for (int lane = 0; lane < 64; ++lane)
                    for (int ks = 0; ks < D / 16; ++ks) load("attention operand", p.pair, own + (lane & 31), (lane >> 5) * 16 + ks * 32);
                for (int tile = first; tile < tiles; ++tile) {
                    const bool masked = keys ? tile < clear : tile >= clear;
                    if (masked && (keys ? (tile + 1) * 32 <= own : tile * 32 >= own + 32)) continue;
                    const int query = keys ? tile * 32 : own, key = keys ? own : tile * 32;
                    if (query >= seq || key >= seq) continue;       // rows that are zeros
                    if (!masked && key + 31 > query) r.fail("attention: queries from %d and keys from %d without a mask", query, key);
                    ++done[((size_t)p.pair * all + query / 32) * all + key / 32];
                }
                for (int row = own; row < own + 32; ++row) {
                    if (row < seq) {
                        ++row_stored[(size_t)(p.pair * seq + row)];
                        r.access("attention result", (p.pair / heads) * sb + (p.pair % heads) * sh + row * ss, D, elems, w, row);
                    }
                    if (!keys && row < padded)
                        for (int half = 0; half < 2; ++half)
                            if (r.access("attention workspace", ((int64_t)p.pair * 2 + half) * padded + row, 1, words, w, row)) ++word_stored[(size_t)((p.pair * 2 + half) * padded + row)];
                }
            }
        }
        for (int pair = 0; pair < pairs && !r.bad; ++pair)
            for (int m = 0; m < all; ++m)
                for (int n = 0; n < all; ++n)
                    if (done[((size_t)pair * all + m) * all + n] != (n <= m)) r.fail("attention: tile (%d, %d) of pair %d is computed %d times", m, n, pair, (int)done[((size_t)pair * all + m) * all + n]);
        for (size_t i = 0; i < row_stored.size() && !r.bad; ++i)
            if (row_stored[i] != 1) r.fail("attention: row %zu is stored %d times", i, (int)row_stored[i]);
        for (size_t i = 0; !keys && i < word_stored.size() && !r.bad; ++i)
            if (word_stored[i] != 1) r.fail("attention: word %zu is stored %d times", i, (int)word_stored[i]);
    }
    *n_checked = r.checked;
    return r.bad;
}

int attention_takes_stride(int64_t stride, int64_t seq, int64_t head_dim) { return attention_stride_ok(stride, seq, head_dim); }

struct ScaleArg {
    int mode;
    int64_t bs, rs, ks, elems;
};

// ti8_gemm_i8_nt / ti8_gemm_i8_nt_i32 -> gemm_i8_kernel<BM, BN, WM, WN, EPI> (gemm.hip); the
// tile shape and epilogue kind are chosen as the entry point chooses them (raw_i32 = 1: the
// int32-output entry point, always 256 x 256 tiles).  epi: 0 raw int32, 1 rows, 2 promote,
// 3 literal, 4 per-lane B factors, 5 chained promote.
int walk_gemm(int64_t bsa, int64_t lda, int64_t bsb, int64_t ldb, int64_t bsc, int64_t ldc, const ScaleArg* sa_in,
              const ScaleArg* sb_in, int64_t batch, int64_t M, int64_t N, int64_t K, int acc_i32_full, int strict, int large,
              int raw_i32, int num_cu, int64_t a_elems, int64_t b_elems, int64_t c_elems, int* picked, int64_t* n_checked,
              char* msg, int msglen) {
    Report r{msg, msglen};
    ScaleArg sa = sa_in ? *sa_in : ScaleArg{0, 0, 0, 0, 0}, sb = sb_in ? *sb_in : ScaleArg{0, 0, 0, 0, 0};
    GemmConfig cfg = raw_i32 ? GemmConfig{256, 256, 2, 4, 0}
                             : gemm_config(M, N, K, batch, acc_i32_full != 0, strict != 0, sa.mode, sb.mode, large != 0, num_cu);
    picked[0] = cfg.bm; picked[1] = cfg.bn; picked[2] = cfg.epi;
    const int BM = cfg.bm, BN = cfg.bn, WM = cfg.wm, WN = cfg.wn, EPI = cfg.epi;
    const int NW = WM * WN, TM = BM / WM / 32, TN = BN / WN / 32, A_INSTR = BM / 8 / NW, B_INSTR = BN / 8 / NW;
    const int A_BYTES = BM * 128, B_BYTES = BN * 128;
    const bool CHAIN = EPI == 5 || EPI == 6, LANEB = EPI == 4 || EPI == 6, FAST = EPI == 2 || EPI == 4 || CHAIN;
    const int tiles_m = (int)((M + BM - 1) / BM), tiles_n = (int)((N + BN - 1) / BN);
    const int nk = (int)(K >> 7), klast = (nk - 1) * 128;
    const int WCOLS = TN * 32, LPR = WCOLS / 8, RPI = 64 / LPR, NRR = 32 / RPI;
    const int GROUP = gemm_group_rows(BM);
    (void)CHAIN;
    std::vector<uint8_t> stored(c_elems <= (int64_t)1 << 30 ? (size_t)c_elems : 0, 0);
    std::vector<uint8_t> tile_seen((size_t)tiles_m * tiles_n, 0);
    // K tiles whose loads are checked: offsets grow with kt up to the clamp, so the first two and
    // the clamped ones (nk - 1, nk, nk + 1: the loop fetches up to two tiles ahead) cover all
    const int kts[5] = {0, 1, nk - 1, nk, nk + 1};
    for (int64_t by = 0; by < batch && !r.bad; ++by) {
        std::fill(tile_seen.begin(), tile_seen.end(), 0);
        for (int bx = 0; bx < tiles_m * tiles_n && !r.bad; ++bx) {
            const TileCoord tc = gemm_tile_of(bx, tiles_m, tiles_n, GROUP, false);
            if (tc.tile_m < 0 || tc.tile_m >= tiles_m || tc.tile_n < 0 || tc.tile_n >= tiles_n) {
                r.fail("gemm: workgroup %d maps to tile (%d, %d) outside %d x %d", bx, tc.tile_m, tc.tile_n, tiles_m, tiles_n);
                break;
            }
            ++tile_seen[(size_t)tc.tile_m * tiles_n + tc.tile_n];
            const int m0 = tc.tile_m * BM, n0 = tc.tile_n * BN;
            for (int wave = 0; wave < NW; ++wave) {
                const int wm = wave / WN, wn = wave % WN;
                const int rA0 = gemm_wave_first_row(m0, wave, A_INSTR, (int)M), rB0 = gemm_wave_first_row(n0, wave, B_INSTR, (int)N);
                const int tA0 = wave * A_INSTR, tB0 = wave * B_INSTR;
                for (int lane = 0; lane < 64; ++lane) {
                    // ---- global -> LDS loads (gemm.hip: voffA/voffB, baseA/baseB, issue_tile_loads)
                    for (int q = 0; q < 5; ++q) {
                        const int koff = gemm_k_offset(kts[q], klast);
                        for (int i = 0; i < A_INSTR; ++i) {
                            const uint32_t vo = gemm_lane_offset_bytes(lane, (tA0 + i) & 1, (int)lda);
                            r.access("gemm A", by * bsa + gemm_load_offset_bytes(rA0, lda, koff, i, vo), 16, a_elems, bx, wave, lane, kts[q]);
                            const int64_t lds = (int64_t)wave * A_INSTR * 1024 + i * 1024 + lane * 16;
                            r.access("gemm LDS A", lds, 16, A_BYTES, bx, wave, lane, i);
                        }
                        for (int i = 0; i < B_INSTR; ++i) {
                            const uint32_t vo = gemm_lane_offset_bytes(lane, (tB0 + i) & 1, (int)ldb);
                            r.access("gemm B", by * bsb + gemm_load_offset_bytes(rB0, ldb, koff, i, vo), 16, b_elems, bx, wave, lane, kts[q]);
                            const int64_t lds = (int64_t)wave * B_INSTR * 1024 + i * 1024 + lane * 16;
                            r.access("gemm LDS B", lds, 16, B_BYTES, bx, wave, lane, i);
                        }
                    }
                    const int fr_row = lane & 31, fr_half = lane >> 5;
                    // ---- per-K-tile factors of the fast promotion (gemm.hip: fraw_a / fraw_b, pfb)
                    if (FAST) {
                        const bool a_in = sa.mode != 0, b_in = sb.mode != 0;
                        const int sha = sa.mode == 3 ? 1 : 0, shb = sb.mode == 3 ? 1 : 0;
                        const int rowblk = gemm_factor_block(m0 + wm * TM * 32, (int)M), colblk = gemm_factor_block(n0 + wn * TN * 32, (int)N);
                        const int64_t ska = a_in ? sa.ks : 0, skb = (b_in && !LANEB) ? sb.ks : 0;
                        for (int c = 0; c < 4; ++c) {
                            const int kt = gemm_factor_kt(c, lane, nk);
                            r.access("gemm factor A", gemm_factor_index(by, sa.bs, rowblk, sa.rs, kt, sha, ska), 1, sa.elems, bx, wave, lane, c);
                            r.access("gemm factor B", gemm_factor_index(by, sb.bs, colblk, sb.rs, kt, shb, skb), 1, sb.elems, bx, wave, lane, c);
                        }
                        if (LANEB)
                            for (int j = 0; j < TN; ++j) {
                                const int64_t base = epi_col_scale_index(by, sb.bs, n0 + (wn * TN + j) * 32 + fr_row, (int)N, sb.rs);
                                for (int kt = 0; kt < nk; ++kt) r.access("gemm lane factor B", base + (int64_t)kt * sb.ks, 1, sb.elems, bx, wave, lane, kt);
                            }
                    }
                    // ---- literal promotion: one scale per element and K tile (gemm.hip: EPI_STRICT block)
                    if (EPI == 3) {
                        const int kk[2] = {0, nk - 1};
                        for (int q = 0; q < 2; ++q)
                            for (int i = 0; i < TM; ++i)
                                for (int j = 0; j < TN; ++j) {
                                    const int col = imin(n0 + (wn * TN + j) * 32 + fr_row, (int)N - 1);
                                    r.access("gemm strict B scale", scale_index(sb.mode, sb.bs, sb.rs, sb.ks, by, col, kk[q]), 1, sb.elems, bx, wave, lane, kk[q]);
                                    for (int e = 0; e < 16; ++e) {
                                        const int mrow = imin(m0 + (wm * TM + i) * 32 + 8 * (e >> 2) + 4 * fr_half + (e & 3), (int)M - 1);
                                        r.access("gemm strict A scale", scale_index(sa.mode, sa.bs, sa.rs, sa.ks, by, mrow, kk[q]), 1, sa.elems, bx, wave, lane, kk[q]);
                                    }
                                }
                    }
                    // ---- epilogue (gemm.hip: coln, cm, prow0 / rm_all, store_tile)
                    const bool col_part = EPI == 1 || (FAST && sb.mode == 0), row_part = EPI == 1 || (FAST && sa.mode == 0);
                    if (EPI == 1 || FAST) {   // column scales, fetched before the main loop by every wave
                        const int64_t cs = col_part ? sb.rs : 0;
                        const int ncol0 = n0 + wn * WCOLS + epi_scale_col_of_lane(lane);
                        for (int c = 0; c < 4; ++c) r.access("gemm column scale", epi_col_scale_index(by, sb.bs, ncol0 + c, (int)N, cs), 1, sb.elems, bx, wave, lane, c);
                    }
                    // a wave whose tile lies outside the output stops here
                    if (m0 + wm * TM * 32 >= M || n0 + wn * WCOLS >= N) continue;
                    const int rb_col = epi_col_of_lane(lane, WCOLS), rb_row = epi_row_of_lane(lane, WCOLS);
                    for (int c = 0; c < 8; ++c) {   // the lane that holds this lane's column scale c, and the column it fetched
                        const int src = epi_scale_lane(lane, c);
                        if (src < 0 || src >= 64 || epi_scale_col_of_lane(src) + (c & 3) != rb_col + c)
                            r.fail("gemm: lane %d takes column scale %d from lane %d, which holds column %d, not %d", lane, c, src,
                                   epi_scale_col_of_lane(src) + (c & 3), rb_col + c);
                    }
                    const int row0 = m0 + wm * TM * 32 + rb_row;
                    if (row_part) {
                        const int64_t base = epi_row_scale_base(by, sa.bs, row0, sa.rs);
                        for (int i = 0; i < TM; ++i)
                            for (int k = 0; k < NRR; ++k)
                                r.access("gemm row scale", base + (int64_t)(i * 32 + k * RPI) * sa.rs, 1, sa.elems, bx, wave, lane, i * NRR + k);
                    }
                    // slab: 32 rows of EPI_SLAB_LD words per wave, inside the operand buffers
                    for (int e = 0; e < 16; ++e)
                        for (int j = 0; j < TN; ++j) {
                            const int rr = 8 * (e >> 2) + 4 * fr_half + (e & 3);
                            r.access("gemm slab write", (int64_t)wave * 32 * EPI_SLAB_LD(WCOLS) + rr * EPI_SLAB_LD(WCOLS) + j * 32 + fr_row, 1,
                                     (2 * (A_BYTES + B_BYTES)) / 4, bx, wave, lane, e);
                        }
                    for (int k = 0; k < NRR; ++k)
                        r.access("gemm slab read", (int64_t)wave * 32 * EPI_SLAB_LD(WCOLS) + (rb_row + k * RPI) * EPI_SLAB_LD(WCOLS) + rb_col, 8,
                                 (2 * (A_BYTES + B_BYTES)) / 4, bx, wave, lane, k);
                    int64_t off = epi_out_offset(by, bsc, row0, ldc, n0 + wn * WCOLS + rb_col);
                    const int64_t c_step = (int64_t)RPI * ldc;
                    for (int i = 0; i < TM; ++i)
                        for (int k = 0; k < NRR; ++k, off += c_step) {
                            if (r.access("gemm C", off, 8, c_elems, bx, wave, lane, i * NRR + k) && !stored.empty())
                                for (int c = 0; c < 8; ++c) ++stored[(size_t)(off + c)];
                        }
                }
            }
        }
        for (size_t t = 0; t < tile_seen.size() && !r.bad; ++t)
            if (tile_seen[t] != 1) r.fail("gemm: tile %zu of batch %lld is computed %d times", t, (long long)by, (int)tile_seen[t]);
    }
    // every element of C [batch][M][N] stored exactly once, nothing else touched
    if (!stored.empty() && !r.bad) {
        int64_t expect = 0;
        for (int64_t b = 0; b < batch && !r.bad; ++b)
            for (int64_t m = 0; m < M && !r.bad; ++m)
                for (int64_t n = 0; n < N; ++n) {
                    const int64_t o = b * bsc + m * ldc + n;
                    if (stored[(size_t)o] != 1) {
                        r.fail("gemm: C[%lld][%lld][%lld] stored %d times", (long long)b, (long long)m, (long long)n, (int)stored[(size_t)o]);
                        break;
                    }
                    ++expect;
                }
        int64_t total = 0;
        for (size_t i = 0; i < stored.size(); ++i) total += stored[i];
        if (!r.bad && total != expect) r.fail("gemm: %lld stores, %lld elements of C", (long long)total, (long long)expect);
    }
    *n_checked = r.checked;
    return r.bad;
}

// Persistent chained kernel (gemm_chain.hip: gemm_i8_chain_kernel) on one GEMM with `batch` batches and `grid`
// workgroups: workgroup w walks tiles w, w + grid, ...; a tile's K tiles are fetched by its own iterations except
// K tiles 0 and 1, which the previous tile's last iterations (or, for a workgroup's first tile, its start) fetch, and
// the workgroup's last tile fetches its own K tiles 0 and 1 once more.  Checked: every tile of every batch is taken
// exactly once, every global -> LDS load, scale load, slab access and store lies inside its buffer, every element
// of C is stored exactly once.
int walk_gemm_chain(int64_t bsa, int64_t lda, int64_t bsb, int64_t ldb, int64_t bsc, int64_t ldc, const ScaleArg* sa_in,
                    const ScaleArg* sb_in, int64_t batch, int64_t M, int64_t N, int64_t K, int grid, int64_t a_elems,
                    int64_t b_elems, int64_t c_elems, int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    const ScaleArg sa = *sa_in, sb = *sb_in;
    const int BM = 256, BN = 256, WN = 4, NW = 8, TM = 4, TN = 2, A_INSTR = 4, B_INSTR = 4, WCOLS = 64, RPI = 8;
    const int tiles_m = (int)((M + BM - 1) / BM), tiles_n = (int)((N + BN - 1) / BN), per_batch = tiles_m * tiles_n;
    const int total = per_batch * (int)batch, nk = (int)(K >> 7), GROUP = gemm_group_rows(BM);
    const int64_t lds_words = (2 * (BM + BN) * 128 + NW * 16 * WCOLS * 4) / 4, slab0 = 2 * (BM + BN) * 128 / 4;
    if (!chain_takes(nk, true)) { r.fail("gemm chain: not over K / 128 = %d", nk); *n_checked = 0; return 1; }
    const int walked = chain_walked(nk);
    if (walked < nk || walked & 1 || walked > 256) r.fail("gemm chain: %d K tiles are walked as %d", nk, walked);
    std::vector<uint8_t> stored(c_elems <= (int64_t)1 << 30 ? (size_t)c_elems : 0, 0);
    std::vector<uint8_t> seen((size_t)total, 0);
    const bool a_in = sa.mode != 0, b_in = sb.mode != 0;
    for (int w = 0; w < grid && !r.bad; ++w)
        for (int T = w; T < total && !r.bad; T += grid) {
            ++seen[(size_t)T];
            const int64_t by = T / per_batch;
            const TileCoord tc = gemm_tile_of(T - (int)by * per_batch, tiles_m, tiles_n, GROUP, true);
            if (tc.tile_m < 0 || tc.tile_m >= tiles_m || tc.tile_n < 0 || tc.tile_n >= tiles_n) {
                r.fail("gemm chain: tile %d maps to (%d, %d) outside %d x %d", T, tc.tile_m, tc.tile_n, tiles_m, tiles_n);
                break;
            }
            const int m0 = tc.tile_m * BM, n0 = tc.tile_n * BN;
            for (int wave = 0; wave < NW; ++wave) {
                const int wm = wave / WN, wn = wave % WN;
                const int rA0 = gemm_wave_first_row(m0, wave, A_INSTR, (int)M), rB0 = gemm_wave_first_row(n0, wave, B_INSTR, (int)N);
                const int tA0 = wave * A_INSTR, tB0 = wave * B_INSTR;
                const int kts[4] = {0, 1, walked - 2, walked - 1};
                for (int lane = 0; lane < 64; ++lane) {
                    for (int q = 0; q < 4; ++q) {
                        const int koff = gemm_k_offset(kts[q], (nk - 1) * 128);
                        for (int i = 0; i < A_INSTR; ++i) {
                            const uint32_t vo = gemm_lane_offset_bytes(lane, (tA0 + i) & 1, (int)lda);
                            r.access("gemm chain A", by * bsa + gemm_load_offset_bytes(rA0, lda, koff, i, vo), 16, a_elems, T, wave, lane, kts[q]);
                        }
                        for (int i = 0; i < B_INSTR; ++i) {
                            const uint32_t vo = gemm_lane_offset_bytes(lane, (tB0 + i) & 1, (int)ldb);
                            r.access("gemm chain B", by * bsb + gemm_load_offset_bytes(rB0, ldb, koff, i, vo), 16, b_elems, T, wave, lane, kts[q]);
                        }
                    }
                    // per-K-tile factors: scalar base + (K tile >> shift) * stride per lane
                    const int64_t fa = gemm_factor_index(by, sa.bs, gemm_factor_block(m0 + wm * TM * 32, (int)M), sa.rs, 0, 0, 0);
                    const int64_t fb = gemm_factor_index(by, sb.bs, gemm_factor_block(n0 + wn * TN * 32, (int)N), sb.rs, 0, 0, 0);
                    for (int c = 0; c <= (walked - 1) >> 6; ++c) {   // the factor register is refilled every 64 K tiles
                        const uint32_t kt = (uint32_t)gemm_factor_kt(c, lane, nk);
                        r.access("gemm chain factor A", fa + (int64_t)((kt >> (sa.mode == 3 ? 1 : 0)) * (uint32_t)(a_in ? sa.ks : 0)), 1, sa.elems, T, wave, lane, c);
                        r.access("gemm chain factor B", fb + (int64_t)((kt >> (sb.mode == 3 ? 1 : 0)) * (uint32_t)(b_in ? sb.ks : 0)), 1, sb.elems, T, wave, lane, c);
                    }
                    // column scales: 4 per lane from the wave tile's first column (clamped for a tile outside N)
                    const uint32_t cs = b_in ? 0u : (uint32_t)sb.rs;
                    const int64_t colp = epi_col_scale_index(by, sb.bs, chain_col_scale_first(n0 + wn * WCOLS, (int)N), (int)N, cs);
                    for (int c = 0; c < 4; ++c)
                        r.access("gemm chain column scale", colp + (int64_t)(((uint32_t)epi_scale_col_of_lane(lane) + c) * cs), 1, sb.elems, T, wave, lane, c);
                    if (m0 + wm * TM * 32 >= M || n0 + wn * WCOLS >= N) continue;   // this wave stores nothing
                    const int rb_col = epi_col_of_lane(lane, WCOLS), rb_row = epi_row_of_lane(lane, WCOLS);
                    for (int c = 0; c < 8; ++c) {
                        const int src = epi_scale_lane(lane, c);
                        if (src < 0 || src >= 64 || epi_scale_col_of_lane(src) + (c & 3) != rb_col + c)
                            r.fail("gemm chain: lane %d takes column scale %d from lane %d", lane, c, src);
                    }
                    const int row0 = m0 + wm * TM * 32 + rb_row;
                    if (!a_in) {
                        const int64_t base = epi_row_scale_base(by, sa.bs, row0, sa.rs);
                        for (int q = 0; q < TM * 4; ++q) r.access("gemm chain row scale", base + (int64_t)(q * RPI) * sa.rs, 1, sa.elems, T, wave, lane, q);
                    }
                    const int fr_row = lane & 31, fr_half = lane >> 5;
                    for (int e = 0; e < 8; ++e)
                        for (int j = 0; j < TN; ++j)
                            r.access("gemm chain slab write", slab0 + wave * 16 * WCOLS + epi_chain_slab_word(epi_chain_slab_row(e, fr_half), j * 32 + fr_row), 1,
                                     lds_words, T, wave, lane, e);
                    for (int k = 0; k < 2; ++k)
                        for (int half = 0; half < 2; ++half)
                            r.access("gemm chain slab read", slab0 + wave * 16 * WCOLS + epi_chain_slab_word(rb_row + k * RPI, rb_col + 4 * half), 4, lds_words,
                                     T, wave, lane, k);
                    int64_t off = epi_out_offset(by, bsc, row0, ldc, n0 + wn * WCOLS + rb_col);
                    for (int q = 0; q < TM * 4; ++q, off += (int64_t)RPI * ldc)
                        if (r.access("gemm chain C", off, 8, c_elems, T, wave, lane, q) && !stored.empty())
                            for (int c = 0; c < 8; ++c) ++stored[(size_t)(off + c)];
                }
            }
        }
    for (int T = 0; T < total && !r.bad; ++T)
        if (seen[(size_t)T] != 1) r.fail("gemm chain: tile %d is computed %d times", T, (int)seen[(size_t)T]);
    if (!stored.empty() && !r.bad) {
        for (int64_t b = 0; b < batch && !r.bad; ++b)
            for (int64_t mm = 0; mm < M && !r.bad; ++mm)
                for (int64_t n = 0; n < N; ++n)
                    if (stored[(size_t)(b * bsc + mm * ldc + n)] != 1) {
                        r.fail("gemm chain: C[%lld][%lld][%lld] stored %d times", (long long)b, (long long)mm, (long long)n, (int)stored[(size_t)(b * bsc + mm * ldc + n)]);
                        break;
                    }
    }
    *n_checked = r.checked;
    return r.bad;
}

// Tiles of the persistent chained kernel's workgroups, round by round: each of `total` exactly once
int walk_chain_rounds(int total, int grid, int several, int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    std::vector<int> seen((size_t)total, 0);
    for (int w = 0; w < grid; ++w) {
        ++seen[(size_t)w];
        for (int base = grid;; base += grid) {
            const int t = chain_tile_of_round(base, grid, total, w, several != 0);
            if (t >= total) break;
            if (t < base || t >= base + grid) r.fail("chain rounds: workgroup %d takes tile %d in the round from %d", w, t, base);
            ++seen[(size_t)t];
        }
    }
    for (int t = 0; t < total && !r.bad; ++t) {
        if (seen[(size_t)t] != 1) r.fail("chain rounds: tile %d is taken %d times", t, seen[(size_t)t]);
        ++r.checked;
    }
    *n_checked = r.checked;
    return r.bad;
}

// Medium-size kernel (gemm_mid.hip: gemm_i8_mid_kernel) on one GEMM: 128 x 128 tiles, M a multiple of 32.  Checked: every tile of every
// batch is computed once; the loads of every K tile, those past the end included, the per-K-tile factors, the scales of the
// epilogue, the LDS slots of loads, fragments, factors and slabs; every element of C stored once.
int walk_gemm_mid(int64_t bsa, int64_t lda, int64_t bsb, int64_t ldb, int64_t bsc, int64_t ldc, const ScaleArg* sa, const ScaleArg* sb,
                  int64_t batch, int64_t M, int64_t N, int64_t K, int i32, int64_t a_elems, int64_t b_elems, int64_t c_elems,
                  int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    const int STAGES = 4, OPERAND = 128 * 128, STAGE = 2 * OPERAND, FACTORS = 256, WCOLS = 64, SLAB = 32 * EPI_SLAB_LD(WCOLS);
    const int tiles_m = (int)((M + 127) / 128), tiles_n = (int)(N / 128), nk = (int)(K >> 7), klast = (nk - 1) * 128;
    if (nk < 1 || nk > FACTORS) r.fail("gemm mid: %d K tiles", nk);
    std::vector<uint8_t> stored((size_t)c_elems, 0), tile_seen((size_t)tiles_m * tiles_n, 0);
    for (int64_t by = 0; by < batch && !r.bad; ++by) {
        std::fill(tile_seen.begin(), tile_seen.end(), 0);
        for (int bx = 0; bx < tiles_m * tiles_n && !r.bad; ++bx) {
            const TileCoord tc = gemm_tile_of(bx, tiles_m, tiles_n, gemm_group_rows(128), false);
            if (tc.tile_m < 0 || tc.tile_m >= tiles_m || tc.tile_n < 0 || tc.tile_n >= tiles_n) {
                r.fail("gemm mid: workgroup %d maps to tile (%d, %d) outside %d x %d", bx, tc.tile_m, tc.tile_n, tiles_m, tiles_n);
                break;
            }
            ++tile_seen[(size_t)tc.tile_m * tiles_n + tc.tile_n];
            const int m0 = tc.tile_m * 128, n0 = tc.tile_n * 128;
            for (int thread = 0; thread < FACTORS && !i32; ++thread) {
                const int kt = imin(thread, nk - 1);
                if (sa->mode != 0) r.access("gemm mid factor A", gemm_factor_index(by, sa->bs, gemm_factor_block(m0, (int)M), sa->rs, kt, sa->mode == 3 ? 1 : 0, sa->ks), 1, sa->elems, bx, thread);
                if (sb->mode != 0) r.access("gemm mid factor B", gemm_factor_index(by, sb->bs, gemm_factor_block(n0, (int)N), sb->rs, kt, sb->mode == 3 ? 1 : 0, sb->ks), 1, sb->elems, bx, thread);
            }
            for (int wave = 0; wave < 8; ++wave) {
                const int grp = wave >> 2, wm = (wave & 3) / 2, wn = wave & 1;
                const int rA0 = gemm_mid_first_row(m0, wave, (int)M), rB0 = gemm_mid_first_row(n0, wave, (int)N);
                for (int lane = 0; lane < 64 && !r.bad; ++lane) {
                    for (int t = 0; t < nk + 4; t = t == 4 && nk > 8 ? nk - 1 : t + 1) {     // offsets grow with t up to the clamp
                        const int koff = gemm_k_offset(t, klast);
                        for (int i = 0; i < 2; ++i) {
                            r.access("gemm mid A", by * bsa + gemm_load_offset_bytes(rA0, lda, koff, i, gemm_lane_offset_bytes(lane, i & 1, (int)lda)), 16, a_elems, bx, wave, lane, t);
                            r.access("gemm mid B", by * bsb + gemm_load_offset_bytes(rB0, ldb, koff, i, gemm_lane_offset_bytes(lane, i & 1, (int)ldb)), 16, b_elems, bx, wave, lane, t);
                            r.access("gemm mid LDS", (t % STAGES) * STAGE + OPERAND + wave * 2048 + i * 1024 + lane * 16, 16, STAGES * STAGE, bx, wave, lane, t);
                        }
                    }
                    const int fr_row = lane & 31, fr_half = lane >> 5, sw = (lane & 7) ^ ((lane >> 3) & 1);
                    for (int ks = 0; ks < 4; ++ks) {
                        const int choff = ((ks * 2 + fr_half) ^ sw) * 16;
                        r.access("gemm mid fragment A", ((wm * 2 + grp) * 32 + fr_row) * 128 + choff, 16, OPERAND, bx, wave, lane, ks);
                        for (int j = 0; j < 2; ++j) r.access("gemm mid fragment B", (wn * 64 + j * 32 + fr_row) * 128 + choff, 16, OPERAND, bx, wave, lane, ks);
                    }
                    const int row0 = m0 + (wm * 2 + grp) * 32, rb_col = epi_col_of_lane(lane, WCOLS), rb_row = epi_row_of_lane(lane, WCOLS);
                    const bool row_part = i32 || sa->mode == 0, col_part = i32 || sb->mode == 0;
                    for (int k = 0; k < 4; ++k)
                        r.access("gemm mid row scale", epi_row_scale_base(by, sa->bs, imin(row0 + rb_row + 8 * k, (int)M - 1), row_part ? sa->rs : 0), 1, sa->elems, bx, wave, lane, k);
                    for (int c = 0; c < 8; ++c)
                        r.access("gemm mid column scale", epi_col_scale_index(by, sb->bs, n0 + wn * WCOLS + rb_col + c, (int)N, col_part ? sb->rs : 0), 1, sb->elems, bx, wave, lane, c);
                    for (int e = 0; e < 16; ++e)
                        for (int j = 0; j < 2; ++j)
                            r.access("gemm mid slab write", (8 * (e >> 2) + 4 * fr_half + (e & 3)) * EPI_SLAB_LD(WCOLS) + j * 32 + fr_row, 1, SLAB, bx, wave, lane, e);
                    r.access("gemm mid slabs", (int64_t)(wave + 1) * SLAB * 4 - 1, 1, STAGES * STAGE, bx, wave);
                    if (row0 >= M) continue;
                    for (int k = 0; k < 4; ++k) {
                        r.access("gemm mid slab read", (rb_row + 8 * k) * EPI_SLAB_LD(WCOLS) + rb_col, 8, SLAB, bx, wave, lane, k);
                        const int64_t off = epi_out_offset(by, bsc, row0 + rb_row, ldc, n0 + wn * WCOLS + rb_col) + (int64_t)(8 * k) * ldc;
                        if (r.access("gemm mid C", off, 8, c_elems, bx, wave, lane, k))
                            for (int c = 0; c < 8; ++c) ++stored[(size_t)(off + c)];
                    }
                }
            }
        }
        for (size_t t = 0; t < tile_seen.size() && !r.bad; ++t)
            if (tile_seen[t] != 1) r.fail("gemm mid: tile %zu of batch %lld is computed %d times", t, (long long)by, (int)tile_seen[t]);
    }
    int64_t total = 0;
    for (int64_t b = 0; b < batch && !r.bad; ++b)
        for (int64_t m = 0; m < M; ++m)
            for (int64_t n = 0; n < N; ++n) {
                const int times = stored[(size_t)(b * bsc + m * ldc + n)];
                if (times != 1) r.fail("gemm mid: C[%lld][%lld][%lld] stored %d times", (long long)b, (long long)m, (long long)n, times);
                total += times;
            }
    for (size_t i = 0; i < stored.size(); ++i) total -= stored[i];
    if (!r.bad && total != 0) r.fail("gemm mid: %lld stores outside C", (long long)-total);
    *n_checked = r.checked;
    return r.bad;
}

// Choice of kernels for a launch of several GEMMs of shapes shape[i] = {M, N, K}: cfg[3 i ..] = bm, bn, mid of GEMM i alone, then of the
// launch (9 values each)
void walk_configs_together(const int64_t* shape, int count, int i32, int num_cu, int* cfg) {
    GemmConfig c[3];
    int64_t s[3][3];
    for (int i = 0; i < count; ++i) {
        for (int d = 0; d < 3; ++d) s[i][d] = shape[3 * i + d];
        c[i] = gemm_config(s[i][0], s[i][1], s[i][2], 1, i32 != 0, false, i32 ? 0 : 1, i32 ? 0 : 1, false, num_cu);
        cfg[3 * i] = c[i].bm; cfg[3 * i + 1] = c[i].bn; cfg[3 * i + 2] = c[i].mid;
    }
    gemm_configs_together(s, count, false, num_cu, c);
    for (int i = 0; i < count; ++i) { cfg[9 + 3 * i] = c[i].bm; cfg[9 + 3 * i + 1] = c[i].bn; cfg[9 + 3 * i + 2] = c[i].mid; }
}

// Workgroup -> (GEMM, tile) map of a several-GEMM launch (gemm.hip: gemm_i8_multi_kernel, launch_multi):
// tiles[i] = workgroups of GEMM i.  Every workgroup of the grid must land in a GEMM i < count with
// a tile index in [0, tiles[i]), and every (GEMM, tile) must be taken exactly once.
// Column sums in one launch (bias.hip): every strip of columns belongs to one workgroup
int walk_column_strips(int strips, int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    std::vector<int> seen((size_t)strips, 0);
    for (int w = 0; w < strips && !r.bad; ++w, ++r.checked) {
        const int s = column_strip(w, strips);
        if (s < 0 || s >= strips || seen[(size_t)s]++) r.fail("column strips: workgroup %d takes strip %d of %d", w, s, strips);
    }
    *n_checked = r.checked;
    return r.bad;
}

// Lists of the persistent chained kernel: every tile of every GEMM is on one workgroup's list of one XCD, each list in the order of the
// launch, no workgroup busier than another by more than a tile that it could have left to it
int walk_chain_list(const int* tiles, const int* cost, int count, int slots, int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    int n[3], base[4] = {0, 0, 0, 0}, first[CHAIN_LIST_SLOTS + 1];
    uint16_t order[CHAIN_LIST_MAX];
    std::vector<std::vector<int>> seen(count);
    for (int i = 0; i < count; ++i) {
        n[i] = (tiles[i] + 7) / 8;
        base[i + 1] = base[i] + 8 * n[i];
        seen[i].assign(tiles[i], 0);
    }
    if (base[count] / 8 > CHAIN_LIST_MAX) { r.fail("chain list: %d entries", base[count] / 8); *n_checked = 0; return 1; }
    for (int i = count; i < 4; ++i) base[i] = base[count];
    const int busiest = chain_list(n, cost, count, slots, first, order);
    if (first[0] != 0 || first[slots] != base[count] / 8) r.fail("chain list: lists from %d to %d", first[0], first[slots]);
    int most = 0, least_but_last = 0x7fffffff;
    for (int s = 0; s < slots && !r.bad; ++s) {
        int load = 0, last = 0;
        for (int at = first[s]; at < first[s + 1] && !r.bad; ++at) {
            if (at > first[s] && order[at] <= order[at - 1]) r.fail("chain list: workgroup %d takes %d behind %d", s, order[at], order[at - 1]);
            for (int xcd = 0; xcd < 8; ++xcd) {
                const int T = order[at] * 8 + xcd, gi = gemm_multi_pick(T, base[1], base[2], count), local = T - base[gi];
                if (local < 0 || local >= 8 * n[gi]) r.fail("chain list: entry %d is none of GEMM %d", order[at], gi);
                else if (local < tiles[gi]) ++seen[gi][(size_t)local], ++r.checked;
                last = cost[gi];
            }
            load += last;
        }
        most = imax(most, load);
        least_but_last = imin(least_but_last, load);
    }
    for (int s = 0; s < slots && !r.bad; ++s) {      // its last tile began when nobody else was free
        int load = 0, last = 0;
        for (int at = first[s]; at < first[s + 1]; ++at) load += last = cost[gemm_multi_pick(order[at] * 8, base[1], base[2], count)];
        if (load - last > least_but_last) r.fail("chain list: workgroup %d of load %d took a tile of %d, another has %d in all", s, load, last, least_but_last);
    }
    if (!r.bad && most != busiest) r.fail("chain list: the busiest has %d, not %d", most, busiest);
    for (int i = 0; i < count && !r.bad; ++i)
        for (int t = 0; t < tiles[i]; ++t)
            if (seen[i][(size_t)t] != 1) { r.fail("chain list: tile %d of GEMM %d is taken %d times", t, i, seen[i][(size_t)t]); break; }
    *n_checked = r.checked;
    return r.bad;
}

// Which GEMMs of a call, over nk[i] K tiles and of tiles[i] 256 x 256 tiles (0: on another kernel), the persistent kernel takes: bit i
int walk_chains_of_call(const int* nk, const int64_t* tiles, int count, int num_cu) {
    bool among[3], alone[3], chains[3];
    int bits = 0;
    for (int i = 0; i < count; ++i) {
        among[i] = chain_takes(nk[i], true);
        alone[i] = chain_takes(nk[i], false);
    }
    chains_of_call(among, alone, tiles, count, num_cu, chains);
    for (int i = 0; i < count; ++i) bits |= chains[i] << i;
    return bits;
}

// Tile map of the LDS-tiled GEMMs: every tile once, and the workgroups of an XCD (every eighth) on tiles that follow each other
int walk_gemm_tile_map(int tiles_m, int tiles_n, int group, int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    const int total = tiles_m * tiles_n;
    std::vector<int> order((size_t)total), seen((size_t)total, 0);       // place of a tile in groups of rows, column by column
    for (int at = 0, m = 0; m < tiles_m; m += group)
        for (int n = 0; n < tiles_n; ++n)
            for (int i = m; i < imin(m + group, tiles_m); ++i) order[(size_t)(i * tiles_n + n)] = at++;
    for (int xcd = 0; xcd < 8; ++xcd)
        for (int w = xcd, last = -1; w < total && !r.bad; w += 8) {
            const TileCoord t = gemm_tile_of(w, tiles_m, tiles_n, group, true);
            if (t.tile_m < 0 || t.tile_m >= tiles_m || t.tile_n < 0 || t.tile_n >= tiles_n) { r.fail("tile map: workgroup %d has (%d, %d)", w, t.tile_m, t.tile_n); break; }
            const int at = order[(size_t)(t.tile_m * tiles_n + t.tile_n)];
            ++seen[(size_t)at];
            if (last >= 0 && at != last + 1) r.fail("tile map: workgroup %d is at %d behind %d", w, at, last);
            last = at;
            ++r.checked;
        }
    for (int w = 0; w < total && !r.bad; ++w) {      // a GEMM alone: every tile once
        const TileCoord t = gemm_tile_of(w, tiles_m, tiles_n, group, false);
        if (t.tile_m < 0 || t.tile_m >= tiles_m || t.tile_n < 0 || t.tile_n >= tiles_n) { r.fail("tile map: workgroup %d alone has (%d, %d)", w, t.tile_m, t.tile_n); break; }
        ++seen[(size_t)order[(size_t)(t.tile_m * tiles_n + t.tile_n)]];
    }
    for (int t = 0; t < total && !r.bad; ++t)
        if (seen[(size_t)t] != 2) r.fail("tile map: tile %d is taken %d times in both", t, seen[(size_t)t]);
    *n_checked = r.checked;
    return r.bad;
}

int walk_gemm_multi_map(const int* tiles, int count, int64_t* n_checked, char* msg, int msglen) {
    Report r{msg, msglen};
    int first[4] = {0, 0, 0, 0};
    int total = 0;
    for (int i = 0; i < count; ++i) {
        first[i] = total;
        total += tiles[i];
    }
    for (int i = count; i < 4; ++i) first[i] = total;
    std::vector<std::vector<int>> seen(count);
    for (int i = 0; i < count; ++i) seen[i].assign(tiles[i], 0);
    for (int w = 0; w < total && !r.bad; ++w) {
        const int i = gemm_multi_pick(w, first[1], first[2], count);
        const int t = w - first[i];
        if (i < 0 || i >= count || t < 0 || t >= tiles[i]) {
            r.fail("gemm multi: workgroup %d maps to GEMM %d tile %d (of %d GEMMs, %d tiles)", w, i, t, count, i >= 0 && i < count ? tiles[i] : -1);
            break;
        }
        ++seen[i][t];
        ++r.checked;
    }
    for (int i = 0; i < count && !r.bad; ++i)
        for (int t = 0; t < tiles[i]; ++t)
            if (seen[i][t] != 1) {
                r.fail("gemm multi: tile %d of GEMM %d is computed %d times", t, i, seen[i][t]);
                break;
            }
    *n_checked = r.checked;
    return r.bad ? 1 : 0;
}

}  // extern "C"
