// The INT8 linear layer -- Y = X W^T, dX = dY W, dW = dY^T X -- enqueued by ONE call: the quantiser launches and the GEMM
// launch(es) of a forward, a backward or a whole step that the Python layer would otherwise issue one entry point at a time, on
// caller-provided outputs and a caller-provided workspace.  Nothing here computes: the entry points of quant.hip, fwht.hip and
// gemm.hip are called in the order of a step with sub-buffers of the workspace, so every tensor (int8 operands, scales, bf16
// outputs) has the bits the separate calls give, also where the GEMM kernels are chosen for the call as a whole.
#include "ti8_common.h"

namespace ti8 {

namespace {

// Sub-buffers of the workspace, each starting on a 256-byte boundary.
struct Carver {
    char* base;
    int64_t used = 0;
    template <class T>
    T* take(int64_t count) {
        T* p = reinterpret_cast<T*>(base + used);
        used += (count * (int64_t)sizeof(T) + 255) / 256 * 256;
        return p;
    }
};

constexpr int64_t ROTATE_TOGETHER_BYTES = (int64_t)192 << 20;

// One call: its arguments with the token dim rounded up, and where every operand lives.
struct Layer {
    const ti8_linear_args* a;
    int64_t T, K, N, tokens;
    int scheme, had;
    bool fwd, bwd, keep;
    // a whole step whose workspace has no room for partial maxima (ti8_linear_fwd_bwd): they live in its outputs, see `quantise`
    bool partials_in_outputs = false;
    // layers that multiply the same X (ti8_linear_group): the one that quantises it (null: this one)
    const Layer* input_of = nullptr;
    // the GEMMs quantise the weight themselves: of its codes there are only the maxima, in their place
    bool raw_weight = false;
    // operands of Y = X W^T, dX = dY W, dW = dY^T X and their scales
    int8_t *xq, *wq, *dq, *wtq, *dytq, *xtq;
    float *xs, *ws, *ds, *wts, *dyts, *xts;
    unsigned int* maxima;       // scratch of the operands quantised both ways, or by columns: pieces of maxima_piece words
    int64_t maxima_words;
    uint16_t* scratch;          // transposed bf16 copy in front of a rotation along the rows

    bool block() const { return scheme == TI8_SCHEME_BLOCK_CHANNEL; }
    bool row_block() const { return scheme == TI8_SCHEME_ROW_BLOCK; }
    bool dbl() const { return scheme == TI8_SCHEME_DOUBLE_CHANNEL; }
    static int64_t maxima_piece(int64_t words) { return (words + 63) / 64 * 64; }
    // bytes of the operands of an unrotated call that are quantised by rows and by columns
    int64_t both_ways_bytes() const {
        const int64_t w = shares() && fwd && !row_block() ? N * K : 0, x = shares() && fwd && dbl() ? T * K : 0, dy = bwd && !block() ? T * N : 0;
        return 2 * (w + x + dy);
    }
    // R + C maxima, and the partial ones behind them where those are collected there
    int64_t partial_words(int64_t R, int64_t C) const { return partials_in_outputs || !quant_together(both_ways_bytes()) ? 0 : maxima_piece(quant_maxima_words(R, C)); }
    int64_t both_ways_words(int64_t R, int64_t C) const { return maxima_piece(R + C) + partial_words(R, C); }
    // whether the transposed copies in front of the rotations are made together (quant_fwht_call): while they find room in the Infinity Cache, and
    // in a workspace of about the operands' size (8192 tokens, 8192 -> 8192 takes 1807 us either way): up to 192 MiB for the copies of a backward, where
    // one after the other they take the largest one's
    bool rotates_together() const { return 2 * (N * K + T * N + T * K) <= ROTATE_TOGETHER_BYTES; }
    // what an unrotated forward quantises for the backward in the same pass
    bool shares() const { return had == 0 && (keep || (fwd && bwd)); }
    bool given_w() const { return a->wq != nullptr; }

    // The sizes alone: laid out at an address that is not null (a buffer already placed is told by that) and not used
    int64_t size(int64_t* saved_bytes) {
        char* const nowhere = reinterpret_cast<char*>(256);
        return carve(nowhere, nowhere, saved_bytes);
    }
    // Lay the buffers out; returns the bytes of workspace, *saved_bytes those of `saved`.
    int64_t carve(char* ws_base, char* saved_base, int64_t* saved_bytes) {
        Carver w{ws_base}, kept{saved_base};
        Carver& k = keep ? kept : w;
        const int64_t gk = K / 128, gn = N / 128, gt = T / 128;
        xq = wq = dq = wtq = dytq = xtq = nullptr;
        xs = ws = ds = wts = dyts = xts = nullptr;
        maxima_words = 0;
        maxima = nullptr;
        scratch = nullptr;
        // Reused by the backward (in `saved` when the two are separate calls): block-channel X^T and its grid, W^T by rows;
        // row-block W^T and its grid; double-channel X^T and W^T by rows
        const bool shared = shares();
        if (shared) {
            if (!row_block()) xtq = input_of ? input_of->xtq : k.take<int8_t>(T * K);
            wtq = k.take<int8_t>(N * K);
            if (block()) { xs = input_of ? input_of->xs : k.take<float>(gt * gk); wts = k.take<float>(K); }
            if (row_block()) ws = k.take<float>(gn * gk);
            if (dbl()) { xts = k.take<float>(K); wts = k.take<float>(K); }
        }
        if (fwd) {
            xq = input_of ? input_of->xq : w.take<int8_t>(T * K);
            if (!xs) xs = w.take<float>(block() ? gt * gk : T);
            if (given_w()) {
                wq = const_cast<int8_t*>(a->wq);
                ws = const_cast<float*>(a->ws);
            } else {
                wq = w.take<int8_t>(N * K);
                if (!ws) ws = w.take<float>(row_block() ? gn * gk : N);
            }
        }
        if (bwd) {
            dq = w.take<int8_t>(T * N);
            ds = w.take<float>(block() ? gt * gn : T);
            dytq = w.take<int8_t>(T * N);
            if (block() && had == 0) dyts = ds;
            else dyts = w.take<float>(block() ? gt * gn : N);
            if (!wtq) wtq = w.take<int8_t>(N * K);
            if (!wts) wts = row_block() ? (ws && had == 0 ? ws : w.take<float>(gn * gk)) : w.take<float>(K);
            if (!xtq) xtq = w.take<int8_t>(T * K);
            if (!xts) xts = block() && had == 0 && xs ? xs : w.take<float>(dbl() ? K : gt * gk);
            if (dbl() && had) {
                int64_t big = N * K;
                if (T * N > big) big = T * N;
                if (T * K > big) big = T * K;
                scratch = w.take<uint16_t>(rotates_together() ? N * K + T * N + T * K : big);
            }
        }
        // maxima: W by rows and columns in the forward (or W by columns in a backward that found nothing saved), dY and, for
        // the double-channel scheme, X likewise
        if (shared && fwd && !row_block()) maxima_words += both_ways_words(N, K);
        if (shared && fwd && dbl()) maxima_words += both_ways_words(T, K);
        if (bwd && had == 0 && !block()) maxima_words += both_ways_words(T, N);
        if (bwd && !shared && !row_block() && !(dbl() && had)) maxima_words += maxima_piece(K);      // W^T by columns
        if (bwd && !shared && dbl() && !had) maxima_words += maxima_piece(K);                        // X^T by columns
        if (bwd && row_block() && had) maxima_words += maxima_piece(N);                              // dY^T by rotated columns
        if (maxima_words) maxima = w.take<unsigned int>(maxima_words);
        if (saved_bytes) *saved_bytes = kept.used;
        return w.used;
    }
};

ti8_gemm_problem gemm2d(const int8_t* A, const float* sA, int modeA, int64_t sa_rs, int64_t sa_ks, const int8_t* B, const float* sB, int modeB,
                        int64_t sb_rs, int64_t sb_ks, void* C, int64_t ldc, int64_t M, int64_t N, int64_t K, int acc_i32_full, float out_scale, float post_scale) {
    ti8_gemm_problem p;
    p.A = A; p.bsa = 0; p.lda = K;
    p.B = B; p.bsb = 0; p.ldb = K;
    p.C = C; p.bsc = 0; p.ldc = ldc;
    p.sA = sA; p.modeA = modeA; p.sa_bs = 0; p.sa_rs = sa_rs; p.sa_ks = sa_ks;
    p.sB = sB; p.modeB = modeB; p.sb_bs = 0; p.sb_rs = sb_rs; p.sb_ks = sb_ks;
    p.batch = 1; p.M = M; p.N = N; p.K = K;
    p.acc_i32_full = acc_i32_full; p.combine = TI8_COMBINE_MUL_MUL;
    p.out_scale = out_scale; p.post_scale = post_scale;
    return p;
}

// Argument checks of every layer call, made before the first launch; fills the part of `L` that describes the call
int check_layer(const char* fn, const ti8_linear_args* a, int64_t T, Layer* L) {
    const int KNOWN = TI8_PART_FORWARD | TI8_PART_BACKWARD | TI8_PART_KEEP;
    L->a = a;
    L->T = T; L->K = a->K; L->N = a->N; L->tokens = a->tokens;
    L->scheme = a->scheme; L->had = a->hadamard;
    L->fwd = (a->parts & TI8_PART_FORWARD) != 0;
    L->bwd = (a->parts & TI8_PART_BACKWARD) != 0;
    L->keep = (a->parts & TI8_PART_KEEP) != 0;
    if (a->scheme < TI8_SCHEME_BLOCK_CHANNEL || a->scheme > TI8_SCHEME_DOUBLE_CHANNEL) return fail(TI8_ERR_MODE, "%s: unknown scheme %d", fn, a->scheme);
    if (a->hadamard != 0 && a->hadamard != (L->dbl() ? TI8_HADAMARD_FULL : 128)) return fail(TI8_ERR_MODE, "%s: rotation %d does not go with scheme %d", fn, a->hadamard, a->scheme);
    if ((a->parts & ~KNOWN) || (!L->fwd && !L->bwd) || (L->fwd && L->bwd && L->keep)) return fail(TI8_ERR_MODE, "%s: bad parts 0x%x", fn, a->parts);
    if (L->given_w() && (L->bwd || L->keep || !a->ws)) return fail(TI8_ERR_MODE, "%s: a weight quantised earlier serves a forward that keeps nothing, and brings its scales", fn);
    const int64_t K = a->K, N = a->N;
    if (T <= 0 || K <= 0 || N <= 0 || T % 128 || K % 128 || N % 128 || T > 0x3fffffff || K > 0x3fffffff || N > 0x3fffffff)
        return fail(TI8_ERR_SHAPE, "%s: T, K and N must be positive multiples of 128 (zero-pad the tokens); got T=%lld K=%lld N=%lld", fn,
                    (long long)T, (long long)K, (long long)N);
    if (a->tokens < 1 || a->tokens > T) return fail(TI8_ERR_SHAPE, "%s: tokens must be in [1, T]; got tokens=%lld T=%lld", fn, (long long)a->tokens, (long long)T);
    return TI8_OK;
}

int check_pointers(const char* fn, const ti8_linear_args* a, const Layer& L) {
    const bool need_w = !L.given_w() && (L.fwd || !L.shares()), need_x = L.fwd || !L.shares() || L.row_block();
    if ((need_x && !a->X) || (need_w && !a->W) || (L.bwd && (!a->dY || !a->dX || !a->dW)) || (L.fwd && !a->Y))
        return fail(TI8_ERR_NULL, "%s: X, W, dY, Y, dX and dW are required", fn);
    const int64_t K = a->K, N = a->N;
    auto rows_ok = [](const void* p, int64_t ld, int64_t cols) { return !p || ld >= cols; };
    auto aligned = [](const void* p, int64_t ld) { return !p || (aligned16(p) && ld % 8 == 0); };
    if (!rows_ok(a->X, a->ldx, K) || !rows_ok(a->W, a->ldw, K) || (L.bwd && (!rows_ok(a->dY, a->lddy, N) || !rows_ok(a->dX, a->lddx, K) || !rows_ok(a->dW, a->lddw, K))) ||
        (L.fwd && !rows_ok(a->Y, a->ldy, N)))
        return fail(TI8_ERR_SHAPE, "%s: leading dimension smaller than the row length", fn);
    // what the quantisers (inputs) and the GEMM epilogues (outputs) need, checked here so that nothing is launched before a rejection
    if (!aligned(a->X, a->ldx) || !aligned(a->W, a->ldw) || (L.bwd && (!aligned(a->dY, a->lddy) || !aligned(a->dX, a->lddx) || !aligned(a->dW, a->lddw))) ||
        (L.fwd && (!aligned(a->Y, a->ldy) || !aligned(a->bias, 0))) || !aligned(a->wq, 0))
        return fail(TI8_ERR_ALIGN, "%s: X, W, dY, Y, dX, dW and the bias must be 16-byte aligned with leading dimensions multiples of 8 elements", fn);
    // limits of the quantisers that this call launches
    const bool shared = L.shares(), row_k = L.fwd && (L.row_block() || ((L.had || !shared) && !(L.block() && L.given_w())));
    const bool row_n = L.bwd && L.had && !L.block();
    if ((row_k && K > 32768) || (row_n && N > 32768) || (L.dbl() && L.had && L.bwd && L.T > 32768))
        return fail(TI8_ERR_SHAPE, "%s: per-row quantisation takes up to 32768 columns", fn);
    // an operand quantised by columns: a workgroup row per 32 rows of it (the token operands, the weight)
    const bool tokens_by_columns = (L.row_block() && L.bwd) || (L.dbl() && !L.had && (L.bwd || shared));
    const bool weight_by_columns = (L.fwd && shared && !L.row_block()) || (L.bwd && !shared && (L.block() || (L.dbl() && !L.had)));
    if ((tokens_by_columns && L.T / 32 > 65535) || (weight_by_columns && N / 32 > 65535)) return fail(TI8_ERR_SHAPE, "%s: too many tiles", fn);
    if (a->gemm_flags & ~(TI8_GEMM_TILED | TI8_GEMM_LARGE_TILES | TI8_GEMM_ONE_TILE)) return fail(TI8_ERR_MODE, "%s: only TI8_GEMM_TILED, TI8_GEMM_LARGE_TILES and TI8_GEMM_ONE_TILE apply here", fn);
    return TI8_OK;
}

// A matrix of bf16 in memory
struct Rows {
    const char* p;
    int64_t rows, ld, cols;
    bool apart(const Rows& o) const {
        if (!p || !o.p || p + ((rows - 1) * ld + cols) * 2 <= o.p || o.p + ((o.rows - 1) * o.ld + o.cols) * 2 <= p) return true;
        if (ld != o.ld) return false;
        const int64_t ahead = ((o.p - p) / 2 % ld + ld) % ld;       // columns of one buffer, beside each other
        return ahead >= cols && ahead + o.cols <= ld;
    }
};
Rows matrix(const void* p, int64_t rows, int64_t ld, int64_t cols) { return Rows{static_cast<const char*>(p), rows, ld, cols}; }

// Whether the outputs of a call share no memory with each other
bool outputs_apart(const ti8_linear_args& a, int64_t T) {
    const bool fwd = (a.parts & TI8_PART_FORWARD) != 0, bwd = (a.parts & TI8_PART_BACKWARD) != 0;
    const Rows y = matrix(fwd ? a.Y : nullptr, T, a.ldy, a.N), dx = matrix(bwd ? a.dX : nullptr, T, a.lddx, a.K), dw = matrix(bwd ? a.dW : nullptr, a.N, a.lddw, a.K);
    return y.apart(dx) && y.apart(dw) && dx.apart(dw);
}

// Whether those of a whole step share none with its inputs, either
bool step_apart(const ti8_linear_args& a, int64_t T) {
    const Rows in[3] = {matrix(a.X, a.tokens, a.ldx, a.K), matrix(a.W, a.N, a.ldw, a.K), matrix(a.dY, a.tokens, a.lddy, a.N)};
    const Rows out[3] = {matrix(a.Y, T, a.ldy, a.N), matrix(a.dX, T, a.lddx, a.K), matrix(a.dW, a.N, a.lddw, a.K)};
    for (const Rows& i : in)
        for (const Rows& o : out)
            if (!i.apart(o)) return false;
    return outputs_apart(a, T);
}

// Operands that go into the two quantiser launches of a call: without a rotation, those quantised by blocks and those quantised by rows and by
// columns, without a launch that only clears maxima (quant_call: 16 tokens, 4096 -> 4096, block-channel 41 -> 37.6 us; 3072 tokens
// row-block 210 -> 204)
struct Operands {
    ti8_qblock_operand by_block[4];
    int64_t by_block_rows[4];
    QRowColOperand both[3];
    int nblocks = 0, nboth = 0;
    QRowOperand rows;
    bool by_rows = false;
    QHadOperand rotated[QHAD_MAX];      // with H_128: all of them
    int nrotated = 0;
    QFwhtOperand whole[QFWHT_MAX];      // with the rotation over whole rows: likewise
    int nwhole = 0;
};
int quantise_operands(const char* fn, const Layer& L, const Operands& o, ti8_stream_t stream) {
    if (o.nwhole) return quant_fwht_call(fn, o.whole, o.nwhole, L.rotates_together(), TI8_Q_CLAMP, TI8_INV_AMAX_DIV_127, stream);
    if (o.nrotated) return quant_had_call(fn, o.rotated, o.nrotated, TI8_Q_CLAMP, TI8_INV_RCP_OF_SCALE, stream);
    return quant_call(fn, o.by_block, o.by_block_rows, o.nblocks, o.both, o.nboth, o.by_rows ? &o.rows : nullptr, TI8_Q_CLAMP,
                      L.dbl() ? TI8_INV_AMAX_DIV_127 : TI8_INV_RCP_OF_SCALE, stream);
}

// Enqueue the quantisers of a call but for those that are added to `o`, and describe its GEMMs.  The order is that of linear_forward +
// linear_backward in the Python layer.
int quantise(const char* fn, Layer& L, Operands& o, ti8_gemm_problem* g, int* count, ti8_stream_t stream) {
    const ti8_linear_args& a = *L.a;
    const int64_t T = L.T, K = L.K, N = L.N, tok = L.tokens;
    const int q = TI8_Q_CLAMP;
    const int inv = L.dbl() ? TI8_INV_AMAX_DIV_127 : TI8_INV_RCP_OF_SCALE;
    const bool shared = L.shares();
    unsigned int* mx = L.maxima;
    auto take_maxima = [&](int64_t words) {
        unsigned int* p = mx;
        mx += Layer::maxima_piece(words);
        return reinterpret_cast<float*>(p);
    };
    // (`out`, `ldout`: the output of the operand's own shape, which a whole step does not write before its GEMMs; with
    // partials_in_outputs the partial maxima live there until the conversion has read them, unless the caller's tensors overlap)
    const bool apart = L.partials_in_outputs && step_apart(a, T);
    auto row_col = [&](const void* x, int64_t ldx, int8_t* oq, float* os, int8_t* oqT, float* osT, int64_t R, int64_t valid, int64_t C, void* out, int64_t ldout) {
        unsigned int* const scratch = reinterpret_cast<unsigned int*>(take_maxima(R + C));
        unsigned int* partial = nullptr;
        if (L.partial_words(R, C)) partial = reinterpret_cast<unsigned int*>(take_maxima(quant_maxima_words(R, C)));
        else if (apart && ldout == C) partial = static_cast<unsigned int*>(out);
        const bool raw = L.raw_weight && x == a.W;
        if (raw) partial = reinterpret_cast<unsigned int*>(oq);
        o.both[o.nboth++] = QRowColOperand{x, ldx, oq, os, oqT, osT, scratch, partial, R, valid, C, raw};
    };
    auto rotated = [&](int kind, const void* x, int64_t ldx, int8_t* oq, float* os, int64_t R, int64_t valid, int64_t C, float* maxima = nullptr) {
        o.rotated[o.nrotated++] = QHadOperand{x, ldx, oq, os, R, valid, C, kind, reinterpret_cast<unsigned int*>(maxima)};
    };
    auto whole = [&](const void* x, int64_t ldx, int8_t* oq, float* os, int64_t R, int64_t valid, int64_t C, uint16_t* scratch = nullptr) {
        o.whole[o.nwhole++] = QFwhtOperand{x, ldx, oq, os, R, valid, C, scratch != nullptr, scratch};
    };
    auto block = [&](const ti8_qblock_operand& operand, int64_t valid) {
        o.by_block_rows[o.nblocks] = valid;
        o.by_block[o.nblocks++] = operand;
    };
    auto blocks = [&](const void* x, int64_t ldx, int8_t* oq, int8_t* oqT, float* os, int64_t R, int64_t C) {
        return ti8_qblock_operand{x, 0, ldx, oq, R * C, C, oqT, R * C, R, os, 0, C / 128, 1, 1, R, C};
    };
    int n = 0;
    const float rot = L.had == 128 ? 0.0078125f : 1.0f;     // 2^-7: both operands carry an un-normalised H_128

    if (L.fwd) {
        float post = 0.0f;
        if (L.block() && L.had) {
            rotated(QHAD_BLOCKS, a.X, a.ldx, L.xq, L.xs, T, tok, K);
            if (!L.given_w()) rotated(QHAD_ROWS, a.W, a.ldw, L.wq, L.ws, N, N, K);
        } else if (L.block()) {
            if (!L.input_of) block(blocks(a.X, a.ldx, L.xq, shared ? L.xtq : nullptr, L.xs, T, K), tok);
            if (shared) row_col(a.W, a.ldw, L.wq, L.ws, L.wtq, L.wts, N, N, K, a.dW, a.lddw);     // rows for Y, columns for dX
            else if (!L.given_w())
                if (int e = ti8_quant_row(a.W, a.ldw, L.wq, K, L.ws, N, K, 0, q, inv, stream)) return e;
        } else if (L.row_block()) {
            if (L.had) {
                rotated(QHAD_ROWS, a.X, a.ldx, L.xq, L.xs, tok, tok, K);
                if (!L.given_w()) rotated(QHAD_BLOCKS, a.W, a.ldw, L.wq, L.ws, N, N, K);
            } else {
                o.rows = QRowOperand{a.X, a.ldx, L.xq, L.xs, tok, K};
                o.by_rows = true;
                if (!L.given_w()) block(blocks(a.W, a.ldw, L.wq, shared ? L.wtq : nullptr, L.ws, N, K), N);
            }
        } else if (L.had) {
            post = (float)(1.0 / (double)K);
            whole(a.X, a.ldx, L.xq, L.xs, tok, tok, K);
            if (!L.given_w()) whole(a.W, a.ldw, L.wq, L.ws, N, N, K);
        } else if (shared) {
            row_col(a.X, a.ldx, L.xq, L.xs, L.xtq, L.xts, T, tok, K, a.dX, a.lddx);
            row_col(a.W, a.ldw, L.wq, L.ws, L.wtq, L.wts, N, N, K, a.dW, a.lddw);
        } else {
            if (int e = ti8_quant_row(a.X, a.ldx, L.xq, K, L.xs, tok, K, 0, q, inv, stream)) return e;
            if (!L.given_w()) if (int e = ti8_quant_row(a.W, a.ldw, L.wq, K, L.ws, N, K, 0, q, inv, stream)) return e;
        }
        const bool xb = L.block(), wb = L.row_block();
        g[n++] = gemm2d(L.xq, L.xs, xb ? TI8_SCALE_BLOCK128 : TI8_SCALE_ROW, xb ? K / 128 : 1, xb ? 1 : 0,
                        L.wq, L.ws, wb ? TI8_SCALE_BLOCK128 : TI8_SCALE_ROW, wb ? K / 128 : 1, wb ? 1 : 0, a.Y, a.ldy, T, N, K, L.dbl(), rot, post);
    }
    if (L.bwd) {
        float post_dx = 0.0f, post_dw = 0.0f;
        int64_t dyts_rs = 1, dyts_ks = 0, xts_rs = 1, xts_ks = 0, wts_rs = 1, wts_ks = 0;
        int dyt_mode = TI8_SCALE_ROW, xt_mode = TI8_SCALE_ROW, wt_mode = TI8_SCALE_ROW;
        // a transposed operand's block scales are the transposed grid: no copy
        auto grid_t = [](int64_t cols, int64_t* rs, int64_t* ks, int* mode) { *rs = 1; *ks = cols / 128; *mode = TI8_SCALE_BLOCK128; };
        if (L.block() && L.had) {
            // H_128 along N for dX, along the tokens for dW: two differently rotated copies
            rotated(QHAD_BLOCKS, a.dY, a.lddy, L.dq, L.ds, T, tok, N);
            rotated(QHAD_COLUMNS, a.W, a.ldw, L.wtq, L.wts, N, N, K, take_maxima(K));
            rotated(QHAD_BLOCKS_T, a.dY, a.lddy, L.dytq, L.dyts, T, tok, N);
            rotated(QHAD_BLOCKS_T, a.X, a.ldx, L.xtq, L.xts, T, tok, K);
        } else if (L.block()) {
            block(blocks(a.dY, a.lddy, L.dq, L.dytq, L.ds, T, N), tok);
            if (!shared) {
                if (int e = quant_col_t_valid(a.W, a.ldw, L.wtq, N, L.wts, take_maxima(K), N, N, K, q, inv, stream)) return e;
                block(blocks(a.X, a.ldx, nullptr, L.xtq, L.xts, T, K), tok);
            }
        } else if (L.row_block() && L.had) {
            rotated(QHAD_ROWS, a.dY, a.lddy, L.dq, L.ds, tok, tok, N);
            rotated(QHAD_BLOCKS_T, a.W, a.ldw, L.wtq, L.wts, N, N, K);
            rotated(QHAD_COLUMNS, a.dY, a.lddy, L.dytq, L.dyts, T, tok, N, take_maxima(N));
            rotated(QHAD_BLOCKS_T, a.X, a.ldx, L.xtq, L.xts, T, tok, K);
        } else if (L.row_block()) {
            row_col(a.dY, a.lddy, L.dq, L.ds, L.dytq, L.dyts, T, tok, N, a.Y, a.ldy);
            if (!shared) block(blocks(a.W, a.ldw, nullptr, L.wtq, L.wts, N, K), N);
            block(blocks(a.X, a.ldx, nullptr, L.xtq, L.xts, T, K), tok);
        } else if (L.had) {
            // the transposed operands are rotated along the rows of the tensors as they lie in memory
            post_dx = (float)(1.0 / (double)N);
            post_dw = (float)(1.0 / (double)T);
            const bool apart_scratch = L.rotates_together();
            whole(a.dY, a.lddy, L.dq, L.ds, tok, tok, N);
            whole(a.W, a.ldw, L.wtq, L.wts, N, N, K, L.scratch);
            whole(a.dY, a.lddy, L.dytq, L.dyts, T, tok, N, L.scratch + (apart_scratch ? N * K : 0));
            whole(a.X, a.ldx, L.xtq, L.xts, T, tok, K, L.scratch + (apart_scratch ? N * K + T * N : 0));
        } else {
            row_col(a.dY, a.lddy, L.dq, L.ds, L.dytq, L.dyts, T, tok, N, a.Y, a.ldy);
            if (!shared) {
                if (int e = quant_col_t_valid(a.W, a.ldw, L.wtq, N, L.wts, take_maxima(K), N, N, K, q, inv, stream)) return e;
                if (int e = quant_col_t_valid(a.X, a.ldx, L.xtq, T, L.xts, take_maxima(K), T, tok, K, q, inv, stream)) return e;
            }
        }
        if (L.block()) { grid_t(N, &dyts_rs, &dyts_ks, &dyt_mode); grid_t(K, &xts_rs, &xts_ks, &xt_mode); }
        if (L.row_block()) { grid_t(K, &wts_rs, &wts_ks, &wt_mode); grid_t(K, &xts_rs, &xts_ks, &xt_mode); }
        g[n++] = gemm2d(L.dq, L.ds, L.block() ? TI8_SCALE_BLOCK128 : TI8_SCALE_ROW, L.block() ? N / 128 : 1, L.block() ? 1 : 0,
                        L.wtq, L.wts, wt_mode, wts_rs, wts_ks, a.dX, a.lddx, T, K, N, L.dbl(), rot, post_dx);
        g[n++] = gemm2d(L.dytq, L.dyts, dyt_mode, dyts_rs, dyts_ks, L.xtq, L.xts, xt_mode, xts_rs, xts_ks, a.dW, a.lddw, N, K, T, L.dbl(), rot, post_dw);
    }
    *count = n;
    return TI8_OK;
}

int gemms(const Layer& L, const ti8_gemm_problem* g, int count, ti8_stream_t stream) {
    const int flags = L.a->gemm_flags;
    // rows of a token operand to multiply: all of them, or with up to 256 (padded) tokens the real ones rounded up to 32 (the padding
    // rows of the 128-row-quantised operand are zeros whose products nobody reads)
    auto live_rows = [&](int64_t contraction) {
        if (L.T > 256 || (flags & (TI8_GEMM_TILED | TI8_GEMM_LARGE_TILES)) || contraction > 32768) return L.T;
        const int64_t r = (L.tokens + 31) / 32 * 32;
        return r < L.T ? r : L.T;
    };
    // outputs that share memory: a launch each, so that the last one stands
    const bool apart = count == 1 || outputs_apart(*L.a, L.T);
    // they go into one launch where none of them has so few rows that it would take the few-rows kernel
    if (L.bwd && (L.T < L.N ? L.T : L.N) > 256) {
        for (int i = 0, n = apart ? count : 1; i < count; i += n) {
            if (int e = ti8_gemm_i8_nt_multi(g + i, n, flags | TI8_GEMM_TOGETHER, stream)) return e;
            if (i == 0 && L.fwd && L.a->bias)       // (before dX or dW may take Y's place)
                if (int e = add_bias(L.a->Y, L.a->ldy, L.a->bias, L.tokens, L.N, stream)) return e;
        }
        return TI8_OK;
    }
    ti8_gemm_problem few[3];
    const void* const bias = L.fwd ? L.a->bias : nullptr;
    for (int i = 0; i < count; ++i) {
        few[i] = g[i];
        if (i + 1 < count || !L.bwd) few[i].M = live_rows(g[i].K);      // dW, the last of a backward, has one row per output feature
    }
    bool launched[3] = {false, false, false};
    if (count > 1 && apart)
        if (int e = gemm_nt_few(few, count, L.bwd, bias, flags, launched, stream)) return e;
    for (int i = 0; i < count; ++i)
        if (!launched[i])
            // launched alone: what ti8_gemm_i8_nt selects for its shape (the few-rows kernel up to 256 rows)
            if (int e = gemm_nt_bias(few[i], i == 0 ? bias : nullptr, flags, stream)) return e;
    return TI8_OK;
}

int run_layer(const char* fn, const ti8_linear_args* a, int64_t T, ti8_gemm_problem* problems, int* count, ti8_stream_t stream, bool partials_in_outputs = false) {
    Layer L;
    if (int e = check_layer(fn, a, T, &L)) return e;
    L.partials_in_outputs = partials_in_outputs;
    if (int e = check_pointers(fn, a, L)) return e;
    int64_t need_saved = 0;
    const int64_t need = L.size(&need_saved);
    if (!a->workspace || (reinterpret_cast<uintptr_t>(a->workspace) & 255) || a->workspace_bytes < need)
        return fail(TI8_ERR_SHAPE, "%s: the workspace must be 256-byte aligned and hold %lld bytes (ti8_linear_workspace); got %lld", fn,
                    (long long)need, (long long)(a->workspace ? a->workspace_bytes : 0));
    if (need_saved && (!a->saved || (reinterpret_cast<uintptr_t>(a->saved) & 255) || a->saved_bytes < need_saved))
        return fail(TI8_ERR_SHAPE, "%s: `saved` must be 256-byte aligned and hold %lld bytes (ti8_linear_workspace); got %lld", fn,
                    (long long)need_saved, (long long)(a->saved ? a->saved_bytes : 0));
    L.carve(static_cast<char*>(a->workspace), static_cast<char*>(a->saved), nullptr);
    // (a kernel that reads X itself cannot write Y where other workgroups are still reading it)
    if (!problems && L.fwd && !L.bwd && !L.had && !L.keep && L.given_w() && matrix(a->X, a->tokens, a->ldx, a->K).apart(matrix(a->Y, 32, a->ldy, a->N))) {
        const int64_t K = L.K, N = L.N;
        bool done = false;
        const bool xb = L.block(), wb = L.row_block();
        if (int e = gemm_nt_decode(gemm2d(L.xq, L.xs, xb ? TI8_SCALE_BLOCK128 : TI8_SCALE_ROW, xb ? K / 128 : 1, xb ? 1 : 0, L.wq, L.ws,
                                          wb ? TI8_SCALE_BLOCK128 : TI8_SCALE_ROW, wb ? K / 128 : 1, wb ? 1 : 0, a->Y, a->ldy, 32, N, K, L.dbl(), 1.0f, 0.0f),
                                   a->X, a->ldx, L.tokens, a->bias, a->gemm_flags, &done, stream)) return e;
        if (done) return TI8_OK;
    }
    L.raw_weight = !problems && T <= 256 && L.fwd && L.bwd && !L.had && L.block() && !a->bias && !(a->gemm_flags & (TI8_GEMM_TILED | TI8_GEMM_LARGE_TILES)) &&
                   quant_together(L.both_ways_bytes()) && gemm_raw_weight_takes(L.tokens, L.K, L.N, a->ldw) && step_apart(*a, T);
    ti8_gemm_problem g[3];
    int n = 0;
    Operands operands;
    if (int e = quantise(fn, L, operands, g, &n, stream)) return e;
    if (int e = quantise_operands(fn, L, operands, stream)) return e;
    if (L.raw_weight) return gemm_nt_raw_weight(g, operands.both[0], L.tokens, stream);
    if (problems) {
        for (int i = 0; i < n; ++i) problems[i] = g[i];
        *count = n;
        return TI8_OK;
    }
    return gemms(L, g, n, stream);
}

// ---- layers on the same X ----------------------------------------------------------------
// The seven linears of a decoder layer are three calls of this kind (q, k, v; gate, up) and two alone: X is quantised once for a
// call, the weights' (the dYs') quantisers are two launches (one) for all of it and the GEMMs one (two).  The whole layer, us apart
// / so: 3 x 1360 tokens, hidden 2048, MLP 4992 1634 / 1497; 4 x 4096, hidden 4096, MLP 14336 18270 / 17930.  In memory, the backward holds the codes of
// all its dY at once (gate and up of 16384 x 14336: 940 MB, apart 470) and a [T][K] dX of each further layer, the layers between the directions
// X's codes and scales once: peak of the larger layer 4779 MiB, apart 4939, of the smaller 589 / 584.
constexpr int GROUP_MAX = 3;
struct Group {
    Layer L[GROUP_MAX];
    int count;
    void* dx[GROUP_MAX];        // backward: dX of each layer, [T][K] but for the first, which is the sum's own place

    // As Layer::carve, of the whole call
    int64_t carve(char* ws_base, char* saved_base, int64_t* saved_bytes) {
        int64_t used = 0, kept = 0;
        for (int i = 0; i < count; ++i) {
            int64_t k = 0;
            L[i].input_of = i ? &L[0] : nullptr;
            used += L[i].carve(ws_base + used, saved_base + kept, &k);
            kept += k;
        }
        for (int i = 1; i < count && L[0].bwd; ++i) {
            dx[i] = ws_base + used;
            used += (L[0].T * L[0].K * 2 + 255) / 256 * 256;
        }
        *saved_bytes = kept;
        return used;
    }
    int64_t size(int64_t* saved_bytes) {
        char* const nowhere = reinterpret_cast<char*>(256);
        return carve(nowhere, nowhere, saved_bytes);
    }
};

int check_group(const char* fn, const ti8_linear_args* a, int count, Group* g) {
    if (count < 2 || count > GROUP_MAX) return fail(TI8_ERR_SHAPE, "%s: between 2 and %d layers, got %d", fn, GROUP_MAX, count);
    g->count = count;
    for (int i = 0; i < count; ++i) {
        if (int e = check_layer(fn, a + i, (a[i].tokens + 127) / 128 * 128, &g->L[i])) return e;
        if (a[i].scheme != TI8_SCHEME_BLOCK_CHANNEL || a[i].hadamard || !g->L[i].keep || a[i].wq || a[i].bias)
            return fail(TI8_ERR_MODE, "%s: block-channel layers without rotation or bias, forward or backward with TI8_PART_KEEP", fn);
        if (a[i].parts != a[0].parts || a[i].tokens != a[0].tokens || a[i].K != a[0].K || a[i].X != a[0].X || a[i].ldx != a[0].ldx || a[i].gemm_flags != a[0].gemm_flags)
            return fail(TI8_ERR_SHAPE, "%s: the layers must have parts, X, tokens, K and gemm_flags in common", fn);
    }
    return TI8_OK;
}

int run_group(const char* fn, const ti8_linear_args* given, int count, ti8_stream_t stream) {
    Group G;
    if (int e = check_group(fn, given, count, &G)) return e;
    const ti8_linear_args& first = given[0];
    int64_t need_saved = 0;
    const int64_t need = G.size(&need_saved);
    if (!first.workspace || (reinterpret_cast<uintptr_t>(first.workspace) & 255) || first.workspace_bytes < need || !first.saved ||
        (reinterpret_cast<uintptr_t>(first.saved) & 255) || first.saved_bytes < need_saved)
        return fail(TI8_ERR_SHAPE, "%s: the first layer's workspace and `saved` must be 256-byte aligned and hold %lld and %lld bytes (ti8_linear_group_workspace)",
                    fn, (long long)need, (long long)need_saved);
    G.carve(static_cast<char*>(first.workspace), static_cast<char*>(first.saved), &need_saved);
    const bool fwd = G.L[0].fwd;
    const int64_t T = G.L[0].T, K = G.L[0].K;
    ti8_linear_args a[GROUP_MAX];
    Rows out[2 * GROUP_MAX];
    int outs = 0;
    for (int i = 0; i < count; ++i) {
        a[i] = given[i];
        if (!fwd && i) {
            a[i].dX = G.dx[i];
            a[i].lddx = K;
        }
        G.L[i].a = &a[i];
        if (int e = check_pointers(fn, &a[i], G.L[i])) return e;
        if (fwd) out[outs++] = matrix(a[i].Y, T, a[i].ldy, a[i].N);
        else out[outs++] = matrix(a[i].dW, a[i].N, a[i].lddw, K);
    }
    if (!fwd) out[outs++] = matrix(first.dX, T, first.lddx, K);
    for (int i = 0; i < outs; ++i)
        for (int j = 0; j < i; ++j)
            if (!out[i].apart(out[j])) return fail(TI8_ERR_SHAPE, "%s: the outputs of the layers must not share memory", fn);

    ti8_gemm_problem g[GROUP_MAX][3], by_kind[3][GROUP_MAX];
    Operands operands;
    int n = 0;
    for (int i = 0; i < count; ++i) {
        if (int e = quantise(fn, G.L[i], operands, g[i], &n, stream)) return e;
        for (int k = 0; k < n; ++k) by_kind[k][i] = g[i][k];
    }
    if (int e = quantise_operands(fn, G.L[0], operands, stream)) return e;
    bool large = T > 256;       // (as for one layer: none of them on the few-rows kernel)
    for (int i = 0; i < count && !fwd; ++i) large = large && a[i].N > 256;
    if (large) {
        for (int k = 0; k < n; ++k)
            if (int e = ti8_gemm_i8_nt_multi(by_kind[k], count, first.gemm_flags | TI8_GEMM_TOGETHER, stream)) return e;
    } else if (fwd) {
        if (int e = gemms(G.L[0], by_kind[0], count, stream)) return e;
    } else {
        for (int i = 0; i < count; ++i)
            if (int e = gemms(G.L[i], g[i], n, stream)) return e;
    }
    if (fwd) return TI8_OK;
    // in the order in which autograd adds up the gradients of layers that were called one after the other
    return add_rows(fn, first.dX, first.lddx, G.dx[1], count > 2 ? G.dx[2] : nullptr, G.L[0].tokens, K, stream);
}

}  // namespace
}  // namespace ti8

using namespace ti8;

extern "C" int64_t ti8_linear_workspace(const ti8_linear_args* a, int64_t* saved_bytes) {
    if (!a || a->tokens < 1) return -1;
    Layer L;
    if (check_layer("ti8_linear_workspace", a, (a->tokens + 127) / 128 * 128, &L)) return -1;
    return L.size(saved_bytes);
}

extern "C" int ti8_linear_quantise(const ti8_linear_args* a, ti8_gemm_problem* problems, int* count, ti8_stream_t stream) {
    const char* fn = "ti8_linear_quantise";
    if (!a || !problems || !count) return fail(TI8_ERR_NULL, "%s: args, problems and count are required", fn);
    if (a->bias) return fail(TI8_ERR_MODE, "%s: the GEMMs that a bias goes with are the caller's", fn);
    return run_layer(fn, a, (a->tokens + 127) / 128 * 128, problems, count, stream);
}

extern "C" int ti8_linear(const ti8_linear_args* a, ti8_stream_t stream) {
    const char* fn = "ti8_linear";
    if (!a) return fail(TI8_ERR_NULL, "%s: args is required", fn);
    return run_layer(fn, a, (a->tokens + 127) / 128 * 128, nullptr, nullptr, stream);
}

extern "C" int64_t ti8_linear_group_workspace(const ti8_linear_args* a, int count, int64_t* saved_bytes) {
    if (!a || !saved_bytes || a->tokens < 1) return -1;
    Group g;
    if (check_group("ti8_linear_group_workspace", a, count, &g)) return -1;
    return g.size(saved_bytes);
}

extern "C" int ti8_linear_group(const ti8_linear_args* a, int count, ti8_stream_t stream) {
    const char* fn = "ti8_linear_group";
    if (!a) return fail(TI8_ERR_NULL, "%s: args is required", fn);
    return run_group(fn, a, count, stream);
}

// The whole step on a token dim that the caller has rounded up itself
static ti8_linear_args step_args(int64_t tokens, int64_t K, int64_t N, int scheme) {
    ti8_linear_args a = {};
    a.tokens = tokens; a.K = K; a.N = N;
    a.scheme = scheme;
    a.parts = TI8_PART_FORWARD | TI8_PART_BACKWARD;
    return a;
}

extern "C" int64_t ti8_linear_fwd_bwd_workspace(int64_t T, int64_t K, int64_t N, int scheme) {
    if (scheme != TI8_SCHEME_BLOCK_CHANNEL && scheme != TI8_SCHEME_DOUBLE_CHANNEL) return -1;
    const ti8_linear_args a = step_args(T, K, N, scheme);
    Layer L;
    if (check_layer("ti8_linear_fwd_bwd_workspace", &a, T, &L)) return -1;
    L.partials_in_outputs = true;
    return L.size(nullptr);
}

extern "C" int ti8_linear_fwd_bwd(const void* X, int64_t ldx, const void* W, int64_t ldw, const void* dY, int64_t lddy,
                                  void* Y, int64_t ldy, void* dX, int64_t lddx, void* dW, int64_t lddw,
                                  int64_t T, int64_t tokens, int64_t K, int64_t N, int scheme, int gemm_flags,
                                  void* workspace, int64_t workspace_bytes, ti8_stream_t stream) {
    const char* fn = "ti8_linear_fwd_bwd";
    if (scheme != TI8_SCHEME_BLOCK_CHANNEL && scheme != TI8_SCHEME_DOUBLE_CHANNEL)
        return fail(TI8_ERR_MODE, "%s: scheme must be TI8_SCHEME_BLOCK_CHANNEL or TI8_SCHEME_DOUBLE_CHANNEL, got %d", fn, scheme);
    ti8_linear_args a = step_args(tokens, K, N, scheme);
    a.X = X; a.ldx = ldx; a.W = W; a.ldw = ldw; a.dY = dY; a.lddy = lddy;
    a.Y = Y; a.ldy = ldy; a.dX = dX; a.lddx = lddx; a.dW = dW; a.lddw = lddw;
    a.gemm_flags = gemm_flags;
    a.workspace = workspace; a.workspace_bytes = workspace_bytes;
    return run_layer(fn, &a, T, nullptr, nullptr, stream, true);
}
