// Y of up to 8 rows of bf16 through a weight with few columns, quantised earlier, in one launch: every workgroup quantises the rows itself
// and multiplies them by 16 rows of the weight, K in quarters over its four waves.
//
// What bounds it at these sizes is latency: the launch, the rows' way from memory, their codes, the weight's way from memory and the sum of
// the waves, each behind the one before.  So the weight does not wait for the codes: a wave asks for 8 K tiles of it at once, straight
// into the registers that the matrix instructions read (16 rows x 64 bytes a load: as many 64-byte pieces as a dense one), while the rows
// are on their way, and for a further K tile whenever one is used up.  The codes of 8 K tiles are made together, 16 columns per lane, so that
// the absmax of a K tile is three steps over 8 lanes and not a reduction over the wave.  16 rows of the weight, half of what
// gemm_i8_decode_kernel takes, fill the CUs with twice as many workgroups; each makes all codes, which is what more columns or more rows cost:
// idx::decode_narrow says where the other is faster.  us in the kernel, 1 / 8 rows, the other one in brackets: 4096 -> 4096 4.9 / 6.6
// (7.5 / 7.4), 12288 -> 4096 11.5 / 15.6 (18.3), 14336 -> 1024 9.5 / 15.5 (17.3), 14336 -> 5120 18.5 / 32.1 (20.6).
//
// Codes, products and sums are those of gemm_i8_wavering_kernel's 32 x 32 blocks behind the quantisers, operation for operation: the same
// quarters, their K tiles in the same order, the same bits.
#include "gemm_args.h"
#include "quant_math.h"

namespace ti8 {

// How operand A's groups are scaled: a K tile of all rows (block-channel), or a row; with a row's scale the sums are promoted by operand B's
// block scales (row-block) or stay int32 over the whole K (double-channel)
enum class Decode { TILES, ROWS, ROWS_I32 };

constexpr int BATCH = idx::DECODE_BATCH;      // K tiles of the weight that a wave has under way, and whose codes it makes together

template <Decode MODE, int ROWS>
__global__ __launch_bounds__(256) void gemm_i8_decode_narrow_kernel(const GemmArgs g, const int rows) {
    constexpr bool I32 = MODE == Decode::ROWS_I32, BY_ROWS = MODE != Decode::TILES;
    __shared__ __attribute__((aligned(16))) int8_t codes[4][BATCH][ROWS][128];      // of the waves, 16-byte chunk c of row r at c ^ r
    __shared__ float4 sums[4][64];
    __shared__ float maxima[4][ROWS];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = blockIdx.x * 16, nk = g.K >> 7;
    const int kbeg = idx::few_k_first(wave, nk), nq = idx::few_k_first(wave + 1, nk) - kbeg;
    const int rot = idx::decode_rot(n0, nq);
    auto tile_of_step = [&](int i) { return idx::few_k_tile(i, rot, kbeg, nq, nk); };      // past the end: the last one again
    const int group = lane >> 3;                        // making the codes: this lane's K tile of a batch
    const int low = lane & 15, quad = lane >> 4;        // multiplying: its row of either operand, and its 16 bytes of 64 columns

    // 16 columns of every row in this lane's K tile of a batch (rows that there are not: the last one again)
    uint4 x[ROWS][2];
    auto row_at = [&](int batch, int r) {
        return reinterpret_cast<const uint16_t*>(g.A) + idx::decode_x_offset(min(r, rows - 1), g.lda, tile_of_step(batch * BATCH + group), lane);
    };
    auto load_rows = [&](int batch) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const uint16_t* const p = row_at(batch, r);
            x[r][0] = *reinterpret_cast<const uint4*>(p);
            x[r][1] = *reinterpret_cast<const uint4*>(p + 8);
        }
    };
    v4i w[BATCH][2];        // the halves of a K tile
    auto load_weight = [&](int step, v4i (&to)[2]) {
        const int8_t* const p = g.B + idx::decode_w_offset(n0, g.ldb, tile_of_step(step), lane);
        to[0] = *reinterpret_cast<const v4i*>(p);
        to[1] = *reinterpret_cast<const v4i*>(p + 64);
    };

    // what the last step needs, in front of all other loads so that it is there by then
    const int e_col = n0 + quad * 4;
    const bool col_part = I32 || g.sb.mode == TI8_SCALE_ROW;
    float coln[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) coln[c] = g.sb.p[col_part ? (int64_t)(e_col + c) * g.sb.rs : 0];
    const uint2 bias = *reinterpret_cast<const uint2*>(g.bias ? reinterpret_cast<const void*>(g.bias + e_col) : reinterpret_cast<const void*>(g.B));
    // operand B's block scale of this lane's K tile
    const float* const block_p = g.sb.p + (int64_t)(n0 >> 7) * g.sb.rs;
    auto block_scale = [&](int batch) { return MODE == Decode::ROWS ? block_p[(int64_t)tile_of_step(batch * BATCH + group) * g.sb.ks] : 1.0f; };

    float f_tile = block_scale(0);      // of this lane's K tile
    load_rows(0);
    __builtin_amdgcn_sched_barrier(0);
    float row_amax[ROWS], row_mult[ROWS], row_scale = 1.0f;     // row_scale: of row `low` of C
    if (BY_ROWS) {
        // the whole rows first: this wave's quarter beyond the K tiles at hand, which is read again for its codes
#pragma unroll
        for (int r = 0; r < ROWS; ++r) row_amax[r] = 0.0f;
        for (int batch = 1; batch * BATCH < nq; ++batch)
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                const uint16_t* const p = row_at(batch, r);
                row_amax[r] = absmax8(*reinterpret_cast<const uint4*>(p + 8), absmax8(*reinterpret_cast<const uint4*>(p), row_amax[r]));
            }
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int t = 0; t < BATCH; ++t)
        if (t < nq) load_weight(t, w[t]);
    __builtin_amdgcn_sched_barrier(0);
    if (BY_ROWS) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const float m = wave_max(nq > 0 ? absmax8(x[r][1], absmax8(x[r][0], row_amax[r])) : 0.0f);
            if (lane == 0) maxima[wave][r] = m;
        }
        // (written out: in front of the barrier that it knows the compiler waits for the weight, too)
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        auto of_row = [&](int r) { return amax_floor(fmaxf(fmaxf(maxima[0][r], maxima[1][r]), fmaxf(maxima[2][r], maxima[3][r])), 0); };
#pragma unroll
        for (int r = 0; r < ROWS; ++r) row_mult[r] = 127.0f / of_row(r);
        const float amax = of_row(low & (ROWS - 1));
        row_scale = I32 ? amax / 127.0f : 1.0f / (127.0f / amax);
    }

    auto quantise = [&]() {
        float scale = 0.0f;
        if (!BY_ROWS) {
            float amax = 0.0f;
#pragma unroll
            for (int r = 0; r < ROWS; ++r) amax = absmax8(x[r][1], absmax8(x[r][0], amax));
            scale = 127.0f / amax_floor(dpp_max<0x141>(dpp_max<0x4E>(dpp_max<0xB1>(amax))), 0);      // over the 8 lanes of a K tile
            f_tile = 1.0f / scale;
        }
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const float s = BY_ROWS ? row_mult[r] : scale;
            const uint2 lo = quant8(x[r][0], s), hi = quant8(x[r][1], s);
            *reinterpret_cast<uint4*>(&codes[wave][group][r][((lane & 7) ^ r) * 16]) = make_uint4(lo.x, lo.y, hi.x, hi.y);
        }
    };

    const v4i zero = {0, 0, 0, 0};
    v4i acc = zero;
    float accf[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    // K tile t of a batch.  C is computed transposed, 16 rows of the weight by 16 rows of X, the further ones of which are copies that nobody stores.
    const int code_row = low & (ROWS - 1);
    auto multiply = [&](int t, float f) {
        v4i d = I32 ? acc : zero;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            d = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[t][h], *reinterpret_cast<const v4i*>(&codes[wave][t][code_row][((4 * h + quad) ^ code_row) * 16]), d, 0, 0, 0);
        if (I32) acc = d;
        else
#pragma unroll
            for (int r = 0; r < 4; ++r) accf[r] = __builtin_fmaf(static_cast<float>(d[r]), f, accf[r]);
    };
    for (int batch = 0; batch * BATCH < nq; ++batch) {
        const int left = nq - batch * BATCH;
        quantise();
        const float f_batch = f_tile;
        if (left > BATCH) {
            f_tile = block_scale(batch + 1);
            load_rows(batch + 1);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < BATCH; ++t) {
            if (t < left) multiply(t, __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f_batch), t * 8)));
            if (t + BATCH < left) load_weight((batch + 1) * BATCH + t, w[t]);
        }
    }

    // lane: row `low` of C, columns 4 quad .. 4 quad + 3
    sums[wave][lane] = I32 ? make_float4(__int_as_float(acc[0]), __int_as_float(acc[1]), __int_as_float(acc[2]), __int_as_float(acc[3]))
                           : make_float4(accf[0], accf[1], accf[2], accf[3]);
    __syncthreads();
    if (wave > 0 || low >= rows) return;
    const float4 s0 = sums[0][lane], s1 = sums[1][lane], s2 = sums[2][lane], s3 = sums[3][lane];
    const float part[4][4] = {{s0.x, s0.y, s0.z, s0.w}, {s1.x, s1.y, s1.z, s1.w}, {s2.x, s2.y, s2.z, s2.w}, {s3.x, s3.y, s3.z, s3.w}};
    float t[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        float v;
        if (I32) {
            v = static_cast<float>(__float_as_int(part[0][c]) + __float_as_int(part[1][c]) + __float_as_int(part[2][c]) + __float_as_int(part[3][c])) * row_scale;
            v = v * coln[c];
        } else {
            v = part[0][c] + part[1][c];
            v = v + part[2][c];
            v = v + part[3][c];
            if (BY_ROWS) v = v * row_scale;
            if (col_part) v = v * coln[c];
        }
        t[c] = v;
    }
    uint2 o = make_uint2(pack_bf16x2(t[0], t[1]), pack_bf16x2(t[2], t[3]));
    if (g.bias) o = make_uint2(add_bf16x2(o.x, bias.x), add_bf16x2(o.y, bias.y));
    *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(g.C) + (int64_t)low * g.ldc + e_col) = o;
}

template <Decode MODE>
static void launch_mode(const GemmArgs& a, int rows, hipStream_t st) {
    const auto kernel = rows == 1 ? gemm_i8_decode_narrow_kernel<MODE, 1> : rows == 2 ? gemm_i8_decode_narrow_kernel<MODE, 2>
                                  : rows <= 4 ? gemm_i8_decode_narrow_kernel<MODE, 4> : gemm_i8_decode_narrow_kernel<MODE, 8>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(a.N / 16)), dim3(256), 0, st, a, rows);
}

int launch_decode_narrow(const GemmArgs& a, int rows, bool i32_full, hipStream_t st) {
    if (i32_full) launch_mode<Decode::ROWS_I32>(a, rows, st);
    else if (a.sa.mode == TI8_SCALE_ROW) launch_mode<Decode::ROWS>(a, rows, st);
    else launch_mode<Decode::TILES>(a, rows, st);
    note_gemm_kernel(TI8_KERNEL_FEW_ROWS, 32, 32, i32_full ? EPI_ROWS : EPI_PROMOTE, TI8_FORM_ROWS_NARROW);
    return check_launch("ti8_gemm_i8_nt");
}

}  // namespace ti8
