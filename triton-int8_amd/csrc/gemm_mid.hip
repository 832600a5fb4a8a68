// INT8 NT GEMM for medium sizes: 128 x 128 tiles on eight waves in two groups, half a K tile apart.
//
// Up to one 128 x 128 tile per CU the time of a GEMM is the time ONE workgroup takes for its K loop, and the tile on four
// waves (gemm.hip, one wave per SIMD) spends that loop waiting: load -> barrier -> LDS read -> MFMA -> convert + fma, one
// after the other, 1.0 us per K tile where the MFMAs take 0.22.  Here each of eight waves owns 32 rows x 64 columns of the
// tile, the upper or lower block row of a 64 x 64 quarter by its group, and every SIMD holds a wave of either group.
//
//  * The groups run half a K tile apart.  Phase M: the products of a K tile whose fragments are in registers, the previous
//    tile's second block folded between the MFMAs (4 vector instructions per MFMA; a second set of product registers lets
//    the MFMAs of both blocks alternate).  Phase F: the next tile's fragments out of LDS, the first block folded between the
//    reads.  While one group is in M the other is in F, so that MFMAs, vector instructions, LDS reads and loads run at the
//    same time; ONE barrier per phase.  (A single wave per SIMD issues a vector instruction every 7 cycles only, two waves
//    one every 4.)
//  * All fragments of a K tile are read in one phase, so a stage is free again when the second group has read it.  Both groups
//    fetch into it in the phase behind that, one in its M and one in its F: with four stages a load has five phases to land,
//    and three K tiles (96 KiB per CU) are in flight.  (Both in their M: group 1 a phase later, and a tile count that spreads
//    badly over the L2s waits: 1280 x 2944 x 8192 int32 44 us, 38 this way.)
//  * The order inside the phases is written out between scheduling barriers, and nothing branches inside a K tile (a loop for
//    each group): left to itself the compiler gathers the conversions in front and spills, or sinks them to the loop's end.
//
// Every sum runs over the K tiles in order, as on the other LDS-tiled kernels, so a GEMM has the same bits on all of them:
// which one serves it is a matter of speed alone.  (The K tiles of either parity on a group of their own, their sums added at
// the end, read a third less from LDS and is no faster; its other association moved the gradients of a decoder layer by up to
// 1.8e-2 through the int8 codes behind them.)
//
// What bounds it: 32 KiB per K tile and CU from L2 into LDS, 96 KiB of fragments out of it, and 512 cycles of MFMA per SIMD
// beside as many of convert + fma.  Promotion / int32, us (parities apart): 1024 rows, N = 4096, K = 14336 84 / 66 = 1.43 /
// 1.82 POP/s (82 / 66; four waves 109 / 74), K = 4096 27 / 23 (27 / 23); 2048 x 2048 x 2048 15.8 / 13.3 (16.6 / 15.4).
#include <type_traits>
#include "gemm_args.h"

namespace ti8 {

namespace {

constexpr int BM = 128, BN = 128, WN = 2, NW = 8;
constexpr int TN = 2;                               // 32 x 32 blocks per wave: one block row of two
constexpr int WCOLS = TN * 32;
constexpr int INSTR = 2;                            // global -> LDS instructions per wave, operand and K tile (16 rows)
constexpr int A_BYTES = BM * 128;
constexpr int STAGE_BYTES = A_BYTES + BN * 128;     // one K tile of both operands
constexpr int STAGES = 4;
constexpr int MAX_K_TILES = 256;
constexpr int LDS_BYTES = STAGES * STAGE_BYTES + MAX_K_TILES * 4;   // 128 KiB of operands, one factor per K tile
constexpr int WAIT_ALL_BUT_TWO_TILES = 0xf70 | (4 * INSTR);    // vmcnt: all but the youngest two K tiles' loads of this wave
static_assert(4 * INSTR < 16, "vmcnt[3:0]");
constexpr int WAIT_LDS = 0xc07f;                    // lgkmcnt(0)
constexpr int SLAB_LD = idx::EPI_SLAB_LD(WCOLS);    // words per row of a wave's 32 x 64 slab
static_assert(NW * 32 * SLAB_LD * 4 <= STAGES * STAGE_BYTES, "the epilogue's slabs lie over the operand buffers");

}  // namespace

template <bool I32>
__global__ __launch_bounds__(64 * NW) void gemm_i8_mid_kernel(const GemmMulti m) {
    extern __shared__ __attribute__((aligned(1024))) int8_t smem[];
    // layout: [stage][A 16 KiB][B 16 KiB], then the factors

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = wave >> 2, quarter = wave & 3;
    const int wm = quarter / WN, wn = quarter % WN;
    const int gi = idx::gemm_multi_pick((int)blockIdx.x, m.first[1], m.first[2], m.count);
    const GemmArgs& g = m.g[gi];
    const int batch = blockIdx.y;
    const idx::TileCoord tc = idx::gemm_tile_of((int)blockIdx.x - m.first[gi], g.tiles_m, g.tiles_n, idx::gemm_group_rows(BM), m.count > 1);
    const int m0 = tc.tile_m * BM, n0 = tc.tile_n * BN;
    const int nk = g.K >> 7, klast = (nk - 1) * 128;

    // ---- global -> LDS: the slab layout and swizzle of the other kernels (gemm.hip) -----------
    uint32_t voffA[2], voffB[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        voffA[p] = idx::gemm_lane_offset_bytes(lane, p, (int)g.lda);
        voffB[p] = idx::gemm_lane_offset_bytes(lane, p, (int)g.ldb);
    }
    const int8_t* const baseA = g.A + (int64_t)batch * g.bsa + (int64_t)idx::gemm_mid_first_row(m0, wave, g.M) * g.lda;
    const int8_t* const baseB = g.B + (int64_t)batch * g.bsb + (int64_t)idx::gemm_mid_first_row(n0, wave, g.N) * g.ldb;
    const int64_t strideA8 = 8 * g.lda, strideB8 = 8 * g.ldb;
    int8_t* const wdst = smem + wave * INSTR * 1024;
    // instruction q (of 4) of K tile t; a tile past the end is the last one again, into a buffer whose products nobody makes
    auto issue_one = [&](int t, int stage, int q) {
        const int koff = idx::gemm_k_offset(t, klast);
        if (q < INSTR) issue_tile_loads<1>(baseA + koff + q * strideA8, strideA8, voffA, q, wdst + stage * STAGE_BYTES + q * 1024);
        else issue_tile_loads<1>(baseB + koff + (q - INSTR) * strideB8, strideB8, voffB, q - INSTR, wdst + stage * STAGE_BYTES + A_BYTES + (q - INSTR) * 1024);
    };

    // ---- per-K-tile factors of the promotion: f_kt = fa_kt * fb_kt (an operand scaled per row contributes its vector in the
    // epilogue instead), the same for the whole tile, through LDS
    const bool divide = !I32 && g.combine == TI8_COMBINE_DIV_PROD;
    float* const factors = reinterpret_cast<float*>(smem + STAGES * STAGE_BYTES);
    if (!I32 && threadIdx.x < MAX_K_TILES) {
        const int kt = min((int)threadIdx.x, nk - 1);
        float f = 1.0f;
        if (g.sa.mode != TI8_SCALE_ROW) f = g.sa.p[idx::gemm_factor_index(batch, g.sa.bs, idx::gemm_factor_block(m0, g.M), g.sa.rs, kt, g.sa.mode == TI8_SCALE_BLOCK_K256 ? 1 : 0, g.sa.ks)];
        if (g.sb.mode != TI8_SCALE_ROW) f = f * g.sb.p[idx::gemm_factor_index(batch, g.sb.bs, idx::gemm_factor_block(n0, g.N), g.sb.rs, kt, g.sb.mode == TI8_SCALE_BLOCK_K256 ? 1 : 0, g.sb.ks)];
        if (divide) f = 1.0f / f;
        factors[threadIdx.x] = f;
    }
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int q = 0; q < 2 * INSTR; ++q) issue_one(t, t, q);

    // ---- LDS -> registers ------------------------------------------------------------------
    // addresses of the first two stages and, 64 KiB on (past the reach of an instruction's offset), of the last two
    const int fr_row = lane & 31, fr_half = lane >> 5;
    const int sw = (lane & 7) ^ ((lane >> 3) & 1);
    uint32_t abase[2][4], bbase[2][4];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const int choff = ((ks * 2 + fr_half) ^ sw) * 16;
            abase[h][ks] = (uint32_t)(2 * h * STAGE_BYTES + ((wm * 2 + grp) * 32 + fr_row) * 128 + choff);
            bbase[h][ks] = (uint32_t)(2 * h * STAGE_BYTES + A_BYTES + (wn * TN * 32 + fr_row) * 128 + choff);
            asm volatile("" : "+v"(abase[h][ks]), "+v"(bbase[h][ks]));
        }

    const v16i vzero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    v16i acc[I32 ? 1 : 2][TN];           // I32: the sums; else the products of the last two K tiles, by parity
    float accf[I32 ? 1 : TN][16];
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[0][j] = acc[I32 ? 0 : 1][j] = vzero;
#pragma unroll
    for (int j = 0; j < (I32 ? 1 : TN); ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) accf[j][r] = 0.0f;

    v4i fa[4], fb[TN][4];
    // instruction q (of 12) of a K tile's fragment reads
    auto read_one = [&](int stage, int q) {
        const int ks = q / 3, b = q % 3, h = stage >> 1, off = (stage & 1) * STAGE_BYTES;
        if (b == 0) fa[ks] = *reinterpret_cast<const v4i*>(smem + abase[h][ks] + off);
        else fb[b - 1][ks] = *reinterpret_cast<const v4i*>(smem + bbase[h][ks] + (off + (b - 1) * 4096));
    };
    // the fragments are in registers HERE: without this the optimiser may move the reads behind the wait, to where the
    // fragments are used, past the point at which their buffer is given back
    auto frags_landed = [&]() {
        __builtin_amdgcn_s_waitcnt(WAIT_LDS);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) asm volatile("" : "+v"(fa[ks]), "+v"(fb[0][ks]), "+v"(fb[1][ks])::"memory");
    };
    // MFMA ks (of 4) of block j into product set p; piece q (of 8) of folding its block j in
    auto mfma = [&](int p, int j, int ks) {
        acc[I32 ? 0 : p][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[ks], fb[j][ks], (!I32 && ks == 0) ? vzero : acc[I32 ? 0 : p][j], 0, 0, 0);
    };
    auto fold = [&](int p, int j, int q, float f) {
        if (I32) return;
#pragma unroll
        for (int r = q * 2; r < q * 2 + 2; ++r) accf[I32 ? 0 : j][r] = __builtin_fmaf(static_cast<float>(acc[I32 ? 0 : p][j][r]), f, accf[I32 ? 0 : j][r]);
    };
    float f_cur = 0.0f, f_next = 0.0f;      // factor of the K tile whose products are being folded; the one read last
    auto read_factor = [&](int t) {
        if (!I32) f_next = factors[min(t, MAX_K_TILES - 1)];
    };
    // Phase M of K tile t (its fragments are in registers): the products.  Phase F behind it: the fragments of tile t + 1.  Both
    // groups fetch the same K tile at the same time, group 0 in its M and group 1 in its F, into the stage that both are past;
    // at the end of that phase all but the youngest two tiles have landed, among them the one that group 0 reads next.
    auto phase_m = [&](auto grp_tag, auto stage_tag, int t) {
        constexpr int STAGE = decltype(stage_tag)::value, P = STAGE & 1;
        constexpr bool FETCH = decltype(grp_tag)::value == 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            __builtin_amdgcn_sched_barrier(0);
            mfma(P, q & 1, q >> 1);
            __builtin_amdgcn_sched_barrier(0);
            fold(P ^ 1, 1, q, f_cur);
            if (FETCH && (q & 1)) issue_one(t + 3, (STAGE + 3) % STAGES, q >> 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        f_cur = f_next;
        if (FETCH) __builtin_amdgcn_s_waitcnt(WAIT_ALL_BUT_TWO_TILES);
    };
    auto phase_f = [&](auto grp_tag, auto stage_tag, int t) {
        constexpr int STAGE = decltype(stage_tag)::value, P = STAGE & 1;
        constexpr bool FETCH = decltype(grp_tag)::value == 1;
        read_factor(t + 1);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < 3; ++k) read_one((STAGE + 1) % STAGES, 3 * q + k);
            __builtin_amdgcn_sched_barrier(0);
            if (FETCH) issue_one(t + 4, STAGE, q);
            fold(P, 0, 2 * q, f_cur);
            fold(P, 0, 2 * q + 1, f_cur);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (FETCH) __builtin_amdgcn_s_waitcnt(WAIT_ALL_BUT_TWO_TILES);
        frags_landed();
    };
    // the barrier is written out: in front of the one it knows the compiler waits for every load in flight
    auto barrier = [&]() { asm volatile("s_barrier" ::: "memory"); };
    auto k_tile = [&](auto grp_tag, auto stage_tag, int t) {
        barrier();
        phase_m(grp_tag, stage_tag, t);
        barrier();
        phase_f(grp_tag, stage_tag, t);
    };
    using G0 = std::integral_constant<int, 0>;
    using G1 = std::integral_constant<int, 1>;
    auto k_loop = [&](auto grp_tag) {
        int t = 0;
        for (; t + 4 <= nk; t += 4) {
            k_tile(grp_tag, std::integral_constant<int, 0>{}, t);
            k_tile(grp_tag, std::integral_constant<int, 1>{}, t + 1);
            k_tile(grp_tag, std::integral_constant<int, 2>{}, t + 2);
            k_tile(grp_tag, std::integral_constant<int, 3>{}, t + 3);
        }
        if (t < nk) k_tile(grp_tag, std::integral_constant<int, 0>{}, t);
        if (t + 1 < nk) k_tile(grp_tag, std::integral_constant<int, 1>{}, t + 1);
        if (t + 2 < nk) k_tile(grp_tag, std::integral_constant<int, 2>{}, t + 2);
    };

    // ---- K loop --------------------------------------------------------------------------------
    __builtin_amdgcn_s_waitcnt(WAIT_LDS & WAIT_ALL_BUT_TWO_TILES);      // tile 0 and the factors
    barrier();
#pragma unroll
    for (int q = 0; q < 12; ++q) read_one(0, q);
    read_factor(0);
    if (grp == 0) {
        frags_landed();
        k_loop(G0{});
        barrier();                      // both groups have met the same number of barriers
    } else {                            // half a K tile behind group 0
#pragma unroll
        for (int q = 0; q < 2 * INSTR; ++q) issue_one(3, 3, q);
        __builtin_amdgcn_s_waitcnt(WAIT_ALL_BUT_TWO_TILES);
        frags_landed();
        barrier();
        k_loop(G1{});
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        if (nk & 1) fold(0, 1, q, f_cur);
        else fold(1, 1, q, f_cur);
    }

    // ---- epilogue: 32 rows x 64 columns per wave, 8 columns per lane ----
    const int e_row0 = m0 + (wm * 2 + grp) * 32;
    const int rb_col = idx::epi_col_of_lane(lane, WCOLS), rb_row = idx::epi_row_of_lane(lane, WCOLS);
    const bool row_part = I32 || g.sa.mode == TI8_SCALE_ROW, col_part = I32 || g.sb.mode == TI8_SCALE_ROW;
    float rowm[4], coln[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        float v = g.sa.p[idx::epi_row_scale_base(batch, g.sa.bs, min(e_row0 + rb_row + 8 * k, g.M - 1), row_part ? g.sa.rs : 0)];
        v = row_part ? v : 1.0f;        // an absent scale vector multiplies by 1 (exact)
        rowm[k] = divide ? 1.0f / v : v;
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        float v = g.sb.p[idx::epi_col_scale_index(batch, g.sb.bs, n0 + wn * WCOLS + rb_col + c, g.N, col_part ? g.sb.rs : 0)];
        v = col_part ? v : 1.0f;
        coln[c] = divide ? 1.0f / v : v;
    }
    uint4 bias = make_uint4(0, 0, 0, 0);
    if (g.bias) bias = *reinterpret_cast<const uint4*>(g.bias + n0 + wn * WCOLS + rb_col);
    // every load has landed and every wave is past its last fragment read: the buffers become the waves' slabs
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    uint32_t* const slab = reinterpret_cast<uint32_t*>(smem) + wave * (32 * SLAB_LD);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int rr = 8 * (r >> 2) + 4 * fr_half + (r & 3);
            slab[rr * SLAB_LD + j * 32 + fr_row] = I32 ? static_cast<uint32_t>(acc[0][j][r]) : __float_as_uint(accf[I32 ? 0 : j][r]);
        }
    __builtin_amdgcn_s_waitcnt(WAIT_LDS);   // the wave reads back what it wrote itself
    __builtin_amdgcn_wave_barrier();
    if (e_row0 >= g.M) return;              // M is a multiple of 32: a wave's 32 rows are all inside or all outside
    uint16_t* dst = reinterpret_cast<uint16_t*>(g.C) + idx::epi_out_offset(batch, g.bsc, e_row0 + rb_row, g.ldc, n0 + wn * WCOLS + rb_col);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t* src = slab + (rb_row + 8 * k) * SLAB_LD + rb_col;
        const uint4 lo = *reinterpret_cast<const uint4*>(src), hi = *reinterpret_cast<const uint4*>(src + 4);
        const uint32_t wb[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        float v[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            v[c] = (I32 ? static_cast<float>(static_cast<int32_t>(wb[c])) : __uint_as_float(wb[c])) * rowm[k];
            v[c] = v[c] * coln[c];
            if (!I32) v[c] = v[c] * g.out_scale;
        }
        if (I32 && g.post_scale != 0.0f) {
#pragma unroll
            for (int c = 0; c < 8; ++c) v[c] = __uint_as_float(pack_bf16x2(v[c], 0.0f) << 16) * g.post_scale;
        }
        uint16_t* const row = dst + (int64_t)(8 * k) * g.ldc;
        uint4 o = make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
        if (g.bias) o = make_uint4(add_bf16x2(o.x, bias.x), add_bf16x2(o.y, bias.y), add_bf16x2(o.z, bias.z), add_bf16x2(o.w, bias.w));
        *reinterpret_cast<uint2*>(row) = make_uint2(o.x, o.y);
        *reinterpret_cast<uint2*>(row + 4) = make_uint2(o.z, o.w);
    }
}

int init_mid_kernels() {
    static OncePerDevice once_i32, once_promote;
    hipError_t e = raise_lds_limit(once_i32, reinterpret_cast<const void*>(gemm_i8_mid_kernel<true>), LDS_BYTES);
    if (e == hipSuccess) e = raise_lds_limit(once_promote, reinterpret_cast<const void*>(gemm_i8_mid_kernel<false>), LDS_BYTES);
    if (e != hipSuccess) return fail(TI8_ERR_HIP, "gemm: cannot raise the LDS limit to %d: %s", LDS_BYTES, hipGetErrorString(e));
    return TI8_OK;
}

int launch_mid(GemmMulti& m, int64_t batch, bool i32_full, hipStream_t st) {
    if (int e = init_mid_kernels()) return e;
    int total = 0;
    for (int i = 0; i < m.count; ++i) {
        m.g[i].tiles_m = (m.g[i].M + BM - 1) / BM;
        m.g[i].tiles_n = m.g[i].N / BN;
        m.first[i] = total;
        total += m.g[i].tiles_m * m.g[i].tiles_n;
    }
    for (int i = m.count; i <= GEMM_MULTI_MAX; ++i) m.first[i] = total;
    for (int i = m.count; i < GEMM_MULTI_MAX; ++i) m.g[i] = m.g[0];
    const dim3 grid((unsigned)total, (unsigned)batch), block(64 * NW);
    if (i32_full) hipLaunchKernelGGL(gemm_i8_mid_kernel<true>, grid, block, LDS_BYTES, st, m);
    else hipLaunchKernelGGL(gemm_i8_mid_kernel<false>, grid, block, LDS_BYTES, st, m);
    note_gemm_kernel(TI8_KERNEL_MID, BM, BN, i32_full ? EPI_ROWS : EPI_PROMOTE_CHAIN);
    return check_launch("ti8_gemm_i8_nt");
}

}  // namespace ti8
