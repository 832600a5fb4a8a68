// INT8 NT GEMM for medium sizes: 128 x 128 tiles, two K tiles at a time on two groups of four waves.
//
// Up to one 128 x 128 tile per CU the time of a GEMM is the time ONE workgroup takes for its K loop, and the tile on four
// waves (gemm.hip, one wave per SIMD) spends that loop waiting: load -> barrier -> LDS read -> MFMA -> convert + fma, one
// after the other, 1.0 us per K tile where the MFMAs take 0.22.  Here group g of a workgroup's eight waves takes the K
// tiles of parity g, each wave a 64 x 64 quarter of the tile with its own accumulators: every SIMD holds two waves, and a K
// tile costs no more LDS reads or convert + fma than on four waves (eight smaller quarters would read half again as much).
//
//  * The groups run half a step apart.  Phase M: the products of a K tile whose fragments are in registers, the previous
//    tile's second block row folded between the MFMAs of the first (8 vector instructions per MFMA), the loads of the tile
//    after the next one per MFMA of the second.  Phase F: the next tile's fragments out of LDS, the first block row folded
//    between the reads.  While one group is in M the other is in F, so that MFMAs, vector instructions, LDS reads and loads
//    run at the same time; ONE barrier per phase.  (Both groups in step: 10 % slower.  Everything folded in F: 19 % slower,
//    a single wave per SIMD issues a vector instruction every 7 cycles only, two waves one every 4.)
//  * All fragments of a K tile are read in one phase, so its LDS buffer is free for three phases: a load has one and a half
//    steps to land, and two K tiles per group (64 to 128 KiB per CU) are in flight.
//  * The order inside the phases is written out between scheduling barriers: left to itself the compiler gathers the
//    conversions in front and spills.
//  * The sums of the two groups meet once, in LDS, behind the loop: each wave hands over one of its two block rows and
//    finishes the other.
//
// What bounds it: 64 KiB per step and CU from L2 into LDS (alone 0.66 us of the 1.15 us that a step takes with all CUs
// busy) in the LDS that 128 KiB of fragments are read from, beside 1024 cycles of MFMA per SIMD.  1024 rows, K = 14336, N =
// 4096: promotion 75.5 us = 1.59 POP/s (four waves: 109), int32 63.9 us (73.8); K = 4096: 28 us (33.6).
//
// Arithmetic: the int32 path (I32) is exact and bit-identical to the other kernels; the promotion adds the K tiles of each
// parity in order and then the two sums (fp32 association only, no rounding more).
#include <type_traits>
#include "gemm_args.h"

namespace ti8 {

namespace {

constexpr int BM = 128, BN = 128, NGROUP = 2, WN = 2, NW = 8;
constexpr int TM = 2, TN = 2;                       // 32 x 32 blocks per wave
constexpr int WCOLS = TN * 32;
constexpr int INSTR = 4;                            // global -> LDS instructions per wave, operand and K tile (32 rows)
constexpr int A_BYTES = BM * 128;
constexpr int STAGE_BYTES = A_BYTES + BN * 128;     // one K tile of both operands
constexpr int GROUP_BYTES = 2 * STAGE_BYTES;        // double buffered, per group
constexpr int MAX_K_TILES = 256;
constexpr int LDS_BYTES = NGROUP * GROUP_BYTES + MAX_K_TILES * 4;   // 128 KiB of operands, one factor per K tile
// vmcnt(2 * INSTR): all but the youngest K tile's loads of this wave
constexpr int WAIT_ALL_BUT_ONE_TILE = 0xf70 | (2 * INSTR);
static_assert(2 * INSTR < 16, "vmcnt[3:0]");
constexpr int WAIT_LDS = 0xc07f;                    // lgkmcnt(0)
constexpr int SLAB_LD = idx::EPI_SLAB_LD(WCOLS);    // words per row of a wave's 32 x 64 slab
static_assert(NW * 32 * SLAB_LD * 4 <= NGROUP * GROUP_BYTES, "the exchange slabs lie over the operand buffers");

}  // namespace

template <bool I32>
__global__ __launch_bounds__(64 * NW) void gemm_i8_mid_kernel(const GemmMulti m) {
    extern __shared__ __attribute__((aligned(1024))) int8_t smem[];
    // layout: [group][buffer][A 16 KiB][B 16 KiB], then the factors

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = wave >> 2, quarter = wave & 3;
    const int wm = quarter / WN, wn = quarter % WN;
    const int gi = idx::gemm_multi_pick((int)blockIdx.x, m.first[1], m.first[2], m.count);
    const GemmArgs& g = m.g[gi];
    const int batch = blockIdx.y;
    const idx::TileCoord tc = idx::gemm_tile_of((int)blockIdx.x - m.first[gi], g.tiles_m, g.tiles_n, idx::gemm_group_rows(BM));
    const int m0 = tc.tile_m * BM, n0 = tc.tile_n * BN;
    const int nk = g.K >> 7;

    // ---- global -> LDS: the slab layout and swizzle of the other kernels (gemm.hip) -----------
    uint32_t voffA[2], voffB[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        voffA[p] = idx::gemm_lane_offset_bytes(lane, p, (int)g.lda);
        voffB[p] = idx::gemm_lane_offset_bytes(lane, p, (int)g.ldb);
    }
    const int8_t* const baseA = g.A + (int64_t)batch * g.bsa + (int64_t)idx::gemm_mid_first_row(m0, quarter, g.M) * g.lda;
    const int8_t* const baseB = g.B + (int64_t)batch * g.bsb + (int64_t)idx::gemm_mid_first_row(n0, quarter, g.N) * g.ldb;
    const int64_t strideA8 = 8 * g.lda, strideB8 = 8 * g.ldb;
    int8_t* const wdst = smem + grp * GROUP_BYTES + quarter * INSTR * 1024;
    // byte offset along K of this group's tile t; past the end (the odd group's last step when nk is odd, and the loads that
    // run ahead) the last K tile is fetched again, into a buffer whose products are dropped or never made
    auto k_offset = [&](int t) { return min(2 * t + grp, nk - 1) * 128; };
    auto issue = [&](int t, int buf) {
        issue_tile_loads<INSTR>(baseA + k_offset(t), strideA8, voffA, 0, wdst + buf * STAGE_BYTES);
        issue_tile_loads<INSTR>(baseB + k_offset(t), strideB8, voffB, 0, wdst + buf * STAGE_BYTES + A_BYTES);
    };
    issue(0, 0);

    // ---- LDS -> registers ------------------------------------------------------------------
    const int fr_row = lane & 31, fr_half = lane >> 5;
    const int sw = (lane & 7) ^ ((lane >> 3) & 1);
    uint32_t abase[4], bbase[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const int choff = ((ks * 2 + fr_half) ^ sw) * 16;
        abase[ks] = (uint32_t)(grp * GROUP_BYTES + (wm * TM * 32 + fr_row) * 128 + choff);
        bbase[ks] = (uint32_t)(grp * GROUP_BYTES + A_BYTES + (wn * TN * 32 + fr_row) * 128 + choff);
        asm volatile("" : "+v"(abase[ks]), "+v"(bbase[ks]));
    }

    // ---- per-K-tile factors of the promotion: f_kt = fa_kt * fb_kt (an operand scaled per row contributes its vector in the
    // epilogue instead), the same for the whole tile, through LDS
    const bool divide = !I32 && g.combine == TI8_COMBINE_DIV_PROD;
    float* const factors = reinterpret_cast<float*>(smem + NGROUP * GROUP_BYTES);
    if (!I32 && threadIdx.x < MAX_K_TILES) {
        const int kt = min((int)threadIdx.x, nk - 1);
        float f = 1.0f;
        if (g.sa.mode != TI8_SCALE_ROW) f = g.sa.p[idx::gemm_factor_index(batch, g.sa.bs, idx::gemm_factor_block(m0, g.M), g.sa.rs, kt, g.sa.mode == TI8_SCALE_BLOCK_K256 ? 1 : 0, g.sa.ks)];
        if (g.sb.mode != TI8_SCALE_ROW) f = f * g.sb.p[idx::gemm_factor_index(batch, g.sb.bs, idx::gemm_factor_block(n0, g.N), g.sb.rs, kt, g.sb.mode == TI8_SCALE_BLOCK_K256 ? 1 : 0, g.sb.ks)];
        if (divide) f = 1.0f / f;
        factors[threadIdx.x] = f;
    }

    const v16i vzero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    v16i acc[TM][TN];       // I32: the sums; else the products of the K tile at hand
    float accf[I32 ? 1 : TM][I32 ? 1 : TN][16];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = vzero;
#pragma unroll
    for (int i = 0; i < (I32 ? 1 : TM); ++i)
#pragma unroll
        for (int j = 0; j < (I32 ? 1 : TN); ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) accf[i][j][r] = 0.0f;

    v4i fa[TM][4], fb[TN][4];
    // instruction pair q (of 8) of a K tile's fragment reads
    auto read_pair = [&](int buf, int q) {
        const int ks = q >> 1, b = q & 1;
        fa[b][ks] = *reinterpret_cast<const v4i*>(smem + abase[ks] + (buf * STAGE_BYTES + b * 4096));
        fb[b][ks] = *reinterpret_cast<const v4i*>(smem + bbase[ks] + (buf * STAGE_BYTES + b * 4096));
    };
    // the fragments are in registers HERE: without this the optimiser may move the reads behind the wait, to where the
    // fragments are used, past the point at which their buffer is given back
    auto frags_landed = [&]() {
        __builtin_amdgcn_s_waitcnt(WAIT_LDS);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) asm volatile("" : "+v"(fa[0][ks]), "+v"(fa[1][ks]), "+v"(fb[0][ks]), "+v"(fb[1][ks])::"memory");
    };
    // MFMA q (of 8) of block row i; piece q (of 8) of folding block row i in
    auto mfma = [&](int i, int q) {
        const int ks = q >> 1, j = q & 1;
        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i][ks], fb[j][ks], (!I32 && ks == 0) ? vzero : acc[i][j], 0, 0, 0);
    };
    auto fold = [&](int i, int q, float f) {
        if (I32) return;
        const int j = q >> 2;
#pragma unroll
        for (int r = (q & 3) * 4; r < (q & 3) * 4 + 4; ++r)
            accf[I32 ? 0 : i][I32 ? 0 : j][r] = __builtin_fmaf(static_cast<float>(acc[i][j][r]), f, accf[I32 ? 0 : i][I32 ? 0 : j][r]);
    };
    float f_cur = 0.0f, f_next = 0.0f;      // factor of the K tile whose products are in acc; the one read last
    auto read_factor = [&](int t) {
        if (!I32) f_next = factors[min(2 * t + grp, MAX_K_TILES - 1)];
    };
    // phase M of K tile `t` of this group (its fragments are in registers, its LDS buffer BUF is free again): the products,
    // the loads of tile t + 2; at the end tile t + 1 (all but the 8 youngest loads) has landed
    auto phase_m = [&](auto buf_tag, int t) {
        constexpr int BUF = decltype(buf_tag)::value;
        const bool live = 2 * t + grp < nk;     // wave-uniform
        if (!I32 || live) {                     // a promoted tile past the end is dropped by its factor instead
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                __builtin_amdgcn_sched_barrier(0);
                mfma(0, q);
                __builtin_amdgcn_sched_barrier(0);
                fold(1, q, f_cur);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (!I32) f_cur = live ? f_next : 0.0f;
        const int8_t* const pA = baseA + k_offset(t + 2);
        const int8_t* const pB = baseB + k_offset(t + 2);
        int8_t* const dst = wdst + BUF * STAGE_BYTES;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            __builtin_amdgcn_sched_barrier(0);
            if (!I32 || live) mfma(1, q);
            if (q < INSTR) issue_tile_loads<1>(pA + q * strideA8, strideA8, voffA, q, dst + q * 1024);
            else issue_tile_loads<1>(pB + (q - INSTR) * strideB8, strideB8, voffB, q, dst + A_BYTES + (q - INSTR) * 1024);
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(WAIT_ALL_BUT_ONE_TILE);
    };
    // phase F behind it: the fragments of tile t + 1 out of buffer BUF ^ 1
    auto phase_f = [&](auto buf_tag, int t) {
        constexpr int BUF = decltype(buf_tag)::value;
        read_factor(t + 1);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            __builtin_amdgcn_sched_barrier(0);
            read_pair(BUF ^ 1, q);
            __builtin_amdgcn_sched_barrier(0);
            fold(0, q, f_cur);
        }
        __builtin_amdgcn_sched_barrier(0);
        frags_landed();
    };
    // the barrier is written out: in front of the one it knows the compiler waits for every load in flight
    auto barrier = [&]() { asm volatile("s_barrier" ::: "memory"); };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;

    // ---- K loop --------------------------------------------------------------------------------
    const int steps = (nk + 1) >> 1;
    __builtin_amdgcn_s_waitcnt(0);      // tile 0 and the factors
    __syncthreads();
    issue(1, 1);
#pragma unroll
    for (int q = 0; q < 8; ++q) read_pair(0, q);
    read_factor(0);
    frags_landed();
    if (grp == 1) barrier();            // half a step behind group 0 from here on
    int t = 0;
    for (; t + 1 < steps; t += 2) {     // (one exit at the end: with a second one in the middle the accumulators are copied)
        barrier();
        phase_m(B0{}, t);
        barrier();
        phase_f(B0{}, t);
        barrier();
        phase_m(B1{}, t + 1);
        barrier();
        phase_f(B1{}, t + 1);
    }
    if (t < steps) {
        barrier();
        phase_m(B0{}, t);
        barrier();
        phase_f(B0{}, t);
    }
    if (grp == 0) barrier();            // both groups have met the same number of barriers
#pragma unroll
    for (int q = 0; q < 8; ++q) fold(1, q, f_cur);

    // ---- epilogue: what this wave finishes is block row `grp` of its quarter, 32 rows x 64 columns, 8 columns per lane ----
    const int e_row0 = m0 + wm * TM * 32 + grp * 32;
    const int rb_col = idx::epi_col_of_lane(lane, WCOLS), rb_row = idx::epi_row_of_lane(lane, WCOLS);
    const bool row_part = I32 || g.sa.mode == TI8_SCALE_ROW, col_part = I32 || g.sb.mode == TI8_SCALE_ROW;
    // (scale loads behind the loop: 12 registers that the loop has no room for)
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
    // every load has landed and every wave is past its last fragment read: the buffers become exchange slabs
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    // wave (grp, quarter) puts block row 1 - grp into its slab and adds to its block row `grp` what the partner wave put
    // there for it
    uint32_t* const slab = reinterpret_cast<uint32_t*>(smem) + wave * (32 * SLAB_LD);
    auto put = [&](int i) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int rr = 8 * (r >> 2) + 4 * fr_half + (r & 3);
                slab[rr * SLAB_LD + j * 32 + fr_row] = I32 ? static_cast<uint32_t>(acc[i][j][r]) : __float_as_uint(accf[I32 ? 0 : i][I32 ? 0 : j][r]);
            }
    };
    if (grp == 0) put(1);
    else put(0);
    __syncthreads();
    const uint32_t* const other = reinterpret_cast<const uint32_t*>(smem) + (wave ^ 4) * (32 * SLAB_LD);
    uint32_t theirs[TN][16];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) theirs[j][r] = other[(8 * (r >> 2) + 4 * fr_half + (r & 3)) * SLAB_LD + j * 32 + fr_row];
    __syncthreads();
    auto sum_into_slab = [&](int i) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int rr = 8 * (r >> 2) + 4 * fr_half + (r & 3);
                uint32_t w;
                if (I32) w = static_cast<uint32_t>(acc[i][j][r]) + theirs[j][r];
                else w = __float_as_uint(accf[I32 ? 0 : i][I32 ? 0 : j][r] + __uint_as_float(theirs[j][r]));
                slab[rr * SLAB_LD + j * 32 + fr_row] = w;
            }
    };
    if (grp == 0) sum_into_slab(0);
    else sum_into_slab(1);
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
