// INT8 NT GEMM for few rows (decode-like shapes: up to 256 rows, in steps of 32).
//
// With so few rows the tiled kernel of gemm.hip has only N/128 workgroups, and each walks the
// whole K behind a two-stage LDS pipeline: its time is load latency, not MFMA.  Here C is cut
// into 32 x 32 blocks, one per workgroup, (N/32) * (M/32) of them, and K is split over the four
// waves of the workgroup, each of which runs its own load -> LDS -> MFMA pipeline with no
// barrier in the loop.
//
// The arithmetic and the epilogue are those of the tiled kernel's int32 and fast-promotion paths,
// operation for operation; only the order in which K tiles are added differs (four partial sums
// per output, K tiles walked from a workgroup-dependent start).  The int32 path is therefore
// bit-identical to the tiled kernel, the promoted path differs by fp32 association only.
#include "gemm_args.h"

namespace ti8 {

// s_waitcnt vmcnt(n) (gfx9 encoding: vmcnt in bits 3:0 and 15:14) and lgkmcnt(0) (bits 11:8),
// expcnt untouched (bits 6:4)
#define TI8_WAIT_VMCNT_LGKM0(n) __builtin_amdgcn_s_waitcnt(((n) & 0xf) | (((n) >> 4) << 14) | 0x0070)

// A workgroup owns 32 x 32 of C and its four waves split K into quarters.  Every wave streams ITS
// quarter of both operands through a private LDS ring (WS_STAGES stages of [A 32 rows][B 32 rows]
// = 8 KiB, filled by global_load_lds in the swizzled layout of the tiled kernel), waits only
// for its own loads and never for another wave; the four partial results meet in LDS at the end
// and are added in the fixed order q0 + q1 + q2 + q3 (int32: exact; fp32: deterministic).
// Independent streams hide the per-tile latency chain (load -> LDS -> MFMA -> convert) that one
// stream per workgroup behind a barrier exposes: a version with 64 x 32 blocks, an 8-stage ring
// shared by the workgroup and one barrier per K tile took 14.4 us where this one takes 11.2 us
// (128 rows, K = N = 4096).  Two stages = 64 KiB per workgroup, so two workgroups share a CU.
constexpr int WS_STAGES = 2;
constexpr int WS_STAGE_BYTES = 2 * 32 * 128;
constexpr int WS_LOADS = 8;  // global->LDS instructions per wave and stage

// `block_x` = index of the workgroup among the blocks of this GEMM and batch.
template <bool I32FULL>
__device__ __forceinline__ void wavering_block(const GemmArgs& g, const int block_x, const int batch) {
    extern __shared__ __attribute__((aligned(1024))) int8_t smem[];  // 4 waves x WS_STAGES x 8 KiB

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int mtiles = g.M >> 5, nstrips = g.N >> 5;
    int strip, mt;
    if ((nstrips & 7) == 0) {   // workgroups that share a strip of B on one XCD (ids 8 apart)
        const int xcd = block_x & 7, idx = block_x >> 3;
        strip = (idx / mtiles) * 8 + xcd;
        mt = idx % mtiles;
    } else {
        strip = block_x / mtiles;
        mt = block_x % mtiles;
    }
    const int n0 = strip * 32, m0 = mt * 32;
    const int nk = g.K >> 7;
    const int kbeg = (wave * nk) >> 2, kend = ((wave + 1) * nk) >> 2;
    const int nq = kend - kbeg;

    // ---- global -> LDS (same slab layout and swizzle as the other kernels): 4 instructions of A
    // (rows 8i .. 8i+7) and 4 of B per stage, all issued by the wave that consumes them
    const int ld_row = lane >> 3;
    uint32_t voffA[2], voffB[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int ch = (lane & 7) ^ ld_row ^ p;
        voffA[p] = (uint32_t)(ld_row * (int)g.lda + ch * 16);
        voffB[p] = (uint32_t)(ld_row * (int)g.ldb + ch * 16);
    }
    const int8_t* baseA = g.A + (int64_t)batch * g.bsa + (int64_t)m0 * g.lda;
    const int8_t* baseB = g.B + (int64_t)batch * g.bsb + (int64_t)n0 * g.ldb;
    const int64_t strideA8 = 8 * g.lda, strideB8 = 8 * g.ldb;
    int8_t* const ring = smem + wave * (WS_STAGES * WS_STAGE_BYTES);
    // step i of this wave's walk is K tile kbeg + (i + rot) mod nq: workgroups start at different
    // tiles so that they do not ask the same memory channels for their lines at the same time
    const int rot = nq > 0 ? (int)((((unsigned)block_x >> 3) * 3u + (unsigned)batch) % (unsigned)nq) : 0;
    auto tile_of_step = [&](int i) {
        int j = min(i, max(nq - 1, 0)) + rot;   // past the end: the last one again, into a free stage
        if (j >= nq) j -= nq;
        return min(kbeg + max(j, 0), nk - 1);
    };
    auto issue_stage = [&](int i) {
        int8_t* st = ring + (i & (WS_STAGES - 1)) * WS_STAGE_BYTES;
        const int koff = tile_of_step(i) * 128;
        issue_tile_loads<4>(baseA + koff, strideA8, voffA, 0, st);
        issue_tile_loads<4>(baseB + koff, strideB8, voffB, 0, st + 4096);
    };

    // ---- scales: unconditional loads (an operand that contributes no in-loop factor is read with
    // stride 0 and dropped; a load under a branch would be waited for on the spot), issued before
    // the tile loads
    const bool divide = !I32FULL && g.combine == TI8_COMBINE_DIV_PROD;
    const bool a_in = !I32FULL && g.sa.mode != TI8_SCALE_ROW, b_in = !I32FULL && g.sb.mode != TI8_SCALE_ROW;
    float fvec[4] = {1.0f, 1.0f, 1.0f, 1.0f};
    if (!I32FULL) {
        const int sha = g.sa.mode == TI8_SCALE_BLOCK_K256 ? 1 : 0, shb = g.sb.mode == TI8_SCALE_BLOCK_K256 ? 1 : 0;
        const float* pa = g.sa.p + (int64_t)batch * g.sa.bs + (a_in ? (int64_t)(m0 >> 7) * g.sa.rs : 0);
        const float* pb = g.sb.p + (int64_t)batch * g.sb.bs + (b_in ? (int64_t)(n0 >> 7) * g.sb.rs : 0);
        const int64_t ska = a_in ? g.sa.ks : 0, skb = b_in ? g.sb.ks : 0;
        float fa[4], fb[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int kt = min(c * 64 + lane, nk - 1);
            fa[c] = pa[(int64_t)(kt >> sha) * ska];
            fb[c] = pb[(int64_t)(kt >> shb) * skb];
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float f = (a_in ? fa[c] : 1.0f) * (b_in ? fb[c] : 1.0f);
            if (divide) f = 1.0f / f;
            fvec[c] = f;
        }
    }
    // epilogue scales of the 4 outputs this thread will finish: row t/8, columns 4*(t%8) .. +3
    const int e_row = threadIdx.x >> 3, e_col = (threadIdx.x & 7) * 4;
    const bool row_part = I32FULL || g.sa.mode == TI8_SCALE_ROW, col_part = I32FULL || g.sb.mode == TI8_SCALE_ROW;
    float rowm = g.sa.p[(int64_t)batch * g.sa.bs + (row_part ? (int64_t)(m0 + e_row) * g.sa.rs : 0)];
    float coln[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) coln[c] = g.sb.p[(int64_t)batch * g.sb.bs + (col_part ? (int64_t)(n0 + e_col + c) * g.sb.rs : 0)];
    if (divide) {
        rowm = 1.0f / rowm;
#pragma unroll
        for (int c = 0; c < 4; ++c) coln[c] = 1.0f / coln[c];
    }

    // the bias of those 4 columns (without one: 8 bytes of B, dropped)
    const uint2 bias = *reinterpret_cast<const uint2*>(g.bias ? reinterpret_cast<const void*>(g.bias + n0 + e_col) : reinterpret_cast<const void*>(g.B));

    const int fr_row = lane & 31, fr_half = lane >> 5;
    const int sw = (lane & 7) ^ ((lane >> 3) & 1);
    int choff[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) choff[ks] = ((ks * 2 + fr_half) ^ sw) * 16;
    const int a_off = fr_row * 128, b_off = 4096 + fr_row * 128;

    const v16i vzero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    v16i acc = vzero;
    float accf[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) accf[i] = 0.0f;

#pragma unroll
    for (int s = 0; s < WS_STAGES - 1; ++s) issue_stage(s);
    // pin the scale vectors to registers here (they are older than the tile loads, so this waits
    // for nothing else): a load still pending at the loop's entry makes the compiler drain the
    // whole load queue at the top of every iteration
    asm volatile("" : "+v"(rowm));
    uint32_t bias_lo = bias.x, bias_hi = bias.y;
    asm volatile("" : "+v"(bias_lo), "+v"(bias_hi));
#pragma unroll
    for (int c = 0; c < 4; ++c) asm volatile("" : "+v"(coln[c]));

    auto factor_of_step = [&](int i) -> float {
        const int kt = tile_of_step(i);
        const int l = kt & 63, c = kt >> 6;
        const float v0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fvec[0]), l));
        const float v1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fvec[1]), l));
        const float v2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fvec[2]), l));
        const float v3 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fvec[3]), l));
        return c == 0 ? v0 : (c == 1 ? v1 : (c == 2 ? v2 : v3));
    };
    v16i d = vzero;
    float f_prev = 0.0f;
    for (int i = 0; i < nq; ++i) {
        // own loads of step i landed (at most the WS_STAGES - 2 younger steps outstanding); own
        // LDS reads of step i - 1 returned, so its stage can be refilled.  No barrier: nobody
        // else touches this wave's ring.
        TI8_WAIT_VMCNT_LGKM0((WS_STAGES - 2) * WS_LOADS);
        issue_stage(i + WS_STAGES - 1);
        const int8_t* st = ring + (i & (WS_STAGES - 1)) * WS_STAGE_BYTES;
        v4i fa[4], fb[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            fa[ks] = *reinterpret_cast<const v4i*>(st + a_off + choff[ks]);
            fb[ks] = *reinterpret_cast<const v4i*>(st + b_off + choff[ks]);
        }
        __builtin_amdgcn_sched_barrier(0);   // all eight reads go out before anything else
        if (I32FULL) {
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[ks], fb[ks], acc, 0, 0, 0);
        } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) accf[r] = __builtin_fmaf(static_cast<float>(d[r]), f_prev, accf[r]);
            __builtin_amdgcn_sched_barrier(0);
            d = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[0], fb[0], vzero, 0, 0, 0);
#pragma unroll
            for (int ks = 1; ks < 4; ++ks) d = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[ks], fb[ks], d, 0, 0, 0);
            f_prev = factor_of_step(i);
        }
    }
    if (!I32FULL) {
#pragma unroll
        for (int r = 0; r < 16; ++r) accf[r] = __builtin_fmaf(static_cast<float>(d[r]), f_prev, accf[r]);
    }
    // every load (the redundant ones of the last steps included) has landed and every wave is
    // done with its ring before the rings are reused for the partial results
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    uint32_t* part = reinterpret_cast<uint32_t*>(smem);   // [K quarter][32 rows][32 columns]
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int row = 8 * (i >> 2) + 4 * fr_half + (i & 3);
        part[(wave * 32 + row) * 32 + fr_row] = I32FULL ? static_cast<uint32_t>(acc[i]) : __float_as_uint(accf[i]);
    }
    __syncthreads();
    uint4 pq[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) pq[q] = *reinterpret_cast<const uint4*>(part + (q * 32 + e_row) * 32 + e_col);
    const uint32_t w0[4] = {pq[0].x, pq[0].y, pq[0].z, pq[0].w}, w1[4] = {pq[1].x, pq[1].y, pq[1].z, pq[1].w};
    const uint32_t w2[4] = {pq[2].x, pq[2].y, pq[2].z, pq[2].w}, w3[4] = {pq[3].x, pq[3].y, pq[3].z, pq[3].w};
    float t[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        float v;
        if (I32FULL) {
            v = static_cast<float>(static_cast<int32_t>(w0[c] + w1[c] + w2[c] + w3[c])) * rowm;
            v = v * coln[c];
            if (g.post_scale != 0.0f) v = __uint_as_float(f32_to_bf16_bits(v) << 16) * g.post_scale;
        } else {
            v = __uint_as_float(w0[c]) + __uint_as_float(w1[c]);
            v = v + __uint_as_float(w2[c]);
            v = v + __uint_as_float(w3[c]);
            if (row_part) v = v * rowm;
            if (col_part) v = v * coln[c];
            if (g.out_scale != 1.0f) v = v * g.out_scale;
        }
        t[c] = v;
    }
    uint2 o;
    o.x = pack_bf16x2(t[0], t[1]);
    o.y = pack_bf16x2(t[2], t[3]);
    if (g.bias) {
        o.x = add_bf16x2(o.x, bias_lo);
        o.y = add_bf16x2(o.y, bias_hi);
    }
    *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(g.C) + (int64_t)batch * g.bsc + (int64_t)(m0 + e_row) * g.ldc + n0 + e_col) = o;
}

template <bool I32FULL>
__global__ __launch_bounds__(256) void gemm_i8_wavering_kernel(const GemmArgs g) {
    wavering_block<I32FULL>(g, blockIdx.x, blockIdx.y);
}

// A GEMM over few K tiles: dW of a step on up to 256 tokens.  Its products are nothing beside its output, so this is made for
// writing that: `workers` workgroups share out the 128 x 128 tiles (worker, worker + workers, ...), the next K tile of the walk is fetched
// while one is multiplied, and a finished tile leaves through LDS in rows of 256 bytes, its stores in flight behind the next tile's
// products.  Each of the four waves computes 64 x 64 with the operands of the MFMA swapped: a lane then holds four neighbouring
// columns of a row, eight bytes of the output.  Sums and epilogue are those of the tiled kernels, operation for operation: the same bits.
// 16 tokens, 4096 -> 4096, Y, dX and dW: 15.6 us in one launch, bound by its 64 MiB (32 of weight, 32 of dW); 8.9 + 11.2 us with dW on
// 256 x 256 tiles in a launch of its own, 18.0 us with a workgroup for each tile of dW that loads, multiplies and stores in turn.
// A_ROW: operand A scaled by rows, else by 128 x 128 blocks; operand B by rows (I32FULL) or by blocks.
constexpr int THIN_K_TILES = 2, THIN_OPERAND = 128 * 128, THIN_STORES = 8;
template <bool I32FULL, bool A_ROW>
__device__ __forceinline__ void thin_walk(const GemmArgs& args, const int worker, const int workers) {
    const GemmArgs g = args;
    extern __shared__ __attribute__((aligned(1024))) int8_t smem[];  // two stages of [A 16 KiB][B 16 KiB]; a tile [128 rows][256 bytes] on its way out
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tiles_n = g.N >> 7, tiles = (g.M >> 7) * tiles_n, nk = g.K >> 7;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;

    const int ld_row = lane >> 3;
    uint32_t voffA[2], voffB[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int ch = (lane & 7) ^ ld_row ^ p;
        voffA[p] = (uint32_t)(ld_row * (int)g.lda + ch * 16);
        voffB[p] = (uint32_t)(ld_row * (int)g.ldb + ch * 16);
    }
    auto issue = [&](int tile, int kt, int stage) {       // each wave 32 rows of either operand
        const int m = (tile / tiles_n) * 128 + wave * 32, n = (tile % tiles_n) * 128 + wave * 32;
        int8_t* const st = smem + stage * 2 * THIN_OPERAND + wave * 4096;
        issue_tile_loads<4>(g.A + (int64_t)m * g.lda + kt * 128, 8 * g.lda, voffA, 0, st);
        issue_tile_loads<4>(g.B + (int64_t)n * g.ldb + kt * 128, 8 * g.ldb, voffB, 0, st + THIN_OPERAND);
    };
    // (a K tile's factors by scalar loads: they count apart from the tiles in flight)
    typedef const float __attribute__((address_space(4))) constant_float;
    constant_float* const fa_p = (constant_float*)(uintptr_t)g.sa.p;
    constant_float* const fb_p = (constant_float*)(uintptr_t)g.sb.p;
    const int fr_row = lane & 31, fr_half = lane >> 5;
    const int sw = (lane & 7) ^ ((lane >> 3) & 1);
    int at[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) at[ks] = fr_row * 128 + ((ks * 2 + fr_half) ^ sw) * 16;
    const v16i vzero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

    v16i acc[2][2];
    float accf[I32FULL ? 1 : 2][I32FULL ? 1 : 2][16];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                acc[i][j] = vzero;
#pragma unroll
                for (int r = 0; r < 16; ++r) accf[I32FULL ? 0 : i][I32FULL ? 0 : j][r] = 0.0f;
            }
    };
    clear();
    float rowm[A_ROW ? 2 : 1];
    float4 cm[I32FULL ? 2 : 1][I32FULL ? 4 : 1];
    int stage = 0, tile = worker, kt = 0;
    bool stored = false;
    issue(tile, kt, stage);
    for (;;) {
        const int m0 = (tile / tiles_n) * 128, n0 = (tile % tiles_n) * 128;
        const bool last = kt + 1 == nk;
        const int next_tile = last ? tile + workers : tile, next_kt = last ? 0 : kt + 1;
        // the loads of this K tile are older than the stores of the tile before, which may stay in flight
        if (stored) TI8_WAIT_VMCNT_LGKM0(THIN_STORES);
        else TI8_WAIT_VMCNT_LGKM0(0);
        asm volatile("s_barrier" ::: "memory");
        int8_t* const st = smem + stage * 2 * THIN_OPERAND;
        stage ^= 1;
        if (last) {      // the vectors of the epilogue, in front of the next loads so that they can be waited for alone
            if (A_ROW)
#pragma unroll
                for (int i = 0; i < 2; ++i) rowm[A_ROW ? i : 0] = g.sa.p[(int64_t)(m0 + wm + i * 32 + fr_row) * g.sa.rs];
            if (I32FULL)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) cm[I32FULL ? j : 0][I32FULL ? q : 0] = *reinterpret_cast<const float4*>(g.sb.p + n0 + wn + j * 32 + 8 * q + 4 * fr_half);
        }
        if (next_tile < tiles) issue(next_tile, next_kt, stage);
        const int8_t* const sa = st + wm * 128;
        const int8_t* const sb = st + THIN_OPERAND + wn * 128;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            v4i fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                fa[i] = *reinterpret_cast<const v4i*>(sa + i * 4096 + at[ks]);
                fb[i] = *reinterpret_cast<const v4i*>(sb + i * 4096 + at[ks]);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[j], fa[i], !I32FULL && ks == 0 ? vzero : acc[i][j], 0, 0, 0);
        }
        if (!I32FULL) {
            const float factor = (A_ROW ? 1.0f : fa_p[(int64_t)(m0 >> 7) * g.sa.rs + kt * g.sa.ks]) * fb_p[(int64_t)(n0 >> 7) * g.sb.rs + kt * g.sb.ks];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) accf[i][j][r] = __builtin_fmaf(static_cast<float>(acc[i][j][r]), factor, accf[i][j][r]);
        }
        if (last) {
            __builtin_amdgcn_s_waitcnt(0xc07f);     // lgkmcnt(0): this wave's reads of the stage that the tile leaves through
            asm volatile("s_barrier" ::: "memory");
            // register 4 q + c of block (i, j): row wm + 32 i + lane % 32, column wn + 32 j + 8 q + 4 (lane / 32) + c.  (Written out: in
            // front of an LDS write that it knows the compiler waits for all loads in flight, which write LDS too.)
            const uint32_t slab = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) int8_t*)st;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int row = wm + i * 32 + fr_row;
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int col = wn + j * 32 + 8 * q + 4 * fr_half;
                        const float4 c4 = cm[I32FULL ? j : 0][I32FULL ? q : 0];
                        const float cn[4] = {c4.x, c4.y, c4.z, c4.w};
                        float t[4];
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            float v;
                            if (I32FULL) {
                                v = static_cast<float>(acc[i][j][4 * q + c]) * rowm[A_ROW ? i : 0];
                                v = v * cn[c];
                                if (g.post_scale != 0.0f) v = __uint_as_float(pack_bf16x2(v, 0.0f) << 16) * g.post_scale;
                            } else {
                                v = accf[I32FULL ? 0 : i][I32FULL ? 0 : j][4 * q + c];
                                if (A_ROW) v = v * rowm[A_ROW ? i : 0];
                                v = v * g.out_scale;       // 1 or a power of two
                            }
                            t[c] = v;
                        }
                        const v2i w = {(int)pack_bf16x2(t[0], t[1]), (int)pack_bf16x2(t[2], t[3])};
                        asm volatile("ds_write_b64 %0, %1" ::"v"(slab + row * 256 + ((col * 2) ^ ((row & 15) << 4))), "v"(w) : "memory");
                    }
            }
            __builtin_amdgcn_s_waitcnt(0xc07f);
            asm volatile("s_barrier" ::: "memory");
            uint16_t* const out = reinterpret_cast<uint16_t*>(g.C) + (int64_t)m0 * g.ldc + n0 + (lane & 15) * 8;
            // row 16 p + 4 wave + lane / 16, chunk lane % 16
            const uint32_t from = slab + (wave * 4 + (lane >> 4)) * 256 + (((lane & 15) ^ ((wave * 4 + (lane >> 4)) & 15)) << 4);
            v4i w[THIN_STORES];
            asm volatile("ds_read_b128 %0, %8\n\tds_read_b128 %1, %8 offset:4096\n\tds_read_b128 %2, %8 offset:8192\n\tds_read_b128 %3, %8 offset:12288\n\t"
                         "ds_read_b128 %4, %8 offset:16384\n\tds_read_b128 %5, %8 offset:20480\n\tds_read_b128 %6, %8 offset:24576\n\tds_read_b128 %7, %8 offset:28672\n\t"
                         "s_waitcnt lgkmcnt(0)"
                         : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]), "=&v"(w[4]), "=&v"(w[5]), "=&v"(w[6]), "=&v"(w[7]) : "v"(from) : "memory");
#pragma unroll
            for (int p = 0; p < THIN_STORES; ++p) *reinterpret_cast<v4i*>(out + (int64_t)(p * 16 + wave * 4 + (lane >> 4)) * g.ldc) = w[p];
            if (next_tile >= tiles) break;
            clear();
        }
        stored = last;
        tile = next_tile;
        kt = next_kt;
    }
}

// The GEMMs of a step, or of its backward, on few tokens (batch of one each) in one launch: Y and dX, which have few blocks each
// and wait for their loads most of the time, and with m.count > few dW behind them, a workgroup per CU.
template <bool I32FULL>
__global__ __launch_bounds__(256) void gemm_i8_few_kernel(const GemmMulti m, const int few) {
    const int i = idx::gemm_multi_pick((int)blockIdx.x, m.first[1], m.first[2], m.count);
    if (i < few) wavering_block<I32FULL>(m.g[i], (int)blockIdx.x - m.first[i], 0);
    else {
        const int worker = (int)blockIdx.x - m.first[i], workers = (int)gridDim.x - m.first[i];
        if (I32FULL || m.g[i].sa.mode == TI8_SCALE_ROW) thin_walk<I32FULL, true>(m.g[i], worker, workers);
        else thin_walk<I32FULL, I32FULL>(m.g[i], worker, workers);
    }
}

bool skinny_supported(const GemmArgs& a) {
    // factors that vary inside a 32 x 32 block (one scale per row or column AND K tile) and more
    // than 256 K tiles are left to the tiled kernels
    if (a.sa.mode == TI8_SCALE_ROW_K128 || a.sb.mode == TI8_SCALE_ROW_K128) return false;
    if (a.K > 256 * 128) return false;
    return (int64_t)(a.N / 32) * (a.M / 32) <= 0x7fffffffLL;
}

bool thin_supported(const GemmArgs& a, bool i32_full) {
    if (a.K > THIN_K_TILES * 128 || a.M % 128 || a.N % 128 || a.strict || a.combine != TI8_COMBINE_MUL_MUL || !aligned16(a.C) || a.ldc % 8) return false;
    if (i32_full ? a.sb.rs != 1 || !aligned16(a.sb.p) : a.sb.mode != TI8_SCALE_BLOCK128 || (a.sa.mode != TI8_SCALE_ROW && a.sa.mode != TI8_SCALE_BLOCK128)) return false;
    return (int64_t)(a.M / 128) * (a.N / 128) <= 0x3fffffff;
}

constexpr size_t WAVERING_LDS_BYTES = (size_t)4 * WS_STAGES * WS_STAGE_BYTES;
static_assert(WAVERING_LDS_BYTES >= (size_t)2 * 2 * THIN_OPERAND, "the tiles of dW share the launch");

int init_skinny_kernels() {
    static OncePerDevice once_i32, once_promote, once_i32_multi, once_promote_multi;
    hipError_t e = raise_lds_limit(once_i32, reinterpret_cast<const void*>(gemm_i8_wavering_kernel<true>), (int)WAVERING_LDS_BYTES);
    if (e == hipSuccess) e = raise_lds_limit(once_promote, reinterpret_cast<const void*>(gemm_i8_wavering_kernel<false>), (int)WAVERING_LDS_BYTES);
    if (e == hipSuccess) e = raise_lds_limit(once_i32_multi, reinterpret_cast<const void*>(gemm_i8_few_kernel<true>), (int)WAVERING_LDS_BYTES);
    if (e == hipSuccess) e = raise_lds_limit(once_promote_multi, reinterpret_cast<const void*>(gemm_i8_few_kernel<false>), (int)WAVERING_LDS_BYTES);
    if (e != hipSuccess) return fail(TI8_ERR_HIP, "gemm: cannot raise the LDS limit to %zu: %s", WAVERING_LDS_BYTES, hipGetErrorString(e));
    return TI8_OK;
}

static int launch_wavering(const GemmArgs& a, int64_t batch, bool i32_full, hipStream_t st) {
    constexpr size_t shmem = WAVERING_LDS_BYTES;
    if (int e = init_skinny_kernels()) return e;
    dim3 grid((unsigned)((a.N / 32) * (a.M / 32)), (unsigned)batch), block(256);
    if (i32_full)
        hipLaunchKernelGGL(gemm_i8_wavering_kernel<true>, grid, block, shmem, st, a);
    else
        hipLaunchKernelGGL(gemm_i8_wavering_kernel<false>, grid, block, shmem, st, a);
    note_gemm_kernel(TI8_KERNEL_FEW_ROWS, 32, 32, i32_full ? EPI_ROWS : EPI_PROMOTE);
    return check_launch("ti8_gemm_i8_nt");
}

int launch_skinny(const GemmArgs& a, int64_t batch, bool i32_full, hipStream_t st) {
    return launch_wavering(a, batch, i32_full, st);
}

int launch_few(GemmMulti& m, int few, bool i32_full, hipStream_t st) {
    if (int e = init_skinny_kernels()) return e;
    int64_t total = 0;
    const int64_t cus = device_cu_count();
    for (int i = 0; i < m.count; ++i) {
        m.first[i] = (int)total;
        const int64_t tiles = (int64_t)(m.g[i].N / 128) * (m.g[i].M / 128);
        total += i < few ? (int64_t)(m.g[i].N / 32) * (m.g[i].M / 32) : tiles < cus ? tiles : cus;
        if (total > 0x7fffffffLL) return fail(TI8_ERR_SHAPE, "gemm: too many blocks");
    }
    for (int i = m.count; i <= GEMM_MULTI_MAX; ++i) m.first[i] = (int)total;
    for (int i = m.count; i < GEMM_MULTI_MAX; ++i) m.g[i] = m.g[0];
    const auto kernel = i32_full ? gemm_i8_few_kernel<true> : gemm_i8_few_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)total), dim3(256), WAVERING_LDS_BYTES, st, m, few);
    note_gemm_kernel(TI8_KERNEL_FEW_ROWS, 32, 32, i32_full ? EPI_ROWS : EPI_PROMOTE);
    return check_launch("ti8_gemm_i8_nt");
}

}  // namespace ti8
