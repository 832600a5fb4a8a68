// INT8 NT GEMM for few rows (decode-like shapes: up to 256 rows, in steps of 32).
//
// With so few rows the tiled kernel of gemm.hip has only N/128 workgroups, and each walks the
// whole K behind a two-stage LDS pipeline: its time is load latency, not MFMA.  Here C is cut
// into 32 x 32 blocks, one or four per workgroup, and K is split over the four
// waves of the workgroup, each of which runs its own load -> LDS -> MFMA pipeline with no
// barrier in the loop.
//
// The arithmetic and the epilogue are those of the tiled kernel's int32 and fast-promotion paths,
// operation for operation; only the order in which K tiles are added differs (four partial sums
// per output, K tiles walked from a workgroup-dependent start).  The int32 path is therefore
// bit-identical to the tiled kernel, the promoted path differs by fp32 association only.
#include "gemm_args.h"
#include "quant_math.h"

namespace ti8 {

// s_waitcnt vmcnt(n) (gfx9 encoding: vmcnt in bits 3:0 and 15:14) and lgkmcnt(0) (bits 11:8),
// expcnt untouched (bits 6:4)
#define TI8_WAIT_VMCNT_LGKM0(n) __builtin_amdgcn_s_waitcnt(((n) & 0xf) | (((n) >> 4) << 14) | 0x0070)

// A workgroup owns 32 x 32 of C (or 64 x 64, with twice the stages' bytes) and its four waves split K into quarters.  Every wave streams ITS
// quarter of both operands through a private LDS ring (WS_STAGES stages of [A 32 rows][B 32 rows]
// = 8 KiB, filled by global_load_lds in the swizzled layout of the tiled kernel), waits only
// for its own loads and never for another wave; the four partial results meet in LDS at the end
// and are added in the fixed order q0 + q1 + q2 + q3 (int32: exact; fp32: deterministic).
// Independent streams hide the per-tile latency chain (load -> LDS -> MFMA -> convert) that one
// stream per workgroup behind a barrier exposes: a version with 64 x 32 blocks, an 8-stage ring
// shared by the workgroup and one barrier per K tile took 14.4 us where this one takes 11.2 us
// (128 rows, K = N = 4096).  Two stages = 64 KiB per workgroup, so two workgroups share a CU.
constexpr int WS_STAGES = 2;
constexpr int DECODE_A_BYTES = DECODE_ROWS * 128;    // a K tile of A that the wave quantises itself

// A workgroup's part of C is MB x NB blocks of 32 x 32, one or four: `block_x` = index of the workgroup among those of this GEMM and
// batch.  What bounds the kernel is the stream into a CU's LDS (55 bytes per ns, half of what the L2 alone delivers; neither more stages
// in flight, 3 or 4 instead of 2, nor leaving the MFMAs out makes a difference), and of four blocks the stream is half as long per
// product.  idx::few_rows_wide says where which is the faster one.  us, one block / four, int32 path: 64 rows, 4096 -> 14336
// 21.0 / 15.3; 128 rows 4096 -> 4096 10.1 / 10.1, 8192 -> 8192 33.4 / 21.1; 256 rows 4096 -> 4096 16.7 / 10.8, 14336 -> 4096 98 / 36;
// 64 rows, 14336 -> 14336 46.6 / 32.1 (31.6 for the weight alone).
// QUANTISE: operand A is bf16 (g.A, g.lda in elements), 1 to 8 rows, and each wave quantises the 128 columns of its K tile on the way to
// LDS, one 16-byte chunk of a row per lane, with the quantisers' own arithmetic: by the absmax of the K tile (BY_TILES), or of the row
// (BY_ROWS), which every workgroup looks for first.  The missing ones of the 32 rows are copies of those 8, and missing ones of the 8 copies
// of the last: rows of C that nobody reads.
enum Quantise { APART, BY_TILES, BY_ROWS };
template <bool I32FULL, int BLOCKS, Quantise QUANTISE = APART>
__device__ __forceinline__ void wavering_block(const GemmArgs& g, const int block_x, const int batch, const int rows = 0) {
    static_assert(QUANTISE == APART || BLOCKS == 1, "up to 8 rows");
    static_assert(QUANTISE != BY_TILES || !I32FULL, "a scale per K tile");
    constexpr int MB = BLOCKS, NB = BLOCKS;
    constexpr int B_AT = QUANTISE ? 0 : MB * 4096, STAGE_BYTES = B_AT + NB * 4096;     // per wave
    extern __shared__ __attribute__((aligned(1024))) int8_t smem[];  // 4 waves x WS_STAGES x STAGE_BYTES

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int mtiles = (g.M + 32 * MB - 1) / (32 * MB), nstrips = g.N / (32 * NB);
    const idx::FewPlace place = idx::few_place(block_x, mtiles, nstrips);
    const int n0 = place.strip * 32 * NB, m0 = place.mt * 32 * MB;
    const int mblocks = min(MB, (g.M - m0) >> 5);      // blocks of rows that exist; what is computed beyond them is not stored
    const int nk = g.K >> 7;
    const int kbeg = idx::few_k_first(wave, nk), kend = idx::few_k_first(wave + 1, nk);
    const int nq = kend - kbeg;

    // ---- global -> LDS (same slab layout and swizzle as the other kernels): 4 instructions per block
    // of A's or B's rows (rows 8i .. 8i+7) and stage, all issued by the wave that consumes them
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
    int8_t* const ring = smem + wave * (WS_STAGES * STAGE_BYTES + (QUANTISE ? DECODE_A_BYTES : 0));
    // QUANTISE: this lane's 16 elements of a K tile, on their way from memory, and where their codes go
    const uint16_t* const x = reinterpret_cast<const uint16_t*>(g.A) + (QUANTISE ? min(ld_row, rows - 1) * g.lda + (lane & 7) * 16 : 0);
    uint4 x_lo = {0, 0, 0, 0}, x_hi = {0, 0, 0, 0};
    int8_t* const a_tile = ring + WS_STAGES * STAGE_BYTES;
    const uint32_t a_to = QUANTISE ? (uint32_t)(uintptr_t)(__attribute__((address_space(3))) int8_t*)(a_tile + ld_row * 128 + ((lane & 7) ^ ld_row) * 16) : 0;
    // step i of this wave's walk is K tile kbeg + (i + rot) mod nq: workgroups of one block start at different
    // tiles so that they do not ask the same memory channels for their lines at the same time.  With more rows what counts is that
    // the workgroups of an XCD read A's columns together, which then need not all fit its L2 (256 rows, K = 14336, N = 4096:
    // 36 us, 55 from different tiles on)
    const int rot = nq > 0 && BLOCKS == 1 ? (int)((((unsigned)block_x >> 3) * 3u + (unsigned)batch) % (unsigned)nq) : 0;
    auto tile_of_step = [&](int i) { return idx::few_k_tile(i, rot, kbeg, nq, nk); };    // past the end: the last one again, into a free stage
    auto issue_stage = [&](int i) {
        int8_t* st = ring + (i & (WS_STAGES - 1)) * STAGE_BYTES;
        const int koff = tile_of_step(i) * 128;
        if (QUANTISE) {
            x_lo = *reinterpret_cast<const uint4*>(x + koff);
            x_hi = *reinterpret_cast<const uint4*>(x + koff + 8);
        } else {
#pragma unroll
            for (int b = 0; b < MB; ++b) issue_tile_loads<4>(baseA + koff + min(b, mblocks - 1) * 4 * strideA8, strideA8, voffA, 0, st + b * 4096);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) issue_tile_loads<4>(baseB + koff + b * 4 * strideB8, strideB8, voffB, 0, st + B_AT + b * 4096);
    };

    // ---- scales: unconditional loads (an operand that contributes no in-loop factor is read with
    // stride 0 and dropped; a load under a branch would be waited for on the spot), issued before
    // the tile loads
    const bool divide = !I32FULL && g.combine == TI8_COMBINE_DIV_PROD;
    const bool a_in = !I32FULL && g.sa.mode != TI8_SCALE_ROW, b_in = !I32FULL && g.sb.mode != TI8_SCALE_ROW;
    float fvec[4] = {1.0f, 1.0f, 1.0f, 1.0f};
    if (!I32FULL && QUANTISE != BY_TILES) {
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
    // epilogue scales of the outputs this thread will finish: row t/8, columns 4*(t%8) .. +3 of every block
    const int e_row = threadIdx.x >> 3, e_col = (threadIdx.x & 7) * 4;
    const bool row_part = I32FULL || g.sa.mode == TI8_SCALE_ROW, col_part = I32FULL || g.sb.mode == TI8_SCALE_ROW;
    float rowm[MB], coln[NB][4];
#pragma unroll
    for (int b = 0; b < MB; ++b)
        rowm[b] = g.sa.p[(int64_t)batch * g.sa.bs + (row_part ? (int64_t)(m0 + min(b, mblocks - 1) * 32 + e_row) * g.sa.rs : 0)];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int c = 0; c < 4; ++c) coln[b][c] = g.sb.p[(int64_t)batch * g.sb.bs + (col_part ? (int64_t)(n0 + b * 32 + e_col + c) * g.sb.rs : 0)];
    if (divide) {
#pragma unroll
        for (int b = 0; b < MB; ++b) rowm[b] = 1.0f / rowm[b];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int c = 0; c < 4; ++c) coln[b][c] = 1.0f / coln[b][c];
    }

    // the bias of those columns (without one: 8 bytes of B, dropped)
    uint32_t bias_lo[NB], bias_hi[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const uint2 bias = *reinterpret_cast<const uint2*>(g.bias ? reinterpret_cast<const void*>(g.bias + n0 + b * 32 + e_col) : reinterpret_cast<const void*>(g.B));
        bias_lo[b] = bias.x;
        bias_hi[b] = bias.y;
    }

    const int fr_row = lane & 31, fr_half = lane >> 5;
    const int sw = (lane & 7) ^ ((lane >> 3) & 1);
    int at[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) at[ks] = fr_row * 128 + ((ks * 2 + fr_half) ^ sw) * 16;
    int at_a[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) at_a[ks] = QUANTISE ? (lane & 7) * 128 + ((ks * 2 + fr_half) ^ (lane & 7)) * 16 : at[ks];

    const v16i vzero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    v16i d[MB][NB];             // int32 sums: of the whole K (I32FULL), or of the step whose products are folded next
    float accf[I32FULL ? 1 : MB][I32FULL ? 1 : NB][16];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            d[i][j] = vzero;
#pragma unroll
            for (int r = 0; r < 16; ++r) accf[I32FULL ? 0 : i][I32FULL ? 0 : j][r] = 0.0f;
        }

    issue_stage(0);
    // pin the scale vectors to registers here (they are older than the tile loads, so this waits
    // for nothing else): a load still pending at the loop's entry makes the compiler drain the
    // whole load queue at the top of every iteration
#pragma unroll
    for (int b = 0; b < MB; ++b) asm volatile("" : "+v"(rowm[b]));
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        asm volatile("" : "+v"(bias_lo[b]), "+v"(bias_hi[b]));
#pragma unroll
        for (int c = 0; c < 4; ++c) asm volatile("" : "+v"(coln[b][c]));
    }

    float row_mult = 0.0f;      // BY_ROWS: of this lane's row of A
    if (QUANTISE == BY_ROWS) {
        float amax = 0.0f;
#pragma unroll 4
        for (int kt = kbeg; kt < kend; ++kt)
            amax = absmax8(*reinterpret_cast<const uint4*>(x + kt * 128 + 8), absmax8(*reinterpret_cast<const uint4*>(x + kt * 128), amax));
        amax = dpp_max<0x141>(dpp_max<0x4E>(dpp_max<0xB1>(amax)));      // over the 8 lanes of a row
        float* const red = reinterpret_cast<float*>(smem + 4 * (WS_STAGES * STAGE_BYTES + DECODE_A_BYTES));     // [wave][row]
        if ((lane & 7) == 0) red[wave * DECODE_ROWS + ld_row] = amax;
        __syncthreads();
        auto of_row = [&](int r) { return amax_floor(fmaxf(fmaxf(red[r], red[DECODE_ROWS + r]), fmaxf(red[2 * DECODE_ROWS + r], red[3 * DECODE_ROWS + r])), 0); };
        row_mult = 127.0f / of_row(ld_row);
        const float out_amax = of_row(e_row & (DECODE_ROWS - 1));
        rowm[0] = I32FULL ? out_amax / 127.0f : 1.0f / (127.0f / out_amax);
    }

    auto factor_of_step = [&](int i) -> float {
        const int kt = tile_of_step(i);
        const int l = kt & 63, c = kt >> 6;
        const float v0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fvec[0]), l));
        const float v1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fvec[1]), l));
        const float v2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fvec[2]), l));
        const float v3 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fvec[3]), l));
        return c == 0 ? v0 : (c == 1 ? v1 : (c == 2 ? v2 : v3));
    };
    float f_prev = 0.0f;
    auto fold = [&]() {
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    float& a = accf[I32FULL ? 0 : i][I32FULL ? 0 : j][r];
                    a = __builtin_fmaf(static_cast<float>(d[i][j][r]), f_prev, a);
                }
    };
    for (int i = 0; i < nq; ++i) {
        // own loads of step i landed; own LDS reads of step i - 1 returned, so its stage can be refilled.  No barrier: nobody
        // else touches this wave's ring.
        TI8_WAIT_VMCNT_LGKM0(0);
        const uint4 now_lo = x_lo, now_hi = x_hi;
        issue_stage(i + 1);
        const int8_t* st = ring + (i & (WS_STAGES - 1)) * STAGE_BYTES;
        float f_now = 0.0f;
        if (QUANTISE) {
            float scale = row_mult;
            if (QUANTISE == BY_TILES) {
                const float amax = amax_floor(wave_max(absmax8(now_hi, absmax8(now_lo, 0.0f))), 0);
                scale = 127.0f / amax;
                f_now = 1.0f / scale;
            }
            const uint2 lo = quant8(now_lo, scale), hi = quant8(now_hi, scale);
            const v4i codes = {(int)lo.x, (int)lo.y, (int)hi.x, (int)hi.y};
            // (a store that the compiler knew of would wait for the loads in flight to LDS; a wave's LDS instructions stay in order)
            asm volatile("ds_write_b128 %0, %1" ::"v"(a_to), "v"(codes) : "memory");
        }
        v4i fa[MB][4], fb[NB][4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
            for (int b = 0; b < MB; ++b) fa[b][ks] = *reinterpret_cast<const v4i*>((QUANTISE ? a_tile : st + b * 4096) + at_a[ks]);
#pragma unroll
            for (int b = 0; b < NB; ++b) fb[b][ks] = *reinterpret_cast<const v4i*>(st + B_AT + b * 4096 + at[ks]);
        }
        __builtin_amdgcn_sched_barrier(0);   // all reads go out before anything else
        if (!I32FULL) {
            fold();
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int a = 0; a < MB; ++a)
#pragma unroll
                for (int b = 0; b < NB; ++b) d[a][b] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[a][ks], fb[b][ks], !I32FULL && ks == 0 ? vzero : d[a][b], 0, 0, 0);
        if (!I32FULL) f_prev = QUANTISE == BY_TILES ? f_now : factor_of_step(i);
    }
    if (!I32FULL) fold();
    // every load (the redundant ones of the last steps included) has landed and every wave is
    // done with its ring before the rings are reused for the partial results
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    uint32_t* part = reinterpret_cast<uint32_t*>(smem);   // [block of the workgroup][K quarter][32 rows][32 columns]
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = 8 * (r >> 2) + 4 * fr_half + (r & 3);
                part[(((i * NB + j) * 4 + wave) * 32 + row) * 32 + fr_row] = I32FULL ? static_cast<uint32_t>(d[i][j][r]) : __float_as_uint(accf[I32FULL ? 0 : i][I32FULL ? 0 : j][r]);
            }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        if (i >= mblocks) break;
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            uint4 pq[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) pq[q] = *reinterpret_cast<const uint4*>(part + (((i * NB + j) * 4 + q) * 32 + e_row) * 32 + e_col);
            const uint32_t w0[4] = {pq[0].x, pq[0].y, pq[0].z, pq[0].w}, w1[4] = {pq[1].x, pq[1].y, pq[1].z, pq[1].w};
            const uint32_t w2[4] = {pq[2].x, pq[2].y, pq[2].z, pq[2].w}, w3[4] = {pq[3].x, pq[3].y, pq[3].z, pq[3].w};
            float t[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                float v;
                if (I32FULL) {
                    v = static_cast<float>(static_cast<int32_t>(w0[c] + w1[c] + w2[c] + w3[c])) * rowm[i];
                    v = v * coln[j][c];
                    if (g.post_scale != 0.0f) v = __uint_as_float(f32_to_bf16_bits(v) << 16) * g.post_scale;
                } else {
                    v = __uint_as_float(w0[c]) + __uint_as_float(w1[c]);
                    v = v + __uint_as_float(w2[c]);
                    v = v + __uint_as_float(w3[c]);
                    if (row_part) v = v * rowm[i];
                    if (col_part) v = v * coln[j][c];
                    if (g.out_scale != 1.0f) v = v * g.out_scale;
                }
                t[c] = v;
            }
            uint2 o;
            o.x = pack_bf16x2(t[0], t[1]);
            o.y = pack_bf16x2(t[2], t[3]);
            if (g.bias) {
                o.x = add_bf16x2(o.x, bias_lo[j]);
                o.y = add_bf16x2(o.y, bias_hi[j]);
            }
            *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(g.C) + (int64_t)batch * g.bsc + (int64_t)(m0 + i * 32 + e_row) * g.ldc + n0 + j * 32 + e_col) = o;
        }
    }
}

template <bool I32FULL, int BLOCKS>
__global__ __launch_bounds__(256) void gemm_i8_wavering_kernel(const GemmArgs g) {
    wavering_block<I32FULL, BLOCKS>(g, blockIdx.x, blockIdx.y);
}

template <bool I32FULL, Quantise QUANTISE>
__global__ __launch_bounds__(256) void gemm_i8_decode_kernel(const GemmArgs g, const int rows) {
    wavering_block<I32FULL, 1, QUANTISE>(g, blockIdx.x, 0, rows);
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
__global__ __launch_bounds__(256) void gemm_i8_few_kernel(const GemmMulti m, const int few, const bool wide) {
    const int i = idx::gemm_multi_pick((int)blockIdx.x, m.first[1], m.first[2], m.count);
    const int block = (int)blockIdx.x - m.first[i];
    if (i < few) {
        if (wide) wavering_block<I32FULL, 2>(m.g[i], block, 0);
        else wavering_block<I32FULL, 1>(m.g[i], block, 0);
        return;
    }
    const int workers = (int)gridDim.x - m.first[i];
    if (I32FULL || m.g[i].sa.mode == TI8_SCALE_ROW) thin_walk<I32FULL, true>(m.g[i], block, workers);
    else thin_walk<I32FULL, I32FULL>(m.g[i], block, workers);
}

// Y (16 columns of it, rows of the weight) or, COLS, dX (32 columns of the weight) of up to 16 TB tokens, the weight quantised on its way from
// memory into the operands of the matrix instructions: by its rows for Y, by its columns for dX.  A weight that is used by so
// few tokens costs more to quantise into memory (its codes written both ways and read again) than to read twice.  16x16x64 products want 16 codes in a row
// along the contraction: for Y what two loads bring; for dX a lane loads 2 columns of 16 rows and the conversion, which
// places single bytes, transposes them (a single column per lane, which gives every CU a workgroup: 22 us for Y and dX instead of 20, the
// weight's cache lines go to four CUs).  What bounds it is the chain of load, conversion (6 instructions per element, about 5 us of issue both ways)
// and product in one or two waves per SIMD: 4096 -> 4096, 13 us for Y alone, 14 for dX, 25 with dW in the launch, where the conversion both ways and
// the GEMMs took 29 in two.  Four waves take
// the K tiles' quarters, each with two of them on their way; walk, sums and epilogue are those of wavering_block, operation for operation: the
// same bits, in all of its 32 rows: with one block of 16 tokens the others are the sums of zeros.
template <bool COLS, int TB>
__device__ __forceinline__ void raw_block(const GemmArgs& g, const RawWeight& w, const int strip) {
    constexpr int SETS = COLS ? 2 : 1;
    constexpr int AHEAD = 2, WORDS = COLS ? 32 : 16;
    extern __shared__ __attribute__((aligned(1024))) int8_t smem[];
    const int lane = threadIdx.x & 63, low = lane & 15, quad = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = strip * (COLS ? idx::RAW_STRIP_DX : idx::RAW_STRIP_Y), nk = g.K >> 7;
    const int kbeg = idx::few_k_first(wave, nk), nq = idx::few_k_first(wave + 1, nk) - kbeg;
    const int rot = idx::decode_rot(n0, nq);
    auto tile_of_step = [&](int i) { return idx::few_k_tile(i, rot, kbeg, nq, nk); };
    const float f_all = g.sa.p[(int64_t)tile_of_step(lane) * g.sa.ks];    // of step `lane` (at most 64 per wave)

    // maxima of this lane's row, or two columns
    // (of up to 32 parts, all asked for at once: one after the other they took longer than the weight)
    uint32_t parts[idx::RAW_PARTS / 4];
#pragma unroll
    for (int i = 0; i < idx::RAW_PARTS / 4; ++i) {
        const int p = idx::raw_part(i, lane, COLS ? w.nrt : w.nct);
        if (COLS) parts[i] = *reinterpret_cast<const uint32_t*>(w.cols + idx::maxima_cols_at(p, w.C, n0 + 2 * low));
        else parts[i] = w.rows[idx::maxima_rows_at(p, w.R, n0 + low)];
    }
    __builtin_amdgcn_sched_barrier(0);

    uint32_t raw[AHEAD][WORDS];
    v4i codes[AHEAD][TB][2];
    const uint32_t lane_bytes = COLS ? idx::raw_col_lane_bytes(w.ldw, lane) : 0;
    auto load = [&](int step, uint32_t (&to)[WORDS], v4i (&a)[TB][2]) {
        const int kt = tile_of_step(step);
        if constexpr (COLS) {
            uint32_t at = lane_bytes;
            asm volatile("" : "+v"(at));        // (a scalar base and a 32-bit offset per load)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const char* row = reinterpret_cast<const char*>(w.w + idx::raw_col_base(n0, w.ldw, kt, h, 0));
#pragma unroll
                for (int j = 0; j < 16; ++j, row += 2 * w.ldw) to[h * 16 + j] = *reinterpret_cast<const uint32_t*>(row + at);      // (raw_col_base of row j)
            }
#pragma unroll
            for (int b = 0; b < TB; ++b)
#pragma unroll
                for (int h = 0; h < 2; ++h) a[b][h] = *reinterpret_cast<const v4i*>(g.A + idx::raw_col_codes_offset(b * 16 + low, g.lda, kt, h, lane));
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint4 v = *reinterpret_cast<const uint4*>(w.w + idx::raw_row_offset(n0, w.ldw, kt, i, lane));
                to[i * 4] = v.x; to[i * 4 + 1] = v.y; to[i * 4 + 2] = v.z; to[i * 4 + 3] = v.w;
            }
#pragma unroll
            for (int b = 0; b < TB; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const v2i v = *reinterpret_cast<const v2i*>(g.A + idx::raw_row_codes_offset(b * 16 + low, g.lda, kt, i, lane));
                    a[b][i >> 1][(i & 1) * 2] = v.x;
                    a[b][i >> 1][(i & 1) * 2 + 1] = v.y;
                }
        }
    };
#pragma unroll
    for (int t = 0; t < AHEAD; ++t) load(t, raw[t], codes[t]);     // (past the last one: that one again)
    __builtin_amdgcn_sched_barrier(0);

    uint32_t m_lo = 0, m_hi = 0;
#pragma unroll
    for (int i = 0; i < idx::RAW_PARTS / 4; ++i) {
        m_lo = max(m_lo, parts[i] & 0xffffu);
        m_hi = max(m_hi, parts[i] >> 16);
    }
    m_lo = max(m_lo, (uint32_t)__shfl_xor((int)m_lo, 16, 64));
    m_lo = max(m_lo, (uint32_t)__shfl_xor((int)m_lo, 32, 64));
    const QMode mode = {1, 0, 0, TI8_INV_RCP_OF_SCALE};
    const float amax_lo = amax_floor(__uint_as_float(m_lo << 16), 0), mult_lo = 127.0f / amax_lo, scale_lo = stored_scale(amax_lo, mult_lo, mode);
    float mult_hi = 0.0f, scale_hi = 0.0f;
    if (COLS) {
        m_hi = max(m_hi, (uint32_t)__shfl_xor((int)m_hi, 16, 64));
        m_hi = max(m_hi, (uint32_t)__shfl_xor((int)m_hi, 32, 64));
        const float amax_hi = amax_floor(__uint_as_float(m_hi << 16), 0);
        mult_hi = 127.0f / amax_hi;
        scale_hi = stored_scale(amax_hi, mult_hi, mode);
    }

    const v4i zero = {0, 0, 0, 0};
    float accf[SETS][TB][4];
#pragma unroll
    for (int s = 0; s < SETS; ++s)
#pragma unroll
        for (int b = 0; b < TB; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) accf[s][b][r] = 0.0f;
    auto multiply = [&](int step, const uint32_t (&v)[WORDS], const v4i (&a)[TB][2]) {
        const float f = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f_all), step));
        v4i d[SETS][TB];
#pragma unroll
        for (int s = 0; s < SETS; ++s)
#pragma unroll
            for (int b = 0; b < TB; ++b) d[s][b] = zero;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            v4i op[SETS];
            if constexpr (COLS) {
                uint32_t lo[4] = {0, 0, 0, 0}, hi[4] = {0, 0, 0, 0};
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    lo[j >> 2] = put_u8(qbiased(bf16_lo(v[h * 16 + j]), mult_lo), j & 3, lo[j >> 2]);
                    hi[j >> 2] = put_u8(qbiased(bf16_hi(v[h * 16 + j]), mult_hi), j & 3, hi[j >> 2]);
                }
                op[0] = v4i{(int)(lo[0] ^ UNBIAS4), (int)(lo[1] ^ UNBIAS4), (int)(lo[2] ^ UNBIAS4), (int)(lo[3] ^ UNBIAS4)};
                op[SETS - 1] = v4i{(int)(hi[0] ^ UNBIAS4), (int)(hi[1] ^ UNBIAS4), (int)(hi[2] ^ UNBIAS4), (int)(hi[3] ^ UNBIAS4)};
            } else {
                const uint32_t* const x = v + h * 8;
                const uint2 p = quant8(make_uint4(x[0], x[1], x[2], x[3]), mult_lo), q = quant8(make_uint4(x[4], x[5], x[6], x[7]), mult_lo);
                op[0] = v4i{(int)p.x, (int)p.y, (int)q.x, (int)q.y};
            }
#pragma unroll
            for (int s = 0; s < SETS; ++s)
#pragma unroll
                for (int b = 0; b < TB; ++b) d[s][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(op[s], a[b][h], d[s][b], 0, 0, 0);
        }
#pragma unroll
        for (int s = 0; s < SETS; ++s)
#pragma unroll
            for (int b = 0; b < TB; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) accf[s][b][r] = __builtin_fmaf(static_cast<float>(d[s][b][r]), f, accf[s][b][r]);
    };
    // one copy of the code (a kernel's instructions come from memory, too): loads past the last K tile ask for that one again
    for (int step = 0; step < nq; step += AHEAD)
#pragma unroll
        for (int t = 0; t < AHEAD; ++t) {
            if (step + t < nq) multiply(step + t, raw[t], codes[t]);
            __builtin_amdgcn_sched_barrier(0);      // the compiler would put off the loads to the end of the batch
            load(step + AHEAD + t, raw[t], codes[t]);
            __builtin_amdgcn_sched_barrier(0);
        }

    // lane: token 16 b + low; columns n0 + 4 quad + r, COLS: n0 + 2 (4 quad + r) + set
    float4* const sums = reinterpret_cast<float4*>(smem);       // [wave][set][b][lane]
#pragma unroll
    for (int s = 0; s < SETS; ++s)
#pragma unroll
        for (int b = 0; b < TB; ++b)
            sums[((wave * SETS + s) * TB + b) * 64 + lane] = make_float4(accf[s][b][0], accf[s][b][1], accf[s][b][2], accf[s][b][3]);
    // a quarter's sum over codes of zero: zero, or NaN where a factor is infinite
    float* const sums_of_zeros = reinterpret_cast<float*>(sums + 4 * SETS * TB * 64);      // [wave]
    if (TB == 1) {
        const float z = lane < nq ? 0.0f * f_all : 0.0f;
        const uint64_t nan = __ballot(z != z);
        if (lane == 0) sums_of_zeros[wave] = 0.0f;
        if (nan && lane == __builtin_ctzll(nan)) sums_of_zeros[wave] = z;
    }
    float scale[SETS][4];       // of those columns
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        scale[0][r] = __shfl(scale_lo, quad * 4 + r, 64);
        if (COLS) scale[SETS - 1][r] = __shfl(scale_hi, quad * 4 + r, 64);
    }
    __syncthreads();
    if (wave >= 2) return;
    const int token = wave * 16 + low;
    float out[SETS][4];
#pragma unroll
    for (int s = 0; s < SETS; ++s) {
        float part[4][4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float4 v;
            if (wave < TB) v = sums[((q * SETS + s) * TB + wave) * 64 + lane];
            else v = make_float4(sums_of_zeros[q], sums_of_zeros[q], sums_of_zeros[q], sums_of_zeros[q]);
            part[q][0] = v.x; part[q][1] = v.y; part[q][2] = v.z; part[q][3] = v.w;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float v = part[0][r] + part[1][r];
            v = v + part[2][r];
            v = v + part[3][r];
            out[s][r] = v * scale[s][r];
        }
    }
    uint16_t* const to = reinterpret_cast<uint16_t*>(g.C) + (int64_t)token * g.ldc + n0 + quad * (4 * SETS);
    if constexpr (COLS)
        *reinterpret_cast<uint4*>(to) = make_uint4(pack_bf16x2(out[0][0], out[SETS - 1][0]), pack_bf16x2(out[0][1], out[SETS - 1][1]),
                                                   pack_bf16x2(out[0][2], out[SETS - 1][2]), pack_bf16x2(out[0][3], out[SETS - 1][3]));
    else
        *reinterpret_cast<uint2*>(to) = make_uint2(pack_bf16x2(out[0][0], out[0][1]), pack_bf16x2(out[0][2], out[0][3]));
}

// dX first: its workgroups have the most to do, two that share the cache lines of the weight on one XCD
template <int TB>
__global__ __launch_bounds__(256) void gemm_i8_raw_weight_kernel(const GemmMulti m, const RawWeight w) {
    const int block = (int)blockIdx.x;
    if (block < m.first[1]) raw_block<true, TB>(m.g[1], w, idx::column_strip(block, m.first[1]));
    else if (block < m.first[2]) raw_block<false, TB>(m.g[0], w, block - m.first[1]);
    else thin_walk<false, false>(m.g[2], block - m.first[2], (int)gridDim.x - m.first[2]);
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

constexpr int wavering_lds_bytes(bool wide) { return 4 * WS_STAGES * 2 * (wide ? 64 : 32) * 128; }
static_assert(wavering_lds_bytes(false) >= 2 * 2 * THIN_OPERAND, "the tiles of dW share the launch");

static bool is_wide(const GemmArgs& a, int64_t batch) { return idx::few_rows_wide(a.M, a.N, a.K, batch, device_cu_count()); }

int init_skinny_kernels() {
    static OncePerDevice all;
    const uint64_t bit = 1ull << (current_device() & 63);
    if (all.done.load(std::memory_order_acquire) & bit) return TI8_OK;
    const void* const kernels[] = {reinterpret_cast<const void*>(gemm_i8_wavering_kernel<false, 2>), reinterpret_cast<const void*>(gemm_i8_wavering_kernel<true, 2>),
                                   reinterpret_cast<const void*>(gemm_i8_few_kernel<false>), reinterpret_cast<const void*>(gemm_i8_few_kernel<true>)};
    for (const void* k : kernels) {
        OncePerDevice once;
        const hipError_t e = raise_lds_limit(once, k, wavering_lds_bytes(true));
        if (e != hipSuccess) return fail(TI8_ERR_HIP, "gemm: cannot raise the LDS limit to %d: %s", wavering_lds_bytes(true), hipGetErrorString(e));
    }
    static_assert(wavering_lds_bytes(false) <= 64 * 1024, "one block needs no raised limit");
    all.done.fetch_or(bit, std::memory_order_release);
    return TI8_OK;
}

int launch_skinny(const GemmArgs& a, int64_t batch, bool i32_full, hipStream_t st) {
    if (int e = init_skinny_kernels()) return e;
    const bool wide = is_wide(a, batch);
    const dim3 grid((unsigned)idx::few_blocks(a.M, a.N, wide), (unsigned)batch);
    const auto kernel = wide ? (i32_full ? gemm_i8_wavering_kernel<true, 2> : gemm_i8_wavering_kernel<false, 2>)
                             : (i32_full ? gemm_i8_wavering_kernel<true, 1> : gemm_i8_wavering_kernel<false, 1>);
    hipLaunchKernelGGL(kernel, grid, dim3(256), wavering_lds_bytes(wide), st, a);
    note_gemm_kernel(TI8_KERNEL_FEW_ROWS, 32, 32, i32_full ? EPI_ROWS : EPI_PROMOTE);
    return check_launch("ti8_gemm_i8_nt");
}

int launch_decode(const GemmArgs& a, int rows, bool i32_full, hipStream_t st) {
    constexpr int lds = 4 * (WS_STAGES * 4096 + DECODE_A_BYTES) + 4 * DECODE_ROWS * 4;
    static_assert(lds >= 4 * 4096 && lds <= 64 * 1024, "the waves' sums meet there");
    const auto kernel = i32_full ? gemm_i8_decode_kernel<true, BY_ROWS>
                                 : a.sa.mode == TI8_SCALE_ROW ? gemm_i8_decode_kernel<false, BY_ROWS> : gemm_i8_decode_kernel<false, BY_TILES>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(a.N / 32)), dim3(256), lds, st, a, rows);
    note_gemm_kernel(TI8_KERNEL_FEW_ROWS, 32, 32, i32_full ? EPI_ROWS : EPI_PROMOTE, TI8_FORM_ROWS);
    return check_launch("ti8_gemm_i8_nt");
}

static int launch_few_group(GemmMulti& m, int few, bool wide, bool i32_full, hipStream_t st) {
    int64_t total = 0;
    const int64_t cus = device_cu_count();
    for (int i = 0; i < m.count; ++i) {
        m.first[i] = (int)total;
        total += i < few ? idx::few_blocks(m.g[i].M, m.g[i].N, wide) : idx::thin_workers(m.g[i].M, m.g[i].N, cus);
        if (total > 0x7fffffffLL) return fail(TI8_ERR_SHAPE, "gemm: too many blocks");
    }
    for (int i = m.count; i <= GEMM_MULTI_MAX; ++i) m.first[i] = (int)total;
    for (int i = m.count; i < GEMM_MULTI_MAX; ++i) m.g[i] = m.g[0];
    const auto kernel = i32_full ? gemm_i8_few_kernel<true> : gemm_i8_few_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)total), dim3(256), wavering_lds_bytes(wide), st, m, few, wide);
    note_gemm_kernel(TI8_KERNEL_FEW_ROWS, 32, 32, i32_full ? EPI_ROWS : EPI_PROMOTE);
    return check_launch("ti8_gemm_i8_nt");
}

int launch_raw_weight(GemmMulti& m, const RawWeight& w, int tokens, hipStream_t st) {
    m.first[0] = 0;
    m.first[1] = w.C / idx::RAW_STRIP_DX;
    m.first[2] = m.first[1] + w.R / idx::RAW_STRIP_Y;
    m.first[3] = m.first[2] + (int)idx::thin_workers(w.R, w.C, device_cu_count());
    const auto kernel = tokens <= 16 ? gemm_i8_raw_weight_kernel<1> : gemm_i8_raw_weight_kernel<2>;
    static_assert(4 * 2 * 2 * 64 * 16 + 4 * 4 <= 2 * 2 * THIN_OPERAND, "the waves' sums share the launch's LDS");
    hipLaunchKernelGGL(kernel, dim3((unsigned)m.first[3]), dim3(256), 2 * 2 * THIN_OPERAND, st, m, w);
    note_gemm_kernel(TI8_KERNEL_FEW_ROWS, 32, 32, EPI_PROMOTE, TI8_FORM_WEIGHT);
    return check_launch("ti8_linear");
}

int launch_few(GemmMulti& m, int few, bool i32_full, hipStream_t st) {
    if (int e = init_skinny_kernels()) return e;
    bool wide[GEMM_MULTI_MAX] = {false, false, false};
    int wides = 0;
    for (int i = 0; i < few; ++i) wides += wide[i] = is_wide(m.g[i], 1);
    if (wides == 0 || wides == few) return launch_few_group(m, few, wides != 0, i32_full, st);
    // both kinds: four blocks in a launch of their own, whose LDS would leave the others one to a CU (100 tokens, 2048 -> 8192, double
    // channel: the step 71 us in one launch)
    GemmMulti four, rest;
    four.count = rest.count = 0;
    for (int i = 0; i < m.count; ++i) (wide[i] ? four.g[four.count++] : rest.g[rest.count++]) = m.g[i];
    if (int e = launch_few_group(four, four.count, true, i32_full, st)) return e;
    return launch_few_group(rest, few - wides, false, i32_full, st);
}

}  // namespace ti8
