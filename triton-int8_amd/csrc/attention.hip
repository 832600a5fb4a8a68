// Backward of causal attention on bf16 tensors: dQ, dK and dV from Q, K, V, the forward's output O and the logarithms of its rows'
// sums.
//
// Two launches, each of which computes the scores again from Q and K and keeps its own sums in registers (seven products per pair
// of tiles instead of five, but nothing is added up in memory and the order of every sum is fixed): attention_dq_kernel walks the
// keys of a block of queries, attention_dkdv_kernel the queries of a block of keys.  Products are v_mfma_f32_32x32x16_bf16 with fp32
// sums; probabilities and score gradients are fp32 and rounded to bf16 as operands of the products behind them.
//
// Scores and their gradients go from one product into the next without leaving the wave's registers: a lane's results of a 32 x 32
// score tile are four rows of every eight in one column, which is an MFMA operand over the rows if the other operand is read in the same
// order, and the transposing LDS read (ds_read_b64_tr_b16) hands out four rows at a time.  A wave owns 32 rows of one operand in
// registers; the other is streamed through LDS in tiles of 32 rows, asked for two tiles ahead without a trip through registers, which
// every wave reads twice, in rows for the scores and transposed for the gradients.  (In front of a step's first transposing read the
// compiler waits for all loads, those of the tile two ahead among them: it takes them for what is read.  A tile so has the products of the
// scores to arrive in.)
//
// Bound by the matrix pipe: batch 4, 32 heads, 4096 x 128: dQ 805 us (1.02 PFLOP/s of its own products), dK and dV 1095 us (1.0
// PFLOP/s), 6.2 ms for torch's three kernels; a large bf16 matrix product reaches 1.17 PFLOP/s.
// A wave that owns 64 rows halves the LDS reads per product but is alone on its SIMD, where nothing covers its vector work: 1090 us
// for dQ, and its dK and dV do not fit the registers.
#include <type_traits>
#include "ti8_common.h"
#include "index_math.h"

namespace ti8 {

namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s lds_v4s;
typedef __attribute__((address_space(3))) void lds_void;

constexpr int TILE_ROWS = 32, STAGES = 3;
constexpr float LOG2E = 1.44269504088896340736f;

struct Strided {        // rows of every (batch, head): element strides, the last dim dense
    const uint16_t* p;
    int64_t sb, sh, ss;
};
struct AttentionArgs {
    Strided q, k, v, o, d_o, dq, dk, dv;
    const float* lse;       // [B, H, S], natural logarithm
    float* rows;            // [B * H, 2, padded]: -lse log2(e) and -sum(dO O) of every query
    int heads, seq, padded, pairs, blocks;      // pairs = B * H; blocks of rows per pair
    float scale;
};

template <int D>
struct Tile {       // 32 rows of D bf16 in LDS, 16-byte chunks permuted within a row against bank conflicts
    static constexpr int ROW = 2 * D, CHUNKS = D / 8, BYTES = TILE_ROWS * ROW, KSTEPS = D / 16, COLS = D / 32;
    static constexpr int SLABS = BYTES / 1024, ROWS_PER_SLAB = 1024 / ROW;      // a wave's load instruction fills a slab
    // the chunks of one number of 16 rows, and four neighbouring ones of 4 rows, fall into different banks each
    __device__ static __forceinline__ int swizzle(int row) {
        return D == 128 ? ((row & 3) << 2) | ((row >> 2) & 3) : (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
    }
    // address of this lane's chunk of an operand whose rows are the tile's: XOR with kstep << 5
    __device__ static __forceinline__ int rows_at(int lane) {
        const int r = lane & 31, h = lane >> 5;
        return r * ROW + ((h ^ swizzle(r)) << 4);
    }
    // the same of an operand over the rows (transposing read): XOR with column tile << 6 and u << 5, plus (16 t + 8 u) ROW
    __device__ static __forceinline__ int columns_at(int lane) {
        const int i = lane & 15, h = lane >> 5, c = ((lane >> 4) & 1) * 2 + ((i >> 1) & 1), r = 4 * h + (i >> 2);
        return r * ROW + ((c ^ swizzle(r)) << 4) + (i & 1) * 8;
    }
};

constexpr int larger(int a, int b) { return a > b ? a : b; }
// stages: two tiles, and for dK and dV 64 floats per wave; the results pass through them at the end, 32 rows per wave
template <int D, int WAVES> constexpr int DKDV_STAGE = 2 * Tile<D>::BYTES + WAVES * 256;
// MFMA steps over D whose values a wave of the dK / dV kernel keeps in LDS: those that its registers do not hold
// (two of eight; with all eight in registers the compiler spills in the loops: 1170 instead of 1095 us at the size above.  Four waves
// are one register short all the same, and keep it in scratch memory between the loops)
template <int D> constexpr int V_IN_LDS = D == 128 ? 2 : 0;
template <int D, int WAVES> constexpr int DKDV_LDS = larger(STAGES * DKDV_STAGE<D, WAVES> + WAVES * V_IN_LDS<D> * 1024, WAVES * Tile<D>::BYTES);
template <int D, int WAVES> constexpr int DQ_STAGE = 2 * Tile<D>::BYTES;
template <int D, int WAVES> constexpr int DQ_LDS = larger(STAGES * DQ_STAGE<D, WAVES>, WAVES * Tile<D>::BYTES);

#if defined(__HIP_DEVICE_COMPILE__)
typedef __amdgpu_buffer_rsrc_t Rsrc;

// the rows of one (batch, head) as a buffer: what lies behind the last row reads as zeros
template <int D>
__device__ __forceinline__ Rsrc rows_of(const Strided& t, int b, int h, int seq) {
    const uint16_t* p = t.p + b * t.sb + h * t.sh;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p), 0, (int)(((int64_t)(seq - 1) * t.ss + D) * 2), 0x00027000);      // = idx::attention_bytes
}
__device__ __forceinline__ v8bf load_chunk(Rsrc r, uint32_t offset) { return __builtin_bit_cast(v8bf, __builtin_amdgcn_raw_buffer_load_b128(r, offset, 0, 0)); }

// Two tensors' tiles of 32 rows on their way into LDS (one behind the other), shared out among the waves of a workgroup
template <int D, int WAVES>
struct TilePair {
    using T = Tile<D>;
    static_assert(T::SLABS % WAVES == 0, "every wave makes the same number of loads of a tile");
    static constexpr int PER_TILE = T::SLABS / WAVES, LOADS = 2 * PER_TILE;     // per wave
    Rsrc x, y;
    uint32_t stride_x, stride_y, at_x, at_y;
    int8_t* lds;
    __device__ __forceinline__ TilePair(Rsrc x_, int64_t ssx, Rsrc y_, int64_t ssy, int wave, int lane, int8_t* lds_) : x(x_), y(y_), lds(lds_ + wave * 1024) {
        const int row = wave * T::ROWS_PER_SLAB + lane / T::CHUNKS, chunk = ((lane % T::CHUNKS) ^ T::swizzle(row)) * 16;
        stride_x = (uint32_t)ssx * 2;
        stride_y = (uint32_t)ssy * 2;
        at_x = row * stride_x + chunk;
        at_y = row * stride_y + chunk;
    }
    // (a wave's slabs of a tile are 16 rows apart, for which the chunks are permuted alike)
    __device__ __forceinline__ void copy(int tile, int offset) const {
#pragma unroll
        for (int i = 0; i < PER_TILE; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(x, (lds_void*)(lds + offset + i * WAVES * 1024), 16, at_x + (tile * TILE_ROWS + i * 16) * stride_x, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < PER_TILE; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(y, (lds_void*)(lds + offset + T::BYTES + i * WAVES * 1024), 16, at_y + (tile * TILE_ROWS + i * 16) * stride_y, 0, 0, 0);
    }
};

// all but this wave's last N loads have landed, its LDS reads have returned, and the same holds for the other waves
template <int N>
__device__ __forceinline__ void wait_and_meet() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((N & 0xf) | ((N >> 4) << 14) | 0x0070);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ v8bf rows_operand(const int8_t* at) { return *reinterpret_cast<const v8bf*>(at); }
template <int D>
__device__ __forceinline__ v8bf columns_operand(const int8_t* tile, int base, int column_tile, int t) {
    const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(tile + ((base ^ (column_tile << 6)) + 16 * t * Tile<D>::ROW)));
    const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(tile + ((base ^ (column_tile << 6) ^ 32) + (16 * t + 8) * Tile<D>::ROW)));
    return __builtin_bit_cast(v8bf, (v8s)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}
__device__ __forceinline__ v16f mfma(v8bf a, v8bf b, v16f c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
// registers 8 t .. 8 t + 7 of a score tile as operand over its rows
__device__ __forceinline__ v8bf operand_of(const v16f& x, int t) {
    const v4u w = {pack_bf16x2(x[8 * t], x[8 * t + 1]), pack_bf16x2(x[8 * t + 2], x[8 * t + 3]), pack_bf16x2(x[8 * t + 4], x[8 * t + 5]), pack_bf16x2(x[8 * t + 6], x[8 * t + 7])};
    return __builtin_bit_cast(v8bf, w);
}

// Store the 32 x D results of a wave, rows 8 g + 4 (lane / 32) + j in register 4 g + j and column lane % 32 of every column tile,
// through 32 rows of LDS that are its own
template <int D>
__device__ __forceinline__ void store_rows(const v16f (&x)[Tile<D>::COLS], float factor, int8_t* slab, const Strided& out, int b, int h, int row0, int seq, int lane) {
    using T = Tile<D>;
#pragma unroll
    for (int db = 0; db < T::COLS; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int row = 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
            *reinterpret_cast<uint16_t*>(slab + row * T::ROW + ((db * 64 + (lane & 31) * 2) ^ ((row & 7) << 4))) = (uint16_t)pack_bf16x2(x[db][i] * factor, 0.0f);
        }
    uint16_t* p = const_cast<uint16_t*>(out.p) + b * out.sb + h * out.sh;
#pragma unroll
    for (int i = 0; i < T::SLABS; ++i) {
        const int row = i * T::ROWS_PER_SLAB + lane / T::CHUNKS, c = lane % T::CHUNKS;
        const uint4 v = *reinterpret_cast<const uint4*>(slab + row * T::ROW + ((c * 16) ^ ((row & 7) << 4)));
        if (row0 + row < seq) *reinterpret_cast<uint4*>(p + (int64_t)(row0 + row) * out.ss + c * 8) = v;
    }
}

__device__ __forceinline__ bool place(const AttentionArgs& a, int& pair, int& block) {
    const idx::AttentionPlace p = idx::attention_place(blockIdx.x, a.blocks);
    pair = p.pair;
    block = p.block;
    return pair < a.pairs;
}
#endif

template <int D, int WAVES>
__global__ __launch_bounds__(WAVES * 64, 2) void attention_dkdv_kernel(const AttentionArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    using T = Tile<D>;
    extern __shared__ __attribute__((aligned(1024))) int8_t smem[];
    int pair, block;
    if (!place(a, pair, block)) return;
    const int b = pair / a.heads, h = pair % a.heads;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = block * (WAVES * 32), nw = n0 + wave * 32;       // first key of the workgroup, of the wave
    const int first = n0 / TILE_ROWS, tiles = (a.seq + TILE_ROWS - 1) / TILE_ROWS;
    const Rsrc rr = __builtin_amdgcn_make_buffer_rsrc(a.rows + (int64_t)pair * 2 * a.padded, 0, a.padded * 8, 0x00027000);
    const TilePair<D, WAVES> stream(rows_of<D>(a.q, b, h, a.seq), a.q.ss, rows_of<D>(a.d_o, b, h, a.seq), a.d_o.ss, wave, lane, smem);
    const uint32_t at_rows = (lane & 31) * 4 + (lane >> 5) * a.padded * 4;
    auto issue = [&](int tile, int stage) {
        const int at = stage * DKDV_STAGE<D, WAVES>;
        stream.copy(tile, at);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rr, (lds_void*)(smem + at + 2 * T::BYTES + wave * 256), 4, at_rows + tile * TILE_ROWS * 4, 0, 0, 0);
    };
    constexpr int LOADS = TilePair<D, WAVES>::LOADS + 1;

    constexpr int VREG = T::KSTEPS - V_IN_LDS<D>;
    v8bf kf[T::KSTEPS], vf[VREG];      // this wave's keys and values as operands over D
    int8_t* const vs = smem + STAGES * DKDV_STAGE<D, WAVES> + wave * V_IN_LDS<D> * 1024;
    {
        const Rsrc rk = rows_of<D>(a.k, b, h, a.seq), rv = rows_of<D>(a.v, b, h, a.seq);
        const uint32_t row = nw + (lane & 31), at = (lane >> 5) * 16;
#pragma unroll
        for (int ks = 0; ks < T::KSTEPS; ++ks) {
            kf[ks] = load_chunk(rk, row * (uint32_t)a.k.ss * 2 + at + ks * 32);
            const uint32_t v = row * (uint32_t)a.v.ss * 2 + at + ks * 32;
            if (ks < VREG) vf[ks < VREG ? ks : 0] = load_chunk(rv, v);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (lds_void*)(vs + (ks - VREG) * 1024), 16, v, 0, 0, 0);
        }
    }
    v16f dk[T::COLS], dv[T::COLS];
#pragma unroll
    for (int db = 0; db < T::COLS; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) dk[db][i] = dv[db][i] = 0.0f;

    issue(first, 0);
    issue(first + 1, 1);
    const int rows_at = T::rows_at(lane), columns_at = T::columns_at(lane);
    const float c = a.scale * LOG2E;

    auto step = [&](const int8_t* st, int m0, auto masked) {
        const int8_t* const qt = st;
        const int8_t* const dt = st + T::BYTES;
        const int8_t* const rt = st + 2 * T::BYTES + wave * 256 + (lane >> 5) * 16;
        v16f s, dp, nl;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < T::KSTEPS; ++ks) s = mfma(rows_operand(qt + (rows_at ^ (ks << 5))), kf[ks], s);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const v4f x = *reinterpret_cast<const v4f*>(rt + g * 32), y = *reinterpret_cast<const v4f*>(rt + 128 + g * 32);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                nl[4 * g + j] = x[j];
                dp[4 * g + j] = y[j];       // dO V^T - sum(dO O), the sum from the start
            }
        }
#pragma unroll
        for (int ks = 0; ks < T::KSTEPS; ++ks) dp = mfma(rows_operand(dt + (rows_at ^ (ks << 5))), ks < VREG ? vf[ks < VREG ? ks : 0] : rows_operand(vs + (ks - VREG) * 1024 + lane * 16), dp);
        const int before = nw + (lane & 31) - m0 - 4 * (lane >> 5);        // queries in front of the key
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], c, nl[i]));
            s[i] = masked && 8 * (i >> 2) + (i & 3) < before ? 0.0f : p;
        }
        const v8bf p0 = operand_of(s, 0), p1 = operand_of(s, 1);
#pragma unroll
        for (int db = 0; db < T::COLS; ++db) {
            dv[db] = mfma(p0, columns_operand<D>(dt, columns_at, db, 0), dv[db]);
            dv[db] = mfma(p1, columns_operand<D>(dt, columns_at, db, 1), dv[db]);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] *= dp[i];
        const v8bf d0 = operand_of(s, 0), d1 = operand_of(s, 1);
#pragma unroll
        for (int db = 0; db < T::COLS; ++db) {
            dk[db] = mfma(d0, columns_operand<D>(qt, columns_at, db, 0), dk[db]);
            dk[db] = mfma(d1, columns_operand<D>(qt, columns_at, db, 1), dk[db]);
        }
    };
    int stage = 0;
    auto walk = [&](int from, int to, auto masked) {
        for (int tile = from; tile < to; ++tile) {
            // own loads of this tile landed (the next tile's may be in flight: as many as every wave issues for a tile); behind the
            // barrier everybody's, and nobody reads the stage of the tile before, which the tile after next goes into
            wait_and_meet<LOADS>();
            issue(tile + 2, stage >= 1 ? stage - 1 : 2);
            if (!masked || (tile + 1) * TILE_ROWS > nw) step(smem + stage * DKDV_STAGE<D, WAVES>, tile * TILE_ROWS, masked);
            stage = stage == 2 ? 0 : stage + 1;
        }
    };
    const int clear = min(tiles, first + WAVES);        // from here on every query comes behind the workgroup's keys
    walk(first, clear, std::true_type{});
    walk(clear, tiles, std::false_type{});
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    int8_t* const slab = smem + wave * T::BYTES;
    store_rows<D>(dk, a.scale, slab, a.dk, b, h, nw, a.seq, lane);
    store_rows<D>(dv, 1.0f, slab, a.dv, b, h, nw, a.seq, lane);
#endif
}

// also writes `rows` for the kernel above
template <int D, int WAVES>
__global__ __launch_bounds__(WAVES * 64, 2) void attention_dq_kernel(const AttentionArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    using T = Tile<D>;
    extern __shared__ __attribute__((aligned(1024))) int8_t smem[];
    int pair, block;
    if (!place(a, pair, block)) return;
    block = a.blocks - 1 - block;       // the longest first
    const int b = pair / a.heads, h = pair % a.heads;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m0 = block * (WAVES * 32), mw = m0 + wave * 32;       // first query of the workgroup, of the wave
    const int tiles = (min(m0 + WAVES * 32, a.seq) + TILE_ROWS - 1) / TILE_ROWS;
    const TilePair<D, WAVES> stream(rows_of<D>(a.k, b, h, a.seq), a.k.ss, rows_of<D>(a.v, b, h, a.seq), a.v.ss, wave, lane, smem);
    auto issue = [&](int tile, int stage) { stream.copy(tile, stage * DQ_STAGE<D, WAVES>); };
    constexpr int LOADS = TilePair<D, WAVES>::LOADS;

    v8bf qf[T::KSTEPS], df[T::KSTEPS];      // this wave's queries and rows of dO as operands over D
    float nl, nd;
    {
        const Rsrc rq = rows_of<D>(a.q, b, h, a.seq), rd = rows_of<D>(a.d_o, b, h, a.seq), ro = rows_of<D>(a.o, b, h, a.seq);
        const int row = mw + (lane & 31);
        const uint32_t at = (lane >> 5) * 16;
        float sum = 0.0f;
#pragma unroll
        for (int ks = 0; ks < T::KSTEPS; ++ks) {
            qf[ks] = load_chunk(rq, row * (uint32_t)a.q.ss * 2 + at + ks * 32);
            df[ks] = load_chunk(rd, row * (uint32_t)a.d_o.ss * 2 + at + ks * 32);
            const v8bf of = load_chunk(ro, row * (uint32_t)a.o.ss * 2 + at + ks * 32);
#pragma unroll
            for (int e = 0; e < 8; ++e) sum = __builtin_fmaf((float)df[ks][e], (float)of[e], sum);
        }
        sum += __shfl_xor(sum, 32, 64);
        nd = -sum;
        nl = row < a.seq ? a.lse[(int64_t)pair * a.seq + row] * -LOG2E : 0.0f;
        if (row < a.padded) a.rows[((int64_t)pair * 2 + (lane >> 5)) * a.padded + row] = lane >> 5 ? nd : nl;
    }
    v16f dq[T::COLS];
#pragma unroll
    for (int db = 0; db < T::COLS; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) dq[db][i] = 0.0f;
    __builtin_amdgcn_s_waitcnt(0);      // from here on nothing but the tiles' loads is in flight: the loop counts them

    issue(0, 0);
    issue(1, 1);
    const int rows_at = T::rows_at(lane), columns_at = T::columns_at(lane);
    const float c = a.scale * LOG2E;
    auto step = [&](const int8_t* st, int n0, auto masked) {
        const int8_t* const kt = st;
        const int8_t* const vt = st + T::BYTES;
        v16f s, dp;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = dp[i] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < T::KSTEPS; ++ks) s = mfma(rows_operand(kt + (rows_at ^ (ks << 5))), qf[ks], s);
#pragma unroll
        for (int ks = 0; ks < T::KSTEPS; ++ks) dp = mfma(rows_operand(vt + (rows_at ^ (ks << 5))), df[ks], dp);
        const int up_to = mw + (lane & 31) - n0 - 4 * (lane >> 5);      // the query's own key
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], c, nl)) * (dp[i] + nd);
            s[i] = masked && 8 * (i >> 2) + (i & 3) > up_to ? 0.0f : p;
        }
        const v8bf d0 = operand_of(s, 0), d1 = operand_of(s, 1);
#pragma unroll
        for (int db = 0; db < T::COLS; ++db) {
            dq[db] = mfma(d0, columns_operand<D>(kt, columns_at, db, 0), dq[db]);
            dq[db] = mfma(d1, columns_operand<D>(kt, columns_at, db, 1), dq[db]);
        }
    };
    int stage = 0;
    auto walk = [&](int from, int to, auto masked) {
        for (int tile = from; tile < to; ++tile) {
            wait_and_meet<LOADS>();
            issue(tile + 2, stage >= 1 ? stage - 1 : 2);
            if (!masked || tile * TILE_ROWS < mw + 32) step(smem + stage * DQ_STAGE<D, WAVES>, tile * TILE_ROWS, masked);
            stage = stage == 2 ? 0 : stage + 1;
        }
    };
    const int clear = m0 / TILE_ROWS;       // up to here every key comes in front of the workgroup's queries
    walk(0, clear, std::false_type{});
    walk(clear, tiles, std::true_type{});
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    store_rows<D>(dq, a.scale, smem + wave * T::BYTES, a.dq, b, h, mw, a.seq, lane);
#endif
}

template <int D, int WAVES_DQ, int WAVES_DKDV>
int prepare(const char* fn) {
    static OncePerDevice once_dq, once_dkdv;
    hipError_t e = raise_lds_limit(once_dq, reinterpret_cast<const void*>(attention_dq_kernel<D, WAVES_DQ>), DQ_LDS<D, WAVES_DQ>);
    if (e == hipSuccess) e = raise_lds_limit(once_dkdv, reinterpret_cast<const void*>(attention_dkdv_kernel<D, WAVES_DKDV>), DKDV_LDS<D, WAVES_DKDV>);
    return e == hipSuccess ? TI8_OK : fail(TI8_ERR_HIP, "%s: cannot raise the LDS limit: %s", fn, hipGetErrorString(e));
}

template <int D, int WAVES_DQ, int WAVES_DKDV>
int launch(const char* fn, AttentionArgs a, hipStream_t st) {
    if (int err = prepare<D, WAVES_DQ, WAVES_DKDV>(fn)) return err;
    const int pairs = (int)idx::round8(a.pairs);
    a.blocks = (a.seq + WAVES_DQ * 32 - 1) / (WAVES_DQ * 32);
    hipLaunchKernelGGL((attention_dq_kernel<D, WAVES_DQ>), dim3((unsigned)(pairs * a.blocks)), dim3(WAVES_DQ * 64), (DQ_LDS<D, WAVES_DQ>), st, a);
    if (int err = check_launch(fn)) return err;
    a.blocks = (a.seq + WAVES_DKDV * 32 - 1) / (WAVES_DKDV * 32);
    hipLaunchKernelGGL((attention_dkdv_kernel<D, WAVES_DKDV>), dim3((unsigned)(pairs * a.blocks)), dim3(WAVES_DKDV * 64), (DKDV_LDS<D, WAVES_DKDV>), st, a);
    return check_launch(fn);
}

int64_t padded_rows(int64_t seq) { return (seq + TILE_ROWS - 1) / TILE_ROWS * TILE_ROWS; }

}  // namespace

int init_attention_kernels() {
    const char* fn = "ti8_init";
    int e = prepare<128, 4, 8>(fn);
    if (!e) e = prepare<128, 4, 4>(fn);
    return e ? e : prepare<64, 4, 4>(fn);
}

}  // namespace ti8

using namespace ti8;

extern "C" int64_t ti8_attention_bwd_workspace(int64_t batch, int64_t heads, int64_t seq) {
    if (batch <= 0 || heads <= 0 || seq <= 0 || seq > (1 << 24) || batch > 0xffffff || heads > 0xffffff || batch * heads > 0xffffff) return -1;
    if (idx::round8(batch * heads) * ((seq + 127) / 128) > 0x7fffffff) return -1;      // workgroups of a launch
    return batch * heads * 2 * padded_rows(seq) * (int64_t)sizeof(float);
}

extern "C" int ti8_attention_bwd(const ti8_attention_args* p, ti8_stream_t stream) {
    const char* fn = "ti8_attention_bwd";
    if (!p || !p->lse || !p->workspace) return fail(TI8_ERR_NULL, "%s: args, lse and workspace are required", fn);
    if (ti8_attention_bwd_workspace(p->batch, p->heads, p->seq) < 0 || (p->head_dim != 64 && p->head_dim != 128))
        return fail(TI8_ERR_SHAPE, "%s: need batch, heads and seq > 0 and head_dim 64 or 128; got batch=%lld heads=%lld seq=%lld head_dim=%lld", fn,
                    (long long)p->batch, (long long)p->heads, (long long)p->seq, (long long)p->head_dim);
    if (!aligned16(p->workspace) || (reinterpret_cast<uintptr_t>(p->lse) & 3)) return fail(TI8_ERR_ALIGN, "%s: workspace or lse is misaligned", fn);
    const ti8_attention_tensor* const tensors[8] = {&p->q, &p->k, &p->v, &p->o, &p->d_o, &p->dq, &p->dk, &p->dv};
    for (const ti8_attention_tensor* x : tensors) {
        if (!x->p) return fail(TI8_ERR_NULL, "%s: q, k, v, o, d_o, dq, dk and dv are required", fn);
        if (!aligned16(x->p) || x->stride_b % 8 || x->stride_h % 8 || x->stride_s % 8)
            return fail(TI8_ERR_ALIGN, "%s: tensors must be 16-byte aligned with strides that are multiples of 8 elements", fn);
        if (!idx::attention_stride_ok(x->stride_s, p->seq, p->head_dim))
            return fail(TI8_ERR_SHAPE, "%s: a row stride of %lld elements does not go with %lld rows of %lld", fn, (long long)x->stride_s, (long long)p->seq, (long long)p->head_dim);
    }
    const auto strided = [](const ti8_attention_tensor& x) { return Strided{static_cast<const uint16_t*>(x.p), x.stride_b, x.stride_h, x.stride_s}; };
    AttentionArgs a;
    a.q = strided(p->q); a.k = strided(p->k); a.v = strided(p->v); a.o = strided(p->o); a.d_o = strided(p->d_o);
    a.dq = strided(p->dq); a.dk = strided(p->dk); a.dv = strided(p->dv);
    a.lse = p->lse;
    a.rows = static_cast<float*>(p->workspace);
    a.heads = (int)p->heads;
    a.seq = (int)p->seq;
    a.padded = (int)padded_rows(p->seq);
    a.pairs = (int)(p->batch * p->heads);
    a.blocks = 0;
    a.scale = p->scale;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    if (p->head_dim == 64) return launch<64, 4, 4>(fn, a, st);
    // eight waves share a stream of tiles where their workgroups fill the chip (dK and dV at 4 x 32 x 4096: 1095 us, 1330 with four; at
    // 32 x 1024, half as many workgroups as CUs, all kernels 88 us with eight and 77 with four)
    return (int64_t)a.pairs * ((a.seq + 255) / 256) >= device_cu_count() ? launch<128, 4, 8>(fn, a, st) : launch<128, 4, 4>(fn, a, st);
}
