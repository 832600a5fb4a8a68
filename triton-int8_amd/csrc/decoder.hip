// What a decoder layer does between its INT8 linears, one pass over memory each: RMSNorm, rotary embedding and the SwiGLU
// product, forward and backward, on bf16 tensors.
//
// All are bound by HBM.  Written as torch expressions they are 60 launches that carry every intermediate through memory, the
// RMSNorm's in fp32: 6.0 ms of a 28 ms layer step (4 x 4096 tokens, hidden 4096, MLP 14336).  Here a tensor is read once and
// a result written once.  Intermediates that the expressions round to bf16 are rounded to bf16 here too (in registers) and rows
// are added up in their order, so that the layer's output and gradients have the bits of the expressions.
#include <type_traits>
#include "ti8_common.h"

namespace ti8 {

namespace {

constexpr int THREADS = 256;
constexpr int NORM_STEP = 2048;                 // RMSNorm: elements of a row per 8 loads of 4 elements that a wave's lanes make
constexpr int NORM_MAX_DIM = 4 * NORM_STEP;     // rows that fit a wave's registers

__device__ __forceinline__ void unpack8(const uint4& v, float* f) {
    f[0] = bf16_lo(v.x); f[1] = bf16_hi(v.x); f[2] = bf16_lo(v.y); f[3] = bf16_hi(v.y);
    f[4] = bf16_lo(v.z); f[5] = bf16_hi(v.z); f[6] = bf16_lo(v.w); f[7] = bf16_hi(v.w);
}
__device__ __forceinline__ uint4 pack8(const float* f) {
    return make_uint4(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]), pack_bf16x2(f[4], f[5]), pack_bf16x2(f[6], f[7]));
}
// each value rounded to bf16 and widened again
__device__ __forceinline__ void round8(float* f) {
    const uint4 v = pack8(f);
    unpack8(v, f);
}

// Sum over a row that a wave holds 4 elements per lane and step, s[e] the lane's sum over its elements e of every step; in every lane.
// The order is that in which torch adds up an fp32 row of up to 4096 elements (lane l: elements 4 l .. 4 l + 3 of every 256, each
// position on its own; then the four, then neighbouring lanes).
__device__ __forceinline__ float row_sum(const float (&s)[4]) {
    float sum = ((s[0] + s[1]) + s[2]) + s[3];
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) sum += __shfl_xor(sum, m, 64);
    return sum;
}

// y = bf16(x * rstd) * w, rstd = 1 / sqrt(mean(x^2) + eps); one wave per row, the row in registers, 4 elements per lane and load.
// The squares are added up in torch's order (row_sum): rstd, and with it y, has the bits of the torch expression.  A difference in
// its last bit would move int8 codes behind it, which the layers that follow spread.
// 16384 x 4096: 56 us (4.8 TB/s; 46 us with 16-byte loads and a workgroup per row, in another order) against about 320 us for the
// seven launches of the expression.
template <int NV>
__global__ __launch_bounds__(THREADS) void rmsnorm_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, uint16_t* __restrict__ y,
                                                          float* __restrict__ rstd, int64_t rows, int dim, float eps) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * (THREADS / 64) + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int nchunk = dim >> 2;
    const uint2* xr = reinterpret_cast<const uint2*>(x + row * dim);
    const uint2* wr = reinterpret_cast<const uint2*>(w);
    uint2 v[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = lane + i * 64;
        v[i] = c < nchunk ? xr[c] : make_uint2(0, 0);
    }
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const float f[4] = {bf16_lo(v[i].x), bf16_hi(v[i].x), bf16_lo(v[i].y), bf16_hi(v[i].y)};
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += f[e] * f[e];
    }
    const float sum = row_sum(s);
    const float r = (float)(1.0 / sqrt((double)(sum * (1.0f / (float)dim) + eps)));   // rounded once; v_rsq_f32 is off by one bit in 7 % of the rows
    if (lane == 0) rstd[row] = r;
    uint2* yr = reinterpret_cast<uint2*>(y + row * dim);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = lane + i * 64;
        if (c < nchunk) {
            const uint2 g = wr[c];
            const uint32_t n0 = pack_bf16x2(bf16_lo(v[i].x) * r, bf16_hi(v[i].x) * r), n1 = pack_bf16x2(bf16_lo(v[i].y) * r, bf16_hi(v[i].y) * r);
            yr[c] = make_uint2(pack_bf16x2(bf16_lo(n0) * bf16_lo(g.x), bf16_hi(n0) * bf16_hi(g.x)), pack_bf16x2(bf16_lo(n1) * bf16_lo(g.y), bf16_hi(n1) * bf16_hi(g.y)));
        }
    }
}

// dx = g rstd + k (2 x) with g = bf16(dy w) and k = -1/2 (sum of g x) rstd^3 / dim, and the products bf16(dy * bf16(x rstd)) whose
// column sums are the weight's gradient: what autograd makes of the expression, rounding by rounding and with the row's sum in torch's
// order (row_sum), so that dx and the products have its bits.  dx goes on into the attention's gradients and the int8 codes behind
// them: summed in another order, dQ and dK came out up to 3.6e-3 away (16384 x 4096).
// The products go through memory because a sum of them in this kernel would be a sum in another order.  One wave per row, the row in
// registers as in the forward.  16384 x 4096: 86 us (6.2 TB/s), and 39 us for torch's sum of the products; the sums in registers with
// 16-byte loads and a workgroup per row took 76 us in all, the launches of the expression about 640.
template <int NV>
__global__ __launch_bounds__(THREADS) void rmsnorm_bwd_kernel(const uint16_t* __restrict__ dy, const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                              const float* __restrict__ rstd, uint16_t* __restrict__ dx, uint16_t* __restrict__ prod,
                                                              int64_t rows, int dim) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * (THREADS / 64) + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int nchunk = dim >> 2;
    const uint2* xr = reinterpret_cast<const uint2*>(x + row * dim);
    const uint2* dr = reinterpret_cast<const uint2*>(dy + row * dim);
    const uint2* wr = reinterpret_cast<const uint2*>(w);
    uint2* pr = reinterpret_cast<uint2*>(prod + row * dim);
    const float r = rstd[row];
    uint2 xv[NV], g[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = lane + i * 64;
        xv[i] = g[i] = make_uint2(0, 0);
        if (c < nchunk) {
            xv[i] = xr[c];
            g[i] = dr[c];
        }
    }
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = lane + i * 64;
        if (c < nchunk) {
            const uint2 wv = wr[c];
            const uint32_t n0 = pack_bf16x2(bf16_lo(xv[i].x) * r, bf16_hi(xv[i].x) * r), n1 = pack_bf16x2(bf16_lo(xv[i].y) * r, bf16_hi(xv[i].y) * r);
            pr[c] = make_uint2(pack_bf16x2(bf16_lo(g[i].x) * bf16_lo(n0), bf16_hi(g[i].x) * bf16_hi(n0)),
                               pack_bf16x2(bf16_lo(g[i].y) * bf16_lo(n1), bf16_hi(g[i].y) * bf16_hi(n1)));
            g[i] = make_uint2(pack_bf16x2(bf16_lo(g[i].x) * bf16_lo(wv.x), bf16_hi(g[i].x) * bf16_hi(wv.x)),
                              pack_bf16x2(bf16_lo(g[i].y) * bf16_lo(wv.y), bf16_hi(g[i].y) * bf16_hi(wv.y)));
            s[0] += bf16_lo(g[i].x) * bf16_lo(xv[i].x);
            s[1] += bf16_hi(g[i].x) * bf16_hi(xv[i].x);
            s[2] += bf16_lo(g[i].y) * bf16_lo(xv[i].y);
            s[3] += bf16_hi(g[i].y) * bf16_hi(xv[i].y);
        }
    }
    const float k = ((-0.5f * row_sum(s)) * ((r * r) * r)) * (1.0f / (float)dim);
    uint2* out = reinterpret_cast<uint2*>(dx + row * dim);
    const auto grad = [&](float gf, float xf) { return gf * r + k * (2.0f * xf); };
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = lane + i * 64;
        if (c < nchunk)
            out[c] = make_uint2(pack_bf16x2(grad(bf16_lo(g[i].x), bf16_lo(xv[i].x)), grad(bf16_hi(g[i].x), bf16_hi(xv[i].x))),
                                pack_bf16x2(grad(bf16_lo(g[i].y), bf16_lo(xv[i].y)), grad(bf16_hi(g[i].y), bf16_hi(xv[i].y))));
    }
}

// out[c] = bf16(sum over g of partial[g][c]), 32 columns per workgroup of 1024 threads: 8 threads side by side take 4 columns
// each (a 128-byte line of a row), 128 of them every 128th row, and LDS adds those up
constexpr int SUM_COLS = 32, SUM_ROWS = 128;
__global__ __launch_bounds__(1024) void column_sum_kernel(const float* __restrict__ partial, int groups, int dim, uint16_t* __restrict__ out) {
    __shared__ float4 acc[SUM_ROWS][8];
    const int c4 = threadIdx.x & 7, r0 = threadIdx.x >> 3;
    const float* p = partial + (int64_t)blockIdx.x * SUM_COLS + c4 * 4;
    float4 s = make_float4(0, 0, 0, 0);
#pragma unroll 8
    for (int g = r0; g < groups; g += SUM_ROWS) {
        const float4 v = *reinterpret_cast<const float4*>(p + (int64_t)g * dim);
        s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    acc[r0][c4] = s;
    __syncthreads();
#pragma unroll
    for (int h = SUM_ROWS / 2; h; h >>= 1) {
        if (r0 < h) {
            const float4 a = acc[r0][c4], b = acc[r0 + h][c4];
            acc[r0][c4] = make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
        }
        __syncthreads();
    }
    if (r0 == 0) {
        const float4 a = acc[0][c4];
        *reinterpret_cast<uint2*>(out + (int64_t)blockIdx.x * SUM_COLS + c4 * 4) = make_uint2(pack_bf16x2(a.x, a.y), pack_bf16x2(a.z, a.w));
    }
}

// cos and sin [seq][half] of position * base^(-2 j / head_dim), rounded to bf16 at the end, with the roundings of the torch expression
// (decoder.rope_tables): one launch for its twelve, which the host took 52 us to launch (8 now).
__global__ __launch_bounds__(THREADS) void rope_tables_kernel(uint16_t* __restrict__ cosv, uint16_t* __restrict__ sinv, int64_t items, int half, float inv_dim, float base) {
    const int64_t i = (int64_t)blockIdx.x * THREADS + threadIdx.x;
    if (i >= items) return;
    const int64_t pos = i / half;
    const int j = (int)(i - pos * half);
    const float angle = (float)pos * (1.0f / powf(base, (float)(2 * j) * inv_dim));
    cosv[i] = (uint16_t)f32_to_bf16_bits(cosf(angle));
    sinv[i] = (uint16_t)f32_to_bf16_bits(sinf(angle));
}

// Rotary embedding of q and k [tokens][heads * D], the two halves of a head's D elements rotated against each other by the
// angle of (position, element); position = token % seq.  One workgroup per token; a thread takes 8 elements of each half.
// 16384 x 4096, q and k together: 83 us (6.4 TB/s), about 700 us in 12 launches before.
// sign = 1, or -1 for the backward (the transposed rotation).  Products and their sum are rounded to bf16 one by one.
__global__ __launch_bounds__(THREADS) void rope_kernel(const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, uint16_t* __restrict__ oq,
                                                       uint16_t* __restrict__ ok, const uint16_t* __restrict__ cosv, const uint16_t* __restrict__ sinv,
                                                       int seq, int heads, int half, float sign) {
    const int64_t t = blockIdx.x;
    const int per_head = half >> 3, items = heads * per_head, dim = heads * half * 2;
    const int pos = (int)(t % seq);
    const uint16_t* const in = blockIdx.y ? k : q;
    uint16_t* const out = blockIdx.y ? ok : oq;
    for (int i = threadIdx.x; i < items; i += THREADS) {
        const int head = i / per_head, j = i - head * per_head;
        const int64_t at = t * dim + (int64_t)head * half * 2 + j * 8;
        float a[8], b[8], c[8], s[8], ac[8], bs[8], bc[8], as[8];
        unpack8(*reinterpret_cast<const uint4*>(in + at), a);
        unpack8(*reinterpret_cast<const uint4*>(in + at + half), b);
        unpack8(*reinterpret_cast<const uint4*>(cosv + (int64_t)pos * half + j * 8), c);
        unpack8(*reinterpret_cast<const uint4*>(sinv + (int64_t)pos * half + j * 8), s);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float se = s[e] * sign;
            ac[e] = a[e] * c[e];
            bs[e] = b[e] * se;
            bc[e] = b[e] * c[e];
            as[e] = a[e] * se;
        }
        round8(ac); round8(bs); round8(bc); round8(as);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            a[e] = ac[e] - bs[e];
            b[e] = bc[e] + as[e];
        }
        *reinterpret_cast<uint4*>(out + at) = pack8(a);
        *reinterpret_cast<uint4*>(out + at + half) = pack8(b);
    }
}

// out = bf16(bf16(silu(gate)) * up), 8 elements per thread; 16384 x 14336: 256 us (5.5 TB/s), 410 us in two launches before
__global__ __launch_bounds__(THREADS) void swiglu_kernel(const uint16_t* __restrict__ gate, const uint16_t* __restrict__ up, uint16_t* __restrict__ out, int64_t chunks) {
    const int64_t i = (int64_t)blockIdx.x * THREADS + threadIdx.x;
    if (i >= chunks) return;
    float g[8], u[8];
    unpack8(reinterpret_cast<const uint4*>(gate)[i], g);
    unpack8(reinterpret_cast<const uint4*>(up)[i], u);
#pragma unroll
    for (int e = 0; e < 8; ++e) g[e] = g[e] / (1.0f + expf(-g[e]));
    round8(g);
#pragma unroll
    for (int e = 0; e < 8; ++e) g[e] = g[e] * u[e];
    reinterpret_cast<uint4*>(out)[i] = pack8(g);
}

// 16384 x 14336: 412 us (5.7 TB/s), 690 us in three launches before.
// dup = bf16(d * bf16(silu(gate))), dgate = bf16(ds * s * (1 + gate * (1 - s))) with s = sigmoid(gate), ds = bf16(d * up)
__global__ __launch_bounds__(THREADS) void swiglu_bwd_kernel(const uint16_t* __restrict__ d, const uint16_t* __restrict__ gate, const uint16_t* __restrict__ up,
                                                             uint16_t* __restrict__ dgate, uint16_t* __restrict__ dup, int64_t chunks) {
    const int64_t i = (int64_t)blockIdx.x * THREADS + threadIdx.x;
    if (i >= chunks) return;
    float df[8], g[8], u[8], s[8], silu[8];
    unpack8(reinterpret_cast<const uint4*>(d)[i], df);
    unpack8(reinterpret_cast<const uint4*>(gate)[i], g);
    unpack8(reinterpret_cast<const uint4*>(up)[i], u);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float t = 1.0f + expf(-g[e]);
        s[e] = 1.0f / t;
        silu[e] = g[e] / t;
        u[e] = df[e] * u[e];
    }
    round8(silu);
    round8(u);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        silu[e] = df[e] * silu[e];
        u[e] = u[e] * s[e] * (1.0f + g[e] * (1.0f - s[e]));
    }
    reinterpret_cast<uint4*>(dup)[i] = pack8(silu);
    reinterpret_cast<uint4*>(dgate)[i] = pack8(u);
}

int check_norm(const char* fn, int64_t rows, int64_t dim) {
    if (rows <= 0 || rows > 0x7fffffff || dim <= 0 || dim % SUM_COLS || dim > NORM_MAX_DIM)
        return fail(TI8_ERR_SHAPE, "%s: need 0<rows<2^31 and dim a multiple of %d up to %d; got rows=%lld dim=%lld", fn, SUM_COLS, NORM_MAX_DIM, (long long)rows, (long long)dim);
    return TI8_OK;
}

// f(loads per lane of a row of `dim` elements)
template <class F>
void with_chunks(int64_t dim, F f) {
    if (dim <= NORM_STEP) f(std::integral_constant<int, 8>{});
    else if (dim <= 2 * NORM_STEP) f(std::integral_constant<int, 16>{});
    else f(std::integral_constant<int, 32>{});
}

}  // namespace
int sum_partials(const char* fn, const float* partial, int groups, int64_t dim, void* out, hipStream_t st) {
    hipLaunchKernelGGL(column_sum_kernel, dim3((unsigned)(dim / SUM_COLS)), dim3(1024), 0, st, partial, groups, (int)dim, static_cast<uint16_t*>(out));
    return check_launch(fn);
}

}  // namespace ti8

using namespace ti8;

extern "C" int ti8_rmsnorm(const void* x, const void* w, void* y, float* rstd, int64_t rows, int64_t dim, float eps, ti8_stream_t stream) {
    const char* fn = "ti8_rmsnorm";
    if (!x || !w || !y || !rstd) return fail(TI8_ERR_NULL, "%s: x, w, y and rstd are required", fn);
    if (int e = check_norm(fn, rows, dim)) return e;
    if (!aligned16(x) || !aligned16(w) || !aligned16(y)) return fail(TI8_ERR_ALIGN, "%s: x, w and y must be 16-byte aligned", fn);
    with_chunks(dim, [&](auto nv) {
        hipLaunchKernelGGL((rmsnorm_kernel<decltype(nv)::value>), dim3((unsigned)((rows + 3) / 4)), dim3(THREADS), 0, static_cast<hipStream_t>(stream),
                           static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w), static_cast<uint16_t*>(y), rstd, rows, (int)dim, eps);
    });
    return check_launch(fn);
}

// the products, then the partial sums of their column sums
static int64_t norm_products_bytes(int64_t rows, int64_t dim) { return (rows * dim * 2 + 255) / 256 * 256; }

extern "C" int64_t ti8_rmsnorm_bwd_workspace(int64_t rows, int64_t dim) {
    if (check_norm("ti8_rmsnorm_bwd_workspace", rows, dim)) return -1;
    const int64_t sums = ti8_column_sum_workspace(rows, dim);
    return sums < 0 ? -1 : norm_products_bytes(rows, dim) + sums;
}

extern "C" int ti8_rmsnorm_bwd(const void* dy, const void* x, const void* w, const float* rstd, void* dx, void* dw, void* workspace, int64_t rows,
                               int64_t dim, ti8_stream_t stream) {
    const char* fn = "ti8_rmsnorm_bwd";
    if (!dy || !x || !w || !rstd || !dx || !workspace) return fail(TI8_ERR_NULL, "%s: dy, x, w, rstd, dx and workspace are required", fn);
    if (int e = check_norm(fn, rows, dim)) return e;
    if (!aligned16(dy) || !aligned16(x) || !aligned16(w) || !aligned16(dx) || !aligned16(dw) || !aligned16(workspace))
        return fail(TI8_ERR_ALIGN, "%s: dy, x, w, dx, dw and workspace must be 16-byte aligned", fn);
    with_chunks(dim, [&](auto nv) {
        hipLaunchKernelGGL((rmsnorm_bwd_kernel<decltype(nv)::value>), dim3((unsigned)((rows + 3) / 4)), dim3(THREADS), 0, static_cast<hipStream_t>(stream),
                           static_cast<const uint16_t*>(dy), static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w), rstd, static_cast<uint16_t*>(dx),
                           static_cast<uint16_t*>(workspace), rows, (int)dim);
    });
    if (int e = check_launch(fn)) return e;
    return dw ? ti8_column_sum(workspace, dim, dw, static_cast<char*>(workspace) + norm_products_bytes(rows, dim), rows, dim, stream) : TI8_OK;
}

extern "C" int ti8_rope(const void* q, const void* k, void* out_q, void* out_k, const void* cos_table, const void* sin_table, int64_t tokens, int64_t seq,
                        int64_t heads, int64_t head_dim, int backward, ti8_stream_t stream) {
    const char* fn = "ti8_rope";
    if (!q || !k || !out_q || !out_k || !cos_table || !sin_table) return fail(TI8_ERR_NULL, "%s: q, k, their outputs and the tables are required", fn);
    if (tokens <= 0 || tokens > 0x7fffffff || seq <= 0 || seq > tokens || heads <= 0 || head_dim <= 0 || head_dim % 16 || heads * head_dim > 0x00ffffff || heads > 0x00ffffff)
        return fail(TI8_ERR_SHAPE, "%s: need 0<seq<=tokens<2^31, heads>0, head_dim a positive multiple of 16; got tokens=%lld seq=%lld heads=%lld head_dim=%lld", fn,
                    (long long)tokens, (long long)seq, (long long)heads, (long long)head_dim);
    if (!aligned16(q) || !aligned16(k) || !aligned16(out_q) || !aligned16(out_k) || !aligned16(cos_table) || !aligned16(sin_table))
        return fail(TI8_ERR_ALIGN, "%s: every tensor must be 16-byte aligned", fn);
    hipLaunchKernelGGL(rope_kernel, dim3((unsigned)tokens, 2), dim3(THREADS), 0, static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(q),
                       static_cast<const uint16_t*>(k), static_cast<uint16_t*>(out_q), static_cast<uint16_t*>(out_k), static_cast<const uint16_t*>(cos_table),
                       static_cast<const uint16_t*>(sin_table), (int)seq, (int)heads, (int)(head_dim / 2), backward ? -1.0f : 1.0f);
    return check_launch(fn);
}

extern "C" int ti8_rope_tables(void* cos_table, void* sin_table, int64_t seq, int64_t head_dim, float base, ti8_stream_t stream) {
    const char* fn = "ti8_rope_tables";
    if (!cos_table || !sin_table) return fail(TI8_ERR_NULL, "%s: both tables are required", fn);
    const int64_t half = (head_dim + 1) / 2, items = seq * half;
    if (seq <= 0 || seq > 0x3fffffff || head_dim <= 0 || head_dim > 0x00ffffff || (items + THREADS - 1) / THREADS > 0x7fffffff)
        return fail(TI8_ERR_SHAPE, "%s: need 0<seq<2^30 and 0<head_dim<2^24; got seq=%lld head_dim=%lld", fn, (long long)seq, (long long)head_dim);
    hipLaunchKernelGGL(rope_tables_kernel, dim3((unsigned)((items + THREADS - 1) / THREADS)), dim3(THREADS), 0, static_cast<hipStream_t>(stream),
                       static_cast<uint16_t*>(cos_table), static_cast<uint16_t*>(sin_table), items, (int)half, 1.0f / (float)head_dim, base);
    return check_launch(fn);
}

static int check_swiglu(const char* fn, int64_t n) {
    if (n <= 0 || n % 8 || n / (8 * THREADS) >= 0x7fffffff) return fail(TI8_ERR_SHAPE, "%s: need a positive multiple of 8 elements, got %lld", fn, (long long)n);
    return TI8_OK;
}

extern "C" int ti8_swiglu(const void* gate, const void* up, void* out, int64_t n, ti8_stream_t stream) {
    const char* fn = "ti8_swiglu";
    if (!gate || !up || !out) return fail(TI8_ERR_NULL, "%s: gate, up and out are required", fn);
    if (int e = check_swiglu(fn, n)) return e;
    if (!aligned16(gate) || !aligned16(up) || !aligned16(out)) return fail(TI8_ERR_ALIGN, "%s: every tensor must be 16-byte aligned", fn);
    hipLaunchKernelGGL(swiglu_kernel, dim3((unsigned)((n / 8 + THREADS - 1) / THREADS)), dim3(THREADS), 0, static_cast<hipStream_t>(stream),
                       static_cast<const uint16_t*>(gate), static_cast<const uint16_t*>(up), static_cast<uint16_t*>(out), n / 8);
    return check_launch(fn);
}

extern "C" int ti8_swiglu_bwd(const void* d, const void* gate, const void* up, void* dgate, void* dup, int64_t n, ti8_stream_t stream) {
    const char* fn = "ti8_swiglu_bwd";
    if (!d || !gate || !up || !dgate || !dup) return fail(TI8_ERR_NULL, "%s: d, gate, up, dgate and dup are required", fn);
    if (int e = check_swiglu(fn, n)) return e;
    if (!aligned16(d) || !aligned16(gate) || !aligned16(up) || !aligned16(dgate) || !aligned16(dup)) return fail(TI8_ERR_ALIGN, "%s: every tensor must be 16-byte aligned", fn);
    hipLaunchKernelGGL(swiglu_bwd_kernel, dim3((unsigned)((n / 8 + THREADS - 1) / THREADS)), dim3(THREADS), 0, static_cast<hipStream_t>(stream),
                       static_cast<const uint16_t*>(d), static_cast<const uint16_t*>(gate), static_cast<const uint16_t*>(up), static_cast<uint16_t*>(dgate),
                       static_cast<uint16_t*>(dup), n / 8);
    return check_launch(fn);
}
