// The bias of a linear layer: adding it behind the GEMMs of a whole step (a GEMM launched alone does that in its epilogue), and its
// gradient, the column sums of dY.
#include "ti8_common.h"
#include "index_math.h"

namespace ti8 {

namespace {

constexpr int THREADS = 256;
constexpr int SUM_COLS = 512;       // columns per workgroup of column_partial_kernel: 64 lanes x 8, a row's share is 1 KiB

}  // namespace

// y[r][c] = bf16(y[r][c] + bias[c]), 8 columns per thread.  Streams y once each way; torch's broadcast add reads the bias through
// its strided path: 1500 x 5632 (34 MB) 11 us, this 6.
__global__ __launch_bounds__(THREADS) void add_bias_kernel(uint16_t* __restrict__ y, int64_t ldy, const uint16_t* __restrict__ bias, int rows, int chunks) {
    const int c = (int)blockIdx.x * THREADS + (int)threadIdx.x;      // group of 8 columns
    if (c >= chunks) return;
    const uint4 b = *reinterpret_cast<const uint4*>(bias + c * 8);
    const int r0 = (int)blockIdx.y * 4;
    uint16_t* const p = y + (int64_t)r0 * ldy + c * 8;
    uint4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (r0 + k < rows) v[k] = *reinterpret_cast<const uint4*>(p + (int64_t)k * ldy);
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (r0 + k < rows)
            *reinterpret_cast<uint4*>(p + (int64_t)k * ldy) =
                make_uint4(add_bf16x2(v[k].x, b.x), add_bf16x2(v[k].y, b.y), add_bf16x2(v[k].z, b.z), add_bf16x2(v[k].w, b.w));
}

// y = bf16(bf16(c + b) + y), 8 elements per thread: gradients of the same input.  Bound by HBM: 16384 x 4096, three of them 93 us (5.7 TB/s).
template <bool THREE>
__global__ __launch_bounds__(THREADS) void add_rows_kernel(uint16_t* __restrict__ y, int64_t ldy, const uint16_t* __restrict__ b, const uint16_t* __restrict__ c,
                                                           int64_t items, int per_row) {
    const int64_t i = (int64_t)blockIdx.x * THREADS + threadIdx.x;
    if (i >= items) return;
    const int64_t row = i / per_row;
    uint4* const to = reinterpret_cast<uint4*>(y + row * ldy + (i - row * per_row) * 8);
    const uint4 first = *to;
    uint4 v = reinterpret_cast<const uint4*>(b)[i];
    if (THREE) {
        const uint4 w = reinterpret_cast<const uint4*>(c)[i];
        v = make_uint4(add_bf16x2(w.x, v.x), add_bf16x2(w.y, v.y), add_bf16x2(w.z, v.z), add_bf16x2(w.w, v.w));
    }
    *to = make_uint4(add_bf16x2(v.x, first.x), add_bf16x2(v.y, first.y), add_bf16x2(v.z, first.z), add_bf16x2(v.w, first.w));
}

// partial[g][c] = sum of x[r][c] over rows r = g * per .. of workgroup row g: each of the four waves takes every fourth row, LDS
// adds their sums.  One read of x; the column sums of a [1500][5632] dY take 4 + 3 us in the two launches (torch's reduction with
// the two memory fills in front of it: 23).
__global__ __launch_bounds__(THREADS) void column_partial_kernel(const uint16_t* __restrict__ x, int64_t ldx, int rows, int per, int cols, float* __restrict__ partial) {
    __shared__ float acc[4][SUM_COLS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c0 = (int)blockIdx.x * SUM_COLS + lane * 8;
    const int r0 = (int)blockIdx.y * per, r1 = min(r0 + per, rows);
    float s[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) s[e] = 0.0f;
    if (c0 < cols) {
#pragma unroll 4
        for (int r = r0 + wave; r < r1; r += 4) {
            const uint4 v = *reinterpret_cast<const uint4*>(x + (int64_t)r * ldx + c0);
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s[2 * e] += bf16_lo(w[e]);
                s[2 * e + 1] += bf16_hi(w[e]);
            }
        }
    }
#pragma unroll
    for (int e = 0; e < 8; e += 4) *reinterpret_cast<float4*>(&acc[wave][lane * 8 + e]) = make_float4(s[e], s[e + 1], s[e + 2], s[e + 3]);
    __syncthreads();
    const int c = threadIdx.x * 2, col = (int)blockIdx.x * SUM_COLS + c;
    if (col >= cols) return;
    *reinterpret_cast<float2*>(partial + (int64_t)blockIdx.y * cols + col) =
        make_float2((acc[0][c] + acc[1][c]) + (acc[2][c] + acc[3][c]), (acc[0][c + 1] + acc[1][c + 1]) + (acc[2][c + 1] + acc[3][c + 1]));
}

// The same in one launch where a workgroup can take all rows of 32 columns in the time that a second launch takes: 4 lanes to a row's 64 bytes,
// 256 rows at a time, whose sums meet across the lanes of a wave and then of the 16 waves, in a fixed order.  Strips that share cache
// lines go to one XCD.  idx::column_sum_narrow says where, with the figures.
constexpr int NARROW_COLS = 32, NARROW_THREADS = 1024;
__global__ __launch_bounds__(NARROW_THREADS) void column_sum_narrow_kernel(const uint16_t* __restrict__ x, int64_t ldx, int rows, int strips, uint16_t* __restrict__ out) {
    __shared__ float acc[NARROW_THREADS / 64][NARROW_COLS];
    const int strip = idx::column_strip((int)blockIdx.x, strips);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint16_t* const p = x + strip * NARROW_COLS + (lane & 3) * 8;
    float s[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) s[e] = 0.0f;
#pragma unroll 8
    for (int r = (int)threadIdx.x >> 2; r < rows; r += NARROW_THREADS / 4) {
        const uint4 v = *reinterpret_cast<const uint4*>(p + (int64_t)r * ldx);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            s[2 * e] += bf16_lo(w[e]);
            s[2 * e + 1] += bf16_hi(w[e]);
        }
    }
#pragma unroll
    for (int m = 4; m < 64; m <<= 1)
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] += __shfl_xor(s[e], m, 64);
    if (lane < 4)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[wave][lane * 8 + e] = s[e];
    __syncthreads();
    if (threadIdx.x >= NARROW_COLS / 2) return;
    float a = 0.0f, b = 0.0f;
#pragma unroll
    for (int w = 0; w < NARROW_THREADS / 64; ++w) {
        a += acc[w][threadIdx.x * 2];
        b += acc[w][threadIdx.x * 2 + 1];
    }
    *reinterpret_cast<uint32_t*>(out + strip * NARROW_COLS + threadIdx.x * 2) = pack_bf16x2(a, b);
}

int add_bias(void* y, int64_t ldy, const void* bias, int64_t rows, int64_t cols, ti8_stream_t stream) {
    const int chunks = (int)(cols / 8);
    for (int64_t r = 0; r < rows; r += 4 * 65535) {     // a launch has at most 65535 workgroup rows
        const int64_t n = rows - r < 4 * 65535 ? rows - r : 4 * 65535;
        hipLaunchKernelGGL(add_bias_kernel, dim3((unsigned)((chunks + THREADS - 1) / THREADS), (unsigned)((n + 3) / 4)), dim3(THREADS), 0,
                           static_cast<hipStream_t>(stream), static_cast<uint16_t*>(y) + r * ldy, ldy, static_cast<const uint16_t*>(bias), (int)n, chunks);
        if (int e = check_launch("ti8_linear")) return e;
    }
    return TI8_OK;
}

int add_rows(const char* fn, void* y, int64_t ldy, const void* b, const void* c, int64_t rows, int64_t cols, ti8_stream_t stream) {
    const int64_t items = rows * (cols / 8), groups = (items + THREADS - 1) / THREADS;
    if (groups > 0x7fffffff) return fail(TI8_ERR_SHAPE, "%s: too many elements", fn);
    const auto kernel = c ? add_rows_kernel<true> : add_rows_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)groups), dim3(THREADS), 0, static_cast<hipStream_t>(stream), static_cast<uint16_t*>(y), ldy,
                       static_cast<const uint16_t*>(b), static_cast<const uint16_t*>(c), items, (int)(cols / 8));
    return check_launch(fn);
}

// Rows per workgroup: about 1024 workgroups, no fewer than 16 rows each (the partial sums are then at most an eighth of the bytes read)
static int64_t rows_per_group(int64_t rows, int64_t cols) {
    const int64_t strips = (cols + SUM_COLS - 1) / SUM_COLS;
    const int64_t wanted = strips < 1024 ? 1024 / strips : 1;
    const int64_t per = (rows + wanted - 1) / wanted;
    return per < 16 ? 16 : per;
}

static bool column_sum_takes(int64_t rows, int64_t cols) {
    return rows > 0 && rows <= 0x3fffffff && cols > 0 && cols % 32 == 0 && cols <= 0x3fffffff;
}

}  // namespace ti8

using namespace ti8;

extern "C" int64_t ti8_column_sum_workspace(int64_t rows, int64_t cols) {
    if (!column_sum_takes(rows, cols)) return -1;
    const int64_t per = rows_per_group(rows, cols);
    return (rows + per - 1) / per * cols * (int64_t)sizeof(float);
}

extern "C" int ti8_column_sum(const void* x, int64_t ldx, void* out, void* workspace, int64_t rows, int64_t cols, ti8_stream_t stream) {
    const char* fn = "ti8_column_sum";
    if (!x || !out || !workspace) return fail(TI8_ERR_NULL, "%s: x, out and the workspace are required", fn);
    if (!column_sum_takes(rows, cols) || ldx < cols)
        return fail(TI8_ERR_SHAPE, "%s: need rows>0, cols a positive multiple of 32 and ldx>=cols; got rows=%lld cols=%lld ldx=%lld", fn, (long long)rows, (long long)cols, (long long)ldx);
    if (!aligned16(x) || ldx % 8 || !aligned16(out) || !aligned16(workspace)) return fail(TI8_ERR_ALIGN, "%s: x, out and the workspace must be 16-byte aligned, ldx a multiple of 8", fn);
    if (idx::column_sum_narrow(rows, cols)) {
        const int strips = (int)(cols / NARROW_COLS);
        hipLaunchKernelGGL(column_sum_narrow_kernel, dim3((unsigned)strips), dim3(NARROW_THREADS), 0, static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(x), ldx,
                           (int)rows, strips, static_cast<uint16_t*>(out));
        return check_launch(fn);
    }
    const int64_t per = rows_per_group(rows, cols);
    const int groups = (int)((rows + per - 1) / per);
    float* const partial = static_cast<float*>(workspace);
    hipStream_t st = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(column_partial_kernel, dim3((unsigned)((cols + SUM_COLS - 1) / SUM_COLS), (unsigned)groups), dim3(THREADS), 0, st,
                       static_cast<const uint16_t*>(x), ldx, (int)rows, (int)per, (int)cols, partial);
    if (int e = check_launch(fn)) return e;
    return sum_partials(fn, partial, groups, cols, out, st);
}
