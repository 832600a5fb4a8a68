// Shared host/device helpers of libti8 (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>
#include <atomic>

#include "../../include/ti8.h"

namespace ti8 {

// ---- error reporting (host) ------------------------------------------------------
char* err_buf();  // thread-local buffer behind ti8_last_error()

inline int fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(err_buf(), 512, fmt, ap);
    va_end(ap);
    return code;
}

inline int check_launch(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(TI8_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
    return TI8_OK;
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// ---- per-device one-time set-up (host) ---------------------------------------------
inline int current_device() {
    int dev = 0;
    (void)hipGetDevice(&dev);
    return dev;
}

// One bit per device index: whether a kernel's dynamic LDS limit has been raised there.  The call is idempotent,
// so two threads that race through it only repeat it.  ti8_init() goes through every kernel that needs it, so that
// nothing of the kind is left for the first launch.
struct OncePerDevice {
    std::atomic<uint64_t> done{0};
};
inline hipError_t raise_lds_limit(OncePerDevice& once, const void* kern, int bytes) {
    const uint64_t bit = 1ull << (current_device() & 63);
    if (once.done.load(std::memory_order_acquire) & bit) return hipSuccess;
    const hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess) once.done.fetch_or(bit, std::memory_order_release);
    else (void)hipGetLastError();
    return e;
}

// Compute units of the current device (looked up once per device).
int device_cu_count();

// What ti8_init() calls: the per-device set-up of each source file's kernels (LDS limits, device symbols).
int init_gemm_kernels();
int init_chain_kernel();
int init_skinny_kernels();
int init_mid_kernels();
int init_fwht_kernels();
int init_attention_kernels();
int init_quant_scratch();

// ---- pieces of quant.hip and fwht.hip that the layer calls (step.hip) use ----------
// `valid_rows` (of R, the rest counts as zeros and is not read): an activation whose token count is no multiple of the tile
// needs no zero-padded copy.  NULL / R: all of them.
int quant_block_multi_valid(const ti8_qblock_operand* operands, const int64_t* valid_rows, int count, int qflags, int inv_mode, ti8_stream_t stream);
// An operand quantised by rows (q [R][C]) and by columns (qT [C][R]).  Scratch: `maxima` R + C words; `partial` quant_maxima_words words
// (in no more than the operand's own bytes) or null, which leaves the call to the atomics form.
struct QRowColOperand {
    const void* x;
    int64_t ldx;
    int8_t* q;
    float* s_row;
    int8_t* qT;
    float* s_col;
    unsigned int *maxima, *partial;
    int64_t R, valid_rows, C;
    bool maxima_only = false;       // the conversion is somebody else's (with `partial`, not in the atomics form)
};
int64_t quant_maxima_words(int64_t R, int64_t C);
// whether the maxima of so many bytes of such operands are collected in one launch; else `partial` is not looked at
bool quant_together(int64_t bytes);
// An operand quantised by rows alone, dense codes
struct QRowOperand {
    const void* x;
    int64_t ldx;
    int8_t* q;
    float* s;
    int64_t R, C;
};
// Block-quantised operands, operands quantised both ways (up to 4 and 3) and one quantised by rows (or null) in two launches, one where there
// are none of the second kind
int quant_call(const char* fn, const ti8_qblock_operand* blocks, const int64_t* block_rows, int nblocks, const QRowColOperand* both, int nboth,
               const QRowOperand* rows, int qflags, int inv_mode, ti8_stream_t stream);
// An operand rotated by H_128 and quantised, dense codes: by 128 x 128 blocks or by rows, rotated along the rows of x [R][C]; by blocks of x^T or by
// the columns of x (`maxima`: C words of scratch), rotated along the columns, q [C][R].  Up to QHAD_MAX of them in a launch (a clearing one and a
// conversion more with columns)
enum { QHAD_BLOCKS = 0, QHAD_BLOCKS_T = 1, QHAD_COLUMNS = 2, QHAD_ROWS = 3, QHAD_MAX = 6 };
struct QHadOperand {
    const void* x;
    int64_t ldx;
    int8_t* q;
    float* s;
    int64_t R, valid_rows, C;       // by rows: R rows
    int kind;
    unsigned int* maxima;
};
int quant_had_call(const char* fn, const QHadOperand* operands, int count, int qflags, int inv_mode, ti8_stream_t stream);
int quant_col_t_valid(const void* x, int64_t ldx, int8_t* qT, int64_t ldqt, float* s, float* ws, int64_t R, int64_t valid_rows, int64_t C,
                      int qflags, int inv_mode, ti8_stream_t stream);
int quant_block_had128_valid(const void* x, int64_t bsx, int64_t ldx, int8_t* q, int64_t bsq, int64_t ldq, float* s, int64_t ssb, int64_t ssr,
                             int64_t ssc, int64_t B, int64_t R, int64_t valid_rows, int64_t C, int along_rows, int qflags, int inv_mode,
                             ti8_stream_t stream);
// An operand rotated over the whole row by H and quantised by rows: x [R][C] (R its rows that exist), q [R][C]; or, `transposed`, x^T with x [R][C]
// transposed into `scratch` first, q [C][R].  Codes dense; up to QFWHT_MAX of a call, `together` (each with scratch of its own) in a launch per
// length and one for the transposes
enum { QFWHT_MAX = 6 };
struct QFwhtOperand {
    const void* x;
    int64_t ldx;
    int8_t* q;
    float* s;
    int64_t R, valid_rows, C;
    bool transposed;
    void* scratch;
};
int64_t next_pow2_128(int64_t v);       // and at least 128
int quant_fwht_call(const char* fn, const QFwhtOperand* operands, int count, bool together, int qflags, int inv_mode, ti8_stream_t stream);
int fwht_t_quant_row_valid(const void* x, int64_t ldx, void* scratch, int8_t* q, int64_t ldq, float* s, int64_t R, int64_t valid_rows, int64_t C,
                           int qflags, int inv_mode, ti8_stream_t stream);
// ti8_gemm_i8_nt with a bias, which the epilogue adds; y += bias behind the GEMMs of a whole step (bias.hip)
int gemm_nt_bias(const ti8_gemm_problem& p, const void* bias, int gemm_flags, ti8_stream_t stream);
// gemm.hip: the GEMMs of a call on few tokens as one launch, those that go into it (see there)
int gemm_nt_few(const ti8_gemm_problem* problems, int count, bool backward, const void* bias, int gemm_flags, bool* launched, ti8_stream_t stream);
// Y of 1 to 8 rows of bf16 that the GEMM's kernel quantises itself (`p` describes what it would be with the quantiser apart); *done tells
// whether it was launched
int gemm_nt_decode(const ti8_gemm_problem& p, const void* X, int64_t ldx, int64_t rows, const void* bias, int gemm_flags, bool* done, ti8_stream_t stream);
// y = bf16(bf16(c + b) + y) on [rows][cols], b and c dense; without c: bf16(b + y) (bias.hip)
int add_rows(const char* fn, void* y, int64_t ldy, const void* b, const void* c, int64_t rows, int64_t cols, ti8_stream_t stream);
// Y, dX and dW of a block-channel step on up to 32 of up to 256 padded tokens from the weight itself, W [N][K], whose maxima are in `w.partial`, and where that is
// taken
bool gemm_raw_weight_takes(int64_t tokens, int64_t K, int64_t N, int64_t ldw);
int gemm_nt_raw_weight(const ti8_gemm_problem* problems, const QRowColOperand& w, int64_t tokens, ti8_stream_t stream);
int add_bias(void* y, int64_t ldy, const void* bias, int64_t rows, int64_t cols, ti8_stream_t stream);
// out[c] = bf16(sum over g of partial[g][c]), dim a multiple of 32 (decoder.hip)
int sum_partials(const char* fn, const float* partial, int groups, int64_t dim, void* out, hipStream_t st);

// ---- which kernel served the last GEMM call of this thread (ti8_last_gemm_kernel) ---
void note_gemm_kernel(int kind, int bm, int bn, int epi, int form = TI8_FORM_PLAIN);

// ---- device helpers --------------------------------------------------------------
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// fp32 -> bf16 bits, round to nearest even (finite values; NaN stays NaN)
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
    u += 0x7fffu + ((u >> 16) & 1u);
    return u >> 16;
}

// two fp32 -> two bf16 in one dword (`lo` in the low half), round to nearest even: gfx950's
// v_cvt_pk_bf16_f32, same results as f32_to_bf16_bits for every finite value and infinity
typedef __bf16 ti8_bf16x2 __attribute__((ext_vector_type(2)));
typedef float ti8_f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
    const ti8_f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, ti8_bf16x2));
}

// sums of two pairs of bf16, each rounded to bf16
__device__ __forceinline__ uint32_t add_bf16x2(uint32_t a, uint32_t b) { return pack_bf16x2(bf16_lo(a) + bf16_lo(b), bf16_hi(a) + bf16_hi(b)); }

// Reductions over lanes with DPP moves (no LDS traffic).
// max(v, v of the lane that DPP control CTRL names) in the rows of ROW_MASK; other lanes keep v
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ float dpp_max(float v) {
    const int i = __float_as_int(v);
    return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(i, i, CTRL, ROW_MASK, 0xf, false)));
}

// max over each half-wave of 32 lanes without LDS traffic; valid in lanes 16-31 and 48-63.
// quad_perm lane^1, lane^2, then row_half_mirror and row_mirror (all 16 lanes of a row agree),
// then row_bcast:15 into rows 1 and 3 (lane 15 of the row before).
__device__ __forceinline__ float half_wave_max_hi(float v) {
    v = dpp_max<0xB1>(v);
    v = dpp_max<0x4E>(v);
    v = dpp_max<0x141>(v);
    v = dpp_max<0x140>(v);
    return dpp_max<0x142, 0xA>(v);
}

// max over the 16 lanes of a DPP row, in all of them
__device__ __forceinline__ float row16_max(float v) {
    v = dpp_max<0xB1>(v);
    v = dpp_max<0x4E>(v);
    v = dpp_max<0x141>(v);
    return dpp_max<0x140>(v);
}

// max over the wave, in every lane: half_wave_max_hi, row_bcast:31 into rows 2 and 3 (lane 63 then
// holds the maximum), and a read of lane 63
__device__ __forceinline__ float wave_max(float v) {
    v = dpp_max<0x143, 0xC>(half_wave_max_hi(v));
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

}  // namespace ti8
