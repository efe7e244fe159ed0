// float_route.hip - kern.MatMul's float route for one row of activations.
//
// internal/kern/kern.go:185-196 of github.com/xattribution/gorelaxor sends a
// product to the float route when the weight keeps its rows and there is
// one row of activations (m = 1 < intMinM), or when the weight is float32:
// gemvRows (gemm.go:195-259) runs the weight's rows in groups of four with
// the assembly kernels and the last partial group with the Go ones, then
// adds the bias:
//   Q8_0  rows in whole groups of four: dot4q8avx (kernels_amd64.s:340-400):
//         per block, eight lanes l: t = w[l]*x[l], then three fmas with the
//         next 24 values, acc[l] = fma(t, d, acc[l]); HSUM at the end.
//         Other rows: dotQ8Go (kern.go:248-266): per block four running sums,
//         s += d*(a0+a1+a2+a3).
//   F32   rows in whole groups of four: dotF32x4 (dot4f32avx over k &^ 15,
//         dotF32Go over the rest); other rows dotF32Go.
// Several threads per output row, each keeping whole lane chains of the
// reference's assembly; the Q8_0 weight is the one packed for the int8
// route (grx_weight tiles), so one weight serves both routes.  x is staged
// in LDS.
#include "grx_float.h"
#include "grx_internal.h"
#include "grx_ln.h"

namespace {

// kern.Linear of a float32 weight (kern.go:185-201 -> ws.matmul,
// gemm.go:116-185) applied to each of B groups of `per` rows: with more than
// 16 rows, the rows in whole groups of six take k6x16 (kernels_amd64.s:5-88):
// from the bias (0 without one), each chunk of 256 k's fma chain (from zero)
// is added in.  This kernel computes that form for every row; the rows the
// reference sends to gemvRows are rewritten afterwards by
// f32_rows_gemv_kernel.
//
// On the float32 matrix cores: v_mfma_f32_16x16x4_f32 adds its four products
// to the accumulator one after another in k order with one rounding each,
// which is four steps of the chain (tests hold it to fmaf chains bit for bit,
// with subnormal sums, signed zeros, infinities and NaN).  A workgroup of
// WR x WC waves computes 16 WR RF x 16 WC CF outputs, KC k's a pass through
// LDS, double-buffered.  Within each 16 k's LDS holds k = 4s + l at place
// 4l + s, so that lane (i, l)'s operands of four instructions are one 16-byte
// read; rows are KC + 4 floats apart (those reads of 16 rows fall in distinct
// banks).  A k past the end is staged as the product of -0 and 0, which
// leaves every sum as it is.
//
// Bound by the matrix cores' float32 rate for many rows (128,512 x 256 x 256:
// 321 us on a VALU tile, 189 us here, 89 TFLOP/s), by the passes' memory latency for few, which is why those take
// longer passes and smaller tiles (512 x 256 x 256:
// 63 -> 6.3 us).
typedef float v4f __attribute__((ext_vector_type(4)));

template <int WR, int WC, int RF, int CF, int KC>
struct RowsTile {
    static constexpr int TM = 16 * WR * RF, TN = 16 * WC * CF, NT = 64 * WR * WC, LD = KC + 4;
    static constexpr int kBuf = (TM + TN) * LD;
    static constexpr size_t lds = 2 * kBuf * sizeof(float);
};

template <int WR, int WC, int RF, int CF, int KC, bool VEC>
__global__ __launch_bounds__(64 * WR *WC) void f32_rows_mfma_kernel(const float *__restrict__ x,
                                                                    const float *__restrict__ w,
                                                                    const float *__restrict__ bias,
                                                                    float *__restrict__ y, int rows, int n, int k) {
    using T = RowsTile<WR, WC, RF, CF, KC>;
    static_assert(256 % KC == 0 && KC % 16 == 0, "chunks of 256 k's end with a pass");
    constexpr int P = KC / 4;                                    // 16-byte pieces of a row and pass
    constexpr int NP = ((T::TM + T::TN) * P + T::NT - 1) / T::NT;  // pieces a thread
    extern __shared__ __align__(16) float st[];
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wave / WC, wc = wave % WC;
    const int r0 = blockIdx.y * T::TM, c0 = blockIdx.x * T::TN;
    float4 pre[NP];
    auto gload = [&](int k0) {
#pragma unroll
        for (int u = 0; u < NP; ++u) {
            const int e = tid + u * T::NT, row = e / P, kk = k0 + 4 * (e % P);
            const bool isx = row < T::TM;
            const float pad = isx ? -0.0f : 0.0f;
            float4 v = make_float4(pad, pad, pad, pad);
            const int g = isx ? r0 + row : c0 + row - T::TM;
            if (row < T::TM + T::TN && g < (isx ? rows : n)) {
                const float *p = (isx ? x : w) + (size_t)g * k + kk;
                if constexpr (VEC) {  // k % 4 == 0, 16-byte aligned rows
                    if (kk < k) v = *reinterpret_cast<const float4 *>(p);
                } else {
                    if (kk < k) v.x = p[0];
                    if (kk + 1 < k) v.y = p[1];
                    if (kk + 2 < k) v.z = p[2];
                    if (kk + 3 < k) v.w = p[3];
                }
            }
            pre[u] = v;
        }
    };
    auto lstore = [&](int buf) {
#pragma unroll
        for (int u = 0; u < NP; ++u) {
            const int e = tid + u * T::NT, row = e / P, pc = e % P;
            if (row >= T::TM + T::TN) break;
            float *d = st + buf * T::kBuf + row * T::LD + 16 * (pc >> 2) + (pc & 3);
            d[0] = pre[u].x;
            d[4] = pre[u].y;
            d[8] = pre[u].z;
            d[12] = pre[u].w;
        }
    };
    v4f acc[RF][CF], out[RF][CF];
#pragma unroll
    for (int j = 0; j < CF; ++j) {
        const int col = c0 + 16 * (wc * CF + j) + li;
        const float bj = (bias != nullptr && col < n) ? bias[col] : 0.f;
#pragma unroll
        for (int i = 0; i < RF; ++i) {
            out[i][j] = v4f{bj, bj, bj, bj};
            acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
        }
    }
    gload(0);
    lstore(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < k; k0 += KC) {
        const bool more = k0 + KC < k;
        if (more) gload(k0 + KC);
        const float *a0 = st + buf * T::kBuf + (wr * RF * 16 + li) * T::LD + 4 * lk;
        const float *b0 = st + buf * T::kBuf + (T::TM + wc * CF * 16 + li) * T::LD + 4 * lk;
#pragma unroll
        for (int g = 0; g < KC / 16; ++g) {
            float4 a[RF], b[CF];
#pragma unroll
            for (int i = 0; i < RF; ++i) a[i] = *reinterpret_cast<const float4 *>(a0 + 16 * i * T::LD + 16 * g);
#pragma unroll
            for (int j = 0; j < CF; ++j) b[j] = *reinterpret_cast<const float4 *>(b0 + 16 * j * T::LD + 16 * g);
            auto step = [&](auto get) {
#pragma unroll
                for (int i = 0; i < RF; ++i)
#pragma unroll
                    for (int j = 0; j < CF; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(get(a[i]), get(b[j]), acc[i][j], 0, 0, 0);
            };
            step([](const float4 &v) { return v.x; });
            step([](const float4 &v) { return v.y; });
            step([](const float4 &v) { return v.z; });
            step([](const float4 &v) { return v.w; });
        }
        if ((k0 + KC) % 256 == 0 || !more) {
#pragma unroll
            for (int i = 0; i < RF; ++i)
#pragma unroll
                for (int j = 0; j < CF; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        out[i][j][r] = __fadd_rn(acc[i][j][r], out[i][j][r]);
                        acc[i][j][r] = 0.f;
                    }
        }
        if (more) {
            lstore(buf ^ 1);  // the other buffer: its readers passed the last barrier
            __syncthreads();
            buf ^= 1;
        }
    }
#pragma unroll
    for (int i = 0; i < RF; ++i)
#pragma unroll
        for (int j = 0; j < CF; ++j) {
            const int col = c0 + 16 * (wc * CF + j) + li;
            if (col >= n) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = r0 + 16 * (wr * RF + i) + 4 * lk + r;
                if (row < rows) y[(size_t)row * n + col] = out[i][j][r];
            }
        }
}

template <int WR, int WC, int RF, int CF, int KC>
hipError_t launch_rows(hipStream_t st, const float *x, const float *w, const float *bias, float *y, int rows, int n,
                       int k) {
    using T = RowsTile<WR, WC, RF, CF, KC>;
    const bool vec = k % 4 == 0 && (((uintptr_t)x | (uintptr_t)w) & 15) == 0;
    auto kern = vec ? f32_rows_mfma_kernel<WR, WC, RF, CF, KC, true> : f32_rows_mfma_kernel<WR, WC, RF, CF, KC, false>;
    if constexpr (T::lds > 64 * 1024) {
        static GrxDeviceOnce once;
        const hipError_t e = grx_raise_lds(once, {(const void *)f32_rows_mfma_kernel<WR, WC, RF, CF, KC, true>,
                                                  (const void *)f32_rows_mfma_kernel<WR, WC, RF, CF, KC, false>},
                                           T::lds);
        if (e != hipSuccess) return e;
    }
    kern<<<dim3((n + T::TN - 1) / T::TN, (rows + T::TM - 1) / T::TM), T::NT, T::lds, st>>>(x, w, bias, y, rows, n, k);
    return hipGetLastError();
}

// The rows of each group that ws.matmul sends to gemvRows (gemm.go:
// 182-184, 195-259): rows lo..per-1 of every group (all of them when
// per <= 16): dotF32x4 for whole groups of four columns, dotF32Go for the
// rest, then the bias added (none without one).  Sixteen lanes per output,
// lane c running dot4f32avx's chain c (5 us at 2 rows x 256 x 256,
// 12 with one thread per output); the Go forms are lane 0's.
__global__ __launch_bounds__(256) void f32_rows_gemv_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                                            const float *__restrict__ bias, float *__restrict__ y,
                                                            int B, int per, int lo, int n, int k) {
    const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) >> 4, tail = (size_t)(per - lo);
    const int c = threadIdx.x & 15;
    if (i >= (size_t)B * tail * n) return;
    const int j = (int)(i % n);
    const size_t rr = i / n, row = rr / tail * per + lo + rr % tail;
    const float *xr = x + row * k, *wj = w + (size_t)j * k;
    const bool avx = j < (n & ~3);
    const int kk = avx ? k & ~15 : 0;
    float acc = 0.f;
#pragma unroll 8
    for (int t = c; t < kk; t += 16) acc = __fmaf_rn(xr[t], wj[t], acc);
    // S_l = A_l + B_l (chains l and 8 + l), h_l = S_l + S_{l+4}, (h0 + h1) + (h2 + h3)
    float o = __fadd_rn(acc, __shfl_xor(acc, 8, 16));
    o = __fadd_rn(o, __shfl_xor(o, 4, 16));
    o = __fadd_rn(o, __shfl_xor(o, 1, 16));
    o = __fadd_rn(o, __shfl_xor(o, 2, 16));
    if (c != 0) return;
    if (kk < k) {
        const float g = dot_go(xr + kk, wj + kk, k - kk);
        o = avx ? __fadd_rn(kk > 0 ? o : 0.f, g) : g;
    }
    y[row * n + j] = bias != nullptr ? __fadd_rn(o, bias[j]) : o;
}


// What happens to output row `row` of n after the bias (GrxFloatEpi):
// stored, stored through kern.SiLU (siluAVX's x/(EXP8(0-x)+1) for the rows
// below n &^ 7, siluGo's x/(1+expf(-x)) past them, kernels_amd64.go:241-250),
// or added to h as h += gate*o (unfused).
__device__ __forceinline__ void float_epilogue(const GrxFloatEpi &e, float o, int row, int n, float *y) {
    if (e.kind == GRX_FEPI_SILU) {
        const float a = __fdiv_rn(o, __fadd_rn(grx_exp8(__fsub_rn(0.f, o)), 1.f));
        const float b = __fdiv_rn(o, __fadd_rn(1.f, grx_expf_go(-o)));
        y[row] = row < (n & ~7) ? a : b;
    } else if (e.kind == GRX_FEPI_GATE) {
        y[row] = __fadd_rn(y[row], __fmul_rn(e.gate[row], o));
    } else {
        y[row] = o;
    }
}

// x into LDS: every thread's reads issued before its stores
__device__ __forceinline__ void stage_x(const float *__restrict__ x, int k, float *xs) {
    const int t = threadIdx.x, nt = blockDim.x;
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int i = t + u * nt;
        v[u] = i < k ? x[i] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int i = t + u * nt;
        if (i < k) xs[i] = v[u];
    }
    for (int i = t + 8 * nt; i < k; i += nt) xs[i] = x[i];
    __syncthreads();
}

// The row in xs normalized and modulated in place (GrxFloatPro).  Every
// workgroup does it for itself: a launch of its own in front of a 512 x 512
// product took 4.4 us and its gap for a row of 2 KB.
__device__ __forceinline__ void float_prologue(const GrxFloatPro &p, float *xs, int k) {
    __shared__ double red[48];  // ln_block_reduce
    double mean, inv;
    ln64_stats(xs, k, p.eps, red, mean, inv);
    for (int j = threadIdx.x; j < k; j += blockDim.x) {
        float o = (float)__dmul_rn(__dsub_rn((double)xs[j], mean), inv);
        if (p.w) o = __fadd_rn(__fmul_rn(o, p.w[j]), p.b[j]);
        xs[j] = __fadd_rn(__fmul_rn(o, __fadd_rn(1.f, p.scale[j])), p.shift[j]);
    }
    __syncthreads();
}

// Q8_0: the rows of one tile per workgroup (q8_float_row).
template <bool LN>
__global__ __launch_bounds__(256) void q8_float_gemv_kernel(const float *__restrict__ x, int k,
                                                            const int8_t *__restrict__ qs,
                                                            const uint16_t *__restrict__ ds, int nb, int n,
                                                            const float *__restrict__ bias, float *__restrict__ y,
                                                            GrxFloatEpi e, GrxFloatPro p) {
    extern __shared__ __align__(16) float xs[];
    stage_x(x, k, xs);
    if constexpr (LN) float_prologue(p, xs, k);
    int row;
    bool emit;
    float o = q8_float_row(xs, qs, ds, nb, n, blockIdx.x, row, emit);
    if (!emit) return;
    if (bias) o = __fadd_rn(o, bias[row]);
    float_epilogue(e, o, row, n, y);
}

// float32: eight threads per row; thread l keeps dot4f32avx's two chains
// A[l] and B[l] (16 values a step), S[l] = A[l]+B[l], and the HSUM is formed
// across the eight as (h0+h1)+(h2+h3), h_l = S[l]+S[l+4]; thread 0 adds
// dotF32Go over k past k &^ 15.  Rows past n &^ 3 take dotF32Go in thread 0.
template <bool LN>
__global__ __launch_bounds__(256) void f32_gemv_kernel(const float *__restrict__ x, int k,
                                                       const float *__restrict__ w, int n,
                                                       const float *__restrict__ bias, float *__restrict__ y,
                                                       GrxFloatEpi e, GrxFloatPro p) {
    extern __shared__ __align__(16) float xs[];
    stage_x(x, k, xs);
    if constexpr (LN) float_prologue(p, xs, k);
    const int row = blockIdx.x * 32 + (threadIdx.x >> 3), l = threadIdx.x & 7;
    const bool live = row < n, avx = row < (n & ~3);
    const float *wr = w + (size_t)row * k;
    const int kk = k & ~15;
    float A = 0.f, B = 0.f;
    if (live && avx) {
#pragma unroll 4
        for (int c = 0; c < kk; c += 16) {
            A = __fmaf_rn(xs[c + l], wr[c + l], A);
            B = __fmaf_rn(xs[c + 8 + l], wr[c + 8 + l], B);
        }
    }
    const float S = __fadd_rn(A, B);
    const float hl = __fadd_rn(S, __shfl_down(S, 4, 8));
    const float h1 = __shfl_down(hl, 1, 8), h2 = __shfl_down(hl, 2, 8), h3 = __shfl_down(hl, 3, 8);
    if (!live || l != 0) return;
    float o;
    if (avx) {
        o = kk > 0 ? __fadd_rn(__fadd_rn(hl, h1), __fadd_rn(h2, h3)) : 0.f;
        if (kk < k) o = __fadd_rn(o, dot_go(xs + kk, wr + kk, k - kk));
    } else {
        o = dot_go(xs, wr, k);
    }
    if (bias) o = __fadd_rn(o, bias[row]);
    float_epilogue(e, o, row, n, y);
}

constexpr int kMaxK = 32768;

}  // namespace

grx_status grx_float_gemv_q8(hipStream_t st, const grx_weight *w, const float *x, const float *bias, float *y,
                             GrxFloatEpi e, GrxFloatPro p) {
    if (w->cols > kMaxK) return grx_fail(GRX_ESIZE, "float route: %d columns (at most %d)", w->cols, kMaxK);
    if (w->rows == 0) return GRX_OK;
    auto kern = p.scale ? q8_float_gemv_kernel<true> : q8_float_gemv_kernel<false>;
    kern<<<w->tiles, 256, (size_t)w->cols * 4, st>>>(x, w->cols, w->qs, w->ds, w->nb, w->rows, bias, y, e, p);
    GRX_LAUNCHED("q8_float_gemv_kernel");
    return GRX_OK;
}

grx_status grx_float_gemv_f32(hipStream_t st, const float *w, int n, int k, const float *x, const float *bias,
                              float *y, GrxFloatEpi e, GrxFloatPro p) {
    if (k > kMaxK) return grx_fail(GRX_ESIZE, "float route: %d columns (at most %d)", k, kMaxK);
    if (n == 0) return GRX_OK;
    auto kern = p.scale ? f32_gemv_kernel<true> : f32_gemv_kernel<false>;
    kern<<<grx_ceil_div(n, 32), 256, (size_t)k * 4, st>>>(x, k, w, n, bias, y, e, p);
    GRX_LAUNCHED("f32_gemv_kernel");
    return GRX_OK;
}

// kern.Linear of one row through the float route, host buffers: the
// weight keeps its rows (no DropRows), so m = 1 takes gemvRows.
extern "C" grx_status grx_linear_q8_float(grx_ctx *ctx, float *dst, const float *x, const grx_weight *w,
                                          const float *bias) {
    if (!ctx || !dst || !x || !w) return grx_fail(GRX_EINVAL, "grx_linear_q8_float: NULL argument");
    const size_t xb = (size_t)w->cols * 4, yb = (size_t)w->rows * 4, bb = bias ? yb : 0;
    void *buf;
    grx_status s = grx_ctx_scratch(ctx, xb + yb + bb + 768, &buf);
    if (s != GRX_OK) return s;
    char *p = static_cast<char *>(buf);
    float *dx = reinterpret_cast<float *>(p), *dy = reinterpret_cast<float *>(p + (xb + 255) / 256 * 256);
    float *dbias = bias ? reinterpret_cast<float *>(p + (xb + 255) / 256 * 256 + (yb + 255) / 256 * 256) : nullptr;
    GRX_HIP(hipSetDevice(ctx->device));
    GRX_HIP(hipMemcpyAsync(dx, x, xb, hipMemcpyHostToDevice, ctx->stream));
    if (bias) GRX_HIP(hipMemcpyAsync(dbias, bias, bb, hipMemcpyHostToDevice, ctx->stream));
    if ((s = grx_float_gemv_q8(ctx->stream, w, dx, dbias, dy)) != GRX_OK) return s;
    GRX_HIP(hipMemcpyAsync(dst, dy, yb, hipMemcpyDeviceToHost, ctx->stream));
    GRX_HIP(hipStreamSynchronize(ctx->stream));
    return GRX_OK;
}

// The same for a float32 weight (rows x cols, row-major) in host memory.
extern "C" grx_status grx_linear_f32(grx_ctx *ctx, float *dst, const float *x, const float *w, int rows, int cols,
                                     const float *bias) {
    if (!ctx || !dst || !x || (!w && rows * cols > 0) || rows < 0 || cols < 0)
        return grx_fail(GRX_EINVAL, "grx_linear_f32: NULL argument or negative size");
    const size_t wb = (size_t)rows * cols * 4, xb = (size_t)cols * 4, yb = (size_t)rows * 4, bb = bias ? yb : 0;
    auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    void *buf;
    grx_status s = grx_ctx_scratch(ctx, up(wb) + up(xb) + up(yb) + up(bb) + 256, &buf);
    if (s != GRX_OK) return s;
    char *p = static_cast<char *>(buf);
    float *dw = reinterpret_cast<float *>(p), *dx = reinterpret_cast<float *>(p + up(wb));
    float *dy = reinterpret_cast<float *>(p + up(wb) + up(xb));
    float *dbias = bias ? reinterpret_cast<float *>(p + up(wb) + up(xb) + up(yb)) : nullptr;
    GRX_HIP(hipSetDevice(ctx->device));
    GRX_HIP(hipMemcpyAsync(dw, w, wb, hipMemcpyHostToDevice, ctx->stream));
    GRX_HIP(hipMemcpyAsync(dx, x, xb, hipMemcpyHostToDevice, ctx->stream));
    if (bias) GRX_HIP(hipMemcpyAsync(dbias, bias, bb, hipMemcpyHostToDevice, ctx->stream));
    if ((s = grx_float_gemv_f32(ctx->stream, dw, rows, cols, dx, dbias, dy)) != GRX_OK) return s;
    GRX_HIP(hipMemcpyAsync(dst, dy, yb, hipMemcpyDeviceToHost, ctx->stream));
    GRX_HIP(hipStreamSynchronize(ctx->stream));
    return GRX_OK;
}

// kern.Linear of a float32 weight w [n][k] over B groups of `per` rows of x
// [B*per][k] into y [B*per][n] (bias nullable): the k6x16 form for every
// row when a group has more than 16, then the gemvRows rows rewritten.
grx_status grx_float_rows_f32(hipStream_t st, const float *x, const float *w, const float *bias, float *y, int B,
                              int per, int n, int k) {
    const int rows = B * per, lo = per > 16 ? per / 6 * 6 : 0;
    if (rows == 0 || n == 0) return GRX_OK;
    if (lo > 0) {
        // 16 columns a workgroup for narrow outputs; 64 x 64 tiles once they
        // give two workgroups a CU, 32 x 32 (four times as many) below that
        const long tiles = (long)grx_ceil_div(rows, 64) * grx_ceil_div(n, 64);
        const hipError_t e = n <= 32         ? launch_rows<4, 1, 1, 1, 64>(st, x, w, bias, y, rows, n, k)
                             : tiles >= 512 ? launch_rows<2, 2, 2, 2, 32>(st, x, w, bias, y, rows, n, k)
                                            : launch_rows<2, 2, 1, 1, 128>(st, x, w, bias, y, rows, n, k);
        if (e != hipSuccess) return grx_hip_fail(e, "f32_rows_mfma_kernel");
    }
    const size_t tail = (size_t)B * (per - lo) * n;
    if (tail > 0) {
        f32_rows_gemv_kernel<<<(unsigned)((tail + 15) / 16), 256, 0, st>>>(x, w, bias, y, B, per, lo, n, k);
        GRX_LAUNCHED("f32_rows_gemv_kernel");
    }
    return GRX_OK;
}

extern "C" grx_status grx_debug_rows_f32(grx_ctx *ctx, float *dst, const float *x, int m, const float *w, int rows,
                                         int cols, const float *bias) {
    if (!ctx || m < 0 || rows < 0 || cols < 0 || ((!dst || !x || !w) && m > 0 && rows > 0))
        return grx_fail(GRX_EINVAL, "grx_debug_rows_f32: NULL argument or negative size");
    if (m == 0 || rows == 0) return GRX_OK;
    const size_t wb = (size_t)rows * cols * 4, xb = (size_t)m * cols * 4, yb = (size_t)m * rows * 4;
    const size_t bb = bias ? (size_t)rows * 4 : 0;
    auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    void *buf;
    grx_status s = grx_ctx_scratch(ctx, up(wb) + up(xb) + up(yb) + up(bb) + 256, &buf);
    if (s != GRX_OK) return s;
    char *p = static_cast<char *>(buf);
    float *dw = reinterpret_cast<float *>(p), *dx = reinterpret_cast<float *>(p + up(wb));
    float *dy = reinterpret_cast<float *>(p + up(wb) + up(xb));
    float *dbias = bias ? reinterpret_cast<float *>(p + up(wb) + up(xb) + up(yb)) : nullptr;
    GRX_HIP(hipSetDevice(ctx->device));
    GRX_HIP(hipMemcpyAsync(dw, w, wb, hipMemcpyHostToDevice, ctx->stream));
    GRX_HIP(hipMemcpyAsync(dx, x, xb, hipMemcpyHostToDevice, ctx->stream));
    if (bias) GRX_HIP(hipMemcpyAsync(dbias, bias, bb, hipMemcpyHostToDevice, ctx->stream));
    if ((s = grx_float_rows_f32(ctx->stream, dx, dw, dbias, dy, 1, m, rows, cols)) != GRX_OK) return s;
    GRX_HIP(hipMemcpyAsync(dst, dy, yb, hipMemcpyDeviceToHost, ctx->stream));
    GRX_HIP(hipStreamSynchronize(ctx->stream));
    return GRX_OK;
}
