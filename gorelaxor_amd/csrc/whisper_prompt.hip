// whisper_prompt.hip - cross-attention of many decoder rows at once (a
// prompt's rows) on the float32 matrix cores.
//
// v_mfma_f32_16x16x4_f32 adds its four products to the accumulator one after
// another in k order, each with a single rounding: exactly four steps of a
// fused multiply-add chain (the float32 rows' tests hold it to fmaf chains bit
// for bit, with subnormal sums, signed zeros, infinities and NaN).  dotF32x4
// (kernels_amd64.s:156-204) is sixteen such chains, chain c over the elements
// 16t + c, so a matrix-core tile per chain gives the reference's sixteen lane
// sums of 16 x 16 outputs; the lanes' final sums stay in the reference's order.
#include "grx_float.h"
#include "grx_internal.h"

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kPcRows = 16;      // decoder rows per workgroup
constexpr int kPcThreads = 1024; // one wave per row in the softmax and the output
constexpr int kPcHd = 64;
constexpr int kPcHs = 8 * kPcRows * kPcHd;  // the values' lane sums S_l [8][rows][64]

// Floats from one row's scores to the next: 4 banks apart (mod 32), so that
// the 16-byte reads of eight rows fall in distinct banks.
__host__ __device__ constexpr int pc_ld(int nctx) { return ((nctx + 31) & ~31) + 4; }
size_t pc_lds(int nctx) { return ((size_t)kPcRows * pc_ld(nctx) + kPcHs) * 4; }

// One head (blockIdx.x) of kPcRows rows (group blockIdx.y) of one stream
// (blockIdx.z: its rows `per` apart in q and att, its cross keys and values
// x_stream floats after the previous stream's): scores (decoder.go:94-108),
// softmax (109), weighted values (110-118), rounded to Q8_0 for the
// cross-out product.
//
// What bounds it: the values, 64 x nctx floats of a head that every row needs
// (384 KB at 1500 positions); sixteen rows share each load, where a workgroup
// a row would read them from L2 sixteen times.  Scores stay in LDS (96 KB).
// Measured at 187 rows, 8 heads, 1500 positions: 47 us a layer.
__global__ __launch_bounds__(kPcThreads) void cross_prompt_kernel(
    const float *__restrict__ q, const float *__restrict__ ck, const float *__restrict__ cv, int nctx, int st, int per,
    size_t x_stream, int8_t *__restrict__ att_q, float *__restrict__ att_s) {
    extern __shared__ __align__(16) float sm[];
    const int h = blockIdx.x, r0 = blockIdx.y * kPcRows;
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int LD = pc_ld(nctx);
    float *sc = sm, *hs = sm + kPcRows * LD;
    const size_t row0 = (size_t)blockIdx.z * per;
    q += row0 * st + h * kPcHd;
    ck += blockIdx.z * x_stream + (size_t)h * nctx * kPcHd;
    cv += blockIdx.z * x_stream + (size_t)h * kPcHd * nctx;

    // ---- scores: lane (li, lk) holds row li's and key li's values
    // 16 lk + c, c = 0..15: chain c's four steps are one instruction
    const int n4 = nctx & ~3, nkt = (nctx + 15) >> 4;
    {
        float4 qv[4];
        const float4 *qr = reinterpret_cast<const float4 *>(q + (size_t)min(r0 + li, per - 1) * st + 16 * lk);
#pragma unroll
        for (int i = 0; i < 4; ++i) qv[i] = qr[i];
        float4 kn[4];
        auto kload = [&](int kt) {
            const float4 *kr = reinterpret_cast<const float4 *>(ck + (size_t)min(16 * kt + li, nctx - 1) * kPcHd + 16 * lk);
#pragma unroll
            for (int i = 0; i < 4; ++i) kn[i] = kr[i];
        };
        if (wave < nkt) kload(wave);
        for (int kt = wave; kt < nkt; kt += kPcThreads / 64) {
            float4 kv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) kv[i] = kn[i];
            kload(min(kt + kPcThreads / 64, nkt - 1));
            // lane sums S_l = A_l + B_l (chains l and 8 + l)
            v4f S[8];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const float qa[4] = {qv[i].x, qv[i].y, qv[i].z, qv[i].w}, ka[4] = {kv[i].x, kv[i].y, kv[i].z, kv[i].w};
                const float qb[4] = {qv[i + 2].x, qv[i + 2].y, qv[i + 2].z, qv[i + 2].w};
                const float kb[4] = {kv[i + 2].x, kv[i + 2].y, kv[i + 2].z, kv[i + 2].w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const v4f z = {0.f, 0.f, 0.f, 0.f};
                    const v4f A = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[j], ka[j], z, 0, 0, 0);
                    const v4f B = __builtin_amdgcn_mfma_f32_16x16x4f32(qb[j], kb[j], z, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) S[4 * i + j][r] = __fadd_rn(A[r], B[r]);
                }
            }
            const int key = 16 * kt + li;
            if (key < n4) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float a[8] = {S[0][r], S[1][r], S[2][r], S[3][r], S[4][r], S[5][r], S[6][r], S[7][r]};
                    sc[(4 * lk + r) * LD + key] = hsum8(a);
                }
            }
        }
        // the keys past the last whole group of four: dotF32Go
        if (tid < kPcRows * (nctx - n4)) {
            const int r = tid % kPcRows, key = n4 + tid / kPcRows;
            sc[r * LD + key] = dot_go(q + (size_t)min(r0 + r, per - 1) * st, ck + (size_t)key * kPcHd, kPcHd);
        }
    }
    __syncthreads();

    // ---- softmax: wave w is row w (block_softmax's order)
    {
        float *s = sc + wave * LD;
        float mx = -__builtin_inff();
        for (int j = lane; j < nctx; j += 64) mx = s[j] > mx ? s[j] : mx;
        mx = wave_max(mx);
        const int n8 = nctx & ~7;
        for (int j = lane; j < n8; j += 64) s[j] = grx_exp8(__fsub_rn(s[j], mx));
        if (n8 + lane < nctx) s[n8 + lane] = grx_expf_go(__fsub_rn(s[n8 + lane], mx));
        __syncthreads();
        // the eight lane sums (lanes 0..7), the tail's own sum (lane 8)
        float acc = 0.f;
        const int c = lane & 7, N = n8 >> 3;
        if (lane < 8) {
#pragma unroll 32
            for (int i = 0; i < N; ++i) acc = __fadd_rn(acc, s[8 * i + c]);
        } else if (lane == 8) {
            for (int j = n8; j < nctx; ++j) acc = __fadd_rn(acc, s[j]);
        }
        float a[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) a[i] = __shfl(acc, i);
        const float sa = n8 > 0 ? hsum8(a) : 0.f;
        const float inv = __fdiv_rn(1.0f, __fadd_rn(sa, __shfl(acc, 8)));
        for (int j = lane; j < nctx; j += 64) s[j] = __fmul_rn(s[j], inv);
    }
    __syncthreads();

    // ---- values: wave (dt, g) forms chains 2g, 2g+1 and 8 + those of
    // outputs 16 dt .. +15.  Steps past the last are products of -0 and +0:
    // adding -0 leaves every sum as it is.
    const int steps = nctx >> 4;
    {
        const int dt = wave & 3, g = wave >> 2;
        const float *vr = cv + (size_t)(16 * dt + li) * nctx + 2 * g;
        const float *pr = sc + li * LD + 2 * g;
        v4f acc[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = v4f{0.f, 0.f, 0.f, 0.f};
        constexpr int U = 4;  // groups of four steps with their loads in flight
        struct Set {
            float v[U][4];
        };
        const int nT = (steps + 3) >> 2;
        const bool even = (nctx & 1) == 0;  // 8-byte aligned rows
        auto load = [&](Set &s, int T0) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float *p = vr + 16 * min(4 * (T0 + u) + lk, max(steps - 1, 0));
                if (even) {
                    const float2 a = *reinterpret_cast<const float2 *>(p), b = *reinterpret_cast<const float2 *>(p + 8);
                    s.v[u][0] = a.x, s.v[u][1] = a.y, s.v[u][2] = b.x, s.v[u][3] = b.y;
                } else {
                    s.v[u][0] = p[0], s.v[u][1] = p[1], s.v[u][2] = p[8], s.v[u][3] = p[9];
                }
            }
        };
        auto fold = [&](const Set &s, int T0) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (T0 + u >= nT) break;  // uniform
                const int t = 4 * (T0 + u) + lk;
                const float *pp = pr + 16 * min(t, steps - 1);
                const float2 a = *reinterpret_cast<const float2 *>(pp), b = *reinterpret_cast<const float2 *>(pp + 8);
                const float pv[4] = {a.x, a.y, b.x, b.y};
                const bool in = t < steps;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? pv[i] : -0.0f, in ? s.v[u][i] : 0.0f, acc[i], 0, 0, 0);
            }
        };
        if (nT > 0) {
            Set s0, s1;
            load(s0, 0);
            for (int T = 0; T < nT; T += 2 * U) {
                load(s1, T + U);
                fold(s0, T);
                load(s0, T + 2 * U);
                fold(s1, T + U);
            }
        }
        // S_l = A_l + B_l of lanes l = 2g, 2g + 1
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                hs[((2 * g + i) * kPcRows + 4 * lk + r) * kPcHd + 16 * dt + li] = __fadd_rn(acc[i][r], acc[i + 2][r]);
    }
    __syncthreads();

    // ---- HSUM, the tail's dotF32Go, the output: wave = row, lane = value
    {
        const int kk = nctx & ~15;
        float o = 0.f;
        if (kk > 0) {
            float a[8];
#pragma unroll
            for (int l = 0; l < 8; ++l) a[l] = hs[(l * kPcRows + wave) * kPcHd + lane];
            o = hsum8(a);
        }
        if (kk < nctx) o = __fadd_rn(o, dot_go(sc + wave * LD + kk, cv + (size_t)lane * nctx + kk, nctx - kk));
        const int r = r0 + wave;
        if (r < per) {
            const size_t row = row0 + r, col = (size_t)h * kPcHd + lane;
            quant32_store(o, att_q + row * st + col, att_s + (row * st + col) / 32, lane & 31);
        }
    }
}

}  // namespace

bool grx_cross_prompt_ok(int nctx, int hd) {
    if (hd != kPcHd || pc_lds(nctx) > 160 * 1024) return false;
    static GrxDeviceOnce once;
    const bool ok = grx_raise_lds(once, {(const void *)cross_prompt_kernel}, 160 * 1024) == hipSuccess;
    if (!ok) (void)hipGetLastError();
    return ok;
}

grx_status grx_cross_prompt(hipStream_t stream, const float *q, const float *ck, const float *cv, int nctx, int st,
                            int per, int streams, size_t x_stream, int8_t *att_q, float *att_s) {
    cross_prompt_kernel<<<dim3(st / kPcHd, grx_ceil_div(per, kPcRows), streams), kPcThreads, pc_lds(nctx), stream>>>(
        q, ck, cv, nctx, st, per, x_stream, att_q, att_s);
    GRX_LAUNCHED("cross_prompt_kernel");
    return GRX_OK;
}
