// SPDX-License-Identifier: Apache-2.0
// kda_proj.hip - projections of the drop-in layer: y[t][o] = W[o][:] . x[t][:] (gfx950).
//
// The reference computes every projection as a per-token GEMV with double accumulators
// (k3_matmul, src/core/k3_ops.c:265-291; bf16 weights widened exactly, :1122-1227). These
// kernels keep the double accumulation and the exact widening of the weights, so they
// reproduce the reference to within the last bit of the fp32 result; only the summation
// order differs. One launch takes several matrices over the same x (the layer's q, k, v, f_a,
// b and g), so a token costs one launch for all of them.
//
// Two forms, by the number of tokens:
//  * T <= 4 (fp32 weights: T <= 2), proj_gemv_kernel: a wave owns R rows of W and every token,
//    8 consecutive inputs per lane (a 16-byte load of bf16), double FMAs on the vector unit, a
//    butterfly over the lanes. Bound by reading W: one token of a bf16 layer of hidden 4096
//    and 32 x 128 heads streams its 136 MB of q, k, v, g, f_a and b in about 25 us (the call 390 -> 43 us); one
//    row a wave, one element a lane and eight token accumulators whatever T is took 46 us for
//    each 34 MB matrix (0.7 TB/s).
//  * more tokens, proj_mfma_kernel: v_mfma_f64_16x16x4_f64 tiles of 16 rows x 16 tokens, four
//    waves of a workgroup on interleaved 64-wide K blocks of the same tiles (summed in wave
//    order). An instruction does the work of 16 vector FMAs without their operand traffic
//    and needs no lane reduction. Bound by the fp64 matrix rate from T = 16 on (a 16-token
//    column of that layer is 1.4 GFMA, 36 us at 79 TFLOP/s, about what its weights take to
//    stream). The whole layer call at T = 16, int8: 866 -> 125 us; T = 400, fp32: 20.4 -> 1.39
//    ms, int8: 20.0 -> 1.35 ms (the vector form alone reads W once per 8 tokens).
//
// The int8 draft format (K3_WI8, include/k3/k3.h:266-283; k3_matmul_q8,
// src/core/k3_ops.c:1228-1301) stores row o as [f32 scale][int8 * in] (4 + in bytes, so rows
// are byte-aligned only): the int8 weights are dotted with x in double and the row's scale
// applied once at the end, y = (float)dot * scale. The reference sums in float in its SIMD
// order and states no exactness contract for the format; the double sum is within float
// rounding of it.
#include <type_traits>

#include "k3kda_common.h"
#include "kda_internal.h"

namespace k3kda {

namespace {

constexpr int PJ_WAVES = 4;
// Tokens up to which the GEMV form runs. Layer calls at hidden 4096, 32 x 128 heads, GEMV
// against MFMA form: bf16 T = 2 84 | 123 us, T = 4 101 | 124; int8 T = 4 90 | 121; fp32 T = 2
// 125 | 137, but T = 3 165 | 140 (its weights take twice the load instructions per input).
constexpr int PJ_GEMV_T = 4, PJ_GEMV_T_F32 = 2;
constexpr long PJ_MAX_T = 65535L * 8; // longest T of one call

struct ProjArgs {
    ProjSeg s[PROJ_SEGS];
    int first[PROJ_SEGS];   // first row group (R or 16 rows) of each matrix
    int n, groups;
};

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_a4 __attribute__((aligned(4)));   // a 16-byte load at 4-byte alignment
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef u32x2 u32x2_a4 __attribute__((aligned(4)));

template <int WDT> __device__ __forceinline__ size_t row_bytes(int in)
{
    return WDT == K3_WBF16 ? (size_t)in * 2 : WDT == K3_WI8 ? 4 + (size_t)in : (size_t)in * 4;
}

// Eight consecutive weights of a row, from element k on: raw bits, then as doubles. VEC: k and
// the row length are multiples of 8 and rows start 16-byte aligned (int8 rows: 4-byte), so
// the slice is one or two vector loads; else element by element, zeros past the row's end.
// ONCE: the weights are read once per call, so vector loads stream past the caches.
template <int WDT, bool VEC, bool ONCE> struct Slice {
    static __device__ __forceinline__ u32x4 load16(const u32x4 *p) { return ONCE ? __builtin_nontemporal_load(p) : *p; }
    u32x4 a, b;
    // row: the row's first byte (int8: its scale); live: the slice is inside the row
    __device__ __forceinline__ void load(const unsigned char *row, int k, int in, bool live)
    {
        if constexpr (VEC) {
            const int kk = live ? k : 0;
            if constexpr (WDT == K3_WBF16) {
                a = load16(reinterpret_cast<const u32x4 *>(row + 2 * (size_t)kk));
                if (!live) a = u32x4(0u);
            } else if constexpr (WDT == K3_WI8) {
                const u32x2 v = *reinterpret_cast<const u32x2_a4 *>(row + 4 + kk);
                a = u32x4{live ? v.x : 0u, live ? v.y : 0u, 0u, 0u};
            } else {
                const u32x4 *p = reinterpret_cast<const u32x4 *>(row + 4 * (size_t)kk);
                a = load16(p);
                b = load16(p + 1);
                if (!live) a = b = u32x4(0u);
            }
        } else {
            uint32_t e[8];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const bool ok = live && k + j < in;
                const size_t i = ok ? (size_t)(k + j) : 0;
                uint32_t v;
                if constexpr (WDT == K3_WBF16) v = reinterpret_cast<const uint16_t *>(row)[i];
                else if constexpr (WDT == K3_WI8) v = row[4 + i];
                else v = reinterpret_cast<const uint32_t *>(row)[i];
                e[j] = ok ? v : 0u;
            }
            if constexpr (WDT == K3_WBF16) {
                a = u32x4{e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16)};
            } else if constexpr (WDT == K3_WI8) {
                a = u32x4{e[0] | (e[1] << 8) | (e[2] << 16) | (e[3] << 24),
                          e[4] | (e[5] << 8) | (e[6] << 16) | (e[7] << 24), 0u, 0u};
            } else {
                a = u32x4{e[0], e[1], e[2], e[3]};
                b = u32x4{e[4], e[5], e[6], e[7]};
            }
        }
    }
    __device__ __forceinline__ double at(int j) const   // j a constant 0..7
    {
        if constexpr (WDT == K3_WBF16) {
            const uint32_t u = a[j >> 1];
            return (double)__uint_as_float((j & 1) ? (u & 0xffff0000u) : (u << 16));
        } else if constexpr (WDT == K3_WI8) {
            return (double)((int)(a[j >> 2] << (24 - 8 * (j & 3))) >> 24);
        } else {
            return (double)__uint_as_float(j < 4 ? a[j & 3] : b[j & 3]);
        }
    }
};

// Eight consecutive inputs of a token (fp32), zeros past the end.
template <bool VEC> struct XSlice {
    f4 a, b;
    __device__ __forceinline__ void load(const float *row, int k, int in, bool live)
    {
        if constexpr (VEC) {
            const f4 *p = reinterpret_cast<const f4 *>(row + (live ? k : 0));
            a = p[0];
            b = p[1];
            if (!live) a = b = f4(0.0f);
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const bool ok = live && k + j < in;
                const float v = row[ok ? k + j : 0];
                if (j < 4) a[j] = ok ? v : 0.0f;
                else b[j - 4] = ok ? v : 0.0f;
            }
        }
    }
    __device__ __forceinline__ double at(int j) const { return (double)(j < 4 ? a[j & 3] : b[j & 3]); }
};

__device__ __forceinline__ float q8_scale(const unsigned char *row)   // unaligned little-endian fp32
{
    return __uint_as_float((uint32_t)row[0] | ((uint32_t)row[1] << 8) | ((uint32_t)row[2] << 16) |
                           ((uint32_t)row[3] << 24));
}

__device__ __forceinline__ int find_seg(const ProjArgs &a, int group)
{
    int s = 0;
    while (s + 1 < a.n && group >= a.first[s + 1]) s++;
    return s;
}

// One wave: rows R g .. R g + R - 1 of a matrix, tokens 0..T-1 (T <= TB). Lane l takes inputs
// 512 i + 8 l .. + 7; U blocks of 512 are requested together.
template <int WDT, int TB, int R, int U, bool VEC>
__global__ __launch_bounds__(64 * PJ_WAVES) void proj_gemv_kernel(const ProjArgs a, int T, int in,
                                                                  const float *__restrict__ x)
{
    const int lane = threadIdx.x & 63;
    const int group = __builtin_amdgcn_readfirstlane(blockIdx.x * PJ_WAVES + (threadIdx.x >> 6));
    if (group >= a.groups) return;
    const int si = find_seg(a, group);
    const ProjSeg &sg = a.s[si];
    const int r0 = (group - a.first[si]) * R;
    const size_t rb = row_bytes<WDT>(in);
    const unsigned char *row[R];
#pragma unroll
    for (int r = 0; r < R; r++) row[r] = reinterpret_cast<const unsigned char *>(sg.W) + (size_t)min(r0 + r, sg.rows - 1) * rb;
    double acc[R][TB];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int t = 0; t < TB; t++) acc[r][t] = 0.0;
    // NU blocks of 512 inputs, the lane's first slice at input k
    auto blocks = [&](auto nu, int k) {
        constexpr int NU = decltype(nu)::value;
        Slice<WDT, VEC, true> w[NU][R];
        XSlice<VEC> xs[NU][TB];
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const bool live = k + 512 * u < in;
#pragma unroll
            for (int r = 0; r < R; r++) w[u][r].load(row[r], k + 512 * u, in, live);
        }
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const bool live = k + 512 * u < in;
#pragma unroll
            for (int t = 0; t < TB; t++) xs[u][t].load(x + (size_t)min(t, T - 1) * in, k + 512 * u, in, live);
        }
#pragma unroll
        for (int u = 0; u < NU; u++)
#pragma unroll
            for (int j = 0; j < 8; j++) {
                double xd[TB];
#pragma unroll
                for (int t = 0; t < TB; t++) xd[t] = xs[u][t].at(j);
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const double wd = w[u][r].at(j);
#pragma unroll
                    for (int t = 0; t < TB; t++) acc[r][t] = fma(wd, xd[t], acc[r][t]);
                }
            }
    };
    const int nb = (in + 511) / 512;
    int i = 0;
    for (; i + U <= nb; i += U) blocks(std::integral_constant<int, U>{}, 512 * i + 8 * lane);
    if constexpr (U > 2)
        for (; i + 2 <= nb; i += 2) blocks(std::integral_constant<int, 2>{}, 512 * i + 8 * lane);
    for (; i < nb; i++) blocks(std::integral_constant<int, 1>{}, 512 * i + 8 * lane);
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int t = 0; t < TB; t++) {
            double s = acc[r][t];
#pragma unroll
            for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
            if (lane == 0 && r0 + r < sg.rows && t < T) {
                float v = (float)s;
                if constexpr (WDT == K3_WI8) v *= q8_scale(row[r]);
                sg.y[(size_t)t * sg.rows + r0 + r] = v;
            }
        }
}

typedef double f64x4 __attribute__((ext_vector_type(4)));

// Tiles of 16 rows x 16 NT tokens: A = tokens (lane l: token l % 16), B = rows of W (row
// l % 16), each lane supplying the K values of its 16-lane group; the K values of a block
// are dealt so that a lane's eight are consecutive in memory (group g: 8 g .. 8 g + 7 of each
// 32), which both operands share, so the product is the same. Wave w takes blocks w, w + 4, ..
// of 64. D: lane l holds column (row of W) l % 16, tokens l / 16 + 4 i. Workgroup L runs on
// XCD L % 8: its `ny` token blocks of one row tile are neighbours on one XCD, so the row tile
// is read from memory once and the other blocks find it in that XCD's L2.
template <int WDT, int NT, bool VEC>
__global__ __launch_bounds__(64 * PJ_WAVES) void proj_mfma_kernel(const ProjArgs a, int T, int in,
                                                                  const float *__restrict__ x, int ny)
{
    const int slot = blockIdx.x >> 3, group = (slot / ny) * 8 + (blockIdx.x & 7);
    if (group >= a.groups) return;
    __shared__ double part[PJ_WAVES - 1][NT][4][64];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = lane & 15, g = lane >> 4;
    const int si = find_seg(a, group);
    const ProjSeg &sg = a.s[si];
    const int r0 = (group - a.first[si]) * 16, t0 = (slot % ny) * 16 * NT;
    const unsigned char *row =
        reinterpret_cast<const unsigned char *>(sg.W) + (size_t)min(r0 + m, sg.rows - 1) * row_bytes<WDT>(in);
    const float *xr[NT];
#pragma unroll
    for (int n = 0; n < NT; n++) xr[n] = x + (size_t)min(t0 + 16 * n + m, T - 1) * in;
    f64x4 acc[NT];
#pragma unroll
    for (int n = 0; n < NT; n++) acc[n] = f64x4(0.0);
    // 32 inputs a step; the next step's operands are requested before this one's products
    auto first_k = [&](int i) { return 64 * (wv + PJ_WAVES * (i >> 1)) + 32 * (i & 1); };
    struct Ops {
        Slice<WDT, VEC, NT == 1> w;
        XSlice<VEC> xs[NT];
    } cur, nxt;
    auto load = [&](Ops &o, int k0) {
        const int k = k0 + 8 * g;
        const bool live = k < in;
        o.w.load(row, k, in, live);
#pragma unroll
        for (int n = 0; n < NT; n++) o.xs[n].load(xr[n], k, in, live);
    };
    load(cur, first_k(0));
    for (int i = 0; first_k(i) < in; i++) {
        load(nxt, first_k(i + 1));   // past the end: nothing live
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const double wd = cur.w.at(j);
#pragma unroll
            for (int n = 0; n < NT; n++)
                acc[n] = __builtin_amdgcn_mfma_f64_16x16x4f64(cur.xs[n].at(j), wd, acc[n], 0, 0, 0);
        }
        cur = nxt;
    }
    if (wv > 0) {
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
            for (int i = 0; i < 4; i++) part[wv - 1][n][i][lane] = acc[n][i];
    }
    __syncthreads();
    if (wv > 0 || r0 + m >= sg.rows) return;
    float scale = 1.0f;
    if constexpr (WDT == K3_WI8) scale = q8_scale(row);
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int t = t0 + 16 * n + g + 4 * i;
            if (t >= T) continue;
            double s = acc[n][i];
#pragma unroll
            for (int w = 0; w < PJ_WAVES - 1; w++) s += part[w][n][i][lane];
            float v = (float)s;
            if constexpr (WDT == K3_WI8) v *= scale;
            sg.y[(size_t)t * sg.rows + r0 + m] = v;
        }
}

// groups of `per` rows, no group across two matrices
int deal(ProjArgs &a, int per)
{
    a.groups = 0;
    for (int i = 0; i < a.n; i++) {
        a.first[i] = a.groups;
        a.groups += (a.s[i].rows + per - 1) / per;
    }
    return a.groups;
}

template <int WDT, bool VEC>
int launch(ProjArgs &a, int T, int in, long rows, const float *x, hipStream_t st)
{
    if (T <= (WDT == K3_WF32 ? PJ_GEMV_T_F32 : PJ_GEMV_T)) {
        // Two rows a wave read x half as often, but need twice the rows to fill the GPU:
        // they run from 8192 rows on (32 waves of two rows per CU); below, one row a wave. (Four
        // rows: the token of the bf16 layer above 46.3 us against 43.1, fp32 120 against 81.)
        // One bf16 token keeps four blocks of 512 inputs in flight, its weights being one load
        // each (43.1 us, two blocks 45.7); fp32, twice the loads, two (80.8 against 85.5).
        const int R = rows >= 8192 ? 2 : 1;
        const unsigned blocks = (unsigned)((deal(a, R) + PJ_WAVES - 1) / PJ_WAVES);
#define K3_GEMV(TB, RR, UU) \
    hipLaunchKernelGGL((proj_gemv_kernel<WDT, TB, RR, UU, VEC>), dim3(blocks), dim3(64 * PJ_WAVES), 0, st, a, T, in, x)
        if (R == 2) {
            if (T == 1) {
                if constexpr (WDT == K3_WBF16) K3_GEMV(1, 2, 4);
                else K3_GEMV(1, 2, 2);
            }
            else if (T == 2) K3_GEMV(2, 2, 2);
            else if constexpr (WDT != K3_WF32) K3_GEMV(4, 2, 1);
        } else {
            if (T == 1) K3_GEMV(1, 1, 4);
            else if (T == 2) K3_GEMV(2, 1, 2);
            else if constexpr (WDT != K3_WF32) K3_GEMV(4, 1, 2);
        }
#undef K3_GEMV
    } else {
        // up to four token tiles a workgroup, dealt evenly over the token blocks
        const int tiles = (T + 15) / 16, ny = (tiles + 3) / 4, nt = (tiles + ny - 1) / ny;
        const long wgs = ((long)deal(a, 16) + 7) / 8 * 8 * ny;
        if (wgs > 0x7fffffffL) K3_FAIL(K3HIP_EINVAL, "projection: T=%d too large for %ld rows", T, rows);
        const dim3 grid((unsigned)wgs);
#define K3_F64(NT) hipLaunchKernelGGL((proj_mfma_kernel<WDT, NT, VEC>), grid, dim3(64 * PJ_WAVES), 0, st, a, T, in, x, ny)
        if (nt == 1) K3_F64(1);
        else if (nt == 2) K3_F64(2);
        else if (nt == 3) K3_F64(3);
        else K3_F64(4);
#undef K3_F64
    }
    K3_LAUNCHED();
    return K3HIP_OK;
}

}  // namespace

int proj_multi(int T, int in, const ProjSeg *segs, int n, const float *x, int wdt, hipStream_t st)
{
    if (n < 1 || n > PROJ_SEGS) K3_FAIL(K3HIP_EINVAL, "projection: %d matrices", n);
    ProjArgs a{};
    long rows = 0;
    // vector loads: rows of whole 8-element slices at 16-byte (int8: 4-byte) boundaries
    bool vec = in % 8 == 0 && ((uintptr_t)x & 15) == 0;
    for (int i = 0; i < n; i++) {
        if (segs[i].rows <= 0) continue;
        a.s[a.n++] = segs[i];
        rows += segs[i].rows;
        vec = vec && ((uintptr_t)segs[i].W & (wdt == K3_WI8 ? 3 : 15)) == 0;
    }
    if (T <= 0 || rows == 0) return K3HIP_OK;
    if (T > PJ_MAX_T) K3_FAIL(K3HIP_EINVAL, "projection: T=%d too large for the GEMV path", T);
    switch (wdt) {
    case K3_WBF16: return vec ? launch<K3_WBF16, true>(a, T, in, rows, x, st) : launch<K3_WBF16, false>(a, T, in, rows, x, st);
    case K3_WF32: return vec ? launch<K3_WF32, true>(a, T, in, rows, x, st) : launch<K3_WF32, false>(a, T, in, rows, x, st);
    case K3_WI8: return vec ? launch<K3_WI8, true>(a, T, in, rows, x, st) : launch<K3_WI8, false>(a, T, in, rows, x, st);
    default: K3_FAIL(K3HIP_EUNSUPPORTED, "projection: weight tag %d (fp32=0, bf16=1, int8 rows=2)", wdt);
    }
}

int proj(int T, int in, int out, const float *x, const void *W, int wdt, float *y, hipStream_t st)
{
    const ProjSeg s{W, y, out};
    return proj_multi(T, in, &s, 1, x, wdt, st);
}

}  // namespace k3kda
