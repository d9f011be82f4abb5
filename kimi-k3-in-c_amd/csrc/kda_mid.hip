// SPDX-License-Identifier: Apache-2.0
// kda_mid.hip - products of short and middle-sized prefills: several weights over the same rows
// in one launch, for gfx950.
//
// Replaces the reference's per-token k3_mmw calls (include/k3/k3.h:290-296 ->
// k3_matmul_bf16, src/core/k3_ops.c:1122-1227; call sites :877-886, :946-948):
//   C_s[M][rows_s] = A[M][K] . B_s[rows_s][K]^T     for up to MID_SEGS weights B_s
// with fp32 accumulation. A is one of
//   bf16 rows (the z product of the bf16 prefill, on f_a's split rows),
//   fp32 rows split into bf16 hi + lo, both against the bf16 weight (fp32 accuracy: x = hi + lo
//   to 2.5e-6 relative rms), which needs no split rows or second half of the result in memory
//   (the full-accuracy layer; the bits of kda_mm.hip on split rows and the two halves' sum).
//
// The 256 x 256 tiles of kda_mm.hip leave most of the GPU idle here (333 tokens of a hidden
// 2048, 16 x 128 layer: 2 x 33 tiles over 256 CUs, and 16 for z), and a launch per weight
// costs more than its products. Tiles of 64 rows x 128 columns (64 x 64 where those would not
// give every CU one, 128 x 128 for bf16 rows where those do), four waves in 2 x 2, K in steps of
// 64. Weights and bf16 rows come by direct-to-LDS buffer loads into 2, 3 or 5 buffers, each requested
// 1, 2 or 4 steps before it is read; fp32 rows go through registers one step ahead and are
// split as they are put in LDS (two buffers). Loads come back in order, so the wait for a step's
// fp32 rows is one for all but the newest step's weights, and a third buffer is the last that
// helps (64 x 64 tiles: five 91.6 us, three 90.4 for the 100-token layer at hidden 2048, 16 x 128).
// 56-80 KiB of LDS; where two workgroups share a CU, one's barrier and load waits hide behind the
// other's products. Rows are 128 bytes, the
// 16-byte chunk index XORed with (row & 7) ^ ((row >> 3) & 1): 16-lane fragment reads fall on
// distinct banks. The weight is the MFMA's first operand, so a lane ends with four adjacent
// columns of one row: 16-byte stores. A column tile's row tiles run on one XCD (workgroup id
// % 8), so its weight rows are read from memory once.
//
// Bound by the chain of a K-step (barrier, LDS reads, products) with 1 to 2 waves per SIMD, then
// by LDS bandwidth (a 64 x 128 step reads 192 bytes per clock at the MFMAs' full rate, the LDS
// gives 128).
#include "kda_internal.h"

#include <algorithm>

namespace k3kda {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int BK = 64, NT = 256, ROW = BK * 2;   // ROW: bytes of a staged row

struct MidArgs {
    MidSeg s[MID_SEGS];
    int first[MID_SEGS];   // first column tile of each weight
    int n, tiles_m, tiles_n;
};

[[maybe_unused]] __device__ __forceinline__ int swz(int row) { return (row & 7) ^ ((row >> 3) & 1); }

template <int n> __device__ __forceinline__ void wait_vm()   // vmcnt(n) lgkmcnt(0)
{
    static_assert(n >= 0 && n < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4));
}

[[maybe_unused]] __device__ __forceinline__ f32x4 mfma(const u32x4 &a, const u32x4 &b, const f32x4 &c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// bf16 pair of two floats, and the pair of what the rounding left
__device__ __forceinline__ uint32_t pack2(float a, float b) { return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{a, b}, bf16x2)); }
[[maybe_unused]] __device__ __forceinline__ uint32_t pack2_rest(float a, float b, uint32_t hi)
{
    return pack2(a - __uint_as_float(hi << 16), b - __uint_as_float(hi & 0xffff0000u));
}

template <int AM, int BM, int BN, int NBUF>
__global__ __launch_bounds__(NT, 2) void mid_kernel(const MidArgs ar, int M, int K, const void *__restrict__ Av, long lda)
{
#ifdef __HIP_DEVICE_COMPILE__   // the host pass, which only needs the stub, drops it over the 16-byte LDS loads
    constexpr int PARTS = AM == MID_A_SPLIT ? 2 : 1;
    constexpr int B_STAGE = BN * ROW, A_PART = BM * ROW, TI = BM / 32, TJ = BN / 32, LEAD = NBUF - 1;
    constexpr int NB = BN / 32, NA = AM == MID_A_16 ? BM / 32 : 0;   // direct loads per wave and step
    constexpr int A_OFF = NBUF * B_STAGE;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;

    const int slot = blockIdx.x >> 3, tn = (slot / ar.tiles_m) * 8 + (blockIdx.x & 7), tm = slot % ar.tiles_m;
    if (tn >= ar.tiles_n) return;
    int si = 0;
    while (si + 1 < ar.n && tn >= ar.first[si + 1]) si++;
    const MidSeg &sg = ar.s[si];
    const int n0 = (tn - ar.first[si]) * BN, m0 = tm * BM;
    const int nks = K / BK;

    // direct load j of wave w fills rows 8 q .. 8 q + 7 of a buffer, q = w + 4 j (1 KiB): lane l
    // lands at row 8 q + l / 8, place l % 8, so it loads the chunk whose place that is. Rows past
    // the matrix are its last one (their results are not stored).
    auto rsrc = [&](const void *p) { return __builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, 0x7fffffff, 0x00020000); };
    auto voff = [&](int q, int last, long ld) {
        const int r = min(8 * q + (lane >> 3), last);
        return r * (int)ld * 2 + ((((lane & 7) ^ (lane >> 3) ^ q) & 1) | (((lane & 7) ^ (lane >> 3)) & 6)) * 16;
    };
    const __amdgpu_buffer_rsrc_t rB = rsrc(reinterpret_cast<const uint16_t *>(sg.B) + (long)n0 * K);
    int vB[NB], vA[NA > 0 ? NA : 1];
#pragma unroll
    for (int j = 0; j < NB; j++) vB[j] = voff(wave + 4 * j, sg.rows - 1 - n0, K);
    auto load_b = [&](int ks) {
        char *dst = smem + (ks % NBUF) * B_STAGE + 1024 * wave;
        const int k = min(ks, nks - 1) * ROW;
#pragma unroll
        for (int j = 0; j < NB; j++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rB, (lds_void *)(dst + 4096 * j), 16, vB[j], k, 0, 0);
    };
    [[maybe_unused]] __amdgpu_buffer_rsrc_t rA = rB;
    if constexpr (AM == MID_A_16) {
        rA = rsrc(reinterpret_cast<const uint16_t *>(Av) + (long)m0 * lda);
#pragma unroll
        for (int j = 0; j < NA; j++) vA[j] = voff(wave + 4 * j, M - 1 - m0, lda);
    }
    auto load_a16 = [&](int ks) {
        char *dst = smem + A_OFF + (ks % NBUF) * A_PART + 1024 * wave;
        const int k = min(ks, nks - 1) * ROW;
#pragma unroll
        for (int j = 0; j < NA; j++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rA, (lds_void *)(dst + 4096 * j), 16, vA[j], k, 0, 0);
    };
    // fp32 rows: thread t holds 16 inputs of rows t / 4, t / 4 + 64, ..
    constexpr int AR = BM / 64;
    const int ar_row = tid >> 2, ac = (tid & 3) * 2;
    const float *ap[AR];
#pragma unroll
    for (int r = 0; r < AR; r++)
        ap[r] = reinterpret_cast<const float *>(Av) + (long)min(m0 + ar_row + 64 * r, M - 1) * lda + 8 * ac;
    f4 ra[AR][4];
    auto load_a32 = [&](int ks) {
#pragma unroll
        for (int r = 0; r < AR; r++) {
            const f4 *p = reinterpret_cast<const f4 *>(ap[r] + min(ks, nks - 1) * BK);
#pragma unroll
            for (int i = 0; i < 4; i++) ra[r][i] = p[i];
        }
    };
    auto put_a32 = [&](int ks) {
        char *base = smem + A_OFF + (ks & 1) * PARTS * A_PART + ar_row * ROW;
#pragma unroll
        for (int r = 0; r < AR; r++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const f4 u = ra[r][2 * h], v = ra[r][2 * h + 1];
                const u32x4 hi = {pack2(u.x, u.y), pack2(u.z, u.w), pack2(v.x, v.y), pack2(v.z, v.w)};
                char *d = base + 64 * r * ROW + (((ac + h) ^ swz(ar_row)) << 4);
                *reinterpret_cast<u32x4 *>(d) = hi;
                *reinterpret_cast<u32x4 *>(d + A_PART) = u32x4{pack2_rest(u.x, u.y, hi.x), pack2_rest(u.z, u.w, hi.y),
                                                              pack2_rest(v.x, v.y, hi.z), pack2_rest(v.z, v.w, hi.w)};
            }
    };

    const int r16 = lane & 15, kq = lane >> 4;
    const int fo[2] = {r16 * ROW + ((kq ^ swz(r16)) << 4), r16 * ROW + (((4 + kq) ^ swz(r16)) << 4)};
    // the lo halves' products have an accumulator of their own: added to the hi halves' once, at
    // the end, they are not rounded to its last place at every step
    f32x4 acc[PARTS][TI][TJ];
#pragma unroll
    for (int p = 0; p < PARTS; p++)
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++) acc[p][i][j] = 0.0f;

    if constexpr (AM != MID_A_16) load_a32(0);
#pragma unroll
    for (int i = 0; i < LEAD; i++) {
        if constexpr (AM == MID_A_16) load_a16(i);
        load_b(i);
    }
    if constexpr (AM != MID_A_16) put_a32(0);
    // One barrier a step. Before it, each wave's own loads of step ks have landed (the newer
    // steps' stay in flight) and its LDS writes are done; after it, the buffer last read in step
    // ks - 1 takes step ks + LEAD. Loads past the last step repeat it into a buffer that
    // nothing reads, so that the counts stay the same.
    for (int ks = 0; ks < nks; ks++) {
        wait_vm<(LEAD - 1) * (NA + NB)>();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (AM == MID_A_16) load_a16(ks + LEAD);
        else load_a32(ks + 1);
        load_b(ks + LEAD);
        __builtin_amdgcn_sched_barrier(0);
        const char *bb = smem + (ks % NBUF) * B_STAGE + wn * (BN / 2) * ROW;
        const char *ab = smem + A_OFF + (AM == MID_A_16 ? (ks % NBUF) * A_PART : (ks & 1) * PARTS * A_PART) + wm * (BM / 2) * ROW;
        // every fragment of the step is requested before its first product
        u32x4 a[2][PARTS][TI], b[2][TJ];
#pragma unroll
        for (int s = 0; s < 2; s++) {
#pragma unroll
            for (int j = 0; j < TJ; j++) b[s][j] = *reinterpret_cast<const u32x4 *>(bb + 16 * j * ROW + fo[s]);
#pragma unroll
            for (int p = PARTS - 1; p >= 0; p--)
#pragma unroll
                for (int i = 0; i < TI; i++)
                    a[s][p][i] = *reinterpret_cast<const u32x4 *>(ab + p * A_PART + 16 * i * ROW + fo[s]);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int p = PARTS - 1; p >= 0; p--)
#pragma unroll
                for (int i = 0; i < TI; i++)
#pragma unroll
                    for (int j = 0; j < TJ; j++) acc[p][i][j] = mfma(b[s][j], a[s][p][i], acc[p][i][j]);
        if constexpr (AM != MID_A_16) put_a32(ks + 1);
    }
    wait_vm<0>();   // no load may still be writing this workgroup's LDS when it ends

    // lane: columns n0 + .. + 4 kq .. + 3 of row r16 of each 16 x 16 tile. Columns from `cols`
    // on go to the second output.
#pragma unroll
    for (int i = 0; i < TI; i++) {
        const int m = m0 + wm * (BM / 2) + 16 * i + r16;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < TJ; j++) {
            const int n = n0 + wn * (BN / 2) + 16 * j + 4 * kq;
            f32x4 v = acc[0][i][j];
            if constexpr (PARTS == 2) v += acc[1][i][j];
            if (sg.vec && n + 4 <= sg.cols) {
                *reinterpret_cast<f32x4 *>(sg.C + (long)m * sg.ldc + n) = v;
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (n + e >= sg.rows) continue;
                float *p = n + e < sg.cols ? sg.C + (long)m * sg.ldc + n + e : sg.C1 + (long)m * sg.ldc1 + (n + e - sg.cols);
                *p = v[e];
            }
        }
    }
#endif
}

template <int AM, int BM, int BN, int NBUF>
int launch_tile(MidArgs &a, int M, int K, const void *A, long lda, hipStream_t st)
{
    constexpr int lds = NBUF * BN * ROW + (AM == MID_A_16 ? NBUF : 4) * BM * ROW;
    a.tiles_m = (M + BM - 1) / BM;
    a.tiles_n = 0;
    for (int i = 0; i < a.n; i++) {
        a.first[i] = a.tiles_n;
        a.tiles_n += (a.s[i].rows + BN - 1) / BN;
    }
    const long grid = (long)((a.tiles_n + 7) / 8) * 8 * a.tiles_m;
    if (grid > 0x7fffffffL) K3_FAIL(K3HIP_EUNSUPPORTED, "mid: %d rows need too many workgroups", M);
    K3_HIP(hipFuncSetAttribute((const void *)mid_kernel<AM, BM, BN, NBUF>,
                               hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    hipLaunchKernelGGL((mid_kernel<AM, BM, BN, NBUF>), dim3((unsigned)grid), dim3(NT), lds, st, a, M, K, A, lda);
    K3_LAUNCHED();
    return K3HIP_OK;
}

template <int AM>
int launch(MidArgs &a, int M, int K, const void *A, long lda, hipStream_t st)
{
    int ncu = 0, rc;
    if ((rc = cu_count(ncu))) return rc;
    long wide = 0;
    for (int i = 0; i < a.n; i++) wide += (a.s[i].rows + 127) / 128;
    // 128 x 128 once those tiles give every CU one: half the LDS reads per product. With two
    // buffers, so that two workgroups share a CU (three: one). At K = 256: the table of the z
    // product's rule in kda_layer.hip.
    if constexpr (AM == MID_A_16) {
        if (wide * ((M + 127) / 128) >= ncu) return launch_tile<AM, 128, 128, 2>(a, M, K, A, lda, st);
    }
    // 64 rows, and 128 columns once those tiles give every CU one; 64 below
    if (wide * ((M + 63) / 64) >= ncu) return launch_tile<AM, 64, 128, 3>(a, M, K, A, lda, st);
    return launch_tile<AM, 64, 64, AM == MID_A_16 ? 5 : 3>(a, M, K, A, lda, st);
}

}  // namespace

bool mid_supported(int K, const void *A, long lda, bool a_fp32)
{
    return K > 0 && K % BK == 0 && K <= (1 << 21) && lda >= K && lda <= (1 << 21) && lda % (a_fp32 ? 4 : 8) == 0 &&
           ((uintptr_t)A & 15) == 0;
}

int mid(int M, int K, int a_mode, const void *A, long lda, const MidSeg *segs, int n, hipStream_t st)
{
    if (M <= 0 || n <= 0) return K3HIP_OK;
    if (n > MID_SEGS || !mid_supported(K, A, lda, a_mode != MID_A_16))
        K3_FAIL(K3HIP_EUNSUPPORTED, "mid: %d weights, K=%d (a multiple of %d), lda=%ld, or A misaligned", n, K, BK, lda);
    MidArgs a{};
    for (int i = 0; i < n; i++) {
        MidSeg s = segs[i];
        if (s.rows <= 0) continue;
        if ((uintptr_t)s.B & 15) K3_FAIL(K3HIP_EUNSUPPORTED, "mid: weight %d misaligned", i);
        if (s.cols <= 0 || s.cols > s.rows) s.cols = s.rows;
        s.vec = ((uintptr_t)s.C & 15) == 0 && s.ldc % 4 == 0;
        a.s[a.n++] = s;
    }
    if (a.n == 0) return K3HIP_OK;
    return a_mode == MID_A_16 ? launch<MID_A_16>(a, M, K, A, lda, st) : launch<MID_A_SPLIT>(a, M, K, A, lda, st);
}

}  // namespace k3kda
