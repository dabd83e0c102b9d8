// gemv.hip -- fp32 products with quantised weights, C[m][n] = A[m] . W[n].
//
// The general-purpose kernel behind the reference's vec_matmul_* and
// matmul_quantized_batch entry points (src/ds3_metal.h:90-161).  Lanes split K
// in 32-weight units; a group of G lanes owns one row and decodes each unit
// once for a tile of up to 8 tokens staged in LDS.  It serves F32 rows, rows that
// are no multiple of 256, and the one- and two-token products that gemm32_ok
// leaves to it; the other quantised products run on k_gemm32.
//
// One token over long matrices (the output head, 151,936 x 2048, and the
// decode projections, src/ds3_engine.c:181-247) goes to k_gemv1 instead: the
// rows stream as one contiguous byte range per chunk of rows, not as the
// scattered unit loads of k_gemv.
#include "common.h"
#include "launch.h"
#include "rowstream.h"

namespace ds3k {

// ---------------------------------------------------------------------------
// k_gemv1: y[n] = x . W[n] for one token, Q4_K / Q6_K / Q8_0 rows of
// K = 2048 * UPL weights stored densely (row stride = row bytes) from a
// 16-byte aligned base.  Persistent workgroups walk chunks of R consecutive
// rows, one contiguous byte range each.  Every thread loads 16-byte pieces of
// a chunk into one of NS register sets in rotation (inline asm loads, waited
// by an asm s_waitcnt after which every register of the set is named), so
// NS - 1 chunks are in flight while one is decoded.  A landed chunk goes to
// one of two LDS buffers; each wave takes R/4 of its rows, each lane dots units
// lane + 64 q of a row from LDS with its x values, which stay in registers
// for the whole kernel with their 8-element sums (loaded once per
// workgroup), and a DPP wave sum gives the row's product.
// ---------------------------------------------------------------------------
bool gemv_type_ok(int type, int K);

#ifndef DS3_G1_ROWS
#define DS3_G1_ROWS 4               // rows per chunk at K = 2048 (half at 4096, at least 4)
#endif
// Persistent workgroups per CU.  6, but 3 for Q8_0 rows of 2048: of 6 five fit at
// once (87 VGPRs), and the sixth's share of the chunks runs after them alone;
// with 3 they all run, with as many bytes in flight as the memory needs.  MI355X, us
// per call with 3 / 5 / 6 on weights that come from memory: Q8_0 2048 -> 151,936
// 59.3 / 62.4 / 66.3, -> 20,000 12.2 / 13.8 / 15.6; 4096 -> 300,000 229 / 227 / 229;
// Q4_K 2048 -> 151,936 48.4 / 45.3 / 44.8; Q6_K 55.9 / 57.6 / 55.3.
#ifndef DS3_G1_WPC
#define DS3_G1_WPC 6
#endif
#ifndef DS3_G1_SETS
#define DS3_G1_SETS 2               // register sets of chunks in flight per workgroup
#endif

template <int TYPE, int UPL>
struct G1 {
    static constexpr int RB = G1Row<TYPE>::RB * UPL;             // bytes per row
    static constexpr int R = DS3_G1_ROWS / UPL < 4 ? 4 : DS3_G1_ROWS / UPL;   // rows per chunk (one per wave at least)
    static constexpr int CB = R * RB;                            // chunk bytes
    static constexpr int NL = (CB + G1_LOAD - 1) / G1_LOAD;      // 16-byte loads per thread and chunk
    static constexpr int BUF = NL * G1_LOAD;                     // LDS bytes per buffer
    static_assert(R % 4 == 0 && RB % 16 == 0, "whole rows per wave, 16-byte rows");
};

template <int TYPE, int UPL>
__global__ void __launch_bounds__(G1_TPB)
k_gemv1(const float *__restrict__ x, const uint8_t *__restrict__ W, float *__restrict__ y, int N, int nch)
{
    using P = G1<TYPE, UPL>;
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * P::BUF];
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    float xr[UPL][32], sx[UPL][4];                    // loaded after the first chunks go out
    auto compute = [&](const uint8_t *buf, int c) {
        // one row at a time: four rows' decoded weights at once cost the second wave per SIMD
#pragma unroll 1
        for (int i = 0; i < P::R / 4; i++) {
            const int r = wave + 4 * i;
            float acc = 0.f;
#pragma unroll
            for (int q = 0; q < UPL; q++) acc += g1_unit_dot<TYPE>(buf + r * P::RB, lane + 64 * q, xr[q], sx[q]);
            acc = g1_wave_total(acc);
            const int n = c * P::R + r;
            if (lane == WAVE - 1 && n < N) y[n] = acc;
        }
    };
    const int G = (int)gridDim.x;
    int c = (int)blockIdx.x;
    const int64_t lim = (int64_t)N * P::RB - 16;
    // NS register sets in rotation: chunk k of this workgroup (c = blockIdx.x
    // + k G) loads into set k mod NS, NS - 1 chunks ahead of the one being
    // decoded, and goes to LDS buffer k mod 2
    constexpr int NS = DS3_G1_SETS;
    static_assert(NS >= 2 && (NS - 1) * P::NL <= 63, "register sets in flight vs the vmcnt field");
    G1Set<P::NL> S[NS];
#pragma unroll
    for (int j = 0; j < NS; j++) S[j].issue(W, (int64_t)min(c + j * G, nch - 1) * P::CB, P::CB, lim);
    // x after the first chunks: the wait for x (vmcnt 0, in issue order)
    // then covers them too, one memory latency instead of two
    g1_load_x<TYPE, UPL>(x, lane, xr, sx);
    bool more = true;
    for (int k = 0; more; k += NS) {
#pragma unroll
        for (int j = 0; j < NS; j++) {
            if (more) {                                   // uniform over the workgroup
                S[j].template wait<(NS - 1) * P::NL>();   // the other sets' loads went out after this one's
                uint8_t *buf = lds + ((k + j) & 1) * P::BUF;
                S[j].to_lds(buf);
                __syncthreads();                          // every wave is done with this buffer's previous chunk
                S[j].issue(W, (int64_t)min(c + NS * G, nch - 1) * P::CB, P::CB, lim);
                compute(buf, c);
                c += G;
                more = c < nch;
            }
        }
    }
    // every set still has loads in flight: wait for them, naming the registers
#pragma unroll
    for (int j = 0; j < NS; j++) S[j].template wait<0>();
}

template <int TYPE, int UPL>
static hipError_t gemv1_t(const float *x, const uint8_t *w, float *y, int N, hipStream_t s)
{
    static int n_cu = 0;
    if (n_cu == 0) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n_cu <= 0)
            n_cu = 256;
    }
    const int nch = (N + G1<TYPE, UPL>::R - 1) / G1<TYPE, UPL>::R;
    constexpr int wpc = TYPE == T_Q8_0 && UPL == 1 ? 3 : DS3_G1_WPC;
    const int grid = nch < wpc * n_cu ? nch : wpc * n_cu;
    hipLaunchKernelGGL((k_gemv1<TYPE, UPL>), dim3((unsigned)grid), dim3(G1_TPB), 0, s, x, w, y, N, nch);
    return hipGetLastError();
}

// k_gemv1's shapes: one token, Q4_K / Q6_K / Q8_0, K = 2048 or 4096, dense
// rows from a 16-byte aligned base.
static bool gemv1_ok(int type, const uint8_t *w, uint64_t stride, int M, int K, const float *wnorm2)
{
    if (M != 1 || wnorm2 != nullptr || (K != 2048 && K != 4096) || ((uintptr_t)w & 15) != 0) return false;
    const int upl = K / 2048;
    switch (type) {
    case T_Q4_K: return stride == (uint64_t)G1Row<T_Q4_K>::RB * upl;
    case T_Q6_K: return stride == (uint64_t)G1Row<T_Q6_K>::RB * upl;
    case T_Q8_0: return stride == (uint64_t)G1Row<T_Q8_0>::RB * upl;
    default: return false;
    }
}

bool gemv1_path(int type, const uint8_t *w, uint64_t stride, int M, int K)
{
    return gemv_type_ok(type, K) && gemv1_ok(type, w, stride, M, K, nullptr);
}

static hipError_t launch_gemv1(int type, const float *x, const uint8_t *w, float *y, int N, int K, hipStream_t s)
{
    const bool two = K == 4096;
    switch (type) {
    case T_Q4_K: return two ? gemv1_t<T_Q4_K, 2>(x, w, y, N, s) : gemv1_t<T_Q4_K, 1>(x, w, y, N, s);
    case T_Q6_K: return two ? gemv1_t<T_Q6_K, 2>(x, w, y, N, s) : gemv1_t<T_Q6_K, 1>(x, w, y, N, s);
    case T_Q8_0: return two ? gemv1_t<T_Q8_0, 2>(x, w, y, N, s) : gemv1_t<T_Q8_0, 1>(x, w, y, N, s);
    default: return hipErrorInvalidValue;
    }
}

// ---------------------------------------------------------------------------
// k_gemm32: C[m][n] = A[m] . W[n] for a few rows of A, in fp32 on the matrix
// cores (v_mfma_f32_16x16x4_f32: fp32 operands, fp32 accumulation).
// k_gemv decodes every weight again for each group of 8 rows of A and takes
// one LDS read per multiply; here a weight is decoded once for 16 * MB rows
// and the products leave the VALU.
//
// A workgroup takes 16 rows of W and 16 * MB rows of A; its waves split K in
// steps of 256 (wave w takes steps w, w + NW, ...), so that the few-row
// products of an expert (27 x 2048 -> 768 is 48 such tiles) still put 8 waves
// on every tile.  Lane group g (lanes 16g..16g+15) decodes units g and g + 4
// of its row per step and reads A at the same K positions, so the MFMA's K
// order is a permutation shared by both operands.
//
// Sums: chains of 8 MFMAs (32 products, as long as k_gemv's lane sums), added
// as a tree over the unit, the step and, through LDS, the waves.  One chain
// per wave and step put the error against 64-bit sums at 2.9e-7 (relative
// L2, K = 2048) where k_gemv has 1.2e-7; this order has 1.2e-7 too.
//
// Measured (MI355X, us per call enqueued back to back, k_gemv before): 27 x
// 2048 -> 768 in Q4_K 73.4 -> 7.6, Q6_K 46.0 -> 8.7, Q8_0 128 -> 8.6; 63 x 2048
// -> 4096 480 / 259 / 920 -> 22 / 22 / 34; 40 x 4096 -> 8192 1215 / 657 / 2341
// -> 64 / 66 / 93 (42 / 41 / 29 TFLOP/s; 40 rows take a tile of 64).  Small
// products are bound by the launch and one or two memory latencies.  Large
// ones are bound by the return path of the vector memory, busy 80-85 % of the
// cycles (matrix units 30-44 %): each wave loads its A fragments itself, 64
// pieces of 16 bytes per load, and nothing is loaded ahead of its step.
// ---------------------------------------------------------------------------
typedef float g32_f4 __attribute__((ext_vector_type(4)));
typedef float g32_f4u __attribute__((ext_vector_type(4), aligned(4)));   // rows of A start on any float

constexpr int G32_TILE = 16;
constexpr int G32_STEP = 256;
constexpr int G32_MAX_WAVES = 8;

// unit_decode with Q8_0's 34 bytes read as 10 aligned dwords in three loads
// (any byte alignment) instead of two dwords for each code dword.
template <int TYPE>
__device__ __forceinline__ void g32_decode(const uint8_t *row, int u, float (&w)[32], int (&k0)[4])
{
    if constexpr (TYPE == T_Q8_0) {
        typedef uint32_t u4 __attribute__((ext_vector_type(4), aligned(4)));
        typedef uint32_t u2 __attribute__((ext_vector_type(2), aligned(4)));
        const uint8_t *blk = row + (size_t)u * 34;
        const uint32_t sh = (uint32_t)((uintptr_t)blk & 3);
        const uint8_t *p = blk - sh;
        const u4 a = *(const u4 *)p, b = *(const u4 *)(p + 16);
        const u2 c = *(const u2 *)(p + 32);
        const uint32_t q[10] = { a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, c.x, c.y };
        const float d = h2f(__builtin_amdgcn_alignbyte(q[1], q[0], sh) & 0xffffu);
        const bool up = sh >= 2;                     // the codes start at byte sh + 2
        const uint32_t cs = (sh + 2) & 3;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t v = __builtin_amdgcn_alignbyte(up ? q[i + 2] : q[i + 1], up ? q[i + 1] : q[i], cs);
#pragma unroll
            for (int j = 0; j < 4; j++) w[4 * i + j] = (float)(int8_t)byte_of(v, j) * d;
        }
#pragma unroll
        for (int s = 0; s < 4; s++) k0[s] = 32 * u + 8 * s;
    } else {
        unit_decode<TYPE>(row, u, w, k0);
    }
}

template <int TYPE, int MB>
__global__ void __launch_bounds__(WAVE * G32_MAX_WAVES)
k_gemm32(const float *__restrict__ A, int64_t lda, const uint8_t *__restrict__ W, uint64_t stride,
         float *__restrict__ C, int64_t ldc, int M, int N, int K)
{
    __shared__ g32_f4 part[G32_MAX_WAVES][MB][WAVE];
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
    const int g = lane >> 4, c = lane & 15;
    const int n = blockIdx.x * G32_TILE + c, m0 = blockIdx.y * G32_TILE * MB;
    // rows past the end repeat the last one; their results are not stored
    const uint8_t *row = W + (uint64_t)min(n, N - 1) * stride;
    const float *a[MB];
    g32_f4 acc[2][MB];
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
        a[mb] = A + (int64_t)min(m0 + G32_TILE * mb + c, M - 1) * lda;
        acc[0][mb] = acc[1][mb] = g32_f4{ 0.f, 0.f, 0.f, 0.f };
    }
    for (int s = wave; s < K / G32_STEP; s += nw)
#pragma unroll
        for (int hv = 0; hv < 2; hv++) {
            g32_f4 x[MB][8];
            float w[32];
            int k0[4];
            g32_decode<TYPE>(row, 8 * s + g + 4 * hv, w, k0);
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
#pragma unroll
                for (int i = 0; i < 8; i++) x[mb][i] = *(const g32_f4u *)(a[mb] + k0[i >> 1] + 4 * (i & 1));
            // chains of 8 MFMAs (32 products), added as a tree
            g32_f4 p[4][MB];
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int mb = 0; mb < MB; mb++) p[j][mb] = g32_f4{ 0.f, 0.f, 0.f, 0.f };
#pragma unroll
            for (int i = 0; i < 8; i++)
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int mb = 0; mb < MB; mb++)
                        p[j][mb] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[mb][2 * j + (i >> 2)][i & 3], w[8 * j + i],
                                                                       p[j][mb], 0, 0, 0);
#pragma unroll
            for (int mb = 0; mb < MB; mb++) acc[hv][mb] += (p[0][mb] + p[1][mb]) + (p[2][mb] + p[3][mb]);
        }
#pragma unroll
    for (int mb = 0; mb < MB; mb++) part[wave][mb][lane] = acc[0][mb] + acc[1][mb];
    __syncthreads();
    for (int mb = wave; mb < MB; mb += nw) {
        g32_f4 q[G32_MAX_WAVES];
#pragma unroll
        for (int w = 0; w < G32_MAX_WAVES; w++) q[w] = w < nw ? part[w][mb][lane] : g32_f4{ 0.f, 0.f, 0.f, 0.f };
        const g32_f4 v = ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int m = m0 + G32_TILE * mb + 4 * g + i;
            if (m < M && n < N) C[(int64_t)m * ldc + n] = v[i];
        }
    }
}

constexpr int GEMV_MT = 8;            // tokens per tile
constexpr int GEMV_TPB = 256;

template <int TYPE, int G>
__global__ void __launch_bounds__(GEMV_TPB)
k_gemv(const float *__restrict__ A, int64_t lda, const uint8_t *__restrict__ W, uint64_t stride,
       float *__restrict__ C, int64_t ldc, int M, int N, int K, int mt_max, int rows_per_wg,
       float *__restrict__ wnorm2)
{
    extern __shared__ float xs[];     // [mt][K]
    const int m0 = blockIdx.y * mt_max;
    const int mt = min(mt_max, M - m0);
    for (int i = threadIdx.x; i < mt * K; i += GEMV_TPB) {
        const int m = i / K, k = i - m * K;
        xs[i] = A[(int64_t)(m0 + m) * lda + k];
    }
    __syncthreads();

    constexpr int GPW = WAVE / G;
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    const int gl = lane % G, grp = lane / G;
    const int U = K / 32;
    const bool want_norm = (wnorm2 != nullptr) && blockIdx.y == 0;
    for (int r = wave * GPW + grp; r < rows_per_wg; r += (GEMV_TPB / WAVE) * GPW) {
        const int n = blockIdx.x * rows_per_wg + r;
        const bool valid = n < N;
        float acc[GEMV_MT];
#pragma unroll
        for (int m = 0; m < GEMV_MT; m++) acc[m] = 0.f;
        float w2 = 0.f;
        if (valid) {
            const uint8_t *row = W + (size_t)n * stride;
            for (int u = gl; u < U; u += G) {
                float w[32];
                int k0[4];
                unit_decode<TYPE>(row, u, w, k0);
                if (want_norm) {
#pragma unroll
                    for (int i = 0; i < 32; i++) w2 += w[i] * w[i];
                }
#pragma unroll
                for (int m = 0; m < GEMV_MT; m++) {
                    if (m < mt) {
                        const float *xm = xs + m * K;
                        float a = acc[m];
#pragma unroll
                        for (int s = 0; s < 4; s++)
#pragma unroll
                            for (int i = 0; i < 8; i++) a += w[8 * s + i] * xm[k0[s] + i];
                        acc[m] = a;
                    }
                }
            }
        }
#pragma unroll
        for (int m = 0; m < GEMV_MT; m++) acc[m] = group_sum<G>(acc[m]);
        if (want_norm) w2 = group_sum<G>(w2);
        if (valid && gl == 0) {
#pragma unroll
            for (int m = 0; m < GEMV_MT; m++)
                if (m < mt) C[(int64_t)(m0 + m) * ldc + n] = acc[m];
            if (want_norm) wnorm2[n] = w2;
        }
    }
}

bool gemv_type_ok(int type, int K)
{
    if (K <= 0) return false;
    switch (type) {
    case T_F32:  return K % 32 == 0;
    case T_Q8_0: return K % 32 == 0;
    case T_Q4_K:
    case T_Q6_K: return K % 256 == 0;
    default:     return false;
    }
}

template <int TYPE>
static hipError_t gemv_type(int G, dim3 grid, size_t lds, hipStream_t s, const float *A, int64_t lda,
                            const uint8_t *w, uint64_t stride, float *C, int64_t ldc, int M, int N, int K,
                            int mt, int rpw, float *wn)
{
#define DS3_GEMV_CASE(GV)                                                                       \
    case GV:                                                                                    \
        hipLaunchKernelGGL((k_gemv<TYPE, GV>), grid, dim3(GEMV_TPB), lds, s, A, lda, w, stride, C, \
                           ldc, M, N, K, mt, rpw, wn);                                          \
        break;
    switch (G) {
        DS3_GEMV_CASE(1) DS3_GEMV_CASE(2) DS3_GEMV_CASE(4) DS3_GEMV_CASE(8)
        DS3_GEMV_CASE(16) DS3_GEMV_CASE(32) DS3_GEMV_CASE(64)
    default: return hipErrorInvalidValue;
    }
#undef DS3_GEMV_CASE
    return hipGetLastError();
}

// k_gemm32's grid: as many rows of A per workgroup as leave two workgroups
// per CU.
static GemvPlan gemm32_plan(int M, int N, int K)
{
    const int64_t nt = ((int64_t)N + G32_TILE - 1) / G32_TILE;
    const int steps = K / G32_STEP;
    int mb = 4;
    while (mb > 1 && (M <= G32_TILE * mb / 2 || nt * ((M + G32_TILE * mb - 1) / (G32_TILE * mb)) < 512)) mb /= 2;
    return { GEMV_MFMA, (unsigned)nt, (unsigned)((M + G32_TILE * mb - 1) / (G32_TILE * mb)),
             (unsigned)(WAVE * (steps < G32_MAX_WAVES ? steps : G32_MAX_WAVES)), mb, G32_TILE };
}

template <int TYPE>
static hipError_t gemm32_type(const GemvPlan &p, const float *A, int64_t lda, const uint8_t *w, uint64_t stride,
                              float *C, int64_t ldc, int M, int N, int K, hipStream_t s)
{
    const dim3 grid(p.gx, p.gy), block(p.tpb);
    switch (p.m_tile) {
    case 1: hipLaunchKernelGGL((k_gemm32<TYPE, 1>), grid, block, 0, s, A, lda, w, stride, C, ldc, M, N, K); break;
    case 2: hipLaunchKernelGGL((k_gemm32<TYPE, 2>), grid, block, 0, s, A, lda, w, stride, C, ldc, M, N, K); break;
    default: hipLaunchKernelGGL((k_gemm32<TYPE, 4>), grid, block, 0, s, A, lda, w, stride, C, ldc, M, N, K); break;
    }
    return hipGetLastError();
}

// k_gemm32's shapes: quantised rows of whole 256-wide steps, wherever it beats
// k_gemv.  Measured on MI355X, us per call back to back, k_gemv / k_gemm32:
//   3 rows of A and more: it wins (3 x 256 -> 64 4.7 / 4.2 in Q4_K, 27 x 2048 ->
//     768 73 / 7.6; the worst is Q6_K 3 x 1280 -> 16,384, 1.08 times)
//   2 rows: it wins (2 x 2048 -> 768 10.2 / 7.0, 8.6 / 7.6, 13.6 / 6.6 in Q4_K, Q6_K,
//     Q8_0) but for K = 256 in Q4_K and Q6_K, where a workgroup is one wave (-> 768
//     4.1 / 4.5; -> 12,288 in Q4_K 0.84 times, -> 24,000 in Q6_K 0.89), and Q6_K at
//     K = 1280, whose five waves share four SIMDs (-> 32,000 26.3 / 28.6)
//   one row fills 1/16 of a tile, but every lane group decodes its own unit.
//     Below 2048 rows of W (1024 -> 700 5.9 / 6.4) and at an odd number of steps
//     (768 -> 32,000 11.2 / 13.8) k_gemv wins.
//     Q8_0: it wins (512 -> 4096 4.9 / 4.3, 1024 -> 20,000 44 / 10.0)
//     Q4_K: it wins (1024 -> 20,000 26 / 9.8, 1536 -> 4096 7.6 / 5.3), at K = 512
//       from 12,288 rows (0.69 times; -> 8192 5.3 / 5.4)
//     Q6_K: its decode costs more.  It wins where K / 32 units are whole turns of
//       32 lanes and more than half the CUs get a tile (1024 -> 4096 5.9 / 5.0; ->
//       2048 4.7 / 5.0), else up to one tile a CU (1536 -> 4096 7.0 / 6.2; -> 8192
//       8.0 / 9.8, -> 100,000 76 / 92; past one tile a CU the two cross several
//       times, with 2560 -> 20,000 32 / 28 the other way), at K = 512 from 12,288
//       rows (-> 32,000 0.97 times; -> 8192 4.8 / 6.0)
static bool gemm32_ok(int type, int M, int N, int K, const float *wnorm2)
{
    if (wnorm2 != nullptr || K % G32_STEP != 0 || (type != T_Q4_K && type != T_Q6_K && type != T_Q8_0)) return false;
    // a launch takes fewer than 2^32 threads in x, which 2^27 rows of W reach
    // with 8 waves per 16 rows; k_gemv's workgroups take any number of rows
    const GemvPlan p = gemm32_plan(M, N, K);
    if ((uint64_t)p.gx * p.tpb >= 1ull << 32) return false;
    if (M >= 3) return true;
    if (M == 2) {
        if (type == T_Q8_0) return true;
        if (K == G32_STEP) return N >= (type == T_Q4_K ? 12288 : 24000);
        return type != T_Q6_K || K != 5 * G32_STEP || N <= 12288;
    }
    if (N < 2048 || K % (2 * G32_STEP) != 0) return false;
    if (type == T_Q8_0) return true;
    if (K == 2 * G32_STEP) return N >= 12288;
    if (type == T_Q4_K) return true;
    return K % 1024 == 0 ? N > 2048 : N <= 4096;
}

// Lanes per row: the largest power of two dividing the unit count (no idle
// lanes), capped at 64.
static int lanes_per_row(int units)
{
    int g = 1;
    while (g < 64 && units % (2 * g) == 0) g *= 2;
    return g;
}

GemvPlan gemv_plan(int type, const uint8_t *w, uint64_t stride, int M, int N, int K, const float *wnorm2)
{
    if (gemv1_ok(type, w, stride, M, K, wnorm2)) return { GEMV_ONE, 0, 0, G1_TPB, 1, 0 };
    if (gemm32_ok(type, M, N, K, wnorm2)) return gemm32_plan(M, N, K);
    const int gpw = WAVE / lanes_per_row(K / 32);
    const int rows_step = (GEMV_TPB / WAVE) * gpw;            // rows one pass of the WG covers
    int mt = GEMV_MT;
    while (mt > 1 && (size_t)mt * K * sizeof(float) > 64 * 1024) mt /= 2;
    const int gy = (M + mt - 1) / mt;
    // Aim for ~512 workgroups: fewer rows per WG when there are few token tiles.
    const int steps_total = (N + rows_step - 1) / rows_step;
    int want_x = 512 / gy;
    if (want_x < 1) want_x = 1;
    int steps_per_wg = (steps_total + want_x - 1) / want_x;
    if (steps_per_wg < 1) steps_per_wg = 1;
    const int rpw = steps_per_wg * rows_step;
    return { GEMV_GENERAL, (unsigned)((N + rpw - 1) / rpw), (unsigned)gy, GEMV_TPB, mt, rpw };
}

hipError_t launch_gemv(int type, const float *A, int64_t lda, const uint8_t *w, uint64_t stride,
                       float *C, int64_t ldc, int M, int N, int K, float *wnorm2, hipStream_t s)
{
    if (!gemv_type_ok(type, K) || M <= 0 || N <= 0) return hipErrorInvalidValue;
    const GemvPlan p = gemv_plan(type, w, stride, M, N, K, wnorm2);
    if (p.kernel == GEMV_ONE) return launch_gemv1(type, A, w, C, N, K, s);
    if (p.kernel == GEMV_MFMA) {
        switch (type) {
        case T_Q8_0: return gemm32_type<T_Q8_0>(p, A, lda, w, stride, C, ldc, M, N, K, s);
        case T_Q4_K: return gemm32_type<T_Q4_K>(p, A, lda, w, stride, C, ldc, M, N, K, s);
        default:     return gemm32_type<T_Q6_K>(p, A, lda, w, stride, C, ldc, M, N, K, s);
        }
    }
    const int G = lanes_per_row(K / 32), mt = p.m_tile, rpw = p.rows_per_wg;
    const dim3 grid(p.gx, p.gy);
    const size_t lds = (size_t)mt * K * sizeof(float);
    switch (type) {
    case T_F32:  return gemv_type<T_F32>(G, grid, lds, s, A, lda, w, stride, C, ldc, M, N, K, mt, rpw, wnorm2);
    case T_Q8_0: return gemv_type<T_Q8_0>(G, grid, lds, s, A, lda, w, stride, C, ldc, M, N, K, mt, rpw, wnorm2);
    case T_Q4_K: return gemv_type<T_Q4_K>(G, grid, lds, s, A, lda, w, stride, C, ldc, M, N, K, mt, rpw, wnorm2);
    case T_Q6_K: return gemv_type<T_Q6_K>(G, grid, lds, s, A, lda, w, stride, C, ldc, M, N, K, mt, rpw, wnorm2);
    default:     return hipErrorInvalidValue;
    }
}

}  // namespace ds3k
