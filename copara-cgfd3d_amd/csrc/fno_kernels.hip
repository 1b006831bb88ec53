// Kernels of the Fourier-neural-operator surrogate: every matrix product of
// its forward and backward passes (lifting, pointwise channel mixing,
// per-mode spectral mixing, the truncated transforms, projection, and their
// weight and input gradients) with the bias, residual and GELU of a layer
// fused into the product's epilogue; the GELU backward; and the Adam update
// of all parameters in one launch.
//
//   C[z] = act((C[z] +) A[z] * B[z] + bias + D[z]),  z = 0 .. batch-1
//   (and, on request, C[z] again in bf16: the operand of the next product)
//   A: M x K bf16, element (m, k) at A + z*sAz + m*sAm + k*sAk
//   B: K x N bf16, element (k, n) at B + z*sBz + k*sBk + n*sBn
//   C: M x N fp32, element (m, n) at C + z*sCz + m*sCm + n
//
// General strides let the backward pass read transposed operands in place.
// Products are exact in FP32 and accumulate in FP32 on the matrix cores
// (v_mfma_f32_16x16x32_bf16, gfx950).
#include <hip/hip_runtime.h>

#include "fno_network.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));

constexpr int BM = 64, BN = 64, BK = 32, PAD = 8;

// How a block stages an operand tile: 0 element by element (any strides),
// 1 eight k-consecutive elements per 16-byte load (unit k stride), 2 eight
// m- (or n-) consecutive elements per 16-byte load, transposed into LDS.
// Modes 1 and 2 need a 16-byte aligned base and the other strides in
// multiples of 8 elements; edge groups fall back to single loads.
enum { STAGE_ANY = 0, STAGE_K = 1, STAGE_MN = 2 };

struct GemmArgs {
    const unsigned short *A, *B;
    float *C;
    long sAz, sAm, sAk, sBz, sBk, sBn, sCz, sCm;
    int M, N, K, accumulate, amode, bmode, vec;
    // epilogue
    const float *bias; // [N] or null
    const float *D;    // addend, (m, n) at D + z*sDz + m*sDm + n, or null
    long sDz, sDm;
    float *pre;        // the value before the activation, laid out as C, or null
    int act;           // CGFD_FNO_ACT_*
    unsigned short *Cb; // bf16 copy of the result, (m, n) at Cb + z*sEz + m*sEm + n, or null
    long sEz, sEm;
    // VEC = 2: the result goes to Cb alone, with each index split in two,
    // (z/zq)*sEz1 + (z%zq)*sEz + (m/mq)*sEm1 + (m%mq)*sEm + (n/nq)*sEn1 + n%nq
    int zq, mq, nq;
    long sEz1, sEm1, sEn1;
};

// One lane's share of a 64 x 32 operand tile (rows r0.., k0..) whose element
// (r, k) sits at P + r*sR + k*sK: eight bf16 values, loaded into registers
// so that the next tile's loads overlap the current tile's products.
// EX = 1: no group of eight crosses the operand's edge (K a multiple of 8 in mode
// K, R in mode MN), so a share is loaded whole or is zero.  The element-wise
// path for crossing groups takes 30 registers: without it 6-8 instead of 4-5
// wavefronts fit a SIMD, and a training batch (32 x 80 x 80, width 64) takes 1604
// instead of 1683 us on the GPU.  Fetching 2 or 3 tiles ahead instead of one
// gave nothing (1633, 1682 us).
template <int MODE, int EX>
__device__ __forceinline__ u16x8 fetch(const unsigned short *P, long sR, long sK, int r0, int k0, int R, int K,
                                       int tid)
{
    u16x8 v = 0;
    if (MODE == STAGE_MN) {
        // 8 consecutive rows at one k
        const int r = r0 + (tid & 7) * 8, k = k0 + (tid >> 3);
        if (k < K && r + (EX ? 0 : 7) < R) {
            v = *reinterpret_cast<const u16x8 *>(P + r * sR + k * sK);
        } else if (!EX) {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = (k < K && r + i < R) ? P[(r + i) * sR + k * sK] : (unsigned short)0;
        }
    } else {
        // 8 consecutive k of one row
        const int r = r0 + (tid >> 2), k = k0 + (tid & 3) * 8;
        if (MODE == STAGE_K && r < R && k + (EX ? 0 : 7) < K) {
            v = *reinterpret_cast<const u16x8 *>(P + r * sR + k);
        } else if (MODE == STAGE_ANY || !EX) {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = (r < R && k + j < K) ? P[r * sR + (k + j) * sK] : (unsigned short)0;
        }
    }
    return v;
}

// Store a fetched share into T[r][k] (k contiguous in LDS).
template <int MODE>
__device__ __forceinline__ void park(unsigned short (*T)[BK + PAD], u16x8 v, int tid)
{
    if (MODE == STAGE_MN) {
        const int rg = (tid & 7) * 8, kk = tid >> 3;
#pragma unroll
        for (int i = 0; i < 8; ++i) T[rg + i][kk] = v[i];
    } else {
        *reinterpret_cast<u16x8 *>(&T[tid >> 2][(tid & 3) * 8]) = v;
    }
}

// bf16 of an fp32 value, rounded to nearest even (NaN kept quiet)
__device__ __forceinline__ unsigned short to_bf16(float f)
{
    unsigned u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x007fffffu)) return (unsigned short)((u >> 16) | 0x40);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

// GELU, erf form: x/2 (1 + erf(x/sqrt 2)), and its derivative
// Phi(x) + x phi(x).
__device__ __forceinline__ float gelu(float x) { return x * 0.5f * (1.0f + erff(x * 0.70710678118654752f)); }

__device__ __forceinline__ float gelu_grad(float x)
{
    const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
    const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
    return cdf + x * pdf;
}

// 256 lanes = 4 wavefronts; wavefront w owns the 32x32 block
// (32*(w/2), 32*(w%2)) of the 64x64 output tile as 2x2 MFMA 16x16 blocks.
// A and B tiles are staged in LDS with K contiguous, so each lane reads its
// 8 consecutive k values of a row (A) or column (B) as one 16-byte vector.
// Two LDS buffers: the next tile is fetched into registers before the
// current tile's products and parked in the other buffer after them, so one
// barrier per K step suffices.
//
// The products here have K <= 160 and are bound by HBM: the epilogue's streams
// decide (a pointwise layer of 204800 x 64 x 64 reads 26 MB of A and 52 MB of
// the spectral branch, and writes 131 MB).  The operands enter the MFMA
// swapped, so that a lane ends up with 4 consecutive columns of a row: with
// VEC = 1 every epilogue stream moves 16 bytes per lane (bf16: 8), and the
// addend is fetched before the K loop.  That layer: 62 -> 44 us (4.2 TB/s);
// 262144 rows with residual and GELU 110 -> 56 us.  VEC = 0 takes any
// alignment, element by element.  VEC = 2 stores the product in bf16 only, at
// an address split by index (the spectral layer's transposes).
template <int AM, int BMODE, int VEC, int EX>
__global__ void __launch_bounds__(256) gemm_bf16_kernel(GemmArgs g)
{
    __shared__ __attribute__((aligned(16))) unsigned short As[2][BM][BK + PAD];
    __shared__ __attribute__((aligned(16))) unsigned short Bs[2][BN][BK + PAD];
    const int z = blockIdx.z, m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const unsigned short *A = g.A + z * g.sAz;
    const unsigned short *B = g.B + z * g.sBz;
    float *C = VEC == 2 ? nullptr : g.C + z * g.sCz;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    f32x4 acc[2][2];
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float *D = VEC != 2 && g.D ? g.D + z * g.sDz : nullptr;
    float *pre = VEC != 2 && g.pre ? g.pre + z * g.sCz : nullptr;
    unsigned short *Cb = VEC == 2 ? g.Cb + (z / g.zq) * g.sEz1 + (z % g.zq) * g.sEz : g.Cb ? g.Cb + z * g.sEz : nullptr;
    // lane l holds row l%16 and columns 4*(l/16) .. +3 of each 16x16 block
    const int mr = m0 + wm + (lane & 15), nc = n0 + wn + (lane >> 4) * 4;
    // A rows are m (stride sAm), B "rows" are n (stride sBn)
    u16x8 na = fetch<AM, EX>(A, g.sAm, g.sAk, m0, 0, g.M, g.K, tid);
    u16x8 nb = fetch<BMODE, EX>(B, g.sBn, g.sBk, n0, 0, g.N, g.K, tid);
    f32x4 dv[2][2];
    if (VEC == 1) {
#pragma unroll
        for (int bi = 0; bi < 2; ++bi)
#pragma unroll
            for (int bj = 0; bj < 2; ++bj) {
                const int m = mr + bi * 16, n = nc + bj * 16;
                if (D && m < g.M && n < g.N) dv[bi][bj] = *reinterpret_cast<const f32x4 *>(D + m * g.sDm + n);
            }
    }

    park<AM>(As[0], na, tid);
    park<BMODE>(Bs[0], nb, tid);
    __syncthreads();
    int cur = 0;
    for (int k0 = 0; k0 < g.K; k0 += BK) {
        const bool more = k0 + BK < g.K;
        if (more) {
            na = fetch<AM, EX>(A, g.sAm, g.sAk, m0, k0 + BK, g.M, g.K, tid);
            nb = fetch<BMODE, EX>(B, g.sBn, g.sBk, n0, k0 + BK, g.N, g.K, tid);
        }
        const int kq = (lane >> 4) * 8;
#pragma unroll
        for (int bi = 0; bi < 2; ++bi) {
            const bf16x8 a = *reinterpret_cast<const bf16x8 *>(&As[cur][wm + bi * 16 + (lane & 15)][kq]);
#pragma unroll
            for (int bj = 0; bj < 2; ++bj) {
                const bf16x8 b = *reinterpret_cast<const bf16x8 *>(&Bs[cur][wn + bj * 16 + (lane & 15)][kq]);
                acc[bi][bj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, acc[bi][bj], 0, 0, 0);
            }
        }
        if (more) {
            park<AM>(As[cur ^ 1], na, tid);
            park<BMODE>(Bs[cur ^ 1], nb, tid);
        }
        __syncthreads();
        cur ^= 1;
    }
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int bj = 0; bj < 2; ++bj) {
            const int m = mr + bi * 16, n = nc + bj * 16;
            if (VEC == 2) {
                if (m >= g.M || n >= g.N) continue; // N and nq are multiples of 4
                u16x4 e;
#pragma unroll
                for (int i = 0; i < 4; ++i) e[i] = to_bf16(acc[bi][bj][i]);
                *reinterpret_cast<u16x4 *>(Cb + (m / g.mq) * g.sEm1 + (m % g.mq) * g.sEm + (n / g.nq) * g.sEn1 +
                                           n % g.nq) = e;
            } else if (VEC == 1) {
                if (m >= g.M || n >= g.N) continue; // N is a multiple of 4
                f32x4 v = acc[bi][bj];
                if (g.accumulate) v = *reinterpret_cast<const f32x4 *>(C + m * g.sCm + n) + v;
                if (g.bias) v = v + *reinterpret_cast<const f32x4 *>(g.bias + n);
                if (D) v = v + dv[bi][bj];
                if (pre) *reinterpret_cast<f32x4 *>(pre + m * g.sCm + n) = v;
                if (g.act == CGFD_FNO_ACT_GELU) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = gelu(v[i]);
                }
                if (g.C) *reinterpret_cast<f32x4 *>(C + m * g.sCm + n) = v;
                if (Cb) {
                    u16x4 e;
#pragma unroll
                    for (int i = 0; i < 4; ++i) e[i] = to_bf16(v[i]);
                    *reinterpret_cast<u16x4 *>(Cb + m * g.sEm + n) = e;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (m >= g.M || n + i >= g.N) continue;
                    float *p = C + m * g.sCm + n + i;
                    float v = acc[bi][bj][i];
                    if (g.accumulate) v = *p + v;
                    if (g.bias) v = v + g.bias[n + i];
                    if (D) v = v + D[m * g.sDm + n + i];
                    if (pre) pre[m * g.sCm + n + i] = v;
                    if (g.act == CGFD_FNO_ACT_GELU) v = gelu(v);
                    *p = v;
                    if (Cb) Cb[m * g.sEm + n + i] = to_bf16(v);
                }
            }
        }
}

template <int AM, int BMODE>
void launch_v(const GemmArgs &g, dim3 grid, hipStream_t s)
{
    // whole groups of eight along the staged index of both operands
    const bool ex = (AM != STAGE_K || g.K % 8 == 0) && (AM != STAGE_MN || g.M % 8 == 0) &&
                    (BMODE != STAGE_K || g.K % 8 == 0) && (BMODE != STAGE_MN || g.N % 8 == 0);
    if (g.vec == 2 && ex) hipLaunchKernelGGL((gemm_bf16_kernel<AM, BMODE, 2, 1>), grid, dim3(256), 0, s, g);
    else if (g.vec == 2) hipLaunchKernelGGL((gemm_bf16_kernel<AM, BMODE, 2, 0>), grid, dim3(256), 0, s, g);
    else if (g.vec && ex) hipLaunchKernelGGL((gemm_bf16_kernel<AM, BMODE, 1, 1>), grid, dim3(256), 0, s, g);
    else if (g.vec) hipLaunchKernelGGL((gemm_bf16_kernel<AM, BMODE, 1, 0>), grid, dim3(256), 0, s, g);
    else hipLaunchKernelGGL((gemm_bf16_kernel<AM, BMODE, 0, 0>), grid, dim3(256), 0, s, g);
}

template <int AM>
void launch_b(const GemmArgs &g, dim3 grid, hipStream_t s)
{
    if (g.bmode == STAGE_K) launch_v<AM, STAGE_K>(g, grid, s);
    else if (g.bmode == STAGE_MN) launch_v<AM, STAGE_MN>(g, grid, s);
    else launch_v<AM, STAGE_ANY>(g, grid, s);
}

// 4-element accesses to an epilogue stream: the base aligned to 4 elements,
// both strides multiples of 4
bool vec4(const void *p, long sz, long sm, int elem)
{
    return p == nullptr || ((reinterpret_cast<unsigned long>(p) % (4 * elem)) == 0 && sz % 4 == 0 && sm % 4 == 0);
}

// what a layer's kernels access 16 bytes at a time without another way (null
// where a pointer is optional)
template <typename... P> bool aligned16(P... p)
{
    return ((reinterpret_cast<unsigned long>(p) | ...) & 15) == 0;
}

// staging mode of an operand: unit stride along k (STAGE_K) or along its
// rows (STAGE_MN), with a 16-byte aligned base and the other strides in
// multiples of 8 elements; otherwise element by element
int stage_mode(const void *p, long sZ, long sR, long sK)
{
    if ((reinterpret_cast<unsigned long>(p) & 15) != 0 || sZ % 8 != 0) return STAGE_ANY;
    if (sK == 1 && sR % 8 == 0) return STAGE_K;
    if (sR == 1 && sK % 8 == 0) return STAGE_MN;
    return STAGE_ANY;
}

void launch_gemm(const GemmArgs &g, int batch, hipStream_t s)
{
    const dim3 grid((unsigned)((g.N + BN - 1) / BN), (unsigned)((g.M + BM - 1) / BM), (unsigned)batch);
    if (g.amode == STAGE_K) launch_b<STAGE_K>(g, grid, s);
    else if (g.amode == STAGE_MN) launch_b<STAGE_MN>(g, grid, s);
    else launch_b<STAGE_ANY>(g, grid, s);
}

// One operand of a product inside a layer: element (r, k) of batch z at
// p + z*sz + r*sr + k*sk.
struct Operand {
    const void *p;
    long sz, sr, sk;
};

// Where a bf16-only product goes: plain rows of n, or an address split by index.
struct Place {
    void *p;
    int zq, mq, nq;
    long sz1, sz, sm1, sm, sn1;
};

Place rows(void *p, long sz, long sm) { return {p, 1 << 30, 1 << 30, 1 << 30, 0, sz, 0, sm, 0}; }

// bf16-only product; N and every stride and split of the place are multiples
// of 4, its base aligned to 8 bytes
void product_bf16(Operand a, Operand b, Place c, int M, int N, int K, int batch, hipStream_t s)
{
    GemmArgs g{};
    g.A = (const unsigned short *)a.p;
    g.B = (const unsigned short *)b.p;
    g.sAz = a.sz;
    g.sAm = a.sr;
    g.sAk = a.sk;
    g.sBz = b.sz;
    g.sBn = b.sr;
    g.sBk = b.sk;
    g.M = M;
    g.N = N;
    g.K = K;
    g.amode = stage_mode(a.p, a.sz, a.sr, a.sk);
    g.bmode = stage_mode(b.p, b.sz, b.sr, b.sk);
    g.vec = 2;
    g.Cb = (unsigned short *)c.p;
    g.zq = c.zq;
    g.mq = c.mq;
    g.nq = c.nq;
    g.sEz1 = c.sz1;
    g.sEz = c.sz;
    g.sEm1 = c.sm1;
    g.sEm = c.sm;
    g.sEn1 = c.sn1;
    launch_gemm(g, batch, s);
}

// The realified mode-mixing weights [[re, im], [-im, re]] of every mode in bf16
// (p, 2C x 2C), from fp32 (p, C x C) each; and, from block nspec on, the nw
// pointwise weights in bf16.  Four elements per lane; C is a multiple of 4.
__global__ void __launch_bounds__(256) layer_weights_kernel(const float *__restrict__ re, const float *__restrict__ im,
                                                            unsigned short *__restrict__ wr, long nspec4, int C,
                                                            const float *__restrict__ w,
                                                            unsigned short *__restrict__ wb, int nw, int nspec)
{
    if ((int)blockIdx.x >= nspec) {
        const int i = (blockIdx.x - nspec) * 256 + threadIdx.x;
        if (i < nw) wb[i] = to_bf16(w[i]);
        return;
    }
    const long q = (long)blockIdx.x * 256 + threadIdx.x;
    if (q >= nspec4) return;
    const f32x4 a = reinterpret_cast<const f32x4 *>(re)[q], b = reinterpret_cast<const f32x4 *>(im)[q];
    const long row = q * 4 / C; // p * C + i
    const int j = (int)(q * 4 % C);
    const long p = row / C;
    const int i = (int)(row % C);
    u16x4 r, c, n;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        r[k] = to_bf16(a[k]);
        c[k] = to_bf16(b[k]);
        n[k] = to_bf16(-b[k]);
    }
    unsigned short *o = wr + p * 4 * C * C;
    *reinterpret_cast<u16x4 *>(o + (long)i * 2 * C + j) = r;
    *reinterpret_cast<u16x4 *>(o + (long)i * 2 * C + C + j) = c;
    *reinterpret_cast<u16x4 *>(o + (long)(C + i) * 2 * C + j) = n;
    *reinterpret_cast<u16x4 *>(o + (long)(C + i) * 2 * C + C + j) = r;
}

// gradients of the two parts from that of the realified weights
__global__ void __launch_bounds__(256) layer_weight_grads_kernel(const float *__restrict__ gw, float *__restrict__ gre,
                                                                 float *__restrict__ gim, long nspec4, int C)
{
    const long q = (long)blockIdx.x * 256 + threadIdx.x;
    if (q >= nspec4) return;
    const long row = q * 4 / C, p = row / C;
    const int j = (int)(q * 4 % C), i = (int)(row % C);
    const float *o = gw + p * 4 * C * C;
    const f32x4 rr = *reinterpret_cast<const f32x4 *>(o + (long)i * 2 * C + j);
    const f32x4 ri = *reinterpret_cast<const f32x4 *>(o + (long)i * 2 * C + C + j);
    const f32x4 ir = *reinterpret_cast<const f32x4 *>(o + (long)(C + i) * 2 * C + j);
    const f32x4 ii = *reinterpret_cast<const f32x4 *>(o + (long)(C + i) * 2 * C + C + j);
    reinterpret_cast<f32x4 *>(gre)[q] = rr + ii;
    reinterpret_cast<f32x4 *>(gim)[q] = ri - ir;
}

// Backward of a layer's epilogue over a block of GROUP rows of N columns: gz =
// gy * GELU'(pre) (pre null: gz = gy), its bf16 copy, gz itself on request, and
// the block's column sums, which the bias gradient adds up.  Each lane keeps V
// columns (N a multiple of V, N/V at most 256), so the sums cost no second pass
// over gz.  Bound by HBM: 204800 x 64 with GELU 25 us (5.2 TB/s) without gz,
// where the GELU backward (38 us) and the sums (22 us) were two passes.
// At 64 / 128 / 256 rows per block, with the weight gradient: 204800 x 64 63 / 56 / 57
// us, 262144 x 64 73 / 62 / 58, 16384 x 64 21 / 21 / 25, 65536 x 256 111 / 115 / 137.
constexpr int GROUP = 128;
template <int V>
__global__ void __launch_bounds__(256) layer_grad_kernel(const float *__restrict__ gy, const float *__restrict__ pre,
                                                         float *__restrict__ gz, unsigned short *__restrict__ gzb,
                                                         float *__restrict__ sums, long R, int N)
{
    typedef float fv __attribute__((ext_vector_type(V)));
    typedef unsigned short uv __attribute__((ext_vector_type(V)));
    __shared__ fv part[256];
    const int cols = N / V, per = 256 / cols; // rows in flight
    const int tid = threadIdx.x, c = tid % cols, r = tid / cols;
    const long r0 = (long)blockIdx.x * GROUP, r1 = r0 + GROUP < R ? r0 + GROUP : R;
    fv sum = 0.f;
    if (r < per)
        for (long i = r0 + r; i < r1; i += per) {
            const long o = i * cols + c;
            fv v = reinterpret_cast<const fv *>(gy)[o];
            if (pre) {
                const fv x = reinterpret_cast<const fv *>(pre)[o];
#pragma unroll
                for (int j = 0; j < V; ++j) v[j] = v[j] * gelu_grad(x[j]);
            }
            uv e;
#pragma unroll
            for (int j = 0; j < V; ++j) e[j] = to_bf16(v[j]);
            reinterpret_cast<uv *>(gzb)[o] = e;
            if (gz) reinterpret_cast<fv *>(gz)[o] = v;
            sum = sum + v;
        }
    part[tid] = sum;
    __syncthreads();
    if (tid < cols) {
        for (int k = 1; k < per; ++k) sum = sum + part[tid + k * cols];
        reinterpret_cast<fv *>(sums)[(long)blockIdx.x * cols + tid] = sum;
    }
}

// out[i] = sum over n of part[n][i] for the weight gradient (first blocks) and
// the bias gradient, summed in double.  1024 lanes: 1024/SL columns, each in SL
// slices.  Many parts of few columns need the slices to fill the chip
// (262144 x 64 x 64, 1024 parts, with the whole gradient: 62 us with 16 slices,
// 188 with 1); with few parts most slices have none (1024 x 8192 x 256, 4 parts:
// 120 us with 16, 75 with 1).
template <int SL>
__global__ void __launch_bounds__(1024) layer_reduce_kernel(const float *__restrict__ wpart, int nw, int W,
                                                            float *__restrict__ gw, const float *__restrict__ bpart,
                                                            int nb, int N, float *__restrict__ gb, int wblocks)
{
    constexpr int COLS = 1024 / SL;
    __shared__ double acc[SL][COLS];
    const bool isw = (int)blockIdx.x < wblocks;
    const float *src = isw ? wpart : bpart;
    const int n = isw ? nw : nb, len = isw ? W : N;
    const int col = threadIdx.x % COLS, sl = threadIdx.x / COLS;
    const int c = (isw ? blockIdx.x : blockIdx.x - wblocks) * COLS + col;
    double s = 0.0;
    if (c < len) {
#pragma unroll 4
        for (int k = sl; k < n; k += SL) s += (double)src[(long)k * len + c];
    }
    if (SL > 1) {
        acc[sl][col] = s;
        __syncthreads();
    }
    if (sl == 0 && c < len) {
        for (int k = 1; k < SL; ++k) s += acc[k][col];
        (isw ? gw : gb)[c] = (float)s;
    }
}

// Input fields of the network at every mapped surface point (surrogate.encode's
// 13 channels, in its order of operations): rows are x, y, depth, mxx, myy, mzz,
// mxy, mxz, myz, log10 M0 of a source.  Computed in double and rounded once.
// One lane per point; 48 sources on 80 x 80 points take 10 us, and their
// prediction 2.5 ms where the host's encoding and its upload of 16 MB made it 6.2.
__global__ void __launch_bounds__(256) encode_kernel(const double *__restrict__ src, float *__restrict__ out, int i0,
                                                     int j0, int wi, int wj, double dh, double L)
{
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= wi * wj) return;
    const double *p = src + 10L * blockIdx.y;
    const double X = (double)(i0 + q / wj) * dh, Y = (double)(j0 + q % wj) * dh;
    const double ex = X - p[0], ey = Y - p[1], dx = ex / L, dy = ey / L, dz = p[2] / L;
    const double r = sqrt(dx * dx + dy * dy + dz * dz);
    float *o = out + ((long)blockIdx.y * wi * wj + q) * 13;
    o[0] = (float)(X / L);
    o[1] = (float)(Y / L);
    o[2] = (float)dx;
    o[3] = (float)dy;
    o[4] = (float)exp(-(ex * ex + ey * ey) / (2 * 1000.0 * 1000.0));
    o[5] = (float)dz;
    o[6] = (float)r;
    o[7] = (float)log10(r);
    o[8] = (float)p[3];
    o[9] = (float)p[4];
    o[10] = (float)p[6];
    o[11] = (float)p[7];
    o[12] = (float)p[8];
}

// The last step of a Fourier layer in one launch: for every grid row z = (b,h),
//   forward:  y = act(V W + bias + F T),  pre and the bf16 copy as on request
//   backward: y = V W + F T
// with V [W, C] and T [2m, C] of that row and the constant W [C, C], F [W, 2m]
// (each operand by strides).  Two launches wrote the inverse transform F T in
// fp32 and read it back.  The two products accumulate apart and are added in the
// order of those launches, so the results are theirs bit for bit.  A block of
// 2*WR wavefronts owns 32*WR points of a row by 64 channels, so that 80 or 96
// points are one block (WR = 3) and 128 are one (WR = 4).  Bound by HBM: 2560 rows
// of 80 points, 64 channels and 16 modes with every output take 38 us (183 MB
// moved, 4.8 TB/s) where the two launches took 19 + 39, the backward 28 us for
// 18 + 24.
struct PairArgs {
    const unsigned short *F, *T, *V, *Wt;
    long sFr, sFk, sTz, sTk, sVz, sVr, sWn, sWk;
    int M, N, K1, K2, act;
    const float *bias;
    float *y, *pre;
    unsigned short *yb;
};

template <int WR, int MODE>
__device__ __forceinline__ u16x8 pair_fetch_a(const unsigned short *P, long sR, long sK, int r0, int k0, int R, int K)
{
    const int tid = threadIdx.x;
    u16x8 v = 0;
    const int r = r0 + (MODE == STAGE_MN ? tid % (4 * WR) * 8 : tid >> 2);
    const int k = k0 + (MODE == STAGE_MN ? tid / (4 * WR) : (tid & 3) * 8);
    if (r < R && k < K) v = *reinterpret_cast<const u16x8 *>(P + r * sR + k * sK);
    return v;
}

template <int WR, int MODE>
__device__ __forceinline__ void pair_park_a(unsigned short (*T)[BK + PAD], u16x8 v)
{
    const int tid = threadIdx.x;
    if (MODE == STAGE_MN) {
        const int r = tid % (4 * WR) * 8, k = tid / (4 * WR);
#pragma unroll
        for (int i = 0; i < 8; ++i) T[r + i][k] = v[i];
    } else {
        *reinterpret_cast<u16x8 *>(&T[tid >> 2][(tid & 3) * 8]) = v;
    }
}

template <int WR, int BWD>
__global__ void __launch_bounds__(128 * WR) layer_pair_kernel(PairArgs g)
{
    // staging: F rows by k (forward) or by point (its transpose), T by channel,
    // V by k, W by channel (forward) or by k (its transpose)
    constexpr int FM = BWD ? STAGE_MN : STAGE_K, WM = BWD ? STAGE_K : STAGE_MN;
    __shared__ __attribute__((aligned(16))) unsigned short As[2][32 * WR][BK + PAD];
    __shared__ __attribute__((aligned(16))) unsigned short Bs[2][BN][BK + PAD];
    const int z = blockIdx.z, m0 = blockIdx.y * 32 * WR, n0 = blockIdx.x * BN;
    const unsigned short *T = g.T + z * g.sTz, *V = g.V + z * g.sVz;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    f32x4 accF[2][2], accV[2][2];
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j) accF[i][j] = accV[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int t1 = (g.K1 + BK - 1) / BK, tiles = t1 + (g.K2 + BK - 1) / BK;
    const bool loadb = tid < 256;
    u16x8 na = 0, nb = 0;
    auto get = [&](int t) {
        if (t < t1) {
            na = pair_fetch_a<WR, FM>(g.F, g.sFr, g.sFk, m0, t * BK, g.M, g.K1);
            if (loadb) nb = fetch<STAGE_MN, 1>(T, 1, g.sTk, n0, t * BK, g.N, g.K1, tid);
        } else {
            na = pair_fetch_a<WR, STAGE_K>(V, g.sVr, 1, m0, (t - t1) * BK, g.M, g.K2);
            if (loadb) nb = fetch<WM, 1>(g.Wt, g.sWn, g.sWk, n0, (t - t1) * BK, g.N, g.K2, tid);
        }
    };
    auto put = [&](int t, int buf) {
        if (t < t1) {
            pair_park_a<WR, FM>(As[buf], na);
            if (loadb) park<STAGE_MN>(Bs[buf], nb, tid);
        } else {
            pair_park_a<WR, STAGE_K>(As[buf], na);
            if (loadb) park<WM>(Bs[buf], nb, tid);
        }
    };
    get(0);
    put(0, 0);
    __syncthreads();
    for (int t = 0; t < tiles; ++t) {
        if (t + 1 < tiles) get(t + 1);
        const int cur = t & 1, kq = (lane >> 4) * 8;
#pragma unroll
        for (int bi = 0; bi < 2; ++bi) {
            const bf16x8 a = *reinterpret_cast<const bf16x8 *>(&As[cur][wm + bi * 16 + (lane & 15)][kq]);
#pragma unroll
            for (int bj = 0; bj < 2; ++bj) {
                const bf16x8 b = *reinterpret_cast<const bf16x8 *>(&Bs[cur][wn + bj * 16 + (lane & 15)][kq]);
                if (t < t1) accF[bi][bj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, accF[bi][bj], 0, 0, 0);
                else accV[bi][bj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, accV[bi][bj], 0, 0, 0);
            }
        }
        if (t + 1 < tiles) put(t + 1, cur ^ 1);
        __syncthreads();
    }
    const int mr = m0 + wm + (lane & 15), nc = n0 + wn + (lane >> 4) * 4;
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int bj = 0; bj < 2; ++bj) {
            const int m = mr + bi * 16, n = nc + bj * 16;
            if (m >= g.M || n >= g.N) continue;
            const long o = ((long)z * g.M + m) * g.N + n;
            f32x4 v = accV[bi][bj];
            if (BWD) {
                v = accF[bi][bj] + v;
                *reinterpret_cast<f32x4 *>(g.y + o) = v;
                continue;
            }
            v = v + *reinterpret_cast<const f32x4 *>(g.bias + n);
            v = v + accF[bi][bj];
            if (g.pre) *reinterpret_cast<f32x4 *>(g.pre + o) = v;
            if (g.act == CGFD_FNO_ACT_GELU) {
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = gelu(v[i]);
            }
            if (g.y) *reinterpret_cast<f32x4 *>(g.y + o) = v;
            u16x4 e;
#pragma unroll
            for (int i = 0; i < 4; ++i) e[i] = to_bf16(v[i]);
            *reinterpret_cast<u16x4 *>(g.yb + o) = e;
        }
}

// strips of 32 points per block: the fewest strips in all, then the largest blocks
template <int BWD> void launch_pair(const PairArgs &g, int batch, hipStream_t s)
{
    const int strips = (g.M + 31) / 32;
    int wr = 4;
    for (int c = 3; c >= 2; --c)
        if ((strips + c - 1) / c * c < (strips + wr - 1) / wr * wr) wr = c;
    const dim3 grid((g.N + BN - 1) / BN, (strips + wr - 1) / wr, batch);
    if (wr == 4) hipLaunchKernelGGL((layer_pair_kernel<4, BWD>), grid, dim3(512), 0, s, g);
    else if (wr == 3) hipLaunchKernelGGL((layer_pair_kernel<3, BWD>), grid, dim3(384), 0, s, g);
    else hipLaunchKernelGGL((layer_pair_kernel<2, BWD>), grid, dim3(256), 0, s, g);
}

// Rows of x and gz that one partial weight-gradient product covers: 256, or 512
// for weights of at least 16 tiles where the parts then still are 8 blocks per CU.
// 256 / 512 rows, gw and gb alone: 65536 x 256 x 256 123 / 115 us, 65536 x 2048 x 256
// 655 / 606 (256 rows write twice the partial sums), 32768 x 64 x 64 22.5 / 28.7, 2048
// x 512 x 256 41 / 46 (512 rows leave the chip idle); 300000 x 128 x 128 with its
// forward pass 325 / 332 (the last part runs alone, for longer).
int weight_rows(long R, int K, int N)
{
    const long tiles = (long)((K + BM - 1) / BM) * ((N + BN - 1) / BN);
    return tiles >= 16 && R / 512 * tiles >= 2048 ? 512 : 256;
}

// Gradients of y = x w + b after its epilogue: gzb and (optional) gz from gy
// and pre, gw and gb.  wpart: ceil(R/weight_rows) x K x N, bpart: ceil(R/GROUP) x N.
void linear_grads(const float *gy, const float *pre, const void *xb, float *gz, void *gzb, float *wpart, float *bpart,
                  float *gw, float *gb, long R, int K, int N, hipStream_t s)
{
    const int wrows = weight_rows(R, K, N);
    const int nb = (int)((R + GROUP - 1) / GROUP), nw = (int)((R + wrows - 1) / wrows), full = (int)(R / wrows);
    if (N % 4 == 0 && vec4(gy, 0, 0, 4) && vec4(pre, 0, 0, 4) && vec4(gz, 0, 0, 4) && vec4(gzb, 0, 0, 2) &&
        vec4(bpart, 0, 0, 4))
        hipLaunchKernelGGL(layer_grad_kernel<4>, dim3(nb), dim3(256), 0, s, gy, pre, gz, (unsigned short *)gzb, bpart,
                           R, N);
    else
        hipLaunchKernelGGL(layer_grad_kernel<1>, dim3(nb), dim3(256), 0, s, gy, pre, gz, (unsigned short *)gzb, bpart,
                           R, N);
    auto part = [&](long r0, int rows_, int batch, float *out) {
        GemmArgs g{};
        g.A = (const unsigned short *)xb + r0 * K;
        g.B = (const unsigned short *)gzb + r0 * N;
        g.C = out;
        g.sAz = (long)wrows * K;
        g.sAm = 1;
        g.sAk = K;
        g.sBz = (long)wrows * N;
        g.sBk = N;
        g.sBn = 1;
        g.sCz = (long)K * N;
        g.sCm = N;
        g.M = K;
        g.N = N;
        g.K = rows_;
        g.amode = stage_mode(g.A, g.sAz, g.sAm, g.sAk);
        g.bmode = stage_mode(g.B, g.sBz, g.sBn, g.sBk);
        g.vec = vec4(out, g.sCz, g.sCm, 4);
        for (int z = 0; z < batch; z += 65535) { // grid.z
            GemmArgs h = g;
            h.A += z * g.sAz;
            h.B += z * g.sBz;
            h.C += z * g.sCz;
            launch_gemm(h, batch - z < 65535 ? batch - z : 65535, s);
        }
    };
    if (full) part(0, wrows, full, wpart);
    if (nw > full) part((long)full * wrows, (int)(R - (long)full * wrows), 1, wpart + (long)full * K * N);
    auto reduce = [&](auto kernel, int cols) {
        const int wblocks = (K * N + cols - 1) / cols;
        hipLaunchKernelGGL(kernel, dim3(wblocks + (N + cols - 1) / cols), dim3(1024), 0, s, wpart, nw, K * N, gw, bpart,
                           nb, N, gb, wblocks);
    };
    if (nw >= 64) reduce(layer_reduce_kernel<16>, 64);
    else if (nw > 16) reduce(layer_reduce_kernel<4>, 256);
    else reduce(layer_reduce_kernel<1>, 1024);
}

int check_layer(long B, long H, long W, long C, long m)
{
    if (B <= 0 || H <= 0 || W <= 0 || C <= 0 || m <= 0 || 2 * m > H || m > W / 2) return CGFD_FNO_EINVAL;
    // vector stores need the width in multiples of 8; grid.z and grid.y limits
    if (C % 8 != 0 || C > 256 || B * H > 65535 || 2 * m * m > 65535 || B > 65535 || B * H * W > 0x7fffffffL)
        return CGFD_FNO_EINVAL;
    return 0;
}

// gx may alias gy: each element is read before it is written, by one lane.
// Bound by HBM (14 bytes per element); VEC = 1 moves 4 elements per lane and
// access (all four bases aligned to them), the last n % 4 one by one: 13.1 M
// elements 44.7 -> 38.0 us (4.8 TB/s).
template <int VEC>
__global__ void __launch_bounds__(256) gelu_bwd_kernel(const float *gy, const float *__restrict__ pre, float *gx,
                                                       unsigned short *__restrict__ gxb, long n)
{
    const long stride = (long)gridDim.x * blockDim.x, first = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long n4 = VEC ? n / 4 : 0;
    if (VEC) {
        for (long i = first; i < n4; i += stride) {
            const f32x4 y = reinterpret_cast<const f32x4 *>(gy)[i], x = reinterpret_cast<const f32x4 *>(pre)[i];
            f32x4 v;
            u16x4 e;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v[j] = y[j] * gelu_grad(x[j]);
                e[j] = to_bf16(v[j]);
            }
            reinterpret_cast<f32x4 *>(gx)[i] = v;
            if (gxb) reinterpret_cast<u16x4 *>(gxb)[i] = e;
        }
    }
    for (long i = n4 * 4 + first; i < n; i += stride) {
        const float v = gy[i] * gelu_grad(pre[i]);
        gx[i] = v;
        if (gxb) gxb[i] = to_bf16(v);
    }
}

// One Adam step (no weight decay, no amsgrad), as torch.optim.Adam computes
// it: m += (1-b1) (g - m); v = b2 v + (1-b2) g^2;
// p -= (lr / bc1) m / (sqrt(v) / sqrt(bc2) + eps), with the scalars formed
// in double and rounded once to float; with clear set the gradient is zeroed
// as it is read.  Block b updates chunk b: elements
// [off, off + CGFD_FNO_ADAM_CHUNK) of tensor t, with (t, off) = chunks[2b],
// chunks[2b+1] and the tensor's (p, g, m, v, n) = tensors[5t .. 5t+4].  Bound
// by HBM (32 bytes per element with clear): 16.9 M parameters 96 us in 4-byte
// accesses, 84 us (6.4 TB/s) in 16-byte ones.
__global__ void __launch_bounds__(256) adam_kernel(const long long *__restrict__ tensors,
                                                   const long long *__restrict__ chunks, float w1, float b2,
                                                   float w2, float lr_bc1, float bc2_sqrt, float eps, int clear)
{
    const long long t = chunks[2 * blockIdx.x], off = chunks[2 * blockIdx.x + 1];
    float *p = reinterpret_cast<float *>(tensors[5 * t]);
    float *g = reinterpret_cast<float *>(tensors[5 * t + 1]);
    float *m = reinterpret_cast<float *>(tensors[5 * t + 2]);
    float *v = reinterpret_cast<float *>(tensors[5 * t + 3]);
    const long long n = tensors[5 * t + 4];
    const long long end = off + CGFD_FNO_ADAM_CHUNK < n ? off + CGFD_FNO_ADAM_CHUNK : n;
    auto update = [&](float gi, float &pi, float &mi, float &vi) {
        mi = mi + w1 * (gi - mi);
        vi = vi * b2 + w2 * (gi * gi);
        pi = pi + -lr_bc1 * (mi / (sqrtf(vi) / bc2_sqrt + eps));
    };
    // chunks start at multiples of 8192 elements: 16-byte accesses where the
    // tensor's four arrays are aligned, its last end % 4 elements one by one
    long long head = off;
    if (((tensors[5 * t] | tensors[5 * t + 1] | tensors[5 * t + 2] | tensors[5 * t + 3]) & 15) == 0) {
        head = end / 4 * 4;
        for (long long i = off + 4 * threadIdx.x; i < head; i += 4 * blockDim.x) {
            f32x4 gi = *reinterpret_cast<f32x4 *>(g + i), pi = *reinterpret_cast<f32x4 *>(p + i);
            f32x4 mi = *reinterpret_cast<f32x4 *>(m + i), vi = *reinterpret_cast<f32x4 *>(v + i);
            if (clear) *reinterpret_cast<f32x4 *>(g + i) = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float pj = pi[j], mj = mi[j], vj = vi[j];
                update(gi[j], pj, mj, vj);
                pi[j] = pj;
                mi[j] = mj;
                vi[j] = vj;
            }
            *reinterpret_cast<f32x4 *>(m + i) = mi;
            *reinterpret_cast<f32x4 *>(v + i) = vi;
            *reinterpret_cast<f32x4 *>(p + i) = pi;
        }
    }
    for (long long i = head + threadIdx.x; i < end; i += blockDim.x) {
        const float gi = g[i];
        if (clear) g[i] = 0.0f; // the gradient is read once: the next backward accumulates into zeros
        float pi = p[i], mi = m[i], vi = v[i];
        update(gi, pi, mi, vi);
        m[i] = mi;
        v[i] = vi;
        p[i] = pi;
    }
}

} // namespace

extern "C" int cgfd_fno_gemm_bf16_ex(const void *A, long sAz, long sAm, long sAk, const void *B, long sBz, long sBk,
                                     long sBn, float *C, long sCz, long sCm, int M, int N, int K, int batch,
                                     int accumulate, const float *bias, const float *D, long sDz, long sDm,
                                     float *pre, int act, void *C_bf16, long sEz, long sEm, void *stream)
{
    if (!A || !B || !C || M <= 0 || N <= 0 || K <= 0 || batch <= 0) return CGFD_FNO_EINVAL;
    if (act != CGFD_FNO_ACT_NONE && act != CGFD_FNO_ACT_GELU) return CGFD_FNO_EINVAL;
    const long tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
    if (tm > 65535 || batch > 65535 || tn > 0x7fffffffL) return CGFD_FNO_EINVAL;
    GemmArgs g{(const unsigned short *)A, (const unsigned short *)B, C, sAz, sAm, sAk, sBz, sBk, sBn, sCz, sCm,
               M, N, K, accumulate ? 1 : 0, stage_mode(A, sAz, sAm, sAk), stage_mode(B, sBz, sBn, sBk),
               N % 4 == 0 && vec4(C, sCz, sCm, 4) && vec4(pre, sCz, sCm, 4) && vec4(D, sDz, sDm, 4) &&
                   vec4(bias, 0, 0, 4) && vec4(C_bf16, sEz, sEm, 2),
               bias, D, sDz, sDm, pre, act, (unsigned short *)C_bf16, sEz, sEm, 1, 1, 1, 0, 0, 0};
    launch_gemm(g, batch, (hipStream_t)stream);
    return hipGetLastError() == hipSuccess ? 0 : CGFD_FNO_EHIP;
}


extern "C" int cgfd_fno_gemm_bf16(const void *A, long sAz, long sAm, long sAk, const void *B, long sBz, long sBk,
                                  long sBn, float *C, long sCz, long sCm, int M, int N, int K, int batch,
                                  int accumulate, void *stream)
{
    return cgfd_fno_gemm_bf16_ex(A, sAz, sAm, sAk, B, sBz, sBk, sBn, C, sCz, sCm, M, N, K, batch, accumulate,
                                 nullptr, nullptr, 0, 0, nullptr, CGFD_FNO_ACT_NONE, nullptr, 0, 0, stream);
}

extern "C" int cgfd_fno_gelu_bwd(const float *gy, const float *pre, float *gx, void *gx_bf16, long n, void *stream)
{
    if (!gy || !pre || !gx || n < 0) return CGFD_FNO_EINVAL;
    if (n == 0) return 0;
    const bool vec = vec4(gy, 0, 0, 4) && vec4(pre, 0, 0, 4) && vec4(gx, 0, 0, 4) && vec4(gx_bf16, 0, 0, 2);
    const long work = vec ? n / 4 + 3 : n, blocks = (work + 255) / 256 < 8192 ? (work + 255) / 256 : 8192;
    if (vec)
        hipLaunchKernelGGL(gelu_bwd_kernel<1>, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, gy, pre, gx,
                           (unsigned short *)gx_bf16, n);
    else
        hipLaunchKernelGGL(gelu_bwd_kernel<0>, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, gy, pre, gx,
                           (unsigned short *)gx_bf16, n);
    return hipGetLastError() == hipSuccess ? 0 : CGFD_FNO_EHIP;
}

extern "C" int cgfd_fno_adam(const long long *tensors, const long long *chunks, int nchunks, double lr,
                             double beta1, double beta2, double eps, long long step, int clear_grad, void *stream)
{
    if (!tensors || !chunks || nchunks < 0 || step < 1 || !(lr >= 0.0) || !(eps > 0.0) || !(beta1 >= 0.0) ||
        !(beta1 < 1.0) || !(beta2 >= 0.0) || !(beta2 < 1.0))
        return CGFD_FNO_EINVAL;
    if (nchunks == 0) return 0;
    const double bc1 = 1.0 - __builtin_pow(beta1, (double)step);
    const double bc2 = 1.0 - __builtin_pow(beta2, (double)step);
    hipLaunchKernelGGL(adam_kernel, dim3((unsigned)nchunks), dim3(256), 0, (hipStream_t)stream, tensors, chunks,
                       (float)(1.0 - beta1), (float)beta2, (float)(1.0 - beta2), (float)(lr / bc1),
                       (float)__builtin_sqrt(bc2), (float)eps, clear_grad ? 1 : 0);
    return hipGetLastError() == hipSuccess ? 0 : CGFD_FNO_EHIP;
}

// One Fourier layer, y = act(v w + b + K v).  The spectral branch K v is six
// launches with bf16 operands throughout: the weights, the DFT along w, that
// along h (stored mode by mode), the mode mixing (stored back to rows), and
// the two inverse DFTs.  Every intermediate is a product summed in fp32 and
// rounded to bf16 once, as the operand of the next product.
extern "C" int cgfd_fno_fourier_fwd(const cgfd_fno_fourier *L, void *stream)
{
    if (!L) return CGFD_FNO_EINVAL;
    const int B = L->B, H = L->H, W = L->W, C = L->C, m = L->modes, P = 2 * m * m;
    int rc = check_layer(B, H, W, C, m);
    if (rc) return rc;
    if (!L->vb || !L->fw || !L->gh || !L->gi || !L->fi || !L->wre || !L->wim || !L->w || !L->bias || !L->wr || !L->wb ||
        !L->t1 || !L->x || !L->t2 || !L->t3 || !L->yb)
        return CGFD_FNO_EINVAL;
    if (!aligned16(L->vb, L->fw, L->gh, L->gi, L->fi, L->wre, L->wim, L->wr, L->wb, L->x, L->t1, L->t2, L->t3, L->y, L->pre,
                   L->yb))
        return CGFD_FNO_EINVAL;
    // the last two products in one launch where whole groups of eight can be staged
    const bool pair = m % 4 == 0 && vec4(L->bias, 0, 0, 4);
    if (!pair && (!L->sp || !L->y)) return CGFD_FNO_EINVAL;
    const hipStream_t s = (hipStream_t)stream;
    const long mC = (long)m * C, C2 = 2L * C;
    const long n4 = (long)P * C * C / 4;
    const int nspec = (int)((n4 + 255) / 256);
    hipLaunchKernelGGL(layer_weights_kernel, dim3(nspec + (C * C + 255) / 256), dim3(256), 0, s, L->wre, L->wim,
                       (unsigned short *)L->wr, n4, C, L->w, (unsigned short *)L->wb, C * C, nspec);
    // t1 [(b,h)][(ri,kw)][c]
    product_bf16({L->fw, 0, W, 1}, {L->vb, (long)W * C, 1, C}, rows(L->t1, 2 * mC, C), 2 * m, C, W, B * H, s);
    // x [(kh,kw)][b][(ri,c)] from rows (ri,kh), columns (kw,c)
    product_bf16({L->gh, 0, 2L * H, 1}, {L->t1, 2 * H * mC, 1, mC},
                 {L->x, 1 << 30, 2 * m, C, 0, C2, C, m * B * C2, B * C2}, 4 * m, m * C, 2 * H, B, s);
    // t2 [b][(kh,ri)][(kw,c)] from batch (kh,kw), rows b, columns (ri,c)
    product_bf16({L->x, B * C2, C2, 1}, {L->wr, C2 * C2, 1, C2},
                 {L->t2, m, 1 << 30, C, 2 * mC, C, 0, 4 * m * mC, mC}, B, 2 * C, 2 * C, P, s);
    // t3 [b][(h,ri)][(kw,c)]
    product_bf16({L->gi, 0, 4L * m, 1}, {L->t2, 4 * m * mC, 1, mC}, rows(L->t3, 2 * H * mC, mC), 2 * H, m * C, 4 * m, B,
                 s);
    if (pair) {
        PairArgs g{(const unsigned short *)L->fi, (const unsigned short *)L->t3, (const unsigned short *)L->vb,
                   (const unsigned short *)L->wb, 2 * m, 1, 2 * mC, C, (long)W * C, C, 1, C, W, C, 2 * m, C,
                   L->gelu ? CGFD_FNO_ACT_GELU : CGFD_FNO_ACT_NONE, L->bias, L->y, L->pre, (unsigned short *)L->yb};
        launch_pair<0>(g, B * H, s);
        return hipGetLastError() == hipSuccess ? 0 : CGFD_FNO_EHIP;
    }
    rc = cgfd_fno_gemm_bf16(L->fi, 0, 2 * m, 1, L->t3, 2 * mC, C, 1, L->sp, (long)W * C, C, W, C, 2 * m, B * H, 0,
                            stream);
    if (rc) return rc;
    return cgfd_fno_gemm_bf16_ex(L->vb, 0, C, 1, L->wb, 0, C, 1, L->y, 0, C, B * H * W, C, C, 1, 0, L->bias, L->sp, 0, C,
                                 L->pre, L->gelu ? CGFD_FNO_ACT_GELU : CGFD_FNO_ACT_NONE, L->yb, 0, C, stream);
}

extern "C" int cgfd_fno_fourier_bwd(const cgfd_fno_fourier_grad *L, void *stream)
{
    if (!L) return CGFD_FNO_EINVAL;
    const int B = L->B, H = L->H, W = L->W, C = L->C, m = L->modes, P = 2 * m * m;
    int rc = check_layer(B, H, W, C, m);
    if (rc) return rc;
    if (!L->gy || !L->vb || !L->fw || !L->gh || !L->gi || !L->fi || !L->wr || !L->wb || !L->x || !L->gzb || !L->t1 ||
        !L->g || !L->t2 || !L->t3 || !L->gwr || !L->wpart || !L->bpart || !L->gv || !L->gwre || !L->gwim || !L->gw ||
        !L->gb)
        return CGFD_FNO_EINVAL;
    if (!aligned16(L->vb, L->fw, L->gh, L->gi, L->fi, L->wr, L->wb, L->x, L->gzb, L->g, L->t1, L->t2, L->t3, L->gwr, L->gv,
                   L->gwre, L->gwim))
        return CGFD_FNO_EINVAL;
    const hipStream_t s = (hipStream_t)stream;
    const long mC = (long)m * C, C2 = 2L * C, R = (long)B * H * W;
    linear_grads(L->gy, L->pre, L->vb, nullptr, L->gzb, L->wpart, L->bpart, L->gw, L->gb, R, C, C, s);
    // transposes of the forward products, from the last to the first
    product_bf16({L->fi, 0, 1, 2L * m}, {L->gzb, (long)W * C, 1, C}, rows(L->t1, 2 * mC, C), 2 * m, C, W, B * H, s);
    // g [(kh,kw)][b][(ri,c)] from rows (kh,ri), columns (kw,c)
    product_bf16({L->gi, 0, 1, 4L * m}, {L->t1, 2 * H * mC, 1, mC},
                 {L->g, 1 << 30, 2, C, 0, C2, m * B * C2, C, B * C2}, 4 * m, m * C, 2 * H, B, s);
    // t2 [b][(ri,kh)][(kw,c)] from batch (kh,kw), rows b, columns (ri,c)
    product_bf16({L->g, B * C2, C2, 1}, {L->wr, C2 * C2, C2, 1},
                 {L->t2, m, 1 << 30, C, mC, C, 0, 4 * m * mC, 2 * m * mC}, B, 2 * C, 2 * C, P, s);
    rc = cgfd_fno_gemm_bf16(L->x, B * C2, 1, C2, L->g, B * C2, C2, 1, L->gwr, C2 * C2, C2, 2 * C, 2 * C, B, P, 0, stream);
    if (rc) return rc;
    const long n4 = (long)P * C * C / 4;
    hipLaunchKernelGGL(layer_weight_grads_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, s, L->gwr, L->gwre,
                       L->gwim, n4, C);
    product_bf16({L->gh, 0, 1, 2L * H}, {L->t2, 4 * m * mC, 1, mC}, rows(L->t3, 2 * H * mC, mC), 2 * H, m * C, 4 * m, B,
                 s);
    if (W % 8 == 0) {
        PairArgs g{(const unsigned short *)L->fw, (const unsigned short *)L->t3, (const unsigned short *)L->gzb,
                   (const unsigned short *)L->wb, 1, W, 2 * mC, C, (long)W * C, C, C, 1, W, C, 2 * m, C,
                   CGFD_FNO_ACT_NONE, nullptr, L->gv, nullptr, nullptr};
        launch_pair<1>(g, B * H, s);
        return hipGetLastError() == hipSuccess ? 0 : CGFD_FNO_EHIP;
    }
    rc = cgfd_fno_gemm_bf16(L->fw, 0, 1, W, L->t3, 2 * mC, C, 1, L->gv, (long)W * C, C, W, C, 2 * m, B * H, 0, stream);
    if (rc) return rc;
    return cgfd_fno_gemm_bf16(L->gzb, 0, C, 1, L->wb, 0, 1, C, L->gv, 0, C, (int)R, C, C, 1, 1, stream);
}

extern "C" int cgfd_fno_weight_rows(long R, int K, int N)
{
    return R <= 0 || K <= 0 || N <= 0 ? CGFD_FNO_EINVAL : weight_rows(R, K, N);
}

extern "C" int cgfd_fno_linear_bwd(const float *gy, const float *pre, const void *xb, const void *wb, float *gz,
                                   void *gzb, float *wpart, float *bpart, float *gx, float *gw, float *gb, long R,
                                   int K, int N, void *stream)
{
    if (!gy || !xb || !wb || !gzb || !wpart || !bpart || !gw || !gb || R <= 0 || K <= 0 || N <= 0 || N > 256 ||
        R > 0x7fffffffL || (R + BM - 1) / BM > 65535 || (K + BM - 1) / BM > 65535)
        return CGFD_FNO_EINVAL;
    const hipStream_t s = (hipStream_t)stream;
    linear_grads(gy, pre, xb, gz, gzb, wpart, bpart, gw, gb, R, K, N, s);
    if (gx) return cgfd_fno_gemm_bf16(gzb, 0, N, 1, wb, 0, 1, N, gx, 0, K, (int)R, K, N, 1, 0, stream);
    return hipGetLastError() == hipSuccess ? 0 : CGFD_FNO_EHIP;
}

extern "C" int cgfd_fno_encode(const double *src, float *out, int n, int i0, int j0, int wi, int wj, double dh, double L,
                               void *stream)
{
    if (!src || !out || n < 0 || n > 65535 || wi <= 0 || wj <= 0 || (long)wi * wj > 0x7fffff00L || !(L > 0.0))
        return CGFD_FNO_EINVAL;
    if (n == 0) return 0;
    hipLaunchKernelGGL(encode_kernel, dim3((wi * wj + 255) / 256, n), dim3(256), 0, (hipStream_t)stream, src, out, i0, j0,
                       wi, wj, dh, L);
    return hipGetLastError() == hipSuccess ? 0 : CGFD_FNO_EHIP;
}

// y = act(x w + b) for the layers whose fp32 result nobody reads
extern "C" int cgfd_fno_linear_fwd(const void *xb, const void *wb, const float *bias, float *pre, int act, void *yb,
                                   long R, int K, int N, void *stream)
{
    if (!xb || !wb || !bias || !yb || R <= 0 || R > 0x7fffffffL || (R + BM - 1) / BM > 65535 || K <= 0 || N <= 0 ||
        (act != CGFD_FNO_ACT_NONE && act != CGFD_FNO_ACT_GELU))
        return CGFD_FNO_EINVAL;
    GemmArgs g{};
    g.A = (const unsigned short *)xb;
    g.B = (const unsigned short *)wb;
    g.sAm = K;
    g.sAk = 1;
    g.sBk = N;
    g.sBn = 1;
    g.sCm = N;
    g.M = (int)R;
    g.N = N;
    g.K = K;
    g.amode = stage_mode(xb, 0, K, 1);
    g.bmode = stage_mode(wb, 0, 1, N);
    g.bias = bias;
    g.pre = pre;
    g.act = act;
    g.Cb = (unsigned short *)yb;
    g.sEm = N;
    g.vec = 1;
    if (N % 4 != 0 || !vec4(bias, 0, 0, 4) || !vec4(pre, 0, N, 4) || !vec4(yb, 0, N, 2)) return CGFD_FNO_EINVAL;
    launch_gemm(g, 1, (hipStream_t)stream);
    return hipGetLastError() == hipSuccess ? 0 : CGFD_FNO_EHIP;
}
