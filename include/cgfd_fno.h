/*
 * cgfd_fno.h -- C-ABI of the kernels of the Fourier-neural-operator
 * surrogate: BF16 MFMA products with fused epilogues, the GELU backward and
 * the Adam update (no reference counterpart: the reference has no learned
 * model; the surrogate maps source location, mechanism and moment to surface
 * peak-ground-velocity maps and station seismograms for a fixed medium,
 * trained on runs of this engine).
 */
#ifndef CGFD_FNO_H
#define CGFD_FNO_H

#ifdef __cplusplus
extern "C" {
#endif

#define CGFD_FNO_EINVAL (-1)
#define CGFD_FNO_EHIP (-3)

/* epilogue activations of cgfd_fno_gemm_bf16_ex */
#define CGFD_FNO_ACT_NONE 0
#define CGFD_FNO_ACT_GELU 1 /* x/2 (1 + erf(x / sqrt 2)) */

/* elements of one tensor that one block of cgfd_fno_adam updates */
#define CGFD_FNO_ADAM_CHUNK 8192

/* Batched GEMM on the matrix cores, bf16 inputs, fp32 accumulation:
 *   C[z] = A[z] * B[z]   (accumulate = 0)   or   C[z] += A[z] * B[z]
 * for z < batch.  A is M x K with element (m, k) at A + z*sAz + m*sAm + k*sAk,
 * B is K x N with (k, n) at B + z*sBz + k*sBk + n*sBn (bf16 elements, strides
 * in elements), C is M x N fp32 with (m, n) at C + z*sCz + m*sCm + n.  The
 * caller guarantees that every addressed element lies in its buffer.
 * Asynchronous on `stream` (a hipStream_t; null = the default stream).
 * M/64 and batch must not exceed 65535. */
int cgfd_fno_gemm_bf16(const void *A, long sAz, long sAm, long sAk, const void *B, long sBz, long sBk, long sBn,
                       float *C, long sCz, long sCm, int M, int N, int K, int batch, int accumulate, void *stream);

/* The same product with a layer's epilogue fused into it:
 *   pre[z] = (C[z] +) A[z] * B[z] + bias + D[z],   C[z] = act(pre[z])
 * bias: N fp32 values added to every row, or null.  D: an M x N fp32 addend
 * with (m, n) at D + z*sDz + m*sDm + n, or null.  pre: where the value before
 * the activation is stored (same layout as C; what the activation's backward
 * needs), or null.  act: CGFD_FNO_ACT_NONE or CGFD_FNO_ACT_GELU.  C_bf16:
 * where C is stored again rounded to bf16 (nearest even), (m, n) at C_bf16 +
 * z*sEz + m*sEm + n (the next product's operand), or null. */
int cgfd_fno_gemm_bf16_ex(const void *A, long sAz, long sAm, long sAk, const void *B, long sBz, long sBk, long sBn,
                          float *C, long sCz, long sCm, int M, int N, int K, int batch, int accumulate,
                          const float *bias, const float *D, long sDz, long sDm, float *pre, int act, void *C_bf16,
                          long sEz, long sEm, void *stream);

/* One Fourier layer on channels-last activations, y = act(v w + bias + K v),
 * K the mixing of the lowest modes x modes frequencies: the launches of
 * surrogate.py's spectral and pointwise products, with every intermediate kept
 * in bf16 only (the operand of the next product) and stored in the order that
 * the next product reads.  C is a multiple of 8 and at most 256, B*H at most
 * 65535.  fw, gh, gi, fi: the bf16 DFT matrices [2m, W], [4m, 2H], [2H, 4m],
 * [W, 2m].  Sizes in elements, R = B*H*W, P = 2*modes*modes. */
typedef struct cgfd_fno_fourier {
    int B, H, W, C, modes, gelu;
    const void *vb;                  /* v in bf16 [R, C] */
    const void *fw, *gh, *gi, *fi;
    const float *wre, *wim;          /* mode weights [P, C, C] */
    const float *w, *bias;           /* pointwise weights [C, C], bias [C] */
    void *wr, *wb;                   /* written: the weights in bf16 [P, 2C, 2C], [C, C] */
    void *x;                         /* written: the kept modes in bf16 [P, B, 2C] */
    void *t1, *t2, *t3;              /* scratch, bf16: 2*B*H*m*C, 4*B*m*m*C, 2*B*H*m*C */
    float *sp;                       /* scratch [R, C]; may be null if modes % 4 == 0 */
    float *y, *pre;                  /* the result (or null if modes % 4 == 0) and the value before the GELU (or null) */
    void *yb;                        /* the result in bf16 */
} cgfd_fno_fourier;
int cgfd_fno_fourier_fwd(const cgfd_fno_fourier *layer, void *stream);

/* Its backward: gv, gwre, gwim, gw, gb from gy.  vb, wr, wb, x and pre as the
 * forward call had or wrote them (pre null without GELU). */
typedef struct cgfd_fno_fourier_grad {
    int B, H, W, C, modes, unused;
    const float *gy, *pre;
    const void *vb, *fw, *gh, *gi, *fi, *wr, *wb, *x;
    void *gzb;                       /* scratch, bf16 [R, C] */
    void *g;                         /* scratch, bf16 [P, B, 2C] */
    void *t1, *t2, *t3;              /* scratch as in the forward call */
    float *gwr;                      /* scratch [P, 2C, 2C] */
    float *wpart, *bpart;            /* scratch ceil(R/256)*C*C, ceil(R/128)*C */
    float *gv, *gwre, *gwim, *gw, *gb;
} cgfd_fno_fourier_grad;
int cgfd_fno_fourier_bwd(const cgfd_fno_fourier_grad *layer, void *stream);

/* yb = act(x w + bias) in bf16 only, x [R, K] and w [K, N] in bf16, N a multiple
 * of 4; the value before the activation into pre unless null. */
int cgfd_fno_linear_fwd(const void *xb, const void *wb, const float *bias, float *pre, int act, void *yb, long R,
                        int K, int N, void *stream);

/* Gradients of y = act(x w + b (+ d)) from gy [R, N], x [R, K] and w [K, N] in
 * bf16: gz = gy * GELU'(pre) (pre null: gy), in bf16 into gzb and on request
 * (the gradient of d) into gz; gx = gz w^T unless null, gw = x^T gz, gb = the
 * column sums of gz in fp32.  N is at most 256.  Scratch:
 * wpart ceil(R/256)*K*N, bpart ceil(R/128)*N fp32 elements. */
int cgfd_fno_linear_bwd(const float *gy, const float *pre, const void *xb, const void *wb, float *gz, void *gzb,
                        float *wpart, float *bpart, float *gx, float *gw, float *gb, long R, int K, int N,
                        void *stream);

/* Backward of GELU over n fp32 elements: gx = gy * GELU'(pre), and, when
 * gx_bf16 is not null, the same values rounded to bf16 (nearest even) there
 * (the operand of the next backward products).  gx may alias gy. */
int cgfd_fno_gelu_bwd(const float *gy, const float *pre, float *gx, void *gx_bf16, long n, void *stream);

/* The network's 13 input fields [n, wi, wj, 13] of n sources at the surface
 * points (i0 + i, j0 + j)*dh: src is n rows of 10 doubles on the device (x, y,
 * depth, mxx, myy, mzz, mxy, mxz, myz, log10 M0), L the length the coordinates
 * are scaled by.  n is at most 65535. */
int cgfd_fno_encode(const double *src, float *out, int n, int i0, int j0, int wi, int wj, double dh, double L,
                    void *stream);

/* One Adam step (torch.optim.Adam without weight decay or amsgrad) over many
 * fp32 tensors in one launch.  tensors: device array of 5 int64 per tensor
 * (parameter, gradient, first moment, second moment addresses, element
 * count).  chunks: device array of 2 int64 per block (tensor index, first
 * element, a multiple of CGFD_FNO_ADAM_CHUNK below the count), nchunks
 * blocks.  step counts from 1; the bias corrections 1 - beta^step, lr /
 * (1 - beta1^step) and sqrt(1 - beta2^step) are formed in double.  With
 * clear_grad, each gradient element is set to zero once read (the next
 * backward pass then accumulates into zeros, with no separate clearing). */
int cgfd_fno_adam(const long long *tensors, const long long *chunks, int nchunks, double lr, double beta1,
                  double beta2, double eps, long long step, int clear_grad, void *stream);

#ifdef __cplusplus
}
#endif

#endif
