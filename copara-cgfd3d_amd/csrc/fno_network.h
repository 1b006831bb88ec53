/*
 * fno_network.h -- the calls between surrogate.py and libcgfd_fno.so that run
 * the network's own layers as one chain of launches.  Pointers are on the
 * device; 0 or a negative code of cgfd_fno.h is returned.
 */
#ifndef FNO_NETWORK_H
#define FNO_NETWORK_H

#include "cgfd_fno.h"

#ifdef __cplusplus
extern "C" {
#endif

/* One Fourier layer on channels-last activations, y = act(v w + bias + K v),
 * K the mixing of the lowest modes x modes frequencies: the launches of
 * surrogate.py's spectral and pointwise products, with every intermediate kept
 * in bf16 only (the operand of the next product) and stored in the order that
 * the next product reads.  C is a multiple of 8 and at most 256, B*H at most
 * 65535.  fw, gh, gi, fi: the bf16 DFT matrices [2m, W], [4m, 2H], [2H, 4m],
 * [W, 2m].  Sizes in elements, R = B*H*W, P = 2*modes*modes.  Every pointer but w,
 * bias and sp is aligned to 16 bytes. */
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
 * forward call had or wrote them (pre null without GELU).  Every pointer but gy,
 * pre, wpart, bpart, gw and gb is aligned to 16 bytes. */
typedef struct cgfd_fno_fourier_grad {
    int B, H, W, C, modes, unused;
    const float *gy, *pre;
    const void *vb, *fw, *gh, *gi, *fi, *wr, *wb, *x;
    void *gzb;                       /* scratch, bf16 [R, C] */
    void *g;                         /* scratch, bf16 [P, B, 2C] */
    void *t1, *t2, *t3;              /* scratch as in the forward call */
    float *gwr;                      /* scratch [P, 2C, 2C] */
    float *wpart, *bpart;            /* scratch as of cgfd_fno_linear_bwd with K = N = C */
    float *gv, *gwre, *gwim, *gw, *gb;
} cgfd_fno_fourier_grad;
int cgfd_fno_fourier_bwd(const cgfd_fno_fourier_grad *layer, void *stream);

/* yb = act(x w + bias) in bf16 only, x [R, K] and w [K, N] in bf16, N a multiple
 * of 4; the value before the activation into pre unless null.  bias and pre are
 * aligned to 16 bytes, yb to 8. */
int cgfd_fno_linear_fwd(const void *xb, const void *wb, const float *bias, float *pre, int act, void *yb, long R,
                        int K, int N, void *stream);

/* Gradients of y = act(x w + b (+ d)) from gy [R, N], x [R, K] and w [K, N] in
 * bf16: gz = gy * GELU'(pre) (pre null: gy), in bf16 into gzb and on request
 * (the gradient of d) into gz; gx = gz w^T unless null, gw = x^T gz, gb = the
 * column sums of gz in fp32.  N is at most 256.  Scratch:
 * wpart ceil(R/rows)*K*N, rows = cgfd_fno_weight_rows(R, K, N), and bpart
 * ceil(R/128)*N fp32 elements. */
int cgfd_fno_linear_bwd(const float *gy, const float *pre, const void *xb, const void *wb, float *gz, void *gzb,
                        float *wpart, float *bpart, float *gx, float *gw, float *gb, long R, int K, int N,
                        void *stream);

/* Rows that one partial sum of the weight gradient covers (256 or 512). */
int cgfd_fno_weight_rows(long R, int K, int N);

/* The network's 13 input fields [n, wi, wj, 13] of n sources at the surface
 * points (i0 + i, j0 + j)*dh: src is n rows of 10 doubles on the device (x, y,
 * depth, mxx, myy, mzz, mxy, mxz, myz, log10 M0), L the length the coordinates
 * are scaled by.  n is at most 65535. */
int cgfd_fno_encode(const double *src, float *out, int n, int i0, int j0, int wi, int wj, double dh, double L,
                    void *stream);

#ifdef __cplusplus
}
#endif

#endif
