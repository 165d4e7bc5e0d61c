/*
 * fame_kernels.h -- launch interface between the host solver and the gfx950
 * kernels (not part of the public C-ABI; see include/fame_hip.h for that).
 */
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include "fame_device.hpp"

enum { OUTER_EPS = 0, OUTER_QR = 1, OUTER_QRS = 2 };

#define MAX_LINES_INNER 32   /* lines (b, c) per block of the inner-axis kernels */

/* stage lists an axis plan provides (per precision):
 * FWD  forward transform, INV inverse transform (both unnormalised),
 * EPS  INV, kernel elementwise step, FWD (outer pass of QBQ),
 * FI   FWD, kernel elementwise step, INV (curl-curl inner pass).             */
enum { LIST_FWD = 0, LIST_INV = 1, LIST_EPS = 2, LIST_FI = 3, NLIST = 4 };

/* per-problem CG scalars, device resident */
struct CgScal {
    double rr;        /* current <r,r>                                         */
    double rr0;       /* <b,b> of the solve                                    */
    double pap_re, pap_im;
    double alpha_re, alpha_im;
    double beta;
    double tol2;      /* absolute tolerance squared                           */
    int iters;        /* reference-style counter k (starts at 1)              */
    int maxit;
    int active;       /* 1 while iterating                                      */
    int pend;         /* 1 when x still lacks alpha p of the last iteration    */
    int upd;          /* 1 when rr, beta, iters and active still lack the last iteration's <r,r> */
};

/* what a solve tells the host, in pinned memory that the host polls: the scalar
 * state or a sum, then the sequence number that the host waits for            */
struct CgNote {
    CgScal sc;
    double sum;
    unsigned seq;
};

#ifdef __HIPCC__
/* b = r1 / r0 and the stopping rule (CG.cu:66-78) from the new <r, r> */
__device__ __forceinline__ void cg_rule(double s, double tol2, int maxit, double& rr, double& beta, int& iters, int& active) {
    beta = s / rr;
    rr = s;
    iters += 1;
    active = (s > tol2) && (iters <= maxit);
}
#endif

struct KInner {
    fame::GridDev g;
    const fame::ProbDev* prob;   /* device, one per problem                    */
    fame::LinePlanDev plan;      /* stage list along the inner axis            */
    const int* active;           /* device flags or nullptr                    */
    const void* x;               /* EXPAND: reduced input (padded, 2N/problem) */
    void* y;                     /* !EXPAND: reduced output                    */
    void* f;                     /* field, 3N per problem                      */
    const void* dotvec;          /* !EXPAND: optional d for partial conj(d).y  */
    double* partials;            /* [problem][block][2]                        */
    size_t xstride, fstride;
    int L, P;                    /* lines per block, LDS line pitch            */
    int pikind;                  /* 0 Pi_Qr, 1 Pi_Pr                           */
    /* EXPAND inside CG (cg_r != nullptr): x is the search direction p, and
     * before it is expanded each element is updated in place,
     *   x_sol += alpha p  (when pend),   p = r + beta p,
     * with alpha, beta, pend of the problem's CgScal: the previous iteration's
     * solution and direction updates ride on this pass's reads.             */
    void* cg_r;
    void* cg_x;
    const CgScal* cgsc;
    /* CG residual update on the same pass: with cg_ap set, r -= alpha Ap of
     * the previous iteration (when pend) is applied before p = r + beta p,
     * and <r,r> goes to slot 5 of the partials.
     * !EXPAND with cg_r set: the pass updates r -= alpha y in place instead of
     * storing y (alpha of this iteration, already in cgsc), and puts <r,r> of
     * the updated residual in slot 3 of 6 doubles per block                 */
    const void* cg_ap;
    /* EXPAND, refinement (fx32 set): before it is expanded, x += fx32 + alpha
     * fp32 (the FP32 solve's solution and its pending update, alpha and pend
     * of cgsc, FP32 complex vectors with problem stride xstride) is formed in
     * FP32, added in FP64 and stored back to x                               */
    const void* fx32;
    const void* fp32;
    /* !EXPAND, refinement residual (rb set, complex double like y): instead
     * of y the pass stores the next FP32 solve's start, r32 = p32 = rb - y
     * rounded to FP32 and x32 = 0 (FP32 complex vectors, problem stride
     * xstride), and the block sums of |r32|^2 into rpart[problem][block]   */
    const void* rb;
    void* r32;
    void* p32;
    void* x32;
    double* rpart;
    /* !EXPAND inside CG: <y, y> into slot 2 of 6 doubles per block (the
     * expanding pass puts <r, r> in slot 5; with dotvec, conj(dotvec).y goes
     * to slots 0 and 1), from which the CG takes <r, r> of the next residual
     * without a pass over r                                                  */
    int cgdots;
};

/* one axis of the plane kernels (fame_plane.hpp): Stockham passes, or a direct
 * DFT on the matrix cores */
struct PlaneStage {
    int R, Ns, nb, tstep;        /* radix, radices before it, butterflies per line, twiddle step */
    unsigned mNs;
};
struct PlaneAxis {
    int n, eng, nst;
    unsigned mnl, mn;            /* udiv magics for / lines and / n             */
    int ntab;                    /* entries of W, kept in LDS                   */
    const void* W;               /* Stockham: exp(-2 pi i m / n), n entries; direct DFT: its
                                    (cos, -sin) fragments [tile][K step][64]    */
    /* device arrays: the passes of the inverse transform, and of the forward one
     * (the radices in reverse order)                                          */
    const PlaneStage* st;
    const PlaneStage* sf;
};

/* constants of one line (b, c) of a wave vector: the symbols of the two outer
 * axes, exp(i pi phi / na) of the inner phase, the symbols' sum, squared norm and
 * squared distance                                                            */
struct LineTab { double2 b, c, e, s; double q, d; };

/* the inner-axis kernels of the plane path */
struct KLine {
    fame::GridDev g;
    const fame::ProbDev* prob;
    const int* active;
    PlaneAxis a;
    const LineTab* lt;           /* nb nc per problem                           */
    const void* tw;              /* inner twiddle factors, inner_tw_per_line(na) per line */
    const void* ea;              /* exp(i pi a / na), na complex doubles        */
    void* f;                     /* field, plane layout [component][a][PP]      */
    size_t fstride, xstride;
    int PP, cs;                  /* plane pitch and component stride (na PP)    */
    int L, P;                    /* lines per block, LDS line pitch             */
    unsigned mLs;                /* udiv magic of the field accesses: / (L / 2) in FP32, / L in FP64 */
    const void* x;
    int ref;                     /* reduced vectors in the reference's layout (2 Nd), not padded */
    const double* sig;           /* expand, plain: x scaled by sig[f] (optional) */
    void* r;                     /* CG residual; contract CO_RES: r32           */
    void* xs;                    /* CG solution; contract: y, or x32 of CO_RES  */
    const CgScal* cgsc;
    const void* fx32;
    const void* fp32;
    const void* rb;
    void* p32;
    double* rpart;               /* contract: block sums of <r, r>, every rstep doubles */
    int rstep;
    /* scalars of the iteration formed by the inner kernels themselves (null: cgsc
     * holds them): the expansion reads cgsc and the nrp sums of <r, r> per problem at
     * rpart and writes sc2 and act_out, the contraction reads sc2 and the npap sums
     * of <p, QBQ p> per problem at pap and writes cgsc                          */
    CgScal* sc2;
    CgScal* sc1;                 /* cgsc, for the contraction's write           */
    int* act_out;
    const double* pap;
    int nrp, npap;
};
struct KPlane {
    fame::GridDev g;
    const int* active;
    void* f;
    size_t fstride;
    int PP;
    const void* invB;            /* 1 / (N eps), plane layout                   */
    const void* tw;              /* middle twiddles, nb nc per problem          */
    double* pap;                 /* optional <v, eps^-1 v / N> per block, [problem][component][a] */
    PlaneAxis b, c;
    unsigned mnb;
    int nt;
    int wide;                    /* FP64: the variant of at most 512 threads with 16 elements each */
};

/* what a one-way plane kernel (FP64) does after its inverse transforms (fame_plane64.hip) */
enum { SYN_FIELD = 0, SYN_REF = 1, SYN_EPS = 2, SYN_RES = 3 };
struct KSyn {
    KPlane k;                    /* invB: 1 / (N eps) for SYN_EPS               */
    const double2* outer;        /* exp(2 i pi r0 c / nc), nc per problem       */
    const double2* in;           /* analysis: field in the reference's layout (General), or null: in place */
    double2* out;                /* SYN_REF: field in the reference's layout    */
    const double2* E;            /* SYN_RES: the fields, reference's layout (General) */
    const double* eps;           /* SYN_RES: permittivity, reference's layout   */
    const double* w2;            /* SYN_RES: omega^2 of problem p at w2[p w2step] */
    size_t ostride;              /* problem stride of in / out / E              */
    double* part;                /* SYN_EPS: |E|^2 per block; SYN_RES: |r|^2, |E|^2 per block */
    int w2step;
    int batch;                   /* problems by which the block size is chosen: the sums' order (0: the launch's) */
};

struct KAxis {
    fame::GridDev g;
    const fame::ProbDev* prob;
    fame::LinePlanDev plan;
    const int* active;
    void* f;
    const void* invB;            /* outer EPS mode: 3N reals, internal layout  */
    /* outer EPS mode inside CG (optional): per block, the sum over its lines of
     * conj(v) (scale eps^-1 v) of the real-space values v, i.e. the block's
     * share of <p, QBQ p> when every line transform is an unnormalised DFT;
     * layout [problem][component][gridDim.x], blocks past the last tile write 0 */
    double* pap;
    size_t fstride;
    int L, P;                    /* lines per block, LDS line pitch            */
    unsigned mL;                 /* udiv magic for / L                         */
};

/* inner-axis kernels keep a table of na complex doubles after their lines:
 * its offset in line entries (rounded to 16 bytes for FP32 entries) and the
 * entries it adds to the LDS size                                            */
__host__ __device__ inline int inner_tab_offset(int entries, int prec) {
    return prec == 8 ? entries : ((entries + 1) & ~1);
}
__host__ __device__ inline int inner_tab_extra(int na, int prec) { return prec == 8 ? na : 2 * na + 1; }
/* behind it, per line, the inner twiddle exp(2 i pi phi a / na) split as
 * a = 16 ah + al: 16 entries for al and ceil(na / 16) for ah, in the kernel's
 * precision.  Entries (kernel precision) of both tables for L lines:         */
__host__ __device__ inline int inner_tw_per_line(int na) { return 16 + (na + 15) / 16; }
__host__ __device__ inline int inner_lds_extra(int na, int prec, int L) {
    return inner_tab_extra(na, prec) + 1 + L * inner_tw_per_line(na);
}

/* LDS bytes of a line-transform launch: tables + nl lines + extra entries */
size_t fame_line_lds(const fame::LinePlanDev& pl, int prec, int nl, int P, int extra);

hipError_t fame_launch_inner(const KInner& a, int expand, int prec, int nprob, hipStream_t s);
hipError_t fame_launch_mid(const KAxis& a, int dir, int prec, int nprob, hipStream_t s);
hipError_t fame_launch_outer(const KAxis& a, int mode, int prec, int nprob, hipStream_t s);
/* dynamic LDS of one block that leaves a second one room on the CU (160 KiB,
 * with the kernels' static LDS) */
#define FAME_LDS_HALF (80 * 1024 - 256)
/* LDS bytes of the plane path's kernels */
inline size_t fame_plane_lds(int nb, int nc, int ntab, int prec) {
    return (size_t)(prec == 8 ? 16 : 8) * ((size_t)ntab + (((size_t)nc * (nb | 1) + 1) & ~(size_t)1));
}
inline size_t fame_line_lds2(int na, int ntab, int L, int P, int prec) {
    return 16 * (size_t)na + sizeof(LineTab) * L + (prec == 8 ? 16 : 8) * ((size_t)ntab + (size_t)L * inner_tw_per_line(na) + 3 * (size_t)L * P);
}
hipError_t fame_launch_line32(const KLine& k, int expand, int mode, int nprob, hipStream_t s);
hipError_t fame_launch_line64(const KLine& k, int expand, int mode, int nprob, hipStream_t s);
hipError_t fame_launch_plane32(const KPlane& k, int nprob, hipStream_t s);
hipError_t fame_launch_plane64(const KPlane& k, int nprob, hipStream_t s);
hipError_t fame_prepare_plane32(int eb, int ec);
hipError_t fame_prepare_plane64(int eb, int ec);
hipError_t fame_prepare_syn(int eb, int ec);
hipError_t fame_launch_syn(const KSyn& k, int mode, int nprob, hipStream_t s);
hipError_t fame_launch_ana(const KSyn& k, int nprob, hipStream_t s);
hipError_t fame_launch_curl(const KLine& k, int nprob, hipStream_t s);
/* out = s in^T for `batch` matrices (rows x cols, pitch ip) of each problem, s the
 * square root of scale2[p] (null: 1) */
hipError_t fame_launch_transpose(const double2* in, double2* out, int rows, int cols, int ip, int op, size_t ib, size_t ob,
                                 int batch, size_t is, size_t os, const double* scale2, int nprob, hipStream_t s);
/* partials of |F - w2 eps E|^2 and |E|^2, F in the plane layout [component][a][PP] of a
 * Simple grid, E and eps in its reference layout [component][c b][a] */
hipError_t fame_launch_resid_simple(const double2* F, const double2* E, const double* eps, const double* w2, int w2step,
                                    double* part, int nblk, int na, int nl, int PP, size_t fs, size_t es, int nprob,
                                    hipStream_t s);
/* 1/eps, eps and 1 / (N eps) in the kernels' layouts from the reference's */
hipError_t fame_launch_eps(const fame::GridDev& g, const double* eps, double* eps_int, double* ib64, float* ib32, double* p64,
                           float* p32, int PP, hipStream_t s);
hipError_t fame_launch_line_tab(const fame::GridDev& g, const fame::ProbDev* prob, LineTab* lt, void* tw64, void* tw32,
                                void* mid64, void* mid32, double2* outer, int nprob, hipStream_t s);
hipError_t fame_launch_xz_transpose(const void* in, void* out, int nx, int ny, int nz, int dir, size_t stride,
                                    int ncomp, int nprob, int prec, hipStream_t s);
hipError_t fame_launch_pack(const void* in, void* out, int N, int Nd, int dir, int prec, hipStream_t s);

/* ---- vector / reduction kernels (fame_blas.hip) ------------------------- */

/* x = 0, r = p = b and the partials of <r,r> (stride: problem stride in elements) */
hipError_t fame_cg_begin(void* x, void* r, void* p, const void* b, double* partials, int nblk,
                         size_t n, size_t stride, int nprob, int prec, const int* mask, hipStream_t s);
hipError_t fame_cg_init_scal(CgScal* sc, const double* partials, int nblk, double tol, int maxit, int nprob,
                             int* active, hipStream_t s);
/* CG iteration with Ap stored (any plan): alpha from the summed <r,r>, <r,r>
 * of the next residual by one step of |r - alpha Ap|^2 = |alpha|^2 |Ap|^2 -
 * |r|^2 (conjugacy: <r,Ap> = <p,Ap>), beta and the active flags, from the
 * 6-double partials of the expanding and contracting passes */
/* CG iteration with the residual updated by the contracting pass (when the
 * outer pass sums <p,Ap>): alpha = <r,r> / <p,Ap> from the outer pass's 3 npap
 * block sums per problem, launched before the contracting pass; then beta and
 * the active flags from the exact <r,r> of the updated residual (slot 3 of the
 * inner partials) */
hipError_t fame_cg_alpha(CgScal* sc, const double* pap, int npap, int nprob, const int* active, hipStream_t s);
hipError_t fame_cg_beta(CgScal* sc, const double* partials, int nblk, int step, int nprob, int* active, hipStream_t s,
                        CgNote* note = nullptr, unsigned seq = 0);
/* the scalar state, or the sum of nblk partials per problem, into the notes */
hipError_t fame_cg_note(const CgScal* sc, int nprob, CgNote* note, unsigned seq, hipStream_t s);
hipError_t fame_sum_note(const double* partials, int nblk, int nprob, CgNote* note, unsigned seq, hipStream_t s);
hipError_t fame_cg_alpha_beta(CgScal* sc, const double* partials, int nblk, int nprob, int* active, hipStream_t s);
hipError_t fame_cg_finish_x(void* x, const void* p, const CgScal* sc, size_t n, size_t stride, int nprob, int prec,
                            hipStream_t s);
/* an FP32 solve inside FP64 refinement starting from the FP64 right-hand
 * side: x32 = 0, r32 = p32 = b64 rounded, with the <r,r> partials */
hipError_t fame_cg_begin_mixed(void* x32, void* r32, void* p32, const void* b64, double* partials, int nblk, size_t n,
                               size_t stride, int nprob, const int* mask, hipStream_t s, void* x64 = nullptr);

/* generic helpers (complex double unless prec says float) */
hipError_t fame_scale_real(void* y, const void* x, const double* sreal, size_t n, size_t xstride, size_t sstride,
                           int nprob, int prec, hipStream_t s);
/* mask (device, optional): problems with mask 0 are left untouched */
hipError_t fame_convert(void* dst, int dprec, const void* src, int sprec, size_t n, size_t dstride, size_t sstride,
                        int nprob, hipStream_t s, const int* mask = nullptr);
hipError_t fame_norm2_partials(const void* x, int prec, double* partials, int nblk, size_t n, size_t stride, int nprob,
                               hipStream_t s);
hipError_t fame_reduce_partials(const double* partials, int nblk, int ncomp, double* out, int nprob, hipStream_t s);

/* Lanczos block kernels: V columns of length n (complex double), column stride cstride,
 * problem stride pstride */
hipError_t fame_gemv_h(const void* V, const void* w, double* partials, int nblk, int m, size_t n, size_t cstride,
                       size_t pstride, size_t wstride, int nprob, const int* mask, hipStream_t s);
hipError_t fame_gemv_n(const void* V, void* w, const double* h, int m, size_t n, size_t cstride, size_t pstride,
                       size_t wstride, size_t hstride, int nprob, const int* mask, hipStream_t s);
/* most basis columns (nstep + 1) the Gram and U*Q kernels take */
#define FAME_LZ_MAXCOL 128
hipError_t fame_gram(const void* V, double* partials, int nblk, int m, size_t n, size_t cstride, size_t pstride,
                     int nprob, const int* mask, hipStream_t s);
hipError_t fame_gemm_vq(const void* V, const double* Q, void* W, int m, int q, size_t n, size_t cstride,
                        size_t pstride, size_t wcstride, size_t wpstride, size_t qstride, int nprob, const int* mask,
                        hipStream_t s);
hipError_t fame_lanczos_step(void* V, int j, const double* alpha_beta_prev, double* partials, int nblk, size_t n,
                             size_t cstride, size_t pstride, int nprob, const int* mask, hipStream_t s);
hipError_t fame_launch_sigma(const fame::GridDev& g, const fame::ProbDev* prob, double* sig, double* sig_inv, int nprob,
                             hipStream_t s);

/* Lanczos scalar helpers (fame_blas.hip) */
hipError_t fame_lz_coeffs(const double* hdot, double* T0d, const double* T1d, int ld, int j, double* hout,
                          int nprob, const int* mask, hipStream_t s);
hipError_t fame_lz_second_pass_mask(const double* h, int n, double tau2, const int* in, int* out, int nprob,
                                    hipStream_t s);
hipError_t fame_lz_beta(const double* nrm2, double* T1d, int ld, int j, double* invb, int nprob, const int* mask,
                        hipStream_t s);
hipError_t fame_scale_real_mod(void* y, const void* x, const double* sreal, size_t n, size_t xstride, size_t sstride,
                               size_t smod, int nprob, int prec, hipStream_t s, const int* mask = nullptr);
/* y = s x with separate problem strides for y and x */
hipError_t fame_scale_real_mod2(void* y, size_t ystride, const void* x, size_t xstride, const double* sreal, size_t n,
                                size_t sstride, size_t smod, int nprob, int prec, hipStream_t s,
                                const int* mask = nullptr);
hipError_t fame_cg_init_scal2(CgScal* sc, const double* partials, int nblk, double tol, double reltol, int maxit,
                              int nprob, int* active, const int* mask, hipStream_t s);
