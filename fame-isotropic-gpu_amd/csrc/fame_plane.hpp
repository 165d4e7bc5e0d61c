/*
 * fame_plane.hpp -- operator applies in three passes over the field, for grids
 * whose (b, c) plane of one component fits the LDS of a CU.
 *
 *   k_expand   Pi expansion of the reduced vector, IFFT along a, inner twiddle;
 *              the field is written in the plane layout F[component][a][c][b]
 *   k_plane    one (c, b) plane of one component per block:
 *              IFFT_b . twiddle . IFFT_c . 1/eps . FFT_c . conj twiddle . FFT_b
 *              on one read and one write (the three axis passes k_mid, k_outer,
 *              k_mid of fame_kernels.hip read and write the field three times)
 *   k_contract conj inner twiddle, FFT along a, Pi^H contraction
 *
 * Per line (b, c) and per plane constants (symbols, phases, twiddles) depend on
 * the wave vector only; they are tabulated once per fame_set_wave_vectors
 * (k_line_tab) instead of being recomputed with sincospi in every block.
 * The plane pitch PP is nb nc rounded up to 16 elements, so that every run of a
 * block's 16 (FP32) or 8 (FP64) lines starts on a 128-byte line.
 */
#pragma once
#include "fame_pass.hpp"

namespace fame {

enum { PIF_SIMPLE = 0, PIF_GUARD = 1, PIF_GEN = 2 };
enum { EX_PLAIN = 0, EX_CG = 1, EX_FX = 2 };
enum { CO_PLAIN = 0, CO_CG = 1, CO_RES = 2 };

__device__ __forceinline__ bool al16(const void* q) { return ((uintptr_t)q & 15) == 0; }
template <typename T> struct Rsq;
template <> struct Rsq<double> { static __device__ __forceinline__ double f(double x) { return rsqrt(x); } };
template <> struct Rsq<float> { static __device__ __forceinline__ double f(double x) { return (double)__builtin_amdgcn_rsqf((float)x); } };

__device__ __forceinline__ double2 fmac2(double2 acc, double2 a, double2 b) {   /* acc + a b */
    return make_double2(acc.x + a.x * b.x - a.y * b.y, acc.y + a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 fmas2(double2 acc, double2 a, double2 b) {   /* acc - a b */
    return make_double2(acc.x - a.x * b.x + a.y * b.y, acc.y - a.x * b.y - a.y * b.x);
}
__device__ __forceinline__ double2 fmacc2(double2 acc, double2 a, double2 b) {  /* acc + a conj(b) */
    return make_double2(acc.x + a.x * b.x + a.y * b.y, acc.y + a.y * b.x - a.x * b.y);
}

/* symbols of mode a of a line and the norms of the Pi basis (the gauge and the
 * guard rule of pi_basis): t = w x Lambda for the two cross-product forms */
template <typename T, int PIK>
struct Geo {
    double2 lx, ly, lz, s, t1, t2, t3;
    double q, i1, i2;
    __device__ __forceinline__ Geo(const LineTab& lt, double2 ea, double iha2) {
        const double2 e = cmul(ea, lt.e);
        const double m = e.y * iha2;                   /* La = 2i sin . exp(i pi x) / h */
        const double2 La = make_double2(-m * e.y, m * e.x);
        q = lt.q + La.x * La.x + La.y * La.y;
        if (PIK == PIF_SIMPLE) { lx = La; ly = lt.b; lz = lt.c; }
        else { lx = lt.c; ly = lt.b; lz = La; }
        if (PIK == PIF_GEN) {
            /* 3 q - |s|^2 as the sum of squares it is (pi_d2_general) */
            s = cadd(lt.s, La);
            const double2 d1 = csub(lz, ly), d2 = csub(lx, lz);
            i2 = Rsq<T>::f(lt.d + d1.x * d1.x + d1.y * d1.y + d2.x * d2.x + d2.y * d2.y);
        } else {
            double n2;
            if (PIK == PIF_GUARD) {
                t1 = csub(lz, ly); t2 = csub(lx, lz); t3 = csub(ly, lx);
                n2 = t1.x * t1.x + t1.y * t1.y + t2.x * t2.x + t2.y * t2.y + t3.x * t3.x + t3.y * t3.y;
            }
            if (PIK == PIF_SIMPLE || n2 <= 1e-30 * q) {
                const double al = 3.0, be = 5.0;
                t1 = csub(cscale(lz, be), ly);
                t2 = csub(lx, cscale(lz, al));
                t3 = csub(cscale(ly, al), cscale(lx, be));
                n2 = t1.x * t1.x + t1.y * t1.y + t2.x * t2.x + t2.y * t2.y + t3.x * t3.x + t3.y * t3.y;
            }
            i2 = Rsq<T>::f(n2);
        }
        i1 = i2 * Rsq<T>::f(q);
    }
    __device__ __forceinline__ void expand(double2 x1, double2 x2, double2 u[3]) const {
        const double2 ga = cscale(x2, i2);
        if (PIK == PIF_GEN) {
            const double2 al = cscale(x1, q * i1), be = cscale(cmulc(x1, s), i1);
            u[0] = fmacc2(fmas2(al, lx, be), ga, csub(lz, ly));
            u[1] = fmacc2(fmas2(al, ly, be), ga, csub(lx, lz));
            u[2] = fmacc2(fmas2(al, lz, be), ga, csub(ly, lx));
        } else {
            const double2 x = cscale(x1, i1);
            const double2 ax = cmulc(x, lx), ay = cmulc(x, ly), az = cmulc(x, lz);
            u[0] = fmacc2(fmas2(cmul(t3, ay), t2, az), ga, t1);
            u[1] = fmacc2(fmas2(cmul(t1, az), t3, ax), ga, t2);
            u[2] = fmacc2(fmas2(cmul(t2, ax), t1, ay), ga, t3);
        }
    }
    __device__ __forceinline__ void contract(double2 w0, double2 w1, double2 w2, double2& y1, double2& y2) const {
        if (PIK == PIF_GEN) {
            const double2 sw = cadd(cadd(w0, w1), w2);
            const double2 t = fmacc2(fmacc2(cmulc(w0, lx), w1, ly), w2, lz);
            y1 = cscale(fmas2(cscale(sw, q), s, t), i1);
            y2 = cscale(fmac2(fmac2(cmul(lx, csub(w1, w2)), ly, csub(w2, w0)), lz, csub(w0, w1)), i2);
        } else {
            const double2 c0 = fmas2(cmul(ly, w2), lz, w1), c1 = fmas2(cmul(lz, w0), lx, w2), c2 = fmas2(cmul(lx, w1), ly, w0);
            const double2 z = fmacc2(fmacc2(cmulc(c0, t1), c1, t2), c2, t3);
            y1 = cscale(z, -i1);
            y2 = cscale(fmac2(fmac2(cmul(t1, w0), t2, w1), t3, w2), i2);
        }
    }
};

template <typename T2> __device__ __forceinline__ T2 rnd(double2 v);
template <> __device__ __forceinline__ double2 rnd<double2>(double2 v) { return v; }
template <> __device__ __forceinline__ float2 rnd<float2>(double2 v) { return make_float2((float)v.x, (float)v.y); }
__device__ __forceinline__ double2 dbl(double2 v) { return v; }
__device__ __forceinline__ double2 dbl(float2 v) { return make_double2(v.x, v.y); }
__device__ __forceinline__ float2 lo2(const float4& v) { return make_float2(v.x, v.y); }
__device__ __forceinline__ float2 hi2(const float4& v) { return make_float2(v.z, v.w); }

/* LDS of the inner-axis kernels: the lines, the transform's table, exp(i pi a /
 * na), the lines' constants and twiddle factors */
template <typename T2>
struct InnerLds {
    T2* S; T2* W; double2* ea; LineTab* lt; T2* tw;
    __device__ __forceinline__ InnerLds(unsigned char* m, int na, int ntab, int L, int P) {
        ea = reinterpret_cast<double2*>(m);
        lt = reinterpret_cast<LineTab*>(ea + na);
        W = reinterpret_cast<T2*>(lt + L);
        tw = W + ntab;
        S = tw + L * inner_tw_per_line(na);
    }
};
__device__ __forceinline__ int inner_tile() { return xcd_tile(); }

/* CG scalars inside the inner kernels.  A reduction kernel of one block per problem
 * took 4.4 us, twice per iteration (of 33 us on a 32^3 grid, of 110 at FCC 96);
 * here every block sums the up to 2048 block sums of the kernel before (from L2,
 * behind the loads of its tables), all in the same order, so that all hold the
 * same alpha and beta.  State goes back and forth between two copies, each kernel
 * reading one and its first block writing the other.
 * wave_part: this thread's share, reduced over its wave into red; the block's
 * next barrier makes it visible to wave_total                                */
__device__ __forceinline__ void wave_part(const double* v, int n, double* red) {
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += FFT_THREADS) s += v[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
}
__device__ __forceinline__ double wave_total(const double* red) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < FFT_THREADS / 64; ++w) s += red[w];
    return s;
}

/* copy the tables of a block's lines l0.. (at most L) into LDS */
template <typename T2>
__device__ __forceinline__ void inner_tables(const KLine& k, const InnerLds<T2>& m, int p, int l0, int nl) {
    const int na = k.g.na, tpl = inner_tw_per_line(na), nlines = k.g.nb * k.g.nc;
    const double2* ea = reinterpret_cast<const double2*>(k.ea);
    const T2* W = reinterpret_cast<const T2*>(k.a.W);
    for (int i = threadIdx.x; i < na; i += blockDim.x) m.ea[i] = ea[i];
    for (int i = threadIdx.x; i < k.a.ntab; i += blockDim.x) m.W[i] = W[i];
    const double* ls = reinterpret_cast<const double*>(k.lt + (size_t)p * nlines + l0);
    double* ld = reinterpret_cast<double*>(m.lt);
    for (int i = threadIdx.x; i < nl * (int)(sizeof(LineTab) / 8); i += blockDim.x) ld[i] = ls[i];
    const T2* ts = reinterpret_cast<const T2*>(k.tw) + ((size_t)p * nlines + l0) * tpl;
    for (int i = threadIdx.x; i < nl * tpl; i += blockDim.x) m.tw[i] = ts[i];
}

/* field by field: a struct assignment goes through scratch */
__device__ __forceinline__ void cg_copy(CgScal& o, const CgScal& c) {
    o.rr = c.rr; o.rr0 = c.rr0; o.pap_re = c.pap_re; o.pap_im = c.pap_im;
    o.alpha_re = c.alpha_re; o.alpha_im = c.alpha_im; o.beta = c.beta; o.tol2 = c.tol2;
    o.iters = c.iters; o.maxit = c.maxit; o.active = c.active; o.pend = c.pend; o.upd = c.upd;
}

/* F = twid . IFFT_a(Pi x), field in the plane layout.  EX_CG: x is the search
 * direction p, and x_sol += alpha p (pending), p = r + beta p ride on the read;
 * EX_FX: x += fx32 + alpha fp32 of the FP32 solve that just ended.          */
template <typename T, int ENG, int PIK, int MODE>
__global__ void __launch_bounds__(FFT_THREADS) k_expand(KLine k) {
    typedef typename C2<T>::T2 T2;
    touch_args<sizeof(KLine)>();
    const int p = blockIdx.y;
    const int nlines = k.g.nb * k.g.nc, na = k.g.na, L = k.L, P = k.P;
    const int tile = inner_tile(), l0 = tile * L;
    if (l0 >= nlines) return;
    const bool fold = MODE == EX_CG && k.sc2;
    if (!fold && k.active && !k.active[p]) return;
    /* in a batch the blocks of problems that are done must not load anything; a
     * single problem is rarely done, and its loads need not wait for the flag   */
    if (fold && gridDim.y > 1 && !k.cgsc[p].active) {
        if (tile == 0 && threadIdx.x == 0) { cg_copy(k.sc2[p], k.cgsc[p]); k.act_out[p] = 0; }
        return;
    }
    __shared__ double red[FFT_THREADS / 64];
    const int nl = min(L, nlines - l0);
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const InnerLds<T2> m(smem_raw, na, k.a.ntab, L, P);
    const bool gam = k.prob[p].gamma != 0;
    const double iha2 = 2.0 * k.g.iha;
    T2* X = reinterpret_cast<T2*>(const_cast<void*>(k.x)) + (size_t)p * k.xstride;
    /* reduced vectors: mode f of the first half at [f - off], of the second at
     * [half + f - off]; the reference's layout leaves out mode 0 at Gamma     */
    const unsigned off = k.ref && gam ? 1u : 0u, half = (unsigned)k.g.N - off;
    T beta = 0, al = 0;
    bool pend = true;
    /* under the first loads of the vectors: the tables and the scalars */
    auto start = [&]() -> bool {
        if (fold) wave_part(k.rpart + (size_t)p * k.nrp, k.nrp, red);
        inner_tables<T2>(k, m, p, l0, nl);
        __syncthreads();
        if (MODE == EX_PLAIN) return true;
        const CgScal& c = k.cgsc[p];
        double bd = c.beta;
        pend = c.pend != 0;
        al = (T)c.alpha_re;
        if (fold) {
            double rr = c.rr;
            int it = c.iters, act = c.active;
            if (act && c.upd) cg_rule(wave_total(red), c.tol2, c.maxit, rr, bd, it, act);
            if (tile == 0 && threadIdx.x == 0) {
                CgScal& o = k.sc2[p];
                cg_copy(o, c);
                o.rr = rr; o.beta = bd; o.iters = it; o.active = act; o.upd = 0;
                k.act_out[p] = act;
            }
            if (!act) return false;
        }
        beta = (T)bd;
        return true;
    };
    T2* S = m.S;
    const int tot = nl * na;
    auto put = [&](int line, int a, unsigned f, T2 x1, T2 x2) {
        double2 u[3] = {make_double2(0, 0), make_double2(0, 0), make_double2(0, 0)};
        if (!(gam && f == 0)) {
            const Geo<T, PIK> g(m.lt[line], m.ea[a], iha2);
            g.expand(dbl(x1), dbl(x2), u);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) S[(c * L + line) * P + a] = rnd<T2>(u[c]);
    };
    bool on = true;
    if constexpr (MODE == EX_CG) {
        const T2* R = reinterpret_cast<const T2*>(k.r) + (size_t)p * k.xstride;
        T2* Y = reinterpret_cast<T2*>(k.xs) + (size_t)p * k.xstride;
        bool done = false;
        if constexpr (sizeof(T) == 4) {
            if (!(na & 1) && al16(X) && al16(R) && al16(Y) && !(half & 1)) {
                done = true;
                /* two consecutive modes of a line per thread, 16-byte accesses */
                struct In { float4 x1, x2, r1, r2, s1, s2; };
                on = batched_loop_over<1>(tot >> 1,
                    [&](int i) -> In {
                        const unsigned f = (unsigned)(l0 * na + 2 * i);
                        In d;
                        d.x1 = *reinterpret_cast<const float4*>(X + f);
                        d.x2 = *reinterpret_cast<const float4*>(X + half + f);
                        d.r1 = *reinterpret_cast<const float4*>(R + f);
                        d.r2 = *reinterpret_cast<const float4*>(R + half + f);
                        if (pend) {
                            d.s1 = *reinterpret_cast<const float4*>(Y + f);
                            d.s2 = *reinterpret_cast<const float4*>(Y + half + f);
                        }
                        return d;
                    },
                    start,
                    [&](int i, const In& d) {
                        const int line = udiv(2 * i, k.g.m_na), a = 2 * i - line * na;
                        const unsigned f = (unsigned)(l0 * na + 2 * i);
                        if (pend) {
                            *reinterpret_cast<float4*>(Y + f) = make_float4(d.s1.x + al * d.x1.x, d.s1.y + al * d.x1.y,
                                                                            d.s1.z + al * d.x1.z, d.s1.w + al * d.x1.w);
                            *reinterpret_cast<float4*>(Y + half + f) = make_float4(d.s2.x + al * d.x2.x, d.s2.y + al * d.x2.y,
                                                                                   d.s2.z + al * d.x2.z, d.s2.w + al * d.x2.w);
                        }
                        const float4 p1 = make_float4(d.r1.x + beta * d.x1.x, d.r1.y + beta * d.x1.y,
                                                      d.r1.z + beta * d.x1.z, d.r1.w + beta * d.x1.w);
                        const float4 p2 = make_float4(d.r2.x + beta * d.x2.x, d.r2.y + beta * d.x2.y,
                                                      d.r2.z + beta * d.x2.z, d.r2.w + beta * d.x2.w);
                        *reinterpret_cast<float4*>(X + f) = p1;
                        *reinterpret_cast<float4*>(X + half + f) = p2;
                        put(line, a, f, lo2(p1), lo2(p2));
                        put(line, a + 1, f + 1, hi2(p1), hi2(p2));
                    });
            }
        }
        if (!done) {
            struct In { T2 x1, x2, r1, r2, s1, s2; };
            on = batched_loop_over<2>(tot,
                [&](int i) -> In {
                    const unsigned f = (unsigned)(l0 * na + i);
                    In d;
                    d.x1 = X[f]; d.x2 = X[half + f];
                    d.r1 = R[f]; d.r2 = R[half + f];
                    if (pend) { d.s1 = Y[f]; d.s2 = Y[half + f]; }
                    return d;
                },
                start,
                [&](int i, const In& d) {
                    const int line = udiv(i, k.g.m_na), a = i - line * na;
                    const unsigned f = (unsigned)(l0 * na + i);
                    if (pend) {
                        T2 s1 = d.s1, s2 = d.s2;
                        s1.x += al * d.x1.x; s1.y += al * d.x1.y;
                        s2.x += al * d.x2.x; s2.y += al * d.x2.y;
                        Y[f] = s1; Y[half + f] = s2;
                    }
                    T2 p1, p2;
                    p1.x = d.r1.x + beta * d.x1.x; p1.y = d.r1.y + beta * d.x1.y;
                    p2.x = d.r2.x + beta * d.x2.x; p2.y = d.r2.y + beta * d.x2.y;
                    X[f] = p1; X[half + f] = p2;
                    put(line, a, f, p1, p2);
                });
        }
    } else {
        const float2* FX = MODE == EX_FX ? reinterpret_cast<const float2*>(k.fx32) + (size_t)p * k.xstride : nullptr;
        const float2* FP = MODE == EX_FX ? reinterpret_cast<const float2*>(k.fp32) + (size_t)p * k.xstride : nullptr;
        const double* sg = k.sig ? k.sig + (size_t)p * k.g.N : nullptr;
        struct In { T2 x1, x2; float2 s1, s2, v1, v2; };
        on = batched_loop_over<2>(tot,
            [&](int i) -> In {
                const unsigned f = (unsigned)(l0 * na + i);
                In d;
                d.x1.x = 0; d.x1.y = 0; d.x2 = d.x1;
                if (f >= off) { d.x1 = X[f - off]; d.x2 = X[half + f - off]; }
                if (MODE == EX_FX) {
                    d.s1 = FX[f]; d.s2 = FX[half + f];
                    if (pend) { d.v1 = FP[f]; d.v2 = FP[half + f]; }
                } else if (sg) {
                    const T s = (T)sg[f];
                    d.x1 = cscale(d.x1, s); d.x2 = cscale(d.x2, s);
                }
                return d;
            },
            start,
            [&](int i, const In& d) {
                const int line = udiv(i, k.g.m_na), a = i - line * na;
                const unsigned f = (unsigned)(l0 * na + i);
                T2 x1 = d.x1, x2 = d.x2;
                if (MODE == EX_FX) {
                    float2 u1 = d.s1, u2 = d.s2;
                    if (pend) {
                        const float fa = (float)al;
                        u1.x += fa * d.v1.x; u1.y += fa * d.v1.y;
                        u2.x += fa * d.v2.x; u2.y += fa * d.v2.y;
                    }
                    x1.x += (T)u1.x; x1.y += (T)u1.y; x2.x += (T)u2.x; x2.y += (T)u2.y;
                    X[f] = x1; X[half + f] = x2;
                }
                put(line, a, f, x1, x2);
            });
    }
    if (!on) return;
    if (nl < L) {   /* lines past the last one transform as zeros */
        T2 z; z.x = 0; z.y = 0;
        for (int i = threadIdx.x; i < 3 * (L - nl) * na; i += blockDim.x) {
            const int r = i / na, a = i - r * na, c = r / (L - nl), line = nl + r - c * (L - nl);
            S[(c * L + line) * P + a] = z;
        }
    }
    line_transform<T, T2, ENG, true>(S, 3 * L, P, 1, k.a, m.W);
    __syncthreads();
    /* inner twiddle exp(2 i pi phi a / na) = th[a >> 4] tl[a & 15] of the line, and
     * the store: lanes across the lines, one run of L consecutive positions per a */
    const int tpl = inner_tw_per_line(na);
    T2* F = reinterpret_cast<T2*>(k.f) + (size_t)p * k.fstride + l0;
    const unsigned PP = (unsigned)k.PP, cs = (unsigned)k.cs;
    if constexpr (sizeof(T) == 4) {
        const int Lh = L >> 1;
        for (int i = threadIdx.x; i < Lh * na; i += blockDim.x) {
            const int a = udiv(i, k.mLs), line = 2 * (i - a * Lh);
            const T2* t0 = m.tw + line * tpl;
            const T2* t1 = t0 + tpl;
            const float2 w0 = cmul(t0[16 + (a >> 4)], t0[a & 15]), w1 = cmul(t1[16 + (a >> 4)], t1[a & 15]);
            const unsigned f = (unsigned)a * PP + line;
            if (line + 1 < nl) {
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const float2 v0 = cmul(S[(c * L + line) * P + a], w0), v1 = cmul(S[(c * L + line + 1) * P + a], w1);
                    *reinterpret_cast<float4*>(F + c * cs + f) = make_float4(v0.x, v0.y, v1.x, v1.y);
                }
            } else if (line < nl) {
#pragma unroll
                for (int c = 0; c < 3; ++c) F[c * cs + f] = cmul(S[(c * L + line) * P + a], w0);
            }
        }
    } else {
        for (int i = threadIdx.x; i < L * na; i += blockDim.x) {
            const int a = udiv(i, k.mLs), line = i - a * L;
            if (line >= nl) continue;
            const T2* t0 = m.tw + line * tpl;
            const T2 w = cmul(t0[16 + (a >> 4)], t0[a & 15]);
            const unsigned f = (unsigned)a * PP + line;
#pragma unroll
            for (int c = 0; c < 3; ++c) F[c * cs + f] = cmul(S[(c * L + line) * P + a], w);
        }
    }
}

/* y = Pi^H FFT_a(conj(twid) . F).  CO_CG: r -= alpha y in place of y, with the
 * block sums of <r, r>; CO_RES: the next FP32 solve's start r32 = p32 = b - y,
 * x32 = 0, with the block sums of |r32|^2.                                   */
template <typename T, int ENG, int PIK, int MODE>
__global__ void __launch_bounds__(FFT_THREADS) k_contract(KLine k) {
    typedef typename C2<T>::T2 T2;
    touch_args<sizeof(KLine)>();
    const int p = blockIdx.y;
    const int nlines = k.g.nb * k.g.nc, na = k.g.na, L = k.L, P = k.P;
    const int tile = inner_tile(), l0 = tile * L;
    if (l0 >= nlines) return;
    const bool fold = MODE == CO_CG && k.sc2;
    if (!fold && k.active && !k.active[p]) return;
    if (fold && gridDim.y > 1 && !k.sc2[p].active) {
        if (tile == 0 && threadIdx.x == 0) cg_copy(k.sc1[p], k.sc2[p]);
        return;
    }
    __shared__ double red[FFT_THREADS / 64];
    const int nl = min(L, nlines - l0);
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const InnerLds<T2> m(smem_raw, na, k.a.ntab, L, P);
    T al = 0;
    auto start = [&]() -> bool {
        if (fold) wave_part(k.pap + (size_t)p * k.npap, k.npap, red);
        inner_tables<T2>(k, m, p, l0, nl);
        __syncthreads();
        if (fold) {
            const CgScal& c = k.sc2[p];
            const int act = c.active;
            /* a = r1 / dot  (CG.cu:60-63); the quadratic form is real */
            const double pq = wave_total(red), a = c.rr / pq;
            if (tile == 0 && threadIdx.x == 0) {
                CgScal& o = k.sc1[p];
                cg_copy(o, c);
                if (act) {
                    o.pap_re = pq; o.pap_im = 0.0;
                    o.alpha_re = a; o.alpha_im = 0.0;
                    o.pend = 1; o.upd = 1;
                }
            }
            if (!act) return false;
            al = (T)a;
        } else if (MODE == CO_CG) {
            al = (T)k.cgsc[p].alpha_re;
        }
        return true;
    };
    const bool gam = k.prob[p].gamma != 0;
    const double iha2 = 2.0 * k.g.iha;
    const int tpl = inner_tw_per_line(na);
    T2* S = m.S;
    const T2* F = reinterpret_cast<const T2*>(k.f) + (size_t)p * k.fstride + l0;
    const unsigned PP = (unsigned)k.PP, cs = (unsigned)k.cs;
    bool on;
    if constexpr (sizeof(T) == 4) {
        struct In { float4 v[3]; };
        const int Lh = L >> 1;
        on = batched_loop_over<1>(Lh * na,
            [&](int i) -> In {
                const int a = udiv(i, k.mLs), line = 2 * (i - a * Lh);
                const unsigned f = (unsigned)a * PP + line;
                In d;
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    d.v[c] = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (line + 1 < nl) d.v[c] = *reinterpret_cast<const float4*>(F + c * cs + f);
                    else if (line < nl) { const float2 t = F[c * cs + f]; d.v[c].x = t.x; d.v[c].y = t.y; }
                }
                return d;
            },
            start,
            [&](int i, const In& d) {
                const int a = udiv(i, k.mLs), line = 2 * (i - a * Lh);
                const T2* t0 = m.tw + line * tpl;
                const T2* t1 = t0 + tpl;
                /* past the last line the tables hold no entry: the value is zero there */
                const float2 one = make_float2(1.f, 0.f);
                const float2 w0 = line < nl ? cmul(t0[16 + (a >> 4)], t0[a & 15]) : one;
                const float2 w1 = line + 1 < nl ? cmul(t1[16 + (a >> 4)], t1[a & 15]) : one;
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    S[(c * L + line) * P + a] = cmulc(lo2(d.v[c]), w0);
                    S[(c * L + line + 1) * P + a] = cmulc(hi2(d.v[c]), w1);
                }
            });
    } else {
        struct In { T2 v[3]; };
        on = batched_loop_over<2>(L * na,
            [&](int i) -> In {
                const int a = udiv(i, k.mLs), line = i - a * L;
                const unsigned f = (unsigned)a * PP + line;
                In d;
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    d.v[c].x = 0; d.v[c].y = 0;
                    if (line < nl) d.v[c] = F[c * cs + f];
                }
                return d;
            },
            start,
            [&](int i, const In& d) {
                const int a = udiv(i, k.mLs), line = i - a * L;
                const T2* t0 = m.tw + line * tpl;
                T2 w; w.x = 1; w.y = 0;
                if (line < nl) w = cmul(t0[16 + (a >> 4)], t0[a & 15]);
#pragma unroll
                for (int c = 0; c < 3; ++c) S[(c * L + line) * P + a] = cmulc(d.v[c], w);
            });
    }
    if (!on) return;
    auto transform = [&]() -> bool {
        line_transform<T, T2, ENG, false>(S, 3 * L, P, 1, k.a, m.W);
        __syncthreads();
        return true;
    };
    const unsigned off = k.ref && gam ? 1u : 0u, half = (unsigned)k.g.N - off;
    const int tot = nl * na;
    double rn = 0.0;
    auto take = [&](int line, int a, unsigned f, T2& o1, T2& o2) {
        double2 y1 = make_double2(0, 0), y2 = make_double2(0, 0);
        if (!(gam && f == 0)) {
            const Geo<T, PIK> g(m.lt[line], m.ea[a], iha2);
            g.contract(dbl(S[(0 * L + line) * P + a]), dbl(S[(1 * L + line) * P + a]), dbl(S[(2 * L + line) * P + a]), y1, y2);
        }
        o1 = rnd<T2>(y1); o2 = rnd<T2>(y2);
    };
    if constexpr (MODE == CO_CG) {
        /* the residual's first group is loaded before the transform */
        T2* R = reinterpret_cast<T2*>(k.r) + (size_t)p * k.xstride;
        struct In1 { T2 r1, r2; };
        struct In2 { float4 r1, r2; };
        auto ld1 = [&](int i) -> In1 {
            const unsigned f = (unsigned)(l0 * na + i);
            In1 d;
            d.r1 = R[f]; d.r2 = R[half + f];
            return d;
        };
        auto use1 = [&](int i, const In1& d) {
            const int line = udiv(i, k.g.m_na), a = i - line * na;
            const unsigned f = (unsigned)(l0 * na + i);
            T2 o1, o2, r1 = d.r1, r2 = d.r2;
            take(line, a, f, o1, o2);
            r1.x -= al * o1.x; r1.y -= al * o1.y;
            r2.x -= al * o2.x; r2.y -= al * o2.y;
            rn += (double)r1.x * r1.x + (double)r1.y * r1.y + (double)r2.x * r2.x + (double)r2.y * r2.y;
            R[f] = r1; R[half + f] = r2;
        };
        if constexpr (sizeof(T) == 4) {
            auto ld2 = [&](int i) -> In2 {
                const unsigned f = (unsigned)(l0 * na + 2 * i);
                In2 d;
                d.r1 = *reinterpret_cast<const float4*>(R + f);
                d.r2 = *reinterpret_cast<const float4*>(R + half + f);
                return d;
            };
            const bool pairs = !(na & 1) && al16(R) && !(half & 1);
            In2 d[1];
            if (pairs) batch_load<1>((int)threadIdx.x, tot >> 1, ld2, d);
            transform();
            if (pairs)
                batched_loop_from<1>(tot >> 1, d, ld2, [&](int i, const In2& d) {
                    const int line = udiv(2 * i, k.g.m_na), a = 2 * i - line * na;
                    const unsigned f = (unsigned)(l0 * na + 2 * i);
                    float2 a1, a2, b1, b2;
                    take(line, a, f, a1, a2);
                    take(line, a + 1, f + 1, b1, b2);
                    const float4 r1 = make_float4(d.r1.x - al * a1.x, d.r1.y - al * a1.y, d.r1.z - al * b1.x, d.r1.w - al * b1.y);
                    const float4 r2 = make_float4(d.r2.x - al * a2.x, d.r2.y - al * a2.y, d.r2.z - al * b2.x, d.r2.w - al * b2.y);
                    rn += (double)r1.x * r1.x + (double)r1.y * r1.y + (double)r1.z * r1.z + (double)r1.w * r1.w +
                          (double)r2.x * r2.x + (double)r2.y * r2.y + (double)r2.z * r2.z + (double)r2.w * r2.w;
                    *reinterpret_cast<float4*>(R + f) = r1;
                    *reinterpret_cast<float4*>(R + half + f) = r2;
                });
            else
                batched_loop<2>(tot, ld1, use1);
        } else {
            batched_loop_over<2>(tot, ld1, transform, use1);
        }
    } else if constexpr (MODE == CO_RES) {
        const T2* B = reinterpret_cast<const T2*>(k.rb) + (size_t)p * k.xstride;
        float2* R32 = reinterpret_cast<float2*>(k.r) + (size_t)p * k.xstride;
        float2* P32 = reinterpret_cast<float2*>(k.p32) + (size_t)p * k.xstride;
        float2* X32 = reinterpret_cast<float2*>(k.xs) + (size_t)p * k.xstride;
        struct In { T2 b1, b2; };
        batched_loop_over<2>(tot,
            [&](int i) -> In {
                const unsigned f = (unsigned)(l0 * na + i);
                In d;
                d.b1 = B[f]; d.b2 = B[half + f];
                return d;
            },
            transform,
            [&](int i, const In& d) {
                const int line = udiv(i, k.g.m_na), a = i - line * na;
                const unsigned f = (unsigned)(l0 * na + i);
                T2 o1, o2;
                take(line, a, f, o1, o2);
                const float2 e1 = make_float2((float)(d.b1.x - o1.x), (float)(d.b1.y - o1.y));
                const float2 e2 = make_float2((float)(d.b2.x - o2.x), (float)(d.b2.y - o2.y));
                const float2 z = make_float2(0.f, 0.f);
                R32[f] = e1; R32[half + f] = e2;
                P32[f] = e1; P32[half + f] = e2;
                X32[f] = z; X32[half + f] = z;
                const float s1 = e1.x * e1.x + e1.y * e1.y, s2 = e2.x * e2.x + e2.y * e2.y;
                rn += (double)s1 + (double)s2;
            });
    } else {
        T2* Y = reinterpret_cast<T2*>(k.xs) + (size_t)p * k.xstride;
        transform();
        for (int i = threadIdx.x; i < tot; i += blockDim.x) {
            const int line = udiv(i, k.g.m_na), a = i - line * na;
            const unsigned f = (unsigned)(l0 * na + i);
            T2 o1, o2;
            take(line, a, f, o1, o2);
            if (f >= off) { Y[f - off] = o1; Y[half + f - off] = o2; }
        }
    }
    if (MODE != CO_PLAIN) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) rn += __shfl_xor(rn, o);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = rn;
        __syncthreads();
        if (threadIdx.x == 0) {
            double sum = 0;
            for (int w = 0; w < FFT_THREADS / 64; ++w) sum += red[w];
            const int nblk = (nlines + L - 1) / L;
            k.rpart[((size_t)p * nblk + tile) * k.rstep] = sum;
        }
    }
}

/* a plane of n = nb nc elements between global memory (contiguous, from G) and LDS
 * (pitch Pb = nb | 1).  nb odd: the LDS rows are as long as the plane's, a linear
 * copy.  FP32: 16 bytes per access, the last element of an odd count by itself */
template <typename T, typename T2, int U>
__device__ __forceinline__ void rows_in(T2* S, const T2* G, int nb, int Pb, unsigned mnb, int n) {
    const int tid = threadIdx.x, nt = blockDim.x;
    if constexpr (sizeof(T) == 4) {
        const int np = n >> 1;
        const float4* G4 = reinterpret_cast<const float4*>(G);
        for (int i0 = tid; i0 < np; i0 += U * nt) {
            float4 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) if (i0 + u * nt < np) v[u] = G4[i0 + u * nt];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int e = 2 * (i0 + u * nt);
                if (e < 2 * np) {
                    if (Pb == nb) { *reinterpret_cast<float4*>(S + e) = v[u]; }
                    else { T2* d = S + e + udiv(e, mnb); d[0] = lo2(v[u]); d[1] = hi2(v[u]); }
                }
            }
        }
        /* n odd: nb is odd too, and with it the copy linear */
        if (tid == 0 && (n & 1)) S[n - 1] = G[n - 1];
    } else {
        for (int i0 = tid; i0 < n; i0 += U * nt) {
            T2 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) if (i0 + u * nt < n) v[u] = G[i0 + u * nt];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int e = i0 + u * nt;
                if (e < n) S[Pb == nb ? e : e + udiv(e, mnb)] = v[u];
            }
        }
    }
}
template <typename T, typename T2>
__device__ __forceinline__ void rows_out(const T2* S, T2* G, int nb, int Pb, unsigned mnb, int n) {
    const int tid = threadIdx.x, nt = blockDim.x;
    if constexpr (sizeof(T) == 4) {
        float4* G4 = reinterpret_cast<float4*>(G);
        for (int i = tid; i < n >> 1; i += nt) {
            const int e = 2 * i;
            if (Pb == nb) G4[i] = *reinterpret_cast<const float4*>(S + e);
            else { const T2* d = S + e + udiv(e, mnb); G4[i] = make_float4(d[0].x, d[0].y, d[1].x, d[1].y); }
        }
        if (tid == 0 && (n & 1)) G[n - 1] = S[n - 1];
    } else {
        for (int i = tid; i < n; i += nt) G[i] = S[Pb == nb ? i : i + udiv(i, mnb)];
    }
}

/* IFFT_b . twiddle . IFFT_c . 1/eps . FFT_c . conj twiddle . FFT_b of one plane */
template <typename T, int ENGB, int ENGC, int TB>
__global__ void __launch_bounds__(TB) k_plane(KPlane k) {
    typedef typename C2<T>::T2 T2;
    /* FP64: 16 elements per thread, and with them the compound radices, where a
     * block of 512 threads leaves 256 registers                              */
    constexpr int MAXE = sizeof(T) == 8 && TB == 512 ? 16 : MaxE<T>::v;
    /* every problem's planes go to all XCDs, a run of consecutive ones each: late in
     * a batch's solve only a few problems iterate (a run over all problems' planes
     * kept those on one or two XCDs: 4.62 k-pts/s on the FCC 96 batch of 30)   */
    touch_args<sizeof(KPlane)>();
    const int npl = 3 * k.g.na;
    const int p = blockIdx.y, pl = xcd_tile();
    if (pl >= npl) return;
    if (k.active && !k.active[p]) return;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int nb = k.b.n, nc = k.c.n, plane = nb * nc, Pb = nb | 1;
    T2* S = reinterpret_cast<T2*>(smem_raw);      /* nc Pb elements, rounded up to an even count */
    T2* Wb = S + ((nc * Pb + 1) & ~1);
    T2* Wc = Wb + k.b.ntab;
    const int tb = k.b.ntab, tc = k.c.ntab;
    for (int i = threadIdx.x; i < tb; i += blockDim.x) Wb[i] = reinterpret_cast<const T2*>(k.b.W)[i];
    for (int i = threadIdx.x; i < tc; i += blockDim.x) Wc[i] = reinterpret_cast<const T2*>(k.c.W)[i];
    const size_t po = (size_t)pl * k.PP;
    T2* F = reinterpret_cast<T2*>(k.f) + (size_t)p * k.fstride + po;
    Hook<T, T2> hk;
    hk.tw = reinterpret_cast<const T2*>(k.tw) + (size_t)p * plane;
    hk.eps = reinterpret_cast<const T*>(k.invB) + po;
    hk.ld = nb;
    hk.pap = k.pap != nullptr;
    rows_in<T, T2, 4>(S, F, nb, Pb, k.mnb, plane);
    line_transform<T, T2, ENGB, true, MAXE>(S, nc, Pb, 1, k.b, Wb);
    double vw = column_round_trip<T, T2, ENGC, MAXE>(S, nb, Pb, k.c, Wc, hk);
    line_transform<T, T2, ENGB, false, MAXE>(S, nc, Pb, 1, k.b, Wb);
    __syncthreads();
    rows_out<T, T2>(S, F, nb, Pb, k.mnb, plane);
    if (hk.pap) {
        __shared__ double red[16];
        for (int o = 32; o > 0; o >>= 1) vw += __shfl_xor(vw, o);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = vw;
        __syncthreads();
        if (threadIdx.x == 0) {
            double sum = 0.0;
            for (int w = 0; w < (int)(blockDim.x >> 6); ++w) sum += red[w];
            k.pap[(size_t)p * npl + pl] = sum;
        }
    }
}

/* ------------------------------------------------------------- launchers ---- */
template <typename T, int ENG, int PIK>
static const void* inner_fn(int expand, int mode) {
    if (expand) {
        if (mode == EX_CG) return (const void*)k_expand<T, ENG, PIK, EX_CG>;
        if constexpr (sizeof(T) == 8) if (mode == EX_FX) return (const void*)k_expand<T, ENG, PIK, EX_FX>;
        return (const void*)k_expand<T, ENG, PIK, EX_PLAIN>;
    }
    if (mode == CO_CG) return (const void*)k_contract<T, ENG, PIK, CO_CG>;
    if constexpr (sizeof(T) == 8) if (mode == CO_RES) return (const void*)k_contract<T, ENG, PIK, CO_RES>;
    return (const void*)k_contract<T, ENG, PIK, CO_PLAIN>;
}
template <typename T>
static const void* inner_fn(const KLine& k, int expand, int mode) {
    const int pik = k.g.pi_guard ? PIF_GUARD : (k.g.general ? PIF_GEN : PIF_SIMPLE);
    if (k.a.eng == ENG_MFMA)
        return pik == PIF_GEN ? inner_fn<T, ENG_MFMA, PIF_GEN>(expand, mode)
             : pik == PIF_GUARD ? inner_fn<T, ENG_MFMA, PIF_GUARD>(expand, mode) : inner_fn<T, ENG_MFMA, PIF_SIMPLE>(expand, mode);
    return pik == PIF_GEN ? inner_fn<T, ENG_STOCKHAM, PIF_GEN>(expand, mode)
         : pik == PIF_GUARD ? inner_fn<T, ENG_STOCKHAM, PIF_GUARD>(expand, mode) : inner_fn<T, ENG_STOCKHAM, PIF_SIMPLE>(expand, mode);
}
template <typename T>
static hipError_t launch_line(const KLine& k, int expand, int mode, int nprob, hipStream_t s) {
    KLine q = k;
    void* arg[] = {&q};
    const int nlines = k.g.nb * k.g.nc;
    return hipLaunchKernel(inner_fn<T>(k, expand, mode), dim3(xcd_round((nlines + k.L - 1) / k.L), nprob), dim3(FFT_THREADS),
                           arg, fame_line_lds2(k.g.na, k.a.ntab, k.L, k.P, (int)sizeof(T)), s);
}
/* launch bound TB: 1024 keeps 128 registers, for 16 waves per CU (two blocks of 8,
 * or one of 16).  FP64 planes that fill a CU's LDS with a block of 8 waves take
 * the 512 instance with 256 registers: 56 us against 63 for one wave vector at
 * FCC 96, where the 128 spill.                                               */
template <typename T, int TB>
static const void* plane_fn(int eb, int ec) {
    if (eb == ENG_MFMA) return ec == ENG_MFMA ? (const void*)k_plane<T, ENG_MFMA, ENG_MFMA, TB> : (const void*)k_plane<T, ENG_MFMA, ENG_STOCKHAM, TB>;
    return ec == ENG_MFMA ? (const void*)k_plane<T, ENG_STOCKHAM, ENG_MFMA, TB> : (const void*)k_plane<T, ENG_STOCKHAM, ENG_STOCKHAM, TB>;
}
template <typename T>
static const void* plane_fn(int eb, int ec, int wide) {
    if constexpr (sizeof(T) == 8) if (wide) return plane_fn<T, 512>(eb, ec);
    return plane_fn<T, 1024>(eb, ec);
}
template <typename T>
static hipError_t launch_plane(const KPlane& k, int nprob, hipStream_t s) {
    KPlane q = k;
    void* arg[] = {&q};
    const size_t lds = fame_plane_lds(k.b.n, k.c.n, k.b.ntab + k.c.ntab, (int)sizeof(T));
    return hipLaunchKernel(plane_fn<T>(k.b.eng, k.c.eng, k.wide), dim3(xcd_round(3 * k.g.na), nprob), dim3(k.nt), arg, lds, s);
}
template <typename T>
static hipError_t prepare_plane(int eb, int ec) {
    for (int wide = 0; wide < 2; ++wide) {
        const hipError_t e = hipFuncSetAttribute(plane_fn<T>(eb, ec, wide), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 256);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace fame
