/*
 * fame_pass.hpp -- line transforms of the plane kernels (fame_plane.hpp): the
 * Stockham passes and the matrix-core direct DFT of fame_device.hpp over lines
 * of any element stride in LDS, for any number of lines.
 *
 * Element m of line l is S[l LS + m ES].  Against fft_pass of fame_device.hpp:
 *   - the transform sign is a template parameter (a run-time sign costs a select
 *     and two register moves per twiddle, 7 instead of 4 instructions);
 *   - lanes run across the lines (conflict-free in LDS for an odd line stride or
 *     for LS = 1), and a pass takes its lines in rounds, so that the lines of a
 *     block are not bounded by its registers;
 *   - hooks at the first and last pass of a transform multiply by plane-shaped
 *     arrays in global memory, read coalesced along the lines.
 */
#pragma once
#include "fame_device.hpp"
#include "fame_kernels.h"

namespace fame {

/* stages are read through the constant address space: scalar loads, and no
 * private copy of a by-value argument that is indexed at run time           */
typedef const __attribute__((address_space(4))) PlaneStage CStage;
__device__ __forceinline__ CStage* cstage(const PlaneStage* p) { return (CStage*)(uintptr_t)p; }
__device__ __forceinline__ PlaneStage load_stage(CStage* p) {
    PlaneStage s;
    s.R = p->R; s.Ns = p->Ns; s.nb = p->nb; s.tstep = p->tstep; s.mNs = p->mNs;
    return s;
}

/* One scalar load from each 64-byte line of a kernel's arguments (BYTES of them),
 * all under way together, at its start: the pass descriptors that a small grid's
 * block reads one after another between its barriers then come from the scalar
 * cache instead of one memory round trip each                                 */
template <int BYTES>
__device__ __forceinline__ void touch_args() {
    typedef const __attribute__((address_space(4))) unsigned CUint;
    CUint* a = (CUint*)__builtin_amdgcn_kernarg_segment_ptr();
    unsigned v = 0;
#pragma unroll
    for (int i = 0; i < BYTES / 4; i += 16) v ^= a[i];
    asm volatile("" :: "s"(v));
}

/* lines per round of a pass with nbf butterflies per line, NBT per thread, and
 * id / lpr as (id + 1/2) * (1 / lpr): exact, since the quotient is below 2^13 and
 * its distance from an integer at least 1 / (2 lpr)                          */
struct Rounds {
    int lpr;
    float inv;
    __device__ __forceinline__ Rounds(int nl, int nbf, int slots) {
        lpr = min(nl, slots / nbf);
        inv = 1.0f / (float)lpr;
    }
    __device__ __forceinline__ int div(int id) const { return (int)(((float)id + 0.5f) * inv); }
};

template <typename T> struct C2;
template <> struct C2<double> { typedef double2 T2; };
template <> struct C2<float> { typedef float2 T2; };

/* hook bits of a transform: multiply element m of line l, at [m ld + l],
 *   HK_TIN  by tw before the first pass,
 *   HK_TOUT by conj(tw) after the last pass
 * (eps and pap serve the fused middle pass)                                  */
enum { HK_TIN = 1, HK_TOUT = 2 };
template <typename T, typename T2>
struct Hook {
    const T2* tw;
    const T* eps;
    int ld;
    bool pap;
};

/* element o of a uniform array: a scalar base and a 32-bit byte offset */
template <typename V>
__device__ __forceinline__ V ld_uni(const V* base, unsigned o) {
    return *reinterpret_cast<const V*>(reinterpret_cast<const char*>(base) + (size_t)(o * (unsigned)sizeof(V)));
}

/* One in-place Stockham pass.  It starts with the barrier that closes what came
 * before (a transform ends without one), after the loads of its first round's
 * hook values are under way, and each round fetches the next round's before its
 * own barrier. */
template <typename T, typename T2, int R, int MAXE, bool INV, int HK>
__device__ __forceinline__ void line_pass(T2* S, int nl, int LS, int ES, const PlaneStage& st, const T2* W,
                                          const Hook<T, T2>& hk, bool first, bool last) {
    constexpr int NBT = nbt_of(R, MAXE);
    const int nbf = st.nb, Ns = st.Ns, NT = (int)blockDim.x;
    const Rounds rd(nl, nbf, NT * NBT);
    const int lpr = rd.lpr;
    T2 u[HK ? NBT : 1][HK ? R : 1];
    const bool hooked = (HK == HK_TIN && first) || (HK == HK_TOUT && last);
    auto place = [&](int i, int l0, int& j, int& line) {
        int id = (int)threadIdx.x + i * NT;
        asm volatile("" : "+v"(id));   /* keep the index of each butterfly out of the enclosing loops' live ranges */
        j = rd.div(id);
        line = l0 + id - j * lpr;
        return j < nbf && line < nl;
    };
    auto fetch = [&](int l0) {
        if constexpr (HK != 0) {
            if (hooked) {
#pragma unroll
                for (int i = 0; i < NBT; ++i) {
                    int j, line;
                    if (place(i, l0, j, line)) {
                        /* HK_TOUT: the last pass has Ns = nb, so its outputs are j + t nb too */
                        const unsigned o = (unsigned)(j * hk.ld + line), os = (unsigned)(nbf * hk.ld);
#pragma unroll
                        for (int t = 0; t < R; ++t) u[i][t] = ld_uni(hk.tw, o + t * os);
                    }
                }
            }
        }
    };
    fetch(0);
    __syncthreads();
    for (int l0 = 0; l0 < nl; l0 += lpr) {
        T2 v[NBT][R];
        int ob[NBT], ol[NBT];
#pragma unroll
        for (int i = 0; i < NBT; ++i) {
            int j, line;
            const bool on = place(i, l0, j, line);
            ob[i] = -1;
            ol[i] = line;
            if (on) {
                const int qd = udiv(j, st.mNs);
                const int k = j - qd * Ns;
                const T2* a = S + line * LS + j * ES;
                const int step = nbf * ES;
#pragma unroll
                for (int t = 0; t < R; ++t) v[i][t] = a[t * step];
                if constexpr (HK == HK_TIN) {
                    if (first) {
#pragma unroll
                        for (int t = 0; t < R; ++t) v[i][t] = cmul(v[i][t], u[i][t]);
                    }
                }
                if (Ns > 1) {
                    const int ks = k * st.tstep;
#pragma unroll
                    for (int t = 1; t < R; ++t) {
                        const T2 w = W[t * ks];
                        v[i][t] = INV ? cmulc(v[i][t], w) : cmul(v[i][t], w);
                    }
                }
                dft<T2, R>(v[i], INV);
                if constexpr (HK == HK_TOUT) {
                    if (last) {
#pragma unroll
                        for (int t = 0; t < R; ++t) v[i][t] = cmulc(v[i][t], u[i][t]);
                    }
                }
                ob[i] = qd * Ns * R + k;
            }
        }
        if (l0 + lpr < nl) fetch(l0 + lpr);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NBT; ++i) {
            if (ob[i] >= 0) {
                T2* o = S + ol[i] * LS + ob[i] * ES;
                const int step = Ns * ES;
#pragma unroll
                for (int t = 0; t < R; ++t) o[t * step] = v[i][t];
            }
        }
    }
}

/* the last pass of an inverse transform, the 1/eps step and the first pass of
 * the forward transform of the same radix: the inverse pass's outputs j + t nb
 * are that forward pass's inputs, so the three run in registers on one LDS round
 * trip.  Returns this thread's share of <v, eps^-1 v> (hk.pap).              */
template <typename T, typename T2, int R, int MAXE>
__device__ __forceinline__ double mid_pass(T2* S, int nl, int LS, int ES, const PlaneStage& st, const T2* W,
                                           const Hook<T, T2>& hk, bool only) {
    constexpr int NBT = nbt_of(R, MAXE);
    const int nbf = st.nb, NT = (int)blockDim.x;
    const Rounds rd(nl, nbf, NT * NBT);
    const int lpr = rd.lpr;
    double acc = 0.0;
    T u[NBT][R];
    auto place = [&](int i, int l0, int& j, int& line) {
        int id = (int)threadIdx.x + i * NT;
        asm volatile("" : "+v"(id));
        j = rd.div(id);
        line = l0 + id - j * lpr;
        return j < nbf && line < nl;
    };
    auto fetch = [&](int l0) {
#pragma unroll
        for (int i = 0; i < NBT; ++i) {
            int j, line;
            if (place(i, l0, j, line)) {
                const unsigned o = (unsigned)(j * hk.ld + line), os = (unsigned)(nbf * hk.ld);
#pragma unroll
                for (int t = 0; t < R; ++t) u[i][t] = ld_uni(hk.eps, o + t * os);
            }
        }
    };
    fetch(0);
    __syncthreads();
    for (int l0 = 0; l0 < nl; l0 += lpr) {
        T2 v[NBT][R];
        int ob[NBT], ol[NBT];
#pragma unroll
        for (int i = 0; i < NBT; ++i) {
            int j, line;
            const bool on = place(i, l0, j, line);
            ob[i] = -1;
            ol[i] = line;
            if (on) {
                const T2* a = S + line * LS + j * ES;
                const int step = nbf * ES;
#pragma unroll
                for (int t = 0; t < R; ++t) v[i][t] = a[t * step];
                if (only) {     /* a single pass: the middle twiddle enters and leaves here */
                    const unsigned o = (unsigned)(j * hk.ld + line), os = (unsigned)(nbf * hk.ld);
#pragma unroll
                    for (int t = 0; t < R; ++t) v[i][t] = cmul(v[i][t], ld_uni(hk.tw, o + t * os));
                } else {
                    const int ks = j * st.tstep;
#pragma unroll
                    for (int t = 1; t < R; ++t) v[i][t] = cmulc(v[i][t], W[t * ks]);
                }
                dft<T2, R>(v[i], true);
#pragma unroll
                for (int t = 0; t < R; ++t) {
                    const T2 x = v[i][t], y = cscale(x, u[i][t]);
                    if (hk.pap) acc += (double)x.x * (double)y.x + (double)x.y * (double)y.y;
                    v[i][t] = y;
                }
                dft<T2, R>(v[i], false);
                ob[i] = j * R;
                if (only) {
                    const unsigned o = (unsigned)(j * R * hk.ld + line);
#pragma unroll
                    for (int t = 0; t < R; ++t) v[i][t] = cmulc(v[i][t], ld_uni(hk.tw, o + t * (unsigned)hk.ld));
                }
            }
        }
        if (l0 + lpr < nl) fetch(l0 + lpr);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NBT; ++i) {
            if (ob[i] >= 0) {
                T2* o = S + ol[i] * LS + ob[i] * ES;
#pragma unroll
                for (int t = 0; t < R; ++t) o[t * ES] = v[i][t];
            }
        }
    }
    return acc;
}

/* run CASE(R) for radix r: the compound radices where a thread holds 16 elements */
#define RADIX_SWITCH(r, MAXE, CASE)                                                                                  \
    switch (r) {                                                                                                     \
        case 2: CASE(2); break;                                                                                      \
        case 3: CASE(3); break;                                                                                      \
        case 4: CASE(4); break;                                                                                      \
        case 5: CASE(5); break;                                                                                      \
        case 7: CASE(7); break;                                                                                      \
        case 8: CASE(8); break;                                                                                      \
        case 11: CASE(11); break;                                                                                    \
        case 13: CASE(13); break;                                                                                    \
        default:                                                                                                     \
            if constexpr (MAXE >= 16) {                                                                              \
                switch (r) {                                                                                         \
                    case 6: CASE(6); break;                                                                          \
                    case 9: CASE(9); break;                                                                          \
                    case 10: CASE(10); break;                                                                        \
                    case 12: CASE(12); break;                                                                        \
                    case 15: CASE(15); break;                                                                        \
                    case 16: CASE(16); break;                                                                        \
                    default: break;                                                                                  \
                }                                                                                                    \
            }                                                                                                        \
            break;                                                                                                   \
    }

/* passes s0 .. s1 - 1 of one transform (no barrier after the last one) */
template <typename T, typename T2, bool INV, int HK, int MAXE>
__device__ __forceinline__ void line_passes(T2* S, int nl, int LS, int ES, CStage* st, int s0, int s1, int nst,
                                            const T2* W, const Hook<T, T2>& hk) {
    if (s0 >= s1) return;
    PlaneStage cur = load_stage(st + s0);
#define LP(R) line_pass<T, T2, R, MAXE, INV, HK>(S, nl, LS, ES, cur, W, hk, s == 0, s + 1 == nst)
    for (int s = s0; s < s1; ++s) {
        /* the next pass's descriptor is on its way while this pass runs */
        const PlaneStage next = load_stage(st + (s + 1 < s1 ? s + 1 : s));
        RADIX_SWITCH(cur.R, MAXE, LP)
        cur = next;
    }
#undef LP
}

/* Direct DFTs on the matrix cores, the products of dft_mfma (fame_device.hpp):
 *   lo.x, hi.x = X +- Y,  X = x_0.x + sum cos s_t.x,  Y = sum sin d_t.y      (half 0)
 *   lo.y, hi.y = X' -+ Y', X' = x_0.y + sum cos s_t.y, Y' = sum sin d_t.x    (half 1)
 * with s_t = x_t + x_{n-t}, d_t = x_t - x_{n-t} formed in registers.  The unit of
 * work of a wave is one half of a group of 16 lines, all NQT output tiles: 12
 * units for 96 lines spread evenly over the 4 SIMDs of a block of 8 waves, where
 * whole groups leave two SIMDs with half the work.
 *   - A operands (cos, -sin) come from LDS as ready fragments [tile][K step][lane]
 *     whose padding is zero (the padding steps read other elements of the line);
 *   - x_0 and, for even n, (-1)^q x_{n/2} start the accumulators;
 *   - a step's operands are loaded while the previous step's products run (a
 *     SIMD holds two or three waves, too few to hide the loads otherwise).
 * Lines past nl repeat the last one and are not stored.  n >= 8.             */
template <typename T, int NQT>
struct MfmaHalf {
    typename Mfma<T>::acc_t x[NQT], y[NQT];
};
template <typename T, typename T2, int NQT>
__device__ __forceinline__ void half_products(MfmaHalf<T, NQT>& o, const T2* S, int g0, int half, int nl, int LS, int ES,
                                              int n, const T2* A) {
    typedef typename Mfma<T>::acc_t acc_t;
    const int m = (n - 1) >> 1, nks = (m + 3) >> 2;
    const int lane = threadIdx.x & 63, row = lane & 15, kq = lane >> 4;
    const T2* Sb = S + min(g0 + row, nl - 1) * LS;
    const T2 z0 = Sb[0];
    T2 zh;
    zh.x = 0; zh.y = 0;
    if (!(n & 1)) zh = Sb[(n >> 1) * ES];
    const T x0 = half ? z0.y : z0.x, h = half ? zh.y : zh.x;
#pragma unroll
    for (int w = 0; w < NQT; ++w) {
#pragma unroll
        for (int v = 0; v < 4; ++v) o.x[w][v] = x0 + ((Mfma<T>::row(kq, v) & 1) ? -h : h);
        o.y[w] = (acc_t){0, 0, 0, 0};
    }
    const T2* Sp = Sb + (kq + 1) * ES;
    const T2* Sm = Sb + (n - 1 - kq) * ES;
    A += lane;
    T2 wn[NQT], an = *Sp, bn = *Sm;
#pragma unroll
    for (int w = 0; w < NQT; ++w) wn[w] = A[w * nks * 64];
#pragma unroll 1
    for (int ks = 0; ks < nks; ++ks) {
        T2 wv[NQT];
        const T s = half ? an.y + bn.y : an.x + bn.x, d = half ? an.x - bn.x : an.y - bn.y;
#pragma unroll
        for (int w = 0; w < NQT; ++w) wv[w] = wn[w];
        const int more = ks + 1 < nks ? 1 : 0;
        Sp += more * 4 * ES; Sm -= more * 4 * ES;
        an = *Sp; bn = *Sm;
#pragma unroll
        for (int w = 0; w < NQT; ++w) wn[w] = A[(w * nks + ks + more) * 64];
#pragma unroll
        for (int w = 0; w < NQT; ++w) {
            o.x[w] = Mfma<T>::mac(wv[w].x, s, o.x[w]);
            o.y[w] = Mfma<T>::mac(wv[w].y, d, o.y[w]);
        }
    }
}
/* forward: X_q = A - iB, X_{n-q} = A + iB, B = -(y accumulators); for q = 0 and
 * q = n / 2 both are the same element and value                             */
template <typename T, typename T2, bool INV, int NQT>
__device__ __forceinline__ void half_store(const MfmaHalf<T, NQT>& o, T2* S, int g0, int half, int nl, int LS, int ES, int n) {
    const int Q = (n >> 1) + 1, lane = threadIdx.x & 63, row = lane & 15, kq = lane >> 4;
    if (g0 + row >= nl) return;
    T* So = reinterpret_cast<T*>(S + (g0 + row) * LS) + half;
    /* the sign of the y term in X_q: half 0 forward -, inverse +; half 1 the opposite */
    const bool minus = INV ? half != 0 : half == 0;
#pragma unroll
    for (int w = 0; w < NQT; ++w)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int q = w * 16 + Mfma<T>::row(kq, v);
            if (w < NQT - 1 || q < Q) {
                const T y = minus ? -o.y[w][v] : o.y[w][v];
                So[2 * (q ? n - q : 0) * ES] = o.x[w][v] - y;
                So[2 * q * ES] = o.x[w][v] + y;
            }
        }
}
template <typename T> struct MfmaUnits { static constexpr int v = 2; };   /* units a wave holds per round */
template <typename T, typename T2, bool INV, int NQT>
__device__ __forceinline__ void line_mfma_n(T2* S, int nl, int LS, int ES, int n, const T2* A) {
    constexpr int NU = MfmaUnits<T>::v;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
    const int ng = (nl + 15) >> 4, per = (NU * nw) >> 1;     /* groups per round */
    for (int gr = 0; gr < ng; gr += per) {
        const int nu = 2 * min(per, ng - gr);
        MfmaHalf<T, NQT> o[NU];
        if (gr == 0) __syncthreads();
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            const int u = wave + i * nw;
            if (u < nu) half_products<T, T2, NQT>(o[i], S, 16 * (gr + (u >> 1)), u & 1, nl, LS, ES, n, A);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            const int u = wave + i * nw;
            if (u < nu) half_store<T, T2, INV, NQT>(o[i], S, 16 * (gr + (u >> 1)), u & 1, nl, LS, ES, n);
        }
    }
}
/* every line of the block; begins with a barrier, ends without one */
template <typename T, typename T2, bool INV>
__device__ __forceinline__ void line_mfma(T2* S, int nl, int LS, int ES, int n, const T2* A) {
    switch (((n >> 1) + 16) >> 4) {      /* ceil((n / 2 + 1) / 16) output tiles */
        case 1: line_mfma_n<T, T2, INV, 1>(S, nl, LS, ES, n, A); break;
        case 2: line_mfma_n<T, T2, INV, 2>(S, nl, LS, ES, n, A); break;
        case 3: line_mfma_n<T, T2, INV, 3>(S, nl, LS, ES, n, A); break;
        default: line_mfma_n<T, T2, INV, 4>(S, nl, LS, ES, n, A); break;
    }
}

/* one transform without hooks; begins with a barrier, ends without one */
template <typename T, typename T2, int ENG, bool INV, int MAXE = MaxE<T>::v>
__device__ __forceinline__ void line_transform(T2* S, int nl, int LS, int ES, const PlaneAxis& ax, const T2* W) {
    if constexpr (ENG == ENG_STOCKHAM) {
        Hook<T, T2> hk;
        hk.tw = nullptr; hk.eps = nullptr; hk.ld = 0; hk.pap = false;
        line_passes<T, T2, INV, 0, MAXE>(S, nl, LS, ES, cstage(INV ? ax.st : ax.sf), 0, ax.nst, ax.nst, W, hk);
    } else {
        line_mfma<T, T2, INV>(S, nl, LS, ES, ax.n, W);
    }
}

/* the c axis of a plane (nl columns, element stride ES): middle twiddle, inverse
 * transform, 1/eps, forward transform, conjugate twiddle; returns the <v, eps^-1 v>
 * share.  Begins with a barrier, ends without one.                           */
template <typename T, typename T2, int ENG, int MAXE = MaxE<T>::v>
__device__ __forceinline__ double column_round_trip(T2* S, int nl, int ES, const PlaneAxis& ax, const T2* W,
                                                    const Hook<T, T2>& hk) {
    double acc = 0.0;
    if constexpr (ENG == ENG_STOCKHAM) {
        const int n = ax.nst;
        const PlaneStage ms = load_stage(cstage(ax.st) + n - 1);
        line_passes<T, T2, true, HK_TIN, MAXE>(S, nl, 1, ES, cstage(ax.st), 0, n - 1, n, W, hk);
#define MP(R) acc = mid_pass<T, T2, R, MAXE>(S, nl, 1, ES, ms, W, hk, n == 1)
        RADIX_SWITCH(ms.R, MAXE, MP)
#undef MP
        line_passes<T, T2, false, HK_TOUT, MAXE>(S, nl, 1, ES, cstage(ax.sf), 1, n, n, W, hk);
    } else {
        /* the elementwise steps as passes of their own, columns fastest */
        const int tot = nl * ax.n;
        auto step = [&](auto f) {
            __syncthreads();
            for (int idx = threadIdx.x; idx < tot; idx += blockDim.x) {
                const int m = udiv(idx, ax.mnl), l = idx - m * nl;
                f(S[l + m * ES], (unsigned)(m * hk.ld + l));
            }
        };
        step([&](T2& e, unsigned o) { e = cmul(e, hk.tw[o]); });
        line_mfma<T, T2, true>(S, nl, 1, ES, ax.n, W);
        step([&](T2& e, unsigned o) {
            const T2 x = e, y = cscale(x, hk.eps[o]);
            if (hk.pap) acc += (double)x.x * (double)y.x + (double)x.y * (double)y.y;
            e = y;
        });
        line_mfma<T, T2, false>(S, nl, 1, ES, ax.n, W);
        step([&](T2& e, unsigned o) { e = cmulc(e, hk.tw[o]); });
    }
    return acc;
}

/* one transform along c with the middle twiddle: inverse with it going in, or
 * forward with its conjugate coming out.  Begins with a barrier, ends without. */
template <typename T, typename T2, int ENG, bool INV, int MAXE = MaxE<T>::v>
__device__ __forceinline__ void column_transform(T2* S, int nl, int ES, const PlaneAxis& ax, const T2* W,
                                                 const Hook<T, T2>& hk) {
    if constexpr (ENG == ENG_STOCKHAM) {
        line_passes<T, T2, INV, INV ? HK_TIN : HK_TOUT, MAXE>(S, nl, 1, ES, cstage(INV ? ax.st : ax.sf), 0, ax.nst, ax.nst, W, hk);
    } else {
        const int tot = nl * ax.n;
        if (!INV) line_mfma<T, T2, INV>(S, nl, 1, ES, ax.n, W);
        __syncthreads();
        for (int idx = threadIdx.x; idx < tot; idx += blockDim.x) {
            const int m = udiv(idx, ax.mnl), l = idx - m * nl;
            T2& e = S[l + m * ES];
            const T2 w = hk.tw[(unsigned)(m * hk.ld + l)];
            e = INV ? cmul(e, w) : cmulc(e, w);
        }
        if (INV) line_mfma<T, T2, INV>(S, nl, 1, ES, ax.n, W);
    }
}

}  // namespace fame
