/* fame_plane64.hip -- FP64 instances of the plane kernels (fame_plane.hpp), and
 * the tables of a wave vector that both precisions read */
#include "fame_plane.hpp"

using namespace fame;

hipError_t fame_launch_line64(const KLine& k, int expand, int mode, int nprob, hipStream_t s) { return launch_line<double>(k, expand, mode, nprob, s); }
hipError_t fame_launch_plane64(const KPlane& k, int nprob, hipStream_t s) { return launch_plane<double>(k, nprob, s); }
hipError_t fame_prepare_plane64(int eb, int ec) { return prepare_plane<double>(eb, ec); }

/* per line (b, c) of every problem: its symbols and inner-axis phase, the inner
 * twiddle factors in both precisions, and the middle twiddles of its nb entries'
 * plane (entry gl itself: exp(2 pi i (s0 + s1 c) b / nb))                    */
__global__ void k_line_tab(GridDev g, const ProbDev* prob, LineTab* lt, double2* tw64, float2* tw32, double2* mid64,
                           float2* mid32, double2* outer) {
    const int p = blockIdx.y, nlines = g.nb * g.nc, tpl = inner_tw_per_line(g.na);
    const ProbDev pr = prob[p];
    for (int gl = blockIdx.x * blockDim.x + threadIdx.x; gl < nlines; gl += gridDim.x * blockDim.x) {
        const int c = gl / g.nb, b = gl - c * g.nb;
        const LineSym s = line_sym(g, pr, b, c);
        const size_t o = (size_t)p * nlines + gl;
        LineTab t;
        t.b = s.Lb; t.c = s.Lc; t.s = cadd(s.Lb, s.Lc);
        t.e = expipi(s.phi / (double)g.na);
        t.q = s.Lb.x * s.Lb.x + s.Lb.y * s.Lb.y + s.Lc.x * s.Lc.x + s.Lc.y * s.Lc.y;
        const double2 d = csub(s.Lb, s.Lc);
        t.d = d.x * d.x + d.y * d.y;
        lt[o] = t;
        const double ph = 2.0 * s.phi / (double)g.na;
        for (int q = 0; q < tpl; ++q) {
            const double2 w = expipi(ph * (double)(q < 16 ? q : 16 * (q - 16)));
            tw64[o * tpl + q] = w;
            tw32[o * tpl + q] = make_float2((float)w.x, (float)w.y);
        }
        const double2 w = expipi(2.0 * (pr.s0 + pr.s1 * (double)c) / (double)g.nb * (double)b);
        mid64[o] = w;
        mid32[o] = make_float2((float)w.x, (float)w.y);
        if (b == 0) outer[(size_t)p * g.nc + c] = expipi(2.0 * pr.r0 * (double)c / (double)g.nc);
    }
}
hipError_t fame_launch_line_tab(const GridDev& g, const ProbDev* prob, LineTab* lt, void* tw64, void* tw32, void* mid64,
                                void* mid32, double2* outer, int nprob, hipStream_t s) {
    hipLaunchKernelGGL(k_line_tab, dim3((g.nb * g.nc + 63) / 64, nprob), dim3(64), 0, s, g, prob, lt, (double2*)tw64, (float2*)tw32,
                       (double2*)mid64, (float2*)mid32, outer);
    return hipGetLastError();
}

/* ------------------------------------------------- one-way plane kernels ---- */
/* The plane halves of Qr and Qrs (FP64): the field enters or leaves in the plane
 * layout, or (General lattices, whose real-space planes of fixed z are the planes
 * of fixed a) straight in the reference's layout, transposed on the way through
 * LDS.  They replace k_mid + k_outer + k_xz_transpose (18 N s of field traffic) and
 * the conversions of the reduced vector (8 N s) by one pass (6 N s): Qrs of
 * a 50 x 42 x 36 grid 59 -> 34 us, residuals of 4 wave vectors x 12 bands on the
 * FCC 64 grid 3.27 -> 1.32 ms.  Bound by the LDS passes and, where a plane is over
 * half a CU's LDS, by one block per CU.  The outer phases come from a table in
 * global memory, so that every grid whose k_plane fits the LDS fits here too  */
namespace fame {

__device__ __forceinline__ void plane_tables(const KPlane& k, double2* Wb, double2* Wc) {
    for (int i = threadIdx.x; i < k.b.ntab; i += blockDim.x) Wb[i] = reinterpret_cast<const double2*>(k.b.W)[i];
    for (int i = threadIdx.x; i < k.c.ntab; i += blockDim.x) Wc[i] = reinterpret_cast<const double2*>(k.c.W)[i];
}

__device__ __forceinline__ double block_sum(double v, double* red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += red[w];
    return s;
}

/* inverse transforms along b and c and the outer twiddle of one plane, then
 *   SYN_FIELD  D/N v back in place (plane layout);
 *   SYN_REF    D/N v into out, reference's layout;
 *   SYN_EPS    D v / (N eps) back in place, with its |.|^2 per block;
 *   SYN_RES    |D/N v - w2 eps E|^2 and |E|^2 per block, nothing stored          */
template <int ENGB, int ENGC, int MODE, int TB>
__global__ void __launch_bounds__(TB) k_syn(KSyn a) {
    constexpr int MAXE = TB == 512 ? 16 : 8;     /* as k_plane */
    typedef double2 T2;
    const KPlane& k = a.k;
    const int npl = 3 * k.g.na;
    const int p = blockIdx.y, pl = xcd_tile();
    if (pl >= npl) return;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ double red[8];
    const int nb = k.b.n, nc = k.c.n, plane = nb * nc, Pb = nb | 1;
    T2* S = reinterpret_cast<T2*>(smem_raw);
    T2* Wb = S + ((nc * Pb + 1) & ~1);
    T2* Wc = Wb + k.b.ntab;
    const T2* D = a.outer + (size_t)p * nc;      /* exp(2 i pi r0 c / nc) */
    plane_tables(k, Wb, Wc);
    const size_t po = (size_t)pl * k.PP;
    T2* F = reinterpret_cast<T2*>(k.f) + (size_t)p * k.fstride + po;
    Hook<double, T2> hk;
    hk.tw = reinterpret_cast<const T2*>(k.tw) + (size_t)p * plane;
    hk.eps = nullptr; hk.ld = nb; hk.pap = false;
    rows_in<double, T2, 4>(S, F, nb, Pb, k.mnb, plane);
    line_transform<double, T2, ENGB, true, MAXE>(S, nc, Pb, 1, k.b, Wb);
    column_transform<double, T2, ENGC, true, MAXE>(S, nb, Pb, k.c, Wc, hk);
    __syncthreads();
    const double invN = 1.0 / (double)k.g.N;
    if constexpr (MODE == SYN_FIELD || MODE == SYN_EPS) {
        const double* ie = reinterpret_cast<const double*>(k.invB) + po;
        double acc = 0.0;
        batched_loop<8>(plane, [&](int i) -> double { return MODE == SYN_EPS ? ie[i] : invN; },
            [&](int i, double e) {
                const int c = udiv(i, k.mnb), b = i - c * nb;
                const T2 v = cscale(cmul(S[c * Pb + b], D[c]), e);
                if (MODE == SYN_EPS) acc += v.x * v.x + v.y * v.y;
                F[i] = v;
            });
        if constexpr (MODE == SYN_EPS) {
            const double s = block_sum(acc, red);
            if (threadIdx.x == 0) a.part[(size_t)p * npl + pl] = s;
        }
    } else {
        /* reference's layout: plane a of component comp at comp N + a plane, c fastest */
        const int comp = pl / k.g.na, ai = pl - comp * k.g.na;
        const size_t ro = (size_t)comp * k.g.N + (size_t)ai * plane;
        if constexpr (MODE == SYN_REF) {
            T2* O = a.out + (size_t)p * a.ostride + ro;
            for (int i = threadIdx.x; i < plane; i += blockDim.x) {
                const int b = udiv(i, k.c.mn), c = i - b * nc;
                O[i] = cscale(cmul(S[c * Pb + b], D[c]), invN);
            }
        } else {
            const T2* E = a.E + (size_t)p * a.ostride + ro;
            const double* ep = a.eps + ro;
            const double w2 = a.w2[(size_t)p * a.w2step];
            double r2 = 0.0, e2 = 0.0;
            struct In { T2 e; double ep; };
            batched_loop<4>(plane, [&](int i) -> In { return In{E[i], ep[i]}; },
                [&](int i, const In& d) {
                    const int b = udiv(i, k.c.mn), c = i - b * nc;
                    const T2 v = cscale(cmul(S[c * Pb + b], D[c]), invN), e = d.e;
                    const double s = w2 * d.ep, rx = v.x - s * e.x, ry = v.y - s * e.y;
                    r2 += rx * rx + ry * ry;
                    e2 += e.x * e.x + e.y * e.y;
                });
            r2 = block_sum(r2, red);
            e2 = block_sum(e2, red);
            if (threadIdx.x == 0) {
                a.part[((size_t)p * npl + pl) * 2] = r2;
                a.part[((size_t)p * npl + pl) * 2 + 1] = e2;
            }
        }
    }
}

/* conj outer twiddle and forward transforms along c and b of one plane, read from
 * `in` (reference's layout, General) or in place, stored in the plane layout  */
template <int ENGB, int ENGC, int TB>
__global__ void __launch_bounds__(TB) k_ana(KSyn a) {
    constexpr int MAXE = TB == 512 ? 16 : 8;
    typedef double2 T2;
    const KPlane& k = a.k;
    const int npl = 3 * k.g.na;
    const int p = blockIdx.y, pl = xcd_tile();
    if (pl >= npl) return;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int nb = k.b.n, nc = k.c.n, plane = nb * nc, Pb = nb | 1;
    T2* S = reinterpret_cast<T2*>(smem_raw);
    T2* Wb = S + ((nc * Pb + 1) & ~1);
    T2* Wc = Wb + k.b.ntab;
    const T2* D = a.outer + (size_t)p * nc;
    plane_tables(k, Wb, Wc);
    T2* F = reinterpret_cast<T2*>(k.f) + (size_t)p * k.fstride + (size_t)pl * k.PP;
    if (a.in) {
        const int comp = pl / k.g.na, ai = pl - comp * k.g.na;
        const T2* I = a.in + (size_t)p * a.ostride + (size_t)comp * k.g.N + (size_t)ai * plane;
        batched_loop<4>(plane, [&](int i) -> T2 { return I[i]; },
            [&](int i, T2 v) {
                const int b = udiv(i, k.c.mn), c = i - b * nc;
                S[c * Pb + b] = cmulc(v, D[c]);
            });
    } else {
        batched_loop<4>(plane, [&](int i) -> T2 { return F[i]; },
            [&](int i, T2 v) {
                const int c = udiv(i, k.mnb), b = i - c * nb;
                S[c * Pb + b] = cmulc(v, D[c]);
            });
    }
    Hook<double, T2> hk;
    hk.tw = reinterpret_cast<const T2*>(k.tw) + (size_t)p * plane;
    hk.eps = nullptr; hk.ld = nb; hk.pap = false;
    column_transform<double, T2, ENGC, false, MAXE>(S, nb, Pb, k.c, Wc, hk);
    line_transform<double, T2, ENGB, false, MAXE>(S, nc, Pb, 1, k.b, Wb);
    __syncthreads();
    rows_out<double, T2>(S, F, nb, Pb, k.mnb, plane);
}

/* the inner axis of the curl-curl operator on the plane layout, in place:
 * conj twiddle, FFT_a, -conj(L) x (L x .) on every mode, IFFT_a, twiddle       */
template <int ENG>
__global__ void __launch_bounds__(FFT_THREADS) k_curl(KLine k) {
    typedef double2 T2;
    const int p = blockIdx.y;
    const int nlines = k.g.nb * k.g.nc, na = k.g.na, L = k.L, P = k.P;
    const int l0 = inner_tile() * L;
    if (l0 >= nlines) return;
    const int nl = min(L, nlines - l0);
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const InnerLds<T2> m(smem_raw, na, k.a.ntab, L, P);
    inner_tables<T2>(k, m, p, l0, nl);
    __syncthreads();
    const double iha2 = 2.0 * k.g.iha;
    const int tpl = inner_tw_per_line(na);
    T2* S = m.S;
    T2* F = reinterpret_cast<T2*>(k.f) + (size_t)p * k.fstride + l0;
    const unsigned PP = (unsigned)k.PP, cs = (unsigned)k.cs;
    struct In { T2 v[3]; };
    batched_loop<2>(L * na,
        [&](int i) -> In {
            const int a = udiv(i, k.mLs), line = i - a * L;
            In d;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                d.v[c] = make_double2(0, 0);
                if (line < nl) d.v[c] = F[c * cs + (unsigned)a * PP + line];
            }
            return d;
        },
        [&](int i, const In& d) {
            const int a = udiv(i, k.mLs), line = i - a * L;
            const T2* t0 = m.tw + line * tpl;
            T2 w = make_double2(1, 0);
            if (line < nl) w = cmul(t0[16 + (a >> 4)], t0[a & 15]);
#pragma unroll
            for (int c = 0; c < 3; ++c) S[(c * L + line) * P + a] = cmulc(d.v[c], w);
        });
    line_transform<double, T2, ENG, false>(S, 3 * L, P, 1, k.a, m.W);
    __syncthreads();
    for (int i = threadIdx.x; i < nl * na; i += blockDim.x) {
        const int line = udiv(i, k.g.m_na), a = i - line * na;
        const LineTab& lt = m.lt[line];
        const double2 e = cmul(m.ea[a], lt.e);
        const double q = e.y * iha2;
        const double2 La = make_double2(-q * e.y, q * e.x);
        double2 l[3];
        if (k.g.general) { l[0] = lt.c; l[1] = lt.b; l[2] = La; }
        else { l[0] = La; l[1] = lt.b; l[2] = lt.c; }
        double2 v[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) v[c] = S[(c * L + line) * P + a];
        const double2 u[3] = {fmas2(cmul(l[1], v[2]), l[2], v[1]), fmas2(cmul(l[2], v[0]), l[0], v[2]),
                              fmas2(cmul(l[0], v[1]), l[1], v[0])};
        const double2 n[3] = {make_double2(-l[0].x, l[0].y), make_double2(-l[1].x, l[1].y), make_double2(-l[2].x, l[2].y)};
        S[(0 * L + line) * P + a] = fmas2(cmul(n[1], u[2]), n[2], u[1]);
        S[(1 * L + line) * P + a] = fmas2(cmul(n[2], u[0]), n[0], u[2]);
        S[(2 * L + line) * P + a] = fmas2(cmul(n[0], u[1]), n[1], u[0]);
    }
    line_transform<double, T2, ENG, true>(S, 3 * L, P, 1, k.a, m.W);
    __syncthreads();
    for (int i = threadIdx.x; i < L * na; i += blockDim.x) {
        const int a = udiv(i, k.mLs), line = i - a * L;
        if (line >= nl) continue;
        const T2* t0 = m.tw + line * tpl;
        const T2 w = cmul(t0[16 + (a >> 4)], t0[a & 15]);
#pragma unroll
        for (int c = 0; c < 3; ++c) F[c * cs + (unsigned)a * PP + line] = cmul(S[(c * L + line) * P + a], w);
    }
}

/* tiled transpose of a batch of matrices, scaled per problem */
__global__ void __launch_bounds__(256) k_transpose(const double2* __restrict__ in, double2* __restrict__ out, int rows, int cols,
                                                   int ip, int op, size_t ib, size_t ob, size_t is, size_t os, const double* scale2) {
    __shared__ double2 tile[32][33];
    const int p = blockIdx.z, m = blockIdx.y, tc = (cols + 31) >> 5;
    const double s = scale2 ? sqrt(scale2[p]) : 1.0;
    const double2* I = in + (size_t)p * is + (size_t)m * ib;
    double2* O = out + (size_t)p * os + (size_t)m * ob;
    const int r0 = (int)(blockIdx.x / tc) * 32, c0 = (int)(blockIdx.x % tc) * 32, lx = threadIdx.x & 31, ly = threadIdx.x >> 5;
    for (int r = ly; r < 32; r += 8)
        if (r0 + r < rows && c0 + lx < cols) tile[r][lx] = I[(size_t)(r0 + r) * ip + c0 + lx];
    __syncthreads();
    for (int c = ly; c < 32; c += 8)
        if (c0 + c < cols && r0 + lx < rows) O[(size_t)(c0 + c) * op + r0 + lx] = cscale(tile[lx][c], s);
}

/* Simple grids: F [component][a][PP] against E and eps [component][c b][a]; one
 * block sums a strided set of 32 x 32 tiles */
__global__ void __launch_bounds__(256) k_resid_simple(const double2* __restrict__ F, const double2* __restrict__ E,
                                                      const double* __restrict__ eps, const double* w2, int w2step,
                                                      double* part, int na, int nl, int PP, size_t fs, size_t es) {
    __shared__ double2 tile[32][33];
    __shared__ double red[8];
    const int p = blockIdx.y, ta = (na + 31) >> 5, tl = (nl + 31) >> 5;
    const int lx = threadIdx.x & 31, ly = threadIdx.x >> 5;
    const double om = w2[(size_t)p * w2step];
    double r2 = 0.0, e2 = 0.0;
    for (int t = blockIdx.x; t < 3 * ta * tl; t += gridDim.x) {
        const int comp = t / (ta * tl), u = t - comp * ta * tl, a0 = (u / tl) * 32, l0 = (u % tl) * 32;
        const double2* Fc = F + (size_t)p * fs + (size_t)comp * na * PP;
        const double2* Ec = E + (size_t)p * es + (size_t)comp * na * nl;
        const double* ec = eps + (size_t)comp * na * nl;
        __syncthreads();
        for (int r = ly; r < 32; r += 8)
            if (a0 + r < na && l0 + lx < nl) tile[r][lx] = Fc[(size_t)(a0 + r) * PP + l0 + lx];
        __syncthreads();
        for (int r = ly; r < 32; r += 8)
            if (l0 + r < nl && a0 + lx < na) {
                const size_t o = (size_t)(l0 + r) * na + a0 + lx;
                const double2 f = tile[lx][r], e = Ec[o];
                const double s = om * ec[o], rx = f.x - s * e.x, ry = f.y - s * e.y;
                r2 += rx * rx + ry * ry;
                e2 += e.x * e.x + e.y * e.y;
            }
    }
    r2 = block_sum(r2, red);
    e2 = block_sum(e2, red);
    if (threadIdx.x == 0) {
        part[((size_t)p * gridDim.x + blockIdx.x) * 2] = r2;
        part[((size_t)p * gridDim.x + blockIdx.x) * 2 + 1] = e2;
    }
}

/* the permittivity in the kernels' layouts.  General: the reference's [z][y][x] is
 * the axis passes' [x][y][z] (c, b, a) with x and z exchanged; both that and the
 * plane layout are written from one read of a 32 x 32 (x, z) or (c b, a) tile   */
__global__ void __launch_bounds__(256) k_eps(GridDev g, const double* __restrict__ eps, double* eps_int, double* ib64,
                                             float* ib32, double* p64, float* p32, int PP) {
    __shared__ double tile[32][33];
    const int na = g.na, nb = g.nb, nc = g.nc, nl = nb * nc;
    const size_t N = (size_t)g.N;
    const double sc = 1.0 / (double)g.N;
    const int lx = threadIdx.x & 31, ly = threadIdx.x >> 5;
    const int comp = blockIdx.z;
    auto put_int = [&](size_t o, double v) {
        const double i = 1.0 / v;
        eps_int[comp * N + o] = v;
        ib64[comp * N + o] = i;
        ib32[comp * N + o] = (float)i;
    };
    auto put_plane = [&](size_t o, double v) {
        if (!p64) return;
        const double i = (1.0 / v) * sc;
        p64[(size_t)comp * na * PP + o] = i;
        p32[(size_t)comp * na * PP + o] = (float)i;
    };
    if (g.general) {
        /* tile over (c = x, a = z) for one b = y */
        const int tc = (nc + 31) >> 5, b = blockIdx.y, c0 = (blockIdx.x % tc) * 32, a0 = (blockIdx.x / tc) * 32;
        for (int r = ly; r < 32; r += 8)
            if (a0 + r < na && c0 + lx < nc) {
                const double v = eps[comp * N + ((size_t)(a0 + r) * nb + b) * nc + c0 + lx];
                tile[r][lx] = v;
                put_plane((size_t)(a0 + r) * PP + (size_t)(c0 + lx) * nb + b, v);
            }
        __syncthreads();
        for (int r = ly; r < 32; r += 8)
            if (c0 + r < nc && a0 + lx < na) put_int(((size_t)(c0 + r) * nb + b) * na + a0 + lx, tile[lx][r]);
    } else {
        /* tile over (line, a): the reference's layout is the axis passes' */
        const int ta = (na + 31) >> 5, l0 = (blockIdx.x / ta) * 32, a0 = (blockIdx.x % ta) * 32;
        for (int r = ly; r < 32; r += 8)
            if (l0 + r < nl && a0 + lx < na) {
                const size_t o = (size_t)(l0 + r) * na + a0 + lx;
                const double v = eps[comp * N + o];
                tile[r][lx] = v;
                put_int(o, v);
            }
        __syncthreads();
        for (int r = ly; r < 32; r += 8)
            if (a0 + r < na && l0 + lx < nl) put_plane((size_t)(a0 + r) * PP + l0 + lx, tile[lx][r]);
    }
}

}  // namespace fame

template <int EB, int EC, int TB>
static const void* syn_fn(int mode) {
    switch (mode) {
        case SYN_FIELD: return (const void*)k_syn<EB, EC, SYN_FIELD, TB>;
        case SYN_REF: return (const void*)k_syn<EB, EC, SYN_REF, TB>;
        case SYN_EPS: return (const void*)k_syn<EB, EC, SYN_EPS, TB>;
        case SYN_RES: return (const void*)k_syn<EB, EC, SYN_RES, TB>;
        default: return (const void*)k_ana<EB, EC, TB>;
    }
}
template <int TB>
static const void* syn_fn(int eb, int ec, int mode) {
    if (eb == ENG_MFMA) return ec == ENG_MFMA ? syn_fn<ENG_MFMA, ENG_MFMA, TB>(mode) : syn_fn<ENG_MFMA, ENG_STOCKHAM, TB>(mode);
    return ec == ENG_MFMA ? syn_fn<ENG_STOCKHAM, ENG_MFMA, TB>(mode) : syn_fn<ENG_STOCKHAM, ENG_STOCKHAM, TB>(mode);
}
hipError_t fame_prepare_syn(int eb, int ec) {
    for (int m = 0; m < 10; ++m) {
        const hipError_t e = hipFuncSetAttribute(m < 5 ? syn_fn<512>(eb, ec, m) : syn_fn<1024>(eb, ec, m - 5),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 256);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
/* the wide variant (k.wide) where k_plane starts with it; its 256 registers leave a
 * CU 512 threads, in two blocks where two planes fit and there are that many.
 * The narrow one's two blocks of 512 threads: residuals of 4 wave vectors x 12
 * bands, FCC 64, 1.32 ms against 1.54 with the wide one                       */
static hipError_t launch_syn(const KSyn& k, int mode, int nprob, hipStream_t s) {
    KSyn q = k;
    void* arg[] = {&q};
    const size_t lds = fame_plane_lds(k.k.b.n, k.k.c.n, k.k.b.ntab + k.k.c.ntab, 8);
    const int nt = lds <= FAME_LDS_HALF && k.k.wide && 3 * k.k.g.na * (k.batch ? k.batch : nprob) > 512 ? 256 : 512;
    return hipLaunchKernel(k.k.wide ? syn_fn<512>(k.k.b.eng, k.k.c.eng, mode) : syn_fn<1024>(k.k.b.eng, k.k.c.eng, mode),
                           dim3(xcd_round(3 * k.k.g.na), nprob), dim3(nt), arg, lds, s);
}
hipError_t fame_launch_syn(const KSyn& k, int mode, int nprob, hipStream_t s) { return launch_syn(k, mode, nprob, s); }
hipError_t fame_launch_ana(const KSyn& k, int nprob, hipStream_t s) { return launch_syn(k, 4, nprob, s); }
hipError_t fame_launch_curl(const KLine& k, int nprob, hipStream_t s) {
    KLine q = k;
    void* arg[] = {&q};
    return hipLaunchKernel(k.a.eng == ENG_MFMA ? (const void*)k_curl<ENG_MFMA> : (const void*)k_curl<ENG_STOCKHAM>,
                           dim3(xcd_round((k.g.nb * k.g.nc + k.L - 1) / k.L), nprob), dim3(FFT_THREADS), arg,
                           fame_line_lds2(k.g.na, k.a.ntab, k.L, k.P, 8), s);
}
hipError_t fame_launch_transpose(const double2* in, double2* out, int rows, int cols, int ip, int op, size_t ib, size_t ob,
                                 int batch, size_t is, size_t os, const double* scale2, int nprob, hipStream_t s) {
    hipLaunchKernelGGL(k_transpose, dim3(((cols + 31) / 32) * ((rows + 31) / 32), batch, nprob), dim3(256), 0, s, in, out, rows, cols,
                       ip, op, ib, ob, is, os, scale2);
    return hipGetLastError();
}
hipError_t fame_launch_resid_simple(const double2* F, const double2* E, const double* eps, const double* w2, int w2step,
                                    double* part, int nblk, int na, int nl, int PP, size_t fs, size_t es, int nprob,
                                    hipStream_t s) {
    hipLaunchKernelGGL(k_resid_simple, dim3(nblk, nprob), dim3(256), 0, s, F, E, eps, w2, w2step, part, na, nl, PP, fs, es);
    return hipGetLastError();
}
hipError_t fame_launch_eps(const GridDev& g, const double* eps, double* eps_int, double* ib64, float* ib32, double* p64,
                           float* p32, int PP, hipStream_t s) {
    const int ta = (g.na + 31) / 32, tc = (g.nc + 31) / 32, tl = (g.nb * g.nc + 31) / 32;
    const dim3 grid = g.general ? dim3(tc * ta, g.nb, 3) : dim3(tl * ta, 1, 3);
    hipLaunchKernelGGL(k_eps, grid, dim3(256), 0, s, g, eps, eps_int, ib64, ib32, p64, p32, PP);
    return hipGetLastError();
}
