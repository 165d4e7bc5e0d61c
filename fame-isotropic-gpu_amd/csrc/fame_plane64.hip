/* fame_plane64.hip -- FP64 instances of the plane kernels (fame_plane.hpp), and
 * the tables of a wave vector that both precisions read */
#include "fame_plane.hpp"

using namespace fame;

hipError_t fame_launch_line64(const KLine& k, int expand, int mode, int nprob, hipStream_t s) { return launch_line<double>(k, expand, mode, nprob, s); }
hipError_t fame_launch_plane64(const KPlane& k, int nprob, hipStream_t s) { return launch_plane<double>(k, nprob, s); }
hipError_t fame_prepare_plane64(int eb, int ec, size_t lds) { return prepare_plane<double>(eb, ec, lds); }

/* per line (b, c) of every problem: its symbols and inner-axis phase, the inner
 * twiddle factors in both precisions, and the middle twiddles of its nb entries'
 * plane (entry gl itself: exp(2 pi i (s0 + s1 c) b / nb))                    */
__global__ void k_line_tab(GridDev g, const ProbDev* prob, LineTab* lt, double2* tw64, float2* tw32, double2* mid64,
                           float2* mid32) {
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
    }
}
hipError_t fame_launch_line_tab(const GridDev& g, const ProbDev* prob, LineTab* lt, void* tw64, void* tw32, void* mid64,
                                void* mid32, int nprob, hipStream_t s) {
    hipLaunchKernelGGL(k_line_tab, dim3((g.nb * g.nc + 63) / 64, nprob), dim3(64), 0, s, g, prob, lt, (double2*)tw64, (float2*)tw32,
                       (double2*)mid64, (float2*)mid32);
    return hipGetLastError();
}
