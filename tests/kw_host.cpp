// Host build of the kinematic-wave solve of the kernels (kw_prepare, kw_begin, kw_end) beside the
// reference's loop written out, for CPU tests. Built by the tests with g++ -ffp-contract=off.
#include "wfh_physics.h"

using namespace wfh;

// rows of 6: q_in, q_prev, q_lat, alpha, dt, dx. out rows of 10: q and flow area of the solve, of the
// loop; 1 where the straight updates take the case; of such a case the largest u, the largest
// f(u) + C and f'(u) and the smallest f'(u) of its updates; and of the four updates from every u whose
// f(u) + C is above 1024 |C| + 1e-8 the largest fall of f + C in one update.
extern "C" void host_kw(const double* in, double* out, long n) {
    for (long i = 0; i < n; ++i) {
        const double *r = in + 6 * i, q_in = r[0], q_prev = r[1], q_lat = r[2], alpha = r[3], dt = r[4], dx = r[5];
        double* o = out + 10 * i;
        const KwPrep p = kw_prepare(q_prev, q_lat, alpha, dt, dx);
        kw_solve(q_in, p, alpha, o[0], o[1]);
        o[4] = p.fast;
        o[5] = o[6] = o[7] = o[9] = 0.0;
        o[8] = INFINITY;
        if (q_in + q_prev + q_lat == 0.0) {
            o[2] = o[3] = 0.0;
            o[4] = 0.0;
            continue;
        }
        const double dt_dx = dt / dx, C = dt_dx * q_in + p.a_u3 + dt * q_lat, far = 1024.0 * wfh_fabs(C) + 1e-8;
        if (!(wfh_fabs(C) <= 0x1p60)) o[4] = 0.0;
        double u = p.u_prev > 0.0 ? p.u_prev : wfh_cbrt(C / alpha), g_before = 0.0;
        int falling = 0;
        for (int k = 0; k < 3000; ++k) {
            double g, df;
            kw_terms(u, dt_dx, alpha, g, df);
            const double f = g - C;
            if (falling > 0 && g_before / g > o[9]) o[9] = g_before / g;
            falling = g > far && u > 0.0 && u < 0x1p100 ? 4 : falling - 1;
            g_before = g;
            if (o[4] != 0.0) {
                o[5] = wfh_fabs(u) > o[5] || u != u ? wfh_fabs(u) : o[5];
                o[6] = wfh_fabs(g) > o[6] || g != g ? wfh_fabs(g) : o[6];
                o[7] = df > o[7] || df != df ? df : o[7];
                o[8] = df < o[8] ? df : o[8];
            }
            if (wfh_fabs(f) <= 1.0e-12) break;
            u = u - f / df;
            if (!(u > 0.0)) u = WFH_KIN_WAVE_MIN_FLOW_QROOT;
        }
        u = wfh_max(u, WFH_KIN_WAVE_MIN_FLOW_QROOT);
        const double u3 = u * u * u;
        o[2] = u3 * u * u;
        o[3] = alpha * u3;
    }
}
