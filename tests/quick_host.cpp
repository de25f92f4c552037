// Host build of the prepared subsurface solve (ssf_quick_prepare / ssf_quick_solve) beside the solve
// it stands for (kinematic_wave_ssf), for CPU tests. Built by the tests with g++ -ffp-contract=off.
#include "wfh_physics.h"

using namespace wfh;

// rows of 16: q_in, q_prev, zi_prev, q_net, slope, sy, d, dt, dx, dw, q_max, kh0, f, z_exp, theta_e, seed
// for the layers' water; out rows of 9: taken by the prepared solve (0/1), then q, zi, exfiltration
// and net flux of it, then those four of kinematic_wave_ssf
extern "C" void host_ssf_pair(const double* in, double* out, long n) {
    const double cfg_thick[4] = {0.1, 0.3, 0.8, NaN_};
    const double cfg_cum[5] = {0.0, 0.1, 0.1 + 0.3, 0.1 + 0.3 + 0.8, NaN_};
    for (long i = 0; i < n; ++i) {
        const double* r = in + 16 * i;
        double* o = out + 9 * i;
        Column<4> col;
        soil_layers<4>(r[6], cfg_cum, cfg_thick, col.act, col.cum);
        col.zi = r[2];
        col.n_unsat = set_layerthickness<4>(col.zi, col.cum, col.act, col.thick);
        col.theta_e = r[14];
        col.theta_fc_r = 0.5 * r[14];
        for (int k = 0; k < 4; ++k) {
            double w = r[15] * (k + 1.0);  // a fraction of the layer's pore space, 1 among them
            w = w - (double)(long)w;
            if (w > 0.9) w = 1.0;
            col.ustore[k] = k < col.n_unsat ? w * col.thick[k] * col.theta_e : 0.0;
        }
        const SsfPrep pp = ssf_prepare(r[1], r[2], r[4], r[5], r[7], r[8], r[11], r[12], r[13]);
        const SsfQuick qk = ssf_quick_prepare<4>(r[1], r[2], r[3], r[5], r[6], r[7], r[8], r[9], r[10], pp, col);
        bool deferred;
        o[0] = ssf_quick_solve(r[0], r[1], r[2], r[3], r[5], r[6], r[7], pp, qk, o[1], o[2], o[3], o[4], deferred);
        const bool d2 = kinematic_wave_ssf<4>(r[0], r[1], r[2], r[3], r[4], r[5], r[6], r[7], r[8], r[9], r[10], r[11],
                                              r[12], r[13], pp, col, true, o[5], o[6], o[7], o[8]);
        if (o[0] != 0.0 && d2 != deferred) o[0] = -1.0;
    }
}

// in-range quotients a / b through a reciprocal formed beforehand
extern "C" void host_div(const double* a, const double* b, double* out, long n) {
    for (long i = 0; i < n; ++i) out[i] = wfh_div_by(a[i], b[i], wfh_rcp(b[i]));
}
