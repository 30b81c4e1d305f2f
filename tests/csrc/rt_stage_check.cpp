/* The run-time Stockham stages of the HIP pressure kernels (wf_rt_stage and
 * WfDiv in wildfires_amd/csrc/hip/wf_fft.h) for the CPU check in
 * tests/test_pressure_passes.py; test code only. */
#include <cmath>
#include <cstddef>
#include <vector>

#include "../../wildfires_amd/csrc/hip/wf_fft.h"

/* The host factoriser's radices: 4s, then 2s, then odd primes. */
static std::vector<int> factor(int n) {
    std::vector<int> rad;
    while (n % 4 == 0) { rad.push_back(4); n /= 4; }
    while (n % 2 == 0) { rad.push_back(2); n /= 2; }
    for (int p = 3; n > 1; p += 2)
        while (n % p == 0) { rad.push_back(p); n /= p; }
    return rad;
}

/* Every stage of length n over nseq sequences by nt threads against
 * wf_stockham_output: the number of values that differ or were not written. */
extern "C" long rt_stages_differ(int n, int nseq, int nt) {
    std::vector<wfc> tw(n), a((size_t)n * nseq), b(a.size());
    for (int e = 0; e < n; e++) {
        const double ang = 2.0 * 3.14159265358979323846 * e / n;
        tw[e].re = std::cos(ang);
        tw[e].im = -std::sin(ang);
    }
    tw[0].im = 0.0;
    for (size_t t = 0; t < a.size(); t++) {
        a[t].re = std::sin(1.0 + 0.7 * (double)t);
        a[t].im = std::cos(2.0 + 1.3 * (double)t);
    }
    long bad = 0;
    int Ns = 1;
    for (int R : factor(n)) {
        for (wfc &v : b) v.re = v.im = NAN;
        for (int tid = 0; tid < nt; tid++) wf_rt_stage(a.data(), b.data(), n, nseq, R, Ns, tw.data(), tid, nt);
        for (int s = 0; s < nseq; s++)
            for (int o = 0; o < n; o++) {
                const wfc want = wf_stockham_output(a.data() + (size_t)s * n, n, R, Ns, tw.data(), o);
                const wfc got = b[(size_t)s * n + o];
                bad += !(got.re == want.re && got.im == want.im);
            }
        a.swap(b);
        Ns *= R;
    }
    return bad;
}

/* quotients that differ, over the range stated at WfDiv */
extern "C" long quotients_differ() {
    long bad = 0;
    for (int d = 1; d <= 1024; d++) {
        const WfDiv by(d);
        for (int t = 0; t < 65536; t++) bad += by(t) != t / d;
    }
    return bad;
}
