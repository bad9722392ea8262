// Plans of products of value and residual rows, asked on the host: what plan_short_pair says has to be something that launch_short_pair takes.
#include "gemm.h"
#include <stdio.h>

using namespace lmhip;

extern "C" void hip_gemm_force_large_m(int policy);

int main()
{
    const int rows[] = {1, 5, 16, 31, 32, 33, 64, 100, 250, 497, 500, 511, 512, 513, 600, 1000, 1024};
    const int shapes[][2] = {{6176, 2560}, {2560, 4096}, {19456, 2560}, {2560, 9728}, {1568, 1152}, {13824, 1152}, {1152, 6912}, {4928, 256}, {260, 416}, {151936, 2560}, {60, 64}};
    long asked = 0, big = 0, bad = 0;
    for (int policy : {0, 1, -1, 2}) {
        hip_gemm_force_large_m(policy);
        for (const auto &sh : shapes)
            for (int M : rows)
                for (int fmt : {0, 1, 2}) {
                    const int N = sh[0], K = sh[1], Kb = tiled_kb(K);
                    const ShortPlan p = plan_short_pair(M, N, K, 0, fmt);
                    asked++;
                    const bool pair = p.big && !(fmt != 0 && large_m_unpacks_q8());      // (tiles that stay quantised: not the pair kernel's)
                    // residual rows in a row block of their own where the pair kernel reads them, else no row between them and the values
                    bool ok = p.lo == (pair ? (M + 31) / 32 * 32 : M);
                    if (pair) {
                        big++;
                        ok = ok && p.steps >= 1;
                    }
                    if (pair && ok) {
                        const PairWalk w{p.steps, Kb};
                        const int blocks = (N + 255) / 256, teams = (blocks * Kb + p.steps - 1) / p.steps;
                        ok = p.chunks == w.planes();
                        for (int b = 0; b < blocks && ok; b++) ok = w.count(b * 256) >= 1 && w.count(b * 256) <= p.chunks && w.first(b) + w.count(b * 256) <= teams;
                    }
                    if (!ok && bad++ < 10) printf("FAIL policy %d fmt %d M %d N %d K %d: big %d lo %d steps %d planes %d\n", policy, fmt, M, N, K, p.big, p.lo, p.steps, p.chunks);
                }
    }
    printf("asked %ld big %ld bad %ld\n", asked, big, bad);
    return bad != 0 || big == 0;
}
