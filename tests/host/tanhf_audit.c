/* tanhf_audit.c - the device's float tanh (k3g_expf.h, compiled here for the host) against the C
 * library's double tanh rounded to float, on every 2^-8-th of the 2^32 float inputs and every
 * input whose magnitude lies in [1/64, 1/32), [0.5, 1) and [8, 10): NaN for NaN, the sign
 * kept, no difference above one float step, and the number of differing results. */
#include <math.h>
#include <stdio.h>
#include <string.h>

#include "k3g_expf.h"

int main(void)
{
    long long n = 0, diff = 0, bad = 0;
#pragma omp parallel for reduction(+ : n, diff, bad) schedule(static, 1 << 16)
    for (long long i = 0; i < (1ll << 32); ++i) {
        const unsigned u = (unsigned)i, m = u & 0x7fffffffu;
        float x;
        memcpy(&x, &u, 4);
        const float ax = fabsf(x);
        const int full = (ax >= 1.0f / 64 && ax < 1.0f / 32) || (ax >= 0.5f && ax < 1.0f) ||
                         (ax >= 8.0f && ax < 10.0f);
        if (!full && (u * 2654435761u) >> 24) continue;
        ++n;
        const float a = (float)tanh((double)x), b = k3x_tanhf(x);
        if (m > 0x7f800000u) {
            if (!isnan(b)) ++bad;
            continue;
        }
        int ua, ub;
        memcpy(&ua, &a, 4);
        memcpy(&ub, &b, 4);
        if (ua == ub) continue;
        ++diff;
        if ((ua < 0) != (ub < 0) || ua - ub > 1 || ub - ua > 1) ++bad;
    }
    printf("inputs %lld differing %lld bad %lld\n", n, diff, bad);
    return bad ? 1 : 0;
}
