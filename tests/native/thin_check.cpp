// Brute-force check of the culls of the Fourier sample planes (kp_thin,
// kp_row_range, gt_ftpatch.h; support_meets_rect, gt_pixel.h) on long slanted
// ellipses: no row or 16 x 32 rectangle of samples may be dropped that holds a
// sample whose exponent, as the kernel forms it, passes the cut.
//   thin_check RATIO ELLIPSES
// prints: samples inside, rows holding one, rows kept, rows
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>

#include "gt_ftpatch.h"
#include "gt_pixel.h"

int main(int argc, char **argv)
{
    const double ratio = std::atof(argv[1]);
    const int ellipses = std::atoi(argv[2]);
    std::mt19937 rng(7);
    std::uniform_real_distribution<double> uni(0.0, 1.0);
    const float cut = -15.0f * 1.44269504f;  // |U^T k|^2 < 30
    constexpr int n = 192, R = 16, C = 32;
    long inside = 0, held = 0, kept = 0, rows = 0;
    for (int t = 0; t < ellipses; t++) {
        // long half-axis of 20 to 80 samples, about the diagonal or at any angle
        const double th = t % 2 ? 2 * M_PI * uni(rng) : M_PI / 4 + 0.1 * (uni(rng) - 0.5);
        const double l0 = std::sqrt(30.0) / (20 + 60 * uni(rng)), l1 = l0 * ratio, shift = uni(rng);
        const double c = std::cos(th), s = std::sin(th), f = -0.5 * 1.4426950408889634;
        const float q0 = (float)(f * (l0 * l0 * c * c + l1 * l1 * s * s));
        const float q1 = (float)(2 * f * (l0 * l0 - l1 * l1) * c * s);
        const float q2 = (float)(f * (l0 * l0 * s * s + l1 * l1 * c * c));
        float k[n];
        for (int i = 0; i < n; i++) k[i] = (float)(i - n / 2 + shift);
        for (int a = 0; a < n; a += R)
            for (int b = 0; b < n; b += C) {
                const bool meets = gt::kp_thin(q0, q1, q2) ||
                                   gt::support_meets_rect(make_float4(0.0f, q0, q1, q2), make_float4(0.0f, 0.0f, 0.0f, 0.0f),
                                                          k[a], k[a + R - 1], k[b], k[b + C - 1], cut);
                float xlo, xhi;
                gt::kp_row_range(q0, q1, q2, cut, k[b], k[b + C - 1], xlo, xhi);
                for (int i = a; i < a + R; i++) {
                    bool in = false;
                    for (int j = b; j < b + C; j++) {
                        const float e = fmaf(fmaf(q0, k[i], q1 * k[j]), k[i], q2 * (k[j] * k[j]));
                        if (!(e > cut)) continue;
                        in = true;
                        inside++;
                    }
                    const bool keep = meets && k[i] >= xlo && k[i] <= xhi;
                    rows++;
                    held += in;
                    kept += keep;
                    if (in && !keep) return 1;
                }
            }
    }
    std::printf("%ld %ld %ld %ld\n", inside, held, kept, rows);
    return 0;
}
