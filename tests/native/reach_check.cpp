// Brute-force check of ft_box_meets and kp_row_range (gt_ftpatch.h): no box or
// row that holds a sample inside a support may be dropped.
//   reach_check ATOMS GRID
// prints: boxes holding a sample, boxes kept, boxes, rows holding a sample, rows kept, rows
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "gt_ftpatch.h"

int main(int argc, char **argv)
{
    const int atoms = std::atoi(argv[1]), n = std::atoi(argv[2]);
    std::mt19937 rng(5);
    std::uniform_real_distribution<float> uni(0.02f, 0.1f);
    std::normal_distribution<float> nor(0.0f, 1.0f);
    std::vector<float> k(n);
    for (int i = 0; i < n; i++) k[i] = (float)(i - n / 2);
    const float sc = 0.84932180f, cut = 30.0f * sc * sc;
    long held = 0, kept = 0, boxes = 0, rheld = 0, rkept = 0, rows = 0;
    for (int a = 0; a < atoms; a++) {
        gt::FtL r{};
        const bool iso = a % 5 == 0;
        const float d = uni(rng);
        for (int c = 0; c < 3; c++) r.u[c] = sc * 6.2831853f * (iso ? d : uni(rng));
        if (!iso)
            for (int c = 3; c < 6; c++) r.u[c] = 0.4f * r.u[c - 3] * nor(rng);
        auto q = [&](float k0, float k1, float k2) {
            const float v0 = r.u[0] * k0, v1 = r.u[1] * k1 + r.u[3] * k0, v2 = r.u[4] * k1 + r.u[5] * k0 + r.u[2] * k2;
            return v0 * v0 + v1 * v1 + v2 * v2;
        };
        const int sizes[2][3] = {{2, 8, 8}, {8, 16, 8}};
        for (const auto &z : sizes)
            for (int b0 = 0; b0 < n; b0 += z[0])
                for (int b1 = 0; b1 < n; b1 += z[1])
                    for (int b2 = 0; b2 < n; b2 += z[2]) {
                        const int lo[3] = {b0, b1, b2};
                        float m[3], x[3];
                        int hi[3];
                        for (int c = 0; c < 3; c++) {
                            hi[c] = std::min(lo[c] + z[c], n) - 1;
                            m[c] = 0.5f * (k[lo[c]] + k[hi[c]]);
                            x[c] = 0.5f * (k[hi[c]] - k[lo[c]]);
                        }
                        const bool keep = gt::ft_box_meets(r, m[0], m[1], m[2], x[0], x[1], x[2], std::sqrt(cut));
                        bool in = false;
                        for (int i = lo[0]; i <= hi[0] && !in; i++)
                            for (int j = lo[1]; j <= hi[1] && !in; j++)
                                for (int l = lo[2]; l <= hi[2] && !in; l++) in = q(k[i], k[j], k[l]) < cut;
                        boxes++;
                        held += in;
                        kept += keep;
                        if (in && !keep) return 1;
                    }
        // the plane k2 = 0 as an ellipse {q0 x^2 + q1 x y + q2 y^2 >= -cut}
        const float q0 = -(r.u[0] * r.u[0] + r.u[3] * r.u[3] + r.u[5] * r.u[5]);
        const float q1 = -2.0f * (r.u[1] * r.u[3] + r.u[4] * r.u[5]), q2 = -(r.u[1] * r.u[1] + r.u[4] * r.u[4]);
        for (int w = 1; w <= 32; w += 31)
            for (int c = 0; c < n; c += w) {
                const int ce = std::min(c + w, n) - 1;
                float xlo, xhi;
                gt::kp_row_range(q0, q1, q2, -cut, k[c], k[ce], xlo, xhi);
                for (int i = 0; i < n; i++) {
                    bool in = false;
                    for (int j = c; j <= ce && !in; j++)
                        in = q0 * k[i] * k[i] + q1 * k[i] * k[j] + q2 * k[j] * k[j] > -cut;
                    const bool keep = k[i] >= xlo && k[i] <= xhi;
                    rows++;
                    rheld += in;
                    rkept += keep;
                    if (in && !keep) return 2;
                }
            }
    }
    std::printf("%ld %ld %ld %ld %ld %ld\n", held, kept, boxes, rheld, rkept, rows);
    return 0;
}
