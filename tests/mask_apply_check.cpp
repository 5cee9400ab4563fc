// Rows applied from neighbourhood masks (mask_aniso_apply) against the assembled
// rows of the oracle times the same values, for the CPU test of the same name.
#include <cstdio>
#include <cstdlib>
#include <cmath>
#include <vector>
#include "aniso_row.h"
extern "C" void orc_assemble_aniso(int nx, int ny, int nz, double dx, double dy, double dz, double alpha, const double *tensor6,
                                   const uint8_t *active, double *out);
template <typename T> static double worst(int trial) {
    const int nx = 9 + trial, ny = 7 + trial % 3, nz = 5 + trial % 2;
    const int64_t n = (int64_t)nx * ny * nz;
    const double dx = 100, dy = 100 + 10 * (trial % 2), dz = 100 - 5 * (trial % 3), alpha = 0.07;
    std::vector<double> lt(nz * 6), t6(n * 6), u(n);
    std::vector<uint8_t> act(n);
    srand(trial + 1);
    for(int z = 0; z < nz; z++) {
        const double th = -1.0 + 2.0 * z / (nz - 1), c = cos(th), s = sin(th), sl = 0.00024, st = 0.000045;
        const double t[6] = {sl * c * c + st * s * s, sl * s * s + st * c * c, st, (sl - st) * c * s, trial % 2 ? 1e-5 * (z + 1) : 0.0, trial % 2 ? -2e-5 * z : 0.0};
        for(int k = 0; k < 6; k++) lt[z * 6 + k] = t[k];
    }
    for(int64_t i = 0; i < n; i++) {
        for(int k = 0; k < 6; k++) t6[i * 6 + k] = lt[(i / (nx * ny)) * 6 + k];
        act[i] = (rand() % 100) >= 15 * (trial % 4) ? 1 : 0;
        u[i] = 2.0 * rand() / RAND_MAX - 1.0;
    }
    std::vector<double> coef(n * 27);
    orc_assemble_aniso(nx, ny, nz, dx, dy, dz, alpha, t6.data(), act.data(), coef.data());
    double far = 0.0;
    for(int64_t c = 0; c < n; c++) {
        const int x = c % nx, y = (c / nx) % ny, z = c / (nx * ny);
        uint32_t m = 0;
        T v[27];
        double want = 0.0;
        for(int k = 0; k < 27; k++) {
            const int xx = x + k % 3 - 1, yy = y + (k / 3) % 3 - 1, zz = z + k / 9 - 1;
            v[k] = T(0);
            if(xx < 0 || xx >= nx || yy < 0 || yy >= ny || zz < 0 || zz >= nz) continue;
            const int64_t j = xx + (int64_t)nx * (yy + (int64_t)ny * zz);
            v[k] = (T)u[j];  // (also of cells that are not active: their values must not matter)
            want += coef[c * 27 + k] * (double)v[k];
            if(act[c] && act[j]) m |= 1u << k;
        }
        const double *l3[3];
        for(int l = 0; l < 3; l++) l3[l] = &lt[(z - 1 + l < 0 ? 0 : (z - 1 + l >= nz ? nz - 1 : z - 1 + l)) * 6];
        double tab[mono::kMaskTable];
        mono::mask_layer_table(l3, dx, dy, dz, tab);
        T xt[mono::kMaskTable], w[4];
        for(int k = 0; k < mono::kMaskTable; k++) xt[k] = (T)tab[k];
        for(int k = 0; k < 4; k++) w[k] = xt[mono::kNormal + k];
        double dg = 0.0;
        const double got = (double)mono::mask_aniso_apply<T>(m, w, (T)alpha, xt, [&](int k) { return v[k]; }, &dg);
        const double d = coef[c * 27 + 13] != 0.0 ? coef[c * 27 + 13] : alpha;
        far = fmax(far, fabs(got - want) / d);
        far = fmax(far, fabs(dg - coef[c * 27 + 13]) / d);
    }
    return far;
}
// Bounds: a product is a sum of some 60 terms, each a weight of at most the
// diagonal times a difference of values below 1, so some 30 roundings of about
// the diagonal: 1e-14 in FP64, 4e-6 in FP32.
int main() {
    int bad = 0;
    for(int trial = 0; trial < 8; trial++) {
        const double d = worst<double>(trial), s = worst<float>(trial);
        printf("trial %d: fp64 %.2e, fp32 %.2e of the diagonal\n", trial, d, s);
        bad += !(d <= 1e-14) + !(s <= 4e-6);
    }
    return bad;
}
