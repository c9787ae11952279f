// Packed image vectors (ann_amd/csrc/common.h) on the host: every field against
// integer arithmetic modulo 1024, and the bits above them untouched.
#include <cstdio>
#include <cstdlib>

#include "common.h"

static int wrap(int n) { return ((n + 512) & 1023) - 512; }

static void check(const int (&x)[3], const int (&y)[3]) {
    using namespace ann;
    const uint32_t a = pack_img(x[0], x[1], x[2]), b = pack_img(y[0], y[1], y[2]);
    int n[3], m[3];
    unpack_img(a, n[0], n[1], n[2]);
    for (uint32_t j = 0; j < 4; ++j) {                  // the two index bits above the fields
        const uint32_t d = img_minus(j << 30 | a, b);
        unpack_img(d, m[0], m[1], m[2]);
        bool ok = a < (1u << 30) && d >> 30 == j;
        for (int t = 0; t < 3; ++t) ok = ok && n[t] == wrap(x[t]) && m[t] == wrap(x[t] - y[t]);
        if (ok) continue;
        std::printf("(%d %d %d) - (%d %d %d): %d %d %d, index bits %u of %u\n", x[0], x[1], x[2], y[0], y[1], y[2], m[0],
                    m[1], m[2], d >> 30, j);
        std::exit(1);
    }
}

int main() {
    const int edge[] = {0, 1, -1, 2, 255, 256, -256, 510, 511, 512, 513, -510, -511, -512, -513, 1000, -1024, 100000000};
    for (int a : edge)
        for (int b : edge)
            for (int c : edge)
                for (int d : edge) {
                    check({a, b, c}, {d, a, b});
                    check({c, a, b}, {b, d, a});
                }
    std::puts("ok");
    return 0;
}
