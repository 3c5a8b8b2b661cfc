// Host driver for the library's field arithmetic (stwo-zig_amd/csrc/fields.hpp): reads
// "q a0 b0 a1 b1 c0 d0 c1 d1", "c a b c d" or "i a" lines and prints the QM31 product, the
// CM31 product or the M31 inverse, "f a b t" (forward butterfly on signed words: the raw and the
// canonical results), "g a b t s" (inverse butterfly on words in [0, p], plain and scaled by s) and
// "m d t" (product of a signed word), so that a test can compare them with an independent
// big-integer restatement of the field laws.
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstring>
#include "../../stwo-zig_amd/csrc/fields.hpp"
using namespace sr;
int main() {
    char op[4];
    while (scanf("%3s", op) == 1) {
        if (!strcmp(op, "q")) {
            uint32_t v[8];
            for (int k = 0; k < 8; k++)
                if (scanf("%u", &v[k]) != 1) return 1;
            const qm31 r = qmul({{v[0], v[1]}, {v[2], v[3]}}, {{v[4], v[5]}, {v[6], v[7]}});
            printf("%u %u %u %u\n", r.c0.a, r.c0.b, r.c1.a, r.c1.b);
        } else if (!strcmp(op, "c")) {
            uint32_t v[4];
            for (int k = 0; k < 4; k++)
                if (scanf("%u", &v[k]) != 1) return 1;
            const cm31 r = cmul({v[0], v[1]}, {v[2], v[3]});
            printf("%u %u\n", r.a, r.b);
        } else if (!strcmp(op, "i")) {
            uint32_t a;
            if (scanf("%u", &a) != 1) return 1;
            printf("%u\n", minv(a));
        } else if (!strcmp(op, "f")) {
            int a, b;
            uint32_t t;
            if (scanf("%d %d %u", &a, &b, &t) != 3) return 1;
            uint32_t x = (uint32_t)a, y = (uint32_t)b;
            mbfly(x, y, mtw2(t), -mtw2(t));
            printf("%d %d %u %u\n", (int)x, (int)y, mcanon(x), mcanon(y));
        } else if (!strcmp(op, "g")) {
            uint32_t a, b, t, sc;
            if (scanf("%u %u %u %u", &a, &b, &t, &sc) != 4) return 1;
            uint32_t x = a, y = b, xs = a, ys = b;
            mibfly(x, y, mtw2(t));
            mibfly_scaled(xs, ys, mtw2(sc), mtw2(mmul(t, sc)));
            printf("%u %u %u %u\n", x, y, xs, ys);
        } else if (!strcmp(op, "m")) {
            int d;
            uint32_t t;
            if (scanf("%d %u", &d, &t) != 2) return 1;
            printf("%u\n", mmul_s((uint32_t)d, mtw2(t)));
        } else {
            return 1;
        }
    }
    return 0;
}
