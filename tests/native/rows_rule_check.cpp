// Host replay of the rule that sends row norms and softmax to the wide kernels (test only, plain C++):
// for rows of any width a call the rule takes has a grid of fewer than 2^32 threads, and only a call that
// would have more is left to the element-wise kernels. Prints "ok" or the first violation and exits 1.
#include <stdio.h>
#include "rows_wide.hpp"

using namespace cdna4;

int main() {
    static const int widths[] = {4, 101, 2047, 2048, 2049, 8191, 8192, 8193, 32001, 65536};
    for (int H : widths)
        for (long long m = 1; m <= 0x7fffffffLL; m = m < 1024 ? m + 1 : m + m / 37) {
            const int M = (int)m;
            for (int vec = 0; vec < 2; ++vec) {
                const bool takes = rows_wide_takes(M, H, vec != 0);
                // launch_op's threads per row: one wave up to 2,048 columns unless the rows are few
                const unsigned long long tpr = H <= 2048 && !rows_few(M, H) ? 64 : H <= 8192 ? 256 : 1024;
                const bool fits = (tpr == 64 ? ((unsigned long long)M + 3) / 4 * 256 : M * tpr) <= 0xffffffffull;
                if (takes && !fits) { printf("grid too large: M %d H %d vec %d\n", M, H, vec); return 1; }
                if (!takes && fits && !vec && (M + 64LL) * (long long)tpr < (1LL << 32)) {
                    printf("not taken: M %d H %d\n", M, H);
                    return 1;
                }
            }
        }
    printf("ok\n");
    return 0;
}
