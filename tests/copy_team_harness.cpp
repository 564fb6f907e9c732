// Shared copies of every length given on the command line, by teams of none to three
// helpers, into a poisoned destination: prints each length that arrives incomplete
// or past its end.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "copy_team.h"

int main(int argc, char **argv)
{
    int bad = 0;
    for (int helpers = 0; helpers <= 3; ++helpers) {
        mbs::CopyTeam team(helpers);
        for (int a = 1; a < argc; ++a) {
            const size_t n = std::strtoull(argv[a], nullptr, 10);
            std::vector<unsigned char> src(n), dst(n + 64, 0xee);
            for (size_t i = 0; i < n; ++i)
                src[i] = (unsigned char)(i * 7 + 1) % 0xee;
            team.copy(dst.data(), src.data(), n);
            size_t wrong = 0;
            for (size_t i = 0; i < n + 64; ++i)
                wrong += dst[i] != (i < n ? src[i] : 0xee);
            const size_t m = n / sizeof(double);
            std::vector<double> x(m + 8, 1.0), y(m);
            for (size_t i = 0; i < m; ++i)
                y[i] = (double)i;
            team.copy(x.data(), y.data(), m * sizeof(double), true);
            for (size_t i = 0; i < m + 8; ++i)
                wrong += x[i] != (i < m ? 1.0 + (double)i : 1.0);
            if (wrong) {
                std::printf("%d helpers, %zu bytes: %zu wrong\n", helpers, n, wrong);
                bad = 1;
            }
        }
    }
    return bad;
}
