// Host check of the sweeps' index schemes (tiles_device.h): see tests/test_tiling.py.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <vector>

#include "tiles_device.h"

using namespace glide;

#define CHECK(c)                                                \
    do {                                                        \
        if (!(c)) return std::printf("line %d: %s\n", __LINE__, #c), 1; \
    } while (0)

int glide::set_error(int code, const char *) { return code; }

int main()
{
    long n_checks = 0;
    // tiles dealt to the XCDs: every tile once, the rest of the grid past the last one
    for (int total = 1; total < 3000; total++) {
        std::vector<int> seen(total);
        const int G = chunked_grid(total);
        CHECK(G >= total && G % NXCD == 0);
        for (int b = 0; b < G; b++) {
            const int t = chunked_tile(b, total);
            CHECK(t >= 0);
            if (t < total) seen[t]++;
        }
        for (int t = 0; t < total; t++) CHECK(seen[t] == 1);
        n_checks += total;
    }
    // several sweeps a launch, one dimension: every cell has one owner, the tile lies in the level, and
    // what goes stale (2 cells a sweep, the faces at the far side one earlier) stays outside the owned cells
    for (int ns = 1; ns <= 3; ns++)
        for (int n = 1; n < 400; n++) {
            const int own = multi_own(n, ns);
            std::vector<int> owners(n);
            for (int b = 0; b < cdiv(n, own); b++) {
                const int io = b * own, i0 = multi_origin(io, n, ns);
                CHECK(i0 >= 0 && i0 <= io && (n <= MS ? i0 == 0 : i0 + MS <= n));
                for (int i = io; i < io + own && i < n; i++) {
                    owners[i]++;
                    CHECK(i - i0 < MS);
                    CHECK(i0 == 0 || i - i0 >= 2 * ns);
                    CHECK(i0 + MS >= n || i0 + MS - 1 - i >= 2 * ns - 1);
                }
            }
            for (int i = 0; i < n; i++) CHECK(owners[i] == 1);
            n_checks += n;
        }
    // pending updates: four arrays a set, two sets, behind the state and inside the scratch of 5 nc doubles
    constexpr int TX = 64, TY = 4;
    static double base[1];
    for (int ny = 1; ny < 300; ny += 1 + ny / 9)
        for (int nx = 1; nx < 700; nx += 1 + nx / 9) {
            if (!fold_fits(ny, nx, TX, TY)) continue;
            const size_t ntx = cdiv(nx, TX), nty = cdiv(ny, TY);
            size_t end = n_t(ny, nx);
            for (int set = 0; set < 2; set++) {
                const FoldPending P = fold_pending<TX, TY>(base, ny, nx, set);
                for (const auto &a : {std::pair<double *, size_t>{P.top, nty * nx}, {P.bot, nty * nx}, {P.lft, ny * ntx},
                                      {P.rgt, ny * ntx}}) {
                    CHECK((size_t)(a.first - base) == end);
                    end += a.second;
                }
            }
            CHECK(end <= 5 * n_c(ny, nx));
            n_checks++;
        }
    std::printf("ok %ld\n", n_checks);
    return 0;
}
