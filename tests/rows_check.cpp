/* Row tables (engine_common.h) against the per column interpolation with its
 * bisection, on the host: for each x and first guess of a row, the number of
 * results that differ. */
#include <cstring>

#include "engine_common.h"

using namespace pg;

/* Column `c` (slopes in c + 1) of `rows` against the tables (k, y, m), all
 * of one material. c < 0: the inverse of column ROW_X, tables (k, y) = (X, K).
 */
extern "C" long rows_check(const double * rows, int n, int c, const double * k,
    const double * y, const double * m, const double * x, const int * guess,
    long count)
{
        RowTables<const double *> r = { n, 1, 0., rows };
        PhysicsView p;
        memset(&p, 0x0, sizeof(p));
        p.n_energies = n;
        p.K = k;
        long bad = 0;
        for (long i = 0; i < count; i++) {
                int last[2] = { n - 2, n - 2 };
                const int row = table_index(k, n, x[i]);
                int g = guess[i];
                double v;
                if (c >= 0) {
                        const Located l = r.locate(0, x[i], &g);
                        const int side =
                            (row < 0) ? -1 : ((row >= n - 1) ? 1 : 0);
                        if (l.side != side) bad++;
                        if (side != 0) {
                                bad += g != guess[i];
                                continue;
                        }
                        bad += (l.row != row) + (g != row);
                        v = r.value(l, c);
                } else {
                        double x0, x1;
                        const int j = r.find(0, ROW_X, x[i], g, x0, x1);
                        bad += j != row;
                        if ((j < 0) || (j >= n - 1)) continue;
                        const double * a = rows + j * ROW_COLUMNS;
                        const double * b = a + ROW_COLUMNS;
                        const double dx = x1 - x0;
                        const double m1 = a[ROW_K_DX] * dx;
                        v = pchip((x[i] - x0) / dx, a[ROW_K], b[ROW_K], m1,
                            (j > 0) ? b[ROW_K_DX] * dx : m1);
                }
                const double w = interpolate(p, last, k, y, m, x[i]);
                bad += memcmp(&v, &w, sizeof(v)) != 0;
        }
        return bad;
}
