/*
 * Packing of the row tables (struct RowTables of engine_common.h) from the
 * columns of a physics file. Host code, without HIP.
 */
#ifndef PUMAS_ROW_TABLES_H
#define PUMAS_ROW_TABLES_H

#include <stddef.h>
#include <stdint.h>

#include <vector>

#include "engine_common.h"

namespace pg {

/* Energy loss schemes with row tables: the CSDA's [0], and the mixed and
 * straggled losses' [1]. */
constexpr int ROW_SCHEMES = 2;

/* A double precision column of the physics file: `count` values, or a NULL
 * pointer when it is missing. */
struct RowSource {
        const double * values;
        uint64_t count;
};

/* Doubles of one scheme's row tables, even (they are copied in 16 B words). */
inline size_t row_tables_size(int n_materials, int n_energies)
{
        return ((size_t)n_materials * n_energies * ROW_COLUMNS + 1) / 2 * 2;
}

/*
 * Packs the row tables of every scheme, one after the other, into `rows`.
 * `find` returns the RowSource of a column. Returns the name of a column that
 * is missing or shorter than the sizes say, NULL when `rows` is packed. The
 * sizes come from the file as well: nothing is allocated or read before every
 * column is known to hold them.
 */
template <class Find>
const char * pack_row_tables(
    Find find, int n_materials, int n_energies, std::vector<double> & rows)
{
        static const struct {
                const char * name;
                int column;
                int first; /* tables before scheme 0's, -1: one for all */
        } columns[] = { { "X", ROW_X, 0 }, { "X_dK", ROW_X_DK, 0 },
                { "K_dX", ROW_K_DX, 0 }, { "dE", ROW_DE, 0 },
                { "dE_dK", ROW_DE_DK, 0 }, { "Omega", ROW_OMEGA, -1 },
                { "Omega_dK", ROW_OMEGA_DK, -1 }, { "CS", ROW_CS, -1 },
                { "CS_dK", ROW_CS_DK, -1 }, { "Mu0", ROW_MU0, -1 },
                { "Mu0_dK", ROW_MU0_DK, -1 },
                /* Led by the tables without energy loss. */
                { "Ms1", ROW_MS1, 1 }, { "Ms1_dK", ROW_MS1_DK, 1 },
                { "Lb", ROW_LB, -1 } };
        const auto holds = [&](const RowSource & s, uint64_t tables) {
                return (s.values != nullptr) &&
                    (s.count / (uint64_t)n_energies >= tables);
        };
        if ((n_materials < 1) || (n_energies < 2)) return "K";
        const uint64_t nM = n_materials;
        const RowSource K = find("K");
        if (!holds(K, 1)) return "K";
        for (const auto & col : columns)
                if (!holds(find(col.name),
                        (col.first < 0) ? nM : nM * (col.first + ROW_SCHEMES)))
                        return col.name;

        const size_t size = row_tables_size(n_materials, n_energies);
        rows.assign(ROW_SCHEMES * size, 0.);
        const auto fill = [&](int scheme, size_t m, int column,
                              const double * src) {
                double * dst = rows.data() + scheme * size +
                    m * n_energies * ROW_COLUMNS + column;
                for (int i = 0; i < n_energies; i++)
                        dst[(size_t)i * ROW_COLUMNS] = src[i];
        };
        for (int scheme = 0; scheme < ROW_SCHEMES; scheme++)
                for (size_t m = 0; m < nM; m++) {
                        fill(scheme, m, ROW_K, K.values);
                        for (const auto & col : columns) {
                                const size_t table = (col.first < 0) ? m :
                                    (col.first + scheme) * nM + m;
                                fill(scheme, m, col.column,
                                    find(col.name).values +
                                        table * n_energies);
                        }
                }
        return nullptr;
}

} /* namespace pg */

#endif
