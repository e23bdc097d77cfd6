// Host build of the 1D gradient pass's steps (libcpab_amd/csrc/cpab_device.hpp) for
// CPU tests.  Test-only; the library never loads this.
#include <math.h>
#include <string.h>
#include <vector>

#include "../libcpab_amd/csrc/cpab_device.hpp"

using namespace cpab;

// Points whose end differs in any bit from the forward's: after the chunks of the
// gradient's pass (which = 0), or the forward's with the whole-cell table (1) or the
// gradient's pass with it (2).
extern "C" int host_signal_mismatches(int nx, const float* A, const float* x, int nP, int which) {
    CellTable<1> plain;
    plain.A = A;
    plain.inv_n = nullptr;
    plain.pl = nullptr;
    plain.nb = nullptr;
    CellTable<1> tab = plain;
    std::vector<float2> hits(2 * nx);
    for (int i = 0; i < 2 * nx; ++i) hits[i] = whole_cell(plain, i >> 1, i & 1, nx);
    if (which) tab.hits = hits.data();
    int bad = 0;
    for (int p = 0; p < nP; ++p) {
        float want[1] = {x[p] * (float)nx}, got[1] = {want[0]}, J[1][1];
        const int c0 = find_cell1(x[p], nx);
        integrate<1, true>(want, c0, 1.f, plain, nx, 0.f, J);
        if (which == 1) {
            integrate<1, true>(got, c0, 1.f, tab, nx, 0.f, J);
        } else {
            PointState<1> st;
            const float q[1] = {got[0]};
            init_point<1>(st, q, c0, 1.f);
            while (point_active<1>(st)) {
                Chunk1 ch;
                advance1(st, tab, nx, ch);
            }
            got[0] = st.q[0];
        }
        bad += memcmp(want, got, sizeof(float)) != 0;
    }
    return bad;
}

extern "C" void host_phis(const float* z, int n, float* p1, float* p2) {
    for (int i = 0; i < n; ++i) phis(z[i], p1[i], p2[i]);
}
