// Host build of the frustum tests' interval cut, for tests/test_frustum_cut.py.
#include "smg_pe_body.hpp"

extern "C" void frustum_cut_n(int n, const float* c, const float* r, float* lo, float* hi) {
    for (int i = 0; i < n; ++i) {
        lo[i] = 0.0f;
        hi[i] = 1.0f;
        smg::frustum_cut(c[i], r[i], lo[i], hi[i]);
    }
}
