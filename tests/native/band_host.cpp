// Host build of the band kernels' tile rule (band_columns in na_common.h)
// against brute force over axis_geometry, for the CPU tests through ctypes.
#include "na_common.h"

extern "C" {

int host_band_columns(int K, int key) { return na::band_columns(K, key != 0); }

// The widest union of any tile of T items (query or key side) of kernel K
// and dilation d, over every extent from K * d to Lmax.
int host_widest_union(int Lmax, int K, int d, int causal, int T, int key) {
    int want = 0;
    const na::FastDiv fd = na::make_fastdiv(static_cast<uint32_t>(d));
    for (int L = K * d; L <= Lmax; ++L) {
        if (!causal && d == 1 && K % 2 == 0 && K == L) continue;
        for (int r = 0; r < d; ++r) {
            const int cn = (L - r + d - 1) / d;
            for (int t = 0; t * T < cn; ++t) {
                const na::AxisGeo g = na::axis_geometry(L, K, d, causal, L % d, 1, L, T, t, r, 0, T - 1, key != 0, fd);
                if (g.U > want) want = g.U;
            }
        }
    }
    return want;
}

}  // extern "C"
