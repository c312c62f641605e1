// Column transforms of 2 to 30 points (the strided first pass of a short azimuth transform: 525 = 5 x 105, 2058 =
// 21 x 98): one lane per column and group holds the whole transform in registers, so there is no LDS, no barrier and
// every row access is 256 contiguous columns. Bounded by launch and memory latency at the shortest (525 x 496 columns:
// 4.6 us a pass, 20 us with the runtime-radix kernel, whose 16 lanes per column share one 5-point butterfly) and by
// memory from 16 points on: pass A of 1512 x 4912 columns 2.8 -> 4.6 TB/s, A' 3.4 -> 5.4; of 2058 lines 3.1 -> 4.8 and
// 3.8 -> 5.8, before with 16 lanes per column and an LDS exchange between two radices of 3 to 7 (col_static.h).
// Both passes, in microseconds, of n x 105 by 4912 columns, LDS kernel -> this one: n = 16 82 -> 60,
// 21 91 -> 73, 25 95 -> 81, 28 99 -> 91, 30 102 -> 95. The line lies at 30 because a transform of n points takes about
// 4.6 n registers: 32 points leave three waves per SIMD and take 113 us against 106, 40 points 162 against 160. (A
// four-wave bound spills from 28 points on: 30 points 101 us, 32 points 130.)
// From 16 points on a launch has to fill the chip first: one lane's chain of n loads, the transform and n twiddle
// loads takes 2 to 5 us longer than sixteen lanes' share of it, so smaller launches keep the LDS kernels. Both passes,
// LDS against this kernel, by workgroups of 256 columns: 21 x 49 by 250 columns (49) 21.5 and 24.4 us, 30 x 105 by
// 500 (210) 33.2 and 39.5, 30 x 49 by 2000 (392) 37.3 and 41.1; 20 x 35 by 4000 (560) 39.1 and 38.2, 25 x 49 by 4000
// (784) 49.0 and 45.4, 30 x 105 by 4000 (1680) 84.5 and 82.0. The line lies at two workgroups per CU.
#include "kernels.h"

namespace asarf {

constexpr long kSmallWorkgroups = 512;  // of 256 columns, from 16 points on

template <bool INV, int N>
__global__ __launch_bounds__(256) void k_col_small(ColFftArgs a) {
    if (a.fused_gate && *a.fused_gate <= kAzCoreReach) return;
    const int x = blockIdx.x * 256 + threadIdx.x;
    if (x >= a.ncols) return;
    for (int g = blockIdx.y; g < a.groups; g += gridDim.y) {  // the same for every lane
        float2 v[N];
#pragma unroll
        for (int m = 0; m < N; ++m) {
            const long r = (long)g * a.in_g + (long)m * a.in_m;
            v[m] = r < a.in_rows ? a.in[r * a.in_stride + x] : make_float2(0.f, 0.f);
        }
        Dft<N, INV>::run(v);
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const long r = (long)g * a.out_g + (long)k * a.out_m;
            if (r >= a.out_rows) continue;
            float2 y = v[k];
            if (a.tw_full) {
                const float2 w = a.tw_full[(long)g * k];
                y = INV ? cmulc(y, w) : cmul(y, w);
            }
            a.out[r * a.out_stride + x] = cscale(y, a.scale);
        }
    }
}

template <int N>
static hipError_t launch_small(const ColFftArgs& a, bool inverse, hipStream_t s) {
    const dim3 grid((a.ncols + 255) / 256, std::min(a.groups, 65535));
    if (inverse)
        hipLaunchKernelGGL((k_col_small<true, N>), grid, dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((k_col_small<false, N>), grid, dim3(256), 0, s, a);
    return hipGetLastError();
}

bool launch_col_small(const ColFftArgs& a, bool inverse, hipStream_t s, hipError_t* err) {
    if (a.ncols < 1 || a.groups < 1) return false;
    if (a.sub.n >= 16 && (long)((a.ncols + 255) / 256) * a.groups < kSmallWorkgroups) return false;
    switch (a.sub.n) {
#define ASARF_COL_SMALL(N) \
    case N: *err = launch_small<N>(a, inverse, s); return true;
        ASARF_COL_SMALL(2) ASARF_COL_SMALL(3) ASARF_COL_SMALL(4) ASARF_COL_SMALL(5) ASARF_COL_SMALL(6)
        ASARF_COL_SMALL(7) ASARF_COL_SMALL(8) ASARF_COL_SMALL(9) ASARF_COL_SMALL(10) ASARF_COL_SMALL(12)
        ASARF_COL_SMALL(14) ASARF_COL_SMALL(15)
        ASARF_COL_SMALL(16) ASARF_COL_SMALL(18) ASARF_COL_SMALL(20) ASARF_COL_SMALL(21) ASARF_COL_SMALL(24)
        ASARF_COL_SMALL(25) ASARF_COL_SMALL(27) ASARF_COL_SMALL(28) ASARF_COL_SMALL(30)
#undef ASARF_COL_SMALL
        default: return false;
    }
}

}  // namespace asarf
