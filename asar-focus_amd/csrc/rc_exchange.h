// LDS exchanges of the row transforms in a padded layout with compile-time offsets (k_rc_pad.hip, rc_block.h):
// element i sits at i + (i >> PS), and a pass's gather positions x[j + r*N/R] and scatter positions
// (j / NS)*NS*R + j % NS + r*NS become a per-butterfly base plus an offset that depends on r alone.
#pragma once
#include "kernels.h"

namespace asarf {
namespace rcpad {

template <int PS>
__host__ __device__ constexpr int lpos(int i) {
    return i + (i >> PS);
}

template <int R, int NS>
__host__ __device__ constexpr int scat_base(int j) {
    return (j / NS) * NS * R + j % NS;
}

// True when lpos(j + r*(N/R)) - lpos(j) depends on r alone.
template <int N, int R, int PS>
constexpr bool gather_const() {
    constexpr int M = N / R;
    for (int j = 0; j < M; ++j)
        for (int r = 1; r < R; ++r)
            if (lpos<PS>(j + r * M) - lpos<PS>(j) != lpos<PS>(r * M)) return false;
    return true;
}

// True when lpos(scat_base(j) + r*NS) - lpos(scat_base(j)) depends on r alone.
template <int N, int R, int NS, int PS>
constexpr bool scatter_const() {
    for (int j = 0; j < N / R; ++j) {
        const int b = scat_base<R, NS>(j);
        for (int r = 1; r < R; ++r)
            if (lpos<PS>(b + r * NS) - lpos<PS>(b) != lpos<PS>(r * NS)) return false;
    }
    return true;
}

// Butterflies j = lane + i*T, i < NB. Lanes past the last butterfly work on a clamped copy (registers written
// unconditionally keep the array in registers); a butterfly past the end for the whole wave is skipped.
template <int N, int R, int T>
struct Pass {
    static constexpr int M = N / R;
    static constexpr int NB = (M + T - 1) / T;
    static constexpr bool partial(int i) { return (i + 1) * T > M; }
};

template <int N, int R, int T, int PS, int E>
__device__ __forceinline__ void ld_gather(float2 (&v)[E], int lane, const float2* lds) {
    using P = Pass<N, R, T>;
    static_assert(P::NB * R <= E, "register array too small");
    constexpr bool C = gather_const<N, R, PS>();
#pragma unroll
    for (int i = 0; i < P::NB; ++i) {
        if (P::partial(i) && !wave_any(lane + i * T < P::M)) break;
        const int j = min(lane + i * T, P::M - 1);
        if constexpr (C) {
            const float2* p = lds + lpos<PS>(j);
#pragma unroll
            for (int r = 0; r < R; ++r) v[i * R + r] = p[lpos<PS>(r * P::M)];
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) v[i * R + r] = lds[lpos<PS>(j + r * P::M)];
        }
    }
}

template <int N, int R, int T, int PS, int E>
__device__ __forceinline__ void st_gather(const float2 (&v)[E], int lane, float2* lds) {
    using P = Pass<N, R, T>;
    constexpr bool C = gather_const<N, R, PS>();
#pragma unroll
    for (int i = 0; i < P::NB; ++i) {
        const int j = lane + i * T;
        if (P::partial(i) && j >= P::M) continue;
        if constexpr (C) {
            float2* p = lds + lpos<PS>(j);
#pragma unroll
            for (int r = 0; r < R; ++r) p[lpos<PS>(r * P::M)] = v[i * R + r];
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) lds[lpos<PS>(j + r * P::M)] = v[i * R + r];
        }
    }
}

template <int N, int R, int NS, int T, int PS, int E>
__device__ __forceinline__ void ld_scatter(float2 (&v)[E], int lane, const float2* lds) {
    using P = Pass<N, R, T>;
    static_assert(P::NB * R <= E, "register array too small");
    constexpr bool C = scatter_const<N, R, NS, PS>();
#pragma unroll
    for (int i = 0; i < P::NB; ++i) {
        if (P::partial(i) && !wave_any(lane + i * T < P::M)) break;
        const int j = min(lane + i * T, P::M - 1);
        const int b = scat_base<R, NS>(j);
        if constexpr (C) {
            const float2* p = lds + lpos<PS>(b);
#pragma unroll
            for (int r = 0; r < R; ++r) v[i * R + r] = p[lpos<PS>(r * NS)];
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) v[i * R + r] = lds[lpos<PS>(b + r * NS)];
        }
    }
}

template <int N, int R, int NS, int T, int PS, int E>
__device__ __forceinline__ void st_scatter(const float2 (&v)[E], int lane, float2* lds) {
    using P = Pass<N, R, T>;
    constexpr bool C = scatter_const<N, R, NS, PS>();
#pragma unroll
    for (int i = 0; i < P::NB; ++i) {
        const int j = lane + i * T;
        if (P::partial(i) && j >= P::M) continue;
        const int b = scat_base<R, NS>(j);
        if constexpr (C) {
            float2* p = lds + lpos<PS>(b);
#pragma unroll
            for (int r = 0; r < R; ++r) p[lpos<PS>(r * NS)] = v[i * R + r];
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) lds[lpos<PS>(b + r * NS)] = v[i * R + r];
        }
    }
}

}  // namespace rcpad
}  // namespace asarf
