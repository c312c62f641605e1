// Range compression in blocks of a line (the reference's RangeCompression, sar/range_compression.cu:57-111).
//
// The kept output samples x < nr - nc are sums of the nc input samples x .. x + nc - 1, so they need no transform of
// the reference's padded length: a circular correlation of any length N gives the N - nc + 1 outputs from x0 on
// exactly when it holds the input samples x0 .. x0 + N - 1 (overlap-save). A workgroup produces one such block of
// one line, and a line of any length runs in as many blocks of a compiled length as it needs. Each line's samples
// beyond nr are never read, so the padding values of the reference's row cannot reach a kept sample either.
//
//   N = 256 X (X = 4 .. 16): radices 16, 16, X on 64 to 256 lanes, one to four butterflies per lane and pass
//   6144: radices 8, 8, 8, 12 on 512 lanes, for lines in place that no shorter length holds
//
// What bounds it: vector issue (0.9 of the SIMD cycles; 30000 lines of 5616 samples in 0.54 to 0.55 ms, the padded
// transforms it replaces 0.64). Per sample and direction three passes cost about 30 FP32 instructions of butterflies and 7.5 of
// twiddle products; the rest is kept off the vector units. The samples are loaded straight into the first pass's registers (no
// staging through LDS, any row alignment). The twiddles of every pass come from a table in global memory (8 to 48 KB,
// held by L1 and L2) instead of being multiplied up from one power, two a 16-byte load: with 8-byte loads the return
// path of the vector memory unit was the bound (94 % busy; 8000 lines 158 us, 140 us with 16-byte loads). The inverse
// runs as the transpose of the forward passes, so both use the same tables and compile-time LDS offsets (see
// k_rc_pad.hip).
#pragma once
#include "rc_exchange.h"

namespace asarf {
namespace rcblock {

using rcpad::ld_gather;
using rcpad::ld_scatter;
using rcpad::lpos;
using rcpad::Pass;
using rcpad::st_gather;
using rcpad::st_scatter;

constexpr int kPadShift = 4;

// Start of pass p's twiddles in the table, in pairs: pass q >= 1 holds W_N^(r k N / (NS R)) for r = 2 s, 2 s + 1 at
// [s * NS + k].
template <class Seq>
constexpr int tw_offset(int p) {
    int o = 0;
    for (int q = 1; q < p; ++q) o += Seq::at(q) / 2 * Seq::prefix(q);
    return o;
}

// The twiddles of every butterfly of the lane in pass (R, NS), in the data's register layout. Issued before the
// pass's LDS reads, so that their latency overlaps the exchange.
template <int N, int R, int NS, int T, int E>
__device__ __forceinline__ void load_twiddles(float2 (&w)[E], int lane, const float4* __restrict__ tab) {
    using P = Pass<N, R, T>;
    static_assert(R % 2 == 0, "twiddles are read in pairs");
#pragma unroll
    for (int i = 0; i < P::NB; ++i) {
        if (P::partial(i) && !wave_any(lane + i * T < P::M)) break;
        const unsigned k = (unsigned)min(lane + i * T, P::M - 1) % NS;
#pragma unroll
        for (int r = 0; r < R; r += 2) {
            const float4 t = (tab + r / 2 * NS)[k];
            w[i * R + r] = make_float2(t.x, t.y);
            w[i * R + r + 1] = make_float2(t.z, t.w);
        }
    }
}

template <int N, int R, int NS, int T, bool INV, int E>
__device__ __forceinline__ void pass(float2 (&v)[E], const float2 (&w)[E], int lane) {
    using P = Pass<N, R, T>;
#pragma unroll
    for (int i = 0; i < P::NB; ++i) {
        if (P::partial(i) && !wave_any(lane + i * T < P::M)) break;
        if constexpr (!INV && NS > 1) {
#pragma unroll
            for (int r = 1; r < R; ++r) v[i * R + r] = cmul(v[i * R + r], w[i * R + r]);
        }
        Dft<R, INV>::run(&v[i * R]);
        if constexpr (INV && NS > 1) {
#pragma unroll
            for (int r = 1; r < R; ++r) v[i * R + r] = cmulc(v[i * R + r], w[i * R + r]);
        }
    }
}

// Range-checked access to a line (the raw-buffer instructions: loads past `bytes` return 0, stores past it are
// dropped): no compare, no branch and no 64-bit address per element. The whole offset goes through the range-checked
// operand, not the scalar one.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const void* p, long bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)max(bytes, 0L), 0x00027000);
}
typedef unsigned uint2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float2 load_b64(__amdgpu_buffer_rsrc_t b, int off) {
    const uint2v u = __builtin_amdgcn_raw_buffer_load_b64(b, off, 0, 0);
    return make_float2(__uint_as_float(u.x), __uint_as_float(u.y));
}
__device__ __forceinline__ unsigned load_b16(__amdgpu_buffer_rsrc_t b, int off) {
    return __builtin_amdgcn_raw_buffer_load_b16(b, off, 0, 0);
}
__device__ __forceinline__ void store_b64(float2 v, __amdgpu_buffer_rsrc_t b, int off) {
    const uint2v u = {__float_as_uint(v.x), __float_as_uint(v.y)};
    __builtin_amdgcn_raw_buffer_store_b64(u, b, off, 0, 0);
}

template <int N>
__host__ __device__ constexpr int data_elems() {
    return (lpos<kPadShift>(N - 1) + 2) & ~1;  // even: what follows is 16-byte aligned
}

// Copies nbytes of a record into LDS (dst 16-byte aligned), 16 bytes a load at any source alignment.
struct __attribute__((packed, aligned(1))) Bytes16 {
    unsigned x, y, z, w;
};
template <int T>
__device__ __forceinline__ void stage_bytes(const uint8_t* __restrict__ src, int nbytes, uint8_t* dst, int lane) {
    for (int c = lane * 16; c + 16 <= nbytes; c += T * 16) {
        const Bytes16 b = *reinterpret_cast<const Bytes16*>(src + c);
        *reinterpret_cast<uint4*>(dst + c) = make_uint4(b.x, b.y, b.z, b.w);
    }
    const int t = max(nbytes, 0) & ~15;
    if (t + lane < nbytes) dst[t + lane] = src[t + lane];
}

// FBAQ-4 blocks (a quantiser id and 63 code bytes) that N consecutive samples can touch.
constexpr int fbaq_blocks(int n) { return (n + 62) / 63 + 1; }

template <int FMT, int N, int T, int WAVES, class Seq>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(WAVES))) void k_rc_block(RcArgs a) {
    static_assert(Seq::product() == N, "radix sequence must factor N");
    constexpr int E = seq_max_elems<N, Seq, T>();
    constexpr int NP = Seq::count;
    constexpr int PS = kPadShift;
    extern __shared__ float2 lds[];
    // A pass of N / 16 butterflies leaves the last waves of the workgroup idle (3072: one of four). Waves go to the
    // SIMDs in order, so the idle ones are rotated from workgroup to workgroup.
    constexpr int WV = T / 64;
    const int lane = WV > 1 ? (int)((threadIdx.x + 64 * (blockIdx.x % WV)) % T) : (int)threadIdx.x;
    const int row = blockIdx.x / a.blocks;
    const int blk = blockIdx.x - row * a.blocks;
    const int x0 = blk * a.block_step;
    float ki = 0.f, kq = 0.f, ii = 1.f, i0 = 0.f, qi = 0.f, qq = 1.f, q0 = 0.f;  // the affine I/Q correction
    if (FMT != RAW_CF32 && a.coef) {
        ki = a.coef->ki;
        kq = a.coef->kq;
        ii = a.coef->ii;
        i0 = a.coef->i0;
        qi = a.coef->qi;
        qq = a.coef->qq;
        q0 = a.coef->q0;
    }
    auto correct = [&](float i, float q) {
        const float di = i - ki, dq = q - kq;
        return make_float2(fmaf(ii, di, i0), fmaf(qi, di, fmaf(qq, dq, q0)));
    };
    float2 v[E], w[E];
    // ---- the block's samples into the first pass's gather positions, corrected on load
    {
        constexpr int R = Seq::at(0);
        using P = Pass<N, R, T>;
        const int left = a.nr_in - x0;  // samples of the line from x0 on (may exceed N)
        // f(register, j, off): block sample j + off, off the same for every lane
        auto each = [&](auto&& f) {
#pragma unroll
            for (int i = 0; i < P::NB; ++i) {
                if (P::partial(i) && !wave_any(lane + i * T < P::M)) break;
                const int j = min(lane + i * T, P::M - 1);
#pragma unroll
                for (int r = 0; r < R; ++r) f(i * R + r, j, r * P::M);
            }
        };
        if constexpr (FMT == RAW_CF32) {
            // samples past the line's end (range-checked loads: 0) reach no kept output sample
            const auto in = buffer(static_cast<const float2*>(a.in) + (long)row * a.in_stride + x0, (long)left * 8);
            each([&](int e, int j, int off) { v[e] = load_b64(in, (j + off) * 8); });
        } else if constexpr (FMT == RAW_ASAR_FBAQ4) {
            // The record bytes of the block's samples and the 16 table entries of each of their quantiser blocks are
            // staged in the data area (16-byte loads), then every sample is one code byte and two entries from LDS.
            // NaN where no sample lands becomes 0 (ZeroNaNs).
            constexpr int NQ = fbaq_blocks(N);
            static_assert(NQ * (64 + 128) <= data_elems<N>() * 8, "the staged record fits the data area");
            uint8_t* bytes = reinterpret_cast<uint8_t*>(lds);
            float4* rows = reinterpret_cast<float4*>(bytes + NQ * 64);
            const uint8_t* rec = static_cast<const uint8_t*>(a.in) + (long)row * a.lines.line_bytes;
            const int len = (int)min((long)fbaq4_record_length(rec), a.lines.line_bytes - 2);
            const int s0 = x0 - a.lines.shift(row);
            const int send = s0 + min(left, N);  // samples [max(s0, 0), send)
            const int q0 = max(s0, 0) / 63;
            const int nq = send > 0 ? (send - 1) / 63 - q0 + 1 : 0;
            const int nb = min(64 * nq, len - 64 * q0);
            stage_bytes<T>(rec + 2 + 64 * q0, nb, bytes, lane);
            __syncthreads();
            const float4* __restrict__ lut = reinterpret_cast<const float4*>(a.lines.lut);
            for (int i = lane; i < 8 * nq && 8 * nb > 64 * (i & ~7); i += T) rows[i] = lut[8 * bytes[8 * (i & ~7)] + (i & 7)];
            __syncthreads();
            each([&](int e, int j, int off) {
                const int s = s0 + j + off;
                const unsigned q = (unsigned)max(s, 0) / 63u - q0;
                const int k = max(s, 0) + (int)(q + q0) + 1 - 64 * q0;  // code byte of the staged ones
                v[e] = make_float2(0.f, 0.f);
                if (j + off < left && s >= 0 && k < nb) {
                    const int code = bytes[k], ci = code >> 4, cq = code & 15;
                    const float2* r = reinterpret_cast<const float2*>(rows) + 16 * q;
                    v[e] = correct(r[ci > 7 ? 15 - ci : 8 + ci].x, r[cq > 7 ? 15 - cq : 8 + cq].y);
                }
            });
        } else {
            // I/Q byte pairs, two bytes a load; all of a lane's loads are in flight before the first is used. (Staged
            // through LDS with 16-byte loads: slower, 158 against 140 us for 8000 lines of 5616 samples.)
            unsigned raw[E];
            auto pair = [&](unsigned u) {
                if constexpr (FMT == RAW_I8)
                    return correct((float)(int)(signed char)(u & 0xFFu), (float)(int)(signed char)((u >> 8) & 0xFFu));
                else
                    return correct((float)(u & 0xFFu), (float)((u >> 8) & 0xFFu));
            };
            if constexpr (FMT == RAW_ERS_LINES) {
                // NaN where the shift puts no sample of the line becomes 0 (ZeroNaNs)
                const int spl = a.lines.spl, s0 = x0 - a.lines.shift(row);
                const auto in = buffer(static_cast<const uint8_t*>(a.in) + (long)row * a.lines.line_bytes, 2L * spl);
                each([&](int e, int j, int off) { raw[e] = load_b16(in, (s0 + j + off) * 2); });
                each([&](int e, int j, int off) {
                    v[e] = (unsigned)(s0 + j + off) < (unsigned)spl && j + off < left ? pair(raw[e])
                                                                                     : make_float2(0.f, 0.f);
                });
            } else {
                // samples past the line's end reach no kept output sample; they are zero so that they add no rounding
                const auto in =
                    buffer(static_cast<const uint8_t*>(a.in) + ((long)row * a.in_stride + x0) * 2, 2L * left);
                each([&](int e, int j, int off) { raw[e] = load_b16(in, (j + off) * 2); });
                each([&](int e, int j, int off) {
                    v[e] = pair(raw[e]);
                    if (off + P::M > left) {  // the same for every lane
                        if (j + off >= left) v[e] = make_float2(0.f, 0.f);
                    }
                });
            }
        }
        if constexpr (FMT == RAW_ASAR_FBAQ4) __syncthreads();  // the staged record is read before the first scatter
    }
    // ---- forward transform, decimation in time: pass p gathers, twiddles (p > 0), DFT, scatters
    static_for<0, NP>([&](auto pc) __attribute__((always_inline)) {
        constexpr int p = decltype(pc)::value;
        constexpr int R = Seq::at(p), NS = Seq::prefix(p);
        if constexpr (p > 0) {
            load_twiddles<N, R, NS, T>(w, lane, a.rc_tw + tw_offset<Seq>(p));
            ld_gather<N, R, T, PS>(v, lane, lds);
            __syncthreads();  // every element is read before the scatter of this pass overwrites LDS
        }
        pass<N, R, NS, T, false>(v, w, lane);
        if constexpr (p + 1 < NP) {
            st_scatter<N, R, NS, T, PS>(v, lane, lds);
            __syncthreads();
        }
    });
    // ---- matched filter: the last forward pass left X[j + r*M] in butterfly j
    {
        constexpr int R = Seq::at(NP - 1);
        using P = Pass<N, R, T>;
        const float4* __restrict__ h = reinterpret_cast<const float4*>(a.hconj);  // pairs, as the twiddles
#pragma unroll
        for (int i = 0; i < P::NB; ++i) {
            if (P::partial(i) && !wave_any(lane + i * T < P::M)) break;
            const unsigned j = min(lane + i * T, P::M - 1);
#pragma unroll
            for (int r = 0; r < R; r += 2) {
                const float4 t = (h + r / 2 * P::M)[j];
                v[i * R + r] = cmul(v[i * R + r], make_float2(t.x, t.y));
                v[i * R + r + 1] = cmul(v[i * R + r + 1], make_float2(t.z, t.w));
            }
        }
    }
    // ---- inverse transform, decimation in frequency: the transposes of the forward passes, last one first
    static_for<0, NP>([&](auto qc) __attribute__((always_inline)) {
        constexpr int p = NP - 1 - decltype(qc)::value;
        constexpr int R = Seq::at(p), NS = Seq::prefix(p);
        if constexpr (p + 1 < NP) {
            if constexpr (NS > 1) load_twiddles<N, R, NS, T>(w, lane, a.rc_tw + tw_offset<Seq>(p));
            ld_scatter<N, R, NS, T, PS>(v, lane, lds);
            __syncthreads();  // every element is read before the gather stores of this pass overwrite LDS
        }
        pass<N, R, NS, T, true>(v, w, lane);
        if constexpr (p > 0) {
            st_gather<N, R, T, PS>(v, lane, lds);
            __syncthreads();
        }
    });
    // ---- output: the last inverse pass (transpose of forward pass 0, NS = 1) holds x[j + r*N/R]; a block keeps its
    // first block_step samples, the last block of a line also clears the columns [nrv, zero_to)
    {
        constexpr int R = Seq::at(0);
        using P = Pass<N, R, T>;
        float2* out = a.out + (long)row * a.out_stride + x0;
        const bool last = blk + 1 == a.blocks;
        const int keep = min(last ? N : a.block_step, a.nrv - x0);
        const int clear = last ? a.zero_to - x0 : 0;
        const auto dst = buffer(out, 8L * keep);  // stores past it are dropped
#pragma unroll
        for (int i = 0; i < P::NB; ++i) {
            const int j = lane + i * T;
            if (P::partial(i) && j >= P::M) continue;
#pragma unroll
            for (int r = 0; r < R; ++r) store_b64(v[i * R + r], dst, (j + r * P::M) * 8);
        }
        for (int x = keep + lane; x < clear; x += T) out[x] = make_float2(0.f, 0.f);
    }
}

template <int N, int T, int WAVES, class Seq>
inline hipError_t launch(const RcArgs& a, int fmt, hipStream_t s) {
    const size_t lds = sizeof(float2) * (size_t)data_elems<N>();
    if (lds > max_lds_bytes()) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(a.rows * a.blocks)), block(T);
    if (fmt == RAW_CF32)
        hipLaunchKernelGGL((k_rc_block<RAW_CF32, N, T, WAVES, Seq>), grid, block, lds, s, a);
    else if (fmt == RAW_U8)
        hipLaunchKernelGGL((k_rc_block<RAW_U8, N, T, WAVES, Seq>), grid, block, lds, s, a);
    else if (fmt == RAW_ERS_LINES)
        hipLaunchKernelGGL((k_rc_block<RAW_ERS_LINES, N, T, WAVES, Seq>), grid, block, lds, s, a);
    else if (fmt == RAW_ASAR_FBAQ4)
        hipLaunchKernelGGL((k_rc_block<RAW_ASAR_FBAQ4, N, T, WAVES, Seq>), grid, block, lds, s, a);
    else
        hipLaunchKernelGGL((k_rc_block<RAW_I8, N, T, WAVES, Seq>), grid, block, lds, s, a);
    return hipGetLastError();
}

template <class Seq>
inline int fill_seq(int* radices) {
    for (int p = 0; p < Seq::count; ++p) radices[p] = Seq::at(p);
    return Seq::count;
}

}  // namespace rcblock
}  // namespace asarf
