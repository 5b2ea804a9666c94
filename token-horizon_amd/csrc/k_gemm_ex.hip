// k_gemm_ex.hip — f32 activations of any row count past 1 on the f16 matrix
// cores, every bit of x and of the weights.
//
// Role: candle's f32 QMatMul::forward on GGUF models (engine/src/
// model.rs:551-562) over prompts and verify steps.  Before it, every f32 call
// with M > 1 ran k_gemv_generic: scalar f32 dots, the weight dequantized again
// for every 8 rows (Q4_K gate/up + down of 4096 / 12288 at M = 300: 19.2 ms,
// now 0.47 ms; a decoder layer at M = 5: 424 us, now 105 us).
//
// Activations (k_xplanes, one launch per call): each row is scaled by a power
// of two and written as three f16 planes, x0 = f16(x), x1 = f16(2^11 (x - x0)),
// x2 = 2^11 (x - x0) - x1, which hold every f32 from the row's largest down to
// 2^-26 of it exactly (the matrix cores do not flush subnormals).  Two planes
// hold 23 bits: one in four f32 values loses its last, and a third of their
// MFMAs is what the 24th costs (the MLP above 0.41 ms, the layer 102 us).
// What the planes do not hold (smaller values, Inf, NaN, a few outliers that
// would push the rest out of their range) is listed per row and dotted in f32
// with the weight as the scalar kernel forms it.  The weights' integers are
// exact in f16 (Q4_K: sc (q - 8), at most 504; affine: q - 8; Q8_0: q; Q6_K:
// code - 32), so each product is exact in f32.  The offsets of the 4-bit
// weights are f32 factors times f32 sums of x.
//
// Sums: a 64-wide part (Q8_0: each 32-wide block of it, Q6_K: each 16-wide
// group) is summed by the matrix core from zero, x0 by itself: a chain that
// starts from the small planes' sum loses its low bits to the alignment with
// the large plane's products (Q6_K, K = 17408: 2.7e-7 in place of 1.1e-7).  The
// parts are scaled and added in f32 over at most EX_CPS chunks of 256, the K
// splits in f64.  Relative error against 64-bit sums (2-norm, 2048 outputs, K =
// 1024 .. 17408): N(0, 1) rows 0.67e-7 .. 1.0e-7, the scalar kernel 1.19e-7 ..
// 1.36e-7; N(0, 1) times exp(N(0, 4)) 0.8e-7 .. 1.42e-7 against 0.95e-7 ..
// 1.35e-7.  As for f32 dots the error is that of sums of the products' size,
// here of x with the integers as centred above: a weight that is zero or small
// because its offset cancels a code (4-bit formats) counts with the code.
//
// Block = 4 waves; a wave owns two 32-row column tiles of weight rows
// (gate/up: the gate and the up rows of the same 32 outputs) and streams them
// into registers a chunk ahead, half a chunk at a time, converting each
// 64-wide part once for the group's rows.  The rows' planes go half a chunk at
// a time into LDS by direct-to-LDS copies, the next half's while the current
// one computes.  Groups of R = 32 rows; up to 16 (8) rows the planes are
// stacked in two (one) 32-row operands and added in the epilogue, two thirds
// (one third) of the MFMAs.  No instance spills.  Bound at prompts: gate/up of
// 24576 x 4096 at M = 300 (280 us) keeps the VALU busy 42 % and the matrix cores
// 35 % of the time with two waves per SIMD, 33 % of a wave's time in waits; the
// conversion repeats per 32 rows.  At verify sizes: latency (one to six chunks
// a block, 20 % waits, 7 % MFMA).
#include "thq_dev.hpp"
#include "thq_kernels.hpp"

#include <type_traits>

namespace thq {
namespace {

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef uint32_t ex_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t ex_u32x2 __attribute__((ext_vector_type(2)));

constexpr float EX_UP = 2048.0f;  // planes 1 and 2 hold 2^11 of what they stand for
constexpr int EX_CPS = 6;         // chunks per K split (the accumulators' error, above)
constexpr int EX_LIST = 32;       // listed elements per row; more, and the whole row is dotted in f32
constexpr int EX_OUT = 8;         // outliers per row that do not set its scale

// an element that the planes do not hold
struct ExItem {
    int k;
    float x;
};

// ------------------------------------------------------------------ activation planes
__device__ __forceinline__ float dpp_quad(float v) {  // sum over each quad of lanes
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, false));
    return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, false));
}
__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
    const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}
// A block per row: its exponent E [M] (the planes hold x 2^-E), its planes
// P [3][M][K], its list (LC [M]: so many items of LK [M][EX_LIST] in ascending
// order, or -1 for the whole row), and for 4-bit weights SA [K/SB][mpad], the
// f32 sums of the scaled row's SB-wide pieces that a weight's offset
// multiplies (Q4_K: SB = 32, affine: 64).  E puts the row's largest magnitude
// into [2^14, 2^15), or the largest once up to EX_OUT outliers, each level
// more than 64 times the rest, are left out.  Listed: outliers, Inf, NaN, and
// what the planes would round.  Bound: latency (the row is read once, KEEP
// 8-wide pieces a thread kept in registers; 512 threads to K = 4096, 1024 past
// it: 5 rows of 12288 1 us less than with 512, 300 rows of 4096 3.5 us more).
template <int QT, int XP_T, int XP_KEEP>
__global__ __launch_bounds__(XP_T) void k_xplanes(const float* __restrict__ X, int K, int64_t plane, h8_t* __restrict__ P,
                                                  int* __restrict__ E, int* __restrict__ LC, ExItem* __restrict__ LK,
                                                  float* __restrict__ SA, int64_t mpad) {
    __shared__ float tops[2][XP_T / 64];
    __shared__ int counts[2][XP_T / 64];
    __shared__ int nlist;
    __shared__ ExItem list[EX_LIST];
    const int64_t row = blockIdx.x;
    const float* x = X + row * K;
    const int n8 = K >> 3, tid = threadIdx.x;
    if (tid == 0) nlist = 0;  // read after the first scan's barrier
    float v[XP_KEEP][8];
#pragma unroll
    for (int j = 0; j < XP_KEEP; ++j) {
        const int p = tid + j * XP_T;
        if (p < n8) load8(x + 8 * p, v[j]);
    }
    auto each = [&](auto&& f) {  // the thread's 8-wide pieces
#pragma unroll
        for (int j = 0; j < XP_KEEP; ++j) {
            const int p = tid + j * XP_T;
            if (p < n8) f(p, v[j]);
        }
        for (int p = tid + XP_KEEP * XP_T; p < n8; p += XP_T) {
            float a[8];
            load8(x + 8 * p, a);
            f(p, a);
        }
    };
    // A scan: this wave's largest magnitude below cut, and how many of its
    // values lie in [from, lim); then every wave's.  (Magnitudes compare as
    // their bits.)
    int turn = 0;
    auto wave_top = [&](float cut) {
        uint32_t m = 0;
        each([&](int, const float (&a)[8]) {
#pragma unroll
            for (int i = 0; i < 8; ++i) m = max(m, fabsf(a[i]) < cut ? __float_as_uint(fabsf(a[i])) : 0u);  // not NaN
        });
        m = max(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0xB1, 0xF, 0xF, false));
        m = max(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0x4E, 0xF, 0xF, false));
        m = max(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0x141, 0xF, 0xF, false));
        m = max(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0x140, 0xF, 0xF, false));
        uint32_t w = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) w = max(w, (uint32_t)__builtin_amdgcn_readlane((int)m, 16 * i));
        return __uint_as_float(w);
    };
    auto wave_count = [&](float from, float lim) {
        int c = 0;
        each([&](int, const float (&a)[8]) {
#pragma unroll
            for (int i = 0; i < 8; ++i) c += fabsf(a[i]) >= from && fabsf(a[i]) < lim;
        });
        c += __builtin_amdgcn_mov_dpp(c, 0xB1, 0xF, 0xF, false);
        c += __builtin_amdgcn_mov_dpp(c, 0x4E, 0xF, 0xF, false);
        c += __builtin_amdgcn_mov_dpp(c, 0x141, 0xF, 0xF, false);
        c += __builtin_amdgcn_mov_dpp(c, 0x140, 0xF, 0xF, false);
        int w = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) w += __builtin_amdgcn_readlane(c, 16 * i);
        return w;
    };
    auto meet = [&](float m, int c) {
        if ((tid & 63) == 0) {
            tops[turn][tid >> 6] = m;
            counts[turn][tid >> 6] = c;
        }
        __syncthreads();
    };
    float lim = INFINITY, top = 0.0f;  // the planes hold magnitudes below lim
    int crowd = 0;                     // of the wave that holds the top: values within 64 times of it
    {
        const float m = wave_top(lim);
        meet(m, m > 0.0f ? wave_count(m * 0.015625f, lim) : 0);
#pragma unroll
        for (int i = 0; i < XP_T / 64; ++i)
            if (tops[0][i] > top) {
                top = tops[0][i];
                crowd = counts[0][i];
            }
    }
    // no outliers where the top's own wave says so (most rows: no second scan)
    for (int left = EX_OUT; crowd <= EX_OUT && top > 0.0f;) {
        const float cut = top * 0.015625f;
        turn ^= 1;
        meet(wave_top(cut), wave_count(cut, lim));
        float rest = 0.0f;
        int count = 0;
#pragma unroll
        for (int i = 0; i < XP_T / 64; ++i) {
            rest = fmaxf(rest, tops[turn][i]);
            count += counts[turn][i];
        }
        if (count > left || rest == 0.0f) break;
        left -= count;  // at least one
        lim = cut;
        top = rest;
    }
    const int e = top > 0.0f ? __builtin_amdgcn_frexp_expf(top) - 15 : 0;
    if (tid == 0) E[row] = e;

    each([&](int p, const float (&a)[8]) {
        h8_t h0, h1, h2;
        float xs[8];
        bool lost[8], any = false;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const bool in = fabsf(a[i]) < lim;
            xs[i] = in ? __builtin_amdgcn_ldexpf(a[i], -e) : 0.0f;
            h0[i] = (_Float16)xs[i];
            const float r1 = (xs[i] - (float)h0[i]) * EX_UP;
            h1[i] = (_Float16)r1;
            const float r2 = r1 - (float)h1[i];
            h2[i] = (_Float16)r2;
            lost[i] = (float)h2[i] != r2 || (xs[i] == 0.0f && a[i] != 0.0f);  // not in, or too small
            any |= lost[i];
        }
        if (any) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (!lost[i]) continue;
                const int at = atomicAdd(&nlist, 1);
                if (at < EX_LIST) list[at] = ExItem{8 * p + i, a[i]};
                h0[i] = h1[i] = h2[i] = (_Float16)0.0f;
                xs[i] = 0.0f;
            }
        }
        P[(row * K >> 3) + p] = h0;
        P[((plane + row * K) >> 3) + p] = h1;
        P[((2 * plane + row * K) >> 3) + p] = h2;
        if constexpr (QT == 12 || QT == 13) {
            float s = ((xs[0] + xs[1]) + (xs[2] + xs[3])) + ((xs[4] + xs[5]) + (xs[6] + xs[7]));
            s = dpp_quad(s);  // 32 values (8-value pieces go to lanes in order; K % 256 == 0: whole waves' octets)
            if constexpr (QT == 13)
                s += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(s), 0x141, 0xF, 0xF, false));
            constexpr int W = QT == 13 ? 8 : 4;
            if ((p & (W - 1)) == 0) SA[(int64_t)(p / W) * mpad + row] = s;
        }
    });
    __syncthreads();
    const int n = nlist;
    if (tid == 0) LC[row] = n > EX_LIST ? -1 : n;
    if (n <= EX_LIST && tid < n) {  // in ascending order, whoever came first
        int rank = 0;
        for (int i = 0; i < n; ++i) rank += list[i].k < list[tid].k;
        LK[row * EX_LIST + rank] = list[tid];
    }
}

// ------------------------------------------------------------------ GEMM
__device__ __forceinline__ uint32_t ex_lds(const void* p) {
    return (uint32_t)(size_t)(__attribute__((address_space(3))) const void*)p;
}
// lane l's 16 bytes at base + voff land at LDS m0 + 16 l; untracked by the
// compiler (the kernel waits for them itself)
__device__ __forceinline__ void ex_dma16(uint32_t lds, const void* base, uint32_t voff) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(lds), "v"(voff), "s"(base) : "memory");
}
__device__ __forceinline__ f32x16_t ex_mfma(const h8_t& a, const h8_t& b, const f32x16_t& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ h2_t as_h2(uint32_t v) {
    h2_t r;
    __builtin_memcpy(&r, &v, 4);
    return r;
}
// eight codes (bytes of a, then of b, each below 256) -> f16 (code - off):
// 0x6400 | code is f16 1024 + code
__device__ __forceinline__ h8_t ex_codes(uint32_t a, uint32_t b, _Float16 off) {
    const uint32_t E = 0x64646464u;
    const _Float16 o = -((_Float16)1024.0f + off);
    const h2_t ov = {o, o};
    const h2_t r0 = as_h2(__builtin_amdgcn_perm(E, a, 0x04010400u)) + ov;
    const h2_t r1 = as_h2(__builtin_amdgcn_perm(E, a, 0x04030402u)) + ov;
    const h2_t r2 = as_h2(__builtin_amdgcn_perm(E, b, 0x04010400u)) + ov;
    const h2_t r3 = as_h2(__builtin_amdgcn_perm(E, b, 0x04030402u)) + ov;
    return h8_t{r0[0], r0[1], r1[0], r1[1], r2[0], r2[1], r3[0], r3[1]};
}

// weight (row, k) in f32, as k_gemv_generic forms it (rows with Inf / NaN only)
template <int QT>
__device__ __forceinline__ float ex_weight(const uint8_t* Wq, const uint8_t* Wa, int64_t row, int K, int64_t nrows,
                                           int k) {
    if constexpr (QT == 8) {
        const int nb = K >> 5, b = k >> 5, i = k & 31;
        const float d = f16_to_f32(reinterpret_cast<const uint16_t*>(Wa)[q8t_d(row, nb, b)]);
        return (float)reinterpret_cast<const int8_t*>(Wq)[q8t_q(row, nb, b, i >> 4) + (i & 15)] * d;
    } else if constexpr (QT == 14) {
        const Q6Layout L = q6k_layout(nrows, K);
        const int j = k >> 6, w = k & 63;
        const int code = ((Wq[row * (K / 2) + 32 * j + (w & 31)] >> (4 * (w >> 5))) & 15) |
                         (((Wq[L.qh + row * (K / 4) + 16 * j + (w & 15)] >> (2 * (w >> 4))) & 3) << 4);
        const float d = f16_to_f32(reinterpret_cast<const uint16_t*>(Wq + L.d)[row * (K / 256) + (j >> 2)]);
        const float ds = d * (float)reinterpret_cast<const int8_t*>(Wq + L.sc)[row * (K / 16) + (k >> 4)];
        return ds * (float)(code - 32);
    } else {
        const int nsb = K >> 8, s = k >> 8, i = k & 255, j = i >> 5, r = i & 31;
        const int q = (Wq[q4k_piece(row, nsb, s, r >> 4, j >> 1) + (r & 15)] >> (4 * (j & 1))) & 15;
        auto hd = [&](int p) { return *reinterpret_cast<const uint32_t*>(Wq + q4k_hdword(row, nsb, s, p)); };
        if constexpr (QT == 13) {
            const uint32_t hw = hd(j >> 1);
            return aff_scale(hw) * (float)q + aff_bias(hw);
        } else {
            const uint4 h = make_uint4(hd(0), hd(1), hd(2), hd(3));
            uint32_t sc, mm;
            q4k_hdr_sm(h, j, sc, mm);
            return q4k_hdr_d(h) * (float)sc * (float)q - q4k_hdr_dmin(h) * (float)mm;
        }
    }
}

// half a chunk (two 64-wide parts) of a lane's weight row
template <int QT>
struct ExHalf;
template <>
struct ExHalf<12> {
    ex_u32x4 w[2];  // the part's nibble piece g
};
template <>
struct ExHalf<13> {
    ex_u32x4 w[2];
};
template <>
struct ExHalf<8> {
    ex_u32x4 w[4];  // one 16-B half per 32-wide block
};
template <>
struct ExHalf<14> {
    ex_u32x2 ql[2][2], qh[2];
};
// the loads of R are waited for here
template <int QT>
__device__ __forceinline__ void ex_settle(ExHalf<QT>& R) {
    if constexpr (QT == 14) {
        asm volatile("" : "+v"(R.ql[0][0]), "+v"(R.ql[0][1]), "+v"(R.ql[1][0]), "+v"(R.ql[1][1]), "+v"(R.qh[0]),
                     "+v"(R.qh[1]));
    } else {
        asm volatile("" : "+v"(R.w[0]), "+v"(R.w[1]));
        if constexpr (QT == 8) asm volatile("" : "+v"(R.w[2]), "+v"(R.w[3]));
    }
}

// R: activation rows per group (8, 16 or 32).
// OUT: 0 = K-split partials f32 [split][M][nrows], 1 = f32, 2 = bf16
template <int QT, int R, bool GU, int OUT>
__global__ __launch_bounds__(256, 2) void k_gemm_ex(const uint8_t* Wq, const uint8_t* Wa, const _Float16* P,
                                                        const int* __restrict__ EX, const int* __restrict__ LC,
                                                        const ExItem* __restrict__ LK, const float* SA, int64_t mpad,
                                                        const float* X, void* __restrict__ Yv, int M, int K,
                                                        int64_t nout, int64_t up_off, int64_t nrows, int cps,
                                                        int tiles, int splits) {
    constexpr int NW = 4;                              // waves
    constexpr int VR = R == 8 ? 32 : 3 * R;            // operand rows in LDS (R = 8: plane 2 twice)
    constexpr int NP = (3 * R + 31) / 32;              // operands
    constexpr int NA = R == 32 ? 1 : NP;               // accumulators per tile
    constexpr int HB = VR * 256;                       // bytes per half chunk
    constexpr int NJ = VR / (4 * NW);                  // copy instructions per wave per half chunk
    constexpr int NSUM = QT == 12 ? 8 : QT == 13 ? 4 : 0;  // offset sums per chunk and row
    constexpr float DOWN = 1.0f / EX_UP;
    __shared__ __attribute__((aligned(16))) uint8_t xs[2 * HB];
    __shared__ __attribute__((aligned(16))) float sas[NSUM ? 2 * NSUM * R : 1];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 31, g = lane >> 5;
    int tile_i, split, group;
    {   // each XCD runs a contiguous range of (split, group) keys, weight tiles fastest
        const int nb = gridDim.x, b = blockIdx.x;
        const int q = (nb + 7) >> 3, tall = (nb & 7) ? (nb & 7) : 8;
        const int xcd = b & 7, local = b >> 3;
        const int v = xcd < tall ? xcd * q + local : tall * q + (xcd - tall) * (q - 1) + local;
        tile_i = v % tiles;
        split = (v / tiles) % splits;
        group = v / (tiles * splits);
    }
    const int nch = K >> 8;
    const int cb = split * cps;
    const int ce = cb + cps < nch ? cb + cps : nch;
    const int m0 = group * R;
    const int Mz = M - m0 < R ? M - m0 : R;

    int64_t orow[2], row[2];
    bool valid[2];
    uint32_t ow[2], oh[2], oq[2], od[2];
    const Q6Layout L6 = q6k_layout(nrows, K);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        orow[t] = GU ? (int64_t)tile_i * (32 * NW) + wave * 32 + n
                     : (int64_t)tile_i * (64 * NW) + wave * 64 + 32 * t + n;
        valid[t] = orow[t] < nout;
        row[t] = valid[t] ? (GU && t ? orow[t] + up_off : orow[t]) : 0;  // in-bounds reads
        oq[t] = od[t] = 0;
        if constexpr (QT == 8) {
            ow[t] = (uint32_t)q8t_q(row[t], K >> 5, 0, g);
            oh[t] = (uint32_t)q8t_d(row[t], K >> 5, 0) * 2u;
        } else if constexpr (QT == 14) {
            ow[t] = (uint32_t)(row[t] * (K / 2)) + 8u * g;
            oq[t] = (uint32_t)(L6.qh + row[t] * (K / 4)) + 8u * g;
            oh[t] = (uint32_t)(L6.sc + row[t] * (K / 16));
            od[t] = (uint32_t)(L6.d + row[t] * (K / 256) * 2);
        } else {
            ow[t] = (uint32_t)q4k_piece(row[t], nch, 0, g, 0);
            oh[t] = (uint32_t)q4k_hdword(row[t], nch, 0, 2 * g);
        }
    }
    auto wload = [&](ExHalf<QT> (&H)[2], int c, int hf) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            if constexpr (QT == 8) {
                const uint8_t* b = Wq + (int64_t)c * 8192 + hf * 4096;
#pragma unroll
                for (int j = 0; j < 4; ++j) H[t].w[j] = *reinterpret_cast<const ex_u32x4*>(b + ow[t] + j * 1024);
            } else if constexpr (QT == 14) {
                const uint8_t* b = Wq + (int64_t)c * 128 + hf * 64;
                const uint8_t* bh = Wq + (int64_t)c * 64 + hf * 32;
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    H[t].ql[u][0] = *reinterpret_cast<const ex_u32x2*>(b + ow[t] + u * 32);
                    H[t].ql[u][1] = *reinterpret_cast<const ex_u32x2*>(b + ow[t] + u * 32 + 16);
                    H[t].qh[u] = *reinterpret_cast<const ex_u32x2*>(bh + oq[t] + u * 16);
                }
            } else {
                const uint8_t* b = Wq + (int64_t)c * 64 + hf * 32;
                H[t].w[0] = *reinterpret_cast<const ex_u32x4*>(b + ow[t]);
                H[t].w[1] = *reinterpret_cast<const ex_u32x4*>(b + ow[t] + 16);
            }
        }
    };
    // a chunk's header: Q4_K / affine four dwords (loaded as two per lane half,
    // h[0..1], and met in hmeet), Q8_0 eight f16 scales, Q6_K sixteen int8 scales (and d)
    struct Hdr {
        ex_u32x4 h;
        uint32_t d;
    };
    auto hload = [&](Hdr (&H)[2], int c) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            H[t].d = 0;
            if constexpr (QT == 8) {
                H[t].h = *reinterpret_cast<const ex_u32x4*>(Wa + (int64_t)c * 512 + oh[t]);
            } else if constexpr (QT == 14) {
                H[t].h = *reinterpret_cast<const ex_u32x4*>(Wq + (int64_t)c * 16 + oh[t]);
                H[t].d = *reinterpret_cast<const uint16_t*>(Wq + (int64_t)c * 2 + od[t]);
            } else {
                const uint8_t* b = Wq + (int64_t)c * 64;
#pragma unroll
                for (int u = 0; u < 2; ++u) H[t].h[u] = *reinterpret_cast<const uint32_t*>(b + oh[t] + u * 16);
            }
        }
    };
    auto hmeet = [&](const Hdr& H) {
        Hdr r = H;
        if constexpr (QT == 12 || QT == 13) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const auto p = __builtin_amdgcn_permlane32_swap(H.h[u], H.h[u], false, false);
                r.h[u] = p[0];  // lane half 0's on both
                r.h[2 + u] = p[1];
            }
        }
        return r;
    };

    // copy j of a wave fills operand rows 4 (wave + NW j) .. + 3 of a half
    // chunk; the 16-B piece p of row r sits at slot p ^ (r & 15); rows past the
    // group copy its last
    uint32_t xoff[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int r = 4 * (wave + NW * j) + (lane >> 4);
        const int pl = r / R < 3 ? r / R : 2, rr = r % R < Mz ? r % R : Mz - 1;
        xoff[j] = ((uint32_t)(pl * M + m0 + rr) * (uint32_t)K) * 2u + 16u * (uint32_t)((lane & 15) ^ (r & 15));
    }
    const uint32_t xs0 = ex_lds(xs);
    auto xcopy = [&](int h, int b) {  // half chunk h into buffer b
        const uint8_t* xc = reinterpret_cast<const uint8_t*>(P) + (int64_t)h * 256;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            ex_dma16(__builtin_amdgcn_readfirstlane(xs0 + (uint32_t)(b * HB + (wave + NW * j) * 1024)), xc, xoff[j]);
    };
    auto aread = [&](int b, int op, int up, int k) {
        const int r = R == 16 && op ? 32 + (n & 15) : 32 * op + n;  // R = 16: plane 2 twice
        const int p = QT == 14 ? 8 * up + 2 * k + g : 8 * up + 2 * g + (k & 1) + 4 * (k >> 1);
        return *reinterpret_cast<const h8_t*>(xs + b * HB + r * 256 + 16 * (p ^ (n & 15)));
    };
    // offset sums of chunk c: thread tid holds (piece tid / R, row tid % R)
    auto sload = [&](int c) {
        if constexpr (!NSUM) return 0.0f;
        const int tid = threadIdx.x & (NSUM * R - 1), r = tid % R;
        const float v = SA[(int64_t)(NSUM * c + tid / R) * mpad + m0 + (r < Mz ? r : 0)];
        return r < Mz ? v : 0.0f;
    };
    auto sstore = [&](float v, int b) {
        if constexpr (NSUM) sas[b * NSUM * R + (threadIdx.x & (NSUM * R - 1))] = v;
    };
    f32x16_t acc[2][NA];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < NA; ++i) acc[t][i] = f32x16_t{};

    // part u (0..3) of a chunk, in half buffer b
    auto part = [&](const ExHalf<QT> (&W)[2], const Hdr (&H)[2], const float (&d)[2], int u, int b) {
        constexpr int SEG = QT == 14 ? 1 : (QT == 8 ? 2 : 4);  // 16-wide steps per scale
        constexpr int NSEG = 4 / SEG;
        constexpr bool SUM = NSEG > 1;  // a part's sum is added to acc once
        const uint32_t M4 = 0x0F0F0F0Fu;
        const int up = u & 1;
        constexpr bool TILES = !(R == 16 && NSEG > 1);  // tiles inside a scale's steps share A; else T would be 64 registers
        f32x16_t T[2][NA];
        h8_t A[NP][SEG];
#pragma unroll
        for (int q = 0; q < 2 * NSEG; ++q) {
            const int t = TILES ? q & 1 : q / NSEG, sg = TILES ? q >> 1 : q % NSEG;
            if (!TILES || t == 0) {
#pragma unroll
                for (int op = 0; op < NP; ++op)
#pragma unroll
                    for (int k = 0; k < SEG; ++k) A[op][k] = aread(b, op, up, SEG * sg + k);
            }
            h8_t B[SEG];
#pragma unroll
            for (int i = 0; i < SEG; ++i) {
                const int k = SEG * sg + i;
                if constexpr (QT == 8) {
                    const ex_u32x4 w = W[t].w[2 * up + (k >> 1)] ^ 0x80808080u;
                    B[i] = ex_codes(w[2 * (k & 1)], w[2 * (k & 1) + 1], (_Float16)128.0f);
                } else if constexpr (QT == 14) {
                    const ex_u32x2 ql = W[t].ql[up][k & 1], qh = W[t].qh[up];
                    uint32_t c[2];
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        c[j] = ((ql[j] >> (4 * (k >> 1))) & M4) | (((qh[j] >> (2 * k)) & 0x03030303u) << 4);
                    B[i] = ex_codes(c[0], c[1], (_Float16)32.0f);
                } else {
                    const ex_u32x4 w = W[t].w[up];
                    const int sh = k < 2 ? 0 : 4, c = 2 * (k & 1);
                    B[i] = ex_codes((w[c] >> sh) & M4, (w[c + 1] >> sh) & M4, (_Float16)8.0f);
                    if constexpr (QT == 12) B[i] *= (_Float16)(uint16_t)((H[t].h[u] >> (k < 2 ? 0 : 12)) & 63u);
                }
            }
            float ds;
            if constexpr (QT == 8)
                ds = f16_to_f32((uint16_t)(sg ? H[t].h[u] >> 16 : H[t].h[u]));
            else if constexpr (QT == 14)
                ds = d[t] * (float)(int8_t)(H[t].h[u] >> (8 * sg));
            else
                ds = QT == 12 ? d[t] : aff_scale(H[t].h[u]);
            f32x16_t D[NP == 3 ? 2 : NP] = {};
            if constexpr (R == 32) {  // plane 0, and planes 1 and 2 together
#pragma unroll
                for (int k = 0; k < SEG; ++k) {
                    D[1] = ex_mfma(A[1][k], B[k], D[1]);
                    D[0] = ex_mfma(A[0][k], B[k], D[0]);
                    D[1] = ex_mfma(A[2][k], B[k], D[1]);
                }
#pragma unroll
                for (int e = 0; e < 16; ++e) D[0][e] = __builtin_fmaf(DOWN, D[1][e], D[0][e]);
            } else {
#pragma unroll
                for (int op = 0; op < NP; ++op)
#pragma unroll
                    for (int k = 0; k < SEG; ++k) D[op] = ex_mfma(A[op][k], B[k], D[op]);
            }
#pragma unroll
            for (int a = 0; a < NA; ++a) {
                f32x16_t& S = SUM ? T[t][a] : acc[t][a];
#pragma unroll
                for (int e = 0; e < 16; ++e) S[e] = SUM && sg == 0 ? ds * D[a][e] : __builtin_fmaf(ds, D[a][e], S[e]);
                asm volatile("" : "+v"(S));  // now: left to the end, every D stays live
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (SUM) {
                if (sg != NSEG - 1) continue;
#pragma unroll
                for (int a = 0; a < NA; ++a) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[t][a][e] += T[t][a][e];
                    asm volatile("" : "+v"(acc[t][a]));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // 4-bit weights: sum_j c_j S_j of a chunk, added to acc once.  Q4_K: c_j =
    // 8 d sc_j - dmin m_j (as 8 d sum sc_j S_j - dmin sum m_j S_j the two large
    // sums' roundings add 1e-7), affine: c_j = 8 scale_j + bias_j.
    auto offset = [&](const Hdr& H, float d, float dm, int j, int half) {  // c_{j + half}, j even
        if constexpr (QT == 12) {
            const uint32_t w = H.h[j >> 1] >> (12 * half);
            return __builtin_fmaf(8.0f * d, (float)(w & 63u), -(dm * (float)((w >> 6) & 63u)));
        }
        const uint32_t w = half ? H.h[(j + 1) & 3] : H.h[j & 3];
        return __builtin_fmaf(8.0f, aff_scale(w), aff_bias(w));
    };
    auto offsets = [&](const Hdr (&H)[2], const float (&d)[2], const float (&dm)[2], int sb) {
        f32x16_t T[2] = {};
        if constexpr (R == 32) {  // on the f32 matrix cores: lane half g holds j + g
#pragma unroll
            for (int j = 0; j < NSUM; j += 2) {
                const float v = sas[(sb * NSUM + j + g) * R + n];
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    T[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, offset(H[t], d[t], dm[t], j, g), T[t], 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int j = 0; j < NSUM; ++j) {
                const float c[2] = {offset(H[0], d[0], dm[0], j & ~1, j & 1), offset(H[1], d[1], dm[1], j & ~1, j & 1)};
#pragma unroll
                for (int i = 0; i < R / 8; ++i) {
                    const f32x4_t v = *reinterpret_cast<const f32x4_t*>(&sas[(sb * NSUM + j) * R + 8 * i + 4 * g]);
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int e = 0; e < 4; ++e) T[t][4 * i + e] = __builtin_fmaf(c[t], v[e], T[t][4 * i + e]);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < R / 2; ++e) acc[t][0][e] += T[t][e];
    };

    ExHalf<QT> W[2][2];
    Hdr Hc[2], Hn[2];
    auto last = [&](int c) { return c < ce ? c : ce - 1; };
    xcopy(2 * cb, 0);
    hload(Hn, cb);
    wload(W[0], cb, 0);
    wload(W[1], cb, 1);
    sstore(sload(cb), 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // Half hf of chunk c computes from buffer hf while the next half's copies
    // go into the other one, read by no wave since the last barrier.  Its own
    // weights are settled before the copies go out (a wait for them behind the
    // copies, which the compiler does not count, would wait for the copies
    // too); the next chunk's are loaded into the same registers at its end and
    // stay in flight across the barrier, for the whole of the next half: its
    // vmcnt(0) is for them and for its copies.  Past the range they repeat the
    // last chunk.
    for (int c = cb; c < ce; ++c) {
        const int sb = (c - cb) & 1;
        float d[2], dm[2], sn = 0.0f;
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
#pragma unroll
            for (int t = 0; t < 2; ++t) ex_settle<QT>(W[hf][t]);
            if (hf == 0) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    if constexpr (QT == 8 || QT == 14)
                        asm volatile("" : "+v"(Hn[t].h), "+v"(Hn[t].d));
                    else
                        asm volatile("" : "+v"(Hn[t].h[0]), "+v"(Hn[t].h[1]));
                    Hc[t] = hmeet(Hn[t]);
                    d[t] = dm[t] = 0.0f;
                    if constexpr (QT == 12) {
                        d[t] = f16_to_f32((uint16_t)__builtin_amdgcn_perm(Hc[t].h[1], Hc[t].h[0], 0x0c0c0703u));
                        dm[t] = f16_to_f32((uint16_t)__builtin_amdgcn_perm(Hc[t].h[3], Hc[t].h[2], 0x0c0c0703u));
                    }
                    if constexpr (QT == 14) d[t] = f16_to_f32((uint16_t)Hc[t].d);
                }
            } else {
                sn = sload(last(c + 1));
            }
            __builtin_amdgcn_sched_barrier(0);
            const int next = 2 * c + hf + 1;
            xcopy(next < 2 * ce ? next : 2 * ce - 1, hf ^ 1);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            part(W[hf], Hc, d, 2 * hf, hf);
            part(W[hf], Hc, d, 2 * hf + 1, hf);
            if constexpr (NSUM)
                if (hf) offsets(Hc, d, dm, sb);
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (hf) sstore(sn, sb ^ 1);
            wload(W[hf], last(c + 1), hf);
            if (hf == 0) hload(Hn, last(c + 1));
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
        }
    }

    // acc[t][a][e] is operand row 8 (e / 4) + 4 g + e % 4; a row's value
    auto value = [&](int t, int e) {
        if constexpr (R == 32) return acc[t][0][e];
        if constexpr (R == 16) return __builtin_fmaf(DOWN, acc[t][0][(e + 8) & 15] + acc[t][NA - 1][e], acc[t][0][e]);
        return __builtin_fmaf(DOWN, acc[t][0][(e + 4) & 15] + acc[t][0][(e + 8) & 15], acc[t][0][e]);
    };
    constexpr int NT = GU && OUT != 0 ? 1 : 2;  // stored tiles (gate/up: one, the gate's)
    // The rows with listed elements, and of those the ones dotted whole: f32
    // dots over the split's K, summed in LDS (xs, no copy is in flight).  Here a
    // lane has one weight row, that of tile g.  The group's listed elements
    // that lie in the split are gathered first, row after row, so that the
    // loads of eight of them are in flight together (one row after the other
    // took 4 times as long as the GEMM at M = 300 with eight in each row).
    const int lc = lane < Mz ? LC[m0 + lane] : 0;
    const uint32_t some = (uint32_t)__ballot(lc != 0), whole = (uint32_t)__ballot(lc < 0);
    constexpr int COLS = 64 * NW;
    float* const side = reinterpret_cast<float*>(xs);  // [row][wave][tile][n]
    if (some) {
        struct Flat {
            int m;
            ExItem it;
        };
        Flat* const flat = reinterpret_cast<Flat*>(side + R * COLS);
        int* const counts = reinterpret_cast<int*>(flat + R * EX_LIST);
        static_assert(2 * HB >= R * COLS * 4 + R * EX_LIST * (int)sizeof(Flat) + R * 4, "all of it in xs");
        constexpr int PER = EX_LIST / 8;  // a row's elements over eight threads
        const int64_t rw = row[g];
        float* const own = side + wave * 64 + lane;
        for (uint32_t left = some; left; left &= left - 1) own[__builtin_ctz(left) * COLS] = 0.0f;
        const int tm = (int)threadIdx.x >> 3, ti = (int)threadIdx.x & 7;
        const int tn = tm < Mz ? LC[m0 + tm] : 0;
        ExItem it[PER];
        int found = 0;  // in the split, and (upper half) before it
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            it[q].k = -1;
            if (ti + 8 * q >= tn) continue;
            it[q] = LK[(int64_t)(m0 + tm) * EX_LIST + ti + 8 * q];
            found += it[q].k < cb * 256 ? 1 << 16 : it[q].k < ce * 256 ? 1 : 0;
        }
#pragma unroll
        for (int off = 1; off < 8; off <<= 1) found += __shfl_xor(found, off, 64);
        if (ti == 0 && tm < R) counts[tm] = found & 0xFFFF;
        __syncthreads();
        int total = 0, base = 0;
        for (int i = 0; i < R; ++i) {
            base = i == tm ? total : base;
            total += counts[i];
        }
#pragma unroll
        for (int q = 0; q < PER; ++q)
            if (it[q].k >= cb * 256 && it[q].k < ce * 256) flat[base + ti + 8 * q - (found >> 16)] = Flat{tm, it[q]};
        __syncthreads();
        for (int i = 0; i < total; i += 8) {
            Flat f[8];
            float w[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) f[j] = flat[i + j < total ? i + j : i];
#pragma unroll
            for (int j = 0; j < 8; ++j) w[j] = ex_weight<QT>(Wq, Wa, rw, K, nrows, f[j].it.k);
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (i + j < total) own[f[j].m * COLS] = __builtin_fmaf(f[j].it.x, w[j], own[f[j].m * COLS]);
        }
        if (whole) {
            for (int k = cb * 256; k < ce * 256; k += 32) {  // the weights once for all those rows
                float w[32];
#pragma unroll
                for (int i = 0; i < 32; ++i) w[i] = ex_weight<QT>(Wq, Wa, rw, K, nrows, k + i);
                for (uint32_t left = whole; left; left &= left - 1) {
                    const int m = __builtin_ctz(left);
                    const float4* x = reinterpret_cast<const float4*>(X + (int64_t)(m0 + m) * K + k);
                    float v = own[m * COLS];
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const float4 q = x[i];
                        v = __builtin_fmaf(q.x, w[4 * i], v);
                        v = __builtin_fmaf(q.y, w[4 * i + 1], v);
                        v = __builtin_fmaf(q.z, w[4 * i + 2], v);
                        v = __builtin_fmaf(q.w, w[4 * i + 3], v);
                    }
                    own[m * COLS] = v;
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int e = 0; e < R / 2; ++e) {
        const int m = 8 * (e >> 2) + 4 * g + (e & 3);
        if (m >= Mz) continue;
        const int ex = EX[m0 + m];
        float v[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) v[t] = ldexpf(value(t, e), ex);
        if ((some >> m) & 1) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const float f = side[m * COLS + wave * 64 + 32 * t + n];
                v[t] = (whole >> m) & 1 ? f : v[t] + f;
            }
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if (!valid[t]) continue;
            if constexpr (OUT == 0) {
                static_cast<float*>(Yv)[((int64_t)split * M + m0 + m) * nrows + row[t]] = v[t];
            } else {
                using YT = std::conditional_t<OUT == 1, float, bf16_t>;
                store_y<YT>(static_cast<YT*>(Yv) + (int64_t)(m0 + m) * nout + orow[t],
                            GU ? silu_mul(v[0], v[1]) : v[t]);
            }
        }
    }
}

// K-split partials P [S][M][ld] summed in split order in f64 (a chain of up to
// K / 256 f32 adds would round more than the splits themselves do), then the
// epilogue; four outputs per thread where rows are multiples of 4.
template <int V, bool GU, typename YT>
__global__ __launch_bounds__(64) void k_ex_reduce(const float* __restrict__ P, YT* __restrict__ Y, int M,
                                                   int64_t nout, int64_t up_off, int64_t ld, int S) {
    const int64_t i = ((int64_t)blockIdx.x * 64 + threadIdx.x) * V;
    if (i >= nout) return;
    const int64_t m = blockIdx.y, step = (int64_t)M * ld;
    typedef float vec_t __attribute__((ext_vector_type(V)));
    double a[V] = {}, u[V] = {};
    const float* p = P + m * ld + i;
    for (int s0 = 0; s0 < S; s0 += 8) {
        vec_t v[8], w[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) {  // eight loads in flight; past S the last again, not added
            const float* q = p + (int64_t)(s0 + s < S ? s0 + s : S - 1) * step;
            __builtin_memcpy(&v[s], q, sizeof(vec_t));
            if (GU) __builtin_memcpy(&w[s], q + up_off, sizeof(vec_t));
        }
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int j = 0; j < V; ++j) {
                a[j] += s0 + s < S ? (double)v[s][j] : 0.0;
                if (GU) u[j] += s0 + s < S ? (double)w[s][j] : 0.0;
            }
    }
#pragma unroll
    for (int j = 0; j < V; ++j)
        store_y<YT>(Y + m * nout + i + j, GU ? silu_mul((float)a[j], (float)u[j]) : (float)a[j]);
}

template <bool GU, typename YT>
hipError_t ex_reduce(const float* P, YT* y, int M, int64_t nout, int64_t up_off, int64_t ld, int S, hipStream_t s) {
    const bool v4 = !((nout | up_off | ld) & 3);
    const int64_t bx = (nout + (v4 ? 256 : 64) - 1) / (v4 ? 256 : 64);
    for (int m0 = 0; m0 < M; m0 += 65535) {  // grid.y limit: row chunks read and write at their own offset
        const dim3 grid((unsigned)bx, (unsigned)(M - m0 < 65535 ? M - m0 : 65535));
        if (v4)
            hipLaunchKernelGGL((k_ex_reduce<4, GU, YT>), grid, dim3(64), 0, s, P + m0 * ld, y + m0 * nout, M, nout,
                               up_off, ld, S);
        else
            hipLaunchKernelGGL((k_ex_reduce<1, GU, YT>), grid, dim3(64), 0, s, P + m0 * ld, y + m0 * nout, M, nout,
                               up_off, ld, S);
    }
    return hipGetLastError();
}

struct ExBufs {
    _Float16* P;
    int *E, *LC;
    ExItem* LK;
    float *SA, *part;
};
size_t ex_align(size_t b) { return (b + 255) & ~(size_t)255; }
// the buffers of a call at `base`, and the bytes of all but the partials
ExBufs ex_bufs(int qtype, int64_t M, int64_t K, void* base, size_t& bytes) {
    char* q = static_cast<char*>(base);
    auto take = [&](size_t n) {
        char* at = q;
        q += ex_align(n);
        return at;
    };
    ExBufs b;
    b.P = reinterpret_cast<_Float16*>(take((size_t)M * K * 6));
    b.E = reinterpret_cast<int*>(take((size_t)M * 4));
    b.LC = reinterpret_cast<int*>(take((size_t)M * 4));
    b.LK = reinterpret_cast<ExItem*>(take((size_t)M * EX_LIST * sizeof(ExItem)));
    const int64_t pieces = qtype == 12 ? K / 32 : qtype == 13 ? K / 64 : 0;
    b.SA = reinterpret_cast<float*>(take((size_t)pieces * ((M + 63) / 64 * 64) * 4));
    b.part = reinterpret_cast<float*>(q);
    bytes = (size_t)(q - static_cast<char*>(base));
    return b;
}

template <int QT, int R, bool GU>
hipError_t run_ex(const ExPlan& p, const WeightView& w, const float* x, const ExBufs& b, void* y, bool yf32, int M,
                  int64_t nout, int64_t up_off, hipStream_t s) {
    const int64_t per = GU ? 128 : 256;
    const int64_t tiles = (nout + per - 1) / per;
    const int64_t nb = tiles * p.splits * p.groups;
    if (nb > 0x7FFFFFFF) return hipErrorInvalidValue;
    const int K = (int)w.K;
    const int64_t mpad = (int64_t)(M + 63) / 64 * 64;
    const auto planes = K <= 4096 ? k_xplanes<QT, 512, 1> : k_xplanes<QT, 1024, 2>;
    hipLaunchKernelGGL(planes, dim3(M), dim3(K <= 4096 ? 512 : 1024), 0, s, x, K, (int64_t)M * K,
                       reinterpret_cast<h8_t*>(b.P), b.E, b.LC, b.LK, b.SA, mpad);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const dim3 grid((unsigned)nb), block(256);
#define THQ_EX(OUT_, Y_)                                                                                              \
    hipLaunchKernelGGL((k_gemm_ex<QT, R, GU, OUT_>), grid, block, 0, s, w.q, w.aux, b.P, b.E, b.LC, b.LK, b.SA, mpad, \
                       x, Y_, M, K, nout, up_off, w.N, p.cps, (int)tiles, p.splits)
    if (p.splits > 1) {
        THQ_EX(0, (void*)b.part);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
        return launch_ex_reduce(b.part, y, yf32, GU, M, nout, up_off, w.N, p.splits, s);
    }
    if (yf32)
        THQ_EX(1, y);
    else
        THQ_EX(2, y);
#undef THQ_EX
    return hipGetLastError();
}

}  // namespace

hipError_t launch_ex_reduce(const float* P, void* y, bool yf32, bool gu, int M, int64_t nout, int64_t up_off,
                            int64_t ld, int S, hipStream_t s) {
    if (yf32)
        return gu ? ex_reduce<true, float>(P, static_cast<float*>(y), M, nout, up_off, ld, S, s)
                  : ex_reduce<false, float>(P, static_cast<float*>(y), M, nout, up_off, ld, S, s);
    return gu ? ex_reduce<true, bf16_t>(P, static_cast<bf16_t*>(y), M, nout, up_off, ld, S, s)
              : ex_reduce<false, bf16_t>(P, static_cast<bf16_t*>(y), M, nout, up_off, ld, S, s);
}

ExPlan plan_gemm_ex(int qtype, int64_t M, int64_t N, int64_t K, bool gu, int cus) {
    ExPlan p;
    if (!(qtype == 8 || qtype == 12 || qtype == 13 || qtype == 14)) return p;
    if (M < 1 || N < 1 || K < 256 || K % 256 || K > (int64_t)1 << 30 || (gu && N % 2)) return p;
    // 32-bit offsets: the weight planes and the activation planes below 4 GiB
    const uint64_t lim = 1ull << 32;
    const uint64_t plane = qtype == 8 ? (uint64_t)q8t_q_bytes(N, K)
                                      : (qtype == 14 ? (uint64_t)q6k_layout(N, K).total
                                                     : (uint64_t)((N + 3) / 4) * (uint64_t)(K / 256) * 576u);
    if (plane >= lim || (uint64_t)M * (uint64_t)K * 6u >= lim) return p;
    // Two blocks per CU.  Cost of a K split count: rounds of resident blocks
    // x chunks (and one of prologue) x a chunk's weight (2.4 us stacked, 4.0 us
    // with 32 rows: less than a chunk takes with both blocks there, but dearer
    // chunks, 3.0 and 8.0, plan more splits at 300 rows: the 4096 / 12288 MLP 487
    // against 465 us), plus the partials' round trip at 4 TB/s.
    const int64_t nch = K / 256, nout = gu ? N / 2 : N, cu = cus > 0 ? cus : 256;
    p.rows = M <= 8 ? 8 : M <= 16 ? 16 : 32;
    p.groups = (int)((M + p.rows - 1) / p.rows);
    const int64_t per = gu ? 128 : 256, tiles = (nout + per - 1) / per;
    const int64_t smin = (nch + EX_CPS - 1) / EX_CPS;
    double best = 1e30;
    for (int64_t s = smin; s <= nch && s <= smin + 32; ++s) {
        const int64_t cps = (nch + s - 1) / s;
        const int64_t rounds = (tiles * p.groups * s + 2 * cu - 1) / (2 * cu);
        const double t = (double)rounds * ((double)cps + 1.0) * (p.rows < 32 ? 2.4 : 4.0) +
                         (s > 1 ? 2.0 + (double)s * (double)M * (double)N * 8.0 / 4.0e6 : 0.0);
        if (t < best - 1e-9) {
            best = t;
            p.cps = (int)cps;
            p.splits = (int)((nch + cps - 1) / cps);
        }
    }
    (void)ex_bufs(qtype, M, K, nullptr, p.workspace_bytes);
    if (p.splits > 1) p.workspace_bytes += (size_t)p.splits * (size_t)M * (size_t)N * 4u;
    return p;
}

hipError_t launch_gemm_ex(const ExPlan& p, const WeightView& w, const float* x, void* y, bool yf32, bool gu, int M,
                          int64_t nout, int64_t up_off, void* ws, hipStream_t s) {
    if (p.groups < 1 || p.splits < 1 || M < 1 || !ws) return hipErrorInvalidValue;
    size_t bytes;
    const ExBufs b = ex_bufs(w.qtype, M, w.K, ws, bytes);
#define THQ_EXG(QT_, R_)                                                           \
    (gu ? run_ex<QT_, R_, true>(p, w, x, b, y, yf32, M, nout, up_off, s)           \
        : run_ex<QT_, R_, false>(p, w, x, b, y, yf32, M, nout, up_off, s))
#define THQ_EXQ(QT_) (p.rows == 8 ? THQ_EXG(QT_, 8) : p.rows == 16 ? THQ_EXG(QT_, 16) : THQ_EXG(QT_, 32))
    switch (w.qtype) {
        case 8: return THQ_EXQ(8);
        case 12: return THQ_EXQ(12);
        case 13: return THQ_EXQ(13);
        case 14: return THQ_EXQ(14);
    }
#undef THQ_EXQ
#undef THQ_EXG
    return hipErrorInvalidValue;
}

}  // namespace thq
