// k_gemm_ex.hip — f32 activations of any row count past 1 on the f16 matrix
// cores, exact weights, no less precise than f32 dots.
//
// Role: candle's f32 QMatMul::forward on GGUF models (engine/src/
// model.rs:551-562) over prompts and verify steps.  Before it, every f32 call
// with M > 1 ran k_gemv_generic: scalar f32 dots, the weight dequantized again
// for every 8 rows (Q4_K gate/up + down of 4096 / 12288 at M = 300: 19.2 ms,
// now 0.41 ms; a decoder layer at M = 5: 424 us, now 102 us).
//
// Activations (k_xplanes, one launch per call): each row is scaled by a power
// of two so that its largest magnitude lies in [2^14, 2^15), then written as
// two f16 planes, x0 = f16(x) and x1 = f16(x - x0): x0 + x1 is x to 2^-24 of
// it, or to 2^-40 of the row's largest value where x1 is subnormal (the
// matrix cores do not flush it).  The weights' integers are exact in f16
// (Q4_K: sc (q - 8), at most 504; affine: q - 8; Q8_0: q; Q6_K: code - 32),
// so each product is exact in f32.
//
// Sums: a 64-wide part (Q8_0: each 32-wide block of it, Q6_K: each 16-wide
// group) is summed by the matrix core from zero, each plane by itself: a
// chain that starts from the small plane's sum loses its low bits to the
// alignment with the large plane's products (Q6_K, K = 17408: 2.7e-7 in
// place of 1.1e-7).  The parts are scaled and added in f32 over at most
// EX_CPS chunks of 256, the K splits in f64.  Relative error against 64-bit
// sums (N(0, 1) rows, 2048 outputs, K = 1024 .. 17408): 0.8e-7 .. 1.33e-7; the
// scalar kernel's is 1.18e-7 .. 1.37e-7, which fixes EX_CPS.
//
// Block = 4 waves; a wave owns two 32-row column tiles of weight rows
// (gate/up: the gate and the up rows of the same 32 outputs) and streams them
// into registers half a chunk ahead, converting each 64-wide part once for
// the group's rows.  The rows' planes go chunk by chunk into LDS by
// direct-to-LDS copies, the next chunk's while the current one computes; one
// A operand read feeds two MFMAs.  Groups of 32 rows; up to 16 rows (ST) the
// two planes are stacked in one 32-row operand and added in the epilogue,
// half the MFMAs.  Groups of 64 rows spill or leave one wave per SIMD (gate/up
// of the MLP above: 335 .. 358 against 268 .. 296 us).  Bound: VALU (the
// conversion, ~2 instructions per weight and 32 rows) at prompts, the weight
// stream's latency at verify sizes.
#include "thq_dev.hpp"
#include "thq_kernels.hpp"

#include <climits>
#include <type_traits>

namespace thq {
namespace {

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef uint32_t ex_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t ex_u32x2 __attribute__((ext_vector_type(2)));

constexpr int EX_NONFINITE = INT_MIN;  // a row's exponent slot: the row holds Inf or NaN
constexpr int EX_CPS = 6;              // chunks per K split (the accumulators' error, above)

// ------------------------------------------------------------------ activation planes
__device__ __forceinline__ float dpp_quad(float v) {  // sum over each quad of lanes
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, false));
    return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, false));
}
__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
    const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}
// A block per row: the row's largest magnitude, then its planes P [2][M][K],
// its exponent E [M], and the sums the offset of a 4-bit weight multiplies:
// Q4_K: SS [M][K/256][2][8] f16, 2^-6 of the scaled row's 32-wide sums in two
// pieces; affine: SA [K/64][mpad] f32 64-wide sums.  A row that holds Inf or
// NaN gets zero planes and EX_NONFINITE (k_gemm_ex dots it in f32).
// Bound: latency (the row is read once, kept in registers up to K = 16384).
constexpr int XP_T = 512, XP_KEEP = 4;
template <int QT>
__global__ __launch_bounds__(XP_T) void k_xplanes(const float* __restrict__ X, int K, int64_t plane, h8_t* __restrict__ P,
                                                  int* __restrict__ E, _Float16* __restrict__ SS,
                                                  float* __restrict__ SA, int64_t mpad) {
    __shared__ float red[XP_T / 64];
    const int64_t row = blockIdx.x;
    const float* x = X + row * K;
    const int n8 = K >> 3, tid = threadIdx.x;
    float v[XP_KEEP][8];
    float mx = 0.0f;
    bool bad = false;
    auto scan = [&](const float (&a)[8]) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float m = fabsf(a[i]);
            bad |= !(m <= 3.402823466e+38f);
            mx = fmaxf(mx, m);
        }
    };
#pragma unroll
    for (int j = 0; j < XP_KEEP; ++j) {
        const int p = tid + j * XP_T;
        if (p < n8) {
            load8(x + 8 * p, v[j]);
            scan(v[j]);
        }
    }
    for (int p = tid + XP_KEEP * XP_T; p < n8; p += XP_T) {
        float a[8];
        load8(x + 8 * p, a);
        scan(a);
    }
    if (bad) mx = INFINITY;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = red[0];
#pragma unroll
    for (int i = 1; i < XP_T / 64; ++i) mx = fmaxf(mx, red[i]);
    const bool fin = mx < INFINITY;
    const int e = fin && mx > 0.0f ? ilogbf(mx) - 14 : 0;
    if (tid == 0) E[row] = fin ? e : EX_NONFINITE;

    auto emit = [&](int p, const float (&a)[8]) {
        h8_t h0, h1;
        float s = 0.0f, xs[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            xs[i] = fin ? ldexpf(a[i], -e) : 0.0f;
            h0[i] = (_Float16)xs[i];
            h1[i] = (_Float16)(xs[i] - (float)h0[i]);
        }
        P[(row * K >> 3) + p] = h0;
        P[((plane + row * K) >> 3) + p] = h1;
        if constexpr (QT == 12 || QT == 13) {
            s = ((xs[0] + xs[1]) + (xs[2] + xs[3])) + ((xs[4] + xs[5]) + (xs[6] + xs[7]));
            s = dpp_quad(s);  // 32 values (8-value pieces go to lanes in order; K % 256 == 0: whole waves' octets)
            if constexpr (QT == 12) {
                if ((p & 3) == 0) {
                    const int j = p >> 2;
                    const float ss = s * 0.015625f;
                    const _Float16 s0 = (_Float16)ss;
                    _Float16* d = SS + (row * (K >> 8) + (j >> 3)) * 16 + (j & 7);
                    d[0] = s0;
                    d[8] = (_Float16)(ss - (float)s0);
                }
            } else {
                s += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(s), 0x141, 0xF, 0xF, false));
                if ((p & 7) == 0) SA[(int64_t)(p >> 3) * mpad + row] = s;
            }
        }
    };
#pragma unroll
    for (int j = 0; j < XP_KEEP; ++j) {
        const int p = tid + j * XP_T;
        if (p < n8) emit(p, v[j]);
    }
    for (int p = tid + XP_KEEP * XP_T; p < n8; p += XP_T) {
        float a[8];
        load8(x + 8 * p, a);
        emit(p, a);
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

// OUT: 0 = K-split partials f32 [split][M][nrows], 1 = f32, 2 = bf16
template <int QT, bool ST, bool GU, int OUT>
__global__ __launch_bounds__(256, 2) void k_gemm_ex(const uint8_t* Wq, const uint8_t* Wa, const _Float16* P,
                                                        const int* __restrict__ EX, const _Float16* SS,
                                                        const float* SA, int64_t mpad, const float* X,
                                                        void* __restrict__ Yv, int M, int K, int64_t nout,
                                                        int64_t up_off, int64_t nrows, int cps, int tiles,
                                                        int splits) {
    constexpr int NW = 4;                      // waves
    constexpr int NP = ST ? 1 : 2;             // operands per 32 rows
    constexpr int MP = ST ? 16 : 32;           // activation rows per group
    constexpr int VR = ST ? 32 : NP * MP;      // operand rows in LDS
    constexpr int XB = VR * 512;               // bytes per buffer
    constexpr int NJ = VR / (2 * NW);          // copy instructions per wave per chunk
    constexpr int SR = 32;                     // rows of the affine sums in LDS
    constexpr bool AFF = QT == 13;
    __shared__ __attribute__((aligned(16))) uint8_t xs[2 * XB];
    __shared__ float sas[AFF ? 2 * 4 * SR : 1];

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
    const int m0 = group * MP;
    const int Mz = M - m0 < MP ? M - m0 : MP;

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
            oh[t] = (uint32_t)q4k_hdword(row[t], nch, 0, 0);
        }
    }
    auto wload = [&](ExHalf<QT> (&R)[2], int c, int hf) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            if constexpr (QT == 8) {
                const uint8_t* b = Wq + (int64_t)c * 8192 + hf * 4096;
#pragma unroll
                for (int j = 0; j < 4; ++j) R[t].w[j] = *reinterpret_cast<const ex_u32x4*>(b + ow[t] + j * 1024);
            } else if constexpr (QT == 14) {
                const uint8_t* b = Wq + (int64_t)c * 128 + hf * 64;
                const uint8_t* bh = Wq + (int64_t)c * 64 + hf * 32;
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    R[t].ql[u][0] = *reinterpret_cast<const ex_u32x2*>(b + ow[t] + u * 32);
                    R[t].ql[u][1] = *reinterpret_cast<const ex_u32x2*>(b + ow[t] + u * 32 + 16);
                    R[t].qh[u] = *reinterpret_cast<const ex_u32x2*>(bh + oq[t] + u * 16);
                }
            } else {
                const uint8_t* b = Wq + (int64_t)c * 64 + hf * 32;
                R[t].w[0] = *reinterpret_cast<const ex_u32x4*>(b + ow[t]);
                R[t].w[1] = *reinterpret_cast<const ex_u32x4*>(b + ow[t] + 16);
            }
        }
    };
    // a chunk's header: Q4_K / affine four dwords, Q8_0 eight f16 scales, Q6_K sixteen int8 scales (and d)
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
                for (int u = 0; u < 4; ++u) H[t].h[u] = *reinterpret_cast<const uint32_t*>(b + oh[t] + u * 16);
            }
        }
    };

    // copy j of a wave fills operand rows 2 (wave + NW j) and the next; the
    // 16-B piece p of row r sits at slot p ^ (r & 15); rows past the group copy its last
    uint32_t xoff[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int r = 2 * (wave + NW * j) + (lane >> 5);
        const int pl = r / MP, rr = r % MP < Mz ? r % MP : Mz - 1;
        xoff[j] = ((uint32_t)(pl * M + m0 + rr) * (uint32_t)K) * 2u + 16u * (uint32_t)((lane & 31) ^ (r & 15));
    }
    const uint32_t xs0 = ex_lds(xs);
    auto xcopy = [&](int c, int b) {
        const uint8_t* xc = reinterpret_cast<const uint8_t*>(P) + (int64_t)c * 512;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            ex_dma16(__builtin_amdgcn_readfirstlane(xs0 + (uint32_t)(b * XB + (wave + NW * j) * 1024)), xc, xoff[j]);
    };
    auto aread = [&](const uint8_t* xb, int pl, int u, int k) {
        const int p = QT == 14 ? 8 * u + 2 * k + g : 8 * u + 2 * g + (k & 1) + 4 * (k >> 1);
        return *reinterpret_cast<const h8_t*>(xb + (pl * MP + n) * 512 + 16 * (p ^ (n & 15)));
    };
    // affine sums of chunk c: thread tid holds (64-wide part tid / SR, row tid % SR)
    auto sload = [&](int c) {
        if constexpr (!AFF) return 0.0f;
        const int tid = threadIdx.x & (4 * SR - 1), r = tid % SR;
        const float v = SA[(int64_t)(4 * c + tid / SR) * mpad + m0 + (r < Mz ? r : 0)];
        return r < Mz ? v : 0.0f;
    };
    auto sstore = [&](float v, int b) {
        if constexpr (AFF) sas[b * 4 * SR + (threadIdx.x & (4 * SR - 1))] = v;
    };

    f32x16_t acc[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) acc[t] = f32x16_t{};

    // one 64-wide part u (0..3) of the chunk in LDS buffer b
    auto part = [&](const ExHalf<QT> (&R)[2], const Hdr (&H)[2], const float (&d)[2], int u, int b) {
        constexpr int SEG = QT == 14 ? 1 : (QT == 8 ? 2 : 4);  // 16-wide steps per scale
        constexpr int NSEG = 4 / SEG;
        const uint8_t* xb = xs + b * XB;
        const uint32_t M4 = 0x0F0F0F0Fu;
        const int up = u & 1;
        h8_t B[2][4];
        float ds[2][NSEG];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if constexpr (QT == 8) {
                    const ex_u32x4 q = R[t].w[2 * up + (k >> 1)] ^ 0x80808080u;
                    B[t][k] = ex_codes(q[2 * (k & 1)], q[2 * (k & 1) + 1], (_Float16)128.0f);
                } else if constexpr (QT == 14) {
                    const ex_u32x2 ql = R[t].ql[up][k & 1], qh = R[t].qh[up];
                    uint32_t c[2];
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        c[i] = ((ql[i] >> (4 * (k >> 1))) & M4) | (((qh[i] >> (2 * k)) & 0x03030303u) << 4);
                    B[t][k] = ex_codes(c[0], c[1], (_Float16)32.0f);
                } else {
                    const ex_u32x4 q = R[t].w[up];
                    const int sh = k < 2 ? 0 : 4, i = 2 * (k & 1);
                    B[t][k] = ex_codes((q[i] >> sh) & M4, (q[i + 1] >> sh) & M4, (_Float16)8.0f);
                    if constexpr (QT == 12) B[t][k] *= (_Float16)(uint16_t)((H[t].h[u] >> (k < 2 ? 0 : 12)) & 63u);
                }
            }
#pragma unroll
            for (int sg = 0; sg < NSEG; ++sg) {
                if constexpr (QT == 8) {
                    ds[t][sg] = f16_to_f32((uint16_t)(sg ? H[t].h[u] >> 16 : H[t].h[u]));
                } else if constexpr (QT == 14) {
                    ds[t][sg] = d[t] * (float)(int8_t)(H[t].h[u] >> (8 * sg));
                } else {
                    ds[t][sg] = QT == 12 ? d[t] : aff_scale(H[t].h[u]);
                }
            }
        }
        h8_t A[NP][4];
#pragma unroll
        for (int pl = 0; pl < NP; ++pl)
#pragma unroll
            for (int k = 0; k < 4; ++k) A[pl][k] = aread(xb, pl, u, k);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            f32x16_t T;  // the part's sum, added to acc once
#pragma unroll
            for (int sg = 0; sg < NSEG; ++sg) {
                f32x16_t D = {}, D1 = {};
#pragma unroll
                for (int k = 0; k < SEG; ++k) {
                    if constexpr (NP == 2) D1 = ex_mfma(A[1][SEG * sg + k], B[t][SEG * sg + k], D1);
                    D = ex_mfma(A[0][SEG * sg + k], B[t][SEG * sg + k], D);
                }
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const float v = NP == 2 ? D[e] + D1[e] : D[e];
                    if constexpr (NSEG == 1 && !AFF)
                        acc[t][e] = __builtin_fmaf(ds[t][0], v, acc[t][e]);
                    else
                        T[e] = sg ? __builtin_fmaf(ds[t][sg], v, T[e]) : ds[t][0] * v;
                }
            }
            if constexpr (AFF) {
                // (bias + 8 scale) x the part's sum of each row
                const float cf = __builtin_fmaf(8.0f, ds[t][0], aff_bias(H[t].h[u]));
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const f32x4_t v =
                        *reinterpret_cast<const f32x4_t*>(&sas[(b * 4 + u) * SR + 8 * i + 4 * g]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) T[4 * i + e] = __builtin_fmaf(cf, v[e], T[4 * i + e]);
                }
            }
            if constexpr (NSEG > 1 || AFF) {
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[t][e] += T[e];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // Q4_K: sum_j c_j S_j of a chunk, c_j = 8 d sc_j - dmin m_j: two MFMAs per
    // tile, the sums' two pieces (lane half g holds piece g) by c_j's two, c
    // scaled by a power of two into f16's range.  (As 8 d sum sc_j S_j - dmin
    // sum m_j S_j the two large sums' roundings add 1e-7.)
    auto offsets = [&](const Hdr (&H)[2], const float (&d)[2], const float (&dm)[2], const h8_t& As) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            float cj[8], mx = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t w = H[t].h[j >> 1] >> (12 * (j & 1));
                cj[j] = __builtin_fmaf(8.0f * d[t], (float)(w & 63u), -(dm[t] * (float)((w >> 6) & 63u)));
                mx = fmaxf(mx, fabsf(cj[j]));
            }
            const int ce_ = __builtin_amdgcn_frexp_expf(mx) - 14;
            const float up = __builtin_amdgcn_ldexpf(1.0f, -ce_), down = __builtin_amdgcn_ldexpf(64.0f, ce_);
            h8_t C0, C1;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float v = cj[j] * up;
                C0[j] = (_Float16)v;
                C1[j] = (_Float16)(v - (float)C0[j]);
            }
            const f32x16_t a = ex_mfma(As, C0, ex_mfma(As, C1, f32x16_t{}));
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[t][e] = __builtin_fmaf(down, a[e], acc[t][e]);
        }
    };

    ExHalf<QT> R0[2], R1[2];
    Hdr Hc[2], Hn[2];
    auto last = [&](int c) { return c < ce ? c : ce - 1; };
    xcopy(cb, 0);
    hload(Hn, cb);
    wload(R0, cb, 0);
    wload(R1, cb, 1);
    sstore(sload(cb), 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // step c (buffer b): chunk c + 1's copies go out first (buffer b ^ 1, read
    // by no wave since the last barrier); each half's weights are loaded again
    // for chunk c + 1 as soon as it is consumed and stay in flight across the
    // barrier: loads complete in order and the first half's and the header's
    // are ten or more instructions behind the copies, so vmcnt(10) waits for
    // the copies only.  Past the range they repeat the last chunk.
    for (int c = cb; c < ce; ++c) {
        const int b = (c - cb) & 1;
        float d[2], dm[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            Hc[t] = Hn[t];
            d[t] = dm[t] = 0.0f;
            if constexpr (QT == 12) {
                d[t] = f16_to_f32((uint16_t)__builtin_amdgcn_perm(Hc[t].h[1], Hc[t].h[0], 0x0c0c0703u));
                dm[t] = f16_to_f32((uint16_t)__builtin_amdgcn_perm(Hc[t].h[3], Hc[t].h[2], 0x0c0c0703u));
            }
            if constexpr (QT == 14) d[t] = f16_to_f32((uint16_t)Hc[t].d);
        }
        xcopy(last(c + 1), b ^ 1);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const float sn = sload(last(c + 1));
        h8_t As = {};
        if constexpr (QT == 12) {
            As = *reinterpret_cast<const h8_t*>(SS + (((int64_t)(m0 + (n < Mz ? n : 0)) * nch + c) * 2 + g) * 8);
            if (n >= Mz) As = h8_t{};
        }
        part(R0, Hc, d, 0, b);
        part(R0, Hc, d, 1, b);
        __builtin_amdgcn_sched_barrier(0);
        wload(R0, last(c + 1), 0);
        hload(Hn, last(c + 1));
        __builtin_amdgcn_sched_barrier(0);
        part(R1, Hc, d, 2, b);
        part(R1, Hc, d, 3, b);
        if constexpr (QT == 12) offsets(Hc, d, dm, As);
        sstore(sn, b ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
        wload(R1, last(c + 1), 1);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
    }

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no copy may land in LDS after the block ends
    // epilogue: acc[t][e] is operand row 8 (e / 4) + 4 g + e % 4
    auto put = [&](int m, int t, float v, float vu) {
        if constexpr (OUT == 0) {
            static_cast<float*>(Yv)[((int64_t)split * M + m0 + m) * nrows + row[t]] = v;
        } else {
            using YT = std::conditional_t<OUT == 1, float, bf16_t>;
            store_y<YT>(static_cast<YT*>(Yv) + (int64_t)(m0 + m) * nout + orow[t], GU ? silu_mul(v, vu) : v);
        }
    };
    constexpr int NT = GU && OUT != 0 ? 1 : 2;  // stored tiles (gate/up: one, the gate's)
#pragma unroll
    for (int e = 0; e < (ST ? 8 : 16); ++e) {
        const int m = 8 * (e >> 2) + 4 * g + (e & 3);
        if (m >= Mz) continue;
        const int ex = EX[m0 + m];
        if (ex == EX_NONFINITE) continue;
        float v[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) v[t] = ldexpf(ST ? acc[t][e] + acc[t][(e + 8) & 15] : acc[t][e], ex);
#pragma unroll
        for (int t = 0; t < NT; ++t)
            if (valid[t]) put(m, t, v[t], v[1]);
    }
    // rows with Inf / NaN: f32 dots over the split's K (lane half g takes every other column)
    for (int m = 0; m < Mz; ++m) {
        if (EX[m0 + m] != EX_NONFINITE) continue;
        float v[2] = {0.0f, 0.0f};
#pragma clang loop unroll(disable)
        for (int k = cb * 256 + g; k < ce * 256; k += 2) {
            const float x = load_x<float>(X + (int64_t)(m0 + m) * K + k);
#pragma unroll
            for (int t = 0; t < 2; ++t) v[t] = __builtin_fmaf(x, ex_weight<QT>(Wq, Wa, row[t], K, nrows, k), v[t]);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) v[t] += __shfl_xor(v[t], 32, 64);
#pragma unroll
        for (int t = 0; t < NT; ++t)
            if (g == 0 && valid[t]) put(m, t, v[t], v[1]);
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
    int* E;
    _Float16* SS;
    float* SA;
    float* part;
};
size_t ex_align(size_t b) { return (b + 255) & ~(size_t)255; }
size_t ex_planes_bytes(int64_t M, int64_t K) { return ex_align((size_t)M * K * 4); }
size_t ex_sums_bytes(int qtype, int64_t M, int64_t K) {
    if (qtype == 12) return ex_align((size_t)M * (K / 256) * 32);
    if (qtype == 13) return ex_align((size_t)(K / 64) * ((M + 63) / 64 * 64) * 4);
    return 0;
}

template <int QT, bool ST, bool GU>
hipError_t run_ex(const ExPlan& p, const WeightView& w, const float* x, const ExBufs& b, void* y, bool yf32, int M,
                  int64_t nout, int64_t up_off, hipStream_t s) {
    const int64_t per = GU ? 128 : 256;
    const int64_t tiles = (nout + per - 1) / per;
    const int64_t nb = tiles * p.splits * p.groups;
    if (nb > 0x7FFFFFFF) return hipErrorInvalidValue;
    const int K = (int)w.K;
    const int64_t mpad = (int64_t)(M + 63) / 64 * 64;
    hipLaunchKernelGGL((k_xplanes<QT>), dim3(M), dim3(XP_T), 0, s, x, K, (int64_t)M * K, reinterpret_cast<h8_t*>(b.P),
                       b.E, b.SS, b.SA, mpad);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const dim3 grid((unsigned)nb), block(256);
#define THQ_EX(OUT_, Y_)                                                                                         \
    hipLaunchKernelGGL((k_gemm_ex<QT, ST, GU, OUT_>), grid, block, 0, s, w.q, w.aux, b.P, b.E, b.SS, b.SA, mpad, x, \
                       Y_, M, K, nout, up_off, w.N, p.cps, (int)tiles, p.splits)
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
    if (plane >= lim || (uint64_t)M * (uint64_t)K * 4u >= lim) return p;
    // Two blocks per CU.  Cost of a K split count: rounds of resident blocks
    // x chunks (and one of prologue) x a chunk's time (2.4 us stacked, 4.0 us
    // with two operands), plus the partials' round trip at 4 TB/s.
    const int64_t nch = K / 256, nout = gu ? N / 2 : N, cu = cus > 0 ? cus : 256;
    p.stacked = M <= 16;
    p.groups = (int)((M + (p.stacked ? 15 : 31)) / (p.stacked ? 16 : 32));
    const int64_t per = gu ? 128 : 256, tiles = (nout + per - 1) / per;
    const int64_t smin = (nch + EX_CPS - 1) / EX_CPS;
    double best = 1e30;
    for (int64_t s = smin; s <= nch && s <= smin + 32; ++s) {
        const int64_t cps = (nch + s - 1) / s;
        const int64_t rounds = (tiles * p.groups * s + 2 * cu - 1) / (2 * cu);
        const double t = (double)rounds * ((double)cps + 1.0) * (p.stacked ? 2.4 : 4.0) +
                         (s > 1 ? 2.0 + (double)s * (double)M * (double)N * 8.0 / 4.0e6 : 0.0);
        if (t < best - 1e-9) {
            best = t;
            p.cps = (int)cps;
            p.splits = (int)((nch + cps - 1) / cps);
        }
    }
    p.workspace_bytes = ex_planes_bytes(M, K) + ex_align((size_t)M * 4) + ex_sums_bytes(qtype, M, K) +
                        (p.splits > 1 ? (size_t)p.splits * (size_t)M * (size_t)N * 4u : 0);
    return p;
}

hipError_t launch_gemm_ex(const ExPlan& p, const WeightView& w, const float* x, void* y, bool yf32, bool gu, int M,
                          int64_t nout, int64_t up_off, void* ws, hipStream_t s) {
    if (p.groups < 1 || p.splits < 1 || M < 1 || !ws) return hipErrorInvalidValue;
    char* q = static_cast<char*>(ws);
    ExBufs b{};
    b.P = reinterpret_cast<_Float16*>(q);
    q += ex_planes_bytes(M, w.K);
    b.E = reinterpret_cast<int*>(q);
    q += ex_align((size_t)M * 4);
    b.SS = reinterpret_cast<_Float16*>(q);
    b.SA = reinterpret_cast<float*>(q);
    q += ex_sums_bytes(w.qtype, M, w.K);
    b.part = reinterpret_cast<float*>(q);
#define THQ_EXG(QT_, ST_)                                                            \
    (gu ? run_ex<QT_, ST_, true>(p, w, x, b, y, yf32, M, nout, up_off, s)            \
        : run_ex<QT_, ST_, false>(p, w, x, b, y, yf32, M, nout, up_off, s))
#define THQ_EXQ(QT_) (p.stacked ? THQ_EXG(QT_, true) : THQ_EXG(QT_, false))
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
