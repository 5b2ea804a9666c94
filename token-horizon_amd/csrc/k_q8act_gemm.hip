// k_q8act_gemm.hip — THQ_MODE_Q8ACT over many activation rows on the int8
// matrix cores (Q4_K and Q8_0 weights in their default layouts).
//
// Role: candle's default CPU arithmetic over prompts ([ext] candle-core 0.11
// k_quants::matmul: every activation row quantized to the weight's dot type,
// then integer block dots scaled in f32).  k_q8act.hip walks the weight again
// for every 8 rows with v_dot4 (Q4_K MLP 4096 / 12288 at M = 256: 1.53 ms, now
// 0.15 ms).
//
// The integers stay exact.  Q4_K: a superblock's aux = sum_j sc_j (q4 . q8)_j
// comes from two int8 planes of the weight, (sc & 7) q and (sc >> 3) q (at
// most 105), each summed over the whole superblock by v_mfma_i32_32x32x32_i8
// without touching the accumulators in between: aux = lo + 8 hi.  One plane
// and a multiply-add per 32-wide sub-block would cost 16 VALU instructions
// for each MFMA.  mins = sum_j m_j xb_j is one f16 MFMA over the 32-wide quant
// sums in two exact pieces (xb & 63 and the rest; every product and sum stays
// below 2^24).  Then y += d_x (d_w aux - dmin_w mins).  Q8_0: one MFMA per
// 32-wide block on the weight's bytes as they are, y += d_w (d_x integer),
// the eight blocks of a chunk summed first.  At most QG_CPS chunks of 256 per
// K split are added in f32, the splits in f64: error against 64-bit sums
// (K = 1024 .. 16384) 0.6e-7 .. 0.8e-7, before 0.7e-7 .. 2.1e-7.
//
// Block = 4 waves, 32 MH activation rows; a wave owns two 32-row column tiles
// (gate/up: gate and up rows of the same outputs), takes them in turn and
// streams each one's 256-wide chunk into registers a chunk ahead; the int8
// rows go into LDS by direct-to-LDS copies, the next chunk's while the
// current one computes.  A lane's 16 nibble bytes are its MFMA operand's 16
// weights, so the conversion is one mask and two v_pk_mul_lo_u16 per 4
// weights.  Bound: no unit alone: gate/up of 24576 x 4096 at M = 256 (94 us)
// keeps the VALU busy 38 % (conversion, the f32 step) and the matrix cores 24 %
// of the time, 27 % of a wave's time in waits (a chunk at MH = 2 takes 2.75 us
// with one block on the CU, 5.4 with two; Q4_K spills 2 to 3 registers there);
// weights by coalesced copies through LDS instead measured slower (MLP at M =
// 256: 180 against 169 us).
#include "thq_dev.hpp"
#include "thq_kernels.hpp"

#include <type_traits>

namespace thq {
namespace {

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));

constexpr int QG_CPS = 16;

__device__ __forceinline__ uint32_t qg_lds(const void* p) {
    return (uint32_t)(size_t)(__attribute__((address_space(3))) const void*)p;
}
// lane l's 16 bytes at base + voff land at LDS m0 + 16 l; untracked by the
// compiler (the kernel waits for them itself)
__device__ __forceinline__ void qg_dma16(uint32_t lds, const void* base, uint32_t voff) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(lds), "v"(voff), "s"(base) : "memory");
}
// four byte codes x s, s small enough that no byte carries (15 x 7)
__device__ __forceinline__ int qg_mul4(uint32_t q, uint16_t s) {
    u16x2_t v;
    __builtin_memcpy(&v, &q, 4);
    v *= u16x2_t{s, s};
    int r;
    __builtin_memcpy(&r, &v, 4);
    return r;
}

// one 256-wide chunk of a lane's weight row, and its header (Q4_K: four
// dwords, Q8_0: eight f16 scales)
template <int QT>
struct QgChunk {
    u32x4_t w[QT == 8 ? 8 : 4];
    u32x4_t h;
};

// OUT: 0 = K-split partials f32 [split][M][nrows], 1 = f32, 2 = bf16
template <int QT, int MH, bool GU, int OUT>
__global__ __launch_bounds__(256, 2) void k_q8act_gemm(const uint8_t* Wq, const uint8_t* Wa, const int8_t* xq,
                                                       const float* xd, const int16_t* xb, void* __restrict__ Yv,
                                                       int M, int K, int64_t nout, int64_t up_off, int64_t nrows,
                                                       int cps, int tiles, int splits) {
    constexpr int MP = 32 * MH;               // activation rows per group
    constexpr int XB = MP * 256;              // bytes per buffer
    constexpr int NJ = MP / 16;               // copy instructions per wave per chunk (4 rows each)
    constexpr int ND = QT == 8 ? 8 : 1;       // activation scales per chunk and row
    __shared__ __attribute__((aligned(16))) uint8_t xs[2 * XB];
    __shared__ __attribute__((aligned(16))) float dxs[2][ND][MP];

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
    uint32_t ow[2], oh[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        orow[t] = GU ? (int64_t)tile_i * 128 + wave * 32 + n : (int64_t)tile_i * 256 + wave * 64 + 32 * t + n;
        valid[t] = orow[t] < nout;
        row[t] = valid[t] ? (GU && t ? orow[t] + up_off : orow[t]) : 0;  // in-bounds reads
        if constexpr (QT == 8) {
            ow[t] = (uint32_t)q8t_q(row[t], K >> 5, 0, g);
            oh[t] = (uint32_t)q8t_d(row[t], K >> 5, 0) * 2u;
        } else {
            ow[t] = (uint32_t)q4k_piece(row[t], nch, 0, g, 0);
            oh[t] = (uint32_t)q4k_hdword(row[t], nch, 0, 0);
        }
    }
    auto wload = [&](QgChunk<QT>& C, int t, int c) {
        if constexpr (QT == 8) {
            const uint8_t* b = Wq + (int64_t)c * 8192;
#pragma unroll
            for (int j = 0; j < 8; ++j) C.w[j] = *reinterpret_cast<const u32x4_t*>(b + ow[t] + j * 1024);
            C.h = *reinterpret_cast<const u32x4_t*>(Wa + (int64_t)c * 512 + oh[t]);
        } else {
            const uint8_t* b = Wq + (int64_t)c * 64;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                C.w[u] = *reinterpret_cast<const u32x4_t*>(b + ow[t] + u * 16);
                C.h[u] = *reinterpret_cast<const uint32_t*>(b + oh[t] + u * 16);
            }
        }
    };
    // copy j of a wave fills operand rows 4 (wave + 4 j) .. + 3; the 16-B piece
    // p of row r sits at slot p ^ (r & 15); rows past the group copy its last
    uint32_t xoff[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int r = 4 * (wave + 4 * j) + (lane >> 4);
        xoff[j] = (uint32_t)(m0 + (r < Mz ? r : Mz - 1)) * (uint32_t)K + 16u * (uint32_t)((lane & 15) ^ (r & 15));
    }
    const uint32_t xs0 = qg_lds(xs);
    auto xcopy = [&](int c, int b) {
        const int8_t* xc = xq + (int64_t)c * 256;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            qg_dma16(__builtin_amdgcn_readfirstlane(xs0 + (uint32_t)(b * XB + (wave + 4 * j) * 1024)), xc, xoff[j]);
    };
    // activation scales of chunk c: one (Q8_0: two at MH = 2) per thread
    constexpr int NS = (ND * MP + 255) / 256;
    auto dload = [&](float (&v)[NS], int c) {
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const int q = ((int)threadIdx.x + 256 * i) & (ND * MP - 1), r = q % MP;
            v[i] = xd[(int64_t)(m0 + (r < Mz ? r : Mz - 1)) * (QT == 8 ? K >> 5 : nch) + c * ND + q / MP];
        }
    };
    auto dstore = [&](const float (&v)[NS], int b) {
#pragma unroll
        for (int i = 0; i < NS; ++i) (&dxs[b][0][0])[((int)threadIdx.x + 256 * i) & (ND * MP - 1)] = v[i];
    };
    auto aread = [&](int b, int h, int j) {  // 32-wide sub-block j
        return *reinterpret_cast<const i32x4_t*>(xs + b * XB + (32 * h + n) * 256 + 16 * ((2 * j + g) ^ (n & 15)));
    };

    f32x16_t acc[2][MH];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int h = 0; h < MH; ++h) acc[t][h] = f32x16_t{};

    // dx of the lane's 16 rows of half h (block j of the chunk)
    auto dxread = [&](float (&v)[16], int b, int h, int j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const f32x4_t q = *reinterpret_cast<const f32x4_t*>(&dxs[b][j][32 * h + 8 * i + 4 * g]);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[4 * i + e] = q[e];
        }
    };
    auto tile4 = [&](const QgChunk<QT>& C, f32x16_t (&a)[MH], const h8_t (&S)[MH], int b) {
        const uint32_t M4 = 0x0F0F0F0Fu;
        i32x16_t lo[MH], hi[MH];
#pragma unroll
        for (int h = 0; h < MH; ++h) lo[h] = hi[h] = i32x16_t{};
        h8_t V;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t hw = C.h[j >> 1] >> (12 * (j & 1));
            const uint16_t s0 = (uint16_t)(hw & 7u), s1 = (uint16_t)((hw >> 3) & 7u);
            V[j] = (_Float16)(uint16_t)((hw >> 6) & 63u);
            i32x4_t B0, B1;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t q = (C.w[j >> 1][i] >> (4 * (j & 1))) & M4;
                B0[i] = qg_mul4(q, s0);
                B1[i] = qg_mul4(q, s1);
            }
#pragma unroll
            for (int h = 0; h < MH; ++h) {
                const i32x4_t A = aread(b, h, j);
                lo[h] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A, B0, lo[h], 0, 0, 0);
                hi[h] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A, B1, hi[h], 0, 0, 0);
            }
        }
        const float dw = f16_to_f32((uint16_t)__builtin_amdgcn_perm(C.h[1], C.h[0], 0x0c0c0703u));
        const float dm = f16_to_f32((uint16_t)__builtin_amdgcn_perm(C.h[3], C.h[2], 0x0c0c0703u));
#pragma unroll
        for (int h = 0; h < MH; ++h) {
            const f32x16_t mins = __builtin_amdgcn_mfma_f32_32x32x16_f16(S[h], V, f32x16_t{}, 0, 0, 0);
            float dx[16];
            dxread(dx, b, h, 0);
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float aux = (float)(lo[h][e] + 8 * hi[h][e]);
                a[h][e] = __builtin_fmaf(dx[e], __builtin_fmaf(dw, aux, -(dm * mins[e])), a[h][e]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto tile8 = [&](const QgChunk<QT>& C, f32x16_t (&a)[MH], int b) {
#pragma unroll
        for (int h = 0; h < MH; ++h) {
            f32x16_t T = {};
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const i32x4_t B = {(int)C.w[j][0], (int)C.w[j][1], (int)C.w[j][2], (int)C.w[j][3]};
                const i32x16_t D = __builtin_amdgcn_mfma_i32_32x32x32_i8(aread(b, h, j), B, i32x16_t{}, 0, 0, 0);
                const uint32_t hw = C.h[j >> 1];
                const float dw = f16_to_f32((uint16_t)((j & 1) ? hw >> 16 : hw));
                float dx[16];
                __builtin_amdgcn_sched_barrier(0);  // hoisted over the blocks, the scales spill
                dxread(dx, b, h, j);
#pragma unroll
                for (int e = 0; e < 16; ++e) T[e] = __builtin_fmaf(dw * dx[e], (float)D[e], T[e]);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int e = 0; e < 16; ++e) a[h][e] += T[e];
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    QgChunk<QT> W[2];
    auto last = [&](int c) { return c < ce ? c : ce - 1; };
    float dn[NS];
    xcopy(cb, 0);
    wload(W[0], 0, cb);
    wload(W[1], 1, cb);
    dload(dn, cb);
    dstore(dn, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // step c (buffer b): chunk c + 1's copies go out first (buffer b ^ 1, read
    // by no wave since the last barrier); each tile's weights are loaded again
    // for chunk c + 1 as soon as they are consumed and stay in flight across
    // the barrier: loads complete in order and the first tile's are eight or
    // more instructions behind the copies, so vmcnt(8) waits for the copies
    // only.  Past the range they repeat the last chunk.
    for (int c = cb; c < ce; ++c) {
        const int b = (c - cb) & 1;
        xcopy(last(c + 1), b ^ 1);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        dload(dn, last(c + 1));
        h8_t S[MH];
        if constexpr (QT == 12) {
            // the rows' 32-wide quant sums: lane half 0 their low 6 bits, half 1 the rest
#pragma unroll
            for (int h = 0; h < MH; ++h) {
                const int r = 32 * h + n;
                const u32x4_t v =
                    *reinterpret_cast<const u32x4_t*>(xb + (int64_t)(m0 + (r < Mz ? r : Mz - 1)) * (K >> 5) + 8 * c);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int s = (int)(int16_t)(v[j >> 1] >> (16 * (j & 1)));
                    S[h][j] = (_Float16)(int16_t)(g ? s & ~63 : s & 63);
                }
            }
        }
        if constexpr (QT == 12)
            tile4(W[0], acc[0], S, b);
        else
            tile8(W[0], acc[0], b);
        wload(W[0], 0, last(c + 1));
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (QT == 12)
            tile4(W[1], acc[1], S, b);
        else
            tile8(W[1], acc[1], b);
        dstore(dn, b ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        wload(W[1], 1, last(c + 1));
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
    }

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no copy may land in LDS after the block ends
    // acc[t][h][e] is activation row 32 h + 8 (e / 4) + 4 g + e % 4 of the group
    constexpr int NT = GU && OUT != 0 ? 1 : 2;  // stored tiles (gate/up: the gate's)
#pragma unroll
    for (int h = 0; h < MH; ++h)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int m = 32 * h + 8 * (e >> 2) + 4 * g + (e & 3);
            if (m >= Mz) continue;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if (!valid[t]) continue;
                if constexpr (OUT == 0) {
                    static_cast<float*>(Yv)[((int64_t)split * M + m0 + m) * nrows + row[t]] = acc[t][h][e];
                } else {
                    using YT = std::conditional_t<OUT == 1, float, bf16_t>;
                    store_y<YT>(static_cast<YT*>(Yv) + (int64_t)(m0 + m) * nout + orow[t],
                                GU ? silu_mul(acc[0][h][e], acc[1][h][e]) : acc[t][h][e]);
                }
            }
        }
}

template <int QT, int MH, bool GU>
hipError_t run_qg(const QgPlan& p, const WeightView& w, const int8_t* xq, const float* xd, const int16_t* xb, void* y,
                  bool yf32, int M, int64_t nout, int64_t up_off, float* ws, hipStream_t s) {
    const int64_t per = GU ? 128 : 256, tiles = (nout + per - 1) / per;
    const int64_t nb = tiles * p.splits * p.groups;
    if (nb > 0x7FFFFFFF) return hipErrorInvalidValue;
#define THQ_QG(OUT_, Y_)                                                                                      \
    hipLaunchKernelGGL((k_q8act_gemm<QT, MH, GU, OUT_>), dim3((unsigned)nb), dim3(256), 0, s, w.q, w.aux, xq, \
                       xd, xb, Y_, M, (int)w.K, nout, up_off, w.N, p.cps, (int)tiles, p.splits)
    if (p.splits > 1) {
        THQ_QG(0, (void*)ws);
        const hipError_t e = hipGetLastError();
        return e != hipSuccess ? e : launch_ex_reduce(ws, y, yf32, GU, M, nout, up_off, w.N, p.splits, s);
    }
    if (yf32)
        THQ_QG(1, y);
    else
        THQ_QG(2, y);
#undef THQ_QG
    return hipGetLastError();
}

}  // namespace

QgPlan plan_q8act_gemm(int qtype, int64_t M, int64_t N, int64_t K, bool gu, int cus) {
    QgPlan p;
    if ((qtype != 8 && qtype != 12) || M < 1 || N < 1 || K < 256 || K % 256 || (gu && N % 2)) return p;
    // 32-bit offsets: the weight plane and the int8 rows below 4 GiB
    const uint64_t lim = 1ull << 32;
    const uint64_t plane =
        qtype == 8 ? (uint64_t)q8t_q_bytes(N, K) : (uint64_t)((N + 3) / 4) * (uint64_t)(K / 256) * 576u;
    if (plane >= lim || (uint64_t)M * (uint64_t)K >= lim) return p;
    // Cost: chunks per block (and one of prologue) x a chunk's time with one or
    // two resident blocks per CU (us, 12288 x 4096 / 4096 x 12288 / gate/up at
    // M = 32 .. 256, every split count), plus the partials' round trip at 4 TB/s.
    static const double chunk_us[2][2][2] = {{{2.0, 4.0}, {2.75, 5.4}}, {{3.0, 4.0}, {5.3, 6.4}}};
    const int64_t nch = K / 256, nout = gu ? N / 2 : N, cu = cus > 0 ? cus : 256;
    const int64_t per = gu ? 128 : 256, tiles = (nout + per - 1) / per, smin = (nch + QG_CPS - 1) / QG_CPS;
    double best = 1e30;
    for (int mh = 1; mh <= 2; ++mh) {
        const int64_t groups = (M + 32 * mh - 1) / (32 * mh);
        const double* us = chunk_us[qtype == 8][mh - 1];
        for (int64_t s = smin; s <= nch && s <= smin + 32; ++s) {
            const int64_t cps = (nch + s - 1) / s, blocks = tiles * groups * s, rem = blocks % (2 * cu);
            const double t = ((double)(blocks / (2 * cu)) * us[1] + (rem == 0 ? 0.0 : us[rem > cu])) * ((double)cps + 1.0) +
                             (s > 1 ? 2.0 + (double)s * (double)M * (double)N * 8.0 / 4.0e6 : 0.0);
            if (t < best - 1e-9) {
                best = t;
                p.mh = mh;
                p.groups = (int)groups;
                p.cps = (int)cps;
                p.splits = (int)((nch + cps - 1) / cps);
            }
        }
    }
    p.workspace_bytes = p.splits > 1 ? (size_t)p.splits * (size_t)M * (size_t)N * 4u : 0;
    return p;
}

hipError_t launch_q8act_gemm(const QgPlan& p, const WeightView& w, const int8_t* xq, const float* xd,
                             const int16_t* xb, void* y, bool yf32, bool gu, int M, int64_t nout, int64_t up_off,
                             float* ws, hipStream_t s) {
    if (p.groups < 1 || p.splits < 1 || M < 1 || (p.splits > 1 && !ws)) return hipErrorInvalidValue;
#define THQ_QGG(QT_, MH_)                                                                         \
    (gu ? run_qg<QT_, MH_, true>(p, w, xq, xd, xb, y, yf32, M, nout, up_off, ws, s)               \
        : run_qg<QT_, MH_, false>(p, w, xq, xd, xb, y, yf32, M, nout, up_off, ws, s))
    if (w.qtype == 8) return p.mh == 1 ? THQ_QGG(8, 1) : THQ_QGG(8, 2);
    if (w.qtype == 12) return p.mh == 1 ? THQ_QGG(12, 1) : THQ_QGG(12, 2);
#undef THQ_QGG
    return hipErrorInvalidValue;
}

}  // namespace thq
