// Quantized GEMM for few rows or narrow outputs: every wave stages its own
// operands through LDS of its own, so the K loop has no workgroup barrier and a
// wave waits only for its own loads, which it keeps NS groups ahead.
//
// A wave owns 16 rows x 16 columns over all of K. A group is four consecutive
// Q8 blocks, 128 bytes of a row. Eight lanes read a row's 128 bytes (a lane per
// row would touch 64 cache lines per load) and the pieces go through the wave's
// LDS rows to the lanes that feed them to the matrix core:
//  * v_mfma_i32_16x16x32_i8 per block gives its exact i32 dots (lane l:
//    activation or weight row l % 16, bytes 8 (l / 16) .. +8 of the block;
//    accumulator v: output row 4 (l / 16) + v, column l % 16);
//  * one v_mfma_f32_16x16x1_4b_f32 gives the scale products of the four blocks
//    in the same lanes, registers 4 j + v (zero C, one nonzero product: the
//    correctly rounded f32 product).
// The vector unit then runs the reference's epilogue in block order: for
// Q8_0x4 slot = fma(isum, wx, slot) (quant.rs:276-288), for the four partial
// sums t[j] += wx * isum (dot.rs:34-45), where register 4 j + v of the group
// belongs to chain j: sixteen independent chains per lane.
#include <hip/hip_runtime.h>

#include "kernrt_hip.h"
#include "device.hpp"
#include "kernels.hpp"
#include "numerics.hpp"

namespace kr {

typedef int d_v4i __attribute__((ext_vector_type(4)));
typedef int d_v16i __attribute__((ext_vector_type(16)));
typedef float d_v16f __attribute__((ext_vector_type(16)));

enum { EPI_PLAIN = 0, EPI_SWI = 1, EPI_ROPE = 2 };

// NW waves side by side: a workgroup's tile is 16 rows x 16 NW columns, of one
// wave in the plain form, of four with an epilogue. EPI_SWI: columns 0..31 are gate rows, 32..63 up rows of hidden block nt;
// EPI_ROPE: the 64 columns are one head.
template <int SEM, int EPI, int NW, int NS, bool DBG>
__global__ __launch_bounds__(64 * NW) void k_gemm_direct(MatSet ms, QuantAct x, uint32_t M, uint32_t K, uint32_t mtiles,
                                                     int32_t* __restrict__ dbg, SwiOut so, RopeOut ro) {
    static_assert(NS % 2 == 0, "results alternate between two register sets");
    constexpr bool FMA = SEM == SEM_FMA_CHAIN, WF16 = SEM != SEM_FOUR_PARTIALS_F32;
    constexpr int NT = FMA ? 4 : 16, TM = 16, LD = 68;
    constexpr int ROW = 128 + 16, SLOT = 32 * ROW + 512;  // a wave's slot: 16 + 16 operand rows, 64 + 64 scales
    __shared__ __align__(16) int8_t lds[NW * 2 * SLOT];
    static_assert(EPI == EPI_PLAIN || (NW == 4 && TM * LD * 4 <= sizeof(lds)), "the epilogue's tile reuses the slots");
    __shared__ uint64_t etab[EPI == EPI_SWI ? 32 : 1];
    const uint32_t nb = K >> 5, ng = (nb + 3) >> 2;
    const uint32_t L = gemm_xcd_tile(blockIdx.x, gridDim.x);
    const uint32_t mt = L % mtiles, nt = L / mtiles;
    const uint32_t tid = threadIdx.x, lane = tid & 63, r = lane & 15, quad = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int mi_ = EPI == EPI_SWI ? (int)(wave >> 1) : nt < ms.tile_end[0] ? 0 : (nt < ms.tile_end[1] ? 1 : 2);
    const uint32_t N = ms.n[mi_], m0 = mt * TM;
    // the wave's first column in its matrix
    const uint32_t n0 = EPI == EPI_SWI ? nt * 32 + 16 * (wave & 1)
                                       : (nt - (mi_ == 0 ? 0 : ms.tile_end[mi_ - 1])) * 16 * NW + 16 * wave;
    if (EPI == EPI_SWI && tid < 32) etab[tid] = kExp2Tab[tid];

    // loader map: lane l reads 16-byte piece l % 8 of rows l / 8 and l / 8 + 8,
    // and the scale of row l / 4, block l % 4. Rows past M or N read the last
    // row, pieces and blocks past the row end its last ones.
    const uint32_t lr = lane >> 3, lc = (lane & 7) * 16, sr = lane >> 2, sb = lane & 3;
    const int8_t* gp[4];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        gp[i] = x.q + (size_t)min(m0 + lr + 8 * i, M - 1) * K;
        gp[2 + i] = ms.q[mi_] + (size_t)min(n0 + lr + 8 * i, N - 1) * K;
    }
    const size_t xsb = (size_t)min(m0 + sr, M - 1) * nb, wsb = (size_t)min(n0 + sr, N - 1) * nb;
    const void* __restrict__ XS = FMA ? (const void*)x.h : (const void*)x.s;
    const void* __restrict__ WS = ms.s[mi_];
    int8_t* const wl = lds + wave * 2 * SLOT;
    struct Stage {
        d_v4i p[4];
        uint32_t xs, ws;
    };
    struct Frag {
        long a[4], b[4];
        uint32_t xs, ws;
    };
    struct Res {
        d_v4i d[4];
        d_v16f p;
    };
    auto gload = [&](Stage& st, uint32_t g) {
        g = min(g, ng - 1);
        const uint32_t col = min(g * 128 + lc, K - 16), blk = min(4 * g + sb, nb - 1);
#pragma unroll
        for (int i = 0; i < 4; i++) st.p[i] = *(const d_v4i*)(gp[i] + col);
        st.xs = scale_bits(FMA, XS, xsb + blk);
        st.ws = scale_bits(WF16, WS, wsb + blk);
    };
    auto lstore = [&](const Stage& st, int slot) {
        int8_t* s = wl + slot * SLOT;
#pragma unroll
        for (int i = 0; i < 4; i++) *(d_v4i*)(s + (lr + 8 * i) * ROW + lc) = st.p[i];
        *(uint32_t*)(s + 32 * ROW + 4 * lane) = st.xs;
        *(uint32_t*)(s + 32 * ROW + 256 + 4 * lane) = st.ws;
    };
    auto fload = [&](Frag& f, int slot) {
        const int8_t* s = wl + slot * SLOT;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            f.a[j] = *(const long*)(s + r * ROW + 32 * j + 8 * quad);
            f.b[j] = *(const long*)(s + (16 + r) * ROW + 32 * j + 8 * quad);
        }
        f.xs = *(const uint32_t*)(s + 32 * ROW + 16 * r + 4 * quad);
        f.ws = *(const uint32_t*)(s + 32 * ROW + 256 + 16 * r + 4 * quad);
    };
    const d_v4i izero = {};
    const d_v16f fzero = {};
    auto mfma = [&](Res& o, const Frag& f) {
        o.p = __builtin_amdgcn_mfma_f32_16x16x1f32(scale_value(FMA, f.xs), scale_value(WF16, f.ws), fzero, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; j++) o.d[j] = __builtin_amdgcn_mfma_i32_16x16x32_i8(f.a[j], f.b[j], izero, 0, 0, 0);
    };
    float t[NT];
#pragma unroll
    for (int v = 0; v < NT; v++) t[v] = 0.0f;
    auto epilogue = [&](const Res& o, uint32_t g, bool last) {
        if (DBG) {
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const uint32_t m = m0 + 4 * quad + (e & 3), n = n0 + r, b = 4 * g + (e >> 2);
                if (m < M && n < N && b < nb) dbg[((size_t)m * N + n) * nb + b] = o.d[e >> 2][e & 3];
            }
        }
        // in the row's last groups a block past its end keeps the sum as it is
        const uint32_t live = nb - 4 * g;
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int e = (4 * j + v) % NT;
                const float s = FMA ? __builtin_fmaf((float)o.d[j][v], o.p[4 * j + v], t[e])
                                    : t[e] + o.p[4 * j + v] * (float)o.d[j][v];
                t[e] = !last || (uint32_t)j < live ? s : t[e];
            }
    };

    // At step g: group g + 2 from registers into LDS and its fragments back,
    // its registers refilled with group g + 2 + NS, group g + 1's matrix work,
    // group g's epilogue. A register set is named at compile time, so its wait
    // covers only its own loads. A wave's LDS operations run in order, so a slot
    // needs no barrier; the fences keep the compiler to that order. Groups past
    // the last are copies of it, staged but never summed.
    auto ordered = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local"); };
    Stage st[NS];
    Frag f[2];
    Res res[2];
#pragma unroll
    for (int s = 0; s < NS; s++) gload(st[s], s);
#pragma unroll
    for (int s = 0; s < 2; s++) {
        lstore(st[s], s);
        gload(st[s], s + NS);
        ordered();
        fload(f[s], s);
    }
    mfma(res[0], f[0]);
    auto step = [&](uint32_t g, int u, bool last) {
        ordered();
        lstore(st[(u + 2) % NS], u & 1);
        gload(st[(u + 2) % NS], g + 2 + NS);
        mfma(res[(u + 1) & 1], f[(u + 1) & 1]);
        ordered();
        fload(f[u & 1], u & 1);
        epilogue(res[u & 1], g, last);
    };
    const uint32_t full = nb / 4 / NS * NS;  // rounds of NS whole groups
    uint32_t g0 = 0;
    for (; g0 < full; g0 += NS) {
#pragma unroll
        for (int u = 0; u < NS; u++) step(g0 + u, u, false);
    }
#pragma unroll
    for (int u = 0; u < NS; u++)
        if (g0 + u < ng) step(g0 + u, u, true);

    auto value = [&](int v) {
        if (FMA) return t[v];
        return ((t[v] + t[(4 + v) % NT]) + t[(8 + v) % NT]) + t[(12 + v) % NT];
    };
    float* Y = ms.y[mi_];
    const uint32_t ld = ms.ld[mi_];
    if constexpr (EPI == EPI_PLAIN) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const uint32_t m = m0 + 4 * quad + v, n = n0 + r;
            if (m < M && n < N) Y[(size_t)m * ld + n] = value(v);
        }
        return;
    }
    float* const sy = (float*)lds;
    __syncthreads();  // other waves may still read their slots
#pragma unroll
    for (int v = 0; v < 4; v++) sy[(4 * quad + v) * LD + 16 * wave + r] = value(v);
    __syncthreads();
    const uint32_t c = tid & 31;
    if constexpr (EPI == EPI_SWI) {
#pragma unroll
        for (int k = 0; k < TM / 8; k++) {  // a half-wave holds one row's hidden block
            const uint32_t row = (tid >> 5) + 8 * k;
            swi_out(so, sy[row * LD + c], sy[row * LD + 32 + c], m0 + row, M, N, nt, c, etab);
        }
    }
    if constexpr (EPI == EPI_ROPE) {
        const uint32_t h0 = n0 - 16 * wave;
#pragma unroll
        for (int k = 0; k < TM / 8; k++) {
            const uint32_t row = (tid >> 5) + 8 * k, m = m0 + row;
            if (m >= M) continue;
            rope_out(ro, mi_, Y, ld, sy[row * LD + c], sy[row * LD + 32 + c], m, h0, c);
        }
    }
}

// Fill in the tile counts (16 NW columns) and launch over 16-row tiles.
template <int SEM, int EPI, int NW, int NS>
static hipError_t direct_go(hipStream_t st, MatSet ms, QuantAct x, size_t rows, size_t k, int32_t* dbg, SwiOut so,
                            RopeOut ro) {
    uint32_t total = 0;
    for (int i = 0; i < 3; i++) {
        if (i < ms.count) total += (uint32_t)((ms.n[i] + 16 * NW - 1) / (16 * NW));
        ms.tile_end[i] = total;
    }
    if (EPI == EPI_SWI) total = ms.n[0] / 32;
    const uint32_t mtiles = (uint32_t)((rows + 15) / 16);
    const dim3 grid(total * mtiles), block(64 * NW);
    if constexpr (EPI == EPI_PLAIN) {
        if (dbg) {
            hipLaunchKernelGGL((k_gemm_direct<SEM, EPI, NW, 2, true>), grid, block, 0, st, ms, x, (uint32_t)rows,
                               (uint32_t)k, mtiles, dbg, so, ro);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((k_gemm_direct<SEM, EPI, NW, NS, false>), grid, block, 0, st, ms, x, (uint32_t)rows, (uint32_t)k,
                       mtiles, nullptr, so, ro);
    return hipGetLastError();
}

hipError_t launch_gemm_direct(hipStream_t st, int sem, const MatSet& ms, size_t k, QuantAct x, size_t rows,
                              int32_t* dbg) {
    switch (sem) {
        case SEM_FMA_CHAIN: return direct_go<SEM_FMA_CHAIN, EPI_PLAIN, 1, 4>(st, ms, x, rows, k, dbg, {}, {});
        case SEM_FOUR_PARTIALS_F32:
            return direct_go<SEM_FOUR_PARTIALS_F32, EPI_PLAIN, 1, 4>(st, ms, x, rows, k, dbg, {}, {});
        case SEM_FOUR_PARTIALS_F16:
            return direct_go<SEM_FOUR_PARTIALS_F16, EPI_PLAIN, 1, 4>(st, ms, x, rows, k, dbg, {}, {});
    }
    return hipErrorInvalidValue;
}

hipError_t launch_direct_swi(hipStream_t st, int sem, const MatSet& ms, size_t k, QuantAct x, size_t rows,
                             SwiOut so) {
    if (sem == SEM_FMA_CHAIN) return direct_go<SEM_FMA_CHAIN, EPI_SWI, 4, 4>(st, ms, x, rows, k, nullptr, so, {});
    return direct_go<SEM_FOUR_PARTIALS_F32, EPI_SWI, 4, 4>(st, ms, x, rows, k, nullptr, so, {});
}

hipError_t launch_direct_rope(hipStream_t st, int sem, const MatSet& ms, size_t k, QuantAct x, size_t rows,
                              RopeOut ro) {
    if (sem == SEM_FMA_CHAIN) return direct_go<SEM_FMA_CHAIN, EPI_ROPE, 4, 4>(st, ms, x, rows, k, nullptr, {}, ro);
    return direct_go<SEM_FOUR_PARTIALS_F32, EPI_ROPE, 4, 4>(st, ms, x, rows, k, nullptr, {}, ro);
}

}  // namespace kr
