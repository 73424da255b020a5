// gemm_tile.h -- one workgroup's tile of a bf16 product with many rows, shared by the
// dense products (matmul.hip) and the grouped expert products (moe.hip).
#pragma once
#include "common.h"

#include <type_traits>

namespace sandy_hip {

// Prefill-sized products: workgroup tile 64 WM x 64 WN of rows x columns,
// 2 x 2 waves of 32 WM x 32 WN on v_mfma_f32_32x32x16_bf16; KS such groups of
// waves take every KS-th chunk of 64 k (their sums added through LDS at the
// end, in group order).  The weight rows are the A operand, so a lane ends with
// four consecutive columns of one activation row.  Both operands go global ->
// registers -> LDS as whole 128-byte lines into XOR-swizzled rows (16-byte
// piece p of row r at p ^ (r / 2) % 8: conflict-free 128-bit writes and
// MFMA-layout reads).  While a chunk multiplies, the next moves from registers
// to the other LDS buffer and the one after is requested, a quarter of each
// per 16 k, so that the matrix cores never wait for a whole chunk's copies.
// Bound: LDS and issue slots beside the MFMA (busy 47% at 2048 x 11264 x 2048);
// see the launch rule for figures.
template <int WM, int WN, int KS>
struct TileGeo {
    static constexpr int BM = 64 * WM, BN = 64 * WN;
    static constexpr int THREADS = 256 * KS;
    static constexpr int kX = BM * 128, kW = BN * 128, kGroup = 2 * (kX + kW);
    static constexpr int XP = BM * 8 / 256, WP = BN * 8 / 256;  // 16-byte pieces a thread stages per chunk
    static constexpr int kRowPitch = 64 * WN + 16;              // bytes of a wave's output row in LDS
    static constexpr int kOut = 4 * 32 * WM * kRowPitch;
    static constexpr int kSums = (KS - 1) * 4 * WM * WN * 64 * 64;
    static constexpr int kLoop = KS * kGroup;
    static constexpr int kBytes = kLoop > kOut ? (kLoop > kSums ? kLoop : kSums) : (kOut > kSums ? kOut : kSums);
};

// One tile: rows x [xrows, K] times the weight rows w [wrows, K], both packed with
// K % 32 == 0 and 16-byte aligned, into out (rows `pitch` apart), plus bias [wrows]
// if given; 1 <= xrows <= BM, 1 <= wrows <= BN, and wrows is BN or ends the rows of
// `out`, so that it divides by what `pitch` divides by.  PART: a wave whose rows all lie past
// xrows multiplies nothing.
template <int WM, int WN, int KS, bool PART>
__device__ __forceinline__ void gemm_tile(unsigned char* lds, const uint16_t* x, int xrows, const uint16_t* w, int wrows,
                                          int64_t K, const uint16_t* bias, uint16_t* out, int64_t pitch) {
    using G_ = TileGeo<WM, WN, KS>;
    typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
    typedef float f32x16_t __attribute__((ext_vector_type(16)));
    typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
    const int tid = threadIdx.x & 255, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int ks = wave >> 2, wm = wave & 1, wn = (wave >> 1) & 1;
    const int col = lane & 31, half = lane >> 5;
    const int chunks = static_cast<int>((K + 63) / 64);
    unsigned char* mine = lds + ks * G_::kGroup;

    // staging: piece i covers tile row tid / 8 + 32 i, 16-byte piece tid % 8, through
    // buffer resources over the tile's rows: the lane's offsets stay put, the chunk's is
    // scalar (no address arithmetic a load), rows past the operand's end read as zero
    const int prow = tid >> 3, ppc = tid & 7;
    // (the resources pinned to scalar registers: left to itself the compiler may compute
    // them on the vector side and loop over the lanes at every load)
    auto uniform = [](const uint16_t* p) {
        const uint64_t v = reinterpret_cast<uint64_t>(p);
        const uint64_t lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
        const uint64_t hi = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v >> 32)));
        return reinterpret_cast<uint16_t*>(hi << 32 | lo);
    };
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
        uniform(x), 0, __builtin_amdgcn_readfirstlane(static_cast<int>(xrows * K * 2)), 0x00020000);
    const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
        uniform(w), 0, __builtin_amdgcn_readfirstlane(static_cast<int>(wrows * K * 2)), 0x00020000);
    int xo[G_::XP], wo[G_::WP];
#pragma unroll
    for (int i = 0; i < G_::XP; i++) xo[i] = static_cast<int>((prow + 32 * i) * K * 2) + 16 * ppc;
#pragma unroll
    for (int i = 0; i < G_::WP; i++) wo[i] = static_cast<int>((prow + 32 * i) * K * 2) + 16 * ppc;
    const int put = prow * 128 + ((ppc ^ ((prow >> 1) & 7)) << 4);  // + 4096 i: (prow + 32 i) / 2 % 8 is the same
    u32x4_t xv[G_::XP], wv[G_::WP];
    // from the last chunk on, where that is half a chunk (k a multiple of 32, not of
    // 64): the pieces past K are put out of range and read as zero
    auto last_half = [&](int c) {
        if ((K & 63) == 0 || c != chunks - 1 || ppc < 4) return;
#pragma unroll
        for (int i = 0; i < G_::XP; i++) xo[i] |= static_cast<int>(0x80000000u);
#pragma unroll
        for (int i = 0; i < G_::WP; i++) wo[i] |= static_cast<int>(0x80000000u);
    };
    auto load1 = [&](int c, int i) {
        if (i < G_::XP)
            xv[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(xres, xo[i], 128 * c, 0));
        else
            wv[i - G_::XP] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(wres, wo[i - G_::XP], 128 * c, 0));
    };
    auto store1 = [&](int b, int i) {
        unsigned char* to = mine + b * (G_::kX + G_::kW) + put;
        if (i < G_::XP) *reinterpret_cast<u32x4_t*>(to + 4096 * i) = xv[i];
        else *reinterpret_cast<u32x4_t*>(to + G_::kX + 4096 * (i - G_::XP)) = wv[i - G_::XP];
    };
    constexpr int kAll = G_::XP + G_::WP;
    auto load = [&](int c) {
        last_half(c);
#pragma unroll
        for (int i = 0; i < kAll; i++) load1(c, i);
    };
    auto store = [&](int b) {
#pragma unroll
        for (int i = 0; i < kAll; i++) store1(b, i);
    };
    f32x16_t acc[WM][WN];
#pragma unroll
    for (int t = 0; t < WM; t++)
#pragma unroll
        for (int c = 0; c < WN; c++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[t][c][i] = 0.0f;
    const int sw = (col >> 1) & 7;
    const bool live = !PART || 32 * WM * wm < xrows;
    const int rounds = (chunks + KS - 1) / KS;
    // past the group's last chunk that chunk is repeated: stored and never read
    const int last = chunks - 1 - (chunks - 1 - ks) % KS;  // this group's last chunk (below ks: none)
    const int n_mine = ks < chunks ? (last - ks) / KS + 1 : 0;
    auto nth = [&](int j) -> int { return min(ks + j * KS, max(last, 0)); };
    load(min(nth(0), chunks - 1));
    store(0);
    load(min(nth(1), chunks - 1));
    __syncthreads();
    int b = 0;
    for (int r = 0; r < rounds; r++, b ^= 1) {
        const unsigned char* xt = mine + b * (G_::kX + G_::kW) + (32 * WM * wm + col) * 128;
        const unsigned char* wt = mine + b * (G_::kX + G_::kW) + G_::kX + (32 * WN * wn + col) * 128;
        bf16x8_t xf[2][WM], wf[2][WN];
        auto frags = [&](int s, int o) {
            const int at = ((2 * s + half) ^ sw) << 4;  // k 16 s + 8 half .. of a row: piece 2 s + half
#pragma unroll
            for (int t = 0; t < WM; t++) xf[o][t] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(xt + 4096 * t + at));
#pragma unroll
            for (int q = 0; q < WN; q++) wf[o][q] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(wt + 4096 * q + at));
        };
        if (KS == 1 || r < n_mine) {
            const int next = min(nth(r + 2), chunks - 1);
            last_half(next);
            if (live) frags(0, 0);
#pragma unroll
            for (int s = 0; s < 4; s++) {
                if (s < 3 && live) frags(s + 1, (s + 1) & 1);
#pragma unroll
                for (int i = kAll * s / 4; i < kAll * (s + 1) / 4; i++) {
                    store1(b ^ 1, i);
                    load1(next, i);
                }
#pragma unroll
                for (int q = 0; q < WN && live; q++)
#pragma unroll
                    for (int t = 0; t < WM; t++)
                        acc[t][q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[s & 1][q], xf[s & 1][t], acc[t][q], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
    }
    if constexpr (KS > 1) {
        float* red = reinterpret_cast<float*>(lds);
        const int w4 = wave & 3;
        if (ks > 0) {
#pragma unroll
            for (int t = 0; t < WM; t++)
#pragma unroll
                for (int c = 0; c < WN; c++)
#pragma unroll
                    for (int i = 0; i < 16; i++)
                        red[((((ks - 1) * 4 + w4) * WM * WN + t * WN + c) * 16 + i) * 64 + lane] = acc[t][c][i];
        }
        __syncthreads();
        if (ks == 0) {
#pragma unroll
            for (int q = 0; q < KS - 1; q++)
#pragma unroll
                for (int t = 0; t < WM; t++)
#pragma unroll
                    for (int c = 0; c < WN; c++)
#pragma unroll
                        for (int i = 0; i < 16; i++)
                            acc[t][c][i] += red[(((q * 4 + w4) * WM * WN + t * WN + c) * 16 + i) * 64 + lane];
        }
        __syncthreads();
        if (ks > 0) return;
    }
    // acc[t][c][i]: row 32 t + col, column 32 c + 8 (i / 4) + 4 half + i % 4 of the wave's part:
    // through LDS (wave-private) into whole row segments
    unsigned char* ot = lds + (wave & 3) * 32 * WM * G_::kRowPitch;
    const int mw = 32 * WM * wm, nw = 32 * WN * wn;
#pragma unroll
    for (int c = 0; c < WN; c++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            float bv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (bias)
#pragma unroll
                for (int j = 0; j < 4; j++) bv[j] = bf16_to_f32(bias[min(nw + 32 * c + 8 * q + 4 * half + j, wrows - 1)]);
#pragma unroll
            for (int t = 0; t < WM; t++)
                *reinterpret_cast<uint2*>(ot + (32 * t + col) * G_::kRowPitch + 2 * (32 * c + 8 * q + 4 * half)) =
                    make_uint2(pack_bf16x2(acc[t][c][4 * q] + bv[0], acc[t][c][4 * q + 1] + bv[1]),
                               pack_bf16x2(acc[t][c][4 * q + 2] + bv[2], acc[t][c][4 * q + 3] + bv[3]));
        }
    __builtin_amdgcn_wave_barrier();
    if ((pitch & 7) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0) {
        constexpr int kLanes = 4 * WN;  // lanes per row, 8 columns each
#pragma unroll
        for (int i = 0; i < 32 * WM * kLanes / 64; i++) {
            const int r = (64 * i + lane) / kLanes, c8 = 8 * ((64 * i + lane) % kLanes);
            const u32x4_t v = *reinterpret_cast<const u32x4_t*>(ot + r * G_::kRowPitch + 2 * c8);
            if (mw + r >= xrows || nw + c8 >= wrows) continue;
            *reinterpret_cast<u32x4_t*>(out + (mw + r) * pitch + nw + c8) = v;
        }
        return;
    }
    // rows of other alignments: two columns a lane or one, so that neighbouring lanes
    // still write neighbouring columns (eight two-byte stores a lane, 16 bytes apart, took
    // 116 us for 2191 x 29614 x 32 where this takes 54; 946 x 13341 x 512 46 -> 37)
    auto put_rows = [&](auto width) {
        constexpr int W = decltype(width)::value, kLanes = 32 * WN / W;
        using Piece = std::conditional_t<W == 2, uint32_t, uint16_t>;
#pragma unroll 1
        for (int i0 = 0; i0 < 32 * WM * kLanes / 64; i0 += 8) {
            Piece v[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int at = 64 * (i0 + i) + lane;
                v[i] = *reinterpret_cast<const Piece*>(ot + at / kLanes * G_::kRowPitch + 2 * W * (at % kLanes));
            }
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int at = 64 * (i0 + i) + lane, r = mw + at / kLanes, c = nw + W * (at % kLanes);
                if (r < xrows && c < wrows) *reinterpret_cast<Piece*>(out + r * pitch + c) = v[i];
            }
        }
    };
    if ((pitch & 1) == 0 && (reinterpret_cast<uintptr_t>(out) & 3) == 0) put_rows(std::integral_constant<int, 2>{});
    else put_rows(std::integral_constant<int, 1>{});
}

} // namespace sandy_hip
