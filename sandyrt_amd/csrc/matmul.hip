// matmul.hip -- dense matmul and linear (the projections and the lm-head).
//
// Semantics (src/core/TensorCalc.cpp):
//   matmul 804-919   for every batch of the broadcast batch shape
//                    (ShapeUtil.cpp:39-71; a smaller batch dim d serves
//                    batch/d consecutive output coordinates, TensorCalc.cpp:
//                    213-240), out[m, n] = sum over k in order of
//                    lhs[m, k] * rhs[k, n], either operand read transposed;
//                    float accumulation
//   linear 722-773   out[r, o] = bias[o] + sum over i in order of
//                    x[r, i] * w[o, i]
// Validation follows launch_cuda_matmul (src/device/cuda/
// CudaMatMulKernels.cu:78-141): same float dtype, contiguous views, rank >= 2,
// matching contracting dims and the exact output shape.
//
// The reference hands both to cuBLAS (cublasGemmEx, CudaMatMulKernels.cu:
// 173-216; its CUDA linear is not implemented, CudaDevice.cpp:536-537).
// Here there are four kernels:
//   - bf16 with the weight read row-major as [n, k] (transpose_rhs, the
//     layout of every projection and the lm-head) runs on bf16 MFMA with fp32
//     accumulation:
//       gemm_waves_kernel for decode-sized products (up to 64 rows),
//         v_mfma_f32_16x16x32_bf16: weight streams, HBM-bound, K split over the waves of a workgroup and, when
//         the column tiles alone cannot fill the chip, over workgroups, with
//         the last-arriving workgroup of each output tile summing the fp32
//         partials in split order -- one launch, no second reduction pass;
//       gemm_tile_kernel for larger row counts, v_mfma_f32_32x32x16_bf16: tiles
//         up to 128 x 192;
//   - f32 in the same layout runs gemm_ordered_kernel, FMA-free float loops
//     that keep the reference's k order per output, so f32 results are
//     bit-identical to the CPU path;
//   - gemm_simt_kernel: every other case (other layouts, unaligned shapes, f32 of
//     short contractions and many outputs), register-tiled, in the same order.
#include "gemm.h"
#include "gemm_tile.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>

namespace sandy_hip {
namespace {

// decode GEMM workgroups resident at once (two per CU on the 256 CUs)
constexpr int64_t kWavesResident = 512;

// The tile of gemm_tile.h over a dense product.
template <int WM, int WN, int KS>
__global__ __launch_bounds__(256 * KS, 2) void gemm_tile_kernel(GemmArgs g) {
    using G_ = TileGeo<WM, WN, KS>;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    // workgroups are dealt round-robin to the 8 XCDs: each XCD takes a run of
    // neighbouring tiles, rows fastest, so its L2 serves the weight tile to every row
    // tile.  The products of a batch follow one another in that run: each product's
    // tiles dealt out by themselves, those of one to eight tiles left XCDs idle
    const int tiles = g.row_tiles * g.col_tiles, all = tiles * g.splits, per = (all + 7) / 8;
    int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (static_cast<int>(blockIdx.x >> 3) >= per || tile >= all) return;
    int64_t product = blockIdx.z;
    if (g.splits > 1) {
        product = tile / tiles;
        tile -= static_cast<int>(product) * tiles;
    }
    const int64_t m0 = static_cast<int64_t>(tile % g.row_tiles) * G_::BM, n0 = static_cast<int64_t>(tile / g.row_tiles) * G_::BN;
    int64_t lo, ro;
    batch_offsets(g.bm, product, lo, ro);
    const int64_t M = g.M, N = g.N, K = g.K;
    gemm_tile<WM, WN, KS, false>(lds, g.a + lo + m0 * K, static_cast<int>(min<int64_t>(G_::BM, M - m0)), g.w + ro + n0 * K,
                                 static_cast<int>(min<int64_t>(G_::BN, N - n0)), K, g.bias ? g.bias + n0 : nullptr,
                                 g.out + (product * M + m0) * N + n0, N);
}

// Any dtype, either operand transposed: 64 x 64 output tile per workgroup,
// 4 x 4 outputs per thread, k staged 16 at a time through LDS.  Each output
// is acc = (bias or 0) then acc = acc + a * b over k in order (no FMA
// contraction), the reference's loop exactly.
template <typename T>
__global__ __launch_bounds__(256) void gemm_simt_kernel(const void* __restrict__ lhs, const void* __restrict__ rhs,
                                                        const void* __restrict__ bias, void* __restrict__ out,
                                                        int64_t M, int64_t N, int64_t K, int32_t tl, int32_t tr,
                                                        int64_t lrs, int64_t rrs, BatchMap bm) {
    constexpr int kT = 64, kK = 16;
    __shared__ float As[kK][kT + 4];
    __shared__ float Bs[kK][kT + 4];
    const int tid = threadIdx.x;
    const int tx = tid & 15, ty = tid >> 4;
    const int64_t m0 = static_cast<int64_t>(blockIdx.y) * kT, n0 = static_cast<int64_t>(blockIdx.x) * kT;
    const int64_t bz = blockIdx.z;
    int64_t lo, ro;
    batch_offsets(bm, bz, lo, ro);
    float acc[4][4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int64_t n = n0 + tx + 16 * j;
        const float b0 = bias && n < N ? Vec8<T>::load1(bias, n) : 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i][j] = b0;
    }
    for (int64_t k0 = 0; k0 < K; k0 += kK) {
        // 1024 elements of each operand tile, 4 per thread; the fast index
        // follows the operand's contiguous dimension
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int e = tid + 256 * q;
            int mm, kk;
            if (tl) { mm = e & 63; kk = e >> 6; } else { kk = e & 15; mm = e >> 4; }
            const int64_t gm = m0 + mm, gk = k0 + kk;
            float v = 0.0f;
            if (gm < M && gk < K) v = Vec8<T>::load1(lhs, lo + (tl ? gk * lrs + gm : gm * lrs + gk));
            As[kk][mm] = v;
            int nn;
            if (tr) { kk = e & 15; nn = e >> 4; } else { nn = e & 63; kk = e >> 6; }
            const int64_t gn = n0 + nn, gk2 = k0 + kk;
            float w = 0.0f;
            if (gn < N && gk2 < K) w = Vec8<T>::load1(rhs, ro + (tr ? gn * rrs + gk2 : gk2 * rrs + gn));
            Bs[kk][nn] = w;
        }
        __syncthreads();
        const int kn = static_cast<int>(min<int64_t>(kK, K - k0));
        for (int kk = 0; kk < kn; kk++) {
            float av[4], bv[4];
#pragma unroll
            for (int i = 0; i < 4; i++) av[i] = As[kk][ty + 16 * i];
#pragma unroll
            for (int j = 0; j < 4; j++) bv[j] = Bs[kk][tx + 16 * j];
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = __fadd_rn(acc[i][j], __fmul_rn(av[i], bv[j]));
        }
        __syncthreads();
    }
    const int64_t ob = bz * M * N;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int64_t m = m0 + ty + 16 * i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t n = n0 + tx + 16 * j;
            if (n < N) Vec8<T>::store1(out, ob + m * N + n, acc[i][j]);
        }
    }
}

// f32 products against a weight read as [n, k] (linear, and matmul with
// transpose_rhs) in the reference's k order: every output is acc = (bias or
// 0), then acc + x * w rounded at each step (no FMA), so results stay
// bit-identical to the CPU path and MFMA, which sums in another order, is out.
// Bound: two VALU instructions a multiply-add, 39 TFLOP/s over 1024 SIMDs; a
// single output's chain alone takes 8 K cycles, so small products want one
// output a lane on as many SIMDs as there are, large ones R rows a lane to
// amortise the operand reads.  A wave owns R rows x 64 columns; chunks of 64 k
// of its operands go global -> registers (a ring of kRing chunks, so that the
// weight stream stays in flight over several short chunks) -> LDS.  A lane
// reads its column 4 k at a time, and of each row the 4 k that its place in a
// quad of lanes names: the multiply takes the quad's lane j by DPP, so an
// activation costs one 16-byte LDS read per 16 k and no instruction of its own.
// Measured (before: 64 x 64 tiles, and one wave per 16 columns up to 8 rows):
// 64 x 768 x 768 119 -> 12 us, 64 x 768 x 3072 542 -> 36, 1000 x 3072 x 768 at
// 35 TFLOP/s, 1 x 50257 x 768 62 -> 33.
typedef float f32v4_t __attribute__((ext_vector_type(4)));

// lane (4 (lane / 4) + Q)'s v
template <int Q>
__device__ __forceinline__ float quad_lane(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), Q * 0x55, 0xf, 0xf, true));
}

template <int R>
__global__ __launch_bounds__(256, R == 1 ? 2 : 3) void gemm_ordered_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                           const float* __restrict__ bias, float* __restrict__ out,
                                                           int64_t M, int64_t N, int64_t K, int32_t row_tiles,
                                                           BatchMap bm) {
    constexpr int kBK = 64;                      // k per chunk
    constexpr int kPitch = kBK + 4;              // floats per weight row in LDS: 64 lanes x 16 bytes, no conflict
    constexpr int kRows = 4 * R;                 // rows and columns of the workgroup
    constexpr int kCols = 64;
    constexpr int kW = kCols * kBK / 4 / 256;    // 16-byte pieces of w a thread stages per chunk
    constexpr int kX = (kRows * kBK / 4 + 255) / 256;
    constexpr int kRing = R == 1 ? 3 : 2;
    static_assert(R <= 4, "x pieces of a chunk: at most one a thread");
    __shared__ __attribute__((aligned(16))) float wl[2][kCols * kPitch];
    __shared__ __attribute__((aligned(16))) float xl[2][kRows * kBK];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t r0 = static_cast<int64_t>(blockIdx.x % row_tiles) * kRows, m0 = r0 + wave * R;
    const int64_t n0 = static_cast<int64_t>(blockIdx.x / row_tiles) * kCols, n = n0 + lane;
    int64_t lo, ro;
    batch_offsets(bm, blockIdx.z, lo, ro);
    const int prow = tid / 16, ppc = tid % 16;   // piece (row prow + 16 i, 4 ppc .. + 3) of a chunk
    const float* wp[kW];
    const float* xp[kX];
#pragma unroll
    for (int i = 0; i < kW; i++) wp[i] = w + ro + min<int64_t>(n0 + prow + 16 * i, N - 1) * K;
#pragma unroll
    for (int i = 0; i < kX; i++) xp[i] = x + lo + min<int64_t>(r0 + prow + 16 * i, M - 1) * K;
    const bool x_on = kRows >= 16 || prow < kRows;
    f32v4_t wv[kRing][kW], xv[kRing][kX];
    auto load = [&](int64_t c, int slot) {
        const int64_t k = min<int64_t>(c * kBK + 4 * ppc, K - 4);  // pieces past K are not used
#pragma unroll
        for (int i = 0; i < kW; i++) wv[slot][i] = *reinterpret_cast<const f32v4_t*>(wp[i] + k);
#pragma unroll
        for (int i = 0; i < kX; i++) xv[slot][i] = *reinterpret_cast<const f32v4_t*>(xp[i] + k);
    };
    float acc[R];
    float b0 = bias && n < N ? bias[n] : 0.0f;
    asm volatile("" : "+v"(b0));  // waited for here, not (with the weights in flight) in the loop
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = b0;
    const float* wr = &wl[0][lane * kPitch];
    const float* xr = &xl[0][wave * R * kBK + 4 * (lane & 3)];
    auto put = [&](int slot, int buf) {
#pragma unroll
        for (int i = 0; i < kW; i++)
            *reinterpret_cast<f32v4_t*>(&wl[buf][(prow + 16 * i) * kPitch + 4 * ppc]) = wv[slot][i];
        if (x_on) {
#pragma unroll
            for (int i = 0; i < kX; i++) *reinterpret_cast<f32v4_t*>(&xl[buf][(prow + 16 * i) * kBK + 4 * ppc]) = xv[slot][i];
        }
        __syncthreads();
    };
    // 16 k (the first 4 `quads` of them) of the chunk in `buf`
    const bool live = m0 < M;  // a wave past the last row only stages
    auto sixteen = [&](int buf, int s, int quads) {
        f32v4_t a[R];
#pragma unroll
        for (int r = 0; r < R; r++) a[r] = *reinterpret_cast<const f32v4_t*>(xr + buf * kRows * kBK + r * kBK + 16 * s);
        auto step = [&](auto quad) {
            constexpr int q = decltype(quad)::value;
            if (q >= quads) return;
            const f32v4_t b = *reinterpret_cast<const f32v4_t*>(wr + buf * kCols * kPitch + 16 * s + 4 * q);
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int r = 0; r < R; r++) acc[r] = __fadd_rn(acc[r], __fmul_rn(quad_lane<q>(a[r][j]), b[j]));
        };
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
    };
    auto whole = [&](int buf) {
        if (!live) return;
#pragma unroll
        for (int s = 0; s < kBK / 16; s++) sixteen(buf, s, 4);
    };
    // rings of whole chunks, every load unconditional so that the wait counts
    // stay exact (past the last chunk its pieces are loaded again); then the
    // chunks left, the last of them perhaps partial
    const int64_t chunks = (K + kBK - 1) / kBK, full = K / kBK;
#pragma unroll
    for (int q = 0; q < kRing; q++) load(q, q);
    int64_t c = 0;
    int buf = 0;
    for (; c + kRing <= full; c += kRing) {
#pragma unroll
        for (int slot = 0; slot < kRing; slot++) {
            put(slot, buf);
            load(c + kRing + slot, slot);
            whole(buf);
            buf ^= 1;
        }
    }
#pragma unroll
    for (int slot = 0; slot < kRing; slot++) {
        if (c + slot < chunks) {
            put(slot, buf);
            const int quads = static_cast<int>(min<int64_t>(kBK, K - (c + slot) * kBK) / 4);
#pragma unroll 1
            for (int s = 0; live && 4 * s < quads; s++) sixteen(buf, s, quads - 4 * s);
            buf ^= 1;
        }
    }
    if (n >= N) return;
#pragma unroll
    for (int r = 0; r < R; r++)
        if (m0 + r < M) out[(static_cast<int64_t>(blockIdx.z) * M + m0 + r) * N + n] = acc[r];
}

// --------------------------------------------------------------------- host
struct Plan {
    int64_t M, N, K, batches;
    int64_t lrs, rrs;  // row strides (last dims) of lhs and rhs
    BatchMap bm;
};

// Fills the plan from operand shapes with the reference's rules; returns an
// error message or null.
const char* plan_matmul(const SandyTensor& l, const SandyTensor& r, const SandyTensor& o, bool tl, bool tr, Plan& p) {
    const int lr = l.rank, rr = r.rank;
    if (lr < 2) return "matmul lhs must have rank >= 2";
    if (rr < 2) return "matmul rhs must have rank >= 2";
    p.M = l.dims[lr - (tl ? 1 : 2)];
    const int64_t lk = l.dims[lr - (tl ? 2 : 1)];
    const int64_t rk = r.dims[rr - (tr ? 1 : 2)];
    p.N = r.dims[rr - (tr ? 2 : 1)];
    if (p.M < 0 || p.N < 0 || lk < 0 || rk < 0) return "matmul matrix dimensions must be static";
    if (lk != rk) return "matmul contracting dimension mismatch";
    p.K = lk;
    const int lb = lr - 2, rb = rr - 2;
    const int brank = std::max(lb, rb);
    if (o.rank != brank + 2) return "matmul output shape mismatch";
    BatchMap& m = p.bm;
    m.rank = brank;
    p.batches = 1;
    // contiguous strides of each operand's batch dims
    int64_t ls[SANDY_HIP_MAX_RANK], rs[SANDY_HIP_MAX_RANK];
    int64_t s = l.dims[lr - 1] * l.dims[lr - 2];
    for (int d = lb - 1; d >= 0; d--) { ls[d] = s; s *= l.dims[d]; }
    s = r.dims[rr - 1] * r.dims[rr - 2];
    for (int d = rb - 1; d >= 0; d--) { rs[d] = s; s *= r.dims[d]; }
    for (int i = 0; i < brank; i++) {
        const int li = lb - brank + i, ri = rb - brank + i;
        const int64_t a = li >= 0 ? l.dims[li] : 1, b = ri >= 0 ? r.dims[ri] : 1;
        int64_t d;
        if (a == b) d = a;
        else if (a == 1) d = b;
        else if (b == 1) d = a;
        else if (a > b && a % b == 0) d = a;
        else if (b > a && b % a == 0) d = b;
        else return "cannot broadcast matmul batch shapes";
        m.dims[i] = d;
        m.l_stride[i] = (li >= 0 && a != 1) ? ls[li] : 0;
        m.l_div[i] = (li >= 0 && a != 1) ? d / a : 1;
        m.r_stride[i] = (ri >= 0 && b != 1) ? rs[ri] : 0;
        m.r_div[i] = (ri >= 0 && b != 1) ? d / b : 1;
        if (o.dims[i] != d) return "matmul output shape mismatch";
        p.batches *= d;
    }
    if (o.dims[brank] != p.M || o.dims[brank + 1] != p.N) return "matmul output shape mismatch";
    p.lrs = l.dims[lr - 1];
    p.rrs = r.dims[rr - 1];
    return nullptr;
}

// The decode GEMM's fused forms: a residual-add epilogue with row sums of
// squares, and an RMSNorm prologue from such sums.
struct Fusion {
    const uint16_t* resid = nullptr;
    double* rsq_out = nullptr;
    int64_t rsq_parts = 0;
    const double* rsq_in = nullptr;
    int64_t rsq_in_parts = 0;
    const uint16_t* norm_w = nullptr;
    float eps = 0.0f;
    const QkvRope* qr = nullptr;  // q/k/v RoPE + paged-append epilogue
    bool dry = false;             // every check and workspace, no launch
};

int launch(const Plan& p, const SandyTensor& l, const SandyTensor& r, const SandyTensor* bias, const SandyTensor& o,
           bool tl, bool tr, hipStream_t stream, Err e, const char* what, int glu = 0, const Fusion* fz = nullptr) {
    if (p.batches == 0 || p.M == 0 || p.N == 0) return ok(e);
    if (p.batches > 65535) return fail(e, SANDY_ERR_UNSUPPORTED, "%s batch count exceeds 65535", what);
    const void* pl = base_ptr(l);
    const void* pr = base_ptr(r);
    const void* pb = bias ? base_ptr(*bias) : nullptr;
    void* po = base_ptr(o);
    const bool aligned = ((reinterpret_cast<uintptr_t>(pl) | reinterpret_cast<uintptr_t>(pr)) & 15) == 0;
    const bool lines = l.dtype == SANDY_BF16 && !tl && tr && p.K % 32 == 0 && p.K > 0 && aligned &&
                       p.K <= (int64_t{1} << 21) && env_int("SANDY_GEMM_SIMT", 0) == 0;
    const bool waves = lines && env_int("SANDY_GEMM_WAVES", p.M <= 64 ? 1 : 0) != 0;
    if ((glu || fz) && !waves)
        return fail(e, SANDY_ERR_UNSUPPORTED, "%s needs bf16 operands, k a multiple of 32 and at most 64 rows", what);
    if (fz && p.batches != 1) return fail(e, SANDY_ERR_UNSUPPORTED, "%s takes one [m, k] matrix", what);
    const bool norm = fz && fz->norm_w;
    // f32 against a weight read as [n, k], in the reference's k order
    // (short contractions with many outputs: the 64 x 64 tiles of gemm_simt_kernel, in the
    // same order, reread the operands less and fill whole store lines.  us, ordered / simt:
    // 1000 x 16000 x 16 49 / 26, 1000 x 4000 x 48 21 / 17, 2000 x 8000 x 96 105 / 97,
    // 1461 x 8606 x 20 44 / 32; k 128 even, 2000 x 8000 x 256 233 / 245; 1000 x 1000 x 24
    // 7.3 / 8.4.  The shorter the contraction, the sooner, and few columns count as the
    // tiles they fill: k 8 235 products of 149 x 12 10.6 / 6.1, 395 x 4689 8.4 / 6.2, k 12
    // 2375 x 834 11.0 / 8.0, k 32 298 of 151 x 5 15.0 / 11.2; k 16 364 x 1849 5.3 / 6.6,
    // 500 x 1837 even, k 24 1012 x 950 7.6 / 8.5, k 32 148 x 9429 9.8 / 10.2)
    const int64_t filled = (p.M + 15) / 16 * 16 * ((p.N + 63) / 64 * 64) * p.batches;
    const bool short_wide = p.M > 8 && p.M <= 65535 * 64 &&
                            ((p.K <= 96 && p.M * p.N * p.batches >= (2 << 20)) || (p.K <= 32 && filled >= (2 << 20)) ||
                             (p.K <= 16 && filled >= 1000000));
    const bool ordered = l.dtype == SANDY_F32 && !tl && tr && p.K % 4 == 0 && p.K > 0 && aligned && !short_wide &&
                         env_int("SANDY_GEMM_SIMT", 0) == 0;
    if (ordered) {
        // one row a lane while that takes at most two waves a SIMD, else four
        // (one wave alone issues a VALU instruction every 7 cycles, several
        // every 4, so small products want more waves, not more rows a wave):
        // us at R = 1 / 4 for rows x columns x k: 64 x 768 x 768 12 / 20,
        // 64 x 768 x 3072 36 / 71, 1 x 50257 x 768 33 / 43; 64 x 3072 x 768
        // 25 / 22, 200 x 768 x 768 23 / 21, 1000 x 3072 x 768 258 / 136
        const int64_t ct = (p.N + 63) / 64;
        const int R = env_int("SANDY_GEMM_ROWS", p.M * ct * p.batches <= 2048 ? 1 : 4) == 1 ? 1 : 4;
        const int64_t rt = (p.M + 4 * R - 1) / (4 * R);
        if (rt * ct > 0x7fffffff) return fail(e, SANDY_ERR_UNSUPPORTED, "%s shape exceeds the launch grid", what);
        const dim3 grid(static_cast<unsigned>(rt * ct), 1, static_cast<unsigned>(p.batches));
        hipLaunchKernelGGL(R == 1 ? gemm_ordered_kernel<1> : gemm_ordered_kernel<4>, grid, dim3(256), 0, stream,
                           static_cast<const float*>(pl), static_cast<const float*>(pr), static_cast<const float*>(pb),
                           static_cast<float*>(po), p.M, p.N, p.K, static_cast<int32_t>(rt), p.bm);
    } else if (waves) {
        GemmArgs g{};
        g.a = static_cast<const uint16_t*>(pl);
        g.w = static_cast<const uint16_t*>(pr);
        g.bias = static_cast<const uint16_t*>(pb);
        g.out = static_cast<uint16_t*>(po);
        g.M = p.M;
        g.N = p.N;
        g.K = p.K;
        g.bm = p.bm;
        g.glu = glu;
        if (fz) {
            g.resid = fz->resid;
            g.rsq_out = fz->rsq_out;
            g.rsq_parts = fz->rsq_parts;
            g.rsq_in = fz->rsq_in;
            g.rsq_in_parts = fz->rsq_in_parts;
            g.norm_w = fz->norm_w;
            g.eps = fz->eps;
            if (fz->qr) g.qr = *fz->qr;
        }
        // tile: 16 * RT rows x 16 * CT columns, variants (RT, CT) = 0 (1, 1),
        // 1 (2, 1), 3 (2, 2), 4 (1, 2), 5 (2, 4), 6 (1, 4), 7 (4, 2; no norm
        // prologue) -- the ones the heuristic below picks (2 is unused); SANDY_GEMM_TILE / SANDY_GEMM_CPS
        // select one of them and a run length for the tests that cover every
        // instantiated form
        static const int kRT[] = {1, 2, 2, 2, 1, 2, 1, 4};
        static const int kCT[] = {1, 1, 1, 2, 2, 4, 4, 2};
        const int64_t chunks = (p.K / 32 + 1) / 2;
        const bool qkv = fz && fz->qr;
        int variant = env_int("SANDY_GEMM_TILE", -1);
        int cps = env_int("SANDY_GEMM_CPS", 0);
        // K: at most 32 chunks (2048 k) per workgroup, split evenly; the
        // per-wave run is rounded up to a built run length
        int64_t ksplits = (chunks + 31) / 32;
        // chunks in flight per wave (4 only for RT * CT <= 2, register bound)
        int qdepth = 2;
        if (variant < 0 || variant > (norm ? 6 : 7) || variant == 2) {
            // Measured on decode shapes with the weights streamed from HBM
            // (rotated over >= 1 GiB of copies):
            //   <= 16 rows: 16 x 16 tiles, 16 x 32 from N >= 16384 (lm-head);
            //   <= 32 rows: 16-row tiles (the second row tile re-reads the
            //     weights from cache), 32 columns from N K >= 5M; 17..32 rows
            //     of N K >= 16M without the norm prologue: one 32-row tile
            //     (weights streamed once);
            //   weights past 64 MB at 32 rows, and batches of 33..64 rows:
            //     32-row tiles, the widest column tile giving >= 120 workgroups;
            //   one product of 33..64 rows (us at 48 / 64 rows, that rule ->
            //     here; the run length and so the sums stay the same): 16 x 16
            //     tiles, four chunks in flight, for weights under 6M elements
            //     (2560 x 2048 8.9 / 9.0 -> 7.5, 1024 x 4096 12.0 / 12.3 -> 8.8,
            //     with the norm prologue 2048 x 2048 11.3 / 12.3 -> 8.4 / 8.9);
            //     32 x 16 up to 20M (5632 x 2048 13.1 -> 9.1 / 9.5, 2048 x 5632
            //     19.4 -> 12.6 / 13.2; not measured with the prologue, which keeps
            //     that rule); 32 x 32 up to 64 MB (11264 x 2048 20.8 / 22.2 -> 15.2 /
            //     15.9, with the prologue 23.4 / 24.8 -> 18.3 / 19.6; 2560 x 10240
            //     30.6 / 32.4 -> 23.1 / 24.7); past it 64 x 32, so that the weights
            //     stream once (32000 x 2048 43.7 / 44.5 -> 33.3 / 36.3, 14336 x 4096
            //     52.0 / 54.2 -> 45.9 / 49.3; the prologue's work would grow with the
            //     rows) -- up to k 4096: with more, and so more splits of K, it loses
            //     (42 x 7616 x 6368 55 against 62, 45 x 14578 x 5408 71 against 76; with
            //     the prologue 33 x 4512 x 5536 41 against 43) and that rule stays;
            //   4 chunks in flight per wave for weights under 8M elements
            //   (o projection at 32 rows 8.3 -> 6.1 us, q/k/v at one row
            //   7.4 -> 5.5 us), 2 for the larger ones;
            //   up to 32 rows with K past 2048: up to 48 chunks per
            //   workgroup and 4 in flight (down projection, 5632 x 2048: two
            //   K splits of runs of 12 against three of 8; 32 rows
            //   12.8 -> 11.6 us, one row 9.2 -> 8.7 us).
            const bool big = p.N * p.K * 2 > (int64_t(64) << 20);
            constexpr int64_t kSmall = 6 << 20, kMiddle = 20 << 20;  // weight elements
            const bool long_big = p.K > 4096 && (big || (norm && p.N * p.K > kMiddle));
            int64_t rt = 1, ct = 1;
            if (p.M <= 16 && !big) {
                ct = p.N >= 16384 ? 2 : 1;
                qdepth = 4;
                if (chunks > 32) ksplits = (chunks + 47) / 48;
            } else if (p.M <= 32 && !big && !norm && p.M > 16 && p.N * p.K >= 16 * (int64_t(1) << 20) && chunks <= 32) {
                // 17..32 rows of a wide projection (gate/up, 2048 x 11264): one
                // 32-row tile, so the weights stream once, non-temporal, with four
                // chunks in flight (15.2 -> 14.2 us; two 16-row tiles re-read
                // them from L2 and must keep them cached).  Not with the RMSNorm
                // prologue, whose work grows with the rows of a tile (gated
                // gate/up 17.0 -> 18.2 us)
                rt = 2;
                qdepth = 4;
            } else if (p.M <= 32 && !big) {
                ct = p.N * p.K >= 5 * (int64_t(1) << 20) ? 2 : 1;
                qdepth = p.N * p.K < 8 * (int64_t(1) << 20) ? 4 : 2;
                if (chunks > 32) {
                    ksplits = (chunks + 47) / 48;
                    qdepth = 4;
                }
            } else if (p.M > 32 && p.batches == 1 && !qkv && !long_big && (!norm || (!big && (p.N * p.K < kSmall || p.N * p.K > kMiddle)))) {
                rt = p.N * p.K < kSmall ? 1 : big ? 4 : 2;
                ct = p.N * p.K <= kMiddle ? 1 : 2;
                qdepth = p.N * p.K < kSmall ? 4 : 2;
            } else {
                rt = p.M <= 16 ? 1 : 2;
                const int64_t rows = (p.M + 16 * rt - 1) / (16 * rt) * p.batches;
                for (int c : {4, 2}) {
                    if ((p.N + 16 * c - 1) / (16 * c) * rows * ksplits >= 120) {
                        ct = c;
                        break;
                    }
                }
            }
            static const int kPick[2][3] = {{0, 4, 6}, {1, 3, 5}};  // [RT 1/2][CT 1/2/4]
            variant = rt == 4 ? 7 : kPick[rt == 1 ? 0 : 1][ct == 1 ? 0 : ct == 2 ? 1 : 2];
        }
        qdepth = env_int("SANDY_GEMM_Q", qdepth);
        // the q/k/v epilogue kernels: 16-row tiles of 16 or 32 columns
        if (qkv) variant = kCT[variant] == 1 ? 0 : 4;
        const int RT = kRT[variant], CT = kCT[variant];
        const int64_t row_tiles = (p.M + 16 * RT - 1) / (16 * RT);
        const int64_t col_tiles = (p.N + 16 * CT - 1) / (16 * CT);
        if (row_tiles > 65535 || col_tiles > (1 << 24))
            return fail(e, SANDY_ERR_UNSUPPORTED, "%s shape exceeds the launch grid", what);
        const int64_t tiles = row_tiles * col_tiles * p.batches;
        if (cps <= 0) cps = static_cast<int>(((chunks + ksplits - 1) / ksplits + 3) / 4);
        // built run lengths: per-split chunks are at most 48 (cps <= 12)
        static const int kRuns[] = {2, 3, 4, 5, 6, 8, 10, 12};
        int run = 12;
        for (int r : kRuns) {
            if (r >= cps) {
                run = r;
                break;
            }
        }
        cps = run;
        const int64_t splits = (chunks + 4 * cps - 1) / (4 * cps);
        g.col_tiles = static_cast<int32_t>(col_tiles);
        g.row_tiles = static_cast<int32_t>(row_tiles);
        g.splits = static_cast<int32_t>(splits);
        g.split_chunks = 4 * cps;
        if (col_tiles * splits > 0x7fffffff) return fail(e, SANDY_ERR_UNSUPPORTED, "%s shape exceeds the launch grid", what);
        if (splits > 1) {
            int status = 0;
            const size_t part = static_cast<size_t>(tiles * splits) * RT * CT * 64 * 4 * sizeof(float);
            g.part = static_cast<float*>(device_workspace(4, part, stream, e, &status));
            if (status) return status;
            g.counters = static_cast<uint32_t*>(device_counters(1, static_cast<size_t>(tiles) * sizeof(uint32_t), stream, e, &status));
            if (status) return status;
        }
        const dim3 grid(static_cast<unsigned>(col_tiles * splits), static_cast<unsigned>(row_tiles),
                        static_cast<unsigned>(p.batches));
        // the weight stream non-temporal where nothing re-reads it from L2 later:
        // one row tile, or every workgroup resident at once (the row tiles of a
        // column tile run together); measured at 1 row: q/k/v 5.2 -> 4.6 us,
        // o 5.1 -> 4.5, gate/up 10.4 -> 9.3, down 8.5 -> 7.8; at 32 rows the
        // 704-workgroup gate/up re-reads its weights after 352 other workgroups
        // (15.3 -> 16.5 us non-temporal) and keeps the default policy
        // (batched products may share one rhs across the batch: only a single
        // matrix counts as read once when the grid is not resident at once)
        const bool nt = (row_tiles == 1 && p.batches == 1) || col_tiles * splits * row_tiles * p.batches <= kWavesResident;
        if (qkv) {
            int status = 0;
            g.qr.arrivals = static_cast<uint32_t*>(
                device_counters(3, static_cast<size_t>(row_tiles) * sizeof(uint32_t), stream, e, &status));
            if (status) return status;
            // column tiles holding a k or v column, times the K splits
            const int64_t q_cols = static_cast<int64_t>(g.qr.hq) * g.qr.d;
            g.qr.kv_arrivals = static_cast<int32_t>((col_tiles - std::min<int64_t>(col_tiles, q_cols / (16 * CT))) * splits);
            if (fz->dry) return ok(e);
            if (nt) launch_waves_qkv<true>(variant, cps, qdepth, norm, grid, stream, g);
            else launch_waves_qkv<false>(variant, cps, qdepth, norm, grid, stream, g);
        } else if (norm) {
            if (nt) launch_waves_norm<true>(variant, cps, qdepth, grid, stream, g);
            else launch_waves_norm<false>(variant, cps, qdepth, grid, stream, g);
        } else {
            if (nt) launch_waves_plain<true>(variant, cps, qdepth, grid, stream, g);
            else launch_waves_plain<false>(variant, cps, qdepth, grid, stream, g);
        }
        SANDY_HIP_TRY(hipGetLastError(), e, what);
        return ok(e);
    } else if (lines) {
        GemmArgs g{};
        g.a = static_cast<const uint16_t*>(pl);
        g.w = static_cast<const uint16_t*>(pr);
        g.bias = static_cast<const uint16_t*>(pb);
        g.out = static_cast<uint16_t*>(po);
        g.M = p.M;
        g.N = p.N;
        g.K = p.K;
        g.bm = p.bm;
        // The tile form with the least estimated time: its chunks of 64 k (over its
        // KS groups) times the time of one plus the tile's own (first loads, output),
        // `alone` up to one workgroup a CU, else `each` for every workgroup of the
        // fullest CU (measured, us).  Cold operands, 64 x 256 tiles before -> the form
        // taken (us): 2048 x 11264 x 2048 163 -> 95-99 (128 x 192 tiles, 955-995 TFLOP/s),
        // 2040 x 2048 x 5632 -> 57 (128 x 128, two K groups), 2048 x 2048 x 2048 39 ->
        // 24 (128 x 64), 1000 x 2048 x 5632 93 -> 33 (128 x 64, two groups), 333 x 2048
        // x 5632 93 -> 22 (64 x 64, two groups).  Without the tile's own time short
        // contractions got too wide tiles, and 64 x 64 of one group suits the smallest
        // (us, 64 x 256 tiles / that rule / here): 915 x 7338 x 224 16.1 / 17.3 / 13.6,
        // 946 x 13341 x 512 42 / 37 / 28, 434 x 2385 x 96 - / 7.2 / 6.0.  Batches (64 x 256
        // tiles / products dealt to the XCDs one by one / here): 185 of 141 x 165 x 576
        // 35 / 47 / 19, 137 of 116 x 5 x 1088 22 / 52 / 12, 164 of 73 x 35 x 160 9.3 / 12 /
        // 5.9, 40 of 85 x 109 x 800 20 / 13 / 7.7.
        struct Form {
            int bm, bn, groups;
            double alone, each, alone_tile, each_tile;
        };
        static const Form kForms[] = {{128, 192, 1, 0.75, 0.78, 2.5, 1.5}, {128, 64, 1, 0.41, 0.36, 0.5, 0.3},
                                      {128, 128, 2, 1.2, 1.4, 2.0, 1.2},   {128, 64, 2, 0.72, 0.8, 0.9, 1.5},
                                      {64, 64, 2, 0.5, 0.5, 0.5, 0.5},     {64, 64, 1, 0.27, 0.25, 0.25, 0.05}};
        const int64_t chunks = (p.K + 63) / 64;
        int form = 0;
        double best = 0.0;
        for (int i = 0; i < 6; i++) {
            const Form& f = kForms[i];
            const double tiles = static_cast<double>((p.M + f.bm - 1) / f.bm) * static_cast<double>((p.N + f.bn - 1) / f.bn) *
                                 static_cast<double>(p.batches);
            const double steps = static_cast<double>((chunks + f.groups - 1) / f.groups);
            const double us = tiles <= 256.0 ? steps * f.alone + f.alone_tile
                                             : std::ceil(tiles / 256.0) * (steps * f.each + f.each_tile);
            if (i == 0 || us < best) {
                best = us;
                form = i;
            }
        }
        form = env_int("SANDY_GEMM_FORM", form);
        auto go = [&](auto geo, auto kernel) -> int {
            using G_ = decltype(geo);
            const int64_t rt = (p.M + G_::BM - 1) / G_::BM, ct = (p.N + G_::BN - 1) / G_::BN;
            if (rt > 0x7fffffff || ct > 0x7fffffff || rt * ct > 0x7ffffff0)
                return fail(e, SANDY_ERR_UNSUPPORTED, "%s shape exceeds the launch grid", what);
            g.row_tiles = static_cast<int32_t>(rt);
            g.col_tiles = static_cast<int32_t>(ct);
            const bool fold = rt * ct * p.batches <= 0x7ffffff0;
            g.splits = fold ? static_cast<int32_t>(p.batches) : 1;
            if (G_::kBytes > 64 * 1024)
                SANDY_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, G_::kBytes), e, what);
            hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>((rt * ct * g.splits + 7) / 8 * 8), 1,
                                            static_cast<unsigned>(fold ? 1 : p.batches)),
                               dim3(G_::THREADS), G_::kBytes, stream, g);
            return SANDY_OK;
        };
        int st = SANDY_OK;
        switch (form) {
            case 0: st = go(TileGeo<2, 3, 1>{}, gemm_tile_kernel<2, 3, 1>); break;
            case 1: st = go(TileGeo<2, 1, 1>{}, gemm_tile_kernel<2, 1, 1>); break;
            case 2: st = go(TileGeo<2, 2, 2>{}, gemm_tile_kernel<2, 2, 2>); break;
            case 3: st = go(TileGeo<2, 1, 2>{}, gemm_tile_kernel<2, 1, 2>); break;
            case 5: st = go(TileGeo<1, 1, 1>{}, gemm_tile_kernel<1, 1, 1>); break;
            default: st = go(TileGeo<1, 1, 2>{}, gemm_tile_kernel<1, 1, 2>); break;
        }
        if (st) return st;
    } else {
        const int64_t gy = (p.M + 63) / 64, gx = (p.N + 63) / 64;
        if (gy > 65535 || gx > 0x7fffffff) return fail(e, SANDY_ERR_UNSUPPORTED, "%s shape exceeds the launch grid", what);
        const dim3 grid(static_cast<unsigned>(gx), static_cast<unsigned>(gy), static_cast<unsigned>(p.batches));
        if (l.dtype == SANDY_BF16)
            hipLaunchKernelGGL(gemm_simt_kernel<BF16>, grid, dim3(256), 0, stream, pl, pr, pb, po, p.M, p.N, p.K,
                               static_cast<int32_t>(tl), static_cast<int32_t>(tr), p.lrs, p.rrs, p.bm);
        else
            hipLaunchKernelGGL(gemm_simt_kernel<F32>, grid, dim3(256), 0, stream, pl, pr, pb, po, p.M, p.N, p.K,
                               static_cast<int32_t>(tl), static_cast<int32_t>(tr), p.lrs, p.rrs, p.bm);
    }
    SANDY_HIP_TRY(hipGetLastError(), e, what);
    return ok(e);
}

} // namespace
} // namespace sandy_hip

using namespace sandy_hip;

extern "C" int sandy_hip_matmul(const SandyTensor* lhs, const SandyTensor* rhs, int32_t transpose_lhs,
                                int32_t transpose_rhs, const SandyTensor* out, void* stream_, char* err,
                                size_t err_cap) {
    Err e{err, err_cap};
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (!valid_rank(lhs) || !valid_rank(rhs) || !valid_rank(out))
        return fail(e, SANDY_ERR_INVALID, "matmul requires lhs, rhs and out");
    if (lhs->dtype != rhs->dtype || lhs->dtype != out->dtype)
        return fail(e, SANDY_ERR_INVALID, "matmul operands must have same dtype");
    if (!is_float(lhs->dtype)) return fail(e, SANDY_ERR_INVALID, "matmul unsupported dtype");
    if (!contiguous(*lhs) || !contiguous(*rhs) || !contiguous(*out))
        return fail(e, SANDY_ERR_UNSUPPORTED, "matmul requires contiguous tensor views");
    Plan p{};
    if (const char* msg = plan_matmul(*lhs, *rhs, *out, transpose_lhs != 0, transpose_rhs != 0, p))
        return fail(e, SANDY_ERR_INVALID, "%s", msg);
    return launch(p, *lhs, *rhs, nullptr, *out, transpose_lhs != 0, transpose_rhs != 0, stream, e, "matmul");
}

extern "C" int sandy_hip_matmul_glu(const SandyTensor* lhs, const SandyTensor* rhs, int32_t activation,
                                    const SandyTensor* out, void* stream_, char* err, size_t err_cap) {
    Err e{err, err_cap};
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (!valid_rank(lhs) || !valid_rank(rhs) || !valid_rank(out))
        return fail(e, SANDY_ERR_INVALID, "matmul requires lhs, rhs and out");
    if (activation != 1 && activation != 2) return fail(e, SANDY_ERR_INVALID, "gated matmul activation must be 1 (silu) or 2 (gelu)");
    if (lhs->dtype != rhs->dtype || lhs->dtype != out->dtype)
        return fail(e, SANDY_ERR_INVALID, "matmul operands must have same dtype");
    if (!contiguous(*lhs) || !contiguous(*rhs) || !contiguous(*out))
        return fail(e, SANDY_ERR_UNSUPPORTED, "matmul requires contiguous tensor views");
    if (rhs->rank != 2 || rhs->dims[0] % 2 != 0)
        return fail(e, SANDY_ERR_INVALID, "gated matmul weight must be [2 * ffn, k] with gate and up rows interleaved");
    // plan the product against the full [.., M, 2 ffn] output; the epilogue writes half of it
    SandyTensor full = *out;
    if (full.rank < 1 || full.dims[full.rank - 1] * 2 != rhs->dims[0])
        return fail(e, SANDY_ERR_INVALID, "matmul output shape mismatch");
    full.dims[full.rank - 1] = rhs->dims[0];
    Plan p{};
    if (const char* msg = plan_matmul(*lhs, *rhs, full, false, true, p)) return fail(e, SANDY_ERR_INVALID, "%s", msg);
    return launch(p, *lhs, *rhs, nullptr, *out, false, true, stream, e, "gated matmul", activation);
}

// Shared checks of the fused decode GEMMs: bf16, lhs [m, k], rhs [n, k]
// (transposed weight), row statistics of ceil(cols / 16) float64 partials.
static int check_fused(const SandyTensor* lhs, const SandyTensor* rhs, const SandyTensor* out, Err e, const char* what) {
    if (!valid_rank(lhs) || !valid_rank(rhs) || !valid_rank(out))
        return fail(e, SANDY_ERR_INVALID, "%s requires lhs, rhs and out", what);
    if (lhs->dtype != SANDY_BF16 || rhs->dtype != SANDY_BF16 || out->dtype != SANDY_BF16)
        return fail(e, SANDY_ERR_UNSUPPORTED, "%s takes bf16 operands", what);
    if (lhs->rank != 2 || rhs->rank != 2 || out->rank != 2)
        return fail(e, SANDY_ERR_INVALID, "%s expects lhs [m, k], rhs [n, k] and out [m, n]", what);
    if (!contiguous(*lhs) || !contiguous(*rhs) || !contiguous(*out))
        return fail(e, SANDY_ERR_UNSUPPORTED, "%s requires contiguous tensor views", what);
    return SANDY_OK;
}

static bool stats_ok(const SandyRowStats* st, int64_t rows, int64_t cols) {
    return st && st->sumsq && st->rows == rows && st->parts == (cols + 15) / 16 &&
           (reinterpret_cast<uintptr_t>(st->sumsq) & 7u) == 0;
}

extern "C" int sandy_hip_matmul_residual(const SandyTensor* lhs, const SandyTensor* rhs, const SandyTensor* residual,
                                         const SandyTensor* out, const SandyRowStats* out_stats, void* stream_,
                                         char* err, size_t err_cap) {
    Err e{err, err_cap};
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const char* what = "residual matmul";
    if (int st = check_fused(lhs, rhs, out, e, what)) return st;
    if (!valid_rank(residual) || residual->dtype != SANDY_BF16 || !same_shape(*residual, *out) || !contiguous(*residual))
        return fail(e, SANDY_ERR_INVALID, "%s residual must be a contiguous bf16 tensor shaped like out", what);
    if (base_ptr(*out) == base_ptr(*lhs)) return fail(e, SANDY_ERR_INVALID, "%s out must not alias lhs", what);
    Plan p{};
    if (const char* msg = plan_matmul(*lhs, *rhs, *out, false, true, p)) return fail(e, SANDY_ERR_INVALID, "%s", msg);
    if (out_stats && !stats_ok(out_stats, p.M, p.N))
        return fail(e, SANDY_ERR_INVALID, "%s row statistics must be [m, ceil(n / 16)] float64", what);
    Fusion fz;
    fz.resid = static_cast<const uint16_t*>(base_ptr(*residual));
    fz.rsq_out = out_stats ? out_stats->sumsq : nullptr;
    fz.rsq_parts = out_stats ? out_stats->parts : 0;
    return launch(p, *lhs, *rhs, nullptr, *out, false, true, stream, e, what, 0, &fz);
}

extern "C" int sandy_hip_matmul_rms(const SandyTensor* lhs, const SandyRowStats* lhs_stats,
                                    const SandyTensor* norm_weight, double eps, const SandyTensor* rhs,
                                    int32_t activation, const SandyTensor* out, void* stream_, char* err,
                                    size_t err_cap) {
    Err e{err, err_cap};
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const char* what = "rms matmul";
    if (int st = check_fused(lhs, rhs, out, e, what)) return st;
    if (activation < 0 || activation > 2) return fail(e, SANDY_ERR_INVALID, "gated matmul activation must be 1 (silu) or 2 (gelu)");
    const int64_t K = lhs->dims[1];
    if (!valid_rank(norm_weight) || norm_weight->dtype != SANDY_BF16 || numel(*norm_weight) != K ||
        !contiguous(*norm_weight) || (reinterpret_cast<uintptr_t>(base_ptr(*norm_weight)) & 15u) != 0)
        return fail(e, SANDY_ERR_INVALID, "%s norm weight must be a 16-byte aligned bf16 [k] vector", what);
    if (!stats_ok(lhs_stats, lhs->dims[0], K))
        return fail(e, SANDY_ERR_INVALID, "%s row statistics must be [m, ceil(k / 16)] float64", what);
    SandyTensor full = *out;
    if (activation) {
        if (rhs->dims[0] % 2 != 0 || out->dims[1] * 2 != rhs->dims[0])
            return fail(e, SANDY_ERR_INVALID, "gated matmul weight must be [2 * ffn, k] with gate and up rows interleaved");
        full.dims[1] = rhs->dims[0];
    }
    Plan p{};
    if (const char* msg = plan_matmul(*lhs, *rhs, full, false, true, p)) return fail(e, SANDY_ERR_INVALID, "%s", msg);
    Fusion fz;
    fz.rsq_in = lhs_stats->sumsq;
    fz.rsq_in_parts = lhs_stats->parts;
    fz.norm_w = static_cast<const uint16_t*>(base_ptr(*norm_weight));
    fz.eps = static_cast<float>(eps);
    return launch(p, *lhs, *rhs, nullptr, *out, false, true, stream, e, what, activation, &fz);
}

namespace sandy_hip {
int matmul_qkv(const SandyTensor* lhs, const SandyRowStats* lhs_stats, const SandyTensor* norm_weight, double eps,
               const SandyTensor* rhs, const QkvRope& qr, hipStream_t stream, Err e, bool dry) {
    const char* what = "qkv matmul";
    if (!valid_rank(lhs) || !valid_rank(rhs)) return fail(e, SANDY_ERR_INVALID, "%s requires lhs and rhs", what);
    if (lhs->dtype != SANDY_BF16 || rhs->dtype != SANDY_BF16) return fail(e, SANDY_ERR_UNSUPPORTED, "%s takes bf16 operands", what);
    if (lhs->rank != 2 || rhs->rank != 2 || !contiguous(*lhs) || !contiguous(*rhs))
        return fail(e, SANDY_ERR_INVALID, "%s expects contiguous lhs [m, k] and rhs [n, k]", what);
    const int64_t M = lhs->dims[0], K = lhs->dims[1];
    if (M > kQkvMaxRows) return fail(e, SANDY_ERR_UNSUPPORTED, "%s takes at most %d rows", what, kQkvMaxRows);
    if (rhs->dims[0] != static_cast<int64_t>(qr.hq + 2 * qr.hkv) * qr.d || rhs->dims[1] != K)
        return fail(e, SANDY_ERR_INVALID, "%s weight must be [(q_heads + 2 kv_heads) head_dim, k]", what);
    const bool norm = lhs_stats || norm_weight;
    if (norm) {
        if (!valid_rank(norm_weight) || norm_weight->dtype != SANDY_BF16 || numel(*norm_weight) != K ||
            !contiguous(*norm_weight) || (reinterpret_cast<uintptr_t>(base_ptr(*norm_weight)) & 15u) != 0)
            return fail(e, SANDY_ERR_INVALID, "%s norm weight must be a 16-byte aligned bf16 [k] vector", what);
        if (!stats_ok(lhs_stats, M, K))
            return fail(e, SANDY_ERR_INVALID, "%s row statistics must be [m, ceil(k / 16)] float64", what);
    }
    // the product is planned against an [m, n] output the epilogue never writes
    SandyTensor full{};
    full.dtype = SANDY_BF16;
    full.rank = 2;
    full.dims[0] = M;
    full.dims[1] = rhs->dims[0];
    full.strides[0] = rhs->dims[0];
    full.strides[1] = 1;
    Plan p{};
    if (const char* msg = plan_matmul(*lhs, *rhs, full, false, true, p)) return fail(e, SANDY_ERR_INVALID, "%s", msg);
    Fusion fz;
    if (norm) {
        fz.rsq_in = lhs_stats->sumsq;
        fz.rsq_in_parts = lhs_stats->parts;
        fz.norm_w = static_cast<const uint16_t*>(base_ptr(*norm_weight));
        fz.eps = static_cast<float>(eps);
    }
    fz.qr = &qr;
    fz.dry = dry;
    return launch(p, *lhs, *rhs, nullptr, full, false, true, stream, e, what, 0, &fz);
}
} // namespace sandy_hip

extern "C" int sandy_hip_linear(const SandyTensor* x, const SandyTensor* weight, const SandyTensor* bias,
                                const SandyTensor* out, void* stream_, char* err, size_t err_cap) {
    Err e{err, err_cap};
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (!valid_rank(x) || !valid_rank(weight) || !valid_rank(bias) || !valid_rank(out))
        return fail(e, SANDY_ERR_INVALID, "linear requires input, weight, bias and out");
    if (!is_float(x->dtype)) return fail(e, SANDY_ERR_INVALID, "linear input unsupported dtype");
    if (weight->dtype != x->dtype || bias->dtype != x->dtype || out->dtype != x->dtype)
        return fail(e, SANDY_ERR_INVALID, "linear operands must have same dtype");
    if (x->rank < 1 || weight->rank != 2 || bias->rank != 1)
        return fail(e, SANDY_ERR_INVALID, "linear expects input [..., in], weight [out, in], bias [out]");
    const int64_t in_f = x->dims[x->rank - 1], out_f = weight->dims[0];
    if (weight->dims[1] != in_f) return fail(e, SANDY_ERR_INVALID, "linear input/weight feature mismatch");
    if (bias->dims[0] != out_f) return fail(e, SANDY_ERR_INVALID, "linear bias shape mismatch");
    if (out->rank != x->rank || out->dims[x->rank - 1] != out_f)
        return fail(e, SANDY_ERR_INVALID, "linear output shape mismatch");
    for (int i = 0; i + 1 < x->rank; i++)
        if (out->dims[i] != x->dims[i]) return fail(e, SANDY_ERR_INVALID, "linear output shape mismatch");
    if (!contiguous(*x) || !contiguous(*weight) || !contiguous(*bias) || !contiguous(*out))
        return fail(e, SANDY_ERR_UNSUPPORTED, "linear requires contiguous tensor views");
    // rows of x flattened: [rows, in] times weight^T
    SandyTensor x2 = *x, o2 = *out;
    int64_t rows = 1;
    for (int i = 0; i + 1 < x->rank; i++) rows *= x->dims[i];
    x2.rank = 2;
    x2.dims[0] = rows;
    x2.dims[1] = in_f;
    x2.strides[0] = in_f;
    x2.strides[1] = 1;
    o2.rank = 2;
    o2.dims[0] = rows;
    o2.dims[1] = out_f;
    o2.strides[0] = out_f;
    o2.strides[1] = 1;
    Plan p{};
    if (const char* msg = plan_matmul(x2, *weight, o2, false, true, p)) return fail(e, SANDY_ERR_INVALID, "%s", msg);
    return launch(p, x2, *weight, bias, o2, false, true, stream, e, "linear");
}
