// attention_prefill.hip -- causal attention of prompts and prompt chunks
// (AttentionKernelOp with Tq > 1, src/core/TensorCalc.cpp:1167-1314), bf16
// and f32, over dense K/V or the reference's paged K/V.
//
// The general kernel (attention.hip) runs one workgroup per (query, head)
// and walks the keys in the reference's order; every query re-reads its K and
// V rows and all products are scalar: 14.4 ms for 2048 queries of 32 heads.
// Here the products run on v_mfma_f32_32x32x16_bf16 with an online softmax:
//   - the rows of one kv head are its (query, head of the group) pairs, query
//     major, so a workgroup's rows are a few neighbouring queries of the whole
//     GQA group: every staged key serves all heads of the group and the
//     causal frontier stays narrow;
//   - S^T = K Q^T (keys are MFMA rows, queries columns), so a lane holds the
//     scores of one query and the softmax needs one cross-lane exchange;
//   - P^T leaves the product in the B-operand layout of O^T += V^T P^T, with
//     V^T read by ds_read_b64_tr_b16 in the same key order;
//   - P enters as three bf16 operands that together are p exactly (two of them
//     kept about 17 bits and were 15% faster at 2048 queries); the row sums are
//     kept in float64.
// f32 takes v_mfma_f32_32x32x2_f32 for both products (f32 operands throughout,
// P straight from its registers) and expf; bound by that instruction's rate, a
// sixteenth of the bf16 one's.
// Four score waves a workgroup: RW of them own 32 rows each and KW = 4 / RW
// share the keys of a chunk (merged at the end), so short prompts still fill
// the chip; at D 256 a second wave per score tile owns half of the head dims.
// Chunks of K and V go global -> registers -> LDS, double buffered where they
// fit, one barrier each.
// Bound: softmax VALU work, the cutting of P included (52% of the cycles at D 64,
// MFMA 26%).  Measured, us a call (general kernel -> here): 2048 queries, 32 / 4
// heads, D 64 14357 -> 48; 777 queries after 1500 keys, window 1024, 8 / 2 heads,
// D 256, pages of 16: 4896 -> 42; 1500 after 300, 16 / 2 heads, D 128: 48; f32, 12
// heads, D 64: 1000 queries 1434 -> 43, 64 queries 23.5 -> 10.
// Against 64 bits (2 to 130 queries after 0 to 2000 keys, scores of three spreads)
// f32 outputs are off by 0.50 to 1.00 of the general kernel's error; of the bf16
// ones that are not the nearest value there are 0.5 to 0.95 as many wherever there
// are enough to count.
#include "attention_prefill.h"
#include "prefill_span.h"

#include <algorithm>
#include <type_traits>

namespace sandy_hip {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kMaxKeys = 1 << 30;
constexpr int kTablePages = 512;  // page addresses of K and V held in LDS

// Geometry of a variant.  LDS rows are padded so that MFMA-layout reads touch
// every bank once: 16 lanes x 16 bytes down a K column (pitch 16 bytes past a
// multiple of 128), 4 rows x 64 bytes of V per transposing read (pitch 64
// bytes past a multiple of 256 or 128), for f32 two V rows 4 apart x 128 bytes.
template <typename T, int D, int RW>
struct Geo {
    static constexpr bool kF32 = std::is_same_v<T, F32>;
    static constexpr int ES = kF32 ? 4 : 2;   // bytes of an element
    // D 256: two waves share a score tile and own half of the head dims each,
    // so that two waves fit a SIMD (one wave with all of O^T in its registers
    // had nothing to run behind its waits)
    static constexpr int DS = D == 256 ? 2 : 1;
    static constexpr int THREADS = 256 * DS;
    static constexpr int DT = D / 32 / DS;    // 32-dim tiles of O^T a wave owns
    static constexpr int KW = 4 / RW;
    static constexpr int CK = KW * 32;        // keys of a chunk, 32 a wave
    static constexpr int KP = ES * D + 16;               // bytes per K row in LDS
    static constexpr int VP = ES * D + (kF32 ? 32 : 64);  // bytes per V row in LDS
    static constexpr int kBuf = CK * (KP + VP);
    // LDS buffers: two where they fit, for f32 only beside a second workgroup
    // (its matrix work per chunk is long enough to cover the copy)
    static constexpr int NB = 2 * kBuf <= (kF32 ? 79 : 159) * 1024 ? 2 : 1;
    static constexpr int NP = CK * D * ES / 16 / THREADS;  // 16-byte pieces of K (and of V) a thread stages
    // final merge: [KW - 1][RW] copies of a wave's accumulators, and (m, l)
    static constexpr int kMerge = (KW - 1) * RW * D * 32 * 4;
    static constexpr int kStats = 4 * 32 * 16;  // of the waves of the first half
    static constexpr int kBytes = (NB * kBuf > kMerge + kStats ? NB * kBuf : kMerge + kStats);
};

// Byte address of row `key` of the page at `at` on page row `row`, rounded
// down to whole elements of `es` bytes.
__device__ __forceinline__ uint64_t paged_row(uint64_t at, int key, int log2_page, int64_t row, int row_bytes, int es) {
    const int64_t in_page = key & ((1 << log2_page) - 1);
    return (at & ~static_cast<uint64_t>(es - 1)) + static_cast<uint64_t>(((row << log2_page) + in_page) * row_bytes);
}

// 16 bytes from a row whose start is only element aligned.
__device__ __forceinline__ u32x4_t load_piece(uint64_t at) {
    if ((at & 15) == 0) return *reinterpret_cast<const u32x4_t*>(at);
    const uint16_t* p = reinterpret_cast<const uint16_t*>(at);
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = static_cast<uint32_t>(p[2 * i]) | (static_cast<uint32_t>(p[2 * i + 1]) << 16);
    return u32x4_t{w[0], w[1], w[2], w[3]};
}

// Up to R neighbouring rows again, by one wave, where outputs were not all finite:
// the general kernel's steps (scores summed over d in order, the max first, then expf
// and a float64 sum; the keys a row does not see and those of score -inf add nothing,
// whatever V holds), so that a non-finite K or V reaches exactly the rows that see its
// key.  Only the rows in `redo` (bit r)
// are stored; q of the rows as float in `qf` [R][D].
// A lane scores one key for all R rows (K is read once for them, twice in all: for
// the max, then for the sums), then each V row of the 64 keys is read once for the R
// rows, p coming from its lane as a scalar.  Bound: VALU and the K and V reads' latency.
// Every row redone (an infinity in V at key 0; us a call through Python: general kernel
// / rows one after another on the whole workgroup / here): 2048 queries, 32 / 4 heads,
// D 64 14363 / 26956 / 951; 777 after 1500, 8 / 2, D 256 7860 / 20702 / 947; 16 after
// 2000, 32 / 4, D 64 447 / 11542 / 451; f32, 12 heads, D 64, 64 queries 28 / 383 / 38,
// 1000 1427 / 5357 / 281.  More loads in flight (8 pieces of K, 32 V rows) gained
// nothing and spilled.
template <typename T, int D, bool PAGED, int R>
__device__ __forceinline__ void careful_rows(const PrefillArgs& a, int b, int kh, int row0, uint32_t redo, int64_t base,
                                             const float* qf) {
    constexpr int ES = std::is_same_v<T, F32> ? 4 : 2;
    constexpr int PE = 16 / ES, NK = 4;  // elements of a 16-byte piece, pieces of K in flight
    constexpr int DL = D / 64, NV = 8;   // dims a lane owns (lane + 64 i), V rows in flight
    const int lane = threadIdx.x & 63;
    const int rows = a.group * a.tq;
    auto last_of = [&](int r) -> int { return static_cast<int>(min<int64_t>(base + min(row0 + r, rows - 1) / a.group, a.tk - 1)); };
    auto first_of = [&](int r) -> int {
        return a.window > 0 ? static_cast<int>(min<int64_t>(max<int64_t>(0, base + min(row0 + r, rows - 1) / a.group + 1 - a.window), kMaxKeys)) : 0;
    };
    // a key's row: null where the page is missing (reported by the caller)
    auto row_of = [&](bool value, int key) -> const char* {
        if constexpr (PAGED) {
            const uint64_t at = (value ? a.v_pages : a.k_pages)[key >> a.log2_page];
            return at ? reinterpret_cast<const char*>(paged_row(at, key, a.log2_page, b * a.kv_rows_b + kh, ES * D, ES)) : nullptr;
        } else {
            const int64_t* st = value ? a.vs : a.ks;
            return static_cast<const char*>(value ? a.v : a.k) + (b * st[0] + kh * st[1] + key * st[2]) * ES;
        }
    };
    const int k_first = first_of(0), k_last = last_of(R - 1);
    // p enters scaled by a power of two of the key count, so that the unnormalised
    // sums stay below the largest |V|
    const float fac = ldexpf(1.0f, -(32 - __clz(max(k_last - k_first, 0))));
    float m[R], acc[R][DL];
    double l[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        m[r] = -INFINITY;
        l[r] = 0.0;
#pragma unroll
        for (int i = 0; i < DL; i++) acc[r][i] = 0.0f;
    }
#pragma unroll 1
    for (int pass = 0; pass < 2; pass++) {
#pragma unroll 1
        for (int k0 = k_first; k0 <= k_last; k0 += 64) {
            const int key = min(k0 + lane, k_last);
            const char* kp = row_of(false, key);
            float s[R];
#pragma unroll
            for (int r = 0; r < R; r++) s[r] = 0.0f;
#pragma unroll 1
            for (int d0 = 0; d0 < D; d0 += NK * PE) {
                u32x4_t kv[NK];
#pragma unroll
                for (int i = 0; i < NK; i++)
                    kv[i] = !PAGED || kp ? load_piece(reinterpret_cast<uint64_t>(kp) + (d0 + i * PE) * ES) : u32x4_t{0, 0, 0, 0};
#pragma unroll
                for (int i = 0; i < NK; i++) {
                    float kf[PE];
#pragma unroll
                    for (int j = 0; j < PE; j++)
                        kf[j] = ES == 4 ? __uint_as_float(kv[i][j & 3])
                                        : __uint_as_float(j & 1 ? kv[i][j >> 1] & 0xffff0000u : kv[i][j >> 1] << 16);
#pragma unroll
                    for (int r = 0; r < R; r++)
#pragma unroll
                        for (int j = 0; j < PE; j++)
                            s[r] = fmaf(qf[r * D + d0 + i * PE + j], kf[j], s[r]);
                }
            }
            uint64_t live[R], all = ~0ull, any = 0;
#pragma unroll
            for (int r = 0; r < R; r++) {
                s[r] = __fmul_rn(s[r], a.scale);
                const bool sees = k0 + lane <= last_of(r) && k0 + lane >= first_of(r) && s[r] != -INFINITY;
                live[r] = __ballot(sees);
                all &= live[r];
                any |= live[r];
                if (pass == 0) {
                    if (sees) m[r] = fmaxf(m[r], s[r]);
                } else {
                    s[r] = sees ? expf(__fsub_rn(s[r], m[r])) : 0.0f;
                    l[r] += static_cast<double>(s[r]);
                    s[r] *= fac;
                }
            }
            if (pass == 0) continue;
            auto weigh = [&](auto whole) {
#pragma unroll 1
                for (int j0 = 0; j0 < 64 && k0 + j0 <= k_last; j0 += NV) {
                    float v[NV][DL];
#pragma unroll
                    for (int j = 0; j < NV; j++) {
                        const char* vp = row_of(true, min(k0 + j0 + j, k_last));
#pragma unroll
                        for (int i = 0; i < DL; i++) v[j][i] = !PAGED || vp ? Vec8<T>::load1(vp, lane + 64 * i) : 0.0f;
                    }
#pragma unroll
                    for (int j = 0; j < NV; j++)
#pragma unroll
                        for (int r = 0; r < R; r++) {
                            const float p = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(s[r]), j0 + j));
                            // all bits where the row takes the key, else none: p is zero there
                            const int mask = decltype(whole)::value ? -1 : -static_cast<int>((live[r] >> (j0 + j)) & 1);
#pragma unroll
                            for (int i = 0; i < DL; i++)
                                acc[r][i] = fmaf(p, __int_as_float(__float_as_int(v[j][i]) & mask), acc[r][i]);
                        }
                }
            };
            if (all == ~0ull) weigh(std::true_type{});
            else if (any) weigh(std::false_type{});
        }
        if (pass == 0) {
#pragma unroll
            for (int r = 0; r < R; r++) m[r] = wave_max(m[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        const double total = wave_sum(l[r]);
        const float inv = (total != 0.0 ? 1.0f / static_cast<float>(total) : 0.0f) / fac;
        const int row = row0 + r;
        if (!((redo >> r) & 1)) continue;
        const int64_t to = b * a.os[0] + (kh * a.group + row % a.group) * a.os[1] + row / a.group * a.os[2] + lane;
#pragma unroll
        for (int i = 0; i < DL; i++) Vec8<T>::store1(a.out, to + 64 * i, m[r] == -INFINITY ? 0.0f : acc[r][i] * inv);
    }
}

template <typename T, int D, int RW, bool PAGED>
__global__ __launch_bounds__((Geo<T, D, RW>::THREADS), (Geo<T, D, RW>::kF32 && D == 128 ? 1 : 2)) void attention_prefill_kernel(PrefillArgs a) {
    using G_ = Geo<T, D, RW>;
    constexpr int KW = G_::KW, SUB = 32, CK = G_::CK, KP = G_::KP, VP = G_::VP, NP = G_::NP, DT = G_::DT;
    constexpr bool kF32 = G_::kF32;
    constexpr int ES = G_::ES;
    constexpr int kPieces = D * ES / 16;  // 16-byte pieces per row
    constexpr int kQ = D * ES / 32;       // 16-byte pieces of q a lane holds
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rw = wave % RW, kw = (wave & 3) / RW, ds = wave >> 2;
    const int col = lane & 31, half = lane >> 5;
    // heads vary fastest: workgroups go round-robin to the 8 XCDs, so one XCD
    // serves few kv heads; the longest row blocks (latest queries) start first
    const int heads = a.batch * a.hkv;
    const int bh = static_cast<int>(blockIdx.x) % heads;
    const int nth = static_cast<int>(blockIdx.x) / heads;
    const int b = bh / a.hkv, kh = bh % a.hkv;
    const int rows = a.group * a.tq;
    int64_t base = 0;
    if (a.pos) {
        base = load_index(a.pos, a.pos_dt, b);
        if (base < 0) {
            if (tid == 0) atomicOr(a.errw, static_cast<uint32_t>(SANDY_DEVERR_ATTN_POS));
            return;
        }
    }
    // keys [first, last] of query t
    auto last_of = [&](int t) -> int { return static_cast<int>(min<int64_t>(base + t, a.tk - 1)); };
    auto first_of = [&](int t) -> int {
        return a.window > 0 ? static_cast<int>(min<int64_t>(max<int64_t>(0, base + t + 1 - a.window), kMaxKeys)) : 0;
    };
    const int rb = a.row_blocks - 1 - nth;
    const int r0 = rb * 32 * RW;
    const int k_begin = first_of(r0 / a.group);
    const int k_end = last_of(min(rows - 1, r0 + 32 * RW - 1) / a.group) + 1;

    // this lane's row (clamped: rows past the end repeat the last and are not stored)
    const int row = r0 + 32 * rw + col;
    const int rc = min(row, rows - 1);
    const int qt = rc / a.group, qg = rc - qt * a.group;
    const int lane_last = last_of(qt), lane_first = first_of(qt);
    // the wave's rows: keys every row sees, and keys some row sees
    const int t_lo = min(rows - 1, r0 + 32 * rw) / a.group, t_hi = min(rows - 1, r0 + 32 * rw + 31) / a.group;
    const int any_first = first_of(t_lo), any_last = last_of(t_hi);
    const int all_first = first_of(t_hi), all_last = last_of(t_lo);

    // B operands: column = query; 16 bytes of q from 32 s + 16 half on (bf16: one
    // step of 16 dims; f32: four steps of 2, slot `half` of step i element i)
    u32x4_t qv[kQ];
    {
        const char* qp = static_cast<const char*>(a.q) + (b * a.qs[0] + (kh * a.group + qg) * a.qs[1] + qt * a.qs[2]) * ES + 16 * half;
#pragma unroll
        for (int s = 0; s < kQ; s++) qv[s] = *reinterpret_cast<const u32x4_t*>(qp + 32 * s);
    }

    // ---- staging: thread piece i covers chunk row prow + i * (256 / kPieces), 16-byte piece ppc
    constexpr int kRowStep = G_::THREADS / kPieces;
    const int prow = tid / kPieces, ppc = tid % kPieces;
    const char* kbase = static_cast<const char*>(a.k) + (PAGED ? 0 : (b * a.ks[0] + kh * a.ks[1]) * ES + 16 * ppc);
    const char* vbase = static_cast<const char*>(a.v) + (PAGED ? 0 : (b * a.vs[0] + kh * a.vs[1]) * ES + 16 * ppc);
    const uint32_t page_row = static_cast<uint32_t>(b * a.kv_rows_b + kh);
    u32x4_t kr[NP], vr[NP];
    bool pages_ok = true;
    // rows past the last key repeat it (they are masked)
    auto key_of = [&](int c0, int i) -> int { return min(c0 + prow + i * kRowStep, k_end - 1); };
    // the page addresses of the workgroup's keys, staged in LDS once where they
    // fit (read from memory per chunk they put a dependent load before each of
    // the chunk's: 777 queries, D 256, 74 us a call against 59) and checked
    // there instead of per piece (46 us against 41)
    u32x4_t* tab = reinterpret_cast<u32x4_t*>(lds + G_::kBytes);
    const int page0 = PAGED ? k_begin >> a.log2_page : 0;
    const int page_mask = (1 << a.log2_page) - 1;
    bool staged = false;
    if (PAGED && a.table_pages > 0) {
        const int pages = k_begin < k_end ? ((k_end - 1) >> a.log2_page) - page0 + 1 : 0;
        const int n = min(pages, a.table_pages);
        bool plain = pages <= a.table_pages;  // all staged, there and 16-byte aligned
        for (int i = tid; i < n; i += G_::THREADS) {
            const uint64_t kp = a.k_pages[page0 + i], vp = a.v_pages[page0 + i];
            plain = plain && kp != 0 && vp != 0 && ((kp | vp) & 15) == 0;
            tab[i] = u32x4_t{static_cast<uint32_t>(kp), static_cast<uint32_t>(kp >> 32), static_cast<uint32_t>(vp),
                             static_cast<uint32_t>(vp >> 32)};
        }
        staged = __syncthreads_and(plain);
    }
    auto load = [&](int c0) {
        if constexpr (PAGED) {
            if (staged) {
#pragma unroll
                for (int i = 0; i < NP; i++) {
                    const int key = key_of(c0, i);
                    const u32x4_t at = tab[(key >> a.log2_page) - page0];
                    // byte offset of the row within the page: below 2^31 (checked on the host)
                    const uint32_t off = ((page_row << a.log2_page) + (key & page_mask)) * (ES * D) + 16 * ppc;
                    kr[i] = *reinterpret_cast<const u32x4_t*>((static_cast<uint64_t>(at[1]) << 32 | at[0]) + off);
                    vr[i] = *reinterpret_cast<const u32x4_t*>((static_cast<uint64_t>(at[3]) << 32 | at[2]) + off);
                }
            } else {
#pragma unroll
                for (int i = 0; i < NP; i++) {
                    const int key = key_of(c0, i);
                    const uint64_t kp = a.k_pages[key >> a.log2_page], vp = a.v_pages[key >> a.log2_page];
                    pages_ok = pages_ok && kp != 0 && vp != 0;
                    kr[i] = vr[i] = u32x4_t{0, 0, 0, 0};
                    if (kp) kr[i] = load_piece(paged_row(kp, key, a.log2_page, page_row, ES * D, ES) + 16 * ppc);
                    if (vp) vr[i] = load_piece(paged_row(vp, key, a.log2_page, page_row, ES * D, ES) + 16 * ppc);
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < NP; i++) {
                kr[i] = *reinterpret_cast<const u32x4_t*>(kbase + key_of(c0, i) * a.ks[2] * ES);
                vr[i] = *reinterpret_cast<const u32x4_t*>(vbase + key_of(c0, i) * a.vs[2] * ES);
            }
        }
    };
    auto store = [&](int buf) {
        unsigned char* kt = lds + buf * G_::kBuf;
        unsigned char* vt = kt + CK * KP;
#pragma unroll
        for (int i = 0; i < NP; i++) {
            *reinterpret_cast<u32x4_t*>(kt + (prow + i * kRowStep) * KP + 16 * ppc) = kr[i];
            *reinterpret_cast<u32x4_t*>(vt + (prow + i * kRowStep) * VP + 16 * ppc) = vr[i];
        }
    };

    f32x16_t acc[DT];
    float m = -INFINITY;  // -inf until a key has been seen
    double l = 0.0;
    // P of a masked key is 0 and lo of an exact P is 0, so an infinity in V
    // would come out as NaN: outputs that are not all finite are computed again
    // below, one key at a time
#pragma unroll
    for (int t = 0; t < DT; t++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[t][i] = 0.0f;
    if (k_begin < k_end) load(k_begin);
    int buf = 0;
    for (int c0 = k_begin; c0 < k_end; c0 += CK, buf ^= G_::NB - 1) {
        if (G_::NB == 1 && c0 > k_begin) __syncthreads();  // the chunk before has been read
        store(buf);
        __syncthreads();
        if (c0 + CK < k_end) load(c0 + CK);
        const int k0 = c0 + kw * SUB;
        if (k0 > any_last || k0 + SUB - 1 < any_first) continue;  // wave-uniform
        const bool partial = k0 + SUB - 1 > all_last || k0 < all_first;
        const unsigned char* kt = lds + buf * G_::kBuf + kw * SUB * KP + col * KP + 16 * half;
        const unsigned char* vt = lds + buf * G_::kBuf + CK * KP + kw * SUB * VP;
        f32x16_t sc;
#pragma unroll
        for (int i = 0; i < 16; i++) sc[i] = 0.0f;
#pragma unroll
        for (int s = 0; s < kQ; s++) {
            const u32x4_t kv = *reinterpret_cast<const u32x4_t*>(kt + 32 * s);
            if constexpr (kF32) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    sc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(kv[i]), __uint_as_float(qv[s][i]), sc, 0, 0, 0);
            } else {
                sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, kv),
                                                             __builtin_bit_cast(bf16x8_t, qv[s]), sc, 0, 0, 0);
            }
        }
        // element i of sc: key k0 + 8 (i / 4) + 4 half + i % 4
        if (partial) {
            int key0 = k0 + 4 * half;
            asm volatile("" : "+v"(key0));  // keeps the compares out of whole tiles
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int key = key0 + 8 * (i >> 2) + (i & 3);
                if (key > lane_last || key < lane_first) sc[i] = -INFINITY;
            }
        }
        float mx = sc[0];
#pragma unroll
        for (int i = 1; i < 16; i++) mx = fmaxf(mx, sc[i]);
        // bf16: exponents in the exp2 domain; f32: expf of scaled scores, as the
        // general kernel takes them
        mx = max_xor32(mx) * (kF32 ? a.scale : a.scale_log2);
        // the reference point m of a row's exponents moves only when its max has
        // grown by 2^8 (p stays below that, its relative precision is the same),
        // so most chunks leave the accumulators alone
        if (__any(mx > m + (kF32 ? 5.5f : 8.0f))) {
            const float m_new = fmaxf(m, mx);
            const float alpha = m == -INFINITY ? 0.0f : kF32 ? expf(m - m_new) : __builtin_amdgcn_exp2f(m - m_new);
            l *= static_cast<double>(alpha);
            if (__any(m != -INFINITY)) {
#pragma unroll
                for (int t = 0; t < DT; t++) acc[t] *= alpha;
            }
            m = m_new;
        }
        const float shift = m == -INFINITY ? 0.0f : m;
        if constexpr (kF32) {
#pragma unroll
            for (int i = 0; i < 16; i++) {
                sc[i] = expf(sc[i] * a.scale - shift);
                l += static_cast<double>(sc[i]);
            }
            // step i: slot `half` is key 8 (i / 4) + 4 half + i % 4, this lane's element i
            const unsigned char* src = vt + 4 * half * VP + 4 * col;
#pragma unroll
            for (int i = 0; i < 16; i++)
#pragma unroll
                for (int t = 0; t < DT; t++)
                    acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                        *reinterpret_cast<const float*>(src + (8 * (i >> 2) + (i & 3)) * VP + 128 * (DT * ds + t)), sc[i], acc[t], 0, 0, 0);
            continue;
        }
#pragma unroll
        for (int i = 0; i < 16; i++) sc[i] = __builtin_amdgcn_exp2f(fmaf(sc[i], a.scale_log2, -shift));
        {  // pairs first: four roundings deep
            float rs[8];
#pragma unroll
            for (int i = 0; i < 8; i++) rs[i] = sc[2 * i] + sc[2 * i + 1];
            l += static_cast<double>(((rs[0] + rs[1]) + (rs[2] + rs[3])) + ((rs[4] + rs[5]) + (rs[6] + rs[7])));
        }
        // contraction slot 8 half + j of step s2: key 16 s2 + 4 half + j (j < 4) or + 8 + j - 4
#pragma unroll
        for (int s2 = 0; s2 < 2; s2++) {
            // p = three bf16 of 8 bits each (cut, not rounded: their sum is p exactly)
            u32x4_t p0, p1, p2;
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
                const float x = sc[8 * s2 + j], y = sc[8 * s2 + j + 1];
                const uint32_t xb = __float_as_uint(x), yb = __float_as_uint(y);
                const float x1 = x - __uint_as_float(xb & 0xffff0000u), y1 = y - __uint_as_float(yb & 0xffff0000u);
                const uint32_t x1b = __float_as_uint(x1), y1b = __float_as_uint(y1);
                const float x2 = x1 - __uint_as_float(x1b & 0xffff0000u), y2 = y1 - __uint_as_float(y1b & 0xffff0000u);
                p0[j / 2] = __builtin_amdgcn_perm(yb, xb, 0x07060302u);  // the upper halves of both
                p1[j / 2] = __builtin_amdgcn_perm(y1b, x1b, 0x07060302u);
                p2[j / 2] = __builtin_amdgcn_perm(__float_as_uint(y2), __float_as_uint(x2), 0x07060302u);
            }
            // ds_read_b64_tr_b16: in each 16-lane group, lane i gets element i % 4 of
            // the 8-byte pieces addressed by lanes 4 n + i / 4 (n = 0..3): pointing
            // lane i at key kb + i / 4, dims d0 + 4 (i % 4) .. + 3 yields V[kb + n][d0 + i]
            const int i16 = lane & 15;
            const unsigned char* src = vt + (16 * s2 + 4 * half + (i16 >> 2)) * VP + 2 * (16 * ((lane >> 4) & 1) + 4 * (i16 & 3));
#pragma unroll
            for (int t = 0; t < DT; t++) {
                const unsigned char* s0 = src + 64 * (DT * ds + t);
                const short4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (short4_t __attribute__((address_space(3)))*)((unsigned char __attribute__((address_space(3)))*)s0));
                const short4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (short4_t __attribute__((address_space(3)))*)((unsigned char __attribute__((address_space(3)))*)(s0 + 8 * VP)));
                const bf16x8_t va = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, __builtin_bit_cast(bf16x8_t, p0), acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, __builtin_bit_cast(bf16x8_t, p1), acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, __builtin_bit_cast(bf16x8_t, p2), acc[t], 0, 0, 0);
            }
        }
    }
    // the two halves of a row's sums; then the key shares of the KW waves
    l += __shfl_xor(l, 32, 64);
    __syncthreads();
    if constexpr (KW > 1) {
        float* red = reinterpret_cast<float*>(lds);
        double* ml = reinterpret_cast<double*>(lds + G_::kMerge);  // [wave][32][2]
        if (half == 0 && ds == 0) {
            ml[((wave & 3) * 32 + col) * 2] = static_cast<double>(m);
            ml[((wave & 3) * 32 + col) * 2 + 1] = l;
        }
        __syncthreads();
        float mm = -INFINITY;
#pragma unroll
        for (int w = 0; w < KW; w++) mm = fmaxf(mm, static_cast<float>(ml[((w * RW + rw) * 32 + col) * 2]));
        const float shift = mm == -INFINITY ? 0.0f : mm;
        double ll = 0.0;
#pragma unroll
        for (int w = 0; w < KW; w++) {
            const double* e = ml + ((w * RW + rw) * 32 + col) * 2;
            const float d = static_cast<float>(e[0]) - shift;
            ll += e[1] * static_cast<double>(kF32 ? expf(d) : __builtin_amdgcn_exp2f(d));
        }
        const float f = kF32 ? expf(m - shift) : __builtin_amdgcn_exp2f(m - shift);
#pragma unroll
        for (int t = 0; t < DT; t++) acc[t] *= f;
        m = mm;
        l = ll;
        if (kw > 0) {
#pragma unroll
            for (int t = 0; t < DT; t++)
#pragma unroll
                for (int i = 0; i < 16; i++) red[(((kw - 1) * RW + rw) * (D / 2) + 16 * (DT * ds + t) + i) * 64 + lane] = acc[t][i];
        }
        __syncthreads();
        if (kw == 0) {
#pragma unroll
            for (int w = 0; w < KW - 1; w++)
#pragma unroll
                for (int t = 0; t < DT; t++)
#pragma unroll
                    for (int i = 0; i < 16; i++) acc[t][i] += red[((w * RW + rw) * (D / 2) + 16 * (DT * ds + t) + i) * 64 + lane];
        }
    }
    if (PAGED && !pages_ok) atomicOr(a.errw, static_cast<uint32_t>(SANDY_DEVERR_BLOCK));
    // f32: the reciprocal as two floats, so that the output is rounded about once
    const double inv64 = 1.0 / l;
    const float inv = kF32 ? static_cast<float>(inv64) : 1.0f / static_cast<float>(l);
    const float inv_lo = kF32 ? static_cast<float>(inv64 - static_cast<double>(inv)) : 0.0f;
    // a row that sees no key (or only NaN scores) is zero, as in the general kernel
    const bool none = m == -INFINITY;
    bool finite = true;
#pragma unroll
    for (int t = 0; kw == 0 && t < DT; t++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            acc[t][i] = none ? 0.0f : kF32 ? fmaf(acc[t][i], inv, acc[t][i] * inv_lo) : acc[t][i] * inv;
            finite = finite && fabsf(acc[t][i]) < INFINITY;
        }
    auto put = [&] {
        char* op = static_cast<char*>(a.out) + (b * a.os[0] + (kh * a.group + qg) * a.os[1] + qt * a.os[2] + 32 * DT * ds + 4 * half) * ES;
#pragma unroll
        for (int t = 0; t < DT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float o[4];
#pragma unroll
                for (int x = 0; x < 4; x++) o[x] = acc[t][4 * i + x];
                char* to = op + (32 * t + 8 * i) * ES;
                if constexpr (kF32) *reinterpret_cast<float4*>(to) = make_float4(o[0], o[1], o[2], o[3]);
                else *reinterpret_cast<uint2*>(to) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
            }
    };
    // rows computed again read their q: where `out` may be `q`, nothing is stored before
    // it is known which those are (elsewhere the stores need not wait for the others)
    if (!a.in_place && kw == 0 && row < rows) put();
    const bool redo = __syncthreads_or(kw == 0 && row < rows && !finite);
    int* bad = reinterpret_cast<int*>(lds);           // [32 * RW] rows to compute again
    float* qf = reinterpret_cast<float*>(lds + 512);  // [32 * RW][D] their q
    if (redo) {
        for (int i = tid; i < 32 * RW; i += G_::THREADS) bad[i] = 0;
        for (int i = tid; i < 32 * RW * D; i += G_::THREADS) {
            const int r = min(r0 + i / D, rows - 1);
            qf[i] = Vec8<T>::load1(a.q, b * a.qs[0] + (kh * a.group + r % a.group) * a.qs[1] + r / a.group * a.qs[2] + i % D);
        }
        __syncthreads();
        if (kw == 0 && row < rows && !finite) bad[32 * rw + col] = 1;
        __syncthreads();
    }
    if (a.in_place && kw == 0 && row < rows && !(redo && bad[32 * rw + col])) put();
    if (!redo) return;
    constexpr int kMine = 32 * RW / (G_::THREADS / 64);  // rows of a wave
    constexpr int R = D == 64 ? 8 : 4;
    static_assert(32 * RW * 4 <= 512 && 512 + 32 * RW * D * 4 <= G_::kBytes && kMine % R == 0, "rows computed again");
#pragma unroll 1
    for (int i = wave * kMine; i < (wave + 1) * kMine && r0 + i < rows; i += R) {
        const uint32_t which = static_cast<uint32_t>(__ballot(lane < R && bad[i + (lane & (R - 1))]));
        if (which) careful_rows<T, D, PAGED, R>(a, b, kh, r0 + i, which, base, qf + i * D);
    }
}

// First and last byte that [batch, hq, tq, dim] elements of `es` bytes at these strides touch.
struct Span {
    uintptr_t first, last;
    Span(const void* p, const int64_t* s, const PrefillArgs& a, int64_t es) {
        const int64_t n[3] = {a.batch - 1, a.hq - 1, a.tq - 1};
        first = last = reinterpret_cast<uintptr_t>(p);
        last += static_cast<uintptr_t>(a.dim * es - 1);
        for (int i = 0; i < 3; i++) (s[i] < 0 ? first : last) += static_cast<uintptr_t>(n[i] * s[i] * es);
    }
};

template <typename T, int D, int RW, bool PAGED>
int launch_form(const PrefillArgs& a, hipStream_t stream, Err e) {
    static_assert(Geo<T, D, RW>::kBytes + kTablePages * 16 <= 160 * 1024 - 256, "LDS of a workgroup");
    PrefillArgs args = a;
    const Span q(a.q, a.qs, a, Geo<T, D, RW>::ES), out(a.out, a.os, a, Geo<T, D, RW>::ES);
    args.in_place = q.first <= out.last && out.first <= q.last;
    size_t bytes = Geo<T, D, RW>::kBytes;
    if (PAGED) {
        const int64_t span = prefill_page_span(a.tk, a.window, RW, a.group, a.log2_page);
        args.table_pages = span <= kTablePages ? static_cast<int32_t>(span) : 0;
        bytes += static_cast<size_t>(args.table_pages) * 16;
    }
    const void* fn = reinterpret_cast<const void*>(&attention_prefill_kernel<T, D, RW, PAGED>);
    if (bytes > 64 * 1024)
        SANDY_HIP_TRY(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)), e,
                      "attention launch");
    const int64_t rows = static_cast<int64_t>(a.group) * a.tq;
    args.row_blocks = static_cast<int32_t>((rows + 32 * RW - 1) / (32 * RW));
    const int64_t wgs = static_cast<int64_t>(args.row_blocks) * a.batch * a.hkv;
    void* params[] = {&args};
    SANDY_HIP_TRY(hipLaunchKernel(fn, dim3(static_cast<unsigned>(wgs)), dim3(Geo<T, D, RW>::THREADS), params, bytes, stream),
                  e, "attention launch");
    return ok(e);
}

template <typename T, int D, bool PAGED>
int launch_dim(const PrefillArgs& a, hipStream_t stream, Err e) {
    const int64_t rows = static_cast<int64_t>(a.group) * a.tq;
    const int64_t heads = static_cast<int64_t>(a.batch) * a.hkv;
    // 64-row workgroups (two waves share the keys) where they nearly fill the 256
    // CUs, else 32-row ones (four share them).  us, 64 / 32 rows, by the number of
    // 64-row workgroups: D 64 100 of them 10.8 / 11.1, 220 12.3 / 13.8, 300 15.4 /
    // 20.5, 1024 50 / 100; D 128 100 15.7 / 13.7, 200 23.8 / 23.2, 226 25.6 / 26.3,
    // 300 33 / 42; D 256 114 41 / 35, 200 64 / 56, 224 72 / 62 and with a window of
    // 1024 54 / 80.  128-row workgroups were slower at every size (two operands of
    // P, 2048 queries, D 64: 45 against 43).
    // f32: 192 workgroups of 64 rows 58 us, 384 of 32 rows 43.
    const int64_t wgs = (rows + 63) / 64 * heads;
    if (env_int("SANDY_PREFILL_RW", wgs >= 224 ? 2 : 1) == 2) return launch_form<T, D, 2, PAGED>(a, stream, e);
    return launch_form<T, D, 1, PAGED>(a, stream, e);
}

} // namespace

bool prefill_takes(const PrefillArgs& a) {
    const bool f32 = a.dtype == SANDY_F32;
    const int64_t D = a.dim, es = f32 ? 4 : 2;
    if ((D != 64 && D != 128 && (D != 256 || f32)) || a.tq < 2 || a.tk <= 0) return false;
    // 16-byte q and dense K/V rows; output pieces of 4 elements
    auto aligned = [es](const void* p, const int64_t* s, int64_t bytes) {
        return (reinterpret_cast<uintptr_t>(p) & static_cast<uintptr_t>(bytes - 1)) == 0 &&
               ((s[0] | s[1] | s[2]) & (bytes / es - 1)) == 0;
    };
    if (!aligned(a.q, a.qs, 16) || !aligned(a.out, a.os, 4 * es)) return false;
    if (!a.k_pages && (!aligned(a.k, a.ks, 16) || !aligned(a.v, a.vs, 16))) return false;
    const int64_t rows = static_cast<int64_t>(a.group) * a.tq;
    if (a.k_pages && ((a.batch * a.kv_rows_b + a.hkv) << a.log2_page) * D * es >= (int64_t{1} << 31)) return false;
    return rows < kMaxKeys && (rows + 31) / 32 * a.batch * a.hkv < (int64_t{1} << 31) &&
           env_int("SANDY_PREFILL_GENERAL", 0) == 0;
}

int launch_prefill(const PrefillArgs& a, hipStream_t stream, Err e) {
    const bool paged = a.k_pages != nullptr;
    if (a.dtype == SANDY_F32) {
        if (a.dim == 64) return paged ? launch_dim<F32, 64, true>(a, stream, e) : launch_dim<F32, 64, false>(a, stream, e);
        return paged ? launch_dim<F32, 128, true>(a, stream, e) : launch_dim<F32, 128, false>(a, stream, e);
    }
    switch (a.dim) {
        case 64: return paged ? launch_dim<BF16, 64, true>(a, stream, e) : launch_dim<BF16, 64, false>(a, stream, e);
        case 128: return paged ? launch_dim<BF16, 128, true>(a, stream, e) : launch_dim<BF16, 128, false>(a, stream, e);
        default: return paged ? launch_dim<BF16, 256, true>(a, stream, e) : launch_dim<BF16, 256, false>(a, stream, e);
    }
}

} // namespace sandy_hip
