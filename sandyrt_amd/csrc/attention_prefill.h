// attention_prefill.h -- attention of several queries a sequence (prompts and
// prompt chunks) on MFMA, called by attention.hip's dispatch.
#pragma once
#include "common.h"

namespace sandy_hip {

struct PrefillArgs {
    const void* q;
    int64_t qs[3];  // element strides over (b, h, t); the head dim is contiguous
    void* out;
    int64_t os[3];
    // dense K/V (element strides over (b, kh, key)), or page address tables:
    // page p of K at k_pages[p], (b, kh) on page row b * kv_rows_b + kh of
    // page_size keys
    const void* k;
    const void* v;
    int64_t ks[3], vs[3];
    const uint64_t* k_pages;
    const uint64_t* v_pages;
    int64_t kv_rows_b;
    int32_t log2_page;
    const void* pos;  // [B] position of the first query, or null (0)
    int32_t pos_dt;
    int32_t batch, hq, hkv, group;
    int32_t tq, tk;
    int32_t row_blocks;  // row tiles per (b, kh)
    int32_t table_pages; // page addresses staged in LDS (0: read from memory)
    int32_t in_place;    // out may share memory with q
    int64_t window;
    float scale, scale_log2;  // scale * log2(e)
    int32_t dtype;            // F32 or BF16
    int64_t dim;              // head dim
    uint32_t* errw;
};

// Whether the kernel takes the shape (the caller's general kernel takes the
// rest), and its launch.
bool prefill_takes(const PrefillArgs& a);
int launch_prefill(const PrefillArgs& a, hipStream_t stream, Err e);

} // namespace sandy_hip
