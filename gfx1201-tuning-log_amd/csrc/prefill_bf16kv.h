// The key-split prefill kernel (prefill_attn.hip) over bf16 caches, as the bf16 entry points
// (prefill_bf16kv.hip) launch it.  Strides of the caches are in bytes.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace fp8kv {

struct PrefillBf16 {
    const void* q;
    const void* k;
    const void* v;
    void* out;
    const int32_t* cu_q;        // null: one sequence, q0 / qlen from the host
    const int32_t* seq_lens;
    const int32_t* bt;
    int64_t q_stride, o_stride, bt_stride;
    int64_t sk0, sk1, sk2, sv0, sv1, sv2;
    float sm_scale;
    int hkv, gqa, pblk;
    int q0, qlen, num_seqs, max_query_len;
};

bool prefill_split_takes_bf16(int hkv, int gqa, int num_seqs, int max_query_len, int ctx_hint);
int launch_prefill_split_bf16(const PrefillBf16& A, bool force_paired, hipStream_t stream);

}  // namespace fp8kv
