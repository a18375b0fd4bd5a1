// A whole decode pass issued by one host call.
//
// A pass of one to a few rows is five or six launches of 5-8 us per layer;
// issued one wrapper call at a time from Python (argument checks, ctypes, an
// output allocation each, 8-10 us) the host took longer than the GPU. The loop
// over the layers is here instead (one token of the 24-layer 0.5B model, LM
// head included: 1212-1269 -> 714 us); the caller checks the layers' operands and
// gives the scratch rows that every layer reuses in stream order. The launches,
// their order and their arguments are those of the calls made one by one.

#include "kve_common.h"

using namespace kve;

extern "C" int kve_small_pass(const void* const* layer_ptrs, const float* layer_consts,
                              int num_layers, void* residual, const void* cos, const void* sin,
                              void* q, void* attn_out, void* act, const int32_t* block_tables,
                              const int32_t* seq_rows, const int32_t* start_pos,
                              const int32_t* q_lens, int num_seqs, int q_len, int hidden, int ffn,
                              int num_q_heads, int num_kv_heads, int head_dim, int block_size,
                              int max_blocks, int num_rows, int num_blocks, int max_ctx,
                              int unit_blocks, int key_waves, const void* plan, void* workspace,
                              size_t workspace_bytes, const void* norm_weight, float norm_eps,
                              void* out, int layout, void* stream) {
  clear_error();
  KVE_REQUIRE(num_layers >= 0 && (num_layers == 0 || (layer_ptrs && layer_consts)),
              "kve_small_pass: %d layers", num_layers);
  KVE_REQUIRE(num_seqs > 0 && q_len > 0 && num_q_heads > 0 && head_dim > 0 && hidden > 0 && ffn > 0,
              "kve_small_pass: bad sizes");
  const int rows = num_seqs * q_len, q_dim = num_q_heads * head_dim;
  for (int i = 0; i < num_layers; ++i) {
    const void* const* p = layer_ptrs + 9 * static_cast<size_t>(i);
    const float* c = layer_consts + 3 * static_cast<size_t>(i);
    // odd layers take the second half of each scratch buffer (one half for every
    // layer: 0.5B, 4 layers of one row in a graph 129.2 -> 131.5 us)
    uint16_t* ql = static_cast<uint16_t*>(q) + (i & 1) * static_cast<size_t>(rows) * q_dim;
    uint16_t* ol = static_cast<uint16_t*>(attn_out) + (i & 1) * static_cast<size_t>(rows) * q_dim;
    uint16_t* al = static_cast<uint16_t*>(act) + (i & 1) * static_cast<size_t>(rows) * ffn;
    int rc = kve_fused_qkv(residual, p[0], c[0], p[1], p[2], cos, sin, ql, const_cast<void*>(p[3]),
                           const_cast<void*>(p[4]), block_tables, seq_rows, start_pos, q_lens,
                           num_seqs, q_len, hidden, num_q_heads, num_kv_heads, head_dim, block_size,
                           max_blocks, num_rows, num_blocks, layout, stream);
    if (rc) return rc;
    rc = kve_paged_verify_attn(ql, p[3], p[4], block_tables, seq_rows, start_pos, q_lens, num_seqs,
                               q_len, num_q_heads, num_kv_heads, head_dim, block_size, max_blocks,
                               num_rows, num_blocks, max_ctx, unit_blocks, key_waves, c[2],
                               KVE_DTYPE_BF16, plan, ol, workspace, workspace_bytes,
                               KVE_LAYOUT_ROWS, stream);
    if (rc) return rc;
    rc = kve_linear_residual(ol, p[5], residual, rows, hidden, q_dim, layout, stream);
    if (rc) return rc;
    rc = kve_fused_gate_up(residual, p[6], c[1], p[7], al, rows, hidden, ffn, layout,
                           KVE_LAYOUT_ROWS, stream);
    if (rc) return rc;
    rc = kve_linear_residual(al, p[8], residual, rows, hidden, ffn, layout, stream);
    if (rc) return rc;
  }
  return kve_rmsnorm(residual, nullptr, nullptr, norm_weight, out, rows, hidden, norm_eps,
                     KVE_DTYPE_BF16, KVE_LAYOUT_ROWS, stream);
}
