// The decode / verify layer in fp32 (the parity configuration), up to 160 rows.
//
// The same cut as the bf16 wide layer of kve_linear.hip: every projection in
// k-slices over the whole chip, their reductions fused with what follows. Per
// layer: q/k/v slices, slice sum + bias + RoPE + K/V write, attention (+ its
// merge), o_proj slices, slice sum + residual + RMSNorm, gate/up with SiLU * up,
// down_proj slices, slice sum + residual + RMSNorm (the next layer's or the
// final one). The weights are 4 bytes each and read once, so the layer is bound
// by how fast the CUs pull them (0.5B: 60 MB per layer, 9.6 us at 6.2 TB/s)
// and by its launches. Library GEMMs with their separate RoPE, SiLU and RMSNorm
// launches, issued one by one from Python, took 180 us per layer at 20 rows.
//
// An fp32 matrix is read as one of uint16 pairs by DmaGemm (kve_gemm.h): its
// k-step of 64 bytes is 16 values, and a lane's 16-byte fragment of both
// operands is 4 consecutive k, fed to four 16x16x4 MFMAs. Every sum is fp32 in a
// fixed order that depends on the weight's shape only, so with a fixed attention
// order (unit_blocks, key_waves) a row's result does not depend on the batch.

#include "kve_common.h"
#include "kve_gemm.h"

#pragma clang fp contract(off)

namespace kve {

constexpr int kF32MaxRows = 160;
constexpr int kF32Slices = 8;

// Slices of an [N, K] weight: about 256 workgroups of 64 columns, at least 4
// k-steps of 16 per slice, at most 8 (the reductions load 8 per round trip).
static int f32_slices(int N, int K) {
  int S = (256 + N / 128) / (N / 64);
  S = S < K / 64 ? S : K / 64;
  S = S < kF32Slices ? S : kF32Slices;
  return S < 1 ? 1 : S;
}

template <int MT_, int NW_, int WN_, int KC_, int LDS_, int NR_>
struct F32Tile {
  using G = typename DmaCfg<MT_, NW_, WN_, KC_, LDS_, NR_>::G;
  static constexpr int NT = 64 * NW_;
};
// Column tiles of 32 (even row tiles, the waves 2 x 2) or 64; chunks of 4
// k-steps (256 bytes of a row) up to 4 row tiles, 2 above. 0.5B at 20 rows,
// chunks of 2 -> 4: gate/up 16.5 -> 15.2 us, the pass of 4 layers 256 -> 246;
// gate/up on 16 columns per workgroup 18.3.
template <int MT>
using F32Split = F32Tile<MT, 4, 1, (MT <= 4 ? 4 : 2), (MT <= 4 ? 80 : 56) * 1024, (MT % 2 == 0 ? 2 : 1)>;
template <int MT>
using F32Gate = F32Tile<MT, 4, 1, (MT <= 4 ? 4 : 2), (MT <= 4 ? 80 : 56) * 1024, 1>;

// part[s] = x[:, slice s] W[:, slice s]^T; grid (N / BN) * S, slice fastest.
template <int MT, typename C>
__global__ __launch_bounds__(C::NT) void f32_splitk_kernel(const uint16_t* x, const uint16_t* w,
                                                           float* part, int M, int N, int K, int S) {
  using G = typename C::G;
  constexpr int WN = G::BN / (16 * G::NC), MTW = G::MTW;
  extern __shared__ __align__(16) uint16_t sm_f32[];
  const int s = blockIdx.x % S, n0 = (blockIdx.x / S) * G::BN;
  const int nks = K / 16, a = nks * s / S, b = nks * (s + 1) / S;
  f32x4 acc[WN][MTW];
#pragma unroll
  for (int j = 0; j < WN; ++j)
#pragma unroll
    for (int mt = 0; mt < MTW; ++mt) acc[j][mt] = f32x4{0, 0, 0, 0};
  G::template run<false, true>(w, [n0](int r) { return n0 + r; }, x, 2 * K, M, 2 * K, a, b, sm_f32, acc);
  const int l = threadIdx.x & 63, lr = l & 15, lg = l >> 4, wv = threadIdx.x >> 6;
  const int wc = wv % G::NC, wr = wv / G::NC;
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) {
    const int m = 16 * (MTW * wr + mt) + lr;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < WN; ++j)
      *reinterpret_cast<f32x4*>(part + (static_cast<size_t>(s) * M + m) * N + n0 +
                                16 * (WN * wc + j) + 4 * lg) = acc[j][mt];
  }
}

// act = silu(gate) * up: workgroup = 32 activation columns (tile rows 0..31
// gate, 32..63 up) of 16 MT rows (blockIdx.y), joined through LDS.
template <int MT, typename C>
__global__ __launch_bounds__(C::NT) void f32_gate_up_kernel(const uint16_t* xn, const uint16_t* w,
                                                            float* act, int M, int H, int F) {
  using G = typename C::G;
  constexpr int WN = G::BN / (16 * G::NC), MTW = G::MTW, HALF = G::BN / 2;
  static_assert(HALF == 32, "32 activation columns");
  extern __shared__ __align__(16) uint16_t sm_f32[];
  const int tid = threadIdx.x, l = tid & 63, lr = l & 15, lg = l >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), wc = wv % G::NC, wr = wv / G::NC;
  const int f0 = blockIdx.x * HALF, m0 = blockIdx.y * G::XROWS, Mb = min(G::XROWS, M - m0);
  f32x4 acc[WN][MTW];
#pragma unroll
  for (int j = 0; j < WN; ++j)
#pragma unroll
    for (int mt = 0; mt < MTW; ++mt) acc[j][mt] = f32x4{0, 0, 0, 0};
  G::template run<false, true>(w, [f0, F](int r) { return r < HALF ? f0 + r : F + f0 + r - HALF; },
                               xn + static_cast<size_t>(m0) * 2 * H, 2 * H, Mb, 2 * H, 0, H / 16, sm_f32,
                               acc);
  float* sy = reinterpret_cast<float*>(sm_f32);  // [16 MT][64]: gate, then up
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
    for (int j = 0; j < WN; ++j)
      *reinterpret_cast<f32x4*>(sy + ((MTW * wr + mt) * 16 + lr) * 64 + 16 * (WN * wc + j) + 4 * lg) =
          acc[j][mt];
  __syncthreads();
  for (int idx = tid; idx < Mb * (HALF / 4); idx += C::NT) {
    const int m = idx / (HALF / 4), c = 4 * (idx % (HALF / 4));
    const f32x4 g = *reinterpret_cast<const f32x4*>(sy + m * 64 + c);
    const f32x4 u = *reinterpret_cast<const f32x4*>(sy + m * 64 + HALF + c);
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      o[e] = __fmul_rn(__fdiv_rn(g[e], __fadd_rn(1.0f, expf(-g[e]))), u[e]);
    *reinterpret_cast<f32x4*>(act + static_cast<size_t>(m0 + m) * F + f0 + c) = o;
  }
}

// The sum of S <= 8 slices of four columns, in slice order. Every slice slot is
// loaded (past S the last one again) and folded by a select, so the loads of
// all slices are in flight together.
__device__ __forceinline__ f32x4 sum_slices(const float* p, size_t plane, int S) {
  f32x4 t[kF32Slices];
#pragma unroll
  for (int i = 0; i < kF32Slices; ++i)
    t[i] = *reinterpret_cast<const f32x4*>(p + min(i, S - 1) * plane);
  f32x4 acc = t[0];
#pragma unroll
  for (int i = 1; i < kF32Slices; ++i) {
    const f32x4 n = acc + t[i];
    acc = i < S ? n : acc;
  }
  return acc;
}

// One workgroup per row: residual += sum of the slices, xn = RMSNorm(residual).
// Thread t owns the 4-column groups t, t + 256 (H <= 2048).
__global__ __launch_bounds__(256) void f32_residual_norm_kernel(const float* part, int S,
                                                                float* residual,
                                                                const float* norm_w, float eps,
                                                                float* xn, int M, int H) {
  constexpr int NG = 2;
  __shared__ float sm_ss[4];
  const int m = blockIdx.x, tid = threadIdx.x, ngr = H / 4;
  f32x4* rrow = reinterpret_cast<f32x4*>(residual + static_cast<size_t>(m) * H);
  const size_t plane = static_cast<size_t>(M) * H;
  f32x4 r[NG], wv[NG];
  float ss = 0.0f;
#pragma unroll
  for (int j = 0; j < NG; ++j) {
    const int g = min(tid + 256 * j, ngr - 1);
    r[j] = rrow[g];
    wv[j] = reinterpret_cast<const f32x4*>(norm_w)[g];
    r[j] += sum_slices(part + static_cast<size_t>(m) * H + 4 * g, plane, S);
    if (tid + 256 * j < ngr) {
#pragma unroll
      for (int e = 0; e < 4; ++e) ss += r[j][e] * r[j][e];
    }
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) sm_ss[tid >> 6] = ss;
  __syncthreads();
  ss = (sm_ss[0] + sm_ss[1]) + (sm_ss[2] + sm_ss[3]);
  const float inv = rsqrtf(__fadd_rn(__fmul_rn(ss, 1.0f / static_cast<float>(H)), eps));
#pragma unroll
  for (int j = 0; j < NG; ++j) {
    const int g = tid + 256 * j;
    if (g >= ngr) break;
    rrow[g] = r[j];
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = __fmul_rn(wv[j][e], __fmul_rn(r[j][e], inv));
    reinterpret_cast<f32x4*>(xn + static_cast<size_t>(m) * H)[g] = o;
  }
}

struct F32QkvArgs {
  const float *part, *bias, *cos, *sin;  // [S, M, N], [N], [M, D], [M, D]
  const int32_t* slots;                  // [M]
  float *q_out, *k_pool, *v_pool;
  int S, M, Hq, Hkv, bs;
};

// Per row: slice sums + bias, RoPE on the q and k heads, q / K / V written.
// Thread: 4 columns of a head's low half and their RoPE partners.
template <int D>
__global__ __launch_bounds__(256) void f32_qkv_rope_kernel(F32QkvArgs a) {
  constexpr int half = D / 2, GPH = half / 4;
  const int m = blockIdx.x, N = (a.Hq + 2 * a.Hkv) * D;
  const int idx = blockIdx.y * 256 + threadIdx.x;
  if (idx >= (a.Hq + 2 * a.Hkv) * GPH) return;
  const int h = idx / GPH, j = 4 * (idx - h * GPH);
  const int slot = a.slots[m];
  const int blk = slot >= 0 ? slot / a.bs : 0, off = slot >= 0 ? slot - blk * a.bs : 0;
  const size_t plane = static_cast<size_t>(a.M) * N;
  const float* p = a.part + static_cast<size_t>(m) * N + h * D + j;
  auto ld = [](const float* q) { return *reinterpret_cast<const f32x4*>(q); };
  const f32x4 bl = ld(a.bias + h * D + j), bh = ld(a.bias + h * D + j + half);
  const float *cr = a.cos + static_cast<size_t>(m) * D + j, *sr = a.sin + static_cast<size_t>(m) * D + j;
  const f32x4 cl = ld(cr), ch = ld(cr + half), sl = ld(sr), sh = ld(sr + half);
  const f32x4 x0 = sum_slices(p, plane, a.S) + bl, x1 = sum_slices(p + half, plane, a.S) + bh;
  if (h >= a.Hq + a.Hkv) {
    if (slot < 0) return;
    float* vb = a.v_pool + (static_cast<size_t>(blk) * a.Hkv + (h - a.Hq - a.Hkv)) * D * a.bs + off;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      vb[static_cast<size_t>(j + e) * a.bs] = x0[e];
      vb[static_cast<size_t>(j + e + half) * a.bs] = x1[e];
    }
    return;
  }
  if (h >= a.Hq && slot < 0) return;
  f32x4 lo, hi;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    lo[e] = __fadd_rn(__fmul_rn(x0[e], cl[e]), __fmul_rn(-x1[e], sl[e]));
    hi[e] = __fadd_rn(__fmul_rn(x1[e], ch[e]), __fmul_rn(x0[e], sh[e]));
  }
  float* dst = h < a.Hq ? a.q_out + (static_cast<size_t>(m) * a.Hq + h) * D
                        : a.k_pool + ((static_cast<size_t>(blk) * a.Hkv + (h - a.Hq)) * a.bs + off) * D;
  *reinterpret_cast<f32x4*>(dst + j) = lo;
  *reinterpret_cast<f32x4*>(dst + j + half) = hi;
}

template <typename K, typename... A>
static int launch_f32(K kernel, size_t& granted, dim3 grid, int threads, size_t lds, hipStream_t st,
                      A... args) {
  if (lds > 64 * 1024 && lds > granted) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize,
                            static_cast<int>(lds)) != hipSuccess) {
      set_error("kve_f32_pass: %zu bytes of LDS refused", lds);
      return KVE_ELAUNCH;
    }
    granted = lds;
  }
  hipLaunchKernelGGL(kernel, grid, dim3(threads), lds, st, args...);
  return KVE_OK;
}

// Row tiles of the k-sliced projections are instantiated for 1-4, 6, 8 and 10.
#define KVE_F32_ROWS(M_, CASE_)         \
  switch (cdiv(M_, 16)) {               \
    case 1: CASE_(1); break;            \
    case 2: CASE_(2); break;            \
    case 3: CASE_(3); break;            \
    case 4: CASE_(4); break;            \
    case 5:                             \
    case 6: CASE_(6); break;            \
    case 7:                             \
    case 8: CASE_(8); break;            \
    default: CASE_(10); break;          \
  }

static int f32_splitk(const void* x, const void* w, float* part, int M, int N, int K, hipStream_t st) {
  const int S = f32_slices(N, K);
  int rc = KVE_OK;
#define KVE_CASE(MT_)                                                                          \
  do {                                                                                         \
    using C = F32Split<MT_>;                                                                   \
    static size_t granted_ = 0;                                                                \
    rc = launch_f32(f32_splitk_kernel<MT_, C>, granted_, dim3(N / C::G::BN * S), C::NT,         \
                    C::G::LDS_BYTES, st, static_cast<const uint16_t*>(x),                      \
                    static_cast<const uint16_t*>(w), part, M, N, K, S);                        \
  } while (0)
  KVE_F32_ROWS(M, KVE_CASE)
#undef KVE_CASE
  return rc;
}

// Row tiles per gate/up workgroup. All of them on F / 32 workgroups left the
// chip half idle from about 90 rows on (0.5B: 152 workgroups), and the fp32 MFMAs
// bound those passes; groups of rows read the weights again, from L2. The cost
// of a workgroup is modelled as its row tiles and one more (weights, outputs),
// and the rows are divided only for a clear gain. Pass of 2 layers in a HIP graph,
// one group -> as picked (library GEMMs), us: 0.5B 20 x 5 rows 211 -> 193 (196),
// 32 x 5 241 -> 214 (245); 3B 20 x 5 610 -> 559 (606), 32 x 5 738 -> 670 (666), 1
// x 160 677 -> 615 (601); 0.5B 10 x 5 stays whole (two groups 2 % slower).
static int f32_gate_tiles(int M, int F) {
  const int tiles = cdiv(M, 16);
  int best = 0;
  float least = 0.0f;
  // at most 6: the four chains of more tiles leave room for one workgroup per CU
  for (int groups = cdiv(tiles, 6); groups <= tiles; ++groups) {
    const int mt = cdiv(tiles, groups);
    const float cost = tile_rounds(static_cast<int64_t>(F / 32) * cdiv(tiles, mt)) * (mt + 1);
    if (!best || cost < least) {
      best = mt;
      least = groups == 1 ? 0.93f * cost : cost;
    }
  }
  return best;
}

static int f32_gate_up(const void* xn, const void* w, float* act, int M, int H, int F, hipStream_t st) {
  int rc = KVE_OK;
#define KVE_CASE(MT_)                                                                          \
  do {                                                                                         \
    using C = F32Gate<MT_>;                                                                    \
    constexpr size_t stage = static_cast<size_t>(16) * MT_ * 64 * 4;                           \
    constexpr size_t lds = C::G::LDS_BYTES > stage ? C::G::LDS_BYTES : stage;                  \
    static size_t granted_ = 0;                                                                \
    rc = launch_f32(f32_gate_up_kernel<MT_, C>, granted_, dim3(F / 32, cdiv(M, 16 * MT_)), C::NT, lds, st, \
                    static_cast<const uint16_t*>(xn), static_cast<const uint16_t*>(w), act, M, \
                    H, F);                                                                     \
  } while (0)
  switch (f32_gate_tiles(M, F)) {
    case 1: KVE_CASE(1); break;
    case 2: KVE_CASE(2); break;
    case 3: KVE_CASE(3); break;
    case 4: KVE_CASE(4); break;
    case 5: KVE_CASE(5); break;
    default: KVE_CASE(6); break;
  }
#undef KVE_CASE
  return rc;
}

}  // namespace kve

using namespace kve;

extern "C" int kve_f32_pass(const void* const* layer_ptrs, const float* layer_consts, int num_layers,
                            void* residual, const void* cos, const void* sin, const int32_t* slots,
                            void* xn, void* q, void* attn_out, void* act, void* partials,
                            size_t partials_bytes, const int32_t* block_tables,
                            const int32_t* seq_rows, const int32_t* start_pos,
                            const int32_t* q_lens, int num_seqs, int q_len, int hidden, int ffn,
                            int num_q_heads, int num_kv_heads, int head_dim, int block_size,
                            int max_blocks, int num_rows, int num_blocks, int max_ctx,
                            int unit_blocks, int key_waves, const void* plan, void* workspace,
                            size_t workspace_bytes, const void* norm_weight, float norm_eps,
                            void* out, void* stream) {
  clear_error();
  if (num_layers == 0) return KVE_OK;
  KVE_REQUIRE(num_layers > 0 && layer_ptrs && layer_consts, "kve_f32_pass: %d layers", num_layers);
  KVE_REQUIRE(residual && cos && sin && slots && xn && q && attn_out && act && partials && norm_weight &&
                  out,
              "kve_f32_pass: null pointer argument");
  KVE_REQUIRE(num_seqs > 0 && q_len > 0 && num_seqs <= kF32MaxRows && q_len <= kF32MaxRows &&
                  num_seqs * q_len <= kF32MaxRows,
              "kve_f32_pass: %d x %d rows (at most %d)", num_seqs, q_len, kF32MaxRows);
  KVE_REQUIRE(head_dim == 64 || head_dim == 128, "kve_f32_pass: head_dim %d", head_dim);
  KVE_REQUIRE(num_q_heads > 0 && num_kv_heads > 0 && block_size > 0, "kve_f32_pass: bad sizes");
  KVE_REQUIRE(hidden > 0 && hidden % 64 == 0 && hidden <= 2048 && ffn > 0 && ffn % 64 == 0,
              "kve_f32_pass: hidden %d (multiple of 64, <= 2048), ffn %d (multiple of 64)", hidden, ffn);
  const int M = num_seqs * q_len, q_dim = num_q_heads * head_dim;
  const int N = (num_q_heads + 2 * num_kv_heads) * head_dim;
  const int S_qkv = f32_slices(N, hidden), S_o = f32_slices(hidden, q_dim), S_d = f32_slices(hidden, ffn);
  size_t need = static_cast<size_t>(S_qkv) * M * N;
  need = need > static_cast<size_t>(S_o) * M * hidden ? need : static_cast<size_t>(S_o) * M * hidden;
  need = need > static_cast<size_t>(S_d) * M * hidden ? need : static_cast<size_t>(S_d) * M * hidden;
  if (partials_bytes < need * 4) {
    set_error("kve_f32_pass: partials %zu bytes, need %zu", partials_bytes, need * 4);
    return KVE_EWORKSPACE;
  }
  uintptr_t al = 0;
  for (const void* p : {static_cast<const void*>(residual), cos, sin, static_cast<const void*>(xn),
                        static_cast<const void*>(q), static_cast<const void*>(attn_out),
                        static_cast<const void*>(act), static_cast<const void*>(partials), norm_weight,
                        static_cast<const void*>(out)})
    al |= reinterpret_cast<uintptr_t>(p);
  for (int i = 0; i < 9 * num_layers; ++i) {
    KVE_REQUIRE(layer_ptrs[i], "kve_f32_pass: null layer pointer %d", i);
    al |= reinterpret_cast<uintptr_t>(layer_ptrs[i]);
  }
  KVE_REQUIRE((al & 15) == 0, "kve_f32_pass: buffers must be 16-byte aligned");
  hipStream_t st = static_cast<hipStream_t>(stream);
  float* part = static_cast<float*>(partials);
  float* res = static_cast<float*>(residual);
  int rc = kve_rmsnorm(residual, nullptr, nullptr, layer_ptrs[0], xn, M, hidden, layer_consts[0],
                       KVE_DTYPE_F32, KVE_LAYOUT_ROWS, stream);
  for (int i = 0; i < num_layers && rc == KVE_OK; ++i) {
    const void* const* p = layer_ptrs + 9 * static_cast<size_t>(i);
    const float* c = layer_consts + 3 * static_cast<size_t>(i);
    const bool last = i + 1 == num_layers;
    rc = f32_splitk(xn, p[1], part, M, N, hidden, st);
    if (rc) return rc;
    F32QkvArgs a{part, static_cast<const float*>(p[2]), static_cast<const float*>(cos),
                 static_cast<const float*>(sin), slots, static_cast<float*>(q),
                 static_cast<float*>(const_cast<void*>(p[3])),
                 static_cast<float*>(const_cast<void*>(p[4])), S_qkv, M, num_q_heads, num_kv_heads,
                 block_size};
    const dim3 grid(M, cdiv(N / 8, 256));
    if (head_dim == 64) hipLaunchKernelGGL(f32_qkv_rope_kernel<64>, grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL(f32_qkv_rope_kernel<128>, grid, dim3(256), 0, st, a);
    rc = kve_paged_verify_attn(q, p[3], p[4], block_tables, seq_rows, start_pos, q_lens, num_seqs,
                               q_len, num_q_heads, num_kv_heads, head_dim, block_size, max_blocks,
                               num_rows, num_blocks, max_ctx, unit_blocks, key_waves, c[2],
                               KVE_DTYPE_F32, plan, attn_out, workspace, workspace_bytes,
                               KVE_LAYOUT_ROWS, stream);
    if (rc) return rc;
    rc = f32_splitk(attn_out, p[5], part, M, hidden, q_dim, st);
    if (rc) return rc;
    hipLaunchKernelGGL(f32_residual_norm_kernel, dim3(M), dim3(256), 0, st, part, S_o, res,
                       static_cast<const float*>(p[6]), c[1], static_cast<float*>(xn), M, hidden);
    rc = f32_gate_up(xn, p[7], static_cast<float*>(act), M, hidden, ffn, st);
    if (rc) return rc;
    rc = f32_splitk(act, p[8], part, M, hidden, ffn, st);
    if (rc) return rc;
    hipLaunchKernelGGL(f32_residual_norm_kernel, dim3(M), dim3(256), 0, st, part, S_d, res,
                       static_cast<const float*>(last ? norm_weight : p[9]),
                       last ? norm_eps : c[3], static_cast<float*>(last ? out : xn), M, hidden);
    rc = check_launch("kve_f32_pass");
  }
  return rc;
}

extern "C" size_t kve_f32_pass_bytes(int rows, int hidden, int ffn, int num_q_heads,
                                     int num_kv_heads, int head_dim) {
  if (rows <= 0 || hidden < 64 || ffn < 64 || num_q_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0)
    return 0;
  const int N = (num_q_heads + 2 * num_kv_heads) * head_dim;
  size_t cols = static_cast<size_t>(f32_slices(N, hidden)) * N;
  const size_t o = static_cast<size_t>(f32_slices(hidden, num_q_heads * head_dim)) * hidden;
  const size_t d = static_cast<size_t>(f32_slices(hidden, ffn)) * hidden;
  cols = cols > o ? cols : o;
  cols = cols > d ? cols : d;
  return cols * rows * sizeof(float);
}
