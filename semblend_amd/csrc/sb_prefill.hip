// Stages of the single-layer partial prefill (semblend_core/triton_kernels.py:769-923) around
// its projection and attention:
//   index     per target position: the donor row it takes, or "computed", or nothing;
//   assemble  the whole target cache [L, 2, H, S, D] in one pass, every row written once;
//   output    the output projection of the computed rows in fp32, rounded to the tensors' type,
//             the other rows zero.
// The composed form wrote the cache up to three times (zero fill, donor scatter, a select over
// every layer) and read it back twice. 1024 positions, 24 layers, 14 heads x 64, bf16, 30%
// computed: 168 us of launches for the cache before, one launch of 24 us here; the output projection
// with its conversions, select and zero fill 33 us before, 17 us here; the whole call 498 -> 146 us.

#include <algorithm>
#include <type_traits>

#include "sb_common.h"

namespace sb {
namespace {

typedef float pf32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t pu32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t pu32x2_t __attribute__((ext_vector_type(2)));
#define SB_PGLOBAL __attribute__((address_space(1)))

// index[t] of a target position: a donor row (>= 0), kRowNone (zero) or kRowComputed.
constexpr int kRowNone = -1;
constexpr int kRowComputed = -2;
constexpr int kPrefillIndexThreads = 1024;

// Workgroup 0 compacts the mask; workgroup b > 0 resolves target positions [1024 (b - 1), 1024 b)
// in an LDS table: the last valid pair that names a position wins. Each of them scans the whole
// pair list (a few loads per thread), which spares a second launch and global atomics.
__global__ __launch_bounds__(kPrefillIndexThreads) void prefill_index_kernel(
    const uint8_t* mask, const int32_t* donor_pos, const int32_t* target_pos, int64_t num_pairs,
    int64_t seq_len, int64_t donor_seq_len, int32_t* index, int32_t* positions) {
  if (blockIdx.x == 0) {
    mask_compact_unit(mask, seq_len, positions, positions + seq_len);
    return;
  }
  __shared__ int win[kPrefillIndexThreads];
  const int tid = threadIdx.x;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x - 1) * kPrefillIndexThreads;
  win[tid] = -1;
  __syncthreads();
  for (int64_t i = tid; i < num_pairs; i += kPrefillIndexThreads) {
    const int64_t t = target_pos[i] - t0;
    const int d = donor_pos[i];
    if (t >= 0 && t < kPrefillIndexThreads && t0 + t < seq_len && d >= 0 && d < donor_seq_len)
      atomicMax(&win[t], static_cast<int>(i));
  }
  __syncthreads();
  const int64_t t = t0 + tid;
  if (t >= seq_len) return;
  const int w = win[tid];
  index[t] = mask[t] ? kRowComputed : (w >= 0 ? donor_pos[w] : kRowNone);
}

struct AssembleArgs {
  char* out;              // [L, 2, H, S, row] contiguous
  const char* donor;
  int64_t d_s_layer, d_s_kv, d_s_head, d_s_seq;  // byte strides
  const char* qkv;        // [S, 3, H, row] rows
  int64_t q_s_row;        // bytes
  const int32_t* index;
  int64_t seq_len;
  int num_heads;
  int row_bytes;
  int vpr_log2;           // log2(16-byte vectors per row)
};

// One thread per 16-byte vector of a target position; grid.y walks (layer, K/V) planes, grid.z
// groups of kAssembleHeads heads. Bound: HBM writes of the cache and reads of its donor rows;
// consecutive threads write consecutive bytes of a plane.
constexpr int kAssembleHeads = 4;
__global__ __launch_bounds__(256) void prefill_assemble_kernel(const AssembleArgs a) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t t = idx >> a.vpr_log2;
  if (t >= a.seq_len) return;
  const int64_t vofs = (idx & ((1 << a.vpr_log2) - 1)) * 16;
  const int plane = blockIdx.y, kv = plane & 1;
  const int h0 = blockIdx.z * kAssembleHeads;
  const int nh = min(kAssembleHeads, a.num_heads - h0);
  const int from = a.index[t];
  pu32x4_t w[kAssembleHeads];
#pragma unroll
  for (int b = 0; b < kAssembleHeads; ++b) w[b] = pu32x4_t{0u, 0u, 0u, 0u};
  if (from != kRowNone) {
    const char* src;
    int64_t s_head;
    if (from == kRowComputed) {
      src = a.qkv + t * a.q_s_row + static_cast<int64_t>(1 + kv) * a.num_heads * a.row_bytes;
      s_head = a.row_bytes;
    } else {
      src = a.donor + (plane >> 1) * a.d_s_layer + kv * a.d_s_kv + from * a.d_s_seq;
      s_head = a.d_s_head;
    }
    src += h0 * s_head + vofs;
#pragma unroll
    for (int b = 0; b < kAssembleHeads; ++b)
      if (b < nh) w[b] = *(const SB_PGLOBAL pu32x4_t*)(src + b * s_head);
  }
  char* dst = a.out + ((static_cast<int64_t>(plane) * a.num_heads + h0) * a.seq_len + t) * a.row_bytes +
              vofs;
  const int64_t s_out = a.seq_len * a.row_bytes;
#pragma unroll
  for (int b = 0; b < kAssembleHeads; ++b)
    if (b < nh) __builtin_nontemporal_store(w[b], (SB_PGLOBAL pu32x4_t*)(dst + b * s_out));
}

struct OutProjArgs {
  char* out;
  int64_t o_s_row;        // bytes
  const float* attn;      // [S, K] rows
  int64_t a_s_row;        // floats
  const char* weight;     // [F, K] rows
  int64_t w_s_row;        // bytes
  const float* bias;      // [F], or nullptr
  const uint8_t* mask;
  const int32_t* positions;  // computed positions, their count at [seq_len]
  int64_t seq_len;
  int64_t num_features;
  int steps;              // K / 16
};

template <int IT>
__device__ __forceinline__ pf32x4_t load4_wide(const char* p) {
  if (IT == SB_DTYPE_F32) return *(const SB_PGLOBAL pf32x4_t*)p;
  const pu32x2_t w = *(const SB_PGLOBAL pu32x2_t*)p;
  if (IT == SB_DTYPE_BF16)
    return pf32x4_t{__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u),
                    __uint_as_float(w.y << 16), __uint_as_float(w.y & 0xffff0000u)};
  return pf32x4_t{f16_to_f32(static_cast<uint16_t>(w.x & 0xffffu)),
                  f16_to_f32(static_cast<uint16_t>(w.x >> 16)),
                  f16_to_f32(static_cast<uint16_t>(w.y & 0xffffu)),
                  f16_to_f32(static_cast<uint16_t>(w.y >> 16))};
}

template <int IT>
__device__ __forceinline__ void store4_round(char* p, pf32x4_t v) {
  if (IT == SB_DTYPE_F32) {
    *(SB_PGLOBAL pf32x4_t*)p = v;
    return;
  }
  pu32x2_t w;
  if (IT == SB_DTYPE_BF16)
    w = pu32x2_t{pack2_bf16(v.x, v.y), pack2_bf16(v.z, v.w)};
  else
    w = pu32x2_t{static_cast<uint32_t>(f32_to_f16(v.x)) | (static_cast<uint32_t>(f32_to_f16(v.y)) << 16),
                 static_cast<uint32_t>(f32_to_f16(v.z)) | (static_cast<uint32_t>(f32_to_f16(v.w)) << 16)};
  *(SB_PGLOBAL pu32x2_t*)p = w;
}

// Output projection, out[p, f] = sum_k attn[p, k] W[f, k] (+ bias) of the computed positions, in
// fp32 on v_mfma_f32_16x16x4_f32 (IEEE fp32 products and sums), rounded once; positions that are
// not computed get zeros.
//   * A wave multiplies 32 features x 32 rows. Operands come straight from memory (both have k
//     contiguous): with the contraction index permuted alike on both sides, one 4-element load of
//     a row per lane feeds MFMA j with elements 16 s + 4 (lane / 16) + j, each j summed in a chain
//     of its own (the error of K / 4 sums).
//   * WIDE false: a workgroup is one 32 x 32 tile, its four waves taking every fourth 16-wide step
//     and adding their sums through LDS: a few hundred rows still give every CU a workgroup.
//     WIDE true: 64 x 64 tiles, one 32 x 32 block per wave, half the operand traffic.
template <int IT, bool WIDE>
__global__ __launch_bounds__(256) void prefill_output_kernel(const OutProjArgs a) {
  constexpr int TN = WIDE ? 64 : 32;
  constexpr int kEs = IT == SB_DTYPE_F32 ? 4 : 2;
  __shared__ __align__(16) float part[WIDE ? 1 : 4 * 32 * 36];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int64_t f0 = static_cast<int64_t>(blockIdx.x) * TN;
  const int64_t n0 = static_cast<int64_t>(blockIdx.y) * TN;

  // Zeros for the positions of [n0, n0 + TN) that are not computed.
  constexpr int kQuads = TN / 4;
  for (int i = tid; i < TN * kQuads; i += 256) {
    const int64_t t = n0 + i / kQuads, f = f0 + 4 * (i % kQuads);
    if (t < a.seq_len && f < a.num_features && !a.mask[t])
      store4_round<IT>(a.out + t * a.o_s_row + f * kEs, pf32x4_t{0.f, 0.f, 0.f, 0.f});
  }

  const int64_t rows = min(static_cast<int64_t>(a.positions[a.seq_len]), a.seq_len);
  if (n0 >= rows) return;  // uniform
  const int64_t fw = f0 + (WIDE ? 32 * (wave & 1) : 0);
  const int64_t nw = n0 + (WIDE ? 32 * (wave >> 1) : 0);
  const char* wp[2];
  const float* ap[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int64_t f = min(fw + 16 * b + lr, a.num_features - 1);
    wp[b] = a.weight + f * a.w_s_row + 4 * lg * kEs;
    const int64_t n = min(nw + 16 * b + lr, rows - 1);
    ap[b] = a.attn + a.positions[n] * a.a_s_row + 4 * lg;
  }
  pf32x4_t acc[2][2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[i][j][c] = pf32x4_t{0.f, 0.f, 0.f, 0.f};

  constexpr int kInc = WIDE ? 1 : 4;
  // Steps whose operands are loaded before the first is multiplied. (Eight take 184 VGPRs, one
  // workgroup per CU: 25 us where four take 16.)
  constexpr int kUnroll = 4;
  const int s_begin = WIDE ? 0 : wave;
  auto batch = [&](int s0, auto whole_c) {
    constexpr bool WHOLE = decltype(whole_c)::value;
    pf32x4_t wf[kUnroll][2], af[kUnroll][2];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int s = WHOLE ? s0 + u * kInc : min(s0 + u * kInc, a.steps - 1);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        wf[u][b] = load4_wide<IT>(wp[b] + static_cast<int64_t>(s) * (16 * kEs));
        af[u][b] = *(const SB_PGLOBAL pf32x4_t*)(ap[b] + static_cast<int64_t>(s) * 16);
      }
    }
    if (!WHOLE) {                       // steps past the end multiply zeros
#pragma unroll
      for (int u = 0; u < kUnroll; ++u)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          if (s0 + u * kInc >= a.steps) wf[u][b] = af[u][b] = pf32x4_t{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u)
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[i][j][c] =
                __builtin_amdgcn_mfma_f32_16x16x4f32(wf[u][i][c], af[u][j][c], acc[i][j][c], 0, 0, 0);
  };
  int s0 = s_begin;
  for (; s0 + (kUnroll - 1) * kInc < a.steps; s0 += kInc * kUnroll) batch(s0, std::true_type{});
  if (s0 < a.steps) batch(s0, std::false_type{});
  // Lane (lr, lg) of block (i, j) holds features 16 i + 4 lg .. + 3 of row 16 j + lr.
  auto finish = [&](int64_t n, int64_t f, pf32x4_t v) {
    if (n >= rows || f >= a.num_features) return;
    if (a.bias) v += *(const SB_PGLOBAL pf32x4_t*)(a.bias + f);
    store4_round<IT>(a.out + a.positions[n] * a.o_s_row + f * kEs, v);
  };
  if (WIDE) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        finish(nw + 16 * j + lr, fw + 16 * i + 4 * lg,
               (acc[i][j][0] + acc[i][j][1]) + (acc[i][j][2] + acc[i][j][3]));
    return;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      *reinterpret_cast<pf32x4_t*>(&part[(wave * 32 + 16 * j + lr) * 36 + 16 * i + 4 * lg]) =
          (acc[i][j][0] + acc[i][j][1]) + (acc[i][j][2] + acc[i][j][3]);
  __syncthreads();
  const int row = tid / 8, col = 4 * (tid % 8);
  pf32x4_t sum = *reinterpret_cast<const pf32x4_t*>(&part[row * 36 + col]);
#pragma unroll
  for (int w = 1; w < 4; ++w)
    sum += *reinterpret_cast<const pf32x4_t*>(&part[(w * 32 + row) * 36 + col]);
  finish(n0 + row, f0 + col, sum);
}

}  // namespace
}  // namespace sb

using namespace sb;

extern "C" int sb_prefill_index(const uint8_t* compute_mask, const int32_t* donor_pos,
                                const int32_t* target_pos, int64_t num_pairs, int64_t seq_len,
                                int64_t donor_seq_len, int32_t* index, int32_t* positions,
                                void* stream) {
  const char* fn = "sb_prefill_index";
  clear_error();
  if (seq_len == 0) return SB_OK;
  if (seq_len < 0 || seq_len > 0x7ffffffe || num_pairs < 0 || num_pairs > 0x7ffffffe)
    return fail(fn, "invalid sizes");
  if (!compute_mask || !index || !positions || (num_pairs > 0 && (!donor_pos || !target_pos)))
    return fail(fn, "null pointer argument");
  const int64_t blocks = 1 + (seq_len + kPrefillIndexThreads - 1) / kPrefillIndexThreads;
  SB_LAUNCH("prefill_index", prefill_index_kernel, dim3(static_cast<unsigned>(blocks)),
            dim3(kPrefillIndexThreads), static_cast<hipStream_t>(stream), compute_mask, donor_pos,
            target_pos, num_pairs, seq_len, donor_seq_len, index, positions);
  return check_launch(fn);
}

extern "C" int sb_prefill_assemble(void* cache, const void* donor, const void* qkv,
                                   const int32_t* index, int64_t num_layers, int64_t num_heads,
                                   int64_t seq_len, int64_t head_dim, const int64_t* ds,
                                   int64_t qkv_stride, int32_t dtype, void* stream) {
  const char* fn = "sb_prefill_assemble";
  clear_error();
  if (num_layers == 0 || num_heads == 0 || seq_len == 0 || head_dim == 0) return SB_OK;
  if (elem_size(dtype) == 0) return fail(fn, "invalid dtype");
  if (!cache || !donor || !qkv || !index || !ds) return fail(fn, "null pointer argument");
  if (num_layers < 0 || 2 * num_layers > 65535 || num_heads < 0 ||
      num_heads > 65535 * kAssembleHeads || seq_len < 0 || head_dim < 0)
    return fail(fn, "invalid sizes");
  if (ds[4] != 1) return fail(fn, "head_dim must be contiguous (stride 1)");
  const int64_t es = elem_size(dtype);
  const int64_t row_bytes = head_dim * es;
  int lg = 0;
  while ((int64_t{16} << lg) < row_bytes && lg < 16) ++lg;
  if ((int64_t{16} << lg) != row_bytes)
    return fail(fn, "rows must be a power of two of 16-byte vectors");
  if (vec_bytes({reinterpret_cast<int64_t>(cache), reinterpret_cast<int64_t>(donor),
                 reinterpret_cast<int64_t>(qkv), ds[0] * es, ds[1] * es, ds[2] * es, ds[3] * es,
                 qkv_stride * es}) < 16)
    return fail(fn, "rows must be 16-byte aligned");
  AssembleArgs a{};
  a.out = static_cast<char*>(cache);
  a.donor = static_cast<const char*>(donor);
  a.d_s_layer = ds[0] * es;
  a.d_s_kv = ds[1] * es;
  a.d_s_head = ds[2] * es;
  a.d_s_seq = ds[3] * es;
  a.qkv = static_cast<const char*>(qkv);
  a.q_s_row = qkv_stride * es;
  a.index = index;
  a.seq_len = seq_len;
  a.num_heads = static_cast<int>(num_heads);
  a.row_bytes = static_cast<int>(row_bytes);
  a.vpr_log2 = lg;
  const int64_t gx = ((seq_len << lg) + 255) / 256;
  if (gx > 0x7fffffff) return fail(fn, "grid too large");
  const dim3 grid(static_cast<unsigned>(gx), static_cast<unsigned>(2 * num_layers),
                  static_cast<unsigned>((num_heads + kAssembleHeads - 1) / kAssembleHeads));
  SB_LAUNCH("prefill_assemble", prefill_assemble_kernel, grid, dim3(256),
            static_cast<hipStream_t>(stream), a);
  return check_launch(fn);
}

extern "C" int sb_prefill_output_projection(void* out, const float* attn, const void* weight,
                                            const float* bias, const uint8_t* compute_mask,
                                            const int32_t* positions, int64_t seq_len,
                                            int64_t in_features, int64_t out_features,
                                            int64_t attn_stride, int64_t weight_stride,
                                            int64_t out_stride, int32_t dtype, void* stream) {
  const char* fn = "sb_prefill_output_projection";
  clear_error();
  if (seq_len == 0 || out_features == 0) return SB_OK;
  if (elem_size(dtype) == 0) return fail(fn, "invalid dtype");
  if (!out || !attn || !weight || !compute_mask || !positions)
    return fail(fn, "null pointer argument");
  if (seq_len < 0 || seq_len > 0x7ffffffe || in_features <= 0 || in_features % 16 != 0 ||
      in_features > 0x7fffffff || out_features < 0 || out_features % 4 != 0)
    return fail(fn, "invalid sizes (input features in 16s, output features in 4s)");
  const int64_t es = elem_size(dtype);
  if (vec_bytes({reinterpret_cast<int64_t>(attn), attn_stride * 4}) < 16 ||
      vec_bytes({reinterpret_cast<int64_t>(weight), reinterpret_cast<int64_t>(out),
                 weight_stride * es, out_stride * es}) < 4 * es ||
      reinterpret_cast<uintptr_t>(bias) % 16)
    return fail(fn, "rows must be aligned to four elements");
  OutProjArgs a{};
  a.out = static_cast<char*>(out);
  a.o_s_row = out_stride * es;
  a.attn = attn;
  a.a_s_row = attn_stride;
  a.weight = static_cast<const char*>(weight);
  a.w_s_row = weight_stride * es;
  a.bias = bias;
  a.mask = compute_mask;
  a.positions = positions;
  a.seq_len = seq_len;
  a.num_features = out_features;
  a.steps = static_cast<int>(in_features / 16);
  // 64 x 64 tiles once a quarter of the positions (a usual computed share) fill every CU's four
  // SIMDs twice with them.
  const bool wide = ((seq_len / 4 + 63) / 64) * ((out_features + 63) / 64) >= 512;
  const int64_t tn = wide ? 64 : 32;
  const int64_t gx = (out_features + tn - 1) / tn, gy = (seq_len + tn - 1) / tn;
  if (gx > 0x7fffffff || gy > 65535) return fail(fn, "grid too large");
  const dim3 grid(static_cast<unsigned>(gx), static_cast<unsigned>(gy));
  hipStream_t st = static_cast<hipStream_t>(stream);
#define SB_OUT_CASE(DT)                                                                        \
  if (dtype == DT) {                                                                           \
    if (wide)                                                                                  \
      SB_LAUNCH("prefill_output", (prefill_output_kernel<DT, true>), grid, dim3(256), st, a);  \
    else                                                                                       \
      SB_LAUNCH("prefill_output", (prefill_output_kernel<DT, false>), grid, dim3(256), st, a); \
    return check_launch(fn);                                                                   \
  }
  SB_OUT_CASE(SB_DTYPE_F32)
  SB_OUT_CASE(SB_DTYPE_F16)
  SB_OUT_CASE(SB_DTYPE_BF16)
#undef SB_OUT_CASE
  return fail(fn, "invalid dtype");
}
