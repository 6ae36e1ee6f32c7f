// fp32 partial-prefill attention on the fp32 matrix cores (included by sb_attn.hip).
//
// Same semantics and work items as the bf16 / fp16 kernel there, for fp32 tensors with head_dim
// 64 or 128: products, softmax weights and sums all in fp32 (v_mfma_f32_16x16x4_f32 multiplies
// and accumulates in IEEE fp32).
//
// Bound: fp32 matrix-core rate (a library fp32 GEMM reaches 152 TFLOP/s on this chip) where
// there are rows to fill it; the VALU kernel it replaces (one wave per row and head) re-read
// every K/V row once per row and head and issued two VALU instructions per product. Per call, merge
// included: 154 rows of 1024 tokens, 14 q / 2 KV heads x 64, 81 -> 17 us; 1000 rows of 3000
// tokens, 28 / 4 x 128, 2274 -> 240 us (75 TFLOP/s of useful products).
//
// Layout: a workgroup of 4 waves owns 64 flattened (row, q-head-in-group) rows of one KV head,
// 16 per wave, and one chunk of the key range, in tiles of 4096 / D keys staged in LDS (33 KB:
// four workgroups per CU hide each other's barriers and loads).
//   * S^T = K Q^T: A = K (lane: key l % 16), B = Q (lane: row l % 16). The contraction index is
//     permuted the same way on both sides so that one ds_read_b128 of a K row feeds four MFMAs:
//     MFMA j of step s takes elements 16 s + 4 (l / 16) + j. K rows are padded by 4 floats: the
//     16 rows of a read fall on disjoint banks.
//   * The accumulator hands each lane 4 keys of ONE row, which are exactly the B operand of
//     O^T += V^T P^T (MFMA r takes keys 4 (l / 16) + r): P never leaves its registers.
//   * V^T's rows are permuted as well (A row m of MFMA t is d = 64 b + 4 m + t), so one
//     ds_read_b128 of a V row feeds four MFMAs and each lane ends with 16 consecutive d of its
//     row: 16-byte stores.
//   * The next tile is loaded to registers while the current one is multiplied.
// Masked keys: a key past a row's position has P = 0, but 0 x a non-finite V would still be NaN.
// Staging notes tiles with a non-finite V element; such a tile, where some row masks part of it,
// adds its products one key at a time over each row's own keys.

namespace sb {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kF32Waves = 4;
constexpr int kF32Rows = 16 * kF32Waves;     // flattened rows per workgroup
constexpr int kF32Threads = 64 * kF32Waves;

// Key split of the fp32 kernel. With 1024 row tiles (four workgroups on each CU) every slot has
// work unsplit; below that the key range splits so that about 1024 chunks run, none shorter
// than two tiles of 4096 / D keys: 1000 tokens, 400 rows, 14 / 2 heads x 64 take 24 us against
// 29.5 us with one tile and 32 us with four (merge and set-up against idle CUs).
// With t < 1024 row tiles x KV heads a split has at most 2048 / t + 1 chunks each: partials of
// 3071 x 64 rows of D + 2 floats, 102 MB, whatever the call.
constexpr int64_t kF32Slots = 1024;
#ifndef SB_F32_MIN_TILES
#define SB_F32_MIN_TILES 2
#endif
__host__ __device__ inline KeySplit key_split_f32(int64_t n_tiles, int64_t num_kv_heads,
                                                  int64_t kv_len, int64_t head_dim) {
  const int64_t kv_pad = (kv_len + 63) / 64 * 64;
  int64_t ks = kv_pad;
  if (n_tiles * num_kv_heads < kF32Slots) {
    const int64_t least = SB_F32_MIN_TILES * 4096 / head_dim;
    ks = (n_tiles * num_kv_heads * (kv_len / 2) / kF32Slots + 63) / 64 * 64;
    if (ks < least) ks = least;
    if (ks > kv_pad) ks = kv_pad;
  }
  const int64_t chunks = (kv_len + ks - 1) / ks;
  return KeySplit{static_cast<int>(ks), static_cast<int>(chunks < 1 ? 1 : chunks)};
}

// Four consecutive elements as fp32.
template <int IT>
__device__ __forceinline__ float4 load4_f32(const char* p) {
  if (IT == SB_DTYPE_F32) {
    const f32x4_t v = *(const SB_GLOBAL f32x4_t*)p;
    return make_float4(v.x, v.y, v.z, v.w);
  }
  const u32x2_t w = *(const SB_GLOBAL u32x2_t*)p;
  auto up = [](uint32_t h) {
    return IT == SB_DTYPE_BF16 ? bf16_to_f32(static_cast<uint16_t>(h))
                               : f16_to_f32(static_cast<uint16_t>(h));
  };
  return make_float4(up(w.x & 0xffffu), up(w.x >> 16), up(w.y & 0xffffu), up(w.y >> 16));
}

// Value of v in lane (lane ^ 16).
__device__ __forceinline__ float xor16(float v) {
  return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x401F));
}

template <int IT, int D, bool PAGED>
__global__ __launch_bounds__(kF32Threads) void attn_f32_kernel(const AttnArgs args) {
  constexpr int TK = 4096 / D;                 // keys per tile (64 or 32)
  constexpr int KB = TK / 16;                  // 16-key blocks
  constexpr int NS = D / 16;                   // 16-element contraction steps of QK^T
  constexpr int NB = D / 64;                   // 64-wide blocks of the output dimension
  constexpr int KST = D + 4;                   // padded K row (floats)
  constexpr int CPR = D / 4;                   // 4-element chunks per row
  constexpr int NLD = TK * CPR / kF32Threads;  // chunks per thread per tile (4)
  constexpr int RPL = kF32Threads / CPR;       // rows one load of every thread covers
  __shared__ __align__(16) float Ks[TK * KST];
  __shared__ __align__(16) float Vs[TK * D];
  __shared__ int red_max[kF32Waves];
  __shared__ int red_min[kF32Waves];
  __shared__ int v_flag;                       // 1 + the last tile with a non-finite V element

  AttnArgs a = args;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int lr = lane & 15;                    // this lane's row of the wave
  const int lg = lane >> 4;                    // its quarter of each 16-key / 16-element group

  const int64_t rows_kv = attn_num_rows(a) * a.group;
  const int64_t n_tiles_live = (rows_kv + kF32Rows - 1) / kF32Rows;
  if (n_tiles_live <= 0) return;  // uniform
  if (a.device_split) {
    const KeySplit sp = key_split_f32(n_tiles_live, a.num_kv_heads, a.kv_len, D);
    a.ksplit = a.ksplit_first = sp.ksplit;
    a.max_chunks = sp.max_chunks;
    a.n_tiles = n_tiles_live;
  }
  const Item item = decode_item(a, n_tiles_live, blockIdx.x);
  if (item.tile < 0 || item.chunk >= a.max_chunks) return;  // uniform
  const int kvh = item.kvh;
  const int k0 = chunk_begin(a, item.chunk);
  if (k0 >= a.kv_len) return;  // uniform
  const int kc = static_cast<int>(min(static_cast<int64_t>(k0) + chunk_len(a, item.chunk), a.kv_len));

  // This lane's row and its query (B operand of S^T = K Q^T).
  const int64_t r = item.tile * kF32Rows + wave * 16 + lr;
  int p = -1, qh = 0;
  int64_t qrow = 0;
  if (r < rows_kv) {
    const int64_t pi = r / a.group;
    qh = kvh * a.group + static_cast<int>(r - pi * a.group);
    int pp = a.positions[pi];
    if (pp >= a.kv_len) pp = static_cast<int>(a.kv_len - 1);
    qrow = a.q_by_position ? max(pp, 0) : pi;
    p = pp < 0 ? -1 : pp;
  }
  if (tid == 0) v_flag = 0;
  const int pmax_w = wave_max_i(p);
  const int pmin_w = wave_min_i(p < 0 ? 0x7fffffff : p);
  if (lane == 0) {
    red_max[wave] = pmax_w;
    red_min[wave] = pmin_w;
  }
  float4 qf[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) qf[s] = make_float4(0.f, 0.f, 0.f, 0.f);
  if (p >= 0) {
    const char* qp = a.q + qrow * a.q_s_row + qh * a.q_s_head;
    constexpr int es = IT == SB_DTYPE_F32 ? 4 : 2;
#pragma unroll
    for (int s = 0; s < NS; ++s) qf[s] = load4_f32<IT>(qp + (16 * s + 4 * lg) * es);
  }
  __syncthreads();
  int kend = red_max[0];
  int pmin = red_min[0];
#pragma unroll
  for (int w = 1; w < kF32Waves; ++w) {
    kend = max(kend, red_max[w]);
    pmin = min(pmin, red_min[w]);
  }
  kend = __builtin_amdgcn_readfirstlane(kend) + 1;
  pmin = __builtin_amdgcn_readfirstlane(pmin);
  if (k0 >= kend) return;  // uniform: kend comes from shared memory
  const int k1 = min(kc, kend);
  const int nchunks = chunk_count(a, kend);
  const int plim = min(p, k1 - 1);
  const int pmax_c = min(__builtin_amdgcn_readfirstlane(pmax_w), k1 - 1);
  const int ntiles = (k1 - k0 + TK - 1) / TK;

  // Tile staging: chunk q of this thread is row q * RPL + tid / CPR, elements 4 (tid % CPR)...
  // Keys past the chunk are clamped to its last one (masked below). The blocks of a tile are
  // looked up one tile before its loads.
  constexpr int es = IT == SB_DTYPE_F32 ? 4 : 2;
  const char* kbase = a.k + kvh * a.k_s_head + (tid % CPR) * 4 * es;
  const char* vbase = a.v + kvh * a.v_s_head + (tid % CPR) * 4 * es;
  int blk[NLD];
  float4 kr[NLD], vr[NLD];
  auto key_of = [&](int t, int q) { return min(k0 + t * TK + q * RPL + tid / CPR, k1 - 1); };
  auto block_of = [&](int key) {
    return a.bs_log2 >= 0 ? key >> a.bs_log2 : key / static_cast<int>(a.block_size);
  };
  auto lookup = [&](int t) {
    if (!PAGED) return;
#pragma unroll
    for (int q = 0; q < NLD; ++q) blk[q] = a.block_table[block_of(key_of(t, q))];
  };
  auto fetch = [&](int t) {
#pragma unroll
    for (int q = 0; q < NLD; ++q) {
      const int key = key_of(t, q);
      int64_t ko, vo;
      if (PAGED) {
        const int in_block = key - block_of(key) * static_cast<int>(a.block_size);
        ko = vo = clamp_block(a, blk[q]) * a.s_block + in_block * a.s_pos;
      } else {
        ko = key * a.k_s_seq;
        vo = key * a.v_s_seq;
      }
      kr[q] = load4_f32<IT>(kbase + ko);
      vr[q] = load4_f32<IT>(vbase + vo);
    }
  };

  float m = -INFINITY, l = 0.f;  // l: this lane's share of the row sum
  f32x4_t o[NB][4];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int t = 0; t < 4; ++t) o[b][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // scale * log2(e) in two parts: rounded to one float it would tilt every weight the same way,
  // by up to 2^-23 times its distance from the row's largest score.
  const float c_log2 = a.scale_log2, c_lo = a.scale_log2_lo;

  lookup(0);
  fetch(0);
  if (ntiles > 1) lookup(1);
  for (int it = 0; it < ntiles; ++it) {
    const int t0 = k0 + it * TK;
    if (it > 0) __syncthreads();  // every wave is done with the tile in LDS
    float probe = 0.f;            // NaN if an element of V is not finite
#pragma unroll
    for (int q = 0; q < NLD; ++q) {
      const int row = q * RPL + tid / CPR, col = 4 * (tid % CPR);
      *reinterpret_cast<float4*>(&Ks[row * KST + col]) = kr[q];
      *reinterpret_cast<float4*>(&Vs[row * D + col]) = vr[q];
      probe = __builtin_fmaf(vr[q].x, 0.f, probe);
      probe = __builtin_fmaf(vr[q].y, 0.f, probe);
      probe = __builtin_fmaf(vr[q].z, 0.f, probe);
      probe = __builtin_fmaf(vr[q].w, 0.f, probe);
    }
    if (probe != probe) v_flag = it + 1;  // same value from every writer
    __syncthreads();
    if (it + 1 < ntiles) {
      fetch(it + 1);
      if (it + 2 < ntiles) lookup(it + 2);
    }
    if (t0 > pmax_c) continue;  // wave-uniform: none of this wave's rows reaches the tile

    // Each score is the sum of four independent chains of D / 4 products (element j of every
    // step): a single chain of D would double the rounding error.
    f32x4_t s[KB];
#pragma unroll
    for (int k2 = 0; k2 < KB; k2 += 2) {
      f32x4_t ac[2][4];
#pragma unroll
      for (int st = 0; st < NS; ++st) {
        const float qe[4] = {qf[st].x, qf[st].y, qf[st].z, qf[st].w};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float4 kf = *reinterpret_cast<const float4*>(
              &Ks[(16 * (k2 + h) + lr) * KST + 16 * st + 4 * lg]);
          const float ke[4] = {kf.x, kf.y, kf.z, kf.w};
#pragma unroll
          for (int j = 0; j < 4; ++j)
            ac[h][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                ke[j], qe[j], st == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : ac[h][j], 0, 0, 0);
        }
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) s[k2 + h] = (ac[h][0] + ac[h][1]) + (ac[h][2] + ac[h][3]);
    }
    const bool masked = t0 + TK - 1 > min(pmin, k1 - 1);  // uniform
    if (masked) {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (t0 + 16 * kb + 4 * lg + i > plim) s[kb][i] = -INFINITY;
    }
    float mx = s[0][0];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[kb][i]);
    mx = fmaxf(mx, xor16(mx));
    mx = fmaxf(mx, xor32(mx));
    const float m_new = fmaxf(m, c_log2 * mx);
    // 2^(m - m_new): 1 unless the maximum moved, 0 for the row's first live tile.
    const float alpha = m_new > m ? (m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - m_new)) : 1.f;
    m = m_new;
    const float negm = m == -INFINITY ? 0.f : -m;
    float tsum = 0.f;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // (a masked score is -inf, which c_lo must not turn into inf - inf)
        const float x = __builtin_fmaf(c_lo, fmaxf(s[kb][i], -3.4e38f),
                                       __builtin_fmaf(c_log2, s[kb][i], negm));
        s[kb][i] = __builtin_amdgcn_exp2f(x);
        tsum += s[kb][i];
      }
    l = l * alpha + tsum;
    if (masked && v_flag == it + 1) {
      // Rare: a non-finite V in a tile some row masks part of; each row adds its own keys only.
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int t = 0; t < 4; ++t) o[b][t] *= alpha;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll 1
          for (int g = 0; g < 4; ++g) {
            const float pk = __shfl(s[kb][i], (g << 4) | lr, 64);
            const int row = 16 * kb + 4 * g + i;
            if (t0 + row > plim) continue;
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float4 v =
                    *reinterpret_cast<const float4*>(&Vs[row * D + 64 * b + 16 * lg + 4 * e]);
                o[b][0][e] += pk * v.x;
                o[b][1][e] += pk * v.y;
                o[b][2][e] += pk * v.z;
                o[b][3][e] += pk * v.w;
              }
          }
    } else {
      // Each CH blocks' product in accumulators of its own (chains of D / 4 keys), their sum
      // added to O: the rounding error of one long chain would be larger.
      constexpr int CH = D / 64;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        f32x4_t sum[4];
#pragma unroll
        for (int k2 = 0; k2 < KB; k2 += CH) {
          f32x4_t pv[4];
#pragma unroll
          for (int h = 0; h < CH; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float4 v = *reinterpret_cast<const float4*>(
                  &Vs[(16 * (k2 + h) + 4 * lg + i) * D + 64 * b + 4 * lr]);
              const float ve[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
              for (int t = 0; t < 4; ++t)
                pv[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                    ve[t], s[k2 + h][i], h + i == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : pv[t], 0, 0, 0);
            }
#pragma unroll
          for (int t = 0; t < 4; ++t) sum[t] = k2 == 0 ? pv[t] : sum[t] + pv[t];
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) o[b][t] = o[b][t] * alpha + sum[t];
      }
    }
  }

  // Lane (row lr, quarter lg) holds d = 64 b + 16 lg + 4 e + t in o[b][t][e].
  l += xor16(l);
  l += xor32(l);
  if (p < 0) return;
  if (nchunks == 1) {
    char* op = a.o + qrow * a.o_s_row + qh * a.o_s_head;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *reinterpret_cast<float4*>(op + (64 * b + 16 * lg + 4 * e) * 4) =
            make_float4(o[b][0][e] / l, o[b][1][e] / l, o[b][2][e] / l, o[b][3][e] / l);
    return;
  }
  const int64_t slot =
      ((static_cast<int64_t>(kvh) * a.n_tiles + item.tile) * a.max_chunks + item.chunk) * kF32Rows +
      wave * 16 + lr;
  float* po = a.part_o + slot * D;
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      *reinterpret_cast<float4*>(po + 64 * b + 16 * lg + 4 * e) =
          make_float4(o[b][0][e], o[b][1][e], o[b][2][e], o[b][3][e]);
  // A row none of whose keys lie in the chunk is marked -inf (its sum is 0); a NaN sum keeps a
  // finite mark, so that the merge carries it to the output.
  if (lg == 0)
    *reinterpret_cast<float2*>(a.part_ml + slot * 2) =
        make_float2(l == 0.f ? -INFINITY : (m == -INFINITY ? 0.f : m), l);
}

}  // namespace sb
