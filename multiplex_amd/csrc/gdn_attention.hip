// Full-attention layers of the hybrid trunk and of the MTP draft head
// (Qwen3.5 gated attention) on gfx950.
//
//   attn_qk_kernel       one wave per token and group of heads: RMSNorm of q and k over
//                        the head dim (y = x / rms(x) * w), the rotary
//                        embedding of the first `rot` dims (rotate-half form,
//                        angle pos * base^(-2i/rot)), q to [B, T, Hq, D]; k and
//                        v appended to the KV cache [B, Hkv, cap, D] at
//                        positions pos0[b] .. pos0[b] + T - 1.
//   attn_fwd_kernel      causal GQA attention over the cache on bf16 MFMA
//                        with an online softmax in fp32.  The query rows of
//                        one kv-head are (token, q-head of its group) pairs,
//                        so the g = Hq / Hkv heads of a group share every K/V
//                        block a workgroup stages in LDS.  RT = 4: four waves
//                        own 16 rows each and walk the same 64-key blocks
//                        (prefill); RT = 1: one 16-row tile, each wave takes
//                        16 keys of every block (decode and draft verify,
//                        where a group has at most 16 rows), and the four
//                        partial softmax states merge in LDS at the end.
//                        Keys may also be split over workgroups; the partial
//                        states then go to a workspace and
//   attn_combine_kernel  merges them.
//   attn_prefill_kernel  long prefills (>= 512 rows per kv-head): 128-row
//                        workgroups, 64-key K / V blocks double-buffered in
//                        LDS (K by direct loads, V transposed on its way in),
//                        one barrier per block; keys split likewise.
//                        The output is multiplied by sigmoid(gate) on the way
//                        out when a gate is given.
//   rms_norm_kernel      the layers' RMSNorm over the hidden size, optionally of
//                        a residual sum it also writes out.
//   pos_add_kernel       the cache offsets' advance and rollback.
//   silu_mul_kernel      the MLP's silu(gate) * up.
#include <cfloat>

#include "gdn_common.hpp"

namespace {

using namespace gdn;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr float kLog2e = 1.4426950408889634f;
constexpr int KB = 64;  // keys per staged block

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x4 mfma16k16(i16x4 a, i16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float sigmoid(float x) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-x * kLog2e));
}

// ------------------------------------------------------------ attn_qk

struct QkParams {
  const uint16_t* qg;  // [B, T, Hq, 2D]: q, then the output gate, per head (token stride qg_ld)
  const uint16_t* kn;  // [B, T, Hkv, D] (token stride kv_ld)
  const uint16_t* vn;  // [B, T, Hkv, D] (token stride kv_ld)
  int64_t qg_ld, kv_ld;
  const void* qw;      // [D] q_norm weight
  const void* kw;      // [D] k_norm weight
  int wdt;
  const int32_t* pos0;  // [B] position of each row's first new token (its cache length)
  uint16_t* q;          // [B, T, Hq, D]
  uint16_t* kc;         // [B, Hkv, cap, D]
  uint16_t* vc;
  int B, T, Hq, Hkv, cap, rot;
  float eps, log2_base;
};

// A row's first position, clamped so that its T new tokens fit in the cache
// (offsets come from device memory and are not validated on the host).
__device__ __forceinline__ int first_pos(const int32_t* pos0, int b, int T, int cap) {
  return min(max(pos0[b], 0), cap - T);
}

// EPL bf16 elements of a row at any 2-byte address, as one load / store (callers
// may pass rows at any element offset; the hardware takes unaligned dwords).
template <int EPL>
struct RowVec {
  typedef uint16_t type __attribute__((ext_vector_type(EPL), aligned(2)));
};

// One wave takes NH heads of one token (q heads, then k, then v), the last
// wave of a token the rest.  The rotary angles depend on the token and the
// lane only, so exp2 and sincos -- most of the arithmetic, computed per head
// it bounded the kernel at 70.6 us for 4096 tokens of 16 + 2 x 4 heads --
// run once for the NH heads, whose rows are all loaded before the first is
// used and whose chains overlap.  A wave with more heads runs longer, so calls
// of few rows (tokens x heads) take few heads a wave (graph-replayed, us, NH =
// 1 / 3 / 6; a wave per head with the angles of its own before them):
//   16 + 2 x 4 heads of 256:   1 token 3.3, 3.5 / 4.3 / 5.5;  160 tokens (3840 rows) 5.4, 5.0 / 5.2 / 5.9;
//      200 (4800) 5.9, 5.5 / 5.3 / 6.0;  600 (14400) 12.3, 11.0 / 7.9 / 8.0;  700 (16800) 13.7, 12.3 / 8.8 / 8.2;
//      2048 34.1, 29.1 / 17.1 / 16.2
//   4 + 2 x 1 of 256:        600 tokens (3600) 5.2, 4.9 / 5.1 / 5.8;  700 (4200) 5.8, 5.5 / 5.2 / 5.9
//   64 + 2 x 8 of 128:   160 tokens (12800) 7.5, 7.2 / 5.4 / 5.5;  256 (20480) 10.5, 9.9 / 6.6 / 6.4
// (4096 tokens of 16 + 2 x 4 heads of 256, 100 MB, 28.3: 3.6 TB/s).
template <int D, int NH>
__global__ __launch_bounds__(256) void attn_qk_kernel(const QkParams p) {
  constexpr int EPL = D / 64;  // elements per lane
  typedef typename RowVec<EPL>::type vec;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int heads = p.Hq + 2 * p.Hkv;  // q heads, k heads, v heads
  const uint32_t per_tok = (heads + NH - 1) / NH;
  const uint32_t item = blockIdx.x * 4u + wave;
  const uint32_t bt = item / per_tok;
  if (bt >= static_cast<uint32_t>(p.B) * p.T) return;  // wave-uniform
  const int h0 = static_cast<int>(item % per_tok) * NH;
  const int t = static_cast<int>(bt % p.T), b = static_cast<int>(bt / p.T);
  const int d0 = EPL * lane;

  vec raw[NH];
#pragma unroll
  for (int n = 0; n < NH; ++n) {
    const int h = min(h0 + n, heads - 1);
    const uint16_t* src;
    if (h < p.Hq) src = p.qg + bt * p.qg_ld + h * 2 * D;
    else if (h < p.Hq + p.Hkv) src = p.kn + bt * p.kv_ld + (h - p.Hq) * D;
    else src = p.vn + bt * p.kv_ld + (h - p.Hq - p.Hkv) * D;
    raw[n] = *reinterpret_cast<const vec*>(src + d0);
  }
  // norm weights as raw bits (converted after every load is issued); a single
  // head's wave loads its own kind's only
  uint32_t qwr[EPL], kwr[EPL];
  const void* qwp = NH > 1 || h0 < p.Hq ? p.qw : p.kw;
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    if (p.wdt == GDN_DTYPE_F32) {
      qwr[e] = static_cast<const uint32_t*>(qwp)[d0 + e];
      if (NH > 1) kwr[e] = static_cast<const uint32_t*>(p.kw)[d0 + e];
    } else {
      qwr[e] = static_cast<const uint16_t*>(qwp)[d0 + e];
      if (NH > 1) kwr[e] = static_cast<const uint16_t*>(p.kw)[d0 + e];
    }
  }
  const int pos = first_pos(p.pos0, b, p.T, p.cap) + t;

  // rotary embedding of dims [0, rot): d < half pairs with d + half
  const int half = p.rot / 2;
  const int shift = half / EPL;  // lanes between partners
  const bool lower = d0 < half;
  const int partner = lower ? lane + shift : lane - shift;
  float sn[EPL], cs[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    sn[e] = 0.0f;
    cs[e] = 1.0f;
  }
  if (d0 < p.rot && h0 < p.Hq + p.Hkv) {
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const int i = half > 0 ? (d0 + e) % half : 0;
      const float inv_freq = exp2f(-2.0f * static_cast<float>(i) / static_cast<float>(p.rot) * p.log2_base);
      sincosf(static_cast<float>(pos) * inv_freq, &sn[e], &cs[e]);
    }
  }
  auto weight = [&](uint32_t u) {
    return p.wdt == GDN_DTYPE_F32 ? __uint_as_float(u)
                                  : (p.wdt == GDN_DTYPE_BF16 ? bf16_to_f32(static_cast<uint16_t>(u))
                                                             : f16_to_f32(static_cast<uint16_t>(u)));
  };
  float qw[EPL], kw[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    qw[e] = weight(qwr[e]);
    kw[e] = NH > 1 ? weight(kwr[e]) : qw[e];
  }

  // the heads' chains (sum, norm, exchange) carry no branch, so they overlap
  float r[NH];
#pragma unroll
  for (int n = 0; n < NH; ++n) {
    float ss = 0.0f;
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const float x = bf16_to_f32(raw[n][e]);
      ss += x * x;
    }
    r[n] = rsqrtf(wave_sum(ss) / D + p.eps);
  }
  vec out[NH];
#pragma unroll
  for (int n = 0; n < NH; ++n) {
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      // RMSNorm, rounded to bf16 (the norm's output dtype)
      const float x = bf16_to_f32(f32_to_bf16(bf16_to_f32(raw[n][e]) * r[n] * (h0 + n < p.Hq ? qw[e] : kw[e])));
      const float other = __shfl(x, partner, 64);
      const float y = d0 < p.rot ? (lower ? x * cs[e] - other * sn[e] : x * cs[e] + other * sn[e]) : x;
      out[n][e] = f32_to_bf16(y);
    }
  }
#pragma unroll
  for (int n = 0; n < NH; ++n) {
    const int h = h0 + n;
    if (h >= heads) return;  // wave-uniform
    if (h < p.Hq) {
      *reinterpret_cast<vec*>(p.q + (static_cast<int64_t>(bt) * p.Hq + h) * D + d0) = out[n];
    } else {
      const bool is_k = h < p.Hq + p.Hkv;  // v goes into the cache as is
      const int hkv = h - p.Hq - (is_k ? 0 : p.Hkv);
      *reinterpret_cast<vec*>((is_k ? p.kc : p.vc) + ((static_cast<int64_t>(b) * p.Hkv + hkv) * p.cap + pos) * D + d0) =
          is_k ? out[n] : raw[n];
    }
  }
}

// ------------------------------------------------------------ attn_fwd

struct AttnParams {
  const uint16_t* q;   // [B, T, Hq, D]
  const uint16_t* qg;  // gate source [B, T, Hq, 2D] (gate = second half of a head; token stride qg_ld) or null
  int64_t qg_ld;
  const uint16_t* kc;  // [B, Hkv, cap, D]
  const uint16_t* vc;
  const int32_t* pos0;  // [B]
  uint16_t* out;        // [B, T, Hq, D]
  float* part;          // split partials: O [B, Hkv, rows_pad, n_split, D], then m and l [.., n_split]
  int B, T, Hq, Hkv, cap;
  int n_split, split_len, rows_pad;
  float scale_log2;  // softmax scale * log2(e)
};

// Partial-state addressing for split keys.
__device__ __forceinline__ int64_t part_row(const AttnParams& p, int b, int hkv, int r) {
  return ((static_cast<int64_t>(b) * p.Hkv + hkv) * p.rows_pad + r) * p.n_split;
}

// Final value of one output element pair / quad: o / l, times the gate.
template <int D>
__device__ __forceinline__ void store_out4(const AttnParams& p, int b, int t, int hq, int d, f32x4 o, float inv_l) {
  const int64_t bt = static_cast<int64_t>(b) * p.T + t;
  const int64_t row = bt * p.Hq + hq;
  f32x4 y = o * inv_l;
  if (p.qg != nullptr) {
    const u32x2 gg = *reinterpret_cast<const u32x2*>(p.qg + bt * p.qg_ld + hq * 2 * D + D + d);
    y[0] *= sigmoid(__uint_as_float(gg.x << 16));
    y[1] *= sigmoid(__uint_as_float(gg.x & 0xffff0000u));
    y[2] *= sigmoid(__uint_as_float(gg.y << 16));
    y[3] *= sigmoid(__uint_as_float(gg.y & 0xffff0000u));
  }
  *reinterpret_cast<u32x2*>(p.out + row * D + d) = u32x2{pk_bf16(y[0], y[1]), pk_bf16(y[2], y[3])};
}

template <int D, int RT>
__global__ __launch_bounds__(256) void attn_fwd_kernel(const AttnParams p) {
  constexpr int KP = D + 8;   // K row stride (bf16): 16-byte fragment reads of 16 rows hit distinct banks
  constexpr int VP = D + 16;  // V row stride: the transposed reads of 4 rows hit distinct banks
  constexpr int KT = RT == 4 ? 4 : 1;  // 16-key tiles per wave and block
  constexpr int NS = D / 32;           // k-steps of q . k
  constexpr int NJ = D / 16;           // 16-wide d tiles of the output
  constexpr int CPT = KB * D / 8 / 256;  // 16-byte chunks per thread of a K (or V) block

  const int b = blockIdx.z;
  const int hkv = blockIdx.y % p.Hkv, rb = blockIdx.y / p.Hkv;
  const int split = blockIdx.x;
  const int g = p.Hq / p.Hkv;
  const int n_rows = p.T * g;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lq = lane >> 4;
  const int p0 = first_pos(p.pos0, b, p.T, p.cap);

  const int row0 = rb * 16 * RT;
  const int t_last = min((row0 + 16 * RT - 1) / g, p.T - 1);
  const int k_lo = split * p.split_len;
  const int k_hi = min(p0 + t_last + 1, k_lo + p.split_len);  // keys of this workgroup: [k_lo, k_hi)
  const int rt = RT == 4 ? wave : 0;
  const int sub = RT == 4 ? 0 : wave;  // first 16-key tile of this wave in each block

  // this wave's 16 rows (lane lr's row): Q as the B operand of S^T = K Q^T
  const int r = row0 + 16 * rt + lr;
  const bool row_ok = r < n_rows;
  const int t = row_ok ? r / g : 0;
  const int hq = hkv * g + (row_ok ? r % g : 0);
  const int kmax = p0 + t;  // last key row r may see
  bf16x8 qf[NS];
  {
    const uint16_t* qrow = p.q + ((static_cast<int64_t>(b) * p.T + t) * p.Hq + hq) * D;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(qrow + 32 * s + 8 * lq);
      qf[s] = __builtin_bit_cast(bf16x8, row_ok ? v : u32x4{0u, 0u, 0u, 0u});
    }
  }

  __shared__ __align__(16) unsigned char smem[KB * (KP + VP) * 2];
  uint16_t(*Ks)[KP] = reinterpret_cast<uint16_t(*)[KP]>(smem);
  uint16_t(*Vs)[VP] = reinterpret_cast<uint16_t(*)[VP]>(smem + KB * KP * 2);

  // the next block, in flight: chunk c = tid + 256 i is row c / (D/8), columns (c % (D/8)) * 8 ..
  // The cache is read with nontemporal loads: each step streams it once, and at
  // decode sizes (1 GB at B=64 and 4096 positions) it cannot stay in the
  // last-level cache, whose allocation on every read cost 15% (180.4 against
  // 152.8 us at B=64).
  u32x4 kr[CPT], vr[CPT];
  const int64_t head_base = (static_cast<int64_t>(b) * p.Hkv + hkv) * p.cap * D;
  auto load_blk = [&](int kb) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int c = tid + 256 * i;
      const int row = c / (D / 8), col = (c % (D / 8)) * 8;
      const int key = kb + row;
      const int64_t off = head_base + static_cast<int64_t>(min(key, k_hi - 1)) * D + col;  // in bounds: k_hi <= cap
      kr[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p.kc + off));
      vr[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p.vc + off));
    }
  };
  auto store_blk = [&](int kb) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int c = tid + 256 * i;
      const int row = c / (D / 8), col = (c % (D / 8)) * 8;
      const bool ok = kb + row < k_hi;  // keys past the range read as zero (the cache there is unset)
      const u32x4 z = {0u, 0u, 0u, 0u};
      *reinterpret_cast<u32x4*>(&Ks[row][col]) = ok ? kr[i] : z;
      *reinterpret_cast<u32x4*>(&Vs[row][col]) = ok ? vr[i] : z;
    }
  };

  float m = -INFINITY, l = 0.0f;  // running max (log2 units) and this lane's share of the sum
  f32x4 o[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) o[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  const int nblk = k_hi > k_lo ? (k_hi - k_lo + KB - 1) / KB : 0;
  if (nblk > 0) load_blk(k_lo);
  for (int blk = 0; blk < nblk; ++blk) {
    const int kb = k_lo + KB * blk;
    __syncthreads();  // the previous block's reads are done
    store_blk(kb);
    __syncthreads();
    if (blk + 1 < nblk) load_blk(kb + KB);

    // S^T = K Q^T for this wave's key tiles: lane (r, q) holds keys 16 kt + 4q + i of row r
    f32x4 sc[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      f32x4 a = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < NS; ++s)
        a = mfma16(*reinterpret_cast<const bf16x8*>(&Ks[16 * (sub + kt) + lr][32 * s + 8 * lq]), qf[s], a);
      sc[kt] = a;
    }
    float mb = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = kb + 16 * (sub + kt) + 4 * lq + i;
        const bool ok = row_ok && key <= kmax && key < k_hi;
        sc[kt][i] = ok ? sc[kt][i] * p.scale_log2 : -INFINITY;
        mb = fmaxf(mb, sc[kt][i]);
      }
    mb = fmaxf(mb, __shfl_xor(mb, 16, 64));
    mb = fmaxf(mb, __shfl_xor(mb, 32, 64));
    const float m_new = fmaxf(m, mb);
    const float m_use = m_new == -INFINITY ? 0.0f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m - m_use);
    m = m_new;
    float ps = 0.0f;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sc[kt][i] = __builtin_amdgcn_exp2f(sc[kt][i] - m_use);
        ps += sc[kt][i];
      }
    l = l * alpha + ps;
#pragma unroll
    for (int j = 0; j < NJ; ++j) o[j] *= alpha;

    // O^T += V^T P^T (P as bf16; V^T by transposed LDS reads)
    if constexpr (RT == 4) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        // k-slots: keys 32 ks + 4q + (0..3), then 32 ks + 16 + 4q + (0..3) -- the rows of
        // accumulator tiles 2 ks and 2 ks + 1 held by lane group q
        const bf16x8 pb = __builtin_bit_cast(
            bf16x8, u32x4{pk_bf16(sc[2 * ks][0], sc[2 * ks][1]), pk_bf16(sc[2 * ks][2], sc[2 * ks][3]),
                          pk_bf16(sc[2 * ks + 1][0], sc[2 * ks + 1][1]), pk_bf16(sc[2 * ks + 1][2], sc[2 * ks + 1][3])});
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const uint16_t* va = &Vs[32 * ks + 4 * lq + (lr >> 2)][16 * j + 4 * (lr & 3)];
          const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(va));
          const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(va + 16 * VP));
          const bf16x8 vt = __builtin_bit_cast(bf16x8, i16x8(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)));
          o[j] = mfma16(vt, pb, o[j]);
        }
      }
    } else {
      const u32x2 pw = {pk_bf16(sc[0][0], sc[0][1]), pk_bf16(sc[0][2], sc[0][3])};
      const i16x4 pb = __builtin_bit_cast(i16x4, pw);
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const uint16_t* va = &Vs[16 * sub + 4 * lq + (lr >> 2)][16 * j + 4 * (lr & 3)];
        o[j] = mfma16k16(__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(va)), pb, o[j]);
      }
    }
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);

  const bool split_out = p.n_split > 1;
  if constexpr (RT == 4) {
    // lane (r, q) holds O[row r][16 j + 4 q + i]
    if (!row_ok) return;
    if (split_out) {
      const int64_t pr = part_row(p, b, hkv, r) + split;
      float* po = p.part + pr * D;
#pragma unroll
      for (int j = 0; j < NJ; ++j) *reinterpret_cast<f32x4*>(po + 16 * j + 4 * lq) = o[j];
      if (lq == 0) {
        float* ml = p.part + static_cast<int64_t>(p.B) * p.Hkv * p.rows_pad * p.n_split * D;
        const int64_t n_part = static_cast<int64_t>(p.B) * p.Hkv * p.rows_pad * p.n_split;
        ml[pr] = m;
        ml[n_part + pr] = l;
      }
      return;
    }
    const float inv_l = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) store_out4<D>(p, b, t, hq, 16 * j + 4 * lq, o[j], inv_l);
  } else {
    // merge the four waves' states for the tile's 16 rows (the K/V buffers are free)
    __syncthreads();
    float* Os = reinterpret_cast<float*>(smem);  // [4][16][D]
    float* Ms = Os + 4 * 16 * D;                 // [4][16]
    float* Ls = Ms + 4 * 16;
    static_assert((4 * 16 * D + 2 * 64) * 4 <= KB * (KP + VP) * 2, "merge buffers must fit in the K/V blocks");
#pragma unroll
    for (int j = 0; j < NJ; ++j) *reinterpret_cast<f32x4*>(&Os[(wave * 16 + lr) * D + 16 * j + 4 * lq]) = o[j];
    if (lq == 0) {
      Ms[wave * 16 + lr] = m;
      Ls[wave * 16 + lr] = l;
    }
    __syncthreads();
    // thread: row tid / 16, columns (tid % 16) * D/16 ..
    constexpr int CW = D / 16;
    const int mr = tid >> 4, c0 = (tid & 15) * CW;
    const int rr = row0 + mr;
    if (rr >= n_rows) return;
    float mw[4], ms = -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      mw[w] = Ms[w * 16 + mr];
      ms = fmaxf(ms, mw[w]);
    }
    const float m_use = ms == -INFINITY ? 0.0f : ms;
    float sw[4], lsum = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      sw[w] = __builtin_amdgcn_exp2f(mw[w] - m_use);
      lsum += sw[w] * Ls[w * 16 + mr];
    }
    if (split_out) {
      const int64_t pr = part_row(p, b, hkv, rr) + split;
      float* po = p.part + pr * D;
#pragma unroll
      for (int c = 0; c < CW; c += 4) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < 4; ++w) acc += sw[w] * *reinterpret_cast<const f32x4*>(&Os[(w * 16 + mr) * D + c0 + c]);
        *reinterpret_cast<f32x4*>(po + c0 + c) = acc;
      }
      if ((tid & 15) == 0) {
        float* ml = p.part + static_cast<int64_t>(p.B) * p.Hkv * p.rows_pad * p.n_split * D;
        const int64_t n_part = static_cast<int64_t>(p.B) * p.Hkv * p.rows_pad * p.n_split;
        ml[pr] = ms;
        ml[n_part + pr] = lsum;
      }
      return;
    }
    const float inv_l = lsum > 0.0f ? 1.0f / lsum : 0.0f;
    const int tt = rr / g, hh = hkv * g + rr % g;
#pragma unroll
    for (int c = 0; c < CW; c += 4) {
      f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int w = 0; w < 4; ++w) acc += sw[w] * *reinterpret_cast<const f32x4*>(&Os[(w * 16 + mr) * D + c0 + c]);
      store_out4<D>(p, b, tt, hh, c0 + c, acc, inv_l);
    }
  }
}

// Causal prefills of at least kPrefillRows rows per kv-head: a workgroup owns
// 128 rows in four row groups of 32, so every K or V fragment a wave reads
// from LDS feeds two 16-row MFMA tiles.  64-key blocks are double-buffered in
// LDS and a block costs one barrier:
//   K  goes in by direct global -> LDS loads (each lane's 16 bytes land at
//      16 * lane past the wave's base), rows of D bf16 whose 16-byte granules
//      are XOR-swizzled by (key & 7), so the fragment reads of 8 consecutive
//      keys hit distinct banks;
//   V  is transposed in registers on its way in: Vt[d][position], with the
//      keys of each 32-key group in the k-slot order of the P^T operand
//      (position 8q + 4h + i holds key 16h + 4q + i), so that a V^T fragment
//      is one 16-byte read, like K's; rows of 64 positions whose 16-byte
//      granules are XOR-swizzled by (d & 7), which keeps both the fragment
//      reads and the 8-byte transposed writes free of bank conflicts.  (Transposed LDS reads of a [key][d]
//      block deliver about 45 bytes per clock per CU, against 128 for 16-byte
//      reads.)  Its loads are issued one block ahead of the transpose.
// KG = 2 (head dim 256, whose workgroup fills a CU's LDS): eight waves, two
// per SIMD, the two of a row group taking 32 keys of every block each with a
// softmax state of their own, merged in LDS at the end.  One wave's MFMAs
// then run beside the other's exponentials: a single wave issues a 16x16x32
// MFMA every 9.6 ns at best and two share a SIMD at 7.6 ns each, with two or
// three vector instructions per MFMA free.  Both must fit in 256 registers
// each without a spill (a reload per block waits for every load in flight:
// +9% per fragment), which is why two k-steps of q stay in LDS and few
// fragments are in flight.  KG = 1 (head dim 128): four waves, and two
// workgroups share a CU.
// Measured at 16 query and 4 kv-heads of 256: 4096 tokens 195 -> 165 us
// (840 TFLOP/s), 512 tokens over a 4096-token prefix in one key range 160 ->
// 128 us; four waves with the next block's scores computed between this
// block's exponentials, in registers enough for both, took 209 and 172 us.
// Few rows leave CUs idle, so the keys may be split over workgroups too
// (n_split; 512 tokens over 4096 in four ranges: 60 us with the combine).
// The softmax max is raised only when a row's block max exceeds it by more
// than 8 (log2 units; P stays below 2^8), which skips the rescale of the
// output on most blocks, and only blocks that cross the diagonal or the end
// of the keys are masked.  Workgroups with the longest key ranges go first.

// A raw buffer descriptor of `bytes` bytes at `base` (wave-uniform): reads past its end return zeros.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), 0x00020000);
}
// The same descriptor as four words, for inline assembly.
__device__ __forceinline__ u32x4 buf_words(const void* base, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  return u32x4{static_cast<uint32_t>(a), static_cast<uint32_t>(a >> 32) & 0xffffu, bytes, 0x00020000u};
}

// 16 bytes per lane from a buffer (byte offset voff) straight into LDS at lds_base + 16 * lane (rsrc and
// lds_base wave-uniform).  Issued from inline assembly: the compiler's wait insertion, seeing an LDS DMA in
// a loop, would otherwise drain every LDS read with lgkmcnt(0).  It increments vmcnt like any load; the
// caller waits for it (vmcnt(0)) before the barrier that publishes the block.
__device__ __forceinline__ void lds_dma16(u32x4 rsrc, uint32_t voff, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
               :
               : "v"(voff), "s"(rsrc), "s"(lds_base)
               : "memory", "m0");
}

// Max / sum over the four 16-lane rows of a wave (lanes r, r + 16, r + 32, r + 48), by the
// gfx950 row-swap moves (VALU, no LDS round trip): permlane16_swap(x, x) yields the even and the
// odd rows, permlane32_swap(x, x) the low and the high halves, each in both places.
__device__ __forceinline__ float rows_max(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float rows_sum(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Max over the 64 lanes.
__device__ __forceinline__ float wave_max(float x) {
  x = fmaxf(x, dpp_f<GDN_DPP_QUAD_XOR1>(x));
  x = fmaxf(x, dpp_f<GDN_DPP_QUAD_XOR2>(x));
  x = fmaxf(x, dpp_f<GDN_DPP_HALF_MIRROR>(x));
  x = fmaxf(x, dpp_f<GDN_DPP_ROW_MIRROR>(x));
  return rows_max(x);
}

constexpr int kPrefillRows = 512;  // rows (tokens x heads of a group) per kv-head from which it is used
constexpr int PR = 128;            // rows per workgroup
constexpr int VTP = KB;            // Vt row stride (bf16); 16-byte granules XOR-swizzled by (d & 7)

template <int D, int KG>
__global__ __launch_bounds__(256 * KG) void attn_prefill_kernel(const AttnParams p) {
  constexpr int NT = 256 * KG;                // threads
  constexpr int NS = D / 32;                  // k-steps of q . k
  constexpr int NJ = D / 16;                  // 16-wide d tiles of the output
  constexpr int KTW = 4 / KG;                 // 16-key tiles of a block per wave
  constexpr int KSW = 2 / KG;                 // 32-key groups of a block per wave
  constexpr int KROW = D / 8;                 // 16-byte granules per K row
  constexpr int KDMA = KB * KROW / NT;        // direct loads per thread and K block
  constexpr int VPAIRS = (KB / 4) * KROW / NT;  // (key quad, d octet) pairs per thread and V block
  constexpr int KSTAGE = KB * D * 2;          // bytes
  constexpr int VSTAGE = D * VTP * 2;
  static_assert(KDMA * NT == KB * KROW && VPAIRS * NT == (KB / 4) * KROW, "block must split evenly over the threads");
  static_assert(KDMA <= NS && 4 * VPAIRS <= NS, "at most one K and one V load per k-step");

  constexpr int QL = KG == 2 ? 2 : 0;         // k-steps of q kept in LDS
  constexpr int kMl = KG == 2 ? 8 * 128 * 4 : 0;  // the waves' (m, l) for the merge
  __shared__ __align__(128) unsigned char smem[2 * (KSTAGE + VSTAGE) + kMl + 4 * 2 * QL * 1024];

  const int b = blockIdx.z, split = blockIdx.y;
  const int n_rb = gridDim.x / p.Hkv;
  const int hkv = blockIdx.x % p.Hkv;
  const int rb = n_rb - 1 - static_cast<int>(blockIdx.x) / p.Hkv;  // longest key ranges first
  const int g = p.Hq / p.Hkv;
  const int n_rows = p.T * g;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = wave & 3, kh = wave >> 2;  // the wave's 32 rows of the workgroup's, and its keys of each block
  const int lr = lane & 15, lq = lane >> 4;
  const int p0 = first_pos(p.pos0, b, p.T, p.cap);

  const int row0 = rb * PR;
  const int t_last = min((row0 + PR - 1) / g, p.T - 1);
  const int k_lo = split * p.split_len;
  const int k_hi = min(p0 + t_last + 1, k_lo + p.split_len);  // keys of this workgroup: [k_lo, k_hi)
  const int k_free = min(p0 + row0 / g + 1, k_hi);             // keys below this are visible to every row
  const int nblk = k_hi > k_lo ? (k_hi - k_lo + KB - 1) / KB : 0;

  // the wave's two 16-row tiles; rows past the end compute on q = 0 and are not stored.  The last QL
  // k-steps of q are kept in LDS (both waves of a row group read one copy)
  auto q_lds = [&](int rt, int s) {
    return reinterpret_cast<bf16x8*>(smem + 2 * (KSTAGE + VSTAGE) + kMl) +
           ((rg * 2 + rt) * QL + s - (NS - QL)) * 64 + lane;
  };
  int kmax[2];
  bf16x8 qf[2][NS - QL];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const int r = row0 + 32 * rg + 16 * rt + lr;
    const bool ok = r < n_rows;
    const int t = ok ? r / g : p.T - 1, hq = hkv * g + (ok ? r % g : 0);
    kmax[rt] = p0 + t;
    const uint16_t* qrow = p.q + ((static_cast<int64_t>(b) * p.T + t) * p.Hq + hq) * D;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(qrow + 32 * s + 8 * lq);
      const bf16x8 f = __builtin_bit_cast(bf16x8, ok ? v : u32x4{0u, 0u, 0u, 0u});
      if (s < NS - QL) qf[rt][s] = f;
      else if (kh == 0) *q_lds(rt, s) = f;
    }
  }

  // K and V blocks are read through descriptors that end at the range's last
  // key, so the lane offsets are constants and keys past the range (masked
  // below) read as zeros
  const unsigned char* kc_head =
      reinterpret_cast<const unsigned char*>(p.kc + (static_cast<int64_t>(b) * p.Hkv + hkv) * p.cap * D);
  const unsigned char* vc_head =
      reinterpret_cast<const unsigned char*>(p.vc + (static_cast<int64_t>(b) * p.Hkv + hkv) * p.cap * D);
  auto block_bytes = [&](int kb) { return min(k_hi - kb, KB) * (D * 2); };
  // K block -> stage st: thread tid's load i fills physical granule i * NT + tid, which is row
  // i * KR + tid / KROW, granule (tid % KROW) ^ (row & 7) of the block (the swizzle does not depend on i)
  constexpr int KR = NT / KROW;
  static_assert(KR % 8 == 0, "the swizzle of a granule must not depend on the load");
  const int k_row0 = tid / KROW;
  const uint32_t k_off = k_row0 * (D * 2) + (((tid % KROW) ^ (k_row0 & 7)) * 16);
  // LDS address of the wave's 1 KB slice of load 0 in stage 0
  const uint32_t k_lds = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem)) + wave * 1024);
  auto k_dma = [&](int kb, int bytes, int st, int i) {  // the block's bytes from load i's first row on
    constexpr int kLoad = KR * D * 2;
    lds_dma16(buf_words(kc_head + static_cast<int64_t>(kb) * (D * 2) + i * kLoad, max(bytes - i * kLoad, 0)), k_off,
              k_lds + st * KSTAGE + i * (NT * 16));
  };
  // V block -> registers: pair i is key quad tid % 16 (4 rows) x d octet i * NT / 16 + tid / 16
  const int v_kq = tid % (KB / 4), v_dq = tid / (KB / 4);
  const uint32_t v_off = 4 * v_kq * (D * 2) + v_dq * 16;
  u32x4 vr[VPAIRS][4];
  auto v_load = [&](__amdgpu_buffer_rsrc_t rsrc, int i, int e) {
    vr[i][e] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, v_off + e * (D * 2) + i * NT, 0, 0);
  };
  // registers -> Vt stage st: for each of the octet's 8 d, the quad's 4 keys as one 8-byte write
  const int v_pos = 32 * (v_kq >> 3) + 8 * (v_kq & 3) + 4 * ((v_kq >> 2) & 1);
  const int v_gran = v_pos >> 3, v_half = v_pos & 7;  // the position's granule and offset in it
  // byte offset of d row 8 v_dq's piece; row + c is at (this ^ (c << 4)) + c rows (a row's 128 bytes are aligned)
  const int v_at = 2 * KSTAGE + 8 * v_dq * (VTP * 2) + 16 * v_gran + 2 * v_half;
  auto v_store = [&](int st, int i, int m) {  // d rows 8 (v_dq + i NT / 16) + 2m, + 2m + 1 (d & 7 = 2m, 2m + 1)
    const int at = v_at + st * VSTAGE + i * (NT / 2) * (VTP * 2);
    const uint32_t k0 = vr[i][0][m], k1 = vr[i][1][m], k2 = vr[i][2][m], k3 = vr[i][3][m];
    // byte permutes: the low (0x05040100) and the high (0x07060302) halves of two keys' words
    const u32x2 even = {__builtin_amdgcn_perm(k1, k0, 0x05040100u), __builtin_amdgcn_perm(k3, k2, 0x05040100u)};
    const u32x2 odd = {__builtin_amdgcn_perm(k1, k0, 0x07060302u), __builtin_amdgcn_perm(k3, k2, 0x07060302u)};
    *reinterpret_cast<u32x2*>(smem + (at ^ (2 * m << 4)) + (2 * m) * (VTP * 2)) = even;
    *reinterpret_cast<u32x2*>(smem + (at ^ ((2 * m + 1) << 4)) + (2 * m + 1) * (VTP * 2)) = odd;
  };

  // a wave may see no key of a row in its range: the running max starts at a
  // finite value, so that exp2 of a masked score is 0 and not exp2(-inf + inf)
  float m[2] = {-FLT_MAX, -FLT_MAX}, l[2] = {0.0f, 0.0f};
  f32x4 o[2][NJ];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt)
#pragma unroll
    for (int j = 0; j < NJ; ++j) o[rt][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // K fragment (tile kt, k-step s) of lane (r, q): row 16 kt + r, granule (4s + q) ^ (r & 7)
  // = 8 (s >> 1) + 4 ((s & 1) ^ x2) + (q ^ x01) with x = r & 7: one base for even s, one for odd,
  // each plus 64 (s & ~1) bytes
  const int x2 = (lr >> 2) & 1, y01 = lq ^ (lr & 3);
  const int kf0 = 16 * KTW * kh * (D * 2) + lr * (D * 2);
  const int kfe = kf0 + (4 * x2 + y01) * 16, kfo = kf0 + (4 * (x2 ^ 1) + y01) * 16;
  // V^T fragment (j, ks) of lane (r, q): d row 16 j + r, positions 32 ks + 8q .., granule (4 ks + q) ^ (r & 7)
  const int vfo0 = lr * (VTP * 2) + (4 * (x2 ^ (KG == 2 ? kh : 0)) + y01) * 16;
  const int vfo1 = lr * (VTP * 2) + (4 * (x2 ^ 1) + y01) * 16;

  // Every wave's LDS writes and direct loads are visible to the others.  The 4 VPAIRS loads of V issued after
  // the direct loads may stay in flight (they go to this thread's registers).
  auto publish = [&]() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(4 * VPAIRS) : "memory");
  };
  if (nblk > 0) {
    const int nb = block_bytes(k_lo);
    const int k1 = nblk > 1 ? k_lo + KB : k_lo;
    const __amdgpu_buffer_rsrc_t vrs = buf_rsrc(vc_head + static_cast<int64_t>(k_lo) * (D * 2), nb);
    const __amdgpu_buffer_rsrc_t vrs1 = buf_rsrc(vc_head + static_cast<int64_t>(k1) * (D * 2), block_bytes(k1));
#pragma unroll
    for (int i = 0; i < KDMA; ++i) k_dma(k_lo, nb, 0, i);
#pragma unroll
    for (int i = 0; i < VPAIRS; ++i) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v_load(vrs, i, e);
    }
#pragma unroll
    for (int i = 0; i < VPAIRS; ++i) {
#pragma unroll
      for (int m4 = 0; m4 < 4; ++m4) v_store(0, i, m4);
#pragma unroll
      for (int e = 0; e < 4; ++e) v_load(vrs1, i, e);
    }
  }
  for (int blk = 0; blk < nblk; ++blk) {
    const int kb = k_lo + KB * blk, st = blk & 1;
    publish();  // block blk is in LDS, stage st ^ 1 is free
    // K of the next block goes in during S^T; its V (in registers since the last iteration) is stored,
    // transposed, during O^T, and the registers take the block after it.  Past the end the loads re-read the
    // last block (never used), so that none sits behind a branch.
    const int kb1 = blk + 1 < nblk ? kb + KB : kb, kb2 = blk + 2 < nblk ? kb + 2 * KB : kb1;
    const int nb1 = block_bytes(kb1);
    const __amdgpu_buffer_rsrc_t vrs = buf_rsrc(vc_head + static_cast<int64_t>(kb2) * (D * 2), block_bytes(kb2));

    // S^T = K Q^T: lane (r, q) holds keys 16 kt + 4q + i of row r, for both row tiles
    const unsigned char* Ks = smem + st * KSTAGE;
    auto k_frag = [&](int s, int kt) {
      return *reinterpret_cast<const bf16x8*>(Ks + ((s & 1) ? kfo : kfe) + kt * 16 * (D * 2) + (s & ~1) * 64);
    };
    f32x4 sc[2][KTW];
#pragma unroll
    for (int kt = 0; kt < KTW; ++kt) sc[0][kt] = sc[1][kt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // fragments f = (k-step f / KTW, tile f % KTW), KPF of them in flight
    constexpr int KPF = KG == 2 ? 3 : 4;
    bf16x8 kf[KPF];
#pragma unroll
    for (int f = 0; f < KPF; ++f) kf[f] = k_frag(f / KTW, f % KTW);
#pragma unroll
    for (int f = 0; f < NS * KTW; ++f) {
      const int s = f / KTW, kt = f % KTW;
      const bf16x8 a = kf[f % KPF];
      if (f + KPF < NS * KTW) kf[f % KPF] = k_frag((f + KPF) / KTW, (f + KPF) % KTW);
      if (kt == 0 && s < KDMA) k_dma(kb1, nb1, st ^ 1, s);
      const bool in_regs = s < NS - QL;
      sc[0][kt] = mfma16(a, in_regs ? qf[0][in_regs ? s : 0] : *q_lds(0, s), sc[0][kt]);
      sc[1][kt] = mfma16(a, in_regs ? qf[1][in_regs ? s : 0] : *q_lds(1, s), sc[1][kt]);
    }
    // issue order: fragment f + KPF read ahead of fragment f's two products
    __builtin_amdgcn_sched_group_barrier(0x100, KPF, 0);
#pragma unroll
    for (int f = 0; f < NS * KTW; ++f) {
      if (f + KPF < NS * KTW) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (f % KTW == 0 && f / KTW >= NS - QL) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // q
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
    }

    if (kb + KB > k_free) {
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int kt = 0; kt < KTW; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int key = kb + 16 * (KTW * kh + kt) + 4 * lq + i;
            if (!(key <= kmax[rt] && key < k_hi)) sc[rt][kt][i] = -INFINITY;
          }
    }
    float mb[2];
    bool grow = false;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      float x = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < KTW; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) x = fmaxf(x, sc[rt][kt][i]);
      mb[rt] = rows_max(x) * p.scale_log2;
      grow |= mb[rt] > m[rt] + 8.0f;
    }
    if (__builtin_amdgcn_ballot_w64(grow) != 0) {
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        const float m_new = fmaxf(m[rt], mb[rt]);
        const float alpha = __builtin_amdgcn_exp2f(m[rt] - m_new);
        m[rt] = m_new;
        l[rt] *= alpha;
#pragma unroll
        for (int j = 0; j < NJ; ++j) o[rt][j] *= alpha;
      }
    }
    // P = exp2(s * scale - m) as the B operand of O^T += V^T P^T: k-slots 8q .. 8q+3 are keys
    // 32 ks + 4q + (0..3) (accumulator tile 2 ks), 8q+4 .. 8q+7 are keys 32 ks + 16 + 4q + (0..3)
    bf16x8 pb[2][KSW];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      float ps = 0.0f;
#pragma unroll
      for (int kt = 0; kt < KTW; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          sc[rt][kt][i] = __builtin_amdgcn_exp2f(fmaf(sc[rt][kt][i], p.scale_log2, -m[rt]));
          ps += sc[rt][kt][i];
        }
      l[rt] += ps;
#pragma unroll
      for (int ks = 0; ks < KSW; ++ks)
        pb[rt][ks] = __builtin_bit_cast(
            bf16x8, u32x4{pk_bf16(sc[rt][2 * ks][0], sc[rt][2 * ks][1]), pk_bf16(sc[rt][2 * ks][2], sc[rt][2 * ks][3]),
                          pk_bf16(sc[rt][2 * ks + 1][0], sc[rt][2 * ks + 1][1]),
                          pk_bf16(sc[rt][2 * ks + 1][2], sc[rt][2 * ks + 1][3])});
    }

    // O^T += V^T P^T
    const unsigned char* Vt = smem + 2 * KSTAGE + st * VSTAGE;
    constexpr int NF = KSW * NJ;  // V^T fragments per block: (ks, j) = (f / NJ, f % NJ)
    constexpr int VPF = 4;        // fragments in flight
    auto v_frag = [&](int f) {
      return *reinterpret_cast<const bf16x8*>(Vt + (f / NJ ? vfo1 : vfo0) + (f % NJ) * 16 * (VTP * 2));
    };
    bf16x8 vf[VPF];
#pragma unroll
    for (int f = 0; f < VPF; ++f) vf[f] = v_frag(f);
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const bf16x8 a = vf[f % VPF];
      if (f + VPF < NF) vf[f % VPF] = v_frag(f + VPF);
      const int j = f % NJ, ks = f / NJ;
      o[0][j] = mfma16(a, pb[0][ks], o[0][j]);
      o[1][j] = mfma16(a, pb[1][ks], o[1][j]);
      // the next block's V into the free stage
      constexpr int VST = NF / (4 * VPAIRS);  // fragments per transposed store
      if (f % VST == VST - 1) {
        v_store(st ^ 1, f / VST / 4, (f / VST) % 4);
        if ((f / VST) % 4 == 3) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v_load(vrs, f / VST / 4, e);
        }
      }
    }
    // issue order: fragment f + VPF read ahead of fragment f's two products
    __builtin_amdgcn_sched_group_barrier(0x100, VPF, 1);
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      if (f + VPF < NF) __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 1);
    }
  }

  __builtin_amdgcn_s_waitcnt(0);  // no direct load may land in LDS after this
  float lt[2] = {rows_sum(l[0]), rows_sum(l[1])};
  // row tile rt's state (lane (r, q): O[row r][16 j + 4 q + i]) to the output, or to the split's partials
  auto store_tile = [&](auto rtc) {
    constexpr int rt = decltype(rtc)::value;
    const int r = row0 + 32 * rg + 16 * rt + lr;
    if (r >= n_rows) return;
    if (p.n_split == 1) {
      const float inv_l = 1.0f / lt[rt];  // (l = 0: every score is -inf, whose softmax is NaN)
#pragma unroll
      for (int j = 0; j < NJ; ++j) store_out4<D>(p, b, r / g, hkv * g + r % g, 16 * j + 4 * lq, o[rt][j], inv_l);
      return;
    }
    const int64_t pr = part_row(p, b, hkv, r) + split;
    const int64_t n_part = static_cast<int64_t>(p.B) * p.Hkv * p.rows_pad * p.n_split;
    if (lq == 0) {
      p.part[n_part * D + pr] = m[rt];
      p.part[n_part * (D + 1) + pr] = lt[rt];
    }
    if (nblk == 0) return;  // the combine does not read the O of a range without keys (l = 0)
#pragma unroll
    for (int j = 0; j < NJ; ++j) *reinterpret_cast<f32x4*>(p.part + pr * D + 16 * j + 4 * lq) = o[rt][j];
  };
  if constexpr (KG == 1) {
    store_tile(std::integral_constant<int, 0>{});
    store_tile(std::integral_constant<int, 1>{});
  } else {
    // the two waves of a row group merge: wave kh finishes row tile kh, and
    // hands its state of the other tile over in LDS (the K / V stages are free)
    float* xo = reinterpret_cast<float*>(smem);  // [8 waves][NJ][64 lanes][4]
    float* xml = xo + 8 * NJ * 256;              // [8 waves][2][64 lanes]
    static_assert(8 * NJ * 256 * 4 <= 2 * (KSTAGE + VSTAGE), "the exchange must fit in the stages");
    __syncthreads();
    auto hand_over = [&](auto rtc) {
      constexpr int rt = decltype(rtc)::value;
#pragma unroll
      for (int j = 0; j < NJ; ++j) *reinterpret_cast<f32x4*>(xo + ((wave * NJ + j) * 64 + lane) * 4) = o[rt][j];
      xml[wave * 128 + lane] = m[rt];
      xml[wave * 128 + 64 + lane] = lt[rt];
    };
    auto finish = [&](auto rtc) {
      constexpr int rt = decltype(rtc)::value;
      const int w = wave ^ 4;
      const float m2 = xml[w * 128 + lane], l2 = xml[w * 128 + 64 + lane];
      const float mm = fmaxf(m[rt], m2);
      const float a1 = __builtin_amdgcn_exp2f(m[rt] - mm), a2 = __builtin_amdgcn_exp2f(m2 - mm);
      m[rt] = mm;
      lt[rt] = a1 * lt[rt] + a2 * l2;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        o[rt][j] = a1 * o[rt][j] + a2 * *reinterpret_cast<const f32x4*>(xo + ((w * NJ + j) * 64 + lane) * 4);
      store_tile(rtc);
    };
    if (kh == 0) hand_over(std::integral_constant<int, 1>{});
    else hand_over(std::integral_constant<int, 0>{});
    __syncthreads();
    if (kh == 0) finish(std::integral_constant<int, 0>{});
    else finish(std::integral_constant<int, 1>{});
  }
}

// One wave per (row, kv-head, batch row): the split partials of a row merged.
// A range without keys of the row (l = 0) may have left its O unwritten: it is
// skipped, its loads read the row's first range with keys instead.
// Lane s takes range s's m and l (64 ranges a pass), and eight ranges' O are
// in flight at a time.
template <int D>
__global__ __launch_bounds__(256) void attn_combine_kernel(const AttnParams p) {
  const int lane = threadIdx.x & 63;
  const int g = p.Hq / p.Hkv;
  const int n_rows = p.T * g;
  const int64_t item =
      static_cast<int64_t>(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  if (item >= static_cast<int64_t>(p.B) * p.Hkv * n_rows) return;
  const int r = static_cast<int>(item % n_rows);
  const int hkv = static_cast<int>((item / n_rows) % p.Hkv);
  const int b = static_cast<int>(item / (static_cast<int64_t>(n_rows) * p.Hkv));
  const int64_t n_part = static_cast<int64_t>(p.B) * p.Hkv * p.rows_pad * p.n_split;
  const int64_t pr = part_row(p, b, hkv, r);
  const float* pm = p.part + n_part * D + pr;
  const float* pl = p.part + n_part * (D + 1) + pr;
  constexpr int EPL = D / 64, NB = 8;
  typedef float vec __attribute__((ext_vector_type(EPL)));
  vec acc = {};
  float m = -FLT_MAX, lsum = 0.0f;
  for (int s0 = 0; s0 < p.n_split; s0 += 64) {
    const int n = min(64, p.n_split - s0);
    const float ls = lane < n ? pl[s0 + lane] : 0.0f;
    const float ms = lane < n && ls != 0.0f ? pm[s0 + lane] : -FLT_MAX;
    const uint64_t has = __builtin_amdgcn_ballot_w64(ls != 0.0f);
    if (has == 0) continue;
    const int first = __builtin_ctzll(has);
    const float m_new = fmaxf(m, wave_max(ms));
    const float keep = __builtin_amdgcn_exp2f(m - m_new);
    m = m_new;
    const float w = __builtin_amdgcn_exp2f(ms - m);  // the lane's range
    acc *= keep;
    lsum = lsum * keep + wave_sum(ls != 0.0f ? w * ls : 0.0f);
    for (int s = 0; s < n; s += NB) {
      vec v[NB];
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const int si = min(s + i, n - 1);
        const int src = (has >> si) & 1 ? si : first;
        v[i] = *reinterpret_cast<const vec*>(p.part + (pr + s0 + src) * D + EPL * lane);
      }
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const int si = min(s + i, n - 1);
        const float wi = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w), si));
        if (s + i < n && ((has >> si) & 1)) acc += wi * v[i];  // wave-uniform
      }
    }
  }
  // l = 0: every score is -inf, whose softmax is NaN (zeros in the kernel of fewer rows)
  const float inv_l = n_rows >= kPrefillRows || lsum > 0.0f ? 1.0f / lsum : 0.0f;
  const int t = r / g, hq = hkv * g + r % g;
  if constexpr (EPL == 4) {
    store_out4<D>(p, b, t, hq, EPL * lane, acc, inv_l);
  } else {
    const int64_t bt = static_cast<int64_t>(b) * p.T + t;
    const int64_t row = bt * p.Hq + hq;
    float y0 = acc[0] * inv_l, y1 = acc[1] * inv_l;
    const int d = EPL * lane;
    if (p.qg != nullptr) {
      const uint16_t* gp = p.qg + bt * p.qg_ld + hq * 2 * D + D + d;
      y0 *= sigmoid(bf16_to_f32(gp[0]));
      y1 *= sigmoid(bf16_to_f32(gp[1]));
    }
    *reinterpret_cast<uint32_t*>(p.out + row * D + d) = pk_bf16(y0, y1);
  }
}

// ------------------------------------------------------------ rms_norm

// Eight weights from index i (a multiple of 8) as floats: one 16-byte load for
// bf16 / fp16, two for fp32 (the branch is uniform).
__device__ __forceinline__ void load_w8(const void* w, int wdt, int i, float out[8]) {
  if (wdt == GDN_DTYPE_F32) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(static_cast<const float*>(w) + i);
    const f32x4 b = *reinterpret_cast<const f32x4*>(static_cast<const float*>(w) + i + 4);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      out[k] = a[k];
      out[4 + k] = b[k];
    }
  } else {
    const u32x4 v = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(w) + i);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint16_t lo = static_cast<uint16_t>(v[k] & 0xffffu), hi = static_cast<uint16_t>(v[k] >> 16);
      out[2 * k] = wdt == GDN_DTYPE_BF16 ? bf16_to_f32(lo) : f16_to_f32(lo);
      out[2 * k + 1] = wdt == GDN_DTYPE_BF16 ? bf16_to_f32(hi) : f16_to_f32(hi);
    }
  }
}

// One workgroup per row; 8 bf16 elements per thread and chunk, chunk c of
// thread t at 8 t + 2048 c.  With a residual, the row is h = bf16(x + res)
// (written to h_out when given) and y = norm(h); y's rows are y_ld elements
// apart.  The first kRegChunks chunks of h stay in registers between the sum
// of squares and the output (one pass over memory up to D = 8192); chunks
// beyond are read again, from h_out when this thread wrote them (h_out may
// alias x), else recomputed.
constexpr int kRegChunks = 4;
__global__ __launch_bounds__(256) void rms_norm_kernel(const uint16_t* x, const uint16_t* res, uint16_t* h_out,
                                                       const void* w, int wdt, uint16_t* y, int64_t y_ld, int D,
                                                       float eps) {
  const int64_t row = blockIdx.x;
  const uint16_t* xr = x + row * D;
  const uint16_t* rr = res != nullptr ? res + row * D : nullptr;
  auto load_h = [&](int c) {
    u32x4 v = *reinterpret_cast<const u32x4*>(xr + c);
    if (rr != nullptr) {
      const u32x4 r = *reinterpret_cast<const u32x4*>(rr + c);
#pragma unroll
      for (int k = 0; k < 4; ++k)
        v[k] = pk_bf16(__uint_as_float(v[k] << 16) + __uint_as_float(r[k] << 16),
                       __uint_as_float(v[k] & 0xffff0000u) + __uint_as_float(r[k] & 0xffff0000u));
    }
    return v;
  };
  auto sq = [](u32x4 v) {
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float a = __uint_as_float(v[k] << 16), bb = __uint_as_float(v[k] & 0xffff0000u);
      ss += a * a + bb * bb;
    }
    return ss;
  };
  const int c0 = 8 * threadIdx.x;
  u32x4 hv[kRegChunks];
  float wv[kRegChunks][8];
  float ss = 0.0f;
#pragma unroll
  for (int j = 0; j < kRegChunks; ++j) {
    const int c = c0 + 2048 * j;
    if (c < D) {
      hv[j] = load_h(c);
      load_w8(w, wdt, c, wv[j]);
    }
  }
#pragma unroll
  for (int j = 0; j < kRegChunks; ++j) {
    const int c = c0 + 2048 * j;
    if (c < D) {
      if (h_out != nullptr) *reinterpret_cast<u32x4*>(h_out + row * D + c) = hv[j];
      ss += sq(hv[j]);
    }
  }
  for (int c = c0 + 2048 * kRegChunks; c < D; c += 2048) {
    const u32x4 v = load_h(c);
    if (h_out != nullptr) *reinterpret_cast<u32x4*>(h_out + row * D + c) = v;
    ss += sq(v);
  }
  __shared__ float part[4];
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float r = rsqrtf((part[0] + part[1] + part[2] + part[3]) / D + eps);
  auto out8 = [&](int c, u32x4 v, const float* wk) {
    u32x4 o;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      o[k] = pk_bf16(__uint_as_float(v[k] << 16) * r * wk[2 * k], __uint_as_float(v[k] & 0xffff0000u) * r * wk[2 * k + 1]);
    *reinterpret_cast<u32x4*>(y + row * y_ld + c) = o;
  };
#pragma unroll
  for (int j = 0; j < kRegChunks; ++j) {
    const int c = c0 + 2048 * j;
    if (c < D) out8(c, hv[j], wv[j]);
  }
  for (int c = c0 + 2048 * kRegChunks; c < D; c += 2048) {
    const u32x4 v = h_out != nullptr ? *reinterpret_cast<const u32x4*>(h_out + row * D + c) : load_h(c);
    float wk[8];
    load_w8(w, wdt, c, wk);
    out8(c, v, wk);
  }
}

// ------------------------------------------------------------ pos_add

// pos[b] = max(pos[b] + delta, lo): a KV cache's advance and rollback, one
// launch each (the rollback was a subtraction and a clamp, two launches of
// 1.5 us and 4 us of host time for a few integers).
__global__ __launch_bounds__(256) void pos_add_kernel(int32_t* pos, int B, int32_t delta, int32_t lo) {
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b < B) pos[b] = max(static_cast<int32_t>(static_cast<uint32_t>(pos[b]) + static_cast<uint32_t>(delta)), lo);
}

// ------------------------------------------------------------ silu_mul

// out[r, i] = silu(gu[r, i]) * gu[r, I + i]; 8 elements per thread.
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* gu, uint16_t* out, int64_t rows, int I) {
  const int64_t i8 = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 8;
  if (i8 >= rows * I) return;
  const int64_t r = i8 / I;
  const int c = static_cast<int>(i8 % I);
  const u32x4 gv = *reinterpret_cast<const u32x4*>(gu + r * 2 * I + c);
  const u32x4 uv = *reinterpret_cast<const u32x4*>(gu + r * 2 * I + I + c);
  u32x4 o;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float g0 = __uint_as_float(gv[k] << 16), g1 = __uint_as_float(gv[k] & 0xffff0000u);
    const float u0 = __uint_as_float(uv[k] << 16), u1 = __uint_as_float(uv[k] & 0xffff0000u);
    o[k] = pk_bf16(silu(g0) * u0, silu(g1) * u1);
  }
  *reinterpret_cast<u32x4*>(out + i8) = o;
}

int64_t attn_rows_pad(int64_t T, int64_t Hq, int64_t Hkv, int rt) {
  const int64_t n_rows = T * (Hq / Hkv);
  const int64_t tile = 16 * rt;
  return (n_rows + tile - 1) / tile * tile;
}

int attn_rt(int64_t T, int64_t Hq, int64_t Hkv) { return T * (Hq / Hkv) <= 16 ? 1 : 4; }

}  // namespace

extern "C" size_t gdn_attn_workspace_bytes(int64_t B, int64_t T, int64_t Hq, int64_t Hkv, int64_t D,
                                           int64_t n_split) {
  if (B <= 0 || T <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || D <= 0 || n_split < 1) return 0;
  if (n_split == 1) return 0;
  const int64_t rows_pad = attn_rows_pad(T, Hq, Hkv, attn_rt(T, Hq, Hkv));
  return static_cast<size_t>(B * Hkv * rows_pad * n_split) * (D + 2) * sizeof(float);
}

extern "C" int gdn_attn_qk(const void* qg, int64_t qg_ld, const void* k_new, const void* v_new, int64_t kv_ld,
                           const void* q_norm_w, const void* k_norm_w, int w_dtype, float eps, const int32_t* pos0,
                           void* q_out, void* k_cache, void* v_cache, int64_t B, int64_t T, int64_t Hq, int64_t Hkv,
                           int64_t D, int64_t cap, int64_t rot, float rope_base, void* stream) {
  using gdn_host::fail;
  if (D != 128 && D != 256) return fail(GDN_ERR_UNSUPPORTED, "gdn_attn_qk: head dim must be 128 or 256 (got %lld)", (long long)D);
  if (B < 0 || T < 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || cap < T || cap > INT32_MAX)
    return fail(GDN_ERR_INVALID, "gdn_attn_qk: bad sizes");
  if (rot < 0 || rot > D || rot % (2 * (D / 64)) != 0 || (rot > 0 && (rot / 2) % (D / 64) != 0))
    return fail(GDN_ERR_UNSUPPORTED, "gdn_attn_qk: rotary dims %lld not supported for head dim %lld", (long long)rot,
                (long long)D);
  if (!gdn_host::dtype_ok(w_dtype) || !(rope_base > 0.0f) || !(eps >= 0.0f))
    return fail(GDN_ERR_INVALID, "gdn_attn_qk: bad norm weight dtype, eps or rope base");
  if (B * T == 0) return GDN_OK;
  if (!qg || !k_new || !v_new || !q_norm_w || !k_norm_w || !pos0 || !q_out || !k_cache || !v_cache)
    return fail(GDN_ERR_INVALID, "gdn_attn_qk: null pointer");
  if (B * T * (Hq + 2 * Hkv) > INT32_MAX) return fail(GDN_ERR_UNSUPPORTED, "gdn_attn_qk: problem too large");
  if (qg_ld == 0) qg_ld = 2 * Hq * D;
  if (kv_ld == 0) kv_ld = Hkv * D;
  if (qg_ld < 2 * Hq * D || kv_ld < Hkv * D) return fail(GDN_ERR_INVALID, "gdn_attn_qk: token strides below the rows");
  QkParams p;
  p.qg = static_cast<const uint16_t*>(qg);
  p.kn = static_cast<const uint16_t*>(k_new);
  p.vn = static_cast<const uint16_t*>(v_new);
  p.qg_ld = qg_ld;
  p.kv_ld = kv_ld;
  p.qw = q_norm_w;
  p.kw = k_norm_w;
  p.wdt = w_dtype;
  p.pos0 = pos0;
  p.q = static_cast<uint16_t*>(q_out);
  p.kc = static_cast<uint16_t*>(k_cache);
  p.vc = static_cast<uint16_t*>(v_cache);
  p.B = static_cast<int>(B);
  p.T = static_cast<int>(T);
  p.Hq = static_cast<int>(Hq);
  p.Hkv = static_cast<int>(Hkv);
  p.cap = static_cast<int>(cap);
  p.rot = static_cast<int>(rot);
  p.eps = eps;
  p.log2_base = log2f(rope_base);
  hipStream_t st = static_cast<hipStream_t>(stream);
  // heads per wave by the rows of all heads (attn_qk_kernel's comment has both sides of each line)
  auto launch = [&](auto nh) {
    constexpr int NH = decltype(nh)::value;
    const dim3 grid(static_cast<unsigned>((B * T * ((Hq + 2 * Hkv + NH - 1) / NH) + 3) / 4));
    if (D == 256) hipLaunchKernelGGL((attn_qk_kernel<256, NH>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((attn_qk_kernel<128, NH>), grid, dim3(256), 0, st, p);
  };
  const int64_t rows = B * T * (Hq + 2 * Hkv);
  if (rows <= 4096) launch(std::integral_constant<int, 1>{});
  else if (rows <= 16384) launch(std::integral_constant<int, 3>{});
  else launch(std::integral_constant<int, 6>{});
  return gdn_host::check_launch("gdn_attn_qk");
}

extern "C" int gdn_attn_fwd(const void* q, const void* qg, int64_t qg_ld, const void* k_cache, const void* v_cache,
                            const int32_t* pos0, void* out, float scale, int64_t B, int64_t T, int64_t Hq,
                            int64_t Hkv, int64_t D, int64_t cap, int64_t kv_len_max, int64_t n_split,
                            void* workspace, size_t workspace_bytes, void* stream) {
  using gdn_host::fail;
  if (D != 128 && D != 256) return fail(GDN_ERR_UNSUPPORTED, "gdn_attn_fwd: head dim must be 128 or 256 (got %lld)", (long long)D);
  if (B < 0 || T < 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || cap < T || cap > INT32_MAX || n_split < 1 ||
      n_split > 65535 || kv_len_max < T || kv_len_max > cap)
    return fail(GDN_ERR_INVALID, "gdn_attn_fwd: bad sizes (kv_len_max must lie in [T, cap])");
  if (!(scale > 0.0f)) return fail(GDN_ERR_INVALID, "gdn_attn_fwd: scale must be positive");
  if (B * T == 0) return GDN_OK;
  if (!q || !k_cache || !v_cache || !pos0 || !out) return fail(GDN_ERR_INVALID, "gdn_attn_fwd: null pointer");
  if (qg_ld == 0) qg_ld = 2 * Hq * D;
  if (qg && qg_ld < 2 * Hq * D) return fail(GDN_ERR_INVALID, "gdn_attn_fwd: gate token stride below the row");
  if (!gdn_host::aligned(q, 16) || !gdn_host::aligned(k_cache, 16) || !gdn_host::aligned(v_cache, 16) ||
      !gdn_host::aligned(out, 8) || (qg && (!gdn_host::aligned(qg, 8) || qg_ld % 4 != 0)))
    return fail(GDN_ERR_INVALID, "gdn_attn_fwd: misaligned pointer");
  const int rt = attn_rt(T, Hq, Hkv);
  const int64_t rows_pad = attn_rows_pad(T, Hq, Hkv, rt);
  const int64_t n_rb = rows_pad / (16 * rt);
  if (B > 65535 || Hkv * n_rb > INT32_MAX || B * Hkv * rows_pad * n_split * (D + 2) > (int64_t(1) << 40))
    return fail(GDN_ERR_UNSUPPORTED, "gdn_attn_fwd: problem too large");
  const size_t need = gdn_attn_workspace_bytes(B, T, Hq, Hkv, D, n_split);
  if (need > 0 && (workspace == nullptr || workspace_bytes < need || !gdn_host::aligned(workspace, 16)))
    return fail(GDN_ERR_INVALID, "gdn_attn_fwd: workspace of %zu bytes is below the %zu needed for %lld splits",
                workspace_bytes, need, (long long)n_split);
  AttnParams p;
  p.q = static_cast<const uint16_t*>(q);
  p.qg = static_cast<const uint16_t*>(qg);
  p.qg_ld = qg_ld;
  p.kc = static_cast<const uint16_t*>(k_cache);
  p.vc = static_cast<const uint16_t*>(v_cache);
  p.pos0 = pos0;
  p.out = static_cast<uint16_t*>(out);
  p.part = static_cast<float*>(workspace);
  p.B = static_cast<int>(B);
  p.T = static_cast<int>(T);
  p.Hq = static_cast<int>(Hq);
  p.Hkv = static_cast<int>(Hkv);
  p.cap = static_cast<int>(cap);
  p.n_split = static_cast<int>(n_split);
  p.split_len = static_cast<int>(((kv_len_max + n_split - 1) / n_split + KB - 1) / KB * KB);
  p.rows_pad = static_cast<int>(rows_pad);
  p.scale_log2 = scale * kLog2e;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (T * (Hq / Hkv) >= kPrefillRows) {
    const int64_t n_prb = (T * (Hq / Hkv) + PR - 1) / PR;
    if (Hkv * n_prb > INT32_MAX) return fail(GDN_ERR_UNSUPPORTED, "gdn_attn_fwd: problem too large");
    const dim3 pgrid(static_cast<unsigned>(Hkv * n_prb), static_cast<unsigned>(n_split), static_cast<unsigned>(B));
    if (D == 256) hipLaunchKernelGGL((attn_prefill_kernel<256, 2>), pgrid, dim3(512), 0, st, p);
    else hipLaunchKernelGGL((attn_prefill_kernel<128, 1>), pgrid, dim3(256), 0, st, p);
  } else if (const dim3 grid(static_cast<unsigned>(n_split), static_cast<unsigned>(Hkv * n_rb), static_cast<unsigned>(B));
             D == 256) {
    if (rt == 4) hipLaunchKernelGGL((attn_fwd_kernel<256, 4>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((attn_fwd_kernel<256, 1>), grid, dim3(256), 0, st, p);
  } else {
    if (rt == 4) hipLaunchKernelGGL((attn_fwd_kernel<128, 4>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((attn_fwd_kernel<128, 1>), grid, dim3(256), 0, st, p);
  }
  int rc = gdn_host::check_launch("gdn_attn_fwd");
  if (rc != GDN_OK || n_split == 1) return rc;
  const int64_t waves = B * Hkv * T * (Hq / Hkv);
  const dim3 cgrid(static_cast<unsigned>((waves + 3) / 4));
  if (D == 256) hipLaunchKernelGGL(attn_combine_kernel<256>, cgrid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL(attn_combine_kernel<128>, cgrid, dim3(256), 0, st, p);
  return gdn_host::check_launch("gdn_attn_fwd/combine");
}

extern "C" int gdn_rms_norm(const void* x, const void* res, void* h_out, const void* w, int w_dtype, void* y,
                            int64_t y_ld, int64_t rows, int64_t D, float eps, void* stream) {
  using gdn_host::fail;
  if (rows < 0 || D <= 0 || D % 8 != 0 || D > INT32_MAX || rows > INT32_MAX)
    return fail(GDN_ERR_INVALID, "gdn_rms_norm: bad sizes (D must be a multiple of 8)");
  if (y_ld == 0) y_ld = D;
  if (y_ld < D || y_ld % 8 != 0) return fail(GDN_ERR_INVALID, "gdn_rms_norm: y row stride must be >= D and a multiple of 8");
  if (!gdn_host::dtype_ok(w_dtype) || !(eps >= 0.0f)) return fail(GDN_ERR_INVALID, "gdn_rms_norm: bad weight dtype or eps");
  if (rows == 0) return GDN_OK;
  if (!x || !w || !y) return fail(GDN_ERR_INVALID, "gdn_rms_norm: null pointer");
  if (!gdn_host::aligned(x, 16) || !gdn_host::aligned(y, 16) || !gdn_host::aligned(w, 16) ||
      (res && !gdn_host::aligned(res, 16)) || (h_out && !gdn_host::aligned(h_out, 16)))
    return fail(GDN_ERR_INVALID, "gdn_rms_norm: misaligned pointer");
  hipLaunchKernelGGL(rms_norm_kernel, dim3(static_cast<unsigned>(rows)), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(res), static_cast<uint16_t*>(h_out),
                     w, w_dtype, static_cast<uint16_t*>(y), y_ld, static_cast<int>(D), eps);
  return gdn_host::check_launch("gdn_rms_norm");
}

extern "C" int gdn_pos_add(int32_t* pos, int64_t B, int32_t delta, int32_t lo, void* stream) {
  using gdn_host::fail;
  if (B < 0 || B > INT32_MAX) return fail(GDN_ERR_INVALID, "gdn_pos_add: bad sizes");
  if (B == 0) return GDN_OK;
  if (!pos) return fail(GDN_ERR_INVALID, "gdn_pos_add: null pointer");
  hipLaunchKernelGGL(pos_add_kernel, dim3(static_cast<unsigned>((B + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), pos, static_cast<int>(B), delta, lo);
  return gdn_host::check_launch("gdn_pos_add");
}

extern "C" int gdn_silu_mul(const void* gate_up, void* out, int64_t rows, int64_t I, void* stream) {
  using gdn_host::fail;
  if (rows < 0 || I <= 0 || I % 8 != 0 || I > INT32_MAX) return fail(GDN_ERR_INVALID, "gdn_silu_mul: bad sizes (I must be a multiple of 8)");
  if (rows == 0) return GDN_OK;
  if (!gate_up || !out) return fail(GDN_ERR_INVALID, "gdn_silu_mul: null pointer");
  if (!gdn_host::aligned(gate_up, 16) || !gdn_host::aligned(out, 16)) return fail(GDN_ERR_INVALID, "gdn_silu_mul: misaligned pointer");
  const int64_t n8 = rows * I / 8;
  if ((n8 + 255) / 256 > INT32_MAX) return fail(GDN_ERR_UNSUPPORTED, "gdn_silu_mul: problem too large");
  hipLaunchKernelGGL(silu_mul_kernel, dim3(static_cast<unsigned>((n8 + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(gate_up), static_cast<uint16_t*>(out),
                     rows, static_cast<int>(I));
  return gdn_host::check_launch("gdn_silu_mul");
}
