// Block-sparse attention forward for fp32 inputs
// (ops/flashprefill_native_forward.py:227-344,
//  ops/flashprefill_varlen_func.py:449-575, run with fp32 q / k / v).
//
// One workgroup (BLK / 32 waves) owns one (query head, sequence, q-block) row,
// or one chunk of a row's list, in the "one query per lane" orientation of
// k_attn. The fp32 products are formed on the bf16 matrix units, which run 16
// times as fast as the fp32 ones: every fp32 value is the exact sum of three
// bf16 parts (8 + 8 + 8 significand bits), x = x1 + x2 + x3, each rounded to
// nearest (|x2| <= 2^-8 |x|, |x3| <= 2^-17 |x|), and
//
//   x y = x1 y1 + (x1 y2 + x2 y1) + (x1 y3 + x2 y2 + x3 y1) + rest,
//   |rest| <= 2^-24 |x y|, one rounding of an fp32 product, of either sign (about
//   2^-27 on average; with x1 truncated instead, 2^-22 and 2^-25),
//
// i.e. six v_mfma_f32_32x32x16_bf16 (192 cycles) per 16 steps of the sum in
// place of eight v_mfma_f32_32x32x2_f32 (512 cycles), with fp32 accumulation
// and fewer roundings of the running sum (6 instead of 8 per 16 terms). Against
// float64 the outputs are no further off than with the fp32 units (2-norm error
// 1.2e-6, there 1.7e-6, on structured 4K inputs).
//
//   S^T = K . Q^T    A = K parts from LDS, B = Q^T parts in registers
//   O^T += V^T . P^T A = V^T parts via ds_read_b64_tr_b16 from the key-major
//                    tile, B = P^T parts split from the S^T accumulators (P
//                    itself stays fp32: its three parts add up to it)
//
// K and V come in tiles of KT keys: loaded to registers one tile ahead, split
// on the way into LDS (one K and one V buffer, 48 KB in all, so that two
// workgroups share a CU and one's splitting and softmax runs beside the
// other's MFMAs), in the swizzled layout of k_attn (conflict free).
//
// Values of 2^56 or more, infinities and NaN do not go through the split
// (x - x1 of an infinity is NaN, and part products could overflow where the
// value's own product does not): a workgroup that meets one among its queries
// or in a tile forms its row (chunk) again with scalar fp32 FMAs at the end.
//
// Numerics follow the reference loop: m starts at -inf and l at 1.0, alpha =
// exp2(m_old - m_new) with NaN -> 1, l = l * alpha + sum p, acc = acc * alpha +
// p . V with p kept in fp32, the diagonal block masks key > query, O = acc / l;
// the tile of the online softmax is KT keys, not the whole block, a
// rounding-level difference. Rows past the sequence end (only in the diagonal
// block, where they are masked) repeat the last row.
//
// Few rows leave the card idle behind the longest one (4K tokens x 8 heads:
// 256 rows of 1 .. 32 blocks on 256 CUs), so launch_attn_f32's caller may give
// every row several chunk slots (AttnArgs::f32_chunks): chunk c takes list
// entries c * f32_chunk_blocks .. of its row, rows of more than one chunk leave
// fp32 partials that k_merge_f32 combines.
//
// Measured (one MI355X), attention alone, against the fp32 units with tiles
// staged between two barriers and one workgroup per row: 4K x 8 q / 2 kv heads,
// d = 64: 315 -> 94 us; the same at d = 128: 630 -> 202; 4K x 32 q / 8 kv heads,
// d = 128: 824 -> 465 us; 8K x 32 heads, d = 64: 1,068 -> 526 us. (Scaling V and P and
// rounding the first parts cost 1 - 3 % of it.) The bf16 units are ~40 % busy
// there: the scaling, splitting, softmax and conversion instructions of a tile
// (~700) take about as long as its 96 MFMAs and two waves per SIMD overlap them
// only in part.
#include "fp_attn_common.h"

namespace fp {

// P and V are split 2^24 times their size: the third part of the smallest fp32
// value is then a normal bf16 value (unscaled, it runs into bf16's last step,
// 2^-133, from 2^-110 on down), and O^T comes out 2^48 times its size. Q and K are
// split as they are: a K below 2^-110 has scores below 2^-47 beside any Q that goes
// through the split, which exp2 does not see.
constexpr float kSplitScale = 16777216.0f;
constexpr float kUnscale = 1.0f / (kSplitScale * kSplitScale);
// |x| from which a value does not go through the split
constexpr float kSplitMax = 7.2057594e16f;  // 2^56

// x0, x1 (times `scale`) -> their three bf16 parts, packed in pairs
__device__ __forceinline__ void split_pair(float x0, float x1, float scale, uint32_t& a,
                                           uint32_t& b, uint32_t& c) {
  x0 *= scale;
  x1 *= scale;
  a = pack2<BF16>(x0, x1);
  const float r0 = x0 - __uint_as_float(a << 16), r1 = x1 - __uint_as_float(a & 0xffff0000u);
  b = pack2<BF16>(r0, r1);
  c = pack2<BF16>(r0 - __uint_as_float(b << 16), r1 - __uint_as_float(b & 0xffff0000u));
}

// acc += A . B over one 16-step with both operands in three parts, the small
// products first
__device__ __forceinline__ f32x16 mfma_split(const bf16x8 (&x)[3], const bf16x8 (&y)[3],
                                             f32x16 acc) {
  acc = BF16::mfma32(x[2], y[0], acc);
  acc = BF16::mfma32(x[0], y[2], acc);
  acc = BF16::mfma32(x[1], y[1], acc);
  acc = BF16::mfma32(x[1], y[0], acc);
  acc = BF16::mfma32(x[0], y[1], acc);
  return BF16::mfma32(x[0], y[0], acc);
}

// keys per tile: two tiles of 3 x KT x D bf16 are 48 KB
template <int D>
constexpr int f32_tile_keys() { return D == 64 ? 64 : 32; }

template <int D, int BLK>
__global__ __launch_bounds__(2 * BLK, BLK == 128 ? 2 : 1) void k_attn_f32(AttnArgs a) {
  constexpr int NT = 2 * BLK;       // threads
  constexpr int KT = f32_tile_keys<D>();
  constexpr int TT = KT / 32;       // 32-key tiles of S^T per LDS tile
  constexpr int NSUB = BLK / KT;    // LDS tiles per block
  constexpr int KS = D / 16;        // MFMA k-steps over the head dim
  constexpr int DT = D / 32;        // 32-dim tiles of O^T
  constexpr int CH = D / 8;         // 16-byte chunks of a part's row
  constexpr int PC = KT * CH / NT;  // chunks per thread and tensor
  static_assert(KT * CH % NT == 0 && BLK % KT == 0, "whole tiles");
  __shared__ uint4 sk[3][KT * CH];
  __shared__ uint4 sv[3][KT * CH];
  __shared__ int s_big;

  // every row has f32_chunks slots, chunk index outermost (heaviest rows first
  // within each)
  const int64_t rows = a.total_slots / a.f32_chunks;
  const int chunk = static_cast<int>(blockIdx.x / rows);
  const int64_t nitems = sld(a.tab.seq_tile + a.B);
  int item, h;
  map_row(static_cast<int>(blockIdx.x % rows), a.Hq, a.Hkv, a.nb_sum_cap, item, h);
  if (item >= nitems) return;
  const ItemRec rec = sld(a.tab.items + item);
  const int i = rec.i, L = rec.L;
  const int64_t t0 = rec.t0;
  const int64_t row_tri = static_cast<int64_t>(h) * a.tri_cap + rec.tri;
  const int64_t row = static_cast<int64_t>(h) * a.nb_sum_cap + rec.tile;
  const int nsel = min(max(sld(a.cnt + row), 0), i + 1);
  const int n0 = chunk * a.f32_chunk_blocks;
  if (chunk > 0 && n0 >= nsel) return;
  const bool split = a.f32_chunks > 1 && nsel > a.f32_chunk_blocks;
  const int ncnt = split ? min(a.f32_chunk_blocks, nsel - n0) : nsel;
  const int32_t* list = a.idx + row_tri + n0;
  const int kvh = h / (a.Hq / a.Hkv);

  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  const int qrow = 32 * w + l32;
  const int qg = i * BLK + qrow;
  const bool qvalid = qg < L;
  const float c = a.sm_scale_log2;
  const float* q = reinterpret_cast<const float*>(a.q);
  const float* kbase = reinterpret_cast<const float*>(a.k) + t0 * a.kst + kvh * a.khs;
  const float* vbase = reinterpret_cast<const float*>(a.v) + t0 * a.vst + kvh * a.vhs;
  const float* qptr = q + (t0 + (qvalid ? qg : 0)) * a.qst + h * a.qhs;

  // tile it of the walk: keys KT (it % NSUB) .. of block list[it / NSUB];
  // thread t holds chunks t, t + NT, ... (8 dims of a key) of K and V
  float4 kf[PC][2], vf[PC][2];
  auto block_of = [&](int it) { return min(max(sld(list + it / NSUB), 0), i); };
  // the lane part of an address is a 32-bit offset (rows t / CH of the tile),
  // the rest wave-uniform
  const uint32_t koff = static_cast<uint32_t>((t / CH) * static_cast<int>(a.kst) + 8 * (t % CH));
  const uint32_t voff = static_cast<uint32_t>((t / CH) * static_cast<int>(a.vst) + 8 * (t % CH));
  auto load_tile = [&](int it) {
    const int key0 = block_of(it) * BLK + (it % NSUB) * KT;
    if (key0 + KT <= L) {
#pragma unroll
      for (int p = 0; p < PC; ++p) {
        const float* kp = kbase + static_cast<int64_t>(key0 + p * (NT / CH)) * a.kst;
        const float* vp = vbase + static_cast<int64_t>(key0 + p * (NT / CH)) * a.vst;
        kf[p][0] = *reinterpret_cast<const float4*>(kp + koff);
        kf[p][1] = *reinterpret_cast<const float4*>(kp + koff + 4);
        vf[p][0] = *reinterpret_cast<const float4*>(vp + voff);
        vf[p][1] = *reinterpret_cast<const float4*>(vp + voff + 4);
      }
    } else {  // rows past the end repeat the last one
#pragma unroll
      for (int p = 0; p < PC; ++p) {
        const int64_t gk = min(key0 + t / CH + p * (NT / CH), L - 1);
        const float* kp = kbase + gk * a.kst + 8 * (t % CH);
        const float* vp = vbase + gk * a.vst + 8 * (t % CH);
        kf[p][0] = *reinterpret_cast<const float4*>(kp);
        kf[p][1] = *reinterpret_cast<const float4*>(kp + 4);
        vf[p][0] = *reinterpret_cast<const float4*>(vp);
        vf[p][1] = *reinterpret_cast<const float4*>(vp + 4);
      }
    }
  };
  auto big4 = [](float m, const float4& x) {
    return fmaxf(fmaxf(fmaxf(m, fabsf(x.x)), fmaxf(fabsf(x.y), fabsf(x.z))), fabsf(x.w));
  };
  auto store_split = [&](uint4 (&dst)[3][KT * CH], const float4 (&x)[PC][2], float scale) {
#pragma unroll
    for (int p = 0; p < PC; ++p) {
      const int cidx = t + p * NT;
      const int r = cidx / CH;
      uint32_t u[3][4];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        split_pair(x[p][e].x, x[p][e].y, scale, u[0][2 * e], u[1][2 * e], u[2][2 * e]);
        split_pair(x[p][e].z, x[p][e].w, scale, u[0][2 * e + 1], u[1][2 * e + 1],
                   u[2][2 * e + 1]);
      }
      const int at = r * CH + ((cidx % CH) ^ swz<D>(r));
#pragma unroll
      for (int s = 0; s < 3; ++s) dst[s][at] = make_uint4(u[s][0], u[s][1], u[s][2], u[s][3]);
    }
  };

  const int ntiles = ncnt * NSUB;
  if (ntiles > 0) load_tile(0);

  // Q^T parts as MFMA B operands: lane's query, dims 16 s + 8 half .. +7
  bf16x8 qb[KS][3];
  float qmax = 0.0f;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    float4 x[2] = {make_float4(0.f, 0.f, 0.f, 0.f), make_float4(0.f, 0.f, 0.f, 0.f)};
    if (qvalid) {
      x[0] = *reinterpret_cast<const float4*>(qptr + 16 * s + 8 * half);
      x[1] = *reinterpret_cast<const float4*>(qptr + 16 * s + 8 * half + 4);
    }
    qmax = big4(big4(qmax, x[0]), x[1]);
    uint32_t u[3][4];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      split_pair(x[e].x, x[e].y, 1.0f, u[0][2 * e], u[1][2 * e], u[2][2 * e]);
      split_pair(x[e].z, x[e].w, 1.0f, u[0][2 * e + 1], u[1][2 * e + 1], u[2][2 * e + 1]);
    }
#pragma unroll
    for (int p = 0; p < 3; ++p)
      qb[s][p] = as_vec8<BF16>(make_uint4(u[p][0], u[p][1], u[p][2], u[p][3]));
  }

  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = f32x16{};
  float m_run = -INFINITY;
  // the two halves' partial sums add up to l: a row starts from the
  // reference's l = 1.0, a chunk of a split row from 0
  float l_part = half == 0 && !split ? 1.0f : 0.0f;
  const int g16 = lane >> 4, i16 = lane & 15;
  const int tr_row = 4 * (g16 >> 1) + (i16 >> 2);
  const int tr_col = 16 * (g16 & 1) + 4 * (i16 & 3);

  if (t == 0) s_big = 0;
  for (int it = 0; it < ntiles; ++it) {
    __syncthreads();  // every wave is done with the previous tile
    float mx = qmax;
#pragma unroll
    for (int p = 0; p < PC; ++p)
      mx = big4(big4(big4(big4(mx, kf[p][0]), kf[p][1]), vf[p][0]), vf[p][1]);
    store_split(sk, kf, 1.0f);
    store_split(sv, vf, kSplitScale);
    if (mx >= kSplitMax) s_big = 1;  // (a NaN alone goes through the split as it is)
    if (it + 1 < ntiles) load_tile(it + 1);  // flies during this tile's products
    // the LDS stores are done; the register loads may still be in flight
    lds_barrier();
    const int j = block_of(it), sub = it % NSUB;
    const bool diag = j == i;
    // 32-key tiles 0 .. live - 1 of this LDS tile are visible to the wave
    const int live = diag ? min(max(w + 1 - sub * TT, 0), TT) : TT;
    if (live == 0) continue;

    f32x16 s[TT];
#pragma unroll
    for (int t4 = 0; t4 < TT; ++t4) s[t4] = f32x16{};
    // one 16-dim step of one 32-key tile's scores: three K part reads, six MFMAs
    auto s_step = [&](int t4, int ks) {
      const int r = 32 * t4 + l32;
      const int at = r * CH + ((2 * ks + half) ^ swz<D>(r));
      const bf16x8 kp[3] = {as_vec8<BF16>(sk[0][at]), as_vec8<BF16>(sk[1][at]),
                            as_vec8<BF16>(sk[2][at])};
      s[t4] = mfma_split(kp, qb[ks], s[t4]);
    };
    if (live == TT) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int t4 = 0; t4 < TT; ++t4) s_step(t4, ks);
      // the part reads run one step (six MFMAs) ahead of their use
      __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 3, 0);
#pragma unroll
      for (int k = 0; k < KS * TT - 1; ++k) {
        __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 3, 0);
        __builtin_amdgcn_sched_group_barrier(kSchedMfma, 6, 0);
      }
      __builtin_amdgcn_sched_group_barrier(kSchedMfma, 6, 0);
    } else {
#pragma unroll
      for (int t4 = 0; t4 < TT; ++t4) {
        if (t4 >= live) continue;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) s_step(t4, ks);
      }
    }
    if (diag) {  // key > query is masked
#pragma unroll
      for (int t4 = 0; t4 < TT; ++t4)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int key = sub * KT + 32 * t4 + 8 * (v >> 2) + 4 * half + (v & 3);
          if (key > qrow) s[t4][v] = -INFINITY;
        }
    }
    // online softmax over this tile (base 2, scores scaled by c)
    float smax = -INFINITY;
#pragma unroll
    for (int t4 = 0; t4 < TT; ++t4)
#pragma unroll
      for (int v = 0; v < 16; ++v) smax = fmaxf(smax, s[t4][v]);
    const float m_new = fmaxf(m_run, pair32_max(smax) * c);
    // the factor is 1 for every lane once the maximum has settled (NaN, from
    // -inf - -inf, counts as 1 as in the reference)
    if (__ballot(m_new != m_run) != 0) {
      float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      if (alpha != alpha) alpha = 1.0f;
      m_run = m_new;
      l_part *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[dt][v] *= alpha;
    }
    float psum = 0.0f;
#pragma unroll
    for (int t4 = 0; t4 < TT; ++t4)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        s[t4][v] = __builtin_amdgcn_exp2f(fmaf(s[t4][v], c, -m_new));
        psum += s[t4][v];
      }
    l_part += psum;

    // O^T += V^T . P^T: B element e of lane (query, half) in 16-key step hh of
    // tile t4 is key 16 hh + (e < 4 ? 4 half + e : 8 + 4 half + e - 4), i.e.
    // accumulator elements 8 hh .. 8 hh + 7
    {
      // one 16-key step: P split into its parts, then per 32 dims six V^T part
      // reads and six MFMAs
      auto pv_step = [&](int t4, int hh) {
        uint32_t u[3][4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          split_pair(s[t4][8 * hh + 2 * e], s[t4][8 * hh + 2 * e + 1], kSplitScale, u[0][e],
                     u[1][e], u[2][e]);
        bf16x8 pb[3];
#pragma unroll
        for (int p = 0; p < 3; ++p)
          pb[p] = as_vec8<BF16>(make_uint4(u[p][0], u[p][1], u[p][2], u[p][3]));
        const int r1 = 32 * t4 + 16 * hh + tr_row;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const int x = 32 * dt + tr_col;
          bf16x8 va[3];
#pragma unroll
          for (int p = 0; p < 3; ++p) {
            const uint16_t* svp = reinterpret_cast<const uint16_t*>(sv[p]);
            const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) i16x4*)(svp + tile_elem<D>(r1, x)));
            const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) i16x4*)(svp + tile_elem<D>(r1 + 8, x)));
            const uint2 lo2 = __builtin_bit_cast(uint2, lo), hi2 = __builtin_bit_cast(uint2, hi);
            va[p] = as_vec8<BF16>(make_uint4(lo2.x, lo2.y, hi2.x, hi2.y));
          }
          o[dt] = mfma_split(va, pb, o[dt]);
        }
      };
      if (live == TT) {
#pragma unroll
        for (int t4 = 0; t4 < TT; ++t4)
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) pv_step(t4, hh);
        __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 6, 0);
#pragma unroll
        for (int k = 0; k < 2 * TT * DT - 1; ++k) {
          __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 6, 0);
          __builtin_amdgcn_sched_group_barrier(kSchedMfma, 6, 0);
        }
        __builtin_amdgcn_sched_group_barrier(kSchedMfma, 6, 0);
      } else {
#pragma unroll
        for (int t4 = 0; t4 < TT; ++t4) {
          if (t4 >= live) continue;
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) pv_step(t4, hh);
        }
      }
    }
  }

  // Values that the split does not take: the row again, with scalar products
  // (32 keys at a time; accumulator element v of a tile is key 8 (v / 4) +
  // 4 half + v % 4, o[dt][x] is dim 32 dt + 8 (x / 4) + 4 half + x % 4). The
  // maximum of the whole row comes first, also for a chunk of it, so that no sum of
  // P V is larger on the way than in the result.
  __syncthreads();
  if (s_big != 0) {
    // scores of tile `it` of the walk over `blocks`
    auto scores = [&](const int32_t* blocks, int it, f32x16& s) {
      const int j = min(max(sld(blocks + it / (BLK / 32)), 0), i);
      const int key0 = 32 * (it % (BLK / 32));
      s = f32x16{};
#pragma unroll 1
      for (int d = 0; d < D; ++d) {
        const float qd = qvalid ? qptr[d] : 0.0f;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int key = key0 + 8 * (v >> 2) + 4 * half + (v & 3);
          s[v] = fmaf(qd, kbase[static_cast<int64_t>(min(j * BLK + key, L - 1)) * a.kst + d], s[v]);
        }
      }
#pragma unroll
      for (int v = 0; v < 16; ++v)
        if (j == i && key0 + 8 * (v >> 2) + 4 * half + (v & 3) > qrow) s[v] = -INFINITY;
    };
    m_run = -INFINITY;
    l_part = 0.0f;
#pragma unroll 1
    for (int it = 0; it < nsel * (BLK / 32); ++it) {
      f32x16 s;
      scores(a.idx + row_tri, it, s);
      float smax = -INFINITY;
#pragma unroll
      for (int v = 0; v < 16; ++v) smax = fmaxf(smax, s[v]);
      m_run = fmaxf(m_run, pair32_max(smax) * c);
      // scores of -inf are P = 0, but NaN (-inf - -inf, as in the reference, whose
      // tile is the block) where they fill a row's first block
      if (chunk == 0 && it == BLK / 32 - 1 && m_run == -INFINITY)
        l_part = __uint_as_float(0x7fc00000u);
    }
    const float ms = m_run == -INFINITY ? 0.0f : m_run;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = f32x16{};
#pragma unroll 1
    for (int it = 0; it < ncnt * (BLK / 32); ++it) {
      const int key0 = min(max(sld(list + it / (BLK / 32)), 0), i) * BLK + 32 * (it % (BLK / 32));
      f32x16 s;
      scores(list, it, s);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        s[v] = __builtin_amdgcn_exp2f(fmaf(s[v], c, -ms));
        l_part += s[v];
        // the other half-wave holds the P of the key 4 apart
        const float other = __uint_as_float(xchg32(__float_as_uint(s[v])));
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          const int key = key0 + 8 * (v >> 2) + 4 * hh + (v & 3);
          const float p = hh == half ? s[v] : other;
          const float* vp = vbase + static_cast<int64_t>(min(key, L - 1)) * a.vst + 4 * half;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
              const float4 y = *reinterpret_cast<const float4*>(vp + 32 * dt + 8 * g4);
              o[dt][4 * g4] = fmaf(p, y.x, o[dt][4 * g4]);
              o[dt][4 * g4 + 1] = fmaf(p, y.y, o[dt][4 * g4 + 1]);
              o[dt][4 * g4 + 2] = fmaf(p, y.z, o[dt][4 * g4 + 2]);
              o[dt][4 * g4 + 3] = fmaf(p, y.w, o[dt][4 * g4 + 3]);
            }
        }
      }
    }
  }

  const float l = pair32_sum(l_part);
  const float unscale = s_big != 0 ? 1.0f : kUnscale;
  if (split) {
    // chunk of a row: unnormalised O^T [BLK][D], then m [BLK], l [BLK]
    float* pp = a.part + (row * a.f32_chunks + chunk) * static_cast<int64_t>(BLK * D + 2 * BLK);
    float* orow = pp + static_cast<int64_t>(qrow) * D;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4)
        *reinterpret_cast<float4*>(orow + 32 * dt + 8 * g4 + 4 * half) =
            make_float4(o[dt][4 * g4] * unscale, o[dt][4 * g4 + 1] * unscale,
                        o[dt][4 * g4 + 2] * unscale, o[dt][4 * g4 + 3] * unscale);
    if (half == 0) {
      pp[BLK * D + qrow] = m_run;
      pp[BLK * D + BLK + qrow] = l;
    }
    return;
  }
  const float rcp = unscale / l;
  if (qvalid) {
    float* op = reinterpret_cast<float*>(a.o) + (t0 + qg) * a.ost + h * a.ohs;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4)
        *reinterpret_cast<float4*>(op + 32 * dt + 8 * g4 + 4 * half) =
            make_float4(o[dt][4 * g4] * rcp, o[dt][4 * g4 + 1] * rcp, o[dt][4 * g4 + 2] * rcp,
                        o[dt][4 * g4 + 3] * rcp);
  }
}

// Output rows of the rows of more than one chunk: m = max_c m_c, w_c =
// exp2(m_c - m), O = sum_c w_c acc_c / sum_c w_c l_c, chunks in order. One
// workgroup per (row, 32 of its queries), eight threads per query.
template <int D, int BLK>
__global__ __launch_bounds__(256) void k_merge_f32(AttnArgs a) {
  constexpr int XT = D / 8;  // dims per thread
  constexpr int64_t S = BLK * D + 2 * BLK;
  const int64_t slot = blockIdx.x / (BLK / 32);
  const int h = static_cast<int>(slot % a.Hq);
  const int64_t item = slot / a.Hq;
  if (item >= sld(a.tab.seq_tile + a.B)) return;
  const ItemRec rec = sld(a.tab.items + item);
  const int64_t row = static_cast<int64_t>(h) * a.nb_sum_cap + rec.tile;
  const int nsel = min(max(sld(a.cnt + row), 0), rec.i + 1);
  const int nc = min((nsel + a.f32_chunk_blocks - 1) / a.f32_chunk_blocks, a.f32_chunks);
  if (nc <= 1) return;
  const int r = 32 * static_cast<int>(blockIdx.x % (BLK / 32)) + static_cast<int>(threadIdx.x >> 3);
  const int qg = rec.i * BLK + r;
  if (qg >= rec.L) return;
  const int x0 = XT * static_cast<int>(threadIdx.x & 7);
  const float* p0 = a.part + row * a.f32_chunks * S;
  float mc[kF32MaxChunks], m = -INFINITY, lsum = 0.0f;
#pragma unroll
  for (int k = 0; k < kF32MaxChunks; ++k) {
    mc[k] = k < nc ? p0[k * S + BLK * D + r] : -INFINITY;
    m = fmaxf(m, mc[k]);
  }
  float4 acc[XT / 4];
#pragma unroll
  for (int e = 0; e < XT / 4; ++e) acc[e] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int k = 0; k < kF32MaxChunks; ++k) {
    if (k >= nc) break;
    const float wc = __builtin_amdgcn_exp2f(mc[k] - m);
    lsum += wc * p0[k * S + BLK * D + BLK + r];
#pragma unroll
    for (int e = 0; e < XT / 4; ++e) {
      const float4 y =
          *reinterpret_cast<const float4*>(p0 + k * S + static_cast<int64_t>(r) * D + x0 + 4 * e);
      acc[e].x += wc * y.x;
      acc[e].y += wc * y.y;
      acc[e].z += wc * y.z;
      acc[e].w += wc * y.w;
    }
  }
  const float rcp = 1.0f / lsum;
  float* op = reinterpret_cast<float*>(a.o) + (rec.t0 + qg) * a.ost + h * a.ohs + x0;
#pragma unroll
  for (int e = 0; e < XT / 4; ++e)
    *reinterpret_cast<float4*>(op + 4 * e) =
        make_float4(acc[e].x * rcp, acc[e].y * rcp, acc[e].z * rcp, acc[e].w * rcp);
}

template <int D, int BLK>
hipError_t launch_attn_f32_t(const AttnArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((k_attn_f32<D, BLK>), dim3(static_cast<unsigned>(a.total_slots)),
                     dim3(2 * BLK), 0, s, a);
  if (a.f32_chunks > 1)
    hipLaunchKernelGGL((k_merge_f32<D, BLK>),
                       dim3(static_cast<unsigned>(a.Hq * a.nb_sum_cap * (BLK / 32))), dim3(256), 0,
                       s, a);
  return hipGetLastError();
}

hipError_t launch_attn_f32(const AttnArgs& a, int head_dim, int block, hipStream_t s) {
  if (a.total_slots <= 0) return hipSuccess;
  if (head_dim == 128)
    return block == 128 ? launch_attn_f32_t<128, 128>(a, s) : launch_attn_f32_t<128, 64>(a, s);
  return block == 128 ? launch_attn_f32_t<64, 128>(a, s) : launch_attn_f32_t<64, 64>(a, s);
}

}  // namespace fp
