// Attention over a paged KV cache: the decode step of the vLLM-style backend
// hook and the prefix-cached prefill of its v0 form (the role of vLLM's
// flash_attn_varlen_func with a block table in the reference's decode branch,
// patches/patch_loader_vllm_0_12_0.py:201-225, patch_loader_vllm_0_10_0.py:
// 270-368). Query row t of sequence b attends to the first
// used[b] - (cu[b + 1] - 1 - t) cached tokens.
//
// A decode step reads every cached key and value once for a handful of query
// rows: HBM-bound. k_paged gives a workgroup one (16-row tile of the G query
// heads of a KV head, KV head, chunk of keys); its four waves take 32 keys in
// turn, straight from the pages into registers (no LDS, no barrier in the
// loop), and merge at the end:
//
//   S^T (keys x rows)  = K . Q^T   v_mfma_f32_16x16x32 on the 16-bit operands;
//                        lane (row r = l % 16, group g = l / 16) then holds
//                        keys 4 g + v of each 16-key tile, v = 0 .. 3
//   O^T (dims x rows) += V^T . P^T v_mfma_f32_16x16x4_f32: k index g of step v
//                        is key 4 g + v, so P stays where it is, in fp32, and
//                        the V operand of MFMA e is element e of the 16-byte
//                        row piece that the lane loaded (dims 8 (l % 16) + e of
//                        key 4 g + v): each load instruction reads four whole
//                        256-byte rows and nothing is transposed
//
// P is never rounded to 16 bits and V converts exactly, so the sums are those
// of an fp32 product. The fp32 MFMAs of 32 keys take ~2,050 cycles per wave,
// a rate of ~18 TB/s over the card, i.e. they stay behind the loads.
//
// Chunks: the host cannot see the lengths without a synchronisation, so it
// fixes only the number of chunk slots (about 8192 workgroups over the card,
// at most 128 per row) and every workgroup derives the chunk length from the
// longest sequence (256 keys at least, whole rounds of 128); workgroups past
// their sequence's end return at once. Rows of one chunk are written out
// directly, the others as (O^T, m, l) partials that k_paged_merge combines.
//
// Measured (one MI355X, d = 128): 32 sequences of 300 .. 15,300 tokens (32 q /
// 8 kv heads, 0.9 GB of cache) 18.8 ms per call as per-sequence torch gathers
// and fp32 products, 0.22 ms here (k_paged 0.20 - 0.21 ms = 4.2 - 4.5 TB/s, where
// a 1 GiB copy reaches 5.24; k_paged_merge 6 us); one sequence of 65,000 tokens
// 6.57 -> 0.056 ms a call among others of its kind, 0.066 with inputs that change
// (127 chunks x 8 KV heads; k_paged 49 us = 5.4 TB/s, k_paged_merge 7).
#include "fp_attn_common.h"

namespace fp {

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(f16x8 a, f16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// entry x of a 32- or 64-bit integer array
__device__ __forceinline__ int64_t ld_int(const void* p, int is64, int64_t x) {
  return is64 ? static_cast<const int64_t*>(p)[x] : static_cast<const int32_t*>(p)[x];
}

// One sequence as the workgroups see it. `bad`: more tokens than the block
// table has room for; its rows are written as NaN. `off`: its query offsets
// descend or lie outside the call's rows.
struct PagedSeq {
  int64_t q0;  // first query row
  int nq;      // query rows
  int64_t nk;  // cached tokens
  bool bad, off;
};

__device__ __forceinline__ PagedSeq paged_seq(const PagedArgs& a, int b) {
  PagedSeq s;
  s.q0 = ld_int(a.cu, a.cu64, b);
  const int64_t q1 = ld_int(a.cu, a.cu64, b + 1);
  s.off = s.q0 < 0 || q1 > a.T || q1 < s.q0;
  s.nq = s.off ? 0 : static_cast<int>(q1 - s.q0);
  s.nk = ld_int(a.used, a.used64, b);
  s.bad = s.nk > static_cast<int64_t>(a.width) * a.bs;
  if (s.bad || s.nk < 0) s.nk = 0;
  return s;
}

__device__ __forceinline__ int64_t shfl64(int64_t x, int lane) {
  return static_cast<int64_t>(
      (static_cast<uint64_t>(static_cast<uint32_t>(__shfl(static_cast<int>(x >> 32), lane))) << 32) |
      static_cast<uint32_t>(__shfl(static_cast<int>(x), lane)));
}

// The sequence that owns row tile `x` (tiles of `rt` rows of nq * G, numbered
// over the sequences) and the tile's index in it, or with tok >= 0 the one
// that owns query row `tok`; and the chunk length all workgroups use. By one
// wave (64 sequences at a time); b < 0 when there is none. Where some sequence's
// offsets do not fit, which rows are whose is unknown: all rows of the call are
// one sequence's then, and bad.
struct PagedTile {
  PagedSeq s;
  int b, tl, chunk;
};
__device__ __forceinline__ PagedTile paged_find(const PagedArgs& a, int rt, int64_t x,
                                                int64_t tok) {
  const int lane = threadIdx.x & 63;
  PagedTile r;
  r.b = -1;
  r.tl = 0;
  r.s = PagedSeq{0, 0, 0, false, false};
  int64_t carry = 0;
  int maxlen = 0;
  bool off = false;
  for (int base = 0; base < a.B; base += 64) {
    PagedSeq s{0, 0, 0, false, false};
    if (base + lane < a.B) s = paged_seq(a, base + lane);
    off = off || __ballot(s.off) != 0;
    const int tiles =
        static_cast<int>((static_cast<int64_t>(s.nq) * a.G + rt - 1) / rt);
    if (s.nq > 0) maxlen = max(maxlen, static_cast<int>(s.nk));
    int incl = tiles;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(incl, o);
      if (lane >= o) incl += y;
    }
    const bool mine = tok >= 0 ? tok >= s.q0 && tok < s.q0 + s.nq
                               : tiles > 0 && x >= carry + incl - tiles && x < carry + incl;
    const uint64_t hit = __ballot(mine);
    if (r.b < 0 && hit) {
      const int l = __ffsll(static_cast<long long>(hit)) - 1;
      r.b = base + l;
      r.tl = static_cast<int>(x - carry) - __shfl(incl - tiles, l);
      r.s.q0 = shfl64(s.q0, l);
      r.s.nq = __shfl(s.nq, l);
      r.s.nk = shfl64(s.nk, l);
      r.s.bad = __shfl(static_cast<int>(s.bad), l) != 0;
    }
    carry += __shfl(incl, 63);
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) maxlen = max(maxlen, __shfl_xor(maxlen, o));
  const int per = (maxlen + a.nc - 1) / a.nc;
  r.chunk = (max(per, kPagedMinChunk) + 127) / 128 * 128;
  if (off) {
    r.b = tok >= 0 || x < (a.T * a.G + rt - 1) / rt ? 0 : -1;
    r.tl = static_cast<int>(x);
    r.s = PagedSeq{0, static_cast<int>(a.T), 0, true, true};
  }
  // wave-uniform values in scalar registers
  r.b = __builtin_amdgcn_readfirstlane(r.b);
  r.tl = __builtin_amdgcn_readfirstlane(r.tl);
  r.chunk = __builtin_amdgcn_readfirstlane(r.chunk);
  r.s.nq = __builtin_amdgcn_readfirstlane(r.s.nq);
  r.s.nk = __builtin_amdgcn_readfirstlane(static_cast<int>(r.s.nk));
  r.s.q0 = __builtin_amdgcn_readfirstlane(static_cast<int>(r.s.q0));
  return r;
}

// Page of cached token `key` of a sequence whose table row is `row`. A page
// number below 0 counts from the end (as the index of a torch gather); one
// outside the cache sets `bad` and reads page 0.
// UNI: `key` is wave-uniform and the lookup goes through the scalar cache (a
// vector load would wait for every K / V load issued before it).
template <bool UNI>
__device__ __forceinline__ int64_t paged_page(const PagedArgs& a, int64_t row, int key, bool& bad) {
  int idx = a.bs_shift >= 0 ? key >> a.bs_shift : key / a.bs;
  int64_t p;
  if constexpr (UNI) {
    idx = __builtin_amdgcn_readfirstlane(idx);
    p = a.table64 ? sld(static_cast<const int64_t*>(a.table) + row + idx)
                  : static_cast<int64_t>(sld(static_cast<const int32_t*>(a.table) + row + idx));
  } else {
    p = ld_int(a.table, a.table64, row + idx);
  }
  if (p < 0) p += a.nblocks;
  if (p < 0 || p >= a.nblocks) {
    bad = true;
    p = 0;
  }
  return p;
}

// max / sum over the lanes l, l ^ 16, l ^ 32, l ^ 48 (one query row), in every lane
__device__ __forceinline__ float row4_max(float x) {
  x = fmaxf(x, __uint_as_float(xchg_xor<16>(__float_as_uint(x))));
  return pair32_max(x);
}
__device__ __forceinline__ float row4_sum(float x) {
  x += __uint_as_float(xchg_xor<16>(__float_as_uint(x)));
  return pair32_sum(x);
}

// P16: the page size is a multiple of 16, so a 16-key tile lies in one page
// (one scalar page lookup and wave-uniform bases); otherwise every lane looks
// up its own key's page.
template <typename T, int D, bool P16>
__global__ __launch_bounds__(256, D > 128 ? 2 : 3) void k_paged(PagedArgs a) {
  constexpr int KS = D / 32;             // MFMA k-steps over the head dim
  constexpr int E = D / 16;              // V elements per lane and key
  constexpr int VW = E / 2;              // the same in 32-bit words
  constexpr int OS = D + 4;              // padded row of the merge buffer (floats)
  __shared__ float sm[4][16][OS];
  __shared__ float sml[4][16][2];
  const int h = static_cast<int>(blockIdx.x % a.Hkv);
  const int64_t x = blockIdx.x / a.Hkv;
  const int c = static_cast<int>(blockIdx.y);
  const PagedTile tile = paged_find(a, 16, x, -1);
  if (tile.b < 0) return;
  const PagedSeq& sq = tile.s;
  const int nk = static_cast<int>(sq.nk), nq = sq.nq;
  const int k0 = c * tile.chunk;
  if (k0 >= nk && c > 0) return;
  const bool single = nk <= tile.chunk;
  const int k1 = min(k0 + tile.chunk, nk);
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int r16 = lane & 15, g = lane >> 4;

  // this lane's query row (B operand column) and its last visible key
  const int rr = tile.tl * 16 + r16;
  const bool rvalid = rr < nq * a.G;
  const int qi = rvalid ? rr / a.G : 0;
  const int lim = rvalid ? nk - nq + qi : nk - 1;
  typename T::vec8 qb[KS];
  {
    const uint16_t* qp = static_cast<const uint16_t*>(a.q) + (sq.q0 + qi) * a.qst +
                         static_cast<int64_t>(h * a.G + (rvalid ? rr % a.G : 0)) * a.qhs + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) qb[s] = as_vec8<T>(rvalid ? ld16(qp + 32 * s) : zero4());
  }

  f32x4 acc[E];
#pragma unroll
  for (int e = 0; e < E; ++e) acc[e] = f32x4{};
  float m_run = -INFINITY, l_part = 0.0f;
  bool bad = false;
  const int64_t row = static_cast<int64_t>(tile.b) * a.table_stride;
  const uint16_t* kc = static_cast<const uint16_t*>(a.kc) + static_cast<int64_t>(h) * a.kch;
  const uint16_t* vc = static_cast<const uint16_t*>(a.vc) + static_cast<int64_t>(h) * a.vch;
  const float scale = a.scale_log2;

  uint4 kf[2][KS];
  uint32_t vf[2][4][VW];
  auto load_v = [&](uint32_t (&dst)[VW], const uint16_t* p) {
    if constexpr (D == 64) {
      const uint2 u = *reinterpret_cast<const uint2*>(p + 4 * r16);
      dst[0] = u.x; dst[1] = u.y;
    } else {
#pragma unroll
      for (int q = 0; q < D / 128; ++q) {
        const uint4 u = ld16(p + 128 * q + 8 * r16);
        dst[4 * q] = u.x; dst[4 * q + 1] = u.y; dst[4 * q + 2] = u.z; dst[4 * q + 3] = u.w;
      }
    }
  };
  // pages and in-page offsets of the two 16-key tiles from `base` (P16); a
  // tile past the sequence repeats the last one (its scores are masked)
  const int last16 = (nk - 1) & ~15;
  int64_t page[2] = {0, 0};
  int inpage[2] = {0, 0};
  auto lookup = [&](int base) {
    if constexpr (P16) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int tb = min(base + 16 * j, last16);
        page[j] = paged_page<true>(a, row, tb, bad);
        inpage[j] = a.bs_shift >= 0 ? tb & (a.bs - 1) : tb % a.bs;
      }
    }
  };
  auto load_k = [&](int base) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint16_t* p;
      if constexpr (P16) {
        p = kc + page[j] * a.kcb + static_cast<int64_t>(inpage[j]) * a.kcs;
        p += static_cast<uint32_t>(r16 * static_cast<int>(a.kcs) + 8 * g);
      } else {
        const int key = min(base + 16 * j + r16, nk - 1);
        const int64_t pg = paged_page<false>(a, row, key, bad);
        p = kc + pg * a.kcb + static_cast<int64_t>(key % a.bs) * a.kcs + 8 * g;
      }
#pragma unroll
      for (int s = 0; s < KS; ++s) kf[j][s] = ld16(p + 32 * s);
    }
  };
  auto load_v_tiles = [&](int base) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const uint16_t* p;
        if constexpr (P16) {
          p = vc + page[j] * a.vcb + static_cast<int64_t>(inpage[j] + v) * a.vcs;
          p += static_cast<uint32_t>(4 * g * static_cast<int>(a.vcs));
        } else {
          const int key = min(base + 16 * j + 4 * g + v, nk - 1);
          const int64_t pg = paged_page<false>(a, row, key, bad);
          p = vc + pg * a.vcb + static_cast<int64_t>(key % a.bs) * a.vcs;
        }
        load_v(vf[j][v], p);
      }
  };

  int base = k0 + 32 * w;
  if (base < k1) {
    lookup(base);
    load_k(base);
    load_v_tiles(base);
  }
  for (; base < k1; base += 128) {
    const int next = base + 128;
    const bool more = next < k1;
    f32x4 s[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      s[j] = f32x4{};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s[j] = mfma16(as_vec8<T>(kf[j][ks]), qb[ks], s[j]);
    }
    // the next round's keys fly during this round's softmax and P.V
    if (more) {
      lookup(next);
      load_k(next);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) s[j][v] *= scale;
    if (base + 31 > nk - nq) {  // some row's causal limit or the end lies in this round
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int key = base + 16 * j + 4 * g + v;
          if (key > lim) s[j][v] = -INFINITY;
          if (key >= nk) {  // slots past the end may hold anything
#pragma unroll
            for (int q = 0; q < VW; ++q) vf[j][v][q] = 0u;
          }
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) mx = fmaxf(mx, s[j][v]);
    const float m_new = fmaxf(m_run, row4_max(mx));
    if (__ballot(m_new > m_run) != 0) {
      // rows with no visible key yet keep m = -inf: their factors are 0
      const float ms = m_new == -INFINITY ? 0.0f : m_new;
      const float alpha = __builtin_amdgcn_exp2f(m_run - ms);
      m_run = m_new;
      l_part *= alpha;
#pragma unroll
      for (int e = 0; e < E; ++e)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[e][v] *= alpha;
    }
    const float ms = m_run == -INFINITY ? 0.0f : m_run;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        s[j][v] = __builtin_amdgcn_exp2f(s[j][v] - ms);
        l_part += s[j][v];
      }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const uint16_t u = static_cast<uint16_t>(vf[j][v][e >> 1] >> (16 * (e & 1)));
          acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(T::to_f32(u), s[j][v], acc[e], 0, 0, 0);
        }
    if (more) load_v_tiles(next);
  }

  // O not finite: P.V again over the keys that each row sees (a masked key's infinite
  // or NaN value times P = 0 is NaN), with P and l 2^off times smaller (m larger), so
  // that values near the largest do not overflow before the division by l
  {
    float nf = 0.0f;
#pragma unroll
    for (int e = 0; e < E; ++e)
#pragma unroll
      for (int v = 0; v < 4; ++v) nf = fmaf(acc[e][v], 0.0f, nf);
    if (__ballot(nf != 0.0f) != 0) {
#pragma unroll
      for (int e = 0; e < E; ++e) acc[e] = f32x4{};
      const float off = static_cast<float>(32 - __clz(k1 - k0));
      m_run += off;
      l_part *= __builtin_amdgcn_exp2f(-off);
      const float ms = m_run == -INFINITY ? 0.0f : m_run;
      int lane2 = static_cast<int>(threadIdx.x);  // (formed here, not kept across the loop)
      asm volatile("" : "+v"(lane2));
      const int g2 = (lane2 >> 4) & 3;
#pragma unroll 1
      for (int i = 0; i < 32 * ((k1 - k0 + 127) / 128); ++i) {
        const int key = k0 + 32 * w + 128 * (i >> 5) + (i & 31);
        if (key >= k1) break;
        const int64_t pg = paged_page<true>(a, row, key, bad);
        const int in = key % a.bs;
        const uint16_t* kp = kc + pg * a.kcb + static_cast<int64_t>(in) * a.kcs + 8 * g2;
        const uint16_t* vp = vc + pg * a.vcb + static_cast<int64_t>(in) * a.vcs;
        float x = 0.0f;  // the lane's dims of q . k
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const uint4 ku = ld16(kp + 32 * ks), qu = __builtin_bit_cast(uint4, qb[ks]);
          const uint32_t kw[4] = {ku.x, ku.y, ku.z, ku.w}, qw[4] = {qu.x, qu.y, qu.z, qu.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            x = fmaf(T::to_f32(static_cast<uint16_t>(qw[e])),
                     T::to_f32(static_cast<uint16_t>(kw[e])), x);
            x = fmaf(T::to_f32(static_cast<uint16_t>(qw[e] >> 16)),
                     T::to_f32(static_cast<uint16_t>(kw[e] >> 16)), x);
          }
        }
        x = row4_sum(x) * scale;
        if (key > lim) continue;
        const float p = __builtin_amdgcn_exp2f(x - ms);
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int e = 0; e < E; e += 4) {
            const int dim = D == 64 ? 4 * (4 * g2 + v)
                                    : 128 * (e >> 3) + 8 * (4 * g2 + v) + (e & 7);
            const uint2 u = *reinterpret_cast<const uint2*>(vp + dim);
            acc[e][v] = fmaf(p, T::to_f32(static_cast<uint16_t>(u.x)), acc[e][v]);
            acc[e + 1][v] = fmaf(p, T::to_f32(static_cast<uint16_t>(u.x >> 16)), acc[e + 1][v]);
            acc[e + 2][v] = fmaf(p, T::to_f32(static_cast<uint16_t>(u.y)), acc[e + 2][v]);
            acc[e + 3][v] = fmaf(p, T::to_f32(static_cast<uint16_t>(u.y >> 16)), acc[e + 3][v]);
          }
      }
    }
  }

  // acc[e][v] is dim 8 (4 g + v) + e (+ 120 per e >= 8 at d = 256: the second
  // 128 dims), d = 64: dim 4 (4 g + v) + e, of row r16
  float l = row4_sum(l_part);
  if (__ballot(bad) != 0) l = __uint_as_float(0x7fc00000u);
#pragma unroll
  for (int e = 0; e < E; ++e)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int dim = D == 64 ? 4 * (4 * g + v) + e : 128 * (e >> 3) + 8 * (4 * g + v) + (e & 7);
      sm[w][r16][dim] = acc[e][v];
    }
  if (g == 0) {
    sml[w][r16][0] = m_run;
    sml[w][r16][1] = l;
  }
  __syncthreads();
  const int orow = t >> 4, od = E * (t & 15);
  const int orr = tile.tl * 16 + orow;
  if (orr >= nq * a.G) return;
  const int64_t tok = sq.q0 + orr / a.G;
  const int hq = h * a.G + orr % a.G;
  float M = -INFINITY;
#pragma unroll
  for (int k = 0; k < 4; ++k) M = fmaxf(M, sml[k][orow][0]);
  float L = 0.0f, o[E];
#pragma unroll
  for (int e = 0; e < E; ++e) o[e] = 0.0f;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float mk = sml[k][orow][0];
    // (a quarter each: four finite sums add up to a finite one)
    const float f = mk == -INFINITY ? 0.0f : 0.25f * __builtin_amdgcn_exp2f(mk - M);
    // (a wave without keys has m = -inf and l = 0; NaN scores leave m = -inf
    // with l = NaN, which the sum keeps)
    L += mk == -INFINITY ? sml[k][orow][1] : f * sml[k][orow][1];
#pragma unroll
    for (int e = 0; e < E; ++e) o[e] += f * sm[k][orow][od + e];
  }
  if (single) {
    uint16_t* op = static_cast<uint16_t*>(a.o) + tok * a.ost + static_cast<int64_t>(hq) * a.ohs + od;
    const float rcp = 1.0f / L;
    uint32_t pk[VW];
#pragma unroll
    for (int q = 0; q < VW; ++q) {
      float lo = o[2 * q] * rcp, hi = o[2 * q + 1] * rcp;
      if (nk == 0) lo = hi = sq.bad ? __uint_as_float(0x7fc00000u) : 0.0f;
      pk[q] = pack2<T>(lo, hi);
    }
#pragma unroll
    for (int q = 0; q < VW; q += 2)
      *reinterpret_cast<uint2*>(op + 2 * q) = make_uint2(pk[q], pk[q + 1]);
  } else {
    const int64_t slot = (tok * a.Hq + hq) * a.nc + c;
    float* pp = a.part + slot * D + od;
#pragma unroll
    for (int e = 0; e < E; e += 4)
      *reinterpret_cast<float4*>(pp + e) = make_float4(o[e], o[e + 1], o[e + 2], o[e + 3]);
    if ((t & 15) == 0) {
      a.ml[2 * slot] = M;
      a.ml[2 * slot + 1] = L;
    }
  }
}

// One output row (query token, query head) per workgroup: the row's chunk
// partials weighted by exp2(m_c - max m) and divided by their l. Wave w adds
// chunks w, w + 4, ... (eight loads in flight), LDS adds the four waves.
template <typename T, int D>
__global__ __launch_bounds__(256) void k_paged_merge(PagedArgs a) {
  constexpr int XD = D / 64;  // dims per lane
  __shared__ float so[4][D];
  const int64_t tok = blockIdx.x / a.Hq;
  const int hq = static_cast<int>(blockIdx.x % a.Hq);
  const PagedTile tile = paged_find(a, 16, 0, tok);
  if (tile.b < 0) return;
  const int nk = static_cast<int>(tile.s.nk);
  if (nk <= tile.chunk) return;  // written by k_paged
  const int n = min((nk + tile.chunk - 1) / tile.chunk, a.nc);
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int64_t slot = (tok * a.Hq + hq) * a.nc;
  // (m, l) of chunks lane and lane + 64 (nc <= 128)
  float m0 = -INFINITY, l0 = 0.0f, m1 = -INFINITY, l1 = 0.0f;
  if (lane < n) {
    m0 = a.ml[2 * (slot + lane)];
    l0 = a.ml[2 * (slot + lane) + 1];
  }
  if (lane + 64 < n) {
    m1 = a.ml[2 * (slot + lane + 64)];
    l1 = a.ml[2 * (slot + lane + 64) + 1];
  }
  const float M = wave_max(fmaxf(m0, m1));
  // (2^-7: the sum over at most 128 chunks stays finite)
  const float f0 = m0 == -INFINITY ? 0.0f : 0x1p-7f * __builtin_amdgcn_exp2f(m0 - M);
  const float f1 = m1 == -INFINITY ? 0.0f : 0x1p-7f * __builtin_amdgcn_exp2f(m1 - M);
  float L = (m0 == -INFINITY ? l0 : f0 * l0) + (m1 == -INFINITY ? l1 : f1 * l1);
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) L += __shfl_xor(L, o);
  float acc[XD];
#pragma unroll
  for (int q = 0; q < XD; ++q) acc[q] = 0.0f;
  const float* pp = a.part + slot * D + XD * lane;
  constexpr int U = 8;
  for (int c0 = w; c0 < n; c0 += 4 * U) {
    float v[U][XD], f[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int ch = c0 + 4 * u;
      const bool on = ch < n;
      f[u] = on ? __shfl(ch < 64 ? f0 : f1, ch & 63) : 0.0f;
#pragma unroll
      for (int q = 0; q < XD; ++q) v[u][q] = on ? pp[static_cast<int64_t>(ch) * D + q] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < XD; ++q) acc[q] += f[u] * v[u][q];
  }
#pragma unroll
  for (int q = 0; q < XD; ++q) so[w][XD * lane + q] = acc[q];
  __syncthreads();
  if (t < D) {
    const float o = (so[0][t] + so[1][t] + so[2][t] + so[3][t]) / L;
    static_cast<uint16_t*>(a.o)[tok * a.ost + static_cast<int64_t>(hq) * a.ohs + t] = T::from_f32(o);
  }
}

// ---------------------------------------------------------------------------
// Many query rows per sequence (prefix-cached prefill)
// ---------------------------------------------------------------------------
// P as three parts of the input type that add up to it: fp32 has 24 significand
// bits, bf16 parts hold 8 each, fp16 parts 11 each. fp16 lacks fp32's exponents,
// so P enters scaled by 2^14 (kPShift; P <= 2^14 < 65504). fp16's last step,
// 2^-24, is 2^-38 of the row's largest P there, too coarse for a small P beside a
// large V, so the third part is taken 2^24 times its size (kLowScale; at most
// 2^14, what two parts leave of a P of 2^14 being 2^-10) and summed apart over 32
// keys: P of 2^-15 of the largest and more is held whole, a smaller one to 2^-51
// of the largest, below what 65504 P can add to an fp16 output. (Three requests of
// 500 new tokens on 6,144, 2,500 and 1,111 cached ones, 28 q / 4 kv heads, d = 128:
// 168 us with the parts summed together, 186 so; bf16 169.)
template <typename T>
struct PParts;
template <>
struct PParts<BF16> {
  static constexpr float kPShift = 0.0f, kLowScale = 1.0f;
};
template <>
struct PParts<F16> {
  static constexpr float kPShift = 14.0f, kLowScale = 16777216.0f;
};
template <typename T>
__device__ __forceinline__ void part_pair(float x0, float x1, uint32_t (&u)[3]) {
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    if (p == 2) {
      x0 *= PParts<T>::kLowScale;
      x1 *= PParts<T>::kLowScale;
    }
    u[p] = pack2<T>(x0, x1);
    x0 -= T::to_f32(static_cast<uint16_t>(u[p]));
    x1 -= T::to_f32(static_cast<uint16_t>(u[p] >> 16));
  }
}

// V^T operand of a 16-key step: keys r .. r + 3 and r + 8 .. r + 11, dim xx of a
// key-major tile
template <typename T, int D>
__device__ __forceinline__ typename T::vec8 read_vt(const uint16_t* sv16, int r, int xx) {
  const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) i16x4*)(sv16 + tile_elem<D>(r, xx)));
  const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) i16x4*)(sv16 + tile_elem<D>(r + 8, xx)));
  const uint2 lo2 = __builtin_bit_cast(uint2, lo), hi2 = __builtin_bit_cast(uint2, hi);
  return as_vec8<T>(make_uint4(lo2.x, lo2.y, hi2.x, hi2.y));
}

// One workgroup (4 waves) per (128-row tile of the G query heads of a KV head,
// KV head, chunk of keys), in the orientation of k_attn: wave w owns rows
// 32 w .. 32 w + 31, S^T = K . Q^T and O^T += V^T . P^T on 32x32x16 MFMA, K and V
// in 64-key tiles through LDS (direct-to-LDS loads, two buffers: a tile lands
// while the one before it is used; one barrier per tile). The rows of a tile
// share every K / V byte, where k_paged reads them once per 16 rows. P stays
// fp32: P.V runs on its three exact 16-bit parts (48 of the 64 MFMAs of a tile
// and wave at d = 128). Bound by these MFMAs and the instructions that form the
// parts. Measured (one MI355X, whole calls): 500 new tokens each on 6,144, 2,500
// and 1,111 cached ones (28 q / 4 kv heads, d = 128) 504 us with k_paged, 169 here
// (the merge 8); 4 x 2,048 new of 4,096 (32 q / 8 kv) 3,045 -> 890 us = 463 TFLOP/s
// (924 of MFMAs).
template <typename T, int D, bool P16>
__global__ __launch_bounds__(256, 2) void k_paged_rows(PagedArgs a) {
  constexpr int KT = 64, TT = KT / 32;
  constexpr int KS = D / 16, DT = D / 32, CH = D / 8;
  constexpr int RPW = 64 / CH;             // rows per load instruction
  constexpr int NI = KT * CH / 64 / 4;     // load instructions per wave and tile
  static_assert(NI * RPW == 16, "a wave loads 16 consecutive keys of a tile");
  __shared__ uint4 sk[2][KT * CH];
  __shared__ uint4 sv[2][KT * CH];
  __shared__ int s_bad;  // some wave looked up a page outside the cache
  const int h = static_cast<int>(blockIdx.x % a.Hkv);
  const int64_t x = blockIdx.x / a.Hkv;
  const int c = static_cast<int>(blockIdx.y);
  const PagedTile tile = paged_find(a, 128, x, -1);
  if (tile.b < 0) return;
  const PagedSeq& sq = tile.s;
  const int nk = static_cast<int>(sq.nk), nq = sq.nq;
  const int k0 = c * tile.chunk;
  if (k0 >= nk && c > 0) return;
  const bool single = nk <= tile.chunk;
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  const int rows = nq * a.G;

  // this lane's query row and its last visible key
  const int rr = tile.tl * 128 + 32 * w + l32;
  const bool rvalid = rr < rows;
  const int qi = (rvalid ? rr : rows - 1) / a.G;
  const int64_t tok = sq.q0 + qi;
  const int hq = h * a.G + (rvalid ? rr : rows - 1) % a.G;
  const int lim = nk - nq + qi;
  // the wave's first and last visible keys' bounds (wave-uniform)
  const int r0 = min(tile.tl * 128 + 32 * w, rows - 1), r1 = min(tile.tl * 128 + 32 * w + 31, rows - 1);
  const int lim_lo = __builtin_amdgcn_readfirstlane(nk - nq + r0 / a.G);
  const int lim_hi = __builtin_amdgcn_readfirstlane(nk - nq + r1 / a.G);
  // keys past the last row of the tile are visible to none of its rows
  const int last_row = min(tile.tl * 128 + 127, rows - 1);
  const int k1 = __builtin_amdgcn_readfirstlane(
      min(min(k0 + tile.chunk, nk), max(nk - nq + last_row / a.G + 1, 0)));

  typename T::vec8 qb[KS];
  {
    const uint16_t* qp = static_cast<const uint16_t*>(a.q) + tok * a.qst +
                         static_cast<int64_t>(hq) * a.qhs + 8 * half;
#pragma unroll
    for (int s = 0; s < KS; ++s) qb[s] = as_vec8<T>(rvalid ? ld16(qp + 16 * s) : zero4());
  }
  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = f32x16{};
  float m_run = -INFINITY, l_part = 0.0f;
  bool bad = false;

  const int64_t row = static_cast<int64_t>(tile.b) * a.table_stride;
  const uint16_t* kc = static_cast<const uint16_t*>(a.kc) + static_cast<int64_t>(h) * a.kch;
  const uint16_t* vc = static_cast<const uint16_t*>(a.vc) + static_cast<int64_t>(h) * a.vch;
  // the lane's byte offsets in the wave's 16 keys (P16)
  uint32_t koff[NI], voff[NI];
#pragma unroll
  for (int q = 0; q < NI; ++q) {
    const int r = q * RPW + lane / CH;
    const int ch = 8 * ((lane % CH) ^ swz<D>(16 * w + r));
    koff[q] = 2 * (static_cast<uint32_t>(r) * static_cast<uint32_t>(a.kcs) + ch);
    voff[q] = 2 * (static_cast<uint32_t>(r) * static_cast<uint32_t>(a.vcs) + ch);
  }
  const int last16 = (nk - 1) & ~15;
  // tile of keys base .. base + 63 into buffer `buf`; keys past the sequence
  // read its last 16-key group (P16: slots past the end are masked and their V
  // zeroed below) or its last key
  auto issue = [&](int base, int buf) {
    if constexpr (P16) {
      const int tb = min(base + 16 * w, last16);
      const int64_t pg = paged_page<true>(a, row, tb, bad);
      const int in = a.bs_shift >= 0 ? tb & (a.bs - 1) : tb % a.bs;
      uint64_t kb = scalar_addr(kc + pg * a.kcb + static_cast<int64_t>(in) * a.kcs);
      uint64_t vb = scalar_addr(vc + pg * a.vcb + static_cast<int64_t>(in) * a.vcs);
      const uint32_t kl = lds_addr(sk[buf] + w * NI * 64), vl = lds_addr(sv[buf] + w * NI * 64);
      // five wait states between the readfirstlane of the bases and their use
      asm volatile("s_nop 4" : "+s"(kb), "+s"(vb));
#pragma unroll
      for (int q = 0; q < NI; ++q) dma16_sbase_m0(kl + q * 1024, kb, koff[q]);
#pragma unroll
      for (int q = 0; q < NI; ++q) dma16_sbase_m0(vl + q * 1024, vb, voff[q]);
    } else {
#pragma unroll
      for (int q = 0; q < NI; ++q) {
        const int r = 16 * w + q * RPW + lane / CH;
        const int key = min(base + r, nk - 1);
        const int64_t pg = paged_page<false>(a, row, key, bad);
        const int in = key % a.bs, ch = 8 * ((lane % CH) ^ swz<D>(r));
        dma16_vaddr(sk[buf] + (w * NI + q) * 64, kc + pg * a.kcb + static_cast<int64_t>(in) * a.kcs + ch);
        dma16_vaddr(sv[buf] + (w * NI + q) * 64, vc + pg * a.vcb + static_cast<int64_t>(in) * a.vcs + ch);
      }
    }
  };
  const int g16 = lane >> 4, i16 = lane & 15;
  const int tr_row = 4 * (g16 >> 1) + (i16 >> 2);
  const int tr_col = 16 * (g16 & 1) + 4 * (i16 & 3);

  // (ordered before the flag by the barrier after the loop)
  if (t == 0) s_bad = 0;
  if (k0 < k1) issue(k0, 0);
  int buf = 0;
  for (int base = k0; base < k1; base += KT, buf ^= 1) {
    // this tile has landed for every wave, and every wave is done with the other
    // buffer
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (base + KT < k1) issue(base + KT, buf ^ 1);
    if (base + KT > nk) {  // V of slots past the sequence: 0 (they may hold anything)
      for (int i = t; i < KT * CH; i += 256)
        if (base + i / CH >= nk) sv[buf][i] = zero4();
      lds_barrier();
    }
    if (base > lim_hi) continue;  // no key of this tile is visible to the wave
    f32x16 s[TT];
#pragma unroll
    for (int t4 = 0; t4 < TT; ++t4) s[t4] = f32x16{};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int t4 = 0; t4 < TT; ++t4) {
        const int r = 32 * t4 + l32;
        const uint4 kop = sk[buf][r * CH + ((2 * ks + half) ^ swz<D>(r))];
        s[t4] = T::mfma32(as_vec8<T>(kop), qb[ks], s[t4]);
      }
    float mx = -INFINITY;
    if (base + KT - 1 > lim_lo) {
#pragma unroll
      for (int t4 = 0; t4 < TT; ++t4)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int key = base + 32 * t4 + 8 * (v >> 2) + 4 * half + (v & 3);
          s[t4][v] = key > lim ? -INFINITY : s[t4][v] * a.scale_log2;
          mx = fmaxf(mx, s[t4][v]);
        }
    } else {
#pragma unroll
      for (int t4 = 0; t4 < TT; ++t4)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          s[t4][v] *= a.scale_log2;
          mx = fmaxf(mx, s[t4][v]);
        }
    }
    const float m_new = fmaxf(m_run, pair32_max(mx));
    if (__ballot(m_new > m_run) != 0) {
      const float ms = m_new == -INFINITY ? 0.0f : m_new;
      const float alpha = __builtin_amdgcn_exp2f(m_run - ms);
      m_run = m_new;
      l_part *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[dt][v] *= alpha;
    }
    // rows with no visible key yet keep m = -inf: their P is 0
    const float ms = (m_run == -INFINITY ? 0.0f : m_run) - PParts<T>::kPShift;
#pragma unroll
    for (int t4 = 0; t4 < TT; ++t4) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        s[t4][v] = __builtin_amdgcn_exp2f(s[t4][v] - ms);
        l_part += s[t4][v];
      }
      if constexpr (PParts<T>::kLowScale == 1.0f) {
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          uint32_t u[4][3];
#pragma unroll
          for (int e = 0; e < 4; ++e)
            part_pair<T>(s[t4][8 * hh + 2 * e], s[t4][8 * hh + 2 * e + 1], u[e]);
          typename T::vec8 pb[3];
#pragma unroll
          for (int p = 0; p < 3; ++p)
            pb[p] = as_vec8<T>(make_uint4(u[0][p], u[1][p], u[2][p], u[3][p]));
          const uint16_t* sv16 = reinterpret_cast<const uint16_t*>(sv[buf]);
          const int r = 32 * t4 + 16 * hh + tr_row;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            const int xx = 32 * dt + tr_col;
            const typename T::vec8 va = read_vt<T, D>(sv16, r, xx);
            o[dt] = T::mfma32(va, pb[2], o[dt]);
            o[dt] = T::mfma32(va, pb[1], o[dt]);
            o[dt] = T::mfma32(va, pb[0], o[dt]);
          }
        }
      } else {
        typename T::vec8 pb[2][3];
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          uint32_t u[4][3];
#pragma unroll
          for (int e = 0; e < 4; ++e)
            part_pair<T>(s[t4][8 * hh + 2 * e], s[t4][8 * hh + 2 * e + 1], u[e]);
#pragma unroll
          for (int p = 0; p < 3; ++p)
            pb[hh][p] = as_vec8<T>(make_uint4(u[0][p], u[1][p], u[2][p], u[3][p]));
        }
        const uint16_t* sv16 = reinterpret_cast<const uint16_t*>(sv[buf]);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          f32x16 low = f32x16{};
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) {
            const int r = 32 * t4 + 16 * hh + tr_row, xx = 32 * dt + tr_col;
            const typename T::vec8 va = read_vt<T, D>(sv16, r, xx);
            low = T::mfma32(va, pb[hh][2], low);
            o[dt] = T::mfma32(va, pb[hh][1], o[dt]);
            o[dt] = T::mfma32(va, pb[hh][0], o[dt]);
          }
#pragma unroll
          for (int v = 0; v < 16; ++v)
            o[dt][v] = fmaf(low[v], 1.0f / PParts<T>::kLowScale, o[dt][v]);
        }
      }
    }
  }

  // An infinite or NaN value times the parts of P is NaN where its product with P
  // is not (a part may be 0 or negative), and sums of values near the largest
  // overflow before they are divided by l: rows whose O is not finite take P.V again
  // in fp32 with P whole, over the keys that each row sees.
  float nf = 0.0f;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int v = 0; v < 16; ++v) nf = fmaf(o[dt][v], 0.0f, nf);
  if (__ballot(nf != 0.0f) != 0) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = f32x16{};
    // P and l 2^off times smaller (m larger): the sum of P V then stays below the
    // largest value, as that of normalised weights does
    const float off = static_cast<float>(32 - __clz(k1 - k0));
    m_run += off;
    l_part *= __builtin_amdgcn_exp2f(-off);
    const float ms = (m_run == -INFINITY ? 0.0f : m_run) - PParts<T>::kPShift;
    // (formed here: kept live across the loop above, the offsets cost d = 64 its
    // third wave per SIMD, 781 -> 826 us for 4 x 2,048 new of 6,144 tokens)
    int half2 = static_cast<int>(threadIdx.x);
    asm volatile("" : "+v"(half2));
    half2 = (half2 >> 5) & 1;
#pragma unroll 1
    for (int key = k0; key < k1; ++key) {
      const int64_t pg = paged_page<true>(a, row, key, bad);
      const int in = key % a.bs;
      const uint16_t* kp = kc + pg * a.kcb + static_cast<int64_t>(in) * a.kcs + 8 * half2;
      const uint16_t* vp = vc + pg * a.vcb + static_cast<int64_t>(in) * a.vcs + 4 * half2;
      float x = 0.0f;  // the lane's dims of q . k
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const uint4 ku = ld16(kp + 16 * s), qu = __builtin_bit_cast(uint4, qb[s]);
        const uint32_t kw[4] = {ku.x, ku.y, ku.z, ku.w}, qw[4] = {qu.x, qu.y, qu.z, qu.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x = fmaf(T::to_f32(static_cast<uint16_t>(qw[e])), T::to_f32(static_cast<uint16_t>(kw[e])), x);
          x = fmaf(T::to_f32(static_cast<uint16_t>(qw[e] >> 16)),
                   T::to_f32(static_cast<uint16_t>(kw[e] >> 16)), x);
        }
      }
      x = pair32_sum(x) * a.scale_log2;
      if (key > lim) continue;
      const float p = __builtin_amdgcn_exp2f(x - ms);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          const uint2 u = *reinterpret_cast<const uint2*>(vp + 32 * dt + 8 * g4);
          o[dt][4 * g4] = fmaf(p, T::to_f32(static_cast<uint16_t>(u.x)), o[dt][4 * g4]);
          o[dt][4 * g4 + 1] = fmaf(p, T::to_f32(static_cast<uint16_t>(u.x >> 16)), o[dt][4 * g4 + 1]);
          o[dt][4 * g4 + 2] = fmaf(p, T::to_f32(static_cast<uint16_t>(u.y)), o[dt][4 * g4 + 2]);
          o[dt][4 * g4 + 3] = fmaf(p, T::to_f32(static_cast<uint16_t>(u.y >> 16)), o[dt][4 * g4 + 3]);
        }
    }
  }

  // A wave looks up the pages of its 16 keys of a tile only, and all four use the
  // tile: a bad page found by one makes the rows of all four NaN.
  float l = pair32_sum(l_part);
  lds_barrier();
  if (bad) s_bad = 1;
  lds_barrier();
  if (s_bad != 0) l = __uint_as_float(0x7fc00000u);
  if (!rvalid) return;
  if (single) {
    const float rcp = 1.0f / l;
    uint16_t* op = static_cast<uint16_t*>(a.o) + tok * a.ost + static_cast<int64_t>(hq) * a.ohs;
    const float nan = __uint_as_float(0x7fc00000u);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          y[e] = o[dt][4 * g4 + e] * rcp;
          if (nk == 0) y[e] = sq.bad ? nan : 0.0f;
        }
        *reinterpret_cast<uint2*>(op + 32 * dt + 8 * g4 + 4 * half) =
            make_uint2(pack2<T>(y[0], y[1]), pack2<T>(y[2], y[3]));
      }
  } else {
    const int64_t slot = (tok * a.Hq + hq) * a.nc + c;
    float* pp = a.part + slot * D;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4)
        *reinterpret_cast<float4*>(pp + 32 * dt + 8 * g4 + 4 * half) =
            make_float4(o[dt][4 * g4], o[dt][4 * g4 + 1], o[dt][4 * g4 + 2], o[dt][4 * g4 + 3]);
    if (half == 0) {
      a.ml[2 * slot] = m_run;
      a.ml[2 * slot + 1] = l;
    }
  }
}

// Output rows of k_paged_rows: one wave per kMergeHeads query heads of a token
// (four waves per workgroup), their chunks (few) in turn; the arithmetic of
// k_paged_merge. Bound by the latency of finding the token's sequence (loads,
// scans over the lanes) and of the (m, l) and partial loads that follow, so a wave
// finds it once for its heads and has the loads of all of them in flight (1,500
// tokens x 28 heads, two chunks, 43 MB of partials: 16.8 us with a wave per head,
// 8.5 with four heads).
constexpr int kMergeHeads = 4;
template <typename T, int D>
__global__ __launch_bounds__(256) void k_paged_merge_rows(PagedArgs a) {
  constexpr int XD = D / 64;  // dims per lane
  constexpr int H = kMergeHeads;
  const int64_t x = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  const int groups = (a.Hq + H - 1) / H;
  const int64_t tok = x / groups;
  if (tok >= a.T) return;
  const int h0 = static_cast<int>(x % groups) * H, lane = threadIdx.x & 63;
  const PagedTile tile = paged_find(a, 128, 0, tok);
  if (tile.b < 0) return;
  const int nk = static_cast<int>(tile.s.nk);
  if (nk <= tile.chunk) return;
  const int n = min((nk + tile.chunk - 1) / tile.chunk, a.nc);
  int64_t slot[H];  // (heads past the last repeat it)
  float M[H], L[H], acc[H][XD];
#pragma unroll
  for (int u = 0; u < H; ++u) {
    slot[u] = (tok * a.Hq + min(h0 + u, a.Hq - 1)) * a.nc;
    M[u] = -INFINITY;
    L[u] = 0.0f;
#pragma unroll
    for (int q = 0; q < XD; ++q) acc[u][q] = 0.0f;
  }
  for (int c = 0; c < n; ++c)
#pragma unroll
    for (int u = 0; u < H; ++u) M[u] = fmaxf(M[u], a.ml[2 * (slot[u] + c)]);
#pragma unroll 2
  for (int c = 0; c < n; ++c)
#pragma unroll
    for (int u = 0; u < H; ++u) {
      const float m = a.ml[2 * (slot[u] + c)], l = a.ml[2 * (slot[u] + c) + 1];
      const float f = m == -INFINITY ? 0.0f : 0x1p-7f * __builtin_amdgcn_exp2f(m - M[u]);
      L[u] += m == -INFINITY ? l : f * l;
#pragma unroll
      for (int q = 0; q < XD; ++q) acc[u][q] += f * a.part[(slot[u] + c) * D + XD * lane + q];
    }
#pragma unroll
  for (int u = 0; u < H; ++u) {
    if (h0 + u >= a.Hq) break;
    uint16_t* op = static_cast<uint16_t*>(a.o) + tok * a.ost +
                   static_cast<int64_t>(h0 + u) * a.ohs + XD * lane;
    const float rcp = 1.0f / L[u];
    if constexpr (XD == 2)
      *reinterpret_cast<uint32_t*>(op) = pack2<T>(acc[u][0] * rcp, acc[u][1] * rcp);
    else
      op[0] = T::from_f32(acc[u][0] * rcp);
  }
}

template <typename T, int D>
hipError_t launch_paged_rows_t(const PagedArgs& a, int64_t tiles, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(tiles * a.Hkv), static_cast<unsigned>(a.nc));
  if (a.bs % 16 == 0) hipLaunchKernelGGL((k_paged_rows<T, D, true>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((k_paged_rows<T, D, false>), grid, dim3(256), 0, s, a);
  if (a.nc > 1) {
    const int64_t waves = a.T * ((a.Hq + kMergeHeads - 1) / kMergeHeads);
    hipLaunchKernelGGL((k_paged_merge_rows<T, D>), dim3(static_cast<unsigned>((waves + 3) / 4)),
                       dim3(256), 0, s, a);
  }
  return hipGetLastError();
}

template <typename T, int D>
hipError_t launch_paged_t(const PagedArgs& a, int64_t tiles, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(tiles * a.Hkv), static_cast<unsigned>(a.nc));
  if (a.bs % 16 == 0) hipLaunchKernelGGL((k_paged<T, D, true>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((k_paged<T, D, false>), grid, dim3(256), 0, s, a);
  if (a.nc > 1)
    hipLaunchKernelGGL((k_paged_merge<T, D>), dim3(static_cast<unsigned>(a.T * a.Hq)), dim3(256), 0,
                       s, a);
  return hipGetLastError();
}

hipError_t launch_paged_rows(const PagedArgs& a, int dtype, int head_dim, int64_t tiles,
                             hipStream_t s) {
  if (head_dim == 128)
    return dtype == FP_DTYPE_BF16 ? launch_paged_rows_t<BF16, 128>(a, tiles, s)
                                  : launch_paged_rows_t<F16, 128>(a, tiles, s);
  return dtype == FP_DTYPE_BF16 ? launch_paged_rows_t<BF16, 64>(a, tiles, s)
                                : launch_paged_rows_t<F16, 64>(a, tiles, s);
}

hipError_t launch_paged(const PagedArgs& a, int dtype, int head_dim, int64_t tiles, hipStream_t s) {
  return with_head_dim(head_dim, [&](auto dc) {
    constexpr int D = decltype(dc)::value;
    return dtype == FP_DTYPE_BF16 ? launch_paged_t<BF16, D>(a, tiles, s)
                                  : launch_paged_t<F16, D>(a, tiles, s);
  });
}

}  // namespace fp
