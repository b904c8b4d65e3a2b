// Flash-attention forward for calls with too few 128-query blocks to fill the device (one decode
// step over a cache, a few new tokens behind it, one short sequence): the wavefronts of a workgroup
// split the keys instead of the queries.
//
// What bounds these calls is not the matrix cores: with one workgroup per 128 queries and the keys
// walked in sequence, a decode step keeps B * H workgroups busy with one useful row of 128 and reads
// every K/V head once per query head. Here
//   * the rows of a workgroup are 32 (query, query head) pairs that read the same K/V head (row r of
//     a K/V head is query r / G, head r % G of its group of G), so grouped heads share one read of
//     the cache;
//   * its W wavefronts each take every W-th tile of 32 keys with an online softmax of their own (no
//     barrier until the end) and their sums are combined through LDS: sum_w 2^(m_w - m) O_w over
//     sum_w 2^(m_w - m) l_w, in wavefront order, in fp32;
//   * a workgroup computes NDB blocks of 32 output dims; with fewer than all of them the workgroups
//     of one (b, K/V head) each read all of K but only their columns of V. K is then re-read from
//     L2 (consecutive workgroups share an XCD), and no partial result leaves the chip: no workspace,
//     no second kernel;
//   * behind a long cache the keys are split over kv_splits workgroups instead, whose sums (unscaled,
//     fp32, with each row's exponent offset and weight sum) a second kernel adds in split order. Where
//     there is no buffer for them one workgroup walks the splits (the _seq kernels): the same bits.
// With every CU reading, HBM bounds it: B 8, H 32, H_kv 8, 1 query, 4096 keys, D 128, bf16 (134 MB of
// K and V): 105 us on the 128-query kernel -> 31 us (4.3 TB/s); 32 K/V heads (537 MB): 125 -> 98 us
// (5.5 TB/s, as a large copy). Short sequences are bound by the latency of a wavefront's tiles, about
// 2 us each (1 x 8 heads x 1023, D 128: 23.6 -> 12.9 us, one tile in flight ahead of the current one).
// Each wavefront stages its own key tiles global -> registers -> LDS (the next tile's loads are in
// flight while the current one is computed), whole rows per load instruction; the products and the
// LDS layouts are those of the 128-query kernel (attention.hpp).
#include "attention.hpp"

namespace mtk {

constexpr int kKvRows = 32;  // rows per workgroup
constexpr int kKvTile = 32;  // keys per wavefront step

__device__ __forceinline__ u32x4 buf_load16_s(rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
}

// Weighted V sums of some keys of a row (8 dims), unscaled, with their exponent offset (log2) and the sum of
// the weights. Sums are added with one rounding per step that is written out (fp contraction is off here
// and in attn_kv, else each kernel's compiler would choose which product to fuse), so that the splits'
// sums come out the same whether one workgroup walks the splits or a second kernel adds them.
struct KvSum {
  float m = -INFINITY, l = 0.0f;
  f32x4 x0 = f32x4{}, x1 = f32x4{};
};
__device__ __forceinline__ f32x4 fma4(float f, f32x4 x, f32x4 y) {
  return f32x4{__builtin_fmaf(f, x.x, y.x), __builtin_fmaf(f, x.y, y.y), __builtin_fmaf(f, x.z, y.z), __builtin_fmaf(f, x.w, y.w)};
}
__device__ __forceinline__ void add_keys(KvSum &s, const KvSum &t) {
#pragma clang fp contract(off)
  const float d = t.m - s.m;  // NaN: no keys on either side
  const float e = __builtin_amdgcn_exp2f(-fabsf(d));
  const float f = d > 0.0f ? e : 1.0f, g = d > 0.0f ? 1.0f : d <= 0.0f ? e : 0.0f;
  s.m = fmaxf(s.m, t.m);
  s.l = __builtin_fmaf(g, t.l, f * s.l);
  s.x0 = fma4(g, t.x0, f * s.x0);
  s.x1 = fma4(g, t.x1, f * s.x1);
}
// N (8 or 4) dims of row (b, q, h) from d on, and the row's log-sum-exp if `lse`.
template <int DT, int N = 8>
__device__ __forceinline__ void store_row(const mtk_attn_kargs &a, int b, int q, int h, int d, const KvSum &s, bool lse) {
  const float inv = s.l > 0.0f ? 1.0f / s.l : 0.0f;
  if (d < a.D) {
    uint16_t *o = (uint16_t *)a.O + (((size_t)b * a.S_q + q) * a.H + h) * a.D + d;
    const u32x2 lo = {pack2<DT>(s.x0.x * inv, s.x0.y * inv), pack2<DT>(s.x0.z * inv, s.x0.w * inv)};
    const u32x2 hi = {pack2<DT>(s.x1.x * inv, s.x1.y * inv), pack2<DT>(s.x1.z * inv, s.x1.w * inv)};
    if constexpr (N == 8)
      *(u32x4 *)o = u32x4{lo.x, lo.y, hi.x, hi.y};
    else
      *(u32x2 *)o = lo;
  }
  if (lse) store_lse(a, b, h, q, 0, s.m, s.l);
}

// SEQ: one workgroup walks all kv_splits splits of the keys in turn (no partial-sum buffer to be had), with
// the sums of each and their order as when the splits are shared out: the same bits.
template <int DT, int DP, int NDB, int W, bool SEQ>
__device__ __forceinline__ void attn_kv(const mtk_attn_kargs &a) {
#pragma clang fp contract(off)
  using L = AttnLayout<DP>;
  constexpr int kKs = L::kKs, kRowB = L::kRowB;
  constexpr int kKI = kKvTile * kRowB / 1024;        // staging instructions per K tile
  constexpr int kVRowB = NDB * 64;                   // bytes of a V row's slice
  constexpr int kVCpr = NDB * 4, kVRpi = 64 / kVCpr; // chunks per slice row, rows per instruction
  constexpr int kVI = kKvTile * kVRowB / 1024;
  constexpr int kWaveB = kKvTile * (kRowB + kVRowB); // staging bytes per wavefront
  constexpr int kOPitch = NDB * 32 + 4;              // floats per row of a wavefront's parked O
  constexpr int kOB = kKvRows * kOPitch * 4;
  constexpr int kMainB = W * (kWaveB > kOB ? kWaveB : kOB);
  __shared__ __attribute__((aligned(1024))) char smem[kMainB];
  __shared__ float sm_m[W][kKvRows], sm_l[W][kKvRows];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, col = lane & 31;
  const int D = a.D;
  const int G = a.H / a.H_kv;
  const int slices = (D + 32 * NDB - 1) / (32 * NDB);

  // consecutive ids: the slices, then the row blocks, of one (b, K/V head)
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int sl = id % slices;
  int rest = id / slices;
  int split = 0;
  if constexpr (!SEQ) {
    split = rest % a.kv_splits;
    rest /= a.kv_splits;
  }
  int rb = rest % a.q_blocks;
  const int bh = rest / a.q_blocks;
  if (a.causal) rb = a.q_blocks - 1 - rb;  // longest first
  const int b = bh / a.H_kv, hk = bh - b * a.H_kv;
  const int d_lo = sl * 32 * NDB;
  const int rows = a.S_q * G;
  const int r0 = rb * kKvRows;
  const int row = r0 + col;
  const int qi = row / G, h = hk * G + (row - qi * G);
  const bool live = row < rows;
  const uint32_t rkv = (uint32_t)a.H_kv * D * 2;
  const uint32_t kvbase = (uint32_t)(((size_t)b * a.S_kv * a.H_kv + hk) * D * 2);
  const size_t obase = (((size_t)b * a.S_q + qi) * a.H + h) * D;  // this lane's row of Q / O
  const rsrc_t rq = make_rsrc(a.Q, a.q_bytes);
  const rsrc_t rk = make_rsrc(a.K, a.kv_bytes);
  const rsrc_t rv = make_rsrc(a.V, a.kv_bytes);
  const int diag = a.S_kv - a.S_q;

  u32x4 qf[kKs];
#pragma unroll
  for (int ds = 0; ds < kKs; ++ds) {
    const int d0 = 16 * ds + 8 * g;
    qf[ds] = buf_load16(rq, (live && d0 < D) ? (uint32_t)(obase * 2) + 2u * d0 : kOOB);
  }

  int kv_end = a.S_kv;
  if (a.causal) kv_end = min(a.S_kv, (min(r0 + kKvRows, rows) - 1) / G + diag + 1);
  int n_tiles = kv_end > 0 ? (kv_end + kKvTile - 1) / kKvTile : 0;
  const int per_split = (n_tiles + a.kv_splits - 1) / a.kv_splits;
  int t0 = split * per_split, t1 = min(n_tiles, t0 + per_split);  // this split's key tiles
  const int first_masked = a.causal ? r0 / G + diag : a.S_kv;  // a tile past this key needs the mask

  char *kt = smem + wave * kWaveB;
  char *vt = kt + kKvTile * kRowB;

  // staging places of this lane: K row i * kRpi + lane / kCpr, chunk lane % kCpr (swizzled in LDS)
  const int kr = lane / L::kCpr, kc = lane % L::kCpr;
  const int vr = lane / kVCpr, vc = lane % kVCpr;
  const uint32_t klane = 8 * kc < D ? (uint32_t)kr * rkv + 16u * kc : kOOB;
  const uint32_t vlane = d_lo + 8 * vc < D ? (uint32_t)vr * rkv + 2u * d_lo + 16u * vc : kOOB;
  auto vswz = [](int r) { return NDB >= 4 ? 4 * (r & 3) : NDB == 2 ? 4 * ((r >> 1) & 1) : 0; };

  u32x4 ks[kKI], vs[kVI];
  auto load = [&](int t) {
    const uint32_t tb = kvbase + (uint32_t)(t * kKvTile) * rkv;
    if ((t + 1) * kKvTile <= a.S_kv) {  // the scalar part is not range-checked: whole tiles only
#pragma unroll
      for (int i = 0; i < kKI; ++i) ks[i] = buf_load16_s(rk, klane, tb + (uint32_t)(i * L::kRpi) * rkv);
#pragma unroll
      for (int i = 0; i < kVI; ++i) vs[i] = buf_load16_s(rv, vlane, tb + (uint32_t)(i * kVRpi) * rkv);
    } else {
#pragma unroll
      for (int i = 0; i < kKI; ++i) {
        const bool in = t * kKvTile + i * L::kRpi + kr < a.S_kv && klane != kOOB;
        ks[i] = buf_load16(rk, in ? tb + (uint32_t)(i * L::kRpi) * rkv + klane : kOOB);
      }
#pragma unroll
      for (int i = 0; i < kVI; ++i) {
        const bool in = t * kKvTile + i * kVRpi + vr < a.S_kv && vlane != kOOB;
        vs[i] = buf_load16(rv, in ? tb + (uint32_t)(i * kVRpi) * rkv + vlane : kOOB);
      }
    }
  };

  const int krow = swap_bits_2_3(col);
  const int ts = lane & 15, th = lane >> 4;

  const float c = a.scale_log2;
  constexpr int kChunks = NDB * 4;  // 8-dim chunks per row
  static_assert(!SEQ || kKvRows * kChunks <= W * 64, "one (row, chunk) per thread");
  KvSum total;  // SEQ: the splits so far, this thread's (row, chunk)

  if (t0 + wave < t1) load(t0 + wave);
  for (;;) {  // one split; SEQ: each in turn
    float m_off = -INFINITY, l_run = 0.0f;
    f32x16 o[NDB];
#pragma unroll
    for (int i = 0; i < NDB; ++i) o[i] = f32x16{};

    for (int t = t0 + wave; t < t1; t += W) {
#pragma unroll
      for (int i = 0; i < kKI; ++i) {
        const int r = i * L::kRpi + kr;
        *(u32x4 *)(kt + r * kRowB + ((kc ^ L::kswz(r)) << 4)) = ks[i];
      }
#pragma unroll
      for (int i = 0; i < kVI; ++i) {
        const int r = i * kVRpi + vr;
        *(u32x4 *)(vt + r * kVRowB + ((vc ^ vswz(r)) << 4)) = vs[i];
      }
      if (t + W < t1) load(t + W);
      // the tile is this wavefront's own: its LDS accesses complete in order, only the compiler has
      // to keep the reads (of other lanes' chunks) behind the writes
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();

      f32x16 s = f32x16{};
#pragma unroll
      for (int ds = 0; ds < kKs; ++ds)
        s = mfma32x32x16<DT>(*(const u32x4 *)(kt + krow * kRowB + (((2 * ds + g) ^ L::kswz(krow)) << 4)), qf[ds], s);

      const int j0 = t * kKvTile;
      if (j0 + kKvTile > a.S_kv || j0 + kKvTile - 1 > first_masked) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = j0 + ((r < 8) ? (8 * g + r) : (16 + 8 * g + (r - 8)));
          s[r] = (key < a.S_kv && (!a.causal || key <= qi + diag)) ? s[r] : -INFINITY;
        }
      }
      float mx = -INFINITY;
#pragma unroll
      for (int r = 0; r < 16; r += 2) mx = vmax3(mx, s[r], s[r + 1]);
      mx = half_max(mx);
      const float m_tile = mx * c;
      float alpha = 1.0f;
      if (m_tile > m_off + kRescaleSlack) {
        alpha = __builtin_amdgcn_exp2f(m_off - m_tile);
        m_off = m_tile;
      }
      const float moff = m_off == -INFINITY ? 0.0f : m_off;
      if (__any(alpha != 1.0f)) {
#pragma unroll
        for (int i = 0; i < NDB; ++i) o[i] *= alpha;
      }
      u32x4 pf[2];
      float psum = 0.0f;
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], c, -moff));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r + 1], c, -moff));
        psum += p0 + p1;
        pf[r >> 3][(r & 7) >> 1] = pack2<DT>(p0, p1);
      }
      l_run = __builtin_fmaf(l_run, alpha, psum);

      // O^T += V^T . P^T: the fragment of d block db, keys 16 js .. +15, as two transposed reads
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int js = 0; js < 2; ++js) {
          const int d = 32 * db + 16 * (th & 1) + 4 * (ts & 3);
          uint32_t w[4];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int r = 16 * js + 8 * (th >> 1) + 4 * e + (ts >> 2);
            const char *p = vt + r * kVRowB + (((d >> 3) ^ vswz(r)) << 4) + 2 * (d & 7);
            const s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)p);
            const u32x2 y = __builtin_bit_cast(u32x2, x);
            w[2 * e] = y.x;
            w[2 * e + 1] = y.y;
          }
          o[db] = mfma32x32x16<DT>(u32x4{w[0], w[1], w[2], w[3]}, pf[js], o[db]);
        }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }

    // ---- combine the wavefronts' sums
    if (SEQ && t1 + wave < min(n_tiles, t1 + per_split)) load(t1 + wave);  // the next split's first tile
    const float l_tot = half_sum(l_run);
    __syncthreads();  // every wavefront is done with its staging region
    if (g == 0) {
      sm_m[wave][col] = m_off;
      sm_l[wave][col] = l_tot;
    }
    float *park = (float *)smem + wave * (kOB / 4);
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *(f32x4 *)(park + col * kOPitch + 32 * db + 8 * q + 4 * g) =
            f32x4{o[db][4 * q], o[db][4 * q + 1], o[db][4 * q + 2], o[db][4 * q + 3]};
    __syncthreads();

    auto sum = [&](int it) {
      const int r = it / kChunks, ch = it % kChunks;
      KvSum s;
#pragma unroll
      for (int w = 0; w < W; ++w) s.m = fmaxf(s.m, sm_m[w][r]);
      const float m0 = s.m == -INFINITY ? 0.0f : s.m;
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const float f = __builtin_amdgcn_exp2f(sm_m[w][r] - m0);
        const float *p = (const float *)smem + w * (kOB / 4) + r * kOPitch + 8 * ch;
        s.l = __builtin_fmaf(f, sm_l[w][r], s.l);
        s.x0 = fma4(f, *(const f32x4 *)p, s.x0);
        s.x1 = fma4(f, *(const f32x4 *)(p + 4), s.x1);
      }
      return s;
    };
    auto store = [&](int it, const KvSum &s) {
      const int r = it / kChunks, ch = it % kChunks, rr = r0 + r;
      const int q = rr / G;
      store_row<DT>(a, b, q, hk * G + (rr - q * G), d_lo + 8 * ch, s, ch == 0 && sl == 0);
    };
    if constexpr (SEQ) {
      const bool mine = tid < kKvRows * kChunks && r0 + tid / kChunks < rows;
      if (mine) add_keys(total, sum(tid));
      t0 = t1;
      if (t0 >= n_tiles) {
        if (mine) store(tid, total);
        break;
      }
      t1 = min(n_tiles, t0 + per_split);
      __syncthreads();  // the parked sums have been read
    } else {
      for (int it = tid; it < kKvRows * kChunks; it += W * 64) {
        const int r = it / kChunks, ch = it % kChunks;
        if (r0 + r >= rows) continue;
        const KvSum s = sum(it);
        if (a.kv_splits > 1) {
          const size_t pr = (((size_t)bh * a.q_blocks + rb) * a.kv_splits + split) * kKvRows + r;
          float *x = a.part + pr * (slices * NDB * 32) + d_lo + 8 * ch;
          *(f32x4 *)x = s.x0;
          *(f32x4 *)(x + 4) = s.x1;
          if (ch == 0 && sl == 0) *(f32x2 *)(a.part_ml + 2 * pr) = f32x2{s.m, s.l};
        } else {
          store(it, s);
        }
      }
      break;
    }
  }
}

// The key splits' sums of every row, in split order. One thread per (row, 4 dims); a row's partials are
// read once. The latency of these reads and the additions of the one or two wavefronts of a row bound it.
// 32 splits of 32 rows, D 128: 4.3 us with 16 splits in flight and one wavefront per workgroup (8 dims per thread:
// 4.9, 8 splits and four wavefronts: 6.8), 16 splits: 3.8 (3.9, 4.6).
template <int DT>
__device__ __forceinline__ void attn_kv_combine(const mtk_attn_kargs &a) {
  const int G = a.H / a.H_kv, rows = a.S_q * G, D = a.D, chunks = D / 4, S = a.kv_splits;
  const long long n = (long long)a.B * a.H_kv * rows * chunks;
  const long long it = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (it >= n) return;
  const int ch = (int)(it % chunks);
  const int rall = (int)(it / chunks);
  const int bh = rall / rows, rr = rall - bh * rows;
  const int b = bh / a.H_kv, hk = bh - b * a.H_kv;
  const size_t pr0 = ((size_t)bh * a.q_blocks + rr / kKvRows) * S * kKvRows + rr % kKvRows;
  const float *ml = a.part_ml + 2 * pr0;
  const float *x = a.part + pr0 * a.part_ld + 4 * ch;
  KvSum total;
  constexpr int kAhead = 16;  // splits whose partials are in flight at once
  for (int s0 = 0; s0 < S; s0 += kAhead) {
    KvSum t[kAhead];  // past the last split: no keys, which add nothing
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
      if (s0 + i < S) {
        const f32x2 e = *(const f32x2 *)(ml + (size_t)(s0 + i) * 2 * kKvRows);
        t[i] = KvSum{e.x, e.y, *(const f32x4 *)(x + (size_t)(s0 + i) * kKvRows * a.part_ld)};
      }
#pragma unroll
    for (int i = 0; i < kAhead; i += 4) {  // few splits: no more than the last four are padding
      if (s0 + i >= S) break;
#pragma unroll
      for (int j = 0; j < 4; ++j) add_keys(total, t[i + j]);
    }
  }
  const int q = rr / G;
  store_row<DT, 4>(a, b, q, hk * G + (rr - q * G), 4 * ch, total, ch == 0);
}

}  // namespace mtk

using namespace mtk;

extern "C" __global__ void __launch_bounds__(64) mtk_attn_kv_combine_f16(const mtk_attn_kargs a) {
  attn_kv_combine<DT_F16>(a);
}
extern "C" __global__ void __launch_bounds__(64) mtk_attn_kv_combine_bf16(const mtk_attn_kargs a) {
  attn_kv_combine<DT_BF16>(a);
}

#define MTK_ATTN_KV_KERNEL_(NAME, DT, DP, NDB, W, SEQ)                                                       \
  extern "C" __global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(W / 4, W / 4))) \
  NAME(const mtk_attn_kargs a) { attn_kv<DT, DP, NDB, W, SEQ>(a); }
#define MTK_ATTN_KV_KERNEL(NAME, DP, NDB, W)                             \
  MTK_ATTN_KV_KERNEL_(NAME##_f16, DT_F16, DP, NDB, W, false)             \
  MTK_ATTN_KV_KERNEL_(NAME##_bf16, DT_BF16, DP, NDB, W, false)
// with the splits in turn
#define MTK_ATTN_KV_SEQ_KERNEL(NAME, DP, NDB, W)                         \
  MTK_ATTN_KV_KERNEL_(NAME##_seq_f16, DT_F16, DP, NDB, W, true)          \
  MTK_ATTN_KV_KERNEL_(NAME##_seq_bf16, DT_BF16, DP, NDB, W, true)

// mtk_attn_kv_d<DP>_<32-dim blocks per workgroup>[_seq]_<type>
MTK_ATTN_KV_KERNEL(mtk_attn_kv_d64_2, 64, 2, 8)
MTK_ATTN_KV_KERNEL(mtk_attn_kv_d64_1, 64, 1, 8)
MTK_ATTN_KV_KERNEL(mtk_attn_kv_d128_4, 128, 4, 8)
MTK_ATTN_KV_KERNEL(mtk_attn_kv_d128_2, 128, 2, 8)
MTK_ATTN_KV_KERNEL(mtk_attn_kv_d128_1, 128, 1, 8)
MTK_ATTN_KV_KERNEL(mtk_attn_kv_d256_4, 256, 4, 4)
MTK_ATTN_KV_KERNEL(mtk_attn_kv_d256_2, 256, 2, 4)
// two or more splits leave at most half of the CUs' worth of workgroups with all blocks, so that the
// kernels with fewer are taken where one workgroup walks them
MTK_ATTN_KV_SEQ_KERNEL(mtk_attn_kv_d64_1, 64, 1, 8)
MTK_ATTN_KV_SEQ_KERNEL(mtk_attn_kv_d128_2, 128, 2, 8)
MTK_ATTN_KV_SEQ_KERNEL(mtk_attn_kv_d128_1, 128, 1, 8)
MTK_ATTN_KV_SEQ_KERNEL(mtk_attn_kv_d256_2, 256, 2, 4)
