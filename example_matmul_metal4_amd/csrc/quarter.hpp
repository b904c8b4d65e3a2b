// GEMM for tile grids that leave most of the device idle: the four 64x64 quarters of a 128x128 tile
// as workgroups of their own, and the K-tiles of each split over the workgroup's W wavefronts.
//
// With one 128x128 tile per CU or fewer, a K loop that all wavefronts walk together costs one memory
// latency per K-tile (about 1.5 us: 1023 cubed has 64 tiles of 16 K-tiles, 31 us for 2.1 GFLOP). Here
//   * every wavefront takes every W-th K-tile of 64 for the whole 64x64 quarter (2 x 2 blocks of
//     32x32x16 MFMAs: one fragment read per MFMA; 96x64: 3 x 2), staged global -> registers -> its own
//     16 KB (20 KB) of LDS: no barrier until the end, and the loads of its next tile in flight meanwhile
//     (two tiles ahead was slower: registers, 18.4 -> 19.5 us at 1024 x 1024 x 4096);
//   * the wavefronts' sums are parked in LDS and added in wavefront order, in fp32.
// Operands stay as stored: rows along K are staged as in the tile kernels and read with 16-byte
// fragment reads, K-major operands with transposed reads. ANY: rows at any 2-byte alignment.
#pragma once

#include "tile_gemm.hpp"

namespace mtk {

// One operand of a step of 64 K: ROWS rows of 64 K (KMAJOR false) or 64 K rows of 64 columns.
template <bool KMAJOR, bool ANY, int ROWS = 64>
struct QuarterOp {
  static_assert(!KMAJOR || ROWS == 64, "K-major operands are 64 columns wide");
  static constexpr int kRows = ROWS, kLoads = ROWS / 8;
  uint32_t lane_off;  // bytes: this lane's chunk of the first load instruction at K-tile 0
  uint32_t step_i;    // bytes between load instructions (8 rows)
  uint32_t step_k;    // bytes between K-tiles

  // Rows (columns) past the operand's end only reach outputs that are not stored; K past its end is
  // zeroed by store().
  __device__ void init(int lane, int first, int ld, uint32_t mis) {
    const uint32_t row = (uint32_t)(KMAJOR ? lane >> 3 : first + (lane >> 3));
    const uint32_t col = (uint32_t)((KMAJOR ? first : 0) + 8 * (lane & 7));
    lane_off = (row * (uint32_t)ld + col) * 2u + mis;
    step_i = 16u * (uint32_t)ld;
    step_k = KMAJOR ? 128u * (uint32_t)ld : 128u;
  }
  __device__ __forceinline__ void load(rsrc_t r, int kt, int, u32x4 (&v)[kLoads], uint32_t (&e)[kLoads]) const {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const uint32_t off = lane_off + ((uint32_t)i * step_i + (uint32_t)kt * step_k);
      if constexpr (ANY) {
        v[i] = buf_load16(r, off & ~3u);
        e[i] = buf_load4(r, (off & ~3u) + 16u);
      } else {
        v[i] = buf_load16(r, off);
      }
    }
  }
  // The staged chunks to LDS; k: K elements from this K-tile on (< 64: the last, partial one).
  __device__ __forceinline__ void store(char *lds, int lane, int kt, int k, u32x4 (&v)[kLoads],
                                        const uint32_t (&e)[kLoads]) const {
    const int r0 = lane >> 3, c = lane & 7;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      u32x4 w = v[i];
      if constexpr (ANY) {
        const uint32_t sh = ((lane_off + ((uint32_t)i * step_i + (uint32_t)kt * step_k)) & 2u) << 3;
        w = u32x4{__builtin_amdgcn_alignbit(w.y, w.x, sh), __builtin_amdgcn_alignbit(w.z, w.y, sh),
                  __builtin_amdgcn_alignbit(w.w, w.z, sh), __builtin_amdgcn_alignbit(e[i], w.w, sh)};
      }
      const int r = 8 * i + r0;
      if (k < kBK) w = keep_halves(w, KMAJOR ? (r < k ? 8 : 0) : k - 8 * c);
      *(u32x4 *)(lds + (KMAJOR ? (uint32_t)(r * 128 + ((c ^ (4 * ((r >> 1) & 1))) << 4)) : lds_off(r, c))) = w;
    }
  }
  // MFMA operand of 32-row (column) block b at k-step ks (16 K).
  __device__ __forceinline__ u32x4 frag(const char *lds, int lane, int b, int ks) const {
    if constexpr (KMAJOR) {
      // two transposed reads: K rows 16 ks + 8 (lane / 32) + 4 e + (lane % 16) / 4, e = 0, 1; the row
      // swizzle depends on the lane only, block b flips bit 6 of the address
      const int s = lane & 15, h = lane >> 4;
      const int d = 16 * (h & 1) + 4 * (s & 3), r = 8 * (h >> 1) + (s >> 2);
      const char *p = lds + ((r * 128 + (((d >> 3) ^ (4 * ((r >> 1) & 1))) << 4) + 2 * (d & 7)) ^ (64 * b)) + 2048 * ks;
      const s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)p);
      const s16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(p + 512));
      const u32x2 v = __builtin_bit_cast(u32x2, x), w = __builtin_bit_cast(u32x2, y);
      return u32x4{v.x, v.y, w.x, w.y};
    } else {
      return *(const u32x4 *)(lds + frag_off(32 * b, ks, lane));
    }
  }
};

// The activation of an implicit-GEMM convolution as the row operand: row m is output pixel (n, oz, oh,
// ow), K element ((kd * KH + kh) * KW + kw) * C + c. With C a multiple of 8 a chunk of 8 lies in one
// filter tap: every lane decodes its chunk's tap once per K-tile and adds it to its 8 rows' window
// origins; rows for which that tap lies in the padding (one bit per tap and dimension, up to 10 taps
// each) and chunks past K are loaded out of range, as zeros.
template <bool ANY>
struct QuarterConv {
  static constexpr int kRows = 64, kLoads = 8;
  const mtk_tile_args &a;
  int base[8];       // element offset of the row's window origin (may be negative)
  uint32_t taps[8];  // in-range taps: depth | height << 10 | width << 20
  uint32_t mis;

  template <typename D>
  static __device__ __forceinline__ int div(int n, const D &d) {
    return d.mul ? (int)(__umulhi((uint32_t)n, d.mul) >> d.shift) : n;
  }
  __device__ void init(int lane, int first, int, uint32_t m) {
    mis = m;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = first + 8 * i + (lane >> 3);
      const int t1 = div(row, a.dOW), ow = row - t1 * a.cOW;
      const int t2 = div(t1, a.dOH), oh = t1 - t2 * a.cOH;
      const int n = div(t2, a.dOD), oz = t2 - n * a.cOD;
      const int iz = oz * a.cSZ - a.cPF, ih = oh * a.cSY - a.cPT, iw = ow * a.cSX - a.cPL;
      uint32_t t = 0;
      for (int k = 0; k < a.cKD; ++k) t |= (uint32_t)((uint32_t)(iz + k * a.cDZ) < (uint32_t)a.cD) << k;
      for (int k = 0; k < a.cKH; ++k) t |= (uint32_t)((uint32_t)(ih + k * a.cDY) < (uint32_t)a.cH) << (10 + k);
      for (int k = 0; k < a.cKW; ++k) t |= (uint32_t)((uint32_t)(iw + k * a.cDX) < (uint32_t)a.cW) << (20 + k);
      taps[i] = row < a.M ? t : 0;
      base[i] = (((n * a.cD + iz) * a.cH + ih) * a.cW + iw) * a.cC;
    }
  }
  __device__ __forceinline__ void load(rsrc_t r, int kt, int lane, u32x4 (&v)[8], uint32_t (&e)[8]) const {
    const int k = kt * kBK + 8 * (lane & 7);
    const int tap = div(k, a.dC), c = k - tap * a.cC;
    const int t = div(tap, a.dKW), kw = tap - t * a.cKW;
    const int kd = div(t, a.dKH), kh = t - kd * a.cKH;
    const int at = ((kd * a.cDZ * a.cH + kh * a.cDY) * a.cW + kw * a.cDX) * a.cC + c;
    const uint32_t need = k < a.K ? 1u << kd | 1u << (10 + kh) | 1u << (20 + kw) : ~0u;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t off = (taps[i] & need) == need ? (uint32_t)(base[i] + at) * 2u : kOOBAny;
      v[i] = buf_load16(r, off);
      if constexpr (ANY) e[i] = buf_load4(r, off + 16u);
    }
  }
  __device__ __forceinline__ void store(char *lds, int lane, int, int, u32x4 (&v)[8], const uint32_t (&e)[8]) const {
    const int r0 = lane >> 3, c = lane & 7;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      u32x4 w = v[i];
      if constexpr (ANY) {  // chunks are 16 bytes apart: all as the activation itself starts
        const uint32_t sh = mis << 3;
        w = u32x4{__builtin_amdgcn_alignbit(w.y, w.x, sh), __builtin_amdgcn_alignbit(w.z, w.y, sh),
                  __builtin_amdgcn_alignbit(w.w, w.z, sh), __builtin_amdgcn_alignbit(e[i], w.w, sh)};
      }
      *(u32x4 *)(lds + lds_off(8 * i + r0, c)) = w;
    }
  }
  __device__ __forceinline__ u32x4 frag(const char *lds, int lane, int b, int ks) const {
    return *(const u32x4 *)(lds + frag_off(32 * b, ks, lane));
  }
};

template <int DT, class AOp, bool BN, bool ANY, int W>
__device__ __forceinline__ void quarter_tile(const mtk_tile_args &a, AOp oa) {
  constexpr int MB = AOp::kRows / 32;                   // 32-row blocks
  constexpr int kWaveB = (AOp::kRows + 64) * 128;
  constexpr int kPasses = MB * 8192 <= kWaveB ? 1 : 2;  // of the final sum: both column blocks at once, or one each
  __shared__ __attribute__((aligned(1024))) char smem[W * kWaveB];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  const int tiles = a.tiles_m * a.tiles_n;
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int split = id / tiles;
  const int t = id - split * tiles;
  const int group = kGroupM * a.tiles_n;
  const int first_m = (t / group) * kGroupM;
  const int gm = min(a.tiles_m - first_m, kGroupM);
  const int m0 = (first_m + (t % group) % gm) * AOp::kRows, n0 = (t % group) / gm * 64;
  const int kt0 = split_first_tile(a, split, t);
  const int kt1 = split_first_tile(a, split + 1, t);

  uint32_t mis_a = 0, mis_b = 0;
  const rsrc_t ra = ANY ? make_rsrc_any(a.A, a.a_bytes, mis_a) : make_rsrc(a.A, a.a_bytes);
  const rsrc_t rb = ANY ? make_rsrc_any(a.B, a.b_bytes, mis_b) : make_rsrc(a.B, a.b_bytes);
  QuarterOp<BN, ANY> ob;
  oa.init(lane, m0, a.lda, mis_a);
  ob.init(lane, n0, a.ldb, mis_b);
  char *la = smem + wave * kWaveB, *lb = la + AOp::kRows * 128;

  f32x16 acc[MB][2] = {};
  u32x4 sa[AOp::kLoads], sb[8];
  uint32_t ea[AOp::kLoads], eb[8];
  int kt = kt0 + wave;
  if (kt < kt1) {
    oa.load(ra, kt, lane, sa, ea);
    ob.load(rb, kt, lane, sb, eb);
  }
  for (; kt < kt1; kt += W) {
    oa.store(la, lane, kt, a.K - kt * kBK, sa, ea);
    ob.store(lb, lane, kt, a.K - kt * kBK, sb, eb);
    if (kt + W < kt1) {
      oa.load(ra, kt + W, lane, sa, ea);
      ob.load(rb, kt + W, lane, sb, eb);
    }
    // this wavefront's own region: LDS accesses of a wavefront complete in order, the compiler has to
    // keep the reads of other lanes' chunks behind the writes
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int ks = 0; ks < kBK / 16; ++ks) {
      u32x4 fa[MB];
#pragma unroll
      for (int i = 0; i < MB; ++i) fa[i] = oa.frag(la, lane, i, ks);
      const u32x4 fb[2] = {ob.frag(lb, lane, 0, ks), ob.frag(lb, lane, 1, ks)};
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma32x32x16<DT>(fa[i], fb[j], acc[i][j]);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }

  // ---- add the wavefronts' sums: accumulator quads parked as [block][quad][lane], 16 bytes each
  constexpr int kCols = 2 / kPasses;  // column blocks per pass
  const uint16_t *bias = (const uint16_t *)a.bias;
#pragma unroll
  for (int pass = 0; pass < kPasses; ++pass) {
    if (pass > 0) __syncthreads();  // the pass before has been read
    f32x4 *park = (f32x4 *)(smem + wave * kWaveB);  // own region
#pragma unroll
    for (int b = 0; b < MB * kCols; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x16 &x = acc[b / kCols][pass + b % kCols];
        park[(4 * b + q) * 64 + lane] = f32x4{x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]};
      }
    __syncthreads();
#pragma unroll
    for (int it = tid; it < MB * kCols * 256; it += 64 * W) {
      f32x4 s = *(const f32x4 *)(smem + it * 16);
#pragma unroll
      for (int w = 1; w < W; ++w) s += *(const f32x4 *)(smem + w * kWaveB + it * 16);
      const int b = it >> 8, q = (it >> 6) & 3, l = it & 63;
      const int row = m0 + 32 * (b / kCols) + 8 * q + 4 * (l >> 5);
      const int col = n0 + 32 * (pass + b % kCols) + (l & 31);
      if (col >= a.N) continue;
      const float v[4] = {s.x, s.y, s.z, s.w};
      if (a.partial != nullptr) {
        float *P = a.partial + (size_t)split * a.M * a.N + col;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (row + r < a.M) P[(size_t)(row + r) * a.N] = v[r];
      } else {
        const float bv = a.has_bias ? from_bits<DT>(bias[col]) : 0.0f;
        uint16_t *C = (uint16_t *)a.C + col;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (row + r < a.M) C[(size_t)(row + r) * a.ldc] = to_bits<DT>(v[r] + bv);
      }
    }
  }
}

template <int DT, bool AT, bool BN, bool ANY, int W>
__device__ __forceinline__ void quarter_gemm(const mtk_tile_args &a) {
  quarter_tile<DT, QuarterOp<AT, ANY>, BN, ANY, W>(a, QuarterOp<AT, ANY>{});
}

// 96 rows of A [M][K] per workgroup, for M where one or two such tiles replace two or three of 64 (B is read
// once for more rows). HBM and the L2 reads of A bound it: 20 KB per K-tile and CU, 8 in flight (160 KB of
// LDS, 254 VGPRs; a spill in the loop waits for the loads in flight: 41 us instead of 33). 77 x 4096 x 14336,
// bf16: 38.0 us on 128x128 tiles, 39.6 on 64x64 quarters -> 33.0.
template <int DT, bool BN, int ROWS, int W>
__device__ __forceinline__ void quarter_tall(const mtk_tile_args &a) {
  using A = QuarterOp<false, false, ROWS>;
  quarter_tile<DT, A, BN, false, W>(a, A{});
}

// Convolution: weights [K][O] as the K-major operand.
template <int DT, bool ANY, int W>
__device__ __forceinline__ void quarter_conv(const mtk_tile_args &a) {
  quarter_tile<DT, QuarterConv<ANY>, true, ANY, W>(a, QuarterConv<ANY>{a});
}

}  // namespace mtk
