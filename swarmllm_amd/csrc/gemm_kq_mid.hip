// gemm_kq_mid.hip — Q4_K and Q6_K products of 17 to 128 activation rows (Q6_K
// to 256) on the int8 matrix cores of gfx950: short prompts, large batches.
//
// dst[m][n] = sum over super-blocks of candle's Q4_K / Q6_K x Q8_K vec_dot
// (vendor/candle/candle-core/src/quantized/k_quants.rs:2031-2111, 2598-2655)
// against the activation quantized as the reference quantizes it
// (BlockQ8K::from_float, :2882-2927): per-256 scale dy, int8 codes y, code
// sums S of 16 values.
//
// Exact integers. Q4_K: sc q (10 bits) enters as two int8 operands, sc =
// 8 sh + sl, sh q and sl q <= 105 (one packed 16-bit multiply makes four of
// them: the products stay inside their bytes), T = 8 T_h + T_l; the min sums
// Tm = sum_j m_j S_j run on one f16 product of small integers (S of 16 values
// and m_j are exact in f16, every sum stays below 2^24). Q6_K: p = sc (q - 32)
// (14 bits) enters as the high byte h and the low byte minus 128, l, of
// 4p + 128: 256 T_h + T_l = 4 sum p y. The f32 epilogue of a super-block is
// acc += dy (d T - dmin Tm), Q6_K acc += dy (d/4 T).
//
// What bounds these products is getting the weight to enough CUs: at 17-128
// rows a weight's bytes (33 MB for 14336 x 4096: 7 us at the 4.8 TB/s a copy
// reaches) and its MFMAs (MT row tiles x 17 x 32 cycles a super-block of 32
// weight rows) are both a few microseconds, while a tile that walks all of K
// alone takes 2 us a super-block (the tiled GEMMs, uncut, at 77 rows: q, k, v
// and o 36 us each, gate and up 39 each, the Q6_K down 110). So K is cut: a workgroup takes
// 128 weight rows, up to 96 activation rows (MT tiles of 32: below 97 rows a
// weight byte is read and expanded once) and one of S ranges of super-blocks; its partial
// goes to a slot and a second launch adds the slots in split order.
//
// Workgroup: 4 waves, each 32 weight rows x MT tiles of
// v_mfma_i32_32x32x32_i8 (one MFMA per 32-value group, tile and operand).
//   - The activation codes of a super-block (32 MT rows x 256 B, pieces
//     XOR-swizzled by row) reach LDS by direct copies, one super-block ahead,
//     double-buffered; the code sums (as f16) and dy through registers.
//   - A wave's weight bytes (32 rows' blocks as their aligned 16-byte
//     pieces) are loaded one super-block ahead into registers, consecutive
//     lanes on consecutive pieces, and written to the wave's own LDS slot
//     when the current super-block is done; lanes read their row back.
//     Q4_K's rows lie 144 bytes apart there, Q6_K's 240 (both spread 16 rows
//     over the banks).
// Rows past M and weight rows past N are read as the last row (valid memory);
// their outputs are never stored.
//
// Measured at 77 rows (an 8B layer, slots added in): q + k + v 24 us, o 19,
// gate + up with its GLU 45, down 34; at 21 rows gate + up with its GLU 28 (the
// two-row-tile few-row kernel before: 54; it keeps the others). At 21 rows gate + up
// reads HBM at 4.9 TB/s, 1.5 x its weight bytes (the 64-byte sector at each
// 144-byte block's edges is fetched twice); at 77 the vector unit is busy 41%
// and the matrix cores 30% of the time. The weight loads are nontemporal:
// plain ones took 50 us at 21 rows, 62 at 77. A second super-block of
// weights in flight changed nothing.
//
// Without room for the slots one workgroup computes a tile's splits one after
// another and adds each to dst, the same sums in the same order (a route for
// the products no other kernel runs faster then: launch_mid_without_slots).
#include "lds_copy.h"
#include "mv_common.h"
#include "qmm_device.h"
#include "qmm_launch.h"

namespace qmm {

namespace {

typedef int i4v __attribute__((ext_vector_type(4)));
typedef int i16v __attribute__((ext_vector_type(16)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pkmul(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b)));
}
__device__ __forceinline__ uint32_t pkmad(uint32_t a, uint32_t b, uint32_t c) {
  return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b) +
                                               __builtin_bit_cast(u16x2, c)));
}

constexpr int kNW = 4, BN = 32 * kNW;  // waves of a workgroup, 32 weight rows each

struct MidArgs {
  const void* w[kMaxTargets];
  float* dst[kMaxTargets];
  int64_t ldd[kMaxTargets];
  int64_t n[kMaxTargets];
  int unit_end[kMaxTargets];      // workgroups of weights 0..t
  int splits[kMaxTargets];        // K ranges of weight t
  int64_t part_off[kMaxTargets];  // its slots in `part` (floats): [split][M][n]
  const int8_t* yq;
  const float* yd;
  const int16_t* ybs;
  float* part;  // null: uncut, a workgroup walks a tile's splits in turn
  int M, nsb, remap;
  int chunks, per;  // row chunks of `per` rows (the last perhaps fewer)
};

template <int FMT>
struct MidFmt {
  static constexpr bool kQ6 = FMT == T_Q6_K;
  static constexpr int kBlock = kQ6 ? 210 : 144;
  static constexpr int kPieces = kQ6 ? 14 : 9;              // aligned pieces around a row's block
  static constexpr int kStride = kQ6 ? 240 : 144;           // LDS bytes a row
  static constexpr int kLoads = (32 * kPieces + 63) / 64;   // a wave's 64-lane loads a super-block
  static constexpr int kSlot = 32 * kStride + (kQ6 ? 16 : 0);
};

template <int FMT, int MT>
__global__ __launch_bounds__(64 * kNW, 2) void gemm_kq_mid_kernel(const MidArgs a) {
  using F = MidFmt<FMT>;
  constexpr bool Q6 = F::kQ6;
  constexpr int kRows = 32 * MT, kThreads = 64 * kNW;
  constexpr int kACopies = 8 * MT / kNW;  // a wave's 1 KB activation copies a super-block
  static_assert(8 * MT % kNW == 0 && 2 * kRows <= kThreads, "copy shapes");
  __shared__ __attribute__((aligned(1024))) int8_t s_a[2][kRows * 256];
  __shared__ __attribute__((aligned(16))) uint8_t s_w[kNW][F::kSlot];
  __shared__ __attribute__((aligned(16))) _Float16 s_bs[2][Q6 ? 1 : kRows][16];
  __shared__ __attribute__((aligned(16))) float s_dy[2][kRows];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, r32 = lane & 31;

  const int total = (int)gridDim.x;
  const int b = (int)blockIdx.x;
  const int idx = a.remap ? (b & 7) * (total >> 3) + (b >> 3) : b;
  const int t = idx < a.unit_end[0] ? 0 : idx < a.unit_end[1] ? 1 : idx < a.unit_end[2] ? 2 : 3;
  auto pick = [&](const auto& arr) { return t == 0 ? arr[0] : t == 1 ? arr[1] : t == 2 ? arr[2] : arr[3]; };
  const int loc0 = idx - (t == 0 ? 0 : t == 1 ? a.unit_end[0] : t == 2 ? a.unit_end[1] : a.unit_end[2]);
  const int64_t N = pick(a.n);
  const int S = pick(a.splits);
  const int nsb = a.nsb;
  // the row chunk: consecutive workgroups share a weight tile
  const int m0 = (loc0 % a.chunks) * a.per;
  const int M = a.M - m0 < a.per ? a.M - m0 : a.per, loc = loc0 / a.chunks;
  const int ctiles = (int)((N + BN - 1) / BN);
  const bool cut = a.part != nullptr;
  const int ct = cut ? loc % ctiles : loc;
  const int s0 = cut ? loc / ctiles : 0, s1 = cut ? s0 + 1 : S;
  const uint8_t* __restrict__ W = (const uint8_t*)pick(a.w);
  const int8_t* __restrict__ yq = a.yq + (int64_t)m0 * nsb * 256;
  const float* __restrict__ yd = a.yd + (int64_t)m0 * nsb;
  const int16_t* __restrict__ ybs = a.ybs + (int64_t)m0 * nsb * 16;
  const int64_t n0 = (int64_t)ct * BN;
  const uint32_t K = (uint32_t)nsb * 256u;
  const uint32_t rowbytes = (uint32_t)nsb * F::kBlock;

  // activation copies: copy i moves rows 4i .. 4i+3; lane L writes row
  // 4i + L/16 at piece position L%16, which holds code piece (L%16) ^ (row & 15)
  uint32_t aoff[kACopies];
#pragma unroll
  for (int u = 0; u < kACopies; u++) {
    const int row = 4 * (wv + kNW * u) + (lane >> 4);
    aoff[u] = (uint32_t)(row < M ? row : M - 1) * K + 16u * (((uint32_t)lane & 15u) ^ ((uint32_t)row & 15u));
  }
  auto copy_a = [&](int sb, int buf) {
#pragma unroll
    for (int u = 0; u < kACopies; u++)
      dma16(yq + 256 * (int64_t)sb, aoff[u], lds_addr(&s_a[buf][1024 * (wv + kNW * u)]));
  };
  // weight pieces: piece f = 64u + lane of the wave's 32 rows (row f / kPieces)
  uint32_t woff[F::kLoads];
#pragma unroll
  for (int u = 0; u < F::kLoads; u++) {
    uint32_t f = 64u * (uint32_t)u + (uint32_t)lane;
    if (f > 32u * F::kPieces - 1u) f = 32u * F::kPieces - 1u;
    const uint32_t row = f / (uint32_t)F::kPieces;
    const int64_t gr = n0 + 32 * wv + row < N ? n0 + 32 * wv + row : N - 1;
    woff[u] = (uint32_t)gr * rowbytes + 16u * (f - (uint32_t)F::kPieces * row);
  }
  uint4 wr[F::kLoads];
  auto load_w = [&](int sb) {
#pragma unroll
    for (int u = 0; u < F::kLoads; u++) {
      if constexpr (Q6)
        wr[u] = ld_stream16(W + ((woff[u] + 210u * (uint32_t)sb) & ~15u));
      else
        wr[u] = ld_stream16(W + 144 * (int64_t)sb + woff[u]);
    }
  };
  auto store_w = [&]() {
#pragma unroll
    for (int u = 0; u < F::kLoads; u++) {
      uint32_t f = 64u * (uint32_t)u + (uint32_t)lane;
      if (32 * F::kPieces % 64 != 0 && u == F::kLoads - 1 && f > 32u * F::kPieces - 1u) f = 32u * F::kPieces - 1u;
      if constexpr (Q6) f += f / (uint32_t)F::kPieces;  // 15 pieces a row in LDS
      *(uint4*)&s_w[wv][16u * f] = wr[u];
    }
  };
  // code sums and dy: thread -> (row, half) and row, threads past them
  // repeating the first ones' (no branch in a step)
  const int bt = tid % (2 * kRows), dt = tid % kRows;
  const int brow = (bt >> 1) < M ? bt >> 1 : M - 1;
  const int drow = dt < M ? dt : M - 1;
  uint4 bs = {};
  float dyr = 0.0f;
  auto load_rows = [&](int sb) {
    if (!Q6) bs = *(const uint4*)(ybs + (int64_t)brow * (K / 16) + 16 * sb + 8 * (bt & 1));
    dyr = yd[(int64_t)drow * nsb + sb];
  };
  auto store_rows = [&](int buf) {
    if (!Q6) {
      const uint32_t w4[4] = {bs.x, bs.y, bs.z, bs.w};
      h8 v;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        v[2 * i] = (_Float16)(int16_t)(w4[i] & 0xFFFFu);
        v[2 * i + 1] = (_Float16)(int16_t)(w4[i] >> 16);
      }
      *(h8*)&s_bs[buf][bt >> 1][8 * (bt & 1)] = v;
    }
    s_dy[buf][dt] = dyr;
  };

  // the lane's weight row in its wave's slot (Q6_K: its block starts at byte
  // (wbase + 210 sb) mod 16 of it), and its activation row's operand address
  const uint8_t* wrow = &s_w[wv][r32 * F::kStride];
  const int64_t grow = n0 + 32 * wv + r32 < N ? n0 + 32 * wv + r32 : N - 1;
  const uint32_t wbase = (uint32_t)grow * rowbytes;
  const uint32_t fa0 = 256u * (uint32_t)r32 + 16u * ((uint32_t)h ^ ((uint32_t)r32 & 15u));

  f16v acc[MT];
  float* __restrict__ dst = pick(a.dst);
  const int64_t ldd = pick(a.ldd);
  const int64_t col = n0 + 32 * wv + r32;

  for (int s = s0; s < s1; s++) {
    const int sb0 = s * nsb / S, sb1 = (s + 1) * nsb / S;
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
      for (int i = 0; i < 16; i++) acc[m][i] = 0.0f;
    copy_a(sb0, 0);
    load_w(sb0);
    load_rows(sb0);
    store_w();
    store_rows(0);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();

    for (int sb = sb0; sb < sb1; sb++) {
      const int cur = (sb - sb0) & 1;
      const int nx = sb + 1 < sb1 ? sb + 1 : sb;  // past the last super-block, the last one's again
      copy_a(nx, cur ^ 1);
      load_w(nx);
      load_rows(nx);

      const int8_t* sa = s_a[cur];
      i16v th[MT], tl[MT];
      h8 mb = {};
      float d = 0.0f, dmin = 0.0f;
      auto afrag = [&](int j, int m) -> i4v { return *(const i4v*)(sa + (fa0 ^ (32u * (uint32_t)j)) + 8192 * m); };
      // The eight 32-value groups, both operands, against every row tile. Group
      // j + 1's operands are made under group j's MFMAs: a tile's activation
      // fragment is read into its registers as soon as its MFMAs have issued.
      auto groups = [&](auto&& prepare, auto&& build) {
        const i16v zero = {};
        i4v af[MT], bh = {}, bl = {};
        prepare(0);
#pragma unroll
        for (int m = 0; m < MT; m++) af[m] = afrag(0, m);
        build(0, bh, bl);
#pragma unroll
        for (int j = 0; j < 8; j++) {
          i4v nh = {}, nl = {};
          if (j < 7) prepare(j + 1);
#pragma unroll
          for (int m = 0; m < MT; m++) {
            th[m] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[m], bh, j == 0 ? zero : th[m], 0, 0, 0);
            tl[m] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[m], bl, j == 0 ? zero : tl[m], 0, 0, 0);
            if (j < 7) af[m] = afrag(j + 1, m);
          }
          if (j < 7) build(j + 1, nh, nl);
          bh = nh;
          bl = nl;
          if constexpr (MT > 1) __builtin_amdgcn_sched_barrier(0);
        }
      };
      if constexpr (!Q6) {
        const uint4 hdr = *(const uint4*)wrow;
        d = h2f((uint16_t)(hdr.x & 0xFFFFu));
        dmin = h2f((uint16_t)(hdr.x >> 16));
        // 6-bit scales and mins (get_scale_min_k4, vendor/candle/candle-core/src/quantized/utils.rs:50-60)
        const uint32_t sc[2] = {hdr.y & 0x3f3f3f3fu, (hdr.w & 0x0f0f0f0fu) | (((hdr.y >> 6) & 0x03030303u) << 4)};
        const uint32_t mn = h ? ((hdr.w >> 4) & 0x0f0f0f0fu) | (((hdr.z >> 6) & 0x03030303u) << 4)
                              : hdr.z & 0x3f3f3f3fu;
        const uint32_t sl[2] = {sc[0] & 0x07070707u, sc[1] & 0x07070707u};
        const uint32_t sh[2] = {(sc[0] >> 3) & 0x07070707u, (sc[1] >> 3) & 0x07070707u};
        // Tm: K slots 8h .. 8h+7 hold the 16-value sums 8h .. and m_j twice each
#pragma unroll
        for (int i = 0; i < 4; i++) {
          // 1024 + m as f16 bits twice, minus 1024: exact
          const h2v v = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, mn, 0x04000400u + 0x00010001u * i)) -
                        (h2v){(_Float16)1024.0f, (_Float16)1024.0f};
          mb[2 * i] = v[0];
          mb[2 * i + 1] = v[1];
        }
        uint4 raw[2];
        auto prepare = [&](int j) {  // the codes of groups j, j + 1 (low and high nibbles)
          if (j % 2 == 0) raw[(j >> 1) & 1] = *(const uint4*)(wrow + 16 + 16 * j + 16 * h);
        };
        auto build = [&](int j, i4v& bh, i4v& bl) {
          const uint4& r = raw[(j >> 1) & 1];
          const uint32_t rw[4] = {r.x, r.y, r.z, r.w};
          const uint32_t sel = 0x0C000C00u + 0x00010001u * (uint32_t)(j & 3);
          const uint32_t hj = __builtin_amdgcn_perm(0u, sh[j >> 2], sel);
          const uint32_t lj = __builtin_amdgcn_perm(0u, sl[j >> 2], sel);
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const uint32_t q = (j & 1 ? rw[e] >> 4 : rw[e]) & 0x0F0F0F0Fu;
            bh[e] = (int)pkmul(q, hj);
            bl[e] = (int)pkmul(q, lj);
          }
        };
        groups(prepare, build);
      } else {
        const int o = (int)((wbase + 210u * (uint32_t)sb) & 15u);
        uint32_t scw[4], ql[2][4], qh[4];
        lds_words<4>(wrow, o + 192, scw);
        d = 0.25f * h2f((uint16_t)lds_u16(wrow, o + 208));
        auto prepare = [&](int j) {  // the code bytes of groups 4 (j / 4) .. + 3
          if (j % 4 != 0) return;
          const int hf = j >> 2;
          lds_words<4>(wrow, o + 64 * hf + 16 * h, ql[0]);
          lds_words<4>(wrow, o + 64 * hf + 32 + 16 * h, ql[1]);
          lds_words<4>(wrow, o + 128 + 32 * hf + 16 * h, qh);
        };
        auto build = [&](int j, i4v& bh, i4v& bl) {
          const int hf = j >> 2, gi = j & 3;
          // scale of 16-value group 8 hf + 2 gi + h
          const uint32_t sw = scw[2 * hf + (gi >> 1)];
          const int sc = (int)(int8_t)((sw >> (16 * (gi & 1) + 8 * h)) & 0xFFu);
          const uint32_t sc4 = ((uint32_t)(4 * sc) & 0xFFFFu) * 0x10001u;
          const uint32_t kb = ((uint32_t)(128 - 128 * sc) & 0xFFFFu) * 0x10001u;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const uint32_t q =
                ((ql[gi & 1][e] >> (4 * (gi >> 1))) & 0x0F0F0F0Fu) | (((qh[e] >> (2 * gi)) & 0x03030303u) << 4);
            const uint32_t pe = pkmad(q & 0x00FF00FFu, sc4, kb);
            const uint32_t po = pkmad((q >> 8) & 0x00FF00FFu, sc4, kb);
            bh[e] = (int)__builtin_amdgcn_perm(po, pe, 0x07030501u);
            bl[e] = (int)(__builtin_amdgcn_perm(po, pe, 0x06020400u) ^ 0x80808080u);
          }
        };
        groups(prepare, build);
      }
      // acc += dy (d T - dmin Tm)
#pragma unroll
      for (int m = 0; m < MT; m++) {
        f16v tm = {};
        if constexpr (!Q6)
          tm = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const h8*)&s_bs[cur][32 * m + r32][8 * h], mb, tm, 0, 0, 0);
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const f4v dy4 = *(const f4v*)&s_dy[cur][32 * m + 8 * g + 4 * h];
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const int i = 4 * g + e;
            const int tt = (int)(((uint32_t)th[m][i] << (Q6 ? 8 : 3)) + (uint32_t)tl[m][i]);
            float u;
            if constexpr (Q6)
              u = d * (float)tt;
            else
              u = __builtin_fmaf(d, (float)tt, -(dmin * tm[i]));
            acc[m][i] = __builtin_fmaf(dy4[e], u, acc[m][i]);
          }
        }
        // consumed here: the compiler would sink the epilogue past the barrier, holding every tile's tm
#pragma unroll
        for (int i = 0; i < 16; i++) asm volatile("" ::"v"(acc[m][i]));
      }
      // the next super-block's bytes, in flight since this one's start
      store_w();
      store_rows(cur ^ 1);
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
    }

    if (col < N) {
      float* __restrict__ out = cut ? a.part + pick(a.part_off) + ((int64_t)s * a.M + m0) * N + col : dst + m0 * ldd + col;
      int64_t ldo = cut ? N : ldd;
      int hrow = 4 * h;
      // the rows and their addresses are formed here, not kept live over the K loop
      asm volatile("" : "+s"(ldo), "+v"(hrow));
      const bool add = !cut && s > 0;
#pragma unroll
      for (int m = 0; m < MT; m++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          float old[4] = {};
          if (add) {
#pragma unroll
            for (int e = 0; e < 4; e++)
              if (32 * m + 8 * g + hrow + e < M) old[e] = out[(32 * m + 8 * g + hrow + e) * ldo];
          }
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (32 * m + 8 * g + hrow + e < M)
              out[(32 * m + 8 * g + hrow + e) * ldo] = add ? old[e] + acc[m][4 * g + e] : acc[m][4 * g + e];
        }
    }
  }
}

// dst of the cut weights: the slots added in split order, 4 neighbouring
// columns a thread where every row of the slots and of dst is 16-byte
// aligned, else one. blockIdx.y: the weight.
__global__ __launch_bounds__(256) void gemm_kq_mid_sum_kernel(const MidArgs a) {
  const int t = (int)blockIdx.y;
  auto pick = [&](const auto& arr) { return t == 0 ? arr[0] : t == 1 ? arr[1] : t == 2 ? arr[2] : arr[3]; };
  const int64_t N = pick(a.n), ldd = pick(a.ldd), total = N * a.M;
  const int S = pick(a.splits);
  float* __restrict__ dst = pick(a.dst);
  const float* __restrict__ p = a.part + pick(a.part_off);
  const uint32_t n32 = (uint32_t)N;  // total < 2^31 (launch_mid)
  if ((N & 3) == 0 && (ldd & 3) == 0 && ((uintptr_t)dst & 15) == 0) {
    for (int64_t i = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x); i < total; i += (int64_t)gridDim.x * 1024) {
      f4v v = *(const f4v*)(p + i);
#pragma unroll 4
      for (int s = 1; s < S; s++) v += *(const f4v*)(p + s * total + i);
      const uint32_t r = (uint32_t)i / n32;
      *(f4v*)(dst + r * ldd + ((uint32_t)i - r * n32)) = v;
    }
    return;
  }
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    float v = p[i];
#pragma unroll 4
    for (int s = 1; s < S; s++) v += p[s * total + i];
    const uint32_t r = (uint32_t)i / n32;
    dst[r * ldd + ((uint32_t)i - r * n32)] = v;
  }
}

// Row chunks of at most 96 rows (three tiles: a fourth leaves too few registers
// for the weights in flight), alike in size.
int64_t chunk_rows(int64_t rows) {
  const int64_t c = (rows + 95) / 96;
  return (rows + c - 1) / c;
}

template <int FMT>
void launch_fmt(const MidArgs& a, int units, hipStream_t st) {
  const dim3 grid((unsigned)units);
  if (a.per <= 32)
    gemm_kq_mid_kernel<FMT, 1><<<grid, 64 * kNW, 0, st>>>(a);
  else if (a.per <= 64)
    gemm_kq_mid_kernel<FMT, 2><<<grid, 64 * kNW, 0, st>>>(a);
  else
    gemm_kq_mid_kernel<FMT, 3><<<grid, 64 * kNW, 0, st>>>(a);
}

}  // namespace

// Up to 32 rows the few-row kernels, which need no second launch, keep what
// fills their rounds of the CUs (4096 weight rows each). This kernel against
// them, us, one weight at 17 / 24 / 32 rows:
//   Q4_K  14336 x 4096   20.6 / 21.3 / 22.3 against 22.1 / 25.1 / 27.9
//         28672 x 2048   17.5 / 17.7 / 18.2         33.1 / 36.9 / 38.8
//         28672 x 512     9.7 /  9.5 /  9.8         21.5 / 24.4 / 24.6
//         14336 x 1024   12.6 / 13.0 / 13.8         11.7 / 12.5 / 12.9
//         9216 x 4096    17.2 / 17.6 / 18.3         18.1 / 20.1 / 22.1
//         12288 x 4096   20.2 / 20.3 / 21.2         18.6 / 21.1 / 22.9
//         8192 x 8192    21.8 / 22.5 / 23.8         20.7 / 23.2 / 26.1
//         5120 x 13824   23.3 / 24.3 / 25.3         30.7 / 34.7 / 39.5
//         8192 x 7168    20.7 / 21.7 / 22.7         19.9 / 21.6 / 24.1
//         8192 x 5120    17.2 / 18.0 / 18.8         15.8 / 17.4 / 18.6
//         4096 x 13824   20.8 / 21.4 / 22.2         20.6 / 22.1 / 23.6
//         1024 x 8192    13.3 / 13.8 / 14.0         13.5 / 14.9 / 15.9
//         1024 x 12288   14.8 / 15.1 / 15.5         18.0 / 19.3 / 20.9
//         2048 x 8192    14.1 / 14.6 / 15.3         14.0 / 15.1 / 15.9
//         4096 x 4096    13.4 / 13.8 / 14.9         10.6 / 10.9 / 11.4
//   Q6_K  9216 x 4096    22.4 / 22.6 / 23.4         27.6 / 29.3 / 30.5
//         8192 x 7168    25.3 / 26.2 / 27.4         27.5 / 29.1 / 31.1
//         4096 x 13824   25.1 / 26.0 / 26.8         25.4 / 26.3 / 27.1
// Gate + up with the GLU gain more (Q4_K 13824 x 4096 at 24 rows 53 -> 29), q + k
// + v sets less, and lose where the kernel takes only some of the weights (two
// launches more: 8192, 2048, 2048 x 8192 at 24 rows 33.8 -> 36.8; 6144, 1024, 1024
// x 6144 all here 23.3, all few-row 19.1). So 4097-8192 rows start at k = 7168 and 24
// rows, and the narrow k and v go with their q (8192, 1024, 1024 x 8192 at 24 rows
// all here 30.2, all few-row 32.5, apart 36.3).
static bool few_rows_leave(int type, int64_t n, int64_t k, int64_t rows) {
  constexpr int64_t kLong = (int64_t)4096 * 13824;
  if (n > 16384 || n * k >= 2 * kLong) return true;
  if (n > 12288 || (type == T_Q6_K && n > 8192 && k < 7168)) return k >= 1536;
  if (n <= 1024) return k >= (rows < 24 ? 10752 : 7168);
  if (rows < 24) return false;
  if (n > 8192) return k >= 3072;
  return n > 4096 ? k >= 7168 : n * k >= kLong;
}

// Past 32 rows the tiled Q6_K GEMM, as exact, keeps what fills its tiles of 128
// rows: this kernel against it, us, at 33 / 64 / 96 rows
//   4096 x 1536    15.7 / 17.2 / 20.6 against 18.3 / 18.5 / 19.6
//   8192 x 1536    16.7 / 19.5 / 23.8         18.3 / 18.6 / 19.7
//   8192 x 2560    19.8 / 22.3 / 26.7         26.0 / 26.3 / 28.4
//   14336 x 2048   22.4 / 25.5 / 30.9         22.6 / 22.8 / 24.7
//   14336 x 2560   25.1 / 28.1 / 33.4         26.4 / 27.2 / 29.6
//   14336 x 4096   31.8 / 34.8 / 41.6         38.3 / 38.7 / 42.5
//   18944 x 1536   22.3 / 24.0 / 27.9         32.3 / 33.0 / 35.3
// at 128 rows
//   4096 x 4096 26.2 against 41.6, 8192 x 8192 55 / 77, 14336 x 8192 86 / 78,
//   28672 x 8192 133 / 150, 65536 x 3072 116 / 93
// and, where the single pass does not take them (k no multiple of 2048), at 160
// / 256 rows
//   1024 x 1536 18.4 / 20.2 against 20.0 / 20.2, 4096 x 1536 21.8 / 20.4 against
//   20.2 / 20.5, 4096 x 2560 24.8 / 29.5 against 29.2 / 29.6, 4096 x 11008 48 / 77
//   against 97 / 98, 8192 x 11008 78 / 131 against 98 / 100.
static bool tiled_q6k_keeps(int64_t n, int64_t k, int64_t rows) {
  if (rows <= 96) {
    if (n <= 4096 || n > 16384) return false;
    return k < (n <= 8192 ? (rows > 64 ? 2560 : 1536) : (rows > 64 ? 4096 : 2560));
  }
  if (rows > 192) return n > 4096 || k < 4096;
  if (n <= 4096) return rows > 128 && n > 2048 && k < 2560;
  return k < 8192 || (rows <= 128 && ((n > 8192 && n <= 16384) || n > 32768));
}

// The products this kernel takes. Above 32 rows the tiled GEMMs keep rows of
// fewer than six super-blocks: of k = 1024 weights of 1024 to 8192 rows take
// 0.89-1.08 (Q4_K) and 1.02-1.22 times (Q6_K) as long here at 33-64 rows,
// 1.05-1.39 and 1.18-1.40 at 65-96, and a launch more of host time; from k = 1536
// 0.71-0.93 and 0.82-1.05. Q4_K keeps past that to 128 rows though the tiled
// (two-pass) GEMM is faster for some: weights of more than 16384 rows at 65-96 rows
// 1.04-1.2 times, at 97-128 1.15-1.25 (65536 rows 1.5: 92 us against 60 at k =
// 3072), and k below 3072 at 65-96 rows 1.05-1.3 (14336 x 1536 26.5 against 20.4):
// it rounds the min sums to f16 (9e-4 of the result's norm where this kernel is
// within 1e-7).
bool gemm_kq_mid_fits(int type, int64_t n, int64_t k, int64_t rows) {
  const int64_t block = type == T_Q4_K ? 144 : type == T_Q6_K ? 210 : 0;
  if (block == 0 || rows < kMidMinRows) return false;
  if (rows <= 32) {
    if (!few_rows_leave(type, n, k, rows)) return false;
  } else if (k < 1536) {
    return false;
  }
  if (type == T_Q6_K && rows > 32 && tiled_q6k_keeps(n, k, rows)) return false;
  if (rows > 128 && (type != T_Q6_K || k % 2048 == 0 || rows > 256)) return false;
  // 32-bit byte offsets inside the kernel
  return k % 256 == 0 && n * (k / 256) * block + 16 < ((int64_t)1 << 31) && 256 * k < ((int64_t)1 << 31) &&
         n * rows < ((int64_t)1 << 31);
}

// K ranges of one weight's product, from its own shape (so a weight's bits do
// not depend on the weights it shares a launch with): as many as bring its
// workgroups to 256 (two fit a CU: gate and up share a launch, and 14336 x 4096
// of either gives 224), at least 2 super-blocks a range. Measured at 77 rows,
// gate + up / q + k + v / down of an 8B layer, slots added: 128 workgroups 54 /
// 24 / 52 us, 256 45 / 24 / 35, 512 56 / 23 / 36.
int gemm_kq_mid_splits(int64_t n, int64_t k, int64_t rows) {
  const int64_t tiles = (n + BN - 1) / BN * ((rows + 95) / 96);
  int64_t s = 256 / tiles;
  const int64_t most = k / 512;
  if (s > most) s = most;
  if (s > 16) s = 16;
  return s < 1 ? 1 : (int)s;
}

size_t gemm_kq_mid_slot_bytes(const MvTargets& t, int64_t k, int64_t rows, bool always) {
  size_t bytes = 0;
  bool cut = always;
  for (int i = 0; i < t.count; i++) {
    const int64_t n = t.row_end[i] - (i ? t.row_end[i - 1] : 0);
    const int S = gemm_kq_mid_splits(n, k, rows);
    cut = cut || S > 1;
    bytes += align_up((size_t)(n * rows) * 4 * S, 256);
  }
  return cut ? bytes : 0;
}

template <int FMT>
static hipError_t launch_mid(const MvTargets& t, int64_t k, const ActPlanes& p, int64_t rows, void* slots,
                             size_t slot_bytes, float** parts, hipStream_t st) {
  if (t.count < 1 || t.count > kMaxTargets) return hipErrorInvalidValue;
  const size_t need = gemm_kq_mid_slot_bytes(t, k, rows, parts != nullptr);
  const bool cut = need > 0 && slots != nullptr && slot_bytes >= need;
  if (parts && !cut) return hipErrorInvalidValue;
  MidArgs a{};
  a.yq = p.codes;
  a.yd = p.d;
  a.ybs = (const int16_t*)p.sums;
  a.M = (int)rows;
  a.per = (int)chunk_rows(rows);
  a.chunks = (int)((rows + a.per - 1) / a.per);
  a.nsb = (int)(k / 256);
  int64_t units = 0, floats = 0, most = 0;
  for (int i = 0; i < kMaxTargets; i++) {
    const int j = i < t.count ? i : t.count - 1;  // unused entries repeat the last weight, with no units
    const int64_t n = t.row_end[j] - (j ? t.row_end[j - 1] : 0);
    a.w[i] = t.w[j];
    a.dst[i] = t.dst[j];
    a.ldd[i] = t.ldd[j];
    a.n[i] = n;
    a.splits[i] = gemm_kq_mid_splits(n, k, rows);
    a.part_off[i] = floats;
    if (i < t.count) {
      units += (n + BN - 1) / BN * a.chunks * (cut ? a.splits[i] : 1);
      if (parts) parts[i] = (float*)slots + floats;
      floats += (int64_t)(align_up((size_t)(n * rows) * 4 * a.splits[i], 256) / 4);
      most = n * rows > most ? n * rows : most;
    }
    a.unit_end[i] = (int)units;
  }
  if (units >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
  a.remap = units % 8 == 0 ? 1 : 0;
  a.part = cut ? (float*)slots : nullptr;
  launch_fmt<FMT>(a, (int)units, st);
  if (cut && !parts) {
    const int64_t blocks = (most / 4 + 255) / 256;
    gemm_kq_mid_sum_kernel<<<dim3((unsigned)(blocks < 1 ? 1 : blocks), (unsigned)t.count), 256, 0, st>>>(a);
  }
  return hipGetLastError();
}

hipError_t launch_gemm_q4k_mid(const MvTargets& t, int64_t k, const ActPlanes& p, int64_t rows, void* slots,
                               size_t slot_bytes, float** parts, hipStream_t st) {
  QMM_NOTE_LAUNCH();
  return launch_mid<T_Q4_K>(t, k, p, rows, slots, slot_bytes, parts, st);
}

hipError_t launch_gemm_q6k_mid(const MvTargets& t, int64_t k, const ActPlanes& p, int64_t rows, void* slots,
                               size_t slot_bytes, float** parts, hipStream_t st) {
  QMM_NOTE_LAUNCH();
  return launch_mid<T_Q6_K>(t, k, p, rows, slots, slot_bytes, parts, st);
}

}  // namespace qmm
