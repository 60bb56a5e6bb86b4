// gemm_b32.hip — Q8_0, IQ4_NL and MXFP4 products of more than 8 activation
// rows on the int8 matrix cores of gfx950.
//
// dst[m][n] = sum over 32-value blocks b of (dx_nb dy_mb) sum_{i in b} x_ni y_mi
// is candle's block dot for each type (Q8_0 vendor/candle/candle-core/src/
// quantized/k_quants.rs:1294-1312, MXFP4 :517-527 with the E2M1 table doubled
// and the e8m0 scale halved, IQ4_NL :754-764) against the activation
// quantized as the reference quantizes it for them (BlockQ8_0::from_float,
// :1240-1269: per-32 f16 scale dy, int8 codes y). The reference's card path
// sends Q8_0 and MXFP4 products above its row line to its int8 MMQ kernels
// (quantized/cuda.rs:1005-1136).
//
// Each block's integer sum T = sum_i x y is exact: a block's 32 values are the
// K of one v_mfma_i32_32x32x32_i8. What bounds these products is the vector
// work after it: one scale pair per 32 values per output. The scale products
// dx dy of a tile come from the matrix cores too, as one
// v_mfma_f32_32x32x16_f16 whose only nonzero K slot holds dy and dx (f16 both;
// the product of two 11-bit numbers is exact in f32), so an output takes two
// vector instructions a block, a conversion and acc += (dx dy) T, instead of
// three. MXFP4's dx = 2^(e - 128) is no f16: its scale products are multiplied
// in f32.
//
// Workgroup: kKG groups of kMW x kNW waves; a wave owns kMT row tiles of 32
// weight rows and a group one of kKG ranges of K, added at the end through LDS
// in group order. The shape follows the rows and the weight (config): 128 x 64
// where such tiles fill the CUs twice, else the same in two K ranges; 64 x 64
// in four up to 64 rows; 32 x 32 in eight up to 32, where a weight byte is
// still read once and eight waves share a tile's latency.
//   - K is staged 128 values (4 blocks) at a time: the activation codes (128 B
//     a row, 16-byte pieces XOR-swizzled by row) and, for each weight row, the
//     aligned 16-byte pieces covering its 4 blocks (clamped to the row, so none
//     leaves the weight's memory; an odd number of pieces a row, which spreads
//     the rows over the LDS banks) reach LDS by direct global-to-LDS copies one
//     stage ahead into the other half of double buffers; the activation scales
//     through registers.
//   - Lane L takes row L%32 of an operand and its values 16 (L/32) .. +15. The
//     lanes of the upper half read their scales from a zeroed piece of LDS.
// Measured: a Q8_0 8B layer's seven products at 512 rows 909 -> 470 us (q + k
// + v, o, gate + up and down: 247 GOP, 0.53 POP/s), where the vector unit is
// busy two thirds of the time and the matrix cores a third; 4096 x 14336 at 24
// rows 233 -> 42 us. Before, tiles of 128 rows x 64 weight rows in
// v_mfma_i32_16x16x32_i8 walked all of K with three vector instructions an
// output and block. Not faster: a block's operands read ahead over the block's
// branch (a wave of 64 x 64 then spills), the two MFMAs of a tile kept apart by
// half an epilogue each (scheduling groups).
// Blocks past the row's last are skipped. Rows past M and weight rows past N
// are read as the last row (valid memory); their outputs are never stored.
#include <type_traits>

#include "b32_common.h"
#include "lds_copy.h"
#include "qmm_launch.h"

namespace qmm {

namespace {

typedef int i4v __attribute__((ext_vector_type(4)));
typedef int i16v __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));

struct B32Args {
  const void* w[kMaxTargets];
  float* dst[kMaxTargets];
  int64_t ldd[kMaxTargets];
  int64_t n[kMaxTargets];
  int unit_end[kMaxTargets];  // workgroups of weights 0..t
  const int8_t* yq;
  const float* yd;
  int M, nb, mtiles, remap;
};

template <int FMT>
struct B32Shape {
  static constexpr int B = Fmt32<FMT>::B;               // bytes a block
  static constexpr int SB = 4 * B;                      // bytes of a row's stage
  static constexpr int Cover = (SB + 15 + 15) / 16;     // 16-byte pieces covering it at any offset
  static constexpr int Head = FMT == T_MXFP4 ? 1 : 2;   // scale bytes before the codes
};

// Four dwords from LDS address a (4-byte aligned), shifted down by sh bytes.
__device__ __forceinline__ void shifted4(const uint8_t* a, uint32_t sh, uint32_t* q) {
  uint32_t w[5];
#pragma unroll
  for (int i = 0; i < 5; i++) w[i] = *(const uint32_t*)(a + 4 * i);
#pragma unroll
  for (int i = 0; i < 4; i++) q[i] = __builtin_amdgcn_alignbyte(w[i + 1], w[i], sh);
}

// Where a lane finds its 16 weights of a stage's blocks (values 16 h ..
// 16 h + 15 of each): block b's bytes start off + B b into the row's window,
// so their dword and byte shift repeat every kCycle blocks.
template <int FMT>
struct B32Lane {
  static constexpr int kCycle = FMT == T_MXFP4 ? 4 : 2;
  const uint8_t* a[kCycle];
  uint32_t sh[kCycle];
  __device__ __forceinline__ B32Lane(const uint8_t* win, int off, int h) {
#pragma unroll
    for (int c = 0; c < kCycle; c++) {
      const int o = off + B32Shape<FMT>::B * c + B32Shape<FMT>::Head + (FMT == T_Q8_0 ? 16 * h : 0);
      a[c] = win + (o & ~3);
      sh[c] = (uint32_t)(o & 3);
    }
  }
  __device__ __forceinline__ i4v operand(int bb, int h, const Lut32<FMT>& lut) const {
    constexpr int B = B32Shape<FMT>::B;
    static_assert(B * kCycle % 4 == 0, "the shifts repeat");
    uint32_t q[4];
    shifted4(a[bb % kCycle] + B * kCycle * (bb / kCycle), sh[bb % kCycle], q);
    if constexpr (FMT != T_Q8_0) {
      // values 0..15 are the low nibbles of bytes 0..15, values 16..31 the high nibbles
#pragma unroll
      for (int i = 0; i < 4; i++) q[i] = (uint32_t)lut16_at(q[i], 4 * h, lut.t0, lut.t1, lut.t2, lut.t3);
    }
    return i4v{(int)q[0], (int)q[1], (int)q[2], (int)q[3]};
  }
};

__device__ __forceinline__ uint32_t swz(uint32_t r) { return (r >> 1) & 7u; }

template <int FMT, int kMW, int kNW, int kKG, int kMT>
__global__ __launch_bounds__(64 * kMW * kNW * kKG, 2) void gemm_b32_kernel(const B32Args a) {
  using S = B32Shape<FMT>;
  constexpr bool kMul = FMT == T_MXFP4;
  constexpr int G = kMW * kNW;                       // waves of a K group
  constexpr int BM = 32 * kMW * kMT, BN = 32 * kNW;
  // 32 rows keep the fewest pieces (eight groups' buffers fill the LDS)
  constexpr int P = BN == 32 ? S::Cover : S::Cover | 1;
  constexpr int kWin = 16 * P;                       // LDS bytes a weight row
  constexpr int kWInstr = (BN * P + 63) / 64;        // 1 KB copies of the weight windows a stage
  constexpr int kAInstr = BM / 8;                    // and of the activation tile
  constexpr int kWCopies = (kWInstr + G - 1) / G, kACopies = kAInstr / G;
  constexpr int kDy = 4 * BM;                        // activation scales a stage
  constexpr int kDyPer = kDy / (64 * G);
  static_assert(kAInstr % G == 0 && kDy % (64 * G) == 0, "copy shapes");
  typedef std::conditional_t<kMul, float, uint16_t> dy_t;
  // kMul: block-major f32 [4][BM]; else row-major f16 [BM][4]
  __shared__ __attribute__((aligned(1024))) int8_t s_a[2][kKG][BM * 128];
  __shared__ __attribute__((aligned(16))) uint8_t s_w[2][kKG][kWInstr * 1024];
  __shared__ __attribute__((aligned(16))) dy_t s_dy[2][kKG][kDy];
  __shared__ __attribute__((aligned(16))) uint8_t s_zero[S::SB + 32];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wv / G, gw = wv % G;  // K group and wave within it
  const int wm = gw % kMW, wn = gw / kMW;
  const int h = lane >> 5, r32 = lane & 31;

  const int total = (int)gridDim.x;
  const int bid = (int)blockIdx.x;
  const int idx = a.remap ? (bid & 7) * (total >> 3) + (bid >> 3) : bid;
  const int t = idx < a.unit_end[0] ? 0 : idx < a.unit_end[1] ? 1 : idx < a.unit_end[2] ? 2 : 3;
  auto pick = [&](const auto& arr) { return t == 0 ? arr[0] : t == 1 ? arr[1] : t == 2 ? arr[2] : arr[3]; };
  const int loc = idx - (t == 0 ? 0 : t == 1 ? a.unit_end[0] : t == 2 ? a.unit_end[1] : a.unit_end[2]);
  const int64_t N = pick(a.n);
  const int M = a.M, nb = a.nb;
  // row tiles of one weight tile next to each other (one XCD's L2, through the remap)
  const int m0 = (loc % a.mtiles) * BM;
  const int64_t n0 = (int64_t)(loc / a.mtiles) * BN;
  const uint8_t* __restrict__ W = (const uint8_t*)pick(a.w);
  const int8_t* __restrict__ yq = a.yq;
  const float* __restrict__ yd = a.yd;
  const uint32_t K = (uint32_t)nb * 32u;
  const uint32_t rowbytes = (uint32_t)nb * S::B;
  // this group's stages: kSteps of them from st0, the last ones perhaps past
  // the row (every group runs the same number of steps, for the barriers)
  const int nst = (nb + 3) / 4, steps = (nst + kKG - 1) / kKG, st0 = kg * steps;

  // Weight copy i: pieces 64 i .. 64 i + 63 of the windows, lane L piece
  // f = 64 i + L: window row f / P, piece f % P of the aligned span at or
  // before the row's stage, clamped to the piece holding the stage's last byte
  // in the row. A wave whose last index passes kWInstr repeats its previous
  // copy. Activation copy i: rows 8i .. 8i+7; lane L row 8i + L/8 at piece
  // position L%8, which holds code piece (L%8) ^ swz(row).
  uint32_t wrow_off[kWCopies], wpc[kWCopies], arow_off[kACopies], apc[kACopies];
#pragma unroll
  for (int u = 0; u < kWCopies; u++) {
    int i = gw + G * u;
    i = i < kWInstr ? i : i - G;
    const uint32_t f = 64u * (uint32_t)i + (uint32_t)lane;
    const uint32_t wr = f / (uint32_t)P < (uint32_t)BN ? f / (uint32_t)P : BN - 1;
    const int64_t r = n0 + wr < N ? n0 + wr : N - 1;
    wrow_off[u] = (uint32_t)r * rowbytes;
    wpc[u] = 16u * (f % (uint32_t)P);
  }
#pragma unroll
  for (int u = 0; u < kACopies; u++) {
    const int tr = 8 * (gw + G * u) + (lane >> 3);
    arow_off[u] = (uint32_t)(m0 + tr < M ? m0 + tr : M - 1) * K;
    apc[u] = 16u * (((uint32_t)lane & 7u) ^ swz((uint32_t)tr));
  }
  // rows of whole stages that start 16-byte aligned: every stage but the last
  // reads what follows it in the row, at offsets that only a scalar moves
  const bool whole = (nb & 3) == 0 && (rowbytes & 15u) == 0;
  auto copy_stage = [&](int st, int buf) {
    if (whole && st + 1 < nst) {
#pragma unroll
      for (int u = 0; u < kACopies; u++)
        dma16(yq + 128 * (int64_t)st, arow_off[u] + apc[u], lds_addr(&s_a[buf][kg][1024 * (gw + G * u)]));
#pragma unroll
      for (int u = 0; u < kWCopies; u++) {
        int i = gw + G * u;
        i = i < kWInstr ? i : i - G;
        dma16(W + ((S::SB * (int64_t)st) & ~(int64_t)15), wrow_off[u] + wpc[u], lds_addr(&s_w[buf][kg][1024 * i]));
      }
      return;
    }
#pragma unroll
    for (int u = 0; u < kACopies; u++) {
      const uint32_t o = 128u * (uint32_t)st + apc[u];
      dma16(yq, arow_off[u] + (o < K - 16u ? o : K - 16u), lds_addr(&s_a[buf][kg][1024 * (gw + G * u)]));
    }
#pragma unroll
    for (int u = 0; u < kWCopies; u++) {
      int i = gw + G * u;
      i = i < kWInstr ? i : i - G;
      const uint32_t s0 = wrow_off[u] + (uint32_t)(S::SB * st);
      const uint32_t rend = wrow_off[u] + rowbytes;
      const uint32_t send = s0 + S::SB < rend ? s0 + S::SB : rend;
      const uint32_t p = (s0 & ~15u) + wpc[u], last = (send - 1u) & ~15u;
      dma16(W, p < last ? p : last, lds_addr(&s_w[buf][kg][1024 * i]));
    }
  };
  // activation scales: thread e of the group loads kDyPer of the (row, block)
  // pairs of a stage, 4 consecutive threads a row (kMul: consecutive rows)
  float sdy[kDyPer];
  const int ge = gw * 64 + lane;
  auto load_dy = [&](int st) {
#pragma unroll
    for (int u = 0; u < kDyPer; u++) {
      const int e = ge + 64 * G * u;
      const int row = e >> 2, blk = e & 3;
      const int gr = m0 + row < M ? m0 + row : M - 1;
      const int gb = 4 * st + blk;
      sdy[u] = yd[(int64_t)gr * nb + (gb < nb ? gb : nb - 1)];
    }
  };
  auto store_dy = [&](int buf) {
#pragma unroll
    for (int u = 0; u < kDyPer; u++) {
      const int e = ge + 64 * G * u;
      if constexpr (kMul)
        s_dy[buf][kg][(e & 3) * BM + (e >> 2)] = sdy[u];
      else
        s_dy[buf][kg][e] = __builtin_bit_cast(uint16_t, (_Float16)sdy[u]);  // an f16's value: exact
    }
  };

  f16v acc[kMT];
#pragma unroll
  for (int m = 0; m < kMT; m++)
#pragma unroll
    for (int i = 0; i < 16; i++) acc[m][i] = 0.0f;

  const Lut32<FMT> lut;
  // the lane's weight row: its bytes' offset, and its window
  const int64_t grow = n0 + 32 * wn + r32;
  const uint32_t wbase = (uint32_t)(grow < N ? grow : N - 1) * rowbytes;
  const int wwin = (32 * wn + r32) * kWin;
  const int arow = 32 * kMT * wm + r32;

  // the scale operands: K slot 0 (lanes 0-31) set block by block, all others zero
  i4v dx8 = {0, 0, 0, 0}, dy8[kMT];
#pragma unroll
  for (int m = 0; m < kMT; m++) dy8[m] = i4v{0, 0, 0, 0};

  auto at = [&](int st) { return st < nst ? st : nst - 1; };  // past the row, its last stage again
  copy_stage(at(st0), 0);
  load_dy(at(st0));
  for (int i = tid; i < (int)sizeof(s_zero) / 4; i += 64 * G * kKG) ((uint32_t*)s_zero)[i] = 0;
  store_dy(0);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();

  auto step = [&](auto parity, int st) {
    constexpr int cur = decltype(parity)::value;
    copy_stage(at(st + 1), cur ^ 1);
    load_dy(at(st + 1));
    const uint8_t* win = &s_w[cur][kg][wwin];
    const int8_t* sa = s_a[cur][kg];
    const dy_t* sdyl = s_dy[cur][kg];
    const int nv = nb - 4 * st;  // blocks of this stage in the row
    const int o = (int)((wbase + (uint32_t)(S::SB * st)) & 15u);
    const B32Lane<FMT> wl(win, o, h);
    const uint8_t* dxp = h && !kMul ? s_zero : win + o;
    uint2 dyw[kMT];
    if constexpr (!kMul) {
#pragma unroll
      for (int m = 0; m < kMT; m++) dyw[m] = *(const uint2*)(h ? (const uint16_t*)s_zero : sdyl + 4 * (arow + 32 * m));
    }
#pragma unroll
    for (int bb = 0; bb < 4; bb++) {
      if (bb >= nv) continue;
      i4v af[kMT];
      float dxf = 0.0f;
      const i4v wf = wl.operand(bb, h, lut);
      if constexpr (kMul)
        dxf = e8m0_half((uint32_t)dxp[S::B * bb]);
      else
        dx8[0] = (int)*(const uint16_t*)(dxp + S::B * bb);
#pragma unroll
      for (int m = 0; m < kMT; m++) {
        const uint32_t row = (uint32_t)(arow + 32 * m);
        af[m] = *(const i4v*)(sa + 128u * row + 16u * ((uint32_t)(2 * bb + h) ^ swz(row)));
        if constexpr (!kMul) {
          const uint32_t w = bb < 2 ? dyw[m].x : dyw[m].y;
          dy8[m][0] = (int)(bb & 1 ? w >> 16 : w & 0xFFFFu);
        }
      }
      const i16v zi = {};
      const f16v zf = {};
      i16v T[kMT];
      f16v Pr[kMT];
#pragma unroll
      for (int m = 0; m < kMT; m++) {
        T[m] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[m], wf, zi, 0, 0, 0);
        if constexpr (!kMul)
          Pr[m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, dy8[m]), __builtin_bit_cast(h8, dx8), zf,
                                                         0, 0, 0);
      }
#pragma unroll
      for (int m = 0; m < kMT; m++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          f4v dy4 = {};
          if constexpr (kMul) dy4 = *(const f4v*)&sdyl[bb * BM + 32 * kMT * wm + 32 * m + 8 * g + 4 * h];
#pragma unroll
          for (int x = 0; x < 4; x++) {
            const int i = 4 * g + x;
            const float p = kMul ? dxf * dy4[x] : Pr[m][i];
            acc[m][i] = __builtin_fmaf(p, (float)T[m][i], acc[m][i]);
          }
        }
    }
    // the next stage's copies and scales, in flight since this one's start
    store_dy(cur ^ 1);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  };
  for (int i = 0; i < steps; i += 2) {
    step(std::integral_constant<int, 0>{}, st0 + i);
    if (i + 1 < steps) step(std::integral_constant<int, 1>{}, st0 + i + 1);
  }

  if constexpr (kKG > 1) {
    // groups 1.. to LDS (the activation buffers, no longer read), added by
    // group 0 in group order
    float* part = (float*)s_a;
    constexpr int kTile = 64 * G * kMT * 16;
    static_assert((kKG - 1) * kTile * 4 <= (int)sizeof(s_a), "partials fit");
    if (kg > 0) {
#pragma unroll
      for (int m = 0; m < kMT; m++)
#pragma unroll
        for (int i = 0; i < 16; i++) part[(kg - 1) * kTile + (16 * m + i) * (64 * G) + ge] = acc[m][i];
    }
    __syncthreads();
    if (kg > 0) return;
    for (int g = 0; g < kKG - 1; g++) {
#pragma unroll
      for (int m = 0; m < kMT; m++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[m][i] += part[g * kTile + (16 * m + i) * (64 * G) + ge];
    }
  }

  float* __restrict__ dst = pick(a.dst);
  int64_t ldd = pick(a.ldd);
  int hrow = m0 + 32 * kMT * wm + 4 * h;
  // the rows and their addresses are formed here, not kept live over the K loop
  asm volatile("" : "+s"(ldd), "+v"(hrow));
  if (grow >= N) return;
#pragma unroll
  for (int m = 0; m < kMT; m++)
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int row = hrow + 32 * m + 8 * (i >> 2) + (i & 3);
      if (row < M) dst[row * ldd + grow] = acc[m][i];
    }
}

// The workgroup shape of one weight's product, from its own size and the rows
// (so a product's bits do not depend on the weights it shares a launch with):
// 0: 128 x 64; 1: 128 x 64, two K ranges; 2: 64 x 64, four; 3: 32 x 32, eight;
// 4: 64 x 32, four.
// Shape 0 where its tiles come to two a CU (Q8_0 gate + up of an 8B layer at
// 512 rows 206 us; 128 x 128 tiles of 64 x 64 a wave, which leave a SIMD two
// waves of 237 registers instead of three of 164, 208, and IQ4_NL's 239 against
// 207); two K ranges give the others eight waves a CU, and the smaller tiles
// serve products whose 128 x 64 tiles would leave CUs idle (4096 x 4096 at 100
// rows, one such tile a workgroup 39 us, now 22; 1024 x 4096 at 300 rows 38, now 22).
int config(int64_t n, int64_t rows) {
  if (rows <= 32) return 3;
  const int64_t wide = (n + 63) / 64 * ((rows + 127) / 128), half = (n + 63) / 64 * ((rows + 63) / 64);
  if (rows > 64 && wide >= 192) return wide >= 512 ? 0 : 1;
  return half > 128 ? 2 : 4;
}
constexpr int kTileRows[5] = {128, 128, 64, 32, 64}, kTileCols[5] = {64, 64, 64, 32, 32};

template <int FMT>
hipError_t launch_config(int c, const MvTargets& t, int64_t k, const ActPlanes& p, int64_t rows, hipStream_t st) {
  B32Args a{};
  a.yq = p.codes;
  a.yd = p.d;
  a.M = (int)rows;
  a.nb = (int)(k / 32);
  a.mtiles = (int)((rows + kTileRows[c] - 1) / kTileRows[c]);
  int64_t units = 0;
  for (int i = 0; i < kMaxTargets; i++) {
    const int j = i < t.count ? i : t.count - 1;  // unused entries repeat the last weight, with no units
    const int64_t n = t.row_end[j] - (j ? t.row_end[j - 1] : 0);
    a.w[i] = t.w[j];
    a.dst[i] = t.dst[j];
    a.ldd[i] = t.ldd[j];
    a.n[i] = n;
    if (i < t.count) units += (n + kTileCols[c] - 1) / kTileCols[c] * a.mtiles;
    if (units >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
    a.unit_end[i] = (int)units;
  }
  a.remap = units % 8 == 0 ? 1 : 0;
  const dim3 grid((unsigned)units);
  if (c == 0)
    gemm_b32_kernel<FMT, 2, 2, 1, 2><<<grid, 256, 0, st>>>(a);
  else if (c == 1)
    gemm_b32_kernel<FMT, 2, 2, 2, 2><<<grid, 512, 0, st>>>(a);
  else if (c == 2)
    gemm_b32_kernel<FMT, 1, 2, 4, 2><<<grid, 512, 0, st>>>(a);
  else if (c == 3)
    gemm_b32_kernel<FMT, 1, 1, 8, 1><<<grid, 512, 0, st>>>(a);
  else
    gemm_b32_kernel<FMT, 1, 1, 4, 2><<<grid, 256, 0, st>>>(a);
  return hipGetLastError();
}

// The weights of one shape share a launch.
template <int FMT>
hipError_t launch_fmt(const MvTargets& t, int64_t k, const ActPlanes& p, int64_t rows, hipStream_t st) {
  for (int c = 0; c < 5; c++) {
    MvTargets g{};
    int64_t end = 0;
    for (int i = 0; i < t.count; i++) {
      const int64_t n = t.row_end[i] - (i ? t.row_end[i - 1] : 0);
      if (config(n, rows) != c) continue;
      g.w[g.count] = t.w[i];
      g.dst[g.count] = t.dst[i];
      g.ldd[g.count] = t.ldd[i];
      end += n;
      g.row_end[g.count++] = end;
    }
    if (g.count == 0) continue;
    const hipError_t e = launch_config<FMT>(c, g, k, p, rows, st);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace

int gemm_b32_min_rows() { return 9; }  // up to 8 rows: the decode kernels

bool gemm_b32_fits(int type, int64_t n, int64_t k, int64_t rows) {
  const int bb = type == T_Q8_0 ? 34 : type == T_IQ4_NL ? 18 : type == T_MXFP4 ? 17 : 0;
  // 32-bit byte offsets inside the kernel; a row of at least one 16-byte piece
  return bb != 0 && k % 32 == 0 && k >= 32 && n * (k / 32) * bb + 16 < ((int64_t)1 << 31) &&
         (rows + 128) * k < ((int64_t)1 << 31);
}

hipError_t launch_gemm_b32(int type, const MvTargets& t, int64_t k, const ActPlanes& p, int64_t rows, hipStream_t st) {
  QMM_NOTE_LAUNCH();
  if (t.count < 1 || t.count > kMaxTargets) return hipErrorInvalidValue;
  if (type == T_Q8_0) return launch_fmt<T_Q8_0>(t, k, p, rows, st);
  if (type == T_IQ4_NL) return launch_fmt<T_IQ4_NL>(t, k, p, rows, st);
  if (type == T_MXFP4) return launch_fmt<T_MXFP4>(t, k, p, rows, st);
  return hipErrorInvalidValue;
}

}  // namespace qmm
