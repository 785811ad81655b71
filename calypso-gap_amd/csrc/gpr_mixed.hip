// Mixed-precision GPR contraction: FP16 (or BF16) hi + lo split operands on
// v_mfma_f32_16x16x32_{f16,bf16} with FP32 accumulation, FP64 norms and FP64
// energy partial sums.
//
// Same mathematics as k_gpr_f64 (gpr.hip): for a row tile against a range of
// sparse points,
//   S = xt mt^T,  d2 = |xt|^2 + |mt|^2 - 2 S  (norms in FP64),
//   W = exp(-d2 / 2) c,  E_i += sum_k W_ik,  G += W mt,
// with the exponential taken as exp2 of log2(e) S - (|xt|^2 + |mt|^2) log2(e) / 2
// (the per-point term and c times the W scale tabulated at model load).
// Every operand x is carried as hi = round(x), lo = round(x - hi) in the
// 16-bit type and each product as hi*hi + hi*lo + lo*hi (the lo*lo term is
// below FP32 rounding).  W is scaled by a power of two chosen from the
// largest |alpha| (GprArgs::wscale) before its split, so that hi cannot
// overflow and lo stays in the normal FP16 range; G is unscaled on output.
//
// Operand layout of the 16x16x32 forms per lane l (l16 = l % 16, lq = l / 16):
// A[l16][8 lq + e], B[8 lq + e][l16] (e = 0..7, one 16-byte register group),
// result D[4 lq + r][l16], r = 0..3.
//
// The kernel computes S^T = mt xt^T (A = sparse points from LDS, B = the
// wave's descriptor rows, held in registers for the whole kernel).  Lane
// (l16, lq) then holds S^T for row l16 and points 4 lq + r of each 16-point
// block, which is, for a 32-point step, exactly the B operand of
// G^T = mt^T W^T when the K index runs over the points in the order
// {4 lq .. 4 lq + 3, 16 + 4 lq .. 16 + 4 lq + 3} for lane group lq.  The
// feature-major copy of mt is stored in that order (api.hip), so W goes from
// the exp straight into MFMA operands without touching LDS.  Each wave owns R
// 16-row blocks, so every LDS fragment feeds 3 R MFMAs.
//
// Sparse points arrive in chunks of 32.  While chunk c's W and G are worked on,
// chunk c + 1's products run beside its exponentials (they do not depend on each
// other, so matrix cores and vector units both have work), and the point-major
// half of chunk c + 2 and the feature-major half of chunk c + 1 travel
// global -> LDS by direct loads (global_load_lds_dwordx4: no registers, counted
// by vmcnt).  Each half has two buffers and a turn one barrier: what the loads of
// a turn overwrite was last read the turn before.
// A point-major half holds the hi/lo tiles of 32 rows of DP halves, a
// feature-major half those of DP rows of 32 halves, each with the chunk's norm
// terms and scaled alphas.
// What bounds it: nothing alone.  Of 375 us for 67,647 atoms (D = 128, 4000
// points), leaving out the chunk loads takes 45 off, the LDS operand reads 25,
// the weights (FP64 conversions and sums, exp) 53, and the products' own time at
// the matrix rate is 164.  Against one chunk at a time between two barriers:
// 390 -> 375 us, energies only (71,644 atoms) 256 -> 210, 32,768 atoms at D = 256
// and 8000 points 759 -> 646.
// A direct load writes 64 consecutive 16-byte pieces per instruction, so the
// tiles have no row padding; instead piece q of row r sits at q ^ swz(r),
// which spreads the 16 rows a 16-lane group reads over all LDS banks.
#include "gapx_internal.h"

#include <type_traits>

namespace gapx {

namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));  // 16 bytes of halves
typedef __attribute__((address_space(3))) void lds_void;

template <bool BF>
struct Half;

template <>
struct Half<false> {
  typedef v8h vec;
  typedef _Float16 scalar;
  static __device__ __forceinline__ v4f mfma(vec a, vec b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

template <>
struct Half<true> {
  typedef v8b vec;
  typedef __bf16 scalar;
  static __device__ __forceinline__ v4f mfma(vec a, vec b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

constexpr int kPC = 32;  // sparse points per chunk

// Piece swizzle of a tile row of P 16-byte pieces: P >= 16 (a row covers
// all banks): XOR with row % 16; P = 8 or 4 (two or four rows per 256 bytes
// of banks): XOR with the row's index among the rows that share bank
// positions.  Rows of other widths are left in order.
template <int P>
__device__ __forceinline__ int swz(int row) {
  if constexpr (P >= 16 && (P & (P - 1)) == 0) return row & 15;
  else if constexpr (P == 8) return (row >> 1) & 7;
  else if constexpr (P == 4) return (row >> 2) & 3;
  else return 0;
}

// A chunk's hi and lo tiles of one kind (point-major or feature-major) and how
// their pieces are spread over the waves: piece s of [hi | lo] goes with DMA
// instruction s / (64 NW) of wave (s / 64) % NW, lane s % 64; instructions past
// the operands fill an unused tail (they reload a valid piece).
template <int DP, int NW>
struct Tiles {
  static constexpr int PM = DP / 8;         // pieces per point-major row
  static constexpr int PF = kPC / 8;        // pieces per feature-major row
  static constexpr int NE = kPC * PM;       // pieces per tile
  static constexpr int NT = 2 * NE;
  static constexpr int PER = 64 * NW;       // pieces per instruction over the workgroup
  static constexpr int NI = (NT + PER - 1) / PER;
  v4u op[NI * PER];
  double ex[128];  // norm terms (kPC doubles), scaled alphas (kPC floats), unused
};

// Offset (halves) of piece s from its tile's chunk origin, bit 31: the lo tile.
template <int DP, int NW, bool POINTS>
__device__ __forceinline__ unsigned piece_src(int s, int Mp) {
  typedef Tiles<DP, NW> C;
  if (s >= C::NT) s = C::NT - 1;
  const int e = s >= C::NE ? s - C::NE : s;
  unsigned off;
  if (POINTS) {
    const int row = e / C::PM, q = (e % C::PM) ^ swz<C::PM>(row);
    off = (unsigned)(row * DP + 8 * q);
  } else {
    const int d = e / C::PF, r = (e % C::PF) ^ swz<C::PF>(d);
    off = (unsigned)(d * Mp + 8 * r);
  }
  return off | (s >= C::NE ? 1u << 31 : 0u);
}

template <int U, int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
  if constexpr (U < N) {
    f(std::integral_constant<int, U>{});
    static_for<U + 1, N>(f);
  }
}

// This wave's direct loads have landed and its LDS reads are done; after the
// barrier every wave's are.  (The barrier's own fence keeps the compiler from
// moving LDS reads across it; it does not wait for direct loads.)
__device__ __forceinline__ void chunk_turn() {
  __builtin_amdgcn_s_waitcnt(7 << 4);  // vmcnt(0) lgkmcnt(0), gfx9 encoding: expcnt left alone
  __syncthreads();
}

template <bool BF, int DP, int R, int NW, bool GRAD>
__device__ __forceinline__ void gpr_mixed(const GprArgs &a) {
  typedef typename Half<BF>::vec vec;
  typedef typename Half<BF>::scalar hs;
  typedef Tiles<DP, NW> C;
  __shared__ __align__(16) C m0;  // point-major halves of even and odd chunks
  __shared__ __align__(16) C m1;
  __shared__ __align__(16) C f0;  // feature-major halves
  __shared__ __align__(16) C f1;

  const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l16 = lane & 15, lq = lane >> 4;
  int tile, split;
  xcd_tile_split(tile, split);
  const int row0 = (a.tile0 + tile) * (16 * R * NW) + wv * (16 * R);
  const int pb = split * a.pts_per_split;
  const int pe = min(a.Mp, pb + a.pts_per_split);
  const int nch = (pe - pb) / kPC;

  // B operands of S^T: row l16 of each row block, 8 features per lane per
  // 32-wide step
  vec xh[R][DP / 32], xl[R][DP / 32];
  double xq[R];  // -|xt|^2 log2(e) / 2 of the row
#pragma unroll
  for (int rb = 0; rb < R; ++rb) {
    const size_t row = (size_t)(row0 + 16 * rb + l16);
#pragma unroll
    for (int t = 0; t < DP / 32; ++t) {
      const size_t off = row * DP + 32 * t + 8 * lq;
      xh[rb][t] = *(const vec *)(a.xt_hi + off);
      xl[rb][t] = *(const vec *)(a.xt_lo + off);
    }
    xq[rb] = -0.5 * kLog2e * a.xn[row];
  }

  // this lane's operand pieces, one per DMA instruction
  unsigned msrc[C::NI], fsrc[C::NI];
#pragma unroll
  for (int u = 0; u < C::NI; ++u) {
    msrc[u] = piece_src<DP, NW, true>((u * NW + wv) * 64 + lane, a.Mp);
    fsrc[u] = piece_src<DP, NW, false>((u * NW + wv) * 64 + lane, a.Mp);
  }

  // the points' norm terms (FP64, two per lane) and scaled alphas (FP32, four
  // per lane); lanes past them reload a norm term into the unused part (the
  // loads are issued under a full lane mask)
  const char *exsrc = lane < kPC / 2       ? (const char *)(a.mnq + 2 * lane)
                      : lane < 3 * kPC / 4 ? (const char *)(a.cq + 4 * (lane - kPC / 2))
                                           : (const char *)a.mnq;
  const int exstride = (lane >= kPC / 2 && lane < 3 * kPC / 4) ? 4 : 8;  // bytes per point

  // one half of the chunk at p0 -> buffer B by direct loads
  auto issue = [&](C &B, const unsigned (&src)[C::NI], const uint16_t *hi, const uint16_t *lo) {
    static_for<0, C::NI>([&](auto uc) {
      constexpr int u = decltype(uc)::value;
      const unsigned o = src[u] & ~(1u << 31);
      const uint16_t *p;
      if constexpr ((u + 1) * C::PER <= C::NE)
        p = hi + o;
      else if constexpr (u * C::PER >= C::NE)
        p = lo + o;
      else
        p = ((src[u] >> 31) ? lo : hi) + o;
      __builtin_amdgcn_global_load_lds((const void *)p, (lds_void *)&B.op[(u * NW + wv) * 64], 16, 0, 0);
    });
  };
  auto issue_m = [&](C &B, int c) {
    const int p0 = pb + c * kPC;
    issue(B, msrc, a.mt_hi + (size_t)p0 * DP, a.mt_lo + (size_t)p0 * DP);
  };
  auto issue_f = [&](C &B, int c) {
    const int p0 = pb + c * kPC;
    if constexpr (GRAD) issue(B, fsrc, a.mtT_hi + p0, a.mtT_lo + p0);
    if (wv == 0)
      __builtin_amdgcn_global_load_lds((const void *)(exsrc + (size_t)p0 * exstride), (lds_void *)&B.ex[0], 16, 0, 0);
  };

  v4f G[R][DP / 16];  // G^T: features 16 b + 4 lq + r of row l16
#pragma unroll
  for (int rb = 0; rb < R; ++rb)
#pragma unroll
    for (int b = 0; b < DP / 16; ++b) G[rb][b] = v4f{0.f, 0.f, 0.f, 0.f};
  double er[R];
#pragma unroll
  for (int rb = 0; rb < R; ++rb) er[rb] = 0.0;

  // S^T of a chunk's two 16-point blocks for the R row blocks: 2 R chains of
  // products, taken in turn so that none waits for the one before
  auto products = [&](const C &B, v4f (&S)[2][R]) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int rb = 0; rb < R; ++rb) S[h][rb] = v4f{0.f, 0.f, 0.f, 0.f};
    // operands of step t + 1 read from LDS while step t's products run
    auto op_at = [&](int h, int t) {
      const int pt = 16 * h + l16;
      return pt * C::PM + ((4 * t + lq) ^ swz<C::PM>(pt));
    };
#pragma unroll
    for (int t = 0; t < DP / 32; ++t) {
      vec mh[2], ml[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        mh[h] = *(const vec *)&B.op[op_at(h, t)];
        ml[h] = *(const vec *)&B.op[C::NE + op_at(h, t)];
      }
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int rb = 0; rb < R; ++rb)
            S[h][rb] = Half<BF>::mfma(k == 1 ? ml[h] : mh[h], k == 2 ? xl[rb][t] : xh[rb][t], S[h][rb]);
    }
  };
  // W of block h from its S^T, in the B layout of the G step
  auto weights = [&](const C &B, int h, const v4f (&Sh)[R], vec (&wh)[R], vec (&wl)[R]) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int pl = 16 * h + 4 * lq + r;
      const double mq = B.ex[pl];
      const float cq = ((const float *)&B.ex[kPC])[pl];
#pragma unroll
      for (int rb = 0; rb < R; ++rb) {
        // -d2 log2(e) / 2 in FP64 (norms minus twice the product), then
        // ws = exp(-d2 / 2) c wscale
        const float e2 = (float)fma((double)Sh[rb][r], kLog2e, xq[rb] + mq);
        float ws = __builtin_amdgcn_exp2f(e2) * cq;
        // one rounded value for all uses: folded into the conversions, the
        // product rounds to another hi than the one lo is the remainder of
        asm("" : "+v"(ws));
        er[rb] += (double)ws;
        const hs hi = (hs)ws;
        wh[rb][4 * h + r] = hi;
        wl[rb][4 * h + r] = (hs)(ws - (float)hi);
      }
    }
  };
  auto gradient = [&](const C &B, const vec (&wh)[R], const vec (&wl)[R]) {
    // chains of products taken in turn (two feature blocks at once for one row
    // block); the next operands read while these products run
    auto top_at = [&](int b) {
      const int d = 16 * b + l16;
      return d * C::PF + (lq ^ swz<C::PF>(d));
    };
    constexpr int QB = R == 1 ? 2 : 1;
    vec th[QB], tl[QB];
#pragma unroll
    for (int q = 0; q < QB; ++q) {
      th[q] = *(const vec *)&B.op[top_at(q)];
      tl[q] = *(const vec *)&B.op[C::NE + top_at(q)];
    }
#pragma unroll
    for (int b = 0; b < DP / 16; b += QB) {
      vec th_n[QB], tl_n[QB];
      if (b + QB < DP / 16) {
#pragma unroll
        for (int q = 0; q < QB; ++q) {
          th_n[q] = *(const vec *)&B.op[top_at(b + QB + q)];
          tl_n[q] = *(const vec *)&B.op[C::NE + top_at(b + QB + q)];
        }
      }
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int q = 0; q < QB; ++q)
#pragma unroll
          for (int rb = 0; rb < R; ++rb)
            G[rb][b + q] = Half<BF>::mfma(k == 1 ? tl[q] : th[q], k == 2 ? wl[rb] : wh[rb], G[rb][b + q]);
#pragma unroll
      for (int q = 0; q < QB; ++q) {
        th[q] = th_n[q];
        tl[q] = tl_n[q];
      }
    }
  };

  // chunk c's weights beside the products of chunk c + 1, then chunk c's G
  v4f S[2][R];  // the current chunk's products
  auto finish = [&](const C &fc) {
    vec wh[R], wl[R];
    weights(fc, 0, S[0], wh, wl);
    weights(fc, 1, S[1], wh, wl);
    if constexpr (GRAD) gradient(fc, wh, wl);
  };
  auto turn = [&](int c, const C &mn, const C &fc, C &mfree, C &ffree) {
    chunk_turn();
    if (c + 2 < nch) issue_m(mfree, c + 2);
    issue_f(ffree, c + 1);
    v4f Sn[2][R];
    products(mn, Sn);
    finish(fc);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int rb = 0; rb < R; ++rb) S[h][rb] = Sn[h][rb];
  };

  // Each buffer is named statically, two turns per trip, so that the compiler
  // does not wait for the direct loads into one buffer before reads of another.
  if (nch > 0) {
    issue_m(m0, 0);
    issue_f(f0, 0);
    if (nch > 1) issue_m(m1, 1);
    chunk_turn();
    products(m0, S);
    int c = 0;
    for (; c + 2 < nch; c += 2) {
      turn(c, m1, f0, m0, f1);
      turn(c + 1, m0, f1, m1, f0);
    }
    if (c + 1 < nch) {
      turn(c, m1, f0, m0, f1);
      chunk_turn();
      finish(f1);
    } else {
      chunk_turn();
      finish(f0);
    }
  }

  const size_t base = (size_t)split * a.Np;
#pragma unroll
  for (int rb = 0; rb < R; ++rb) {
    const size_t row = (size_t)(row0 + 16 * rb + l16);
    if constexpr (GRAD) {
      const float inv = 1.0f / a.wscale;  // a power of two: exact
#pragma unroll
      for (int b = 0; b < DP / 16; ++b) {
        const float4 v = make_float4(G[rb][b][0] * inv, G[rb][b][1] * inv, G[rb][b][2] * inv, G[rb][b][3] * inv);
        *(float4 *)(a.Gpart32 + (base + row) * DP + 16 * b + 4 * lq) = v;
      }
    }
    double v = er[rb];
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    if (lq == 0) a.Epart[base + row] = v * (1.0 / (double)a.wscale);  // a power of two: exact
  }
}

template <bool BF, int DP, int R, int NW>
__global__ __launch_bounds__(64 * NW, 8 / NW) void k_gpr_mixed(GprArgs a) {
  gpr_mixed<BF, DP, R, NW, true>(a);
}

// Energies only: no feature-major loads, no second product (the halves' place in
// LDS stays; only the chunk's norm terms and alphas are kept there).
template <bool BF, int DP, int R, int NW>
__global__ __launch_bounds__(64 * NW, 8 / NW) void k_gpr_mixed_energy(GprArgs a) {
  gpr_mixed<BF, DP, R, NW, false>(a);
}

template <bool BF, int DP, int R, int NW, bool GRAD>
void launch_one(hipStream_t s, const GprArgs &a, int tiles) {
  if constexpr (GRAD)
    k_gpr_mixed<BF, DP, R, NW><<<dim3(tiles, a.splits), 64 * NW, 0, s>>>(a);
  else
    k_gpr_mixed_energy<BF, DP, R, NW><<<dim3(tiles, a.splits), 64 * NW, 0, s>>>(a);
}

// rows per workgroup: 64 (four waves of one 16-row block) or 128 (four
// waves of two blocks up to DP = 128; eight waves of one block above, where
// the four half-chunk buffers fill most of a CU's LDS)
template <bool BF, int DP, bool GRAD>
hipError_t launch_rows(hipStream_t s, const GprArgs &a) {
  const int tiles = a.ntiles > 0 ? a.ntiles : a.Np / a.rows;
  if (a.rows == 128) {
    if constexpr (DP <= 128)
      launch_one<BF, DP, 2, 4, GRAD>(s, a, tiles);
    else
      launch_one<BF, DP, 1, 8, GRAD>(s, a, tiles);
  } else {
    launch_one<BF, DP, 1, 4, GRAD>(s, a, tiles);
  }
  return hipGetLastError();
}

template <bool BF, bool GRAD>
hipError_t launch_typed(hipStream_t s, const GprArgs &a) {
  switch (a.Dp) {
    case 32: return launch_rows<BF, 32, GRAD>(s, a);
    case 64: return launch_rows<BF, 64, GRAD>(s, a);
    case 96: return launch_rows<BF, 96, GRAD>(s, a);
    case 128: return launch_rows<BF, 128, GRAD>(s, a);
    case 160: return launch_rows<BF, 160, GRAD>(s, a);
    case 192: return launch_rows<BF, 192, GRAD>(s, a);
    case 224: return launch_rows<BF, 224, GRAD>(s, a);
    case 256: return launch_rows<BF, 256, GRAD>(s, a);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

int gpr_points_per_chunk(int Dp) { return Dp <= 128 ? 64 : 32; }

hipError_t launch_gpr_mixed(hipStream_t s, const GprArgs &a) {
  if (a.pts_per_split % kPC != 0 || a.Mp % kPC != 0 || (a.rows != 64 && a.rows != 128) || a.Np % a.rows != 0)
    return hipErrorInvalidValue;
  if (a.grad) return a.bf16 ? launch_typed<true, true>(s, a) : launch_typed<false, true>(s, a);
  return a.bf16 ? launch_typed<true, false>(s, a) : launch_typed<false, false>(s, a);
}

}  // namespace gapx
