// Moment GEMMs of Linear and Conv2D on the bf16 matrix cores, with fp32 operands and results.
//
// The fp32 MFMA bounds these products (157 TF/s, the fp32 kernel reaches 115-137); the bf16
// MFMA is 16 times as wide. Every fp32 operand value (the squares formed in fp32 first) is
// split into three bf16 parts h + m + l (8 + 8 + 7 significand bits), exactly where its last
// bit is bf16's smallest, 2^-133, or more: values of 2^-109 (1.5e-33) and up; smaller ones are
// held to 2^-133, as a result of fp32 arithmetic is to 2^-149. A product is the six part
// products h h, h m, m h, m m, h l, l h, each exact in the matrix core; the three left out are
// below 2^-24 of it. The six are added smallest first into a partial sum that
// starts at zero in every 32-wide k tile, and the partial sum is added to the fp32 accumulator
// by the VALU, which rounds to nearest (the bf16 MFMA truncates: added straight to the
// accumulator the small products would be cut off, 1e-5 over 4096 terms). One rounding per 32
// terms instead of one per 2: against float64 the result is 3 to 10 times closer than the fp32
// kernel's (4096 x 4096 x 4096 training products 2.3e-7 against 2.3e-6, a residual block's
// parameter deltas 3.2e-7 against 1.2e-6, 1001 x 1003 x 517 9e-8 against 4e-7).
//
// What bounds it is VALU work beside the MFMAs (they hardly overlap): 11 operations split a
// pair of values. So each value is split once per block: one operand (direct) goes from global
// memory to registers in the MFMA's fragment layout, each wave owning its rows of it; the
// other (staged) is split by the whole block and shared through LDS as bf16 parts. 16x16x32
// MFMAs, which sustain 2.1 PF/s here where 32x32x16 throttles at 1.85 (random operands).
// Measured, fp32 kernel on the left, each in its plan (4096 x 4096 x 4096, one run): forward
// 3021 -> 2166 us (190 TF/s of fp32 products), input deltas 2036 -> 1389, parameter deltas 2107
// -> 1750; a 64-channel 3 x 3 Conv2D at 131072 pixels: forward 246 -> 193, input deltas 183 ->
// 152, parameter deltas 197 -> 170.
#pragma once
#include "tagi_gemm_core.h"

namespace tagi {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pack_hi(float x0, float x1) {
  return __builtin_amdgcn_perm(__float_as_uint(x1), __float_as_uint(x0), 0x07060302u);
}
__device__ __forceinline__ uint32_t pack_bf16(float x0, float x1) {
  bf16x2 p;
  p[0] = (__bf16)x0;
  p[1] = (__bf16)x1;
  return __builtin_bit_cast(uint32_t, p);
}

// Three-way split of two values, packed: h and m rounded to nearest, l what remains (7 bits at
// most). Of a value in [1, 2), |m| <= 2^-8 and |l| <= 2^-17, of either sign whatever the
// value's, so the part products left out average out even where an operand is constant (an
// initial variance). With h truncated they reach 2^-22 and share a sign: 6e-8 of a variance
// whose weights are all 1.0078, which cost 2% less (ResNet-18 step 7.66 against 7.81 ms).
__device__ __forceinline__ void split_pair(float x0, float x1, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = pack_bf16(x0, x1);
  float r0 = x0 - __uint_as_float(h << 16), r1 = x1 - __uint_as_float(h & 0xffff0000u);
  m = pack_bf16(r0, r1);
  r0 -= __uint_as_float(m << 16);
  r1 -= __uint_as_float(m & 0xffff0000u);
  l = pack_hi(r0, r1);
}

// Operand of product P (0: the mean's, then the variance's) formed from the raw moments; s0
// and s1 are the moments and r0 the mean, s0 and s1 both times the same sign
template <int PROD, bool B, int P>
__device__ __forceinline__ float prod_operand(float r0, float s0, float s1) {
  if constexpr (PROD == PROD_FWD) {
    if constexpr (!B) return P == 0 ? s0 : P == 1 ? r0 * s0 : s1;
    else return P == 0 ? s0 : P == 1 ? s1 : r0 * s0 + s1;
  } else if constexpr ((PROD == PROD_SHARED_B) == B) {
    return P == 0 ? s0 : r0 * s0;
  } else {
    return P == 0 ? s0 : s1;
  }
}

__device__ __forceinline__ floatx4 mfma_bf16(uintx4 a, uintx4 b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                 0);
}

template <int KIND>
constexpr bool kfast_kind() {
  return !KindTraits<KIND>::mn_fast;
}

// Waves per SIMD of the register budget: the loaders of any alignment and of scalar patches
// hold more addresses than the budget of three or four waves allows without spills.
template <int PROD, class X, int KA, int KB>
constexpr int split_minw() {
  constexpr bool heavy = KindTraits<KA>::any || KindTraits<KB>::any || !KindTraits<KA>::vec4;
  return X::minw(PROD) > 2 && heavy ? X::minw(PROD) - 1 : X::minw(PROD);
}

template <int PROD, class X, int KA, int KB, int EPI = 0>
__global__ void __launch_bounds__(X::NTH, (split_minw<PROD, X, KA, KB>())) gemm_split_kernel(GemmArgs g) {
  // the operand whose fragments are loaded along the reduction goes to registers directly
  constexpr bool DA = kfast_kind<KA>();
  constexpr int NBUF = X::nbuf(PROD);
  constexpr int BK = X::BK, NTH = X::NTH, DM = X::DM, LM = X::LM, NW = X::NW;
  constexpr int BM = DA ? NW * DM : LM, BN = DA ? LM : NW * DM;
  constexpr int WM = DA ? DM : LM, WN = DA ? LM : DM;
  constexpr int NA = (PROD == PROD_SHARED_A) ? 1 : 2;
  constexpr int NB = (PROD == PROD_SHARED_B) ? 1 : 2;
  constexpr int ND = DA ? NA : NB, NL = DA ? NB : NA;  // raw tensors of each operand
  constexpr int NP = PROD == PROD_FWD ? 3 : 2;
  constexpr int TD = DM / 16, TL = LM / 16;
  constexpr int TM = WM / 16, TN = WN / 16;
  constexpr int EK = !DA ? 2 : KA == LD_CBWD_A4 || KA == LD_CBWD_A_S || KA == LD_CBWD_A4T ? 4 : 1;
  using LD = Loader<DA ? KA : KB, ND, NW * DM, BK, NTH, 1, 2, DM>;
  using LS = Loader<DA ? KB : KA, NL, LM, BK, NTH, 1, 1>;
  // LDS: [buffer][product][part][k / 8][row][8 bf16]; the k / 8 planes are offset by 64
  // bytes and the rows of a group of four permuted (phys below), which spreads the stores of
  // every unit shape over the banks (the counters still read half of the LDS cycles as
  // conflicts, at one LDS instruction per 8 to 18 VALU instructions)
  constexpr int QS = LM * 16 + 64, PS = 4 * QS, BUF = NP * 3 * PS;
  constexpr int RAW = NL * LM * BK * 4;  // fp32 tile of the fallback loop
  constexpr int SM = NBUF * BUF > RAW ? NBUF * BUF : RAW;
  __shared__ __attribute__((aligned(16))) unsigned char smem[SM];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int rl = lane & 15, q = lane >> 4;

  BlockPos bp;
  if (!block_pos<BM, BN>(g, bp)) return;
  const int z = bp.z, kbeg = bp.kbeg, kend = bp.kend;
  const int zz = z * g.splits + bp.split;
  const int d0 = DA ? bp.m0 : bp.n0, l0 = DA ? bp.n0 : bp.m0;
  const Operand& od = DA ? g.a : g.b;
  const Operand& os = DA ? g.b : g.a;

  LD ld;
  LS ls;
  ld.init(od, z, d0, tid, kend);
  ls.init(os, z, l0, tid, kend);

  floatx4 acc[2][TM][TN];
#pragma unroll
  for (int o = 0; o < 2; ++o)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[o][i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  const int nk = kbeg < kend ? (kend - kbeg + BK - 1) / BK : 0;
  if (g.phased && g.partial && nk == 0) return;

  // raw element e of the thread's staged unit u, row j of it
  auto sraw = [&](int t, int u, int j, int e) {
    if constexpr (LS::V4 && !LS::MNF) return ls.elem(t, u * LS::CPU + e / 4, e % 4);
    else return ls.elem(t, u * LS::CPU + e, j);
  };
  // The bf16 MFMA drops the bits below its alignment, so each k tile's partial sums lie a
  // little (1e-8 of their size) below their value: nothing beside one output's rounding, but
  // deltas are summed over 1e5 pixels downstream, where it would add up. The staged operand
  // is negated in every other k tile and every other row of tiles (and the partial sums
  // subtracted), so that the shift cancels along the reduction and over the rows.
  auto sign = [&](int t) { return ((t ^ bp.tmi) & 1) ? -1.f : 1.f; };
  auto phys = [](int row) { return (row & ~3) | ((row & 3) ^ ((row >> 2) & 3)); };
  auto stage = [&](unsigned char* buf, int t) {
    const float sg = sign(t);
#pragma unroll
    for (int u = 0; u < LS::NU; ++u) {
      int mn, k;
      LS::unit_pos(tid, u, mn, k);
#pragma unroll
      for (int j = 0; j < LS::UR; ++j) {
        unsigned char* p = buf + (k >> 3) * QS + phys(mn + j) * 16 + (k & 7) * 2;
        // the raw values with the tile's sign once; squares take one signed factor
        float r0[LS::KG], s0[LS::KG], s1[LS::KG];
#pragma unroll
        for (int e = 0; e < LS::KG; ++e) {
          r0[e] = sraw(0, u, j, e);
          s0[e] = sg * r0[e];
          s1[e] = NL == 2 ? sg * sraw(NL - 1, u, j, e) : 0.f;
        }
        static_for<0, NP>([&](auto P) {
          uint32_t w[3][LS::KG / 2];
#pragma unroll
          for (int e = 0; e < LS::KG; e += 2)
            split_pair(prod_operand<PROD, DA, P>(r0[e], s0[e], s1[e]),
                       prod_operand<PROD, DA, P>(r0[e + 1], s0[e + 1], s1[e + 1]), w[0][e / 2], w[1][e / 2],
                       w[2][e / 2]);
#pragma unroll
          for (int s = 0; s < 3; ++s) {
            unsigned char* d = p + (P * 3 + s) * PS;
            if constexpr (LS::KG == 8) *reinterpret_cast<uintx4*>(d) = uintx4{w[s][0], w[s][1], w[s][2], w[s][3]};
            else if constexpr (LS::KG == 4) *reinterpret_cast<uintx2*>(d) = uintx2{w[s][0], w[s][1]};
            else *reinterpret_cast<uint32_t*>(d) = w[s][0];
          }
        });
      }
    }
  };
  // raw element e of direct fragment f
  auto draw = [&](int t, int f, int e) {
    if constexpr (LD::FV != 0) return ld.elem(t, e, f);
    else if constexpr (LD::V4) return ld.elem(t, f * LD::CPF + e / 4, e % 4);
    else return ld.elem(t, f * LD::CPF + e, 0);
  };
  auto dval = [&](auto P, int f, int e) {
    const float r0 = draw(0, f, e);
    return prod_operand<PROD, !DA, decltype(P)::value>(r0, r0, ND == 2 ? draw(ND - 1, f, e) : 0.f);
  };
  const int lrow = q * QS + phys(rl) * 16;  // the lane's 16 bytes of staged fragment 0

  // Products P .. P + N - 1 of one k tile (N 2: the forward's two variance products, whose
  // partial sums share one chain and one addition)
  auto product = [&](auto P, auto N, const unsigned char* buf, float sg, auto&& after) {
    constexpr int n_ = decltype(N)::value;
    uintx4 fd[n_][TD][3];
    static_for<0, n_>([&](auto n) {
      using Q = std::integral_constant<int, decltype(P)::value + decltype(n)::value>;
#pragma unroll
      for (int f = 0; f < TD; ++f)
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          uint32_t h, m, l;
          split_pair(dval(Q{}, f, e), dval(Q{}, f, e + 1), h, m, l);
          fd[n][f][0][e / 2] = h;
          fd[n][f][1][e / 2] = m;
          fd[n][f][2][e / 2] = l;
        }
    });
    after();
#pragma unroll
    for (int j = 0; j < TL; ++j) {
      uintx4 fl[n_][3];
#pragma unroll
      for (int n = 0; n < n_; ++n)
#pragma unroll
        for (int s = 0; s < 3; ++s)
          fl[n][s] = *reinterpret_cast<const uintx4*>(buf + lrow + ((P + n) * 3 + s) * PS + j * 256);
      floatx4 t[TD];
#pragma unroll
      for (int f = 0; f < TD; ++f) t[f] = floatx4{0.f, 0.f, 0.f, 0.f};
      // smallest part products first, so that each addition loses the least
      constexpr int sd[6] = {0, 2, 1, 0, 1, 0}, sl[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
      for (int c = 0; c < 6; ++c)
#pragma unroll
        for (int n = 0; n < n_; ++n)
#pragma unroll
          for (int f = 0; f < TD; ++f)
            t[f] = DA ? mfma_bf16(fd[n][f][sd[c]], fl[n][sl[c]], t[f]) : mfma_bf16(fl[n][sl[c]], fd[n][f][sd[c]], t[f]);
#pragma unroll
      for (int f = 0; f < TD; ++f) {
        floatx4& a = acc[P == 0 ? 0 : 1][DA ? f : j][DA ? j : f];
#pragma unroll
        for (int v = 0; v < 4; ++v) a[v] = fmaf(sg, t[f][v], a[v]);
      }
      // two staged fragments at a time: more of them read ahead cost registers (the 32 x 128
      // wave tiles spill), one at a time leaves the matrix cores waiting for it
      if (j % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    }
  };
  // The forward's variance products share a chain in the 256 x 64 tiles: a quarter fewer VALU
  // additions (residual block 988 -> 969 us, 64-channel 3 x 3 layer 490 -> 483). In the wider
  // tiles the second set of fragments does not fit the registers, and in the others, and
  // beside element-wise or unaligned loaders, it gains nothing (42 -> 70 channels 119.3 ->
  // 120.1).
  constexpr bool JOIN = PROD == PROD_FWD && NW == 8 && DM == 32 && LM == 64 && KindTraits<KA>::vec4 &&
                        !KindTraits<KA>::any && !KindTraits<KB>::any;
  constexpr int NPASS = JOIN ? 2 : NP;

  if (nk > 0) {
    ls.fetch(os, z, l0, kbeg);
    ld.fetch(od, z, d0, kbeg);
    ls.settle(os, l0, kbeg);
    stage(smem, 0);
  }
  __syncthreads();
  // Tile t is read from buffer t % 2 while tile t + 1 is loaded (before the last product but
  // one), split and stored to the other buffer (after it); the direct operand's next tile is
  // loaded during the last product. The staged and the direct operand's loads in flight are
  // never both held in registers.
  for (int t = 0; t < nk; ++t) {
    const int k0 = kbeg + t * BK;
    const unsigned char* buf = smem + (NBUF == 2 ? (t & 1) * BUF : 0);
    if constexpr (NBUF == 1) ls.fetch(os, z, l0, k0 + BK);
    ld.settle(od, d0, k0);
    static_for<0, NPASS>([&](auto P) {
      if constexpr (NBUF == 2 && P == NPASS - 2) ls.fetch(os, z, l0, k0 + BK);
      product(P, std::integral_constant<int, (JOIN && P == 1) ? 2 : 1>{}, buf, sign(t), [&] {
        if constexpr (P == NPASS - 1) ld.fetch(od, z, d0, k0 + BK);
      });
      if constexpr (NBUF == 2 && P == NPASS - 2) {
        ls.settle(os, l0, k0 + BK);
        stage(smem + ((t + 1) & 1) * BUF, t + 1);
      }
    });
    __syncthreads();
    if constexpr (NBUF == 1) {
      ls.settle(os, l0, k0 + BK);
      stage(smem, t + 1);
      __syncthreads();
    }
  }

  // An infinite or NaN operand, one that h rounds past the bf16 range (above 3.3895e38), or a
  // sum past the fp32 range leaves NaN where the parts of an infinity meet: such a tile is
  // formed again with fp32 MFMAs, so that infinities and NaN come out as fp32 arithmetic gives
  // them (and the tile's other outputs with that kernel's rounding).
  bool bad = false;
#pragma unroll
  for (int o = 0; o < 2; ++o)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) bad |= !(fabsf(acc[o][i][j][v]) <= FLT_MAX);
  if (__syncthreads_or(bad)) {
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[o][i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    float* raw = reinterpret_cast<float*>(smem);
    for (int t = 0; t < nk; ++t) {
      __syncthreads();
      ls.fetch(os, z, l0, kbeg + t * BK);
      ld.fetch(od, z, d0, kbeg + t * BK);
      ls.settle(os, l0, kbeg + t * BK);
      ld.settle(od, d0, kbeg + t * BK);
#pragma unroll
      for (int u = 0; u < LS::NU; ++u) {
        int mn, k;
        LS::unit_pos(tid, u, mn, k);
#pragma unroll
        for (int j = 0; j < LS::UR; ++j)
#pragma unroll
          for (int e = 0; e < LS::KG; ++e)
#pragma unroll
            for (int n = 0; n < NL; ++n) raw[(n * BK + k + e) * LM + mn + j] = sraw(n, u, j, e);
      }
      __syncthreads();
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int j = 0; j < TL; ++j) {
          const float r0 = raw[(8 * q + e) * LM + j * 16 + rl];
          const float r1 = NL == 2 ? raw[((NL - 1) * BK + 8 * q + e) * LM + j * 16 + rl] : 0.f;
          static_for<0, NP>([&](auto P) {
            const float l = prod_operand<PROD, DA, P>(r0, r0, r1);
#pragma unroll
            for (int f = 0; f < TD; ++f) {
              const float d = dval(P, f, e);
              floatx4& a = acc[P == 0 ? 0 : 1][DA ? f : j][DA ? j : f];
              a = DA ? __builtin_amdgcn_mfma_f32_16x16x4f32(d, l, a, 0, 0, 0)
                     : __builtin_amdgcn_mfma_f32_16x16x4f32(l, d, a, 0, 0, 0);
            }
          });
        }
    }
    __syncthreads();
  }
  gemm_epilogue<16, BM, BN, WM, WN, NTH, KA, EPI, false, false, SM / 4, !DA && LD::FV == 2, EK>(
      g, z, zz, bp.R, bp.m0, bp.n0, bp.tmi, tid, acc[0], acc[1], reinterpret_cast<float*>(smem), nullptr, nullptr,
      nullptr);
}

template <int PROD, class CFG, int KA, int KB, int EPI>
void launch_cfg(const GemmArgs& g, int64_t grid_x, int64_t grid_y, hipStream_t s) {
  const dim3 grid((unsigned)grid_x, (unsigned)grid_y);
  if constexpr (CFG::X)
    hipLaunchKernelGGL((gemm_split_kernel<PROD, CFG, KA, KB, EPI>), grid, dim3(CFG::NTH), 0, s, g);
  else
    hipLaunchKernelGGL((gemm_kernel<PROD, CFG, KA, KB, EPI>), grid, dim3(CFG::NTH), 0, s, g);
}

}  // namespace tagi
