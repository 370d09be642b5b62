// Fused dictionary route for 512-wide rows and for few 256-wide ones (plain
// softmax assignment; route.hip has the contract, the variants, the other rows
// and the rule between them).
//
// A workgroup of eight waves owns QT rows and streams the whole dictionary
// past them, KT atoms per step:
//   S^T[j, c] = Dk^T U^T   the step's 16 x 16 blocks are dealt to the waves:
//       each holds its unit rows in VGPRs and reads its key atoms from LDS;
//   P^T                    packed as MFMA B operands (da_common.h) into LDS;
//   O^T[r, c] += Dv P^T    each wave owns R/8 coordinates of all QT rows: it
//       reads P from LDS and its value atoms straight from memory (the
//       32-atom tiles make a wave's 16 coordinates one contiguous KiB, and no
//       other wave of the workgroup needs them).
// Against four 16-row waves that each read every key and value fragment from
// LDS (256 KiB per 32 atoms of 64 rows at R = 512), this reads 160 KiB, and two
// waves share a SIMD.  What bounds it: the chain of one step (key loads, key
// fragments, exponentials, the P exchange, the barrier), about 3000 clocks for
// 1024 of MFMA work at R = 512.  A third key buffer with loads a whole step
// ahead was slower (80 us against 71 at 16384 rows x 1536 atoms).
// Step t multiplies P(t), turns the logits of t+1 into weights and forms those
// of t+2, one barrier per step; key tiles reach a two-buffer LDS ring by
// global->LDS DMA issued at the start of a step.  With the logits a tile ahead,
// the row maxima that a beta above 9.7 needs are exchanged by that barrier, and
// the sums are scaled as a maximum moves: no pass of its own over the atoms, which
// cost 40 % (R = 512, 1536 atoms, 8192 rows 63 us, now 49).  Fixed-reference
// calls pay 1 to 3 % for it, a barrier before the first step.
// Measured (us, bf16 rows, against route.hip's kernel): beta 8, R = 512 with 1536
// atoms 192 rows 40 / 68, 8192 rows 45 / 69, 12000 rows 60 / 70, 16384 rows 63 / 71,
// 32768 rows 124 / 140; R = 256 with 512 atoms 192 rows 11.3 / 12.9, 8192 rows 12.2 /
// 13.8, 12000 rows 19.8 / 25.6.  Beta 12: R = 512 with 1536 atoms 8192 rows 49 / 86,
// 16384 rows 77 / 86; R = 256 with 1536 atoms 8192 rows 28.9 / 30.7, with 4096 atoms 74 / 77.
#include <type_traits>

#include "da_common.h"
#include "da_launch.h"
#include "da_tile.h"

namespace da {

namespace {

constexpr int kWaves = 8;

struct RouteTileParams {
  const void* x;
  int64_t rows, x_stride;
  const void* key_t;
  const _Float16* value;
  int M, n_tiles;
  const void* beta_ptr;
  int beta_dtype;
  float beta_value, eps;
  int flags;
  void* out;
  int64_t out_stride;
};

}  // namespace

template <typename TX, typename TK, typename TO, int R, int QT, int KT>
// 256-wide rows keep two workgroups per CU.
__global__ __launch_bounds__(kWaves * 64, R == 256 ? 4 : 2) void route_tile_kernel(RouteTileParams p) {
  // x and out may alias (in-place routing): the workgroup has read its rows
  // into VGPRs, a barrier or more before any of its waves writes one.
  typedef typename Elem<TK>::v8 k8;
  constexpr int QB = QT / 16;                  // row blocks
  constexpr int KW = KT / 32;                  // 32-atom windows of a step
  constexpr int NKG = KT / 16;                 // waves along the atoms, one 16-atom block each
  static_assert(NKG * QB == kWaves, "a score block per wave");
  constexpr int KS = R / 32;
  constexpr int FB = R / 128;                  // 16-coordinate blocks per wave
  typedef XorTile<KT, R / 8, true> KTile;
  constexpr int KCH = KTile::LOADS / kWaves;   // wave loads of a key tile per wave
  constexpr int PBYTES = KW * QB * 1024;
  constexpr int OFF_P = 2 * KTile::BYTES;
  // The P buffers also take the exchanges of row sums and norms; the maxima of
  // two tiles (a row's from every wave along the atoms) follow them.
  static_assert(NKG * QT * 4 <= PBYTES && kWaves * QT * 4 <= PBYTES, "the exchanges fit a P buffer each");
  constexpr int OFF_M = OFF_P + 2 * PBYTES, MBYTES = QT * NKG * 4;
  __shared__ __attribute__((aligned(1024))) char lds[OFF_M + 2 * MBYTES];

  const int lane = lane_id();
  const int c = lane & 15, g = lane >> 4;
  const int wave = uniform_wave();
  const int kg = wave % NKG, qg = wave / NKG;   // this wave's score block
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * QT;
  const TX* x = static_cast<const TX*>(p.x);

  // One memory round trip: beta, the rows (past the end the last one repeats,
  // never stored) and the first key tiles.
  const ScalarHalves beta_bits = fetch_scalar(p.beta_ptr ? p.beta_ptr : p.x, p.beta_ptr ? p.beta_dtype : kF32, 0);
  typename Elem<TX>::v8 xr[KS];
  const int own = qg * 16 + c;   // this lane's row of the score block
  {
    const int64_t left = p.rows - 1 - row0;
    const TX* src = x + (row0 + (own < left ? own : left)) * p.x_stride + 8 * g;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) xr[kk] = load8(src + kk * 32);
  }
  uint32_t koff[KCH];
#pragma unroll
  for (int i = 0; i < KCH; ++i) {
    int row, ck;
    KTile::slot_chunk((i * kWaves + wave) * 64 + lane, row, ck);
    koff[i] = static_cast<uint32_t>((row * R + ck * 8) * 2);
  }
  // Key atoms of tile t into its buffer (the parity of t); the bank is padded
  // to whole tiles.
  auto load_keys = [&](int t) {
    const char* src = uniform_ptr(static_cast<const char*>(p.key_t) + static_cast<int64_t>(t) * KT * R * 2);
    char* dst = lds + (t & 1) * KTile::BYTES + wave * 1024;
#pragma unroll
    for (int i = 0; i < KCH; ++i) dma16(src + koff[i], dst + i * kWaves * 1024);
  };
  const int n_tiles = p.n_tiles;
  load_keys(0);
  if (n_tiles > 1) load_keys(1);
  // Nothing that uses a loaded value moves above the loads' issue.
  __builtin_amdgcn_sched_barrier(0);
  wait_vmem();

  const float beta_raw = p.beta_ptr ? scalar_value(beta_bits, p.beta_dtype) : p.beta_value;
  const float beta = (p.flags & kRouteBetaIsLog) ? expf(fminf(fmaxf(beta_raw, kLogBetaMin), kLogBetaMax)) : beta_raw;
  // Maxima are taken of raw logits, so a negative beta is folded into the rows.
  const float scale = fabsf(beta) * kLog2e;
  const float sign = beta < 0.f ? -1.f : 1.f;
  // With input normalization the unit row is rounded once to TK; otherwise
  // TK == TX and the raw row passes through unchanged.
  k8 xf[KS];
  float ss = 0.f;
#pragma unroll
  for (int kk = 0; kk < KS; ++kk)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float v = static_cast<float>(xr[kk][e]);
      ss += v * v;
    }
  ss = group_sum(ss);
  const float inv = sign * ((p.flags & kRouteNormalizeInput) ? 1.f / fmaxf(sqrtf(ss), p.eps) : 1.f);
#pragma unroll
  for (int kk = 0; kk < KS; ++kk)
#pragma unroll
    for (int e = 0; e < 8; ++e) xf[kk][e] = static_cast<TK>(static_cast<float>(xr[kk][e]) * inv);

  const _Float16* vbase = p.value + 32 * (wave * FB * 16) + c * 32 + g * 8;
  f16x8 vreg[KW][FB];
  auto load_values = [&](int t) {
    const _Float16* src = vbase + static_cast<int64_t>(t) * KT * R;
#pragma unroll
    for (int w = 0; w < KW; ++w)
#pragma unroll
      for (int f = 0; f < FB; ++f) vreg[w][f] = load8(src + w * 32 * R + f * 16 * 32);
  };

  int kfrag[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) kfrag[k] = KTile::base(c, g, k) + kg * KTile::ROW_BLOCK;
  // Logits of tile t: lane (c, g) element e is atom atom_of(t) + e for row own.
  auto logits = [&](int t) {
    const char* tile = lds + (t & 1) * KTile::BYTES;
    f32x4 st = zero4();
#pragma unroll
    for (int kk = 0; kk < KS; ++kk)
      st = Elem<TK>::mma(lds_v8<TK>(tile + kfrag[kk & 3] + 256 * (kk >> 2)), xf[kk], st);
    // Four fragments stay in flight ahead of their MFMAs.
    constexpr int AHEAD = 4;
    __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
    for (int n = 0; n < KS - AHEAD; ++n) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, AHEAD, 0);
    return st;
  };
  auto atom_of = [&](int t) { return t * KT + 32 * (kg >> 1) + 8 * g + 4 * (kg & 1); };

  // The reference of the exponents: fixed where unit rows and unit atoms bound
  // every logit by 1 and all weights then stay in fp16's normal range, else
  // each row's maximum so far.  The largest weight is at most 2^kRouteP16Lift;
  // the factor cancels in the division by the row sum.
  const bool fixed = (p.flags & kRouteNormalizeInput) && (p.flags & kRouteUnitKeys) && 2.f * scale <= 2.f * kRouteP16Lift;
  float ref = fixed ? kRouteP16Lift - scale : 0.f;

  f32x4 acc[FB][QB];
#pragma unroll
  for (int f = 0; f < FB; ++f)
#pragma unroll
    for (int i = 0; i < QB; ++i) acc[f][i] = zero4();
  float l_part = 0.f;

  // Logits pr of tile t, turned into weights in its P buffer.
  auto weights = [&](int t, f32x4 pr) {
    char* dst = lds + OFF_P + (t & 1) * PBYTES + (kg >> 1) * QB * 1024 + (kg & 1) * 8;
#pragma unroll
    for (int e = 0; e < 4; ++e) pr[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(pr[e], scale, ref));
    if ((t + 1) * KT > p.M) {   // padding atoms weigh nothing
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (atom_of(t) + e >= p.M) pr[e] = 0.f;
    }
    l_part += (pr[0] + pr[1]) + (pr[2] + pr[3]);
    f16x4 h;
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = static_cast<_Float16>(pr[e]);
    *reinterpret_cast<f16x4*>(dst + (qg * 64 + lane) * 16) = h;
  };
  // O^T += Dv(t) P^T(t).
  auto multiply = [&](int t) {
    const char* pb = lds + OFF_P + (t & 1) * PBYTES + lane * 16;
#pragma unroll
    for (int w = 0; w < KW; ++w)
#pragma unroll
      for (int i = 0; i < QB; ++i) {
        const f16x8 pf = lds_v8<_Float16>(pb + (w * QB + i) * 1024);
#pragma unroll
        for (int f = 0; f < FB; ++f) acc[f][i] = Elem<_Float16>::mma(vreg[w][f], pf, acc[f][i]);
      }
    constexpr int FR = KW * QB, AHEAD = FR < 3 ? FR : 3;
    __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
    for (int n = 0; n < FR - AHEAD; ++n) {
      __builtin_amdgcn_sched_group_barrier(0x008, FB, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, AHEAD * FB, 0);
  };

  lds_barrier();   // key tiles 0 and 1
  load_values(0);
  __builtin_amdgcn_sched_barrier(0);
  // Logits run a tile ahead of their weights.  Without the fixed reference the
  // waves along the atoms have so exchanged a tile's row maxima by the step's
  // own barrier.
  auto maxima = [&](int t, const f32x4& st) {
    float mx = -INFINITY;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (atom_of(t) + e < p.M) mx = fmaxf(mx, st[e] * scale);
    mx = group_max(mx);
    if (g == 0) *reinterpret_cast<float*>(lds + OFF_M + (t & 1) * MBYTES + (own * NKG + kg) * 4) = mx;
  };
  float m[QB];   // maxima of rows 16 i + c
#pragma unroll
  for (int i = 0; i < QB; ++i) m[i] = -INFINITY;
  // Tile t's maxima move the reference; the sums so far are scaled to it.
  auto advance = [&](int t) {
#pragma unroll
    for (int i = 0; i < QB; ++i) {
      const float* row = reinterpret_cast<const float*>(lds + OFF_M + (t & 1) * MBYTES) + (16 * i + c) * NKG;
      float mx = m[i];
#pragma unroll
      for (int w = 0; w < NKG; ++w) mx = fmaxf(mx, row[w]);
      if (__ballot(mx > m[i])) {
        const float by = mx > m[i] ? __builtin_amdgcn_exp2f(m[i] - mx) : 1.f;
        m[i] = mx;
#pragma unroll
        for (int f = 0; f < FB; ++f) acc[f][i] *= by;
        if (i == qg) {
          ref = kRouteP16Lift - mx;
          l_part *= by;
        }
      }
    }
  };
  f32x4 st = logits(0);
  if (!fixed) maxima(0, st);
  lds_barrier();   // the maxima of tile 0; its key buffer is free
  if (n_tiles > 2) load_keys(2);
  __builtin_amdgcn_sched_barrier(0);
  if (!fixed) advance(0);
  weights(0, st);
  if (n_tiles > 1) {
    st = logits(1);
    if (!fixed) maxima(1, st);
  }
  // Step t finds P(t), the maxima of t + 1 and the keys of t + 2 in LDS; the
  // key buffer of t + 1 and the P buffer of t - 1 are free.
  wait_vmem();
  for (int t = 0; t + 1 < n_tiles; ++t) {
    lds_barrier();
    if (t + 3 < n_tiles) load_keys(t + 3);
    __builtin_amdgcn_sched_barrier(0);
    multiply(t);
    wait_vmem();
    load_values(t + 1);
    __builtin_amdgcn_sched_barrier(0);
    if (!fixed) advance(t + 1);
    weights(t + 1, st);
    if (t + 2 < n_tiles) {
      st = logits(t + 2);
      if (!fixed) maxima(t + 2, st);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  lds_barrier();
  multiply(n_tiles - 1);

  // Row sums over the waves along the atoms (the first P buffer), then row
  // norms over the waves along the coordinates (the second): r = O / l,
  // z = r / max(||r||, eps).  Lane (c, g) holds coordinates
  // 16 (wave FB + f) + 4g + e of row 16 i + c.
  float* xl = reinterpret_cast<float*>(lds + OFF_P);
  float* xn = reinterpret_cast<float*>(lds + OFF_P + PBYTES);
  lds_barrier();
  l_part = group_sum(l_part);
  if (g == 0) xl[kg * QT + own] = l_part;
  lds_barrier();
  float w[QB];
#pragma unroll
  for (int i = 0; i < QB; ++i) {
    float l = 0.f;
#pragma unroll
    for (int k = 0; k < NKG; ++k) l += xl[k * QT + i * 16 + c];
    w[i] = 1.f / l;
  }
  if (p.flags & kRouteNormalizeOutput) {
#pragma unroll
    for (int i = 0; i < QB; ++i) {
      float rs = 0.f;
#pragma unroll
      for (int f = 0; f < FB; ++f)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = acc[f][i][e] * w[i];
          rs += v * v;
        }
      rs = group_sum(rs);
      if (g == 0) xn[wave * QT + i * 16 + c] = rs;
    }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < QB; ++i) {
      float rs = 0.f;
#pragma unroll
      for (int k = 0; k < kWaves; ++k) rs += xn[k * QT + i * 16 + c];
      w[i] /= fmaxf(sqrtf(rs), p.eps);
    }
  }
#pragma unroll
  for (int i = 0; i < QB; ++i) {
    const int64_t row = row0 + i * 16 + c;
    if (row >= p.rows) continue;
    TO* dst = static_cast<TO*>(p.out) + row * p.out_stride + wave * FB * 16 + 4 * g;
#pragma unroll
    for (int f = 0; f < FB; ++f) {
      typename Elem<TO>::v4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = static_cast<TO>(acc[f][i][e] * w[i]);
      *reinterpret_cast<typename Elem<TO>::v4*>(dst + f * 16) = o;
    }
  }
}

namespace {

template <typename TX, typename TK, typename TO, int R, int QT, int KT>
void launch_k(const RouteArgs& a, hipStream_t s) {
  static_assert(kAtomPad % KT == 0, "the bank is padded to whole tiles");
  RouteTileParams p{};
  p.x = a.x;
  p.rows = a.rows;
  p.x_stride = a.x_stride;
  p.key_t = a.key_t;
  p.value = static_cast<const _Float16*>(a.value);
  p.M = a.M;
  p.n_tiles = static_cast<int>((a.M + KT - 1) / KT);
  p.beta_ptr = a.beta_ptr;
  p.beta_dtype = a.beta_dtype;
  p.beta_value = a.beta_value;
  p.eps = a.eps;
  p.flags = a.flags;
  p.out = a.out;
  p.out_stride = a.out_stride;
  hipLaunchKernelGGL((route_tile_kernel<TX, TK, TO, R, QT, KT>), dim3(static_cast<unsigned>((a.rows + QT - 1) / QT)),
                     dim3(kWaves * 64), 0, s, p);
}

// 512-wide rows: 64 rows per workgroup halve the reads of the dictionary, 32
// spread fewer rows over twice the CUs (1536 atoms: 8192 rows 45 us in one
// round of 32-row workgroups; 12000 rows 60 us in one round of 64-row ones, and
// 83 in two rounds of 32-row ones).
constexpr int64_t kTileCUs = 256;

template <typename TX, typename TK, typename TO>
void launch_t(const RouteArgs& a, hipStream_t s) {
  if (a.R == 256) {
    launch_k<TX, TK, TO, 256, 32, 64>(a, s);
  } else if ((a.rows + 31) / 32 > kTileCUs) {
    launch_k<TX, TK, TO, 512, 64, 32>(a, s);
  } else {
    launch_k<TX, TK, TO, 512, 32, 64>(a, s);
  }
}

}  // namespace

void launch_route_tile(const RouteArgs& a, hipStream_t s) {
  if (a.x_dtype == kBF16) {
    if (a.key_dtype == kF16) {
      if (a.out_dtype == kF16) launch_t<__bf16, _Float16, _Float16>(a, s);
      else launch_t<__bf16, _Float16, __bf16>(a, s);
    } else {
      if (a.out_dtype == kF16) launch_t<__bf16, __bf16, _Float16>(a, s);
      else launch_t<__bf16, __bf16, __bf16>(a, s);
    }
  } else {
    launch_t<_Float16, _Float16, _Float16>(a, s);
  }
}

}  // namespace da
