// Outer attention of one map over long sequences (reference
// src/double_attention/ops.py:65-93): O = softmax(gamma q k^T, causal) V, the
// key range of a query tile cut into pieces that fill the chip.
//
// A workgroup of eight waves owns 128 queries and DS value features.  Per step
// (32 keys):
//   S^T[key, q] = K Q^T   the score tile's 16 x 16 blocks are dealt to the
//       waves: each holds its queries in VGPRs and reads its key rows from LDS;
//   P^T                   packed as MFMA B operands (da_common.h) into LDS;
//   O^T[f, q] += V^T P^T  each wave owns DS/8 features of all QT queries: it
//       reads P from LDS, and its V^T rows straight from global memory (the
//       32-token tiles make a wave's 16 rows one contiguous KiB; no other wave
//       of the workgroup needs them).
// So the scores are formed once for 256 or 512 value features (the general
// kernel's waves keep P in registers and repeat them per slice).  What bounds
// a step at 256-wide scores and 512 features (1536 clocks of MFMA work): 128
// KiB of key and 64 KiB of P reads from LDS at 128 bytes per clock, 48 KiB of
// loads at 64 bytes per clock, and the barrier; measured about 3200 clocks.
// Step u multiplies P(u) while it forms the scores of u+1, so the
// exponentials run beside MFMAs, with one barrier per step.  Key tiles reach
// a two-buffer LDS ring by global->LDS DMA issued at the start of a step; V^T
// loads are issued when the previous tile's registers are free.  Two waves
// share a SIMD (at most 256 registers).  Measured (us, bf16, causal, against
// the general kernel with its stream split): 1 x 8192 tokens at 256-wide scores
// 75 / 91, 4 x 2048 at 512-wide 57 / 68; the modules' forwards 138 -> 118 and
// 179 -> 165.
#include <algorithm>
#include <type_traits>

#include "da_common.h"
#include "da_launch.h"
#include "da_tile.h"

namespace da {

namespace {

constexpr int kTileWaves = 8;
constexpr int kTileQueries = 128;   // queries of a workgroup
constexpr int kTileKeys = 32;       // keys of a step

struct TileParams {
  const void* q;
  const void* k;
  int64_t qk_stride_b, qk_stride_t;
  const void* vt;
  int64_t vt_stride_b;
  int T, D;
  int n_qt, n_slices;
  int items;            // work items per (sequence, slice)
  int piece_group;      // causal split: query tile i has i / piece_group + 1 pieces (0: unsplit)
  int n_pieces;         // pieces of every query tile otherwise
  int piece_len;        // key tiles per piece
  char* part;           // split: [sequence x slice][item] slots
  int piece_es;         // bytes of a piece's element (2: the value type, 4: fp32)
  const void* scales;
  int scales_dtype;
  float scale_mult;
  int flags;
  float score_bound;
  void* out;
  int64_t out_stride_b, out_stride_t;
};

// Work items of a (sequence, slice).  Unsplit: item = query tile, heaviest
// first.  Split: a query tile's keys are cut into pieces of piece_len tiles
// (the last one shorter), and items go piece by piece, so the workgroups of
// one XCD walk the same keys at the same time and its L2 serves them.  In a
// causal problem query tile i has i / piece_group + 1 pieces.
struct Item {
  int qt, piece;
};
__host__ __device__ inline int tile_pieces(int qt, int piece_group, int n_pieces) {
  return piece_group > 0 ? qt / piece_group + 1 : n_pieces;
}
__device__ __forceinline__ Item tile_item(int idx, int n_qt, int piece_group, int n_pieces) {
  if (piece_group == 0) return n_pieces == 1 ? Item{n_qt - 1 - idx, 0} : Item{idx % n_qt, idx / n_qt};
  int y = 0;
  while (idx >= n_qt - y * piece_group) {
    idx -= n_qt - y * piece_group;
    ++y;
  }
  return Item{n_qt - 1 - idx, y};
}
// Slot of piece `piece` of query tile qt.
__host__ __device__ inline int tile_slot(int qt, int piece, int piece_group, int n_pieces) {
  if (piece_group == 0) return qt * n_pieces + piece;
  const int g = qt / piece_group;
  return piece_group * (g * (g + 1) / 2) + (qt - g * piece_group) * (g + 1) + piece;
}

__host__ __device__ inline int64_t piece_slot_bytes(int QT, int DS, int es) {
  return static_cast<int64_t>(QT) * DS * es + 8 * static_cast<int64_t>(QT);
}

// Four features in fp32 or in the value type.
template <typename TV>
__device__ __forceinline__ void store_features(char* dst, int es, f32x4 v) {
  if (es == 4) {
    *reinterpret_cast<f32x4*>(dst) = v;
  } else {
    typename Elem<TV>::v4 h;
#pragma unroll
    for (int r = 0; r < 4; ++r) h[r] = static_cast<TV>(v[r]);
    *reinterpret_cast<typename Elem<TV>::v4*>(dst) = h;
  }
}

}  // namespace

// W: score width.
template <typename TV, int W, int DS>
__global__ __launch_bounds__(kTileWaves * 64) void attention_tile_kernel(TileParams p) {
  typedef _Float16 TQ;
  typedef typename Elem<TQ>::v8 q8;
  typedef typename Elem<TV>::v8 v8;
  constexpr int QT = kTileQueries, KT = kTileKeys;
  // Score blocks of a wave, queries x keys: two query blocks halve the key
  // reads from LDS; with 128 x 512 accumulators only one block's queries fit.
  constexpr int QPW = DS == 512 ? 1 : 2;
  constexpr int KPW = QPW == 1 ? 2 : 1;
  constexpr int QB = QT / 16;                  // query blocks
  constexpr int NKG = KT / 16 / KPW;           // waves along the keys
  static_assert(NKG * (QB / QPW) == kTileWaves, "the score blocks go round the waves");
  constexpr int KS = W / 32;                   // 32-deep steps
  constexpr int FB = DS / 128;                 // 16-feature blocks per wave
  constexpr int NCK = W / 8;
  typedef XorTile<KT, NCK, true> KTile;
  constexpr int KCH = KTile::LOADS / kTileWaves;   // wave loads of a key tile per wave
  constexpr int PBYTES = QB * 1024;
  // The P buffers also take the exchanges of row maxima and sums.
  constexpr int OFF_P = 2 * KTile::BYTES, OFF_X = OFF_P;
  static_assert(NKG * QT * 4 <= 2 * PBYTES, "the exchange fits the P buffers");
  __shared__ __attribute__((aligned(1024))) char lds[OFF_P + 2 * PBYTES];

  const int lane = lane_id();
  const int c = lane & 15, g = lane >> 4;
  const int wave = uniform_wave();
  const int kg = wave % NKG, qg = wave / NKG;   // this wave's score blocks
  const ScalarHalves scale_raw = fetch_scalar(p.scales, p.scales_dtype, 0);   // issued first, used later
  const bool causal = p.flags & kAttnCausal;

  // Workgroups are dealt to the XCDs round-robin; each XCD takes a contiguous
  // range of (sequence, item, slice), so a sequence's keys and values stay in
  // one L2.  Items run heaviest first.
  const int n_wg = static_cast<int>(gridDim.x);
  const int wg = static_cast<int>(blockIdx.x);
  const int xcd = wg % kXcds, per_xcd = n_wg / kXcds, rem_xcd = n_wg % kXcds;
  const int logical = xcd * per_xcd + min(xcd, rem_xcd) + wg / kXcds;
  const int slice = logical % p.n_slices;
  const int bi = logical / p.n_slices;
  const int b = bi / p.items;
  const Item it = tile_item(bi - b * p.items, p.n_qt, p.piece_group, p.n_pieces);
  const int q0 = it.qt * QT;
  const int n_kt = causal ? (min(q0 + QT, p.T) - 1) / KT + 1 : (p.T + KT - 1) / KT;
  const int kt0 = it.piece * p.piece_len, kt1 = min(n_kt, kt0 + p.piece_len);

  const TQ* qbase = static_cast<const TQ*>(p.q) + b * p.qk_stride_b;
  const char* kbase = reinterpret_cast<const char*>(static_cast<const TQ*>(p.k) + b * p.qk_stride_b);
  const int ds0 = slice * DS;
  const TV* vbase = static_cast<const TV*>(p.vt) + b * p.vt_stride_b + 32 * (ds0 + wave * FB * 16) + c * 32 + g * 8;
  const int kstride = static_cast<int>(p.qk_stride_t) * 2;

  // This wave's key loads: 1 KiB of the LDS tile each, filled by global->LDS
  // DMA (lane l's 16 bytes land at slot l).
  uint32_t koff[KCH];
#pragma unroll
  for (int i = 0; i < KCH; ++i) {
    int row, ck;
    KTile::slot_chunk((i * kTileWaves + wave) * 64 + lane, row, ck);
    koff[i] = static_cast<uint32_t>(row * kstride + ck * 16);
  }
  // Keys of tile kt into its buffer (the parity of kt).  Past the run's last
  // tile that one is loaded again, into a buffer that nothing reads any more.
  auto load_keys = [&](int kt) {
    const int k0 = min(kt, kt1 - 1) * KT;
    const char* src = uniform_ptr(kbase + static_cast<int64_t>(k0) * kstride);
    char* dst = lds + (kt & 1) * KTile::BYTES + wave * 1024;
    if (k0 + KT <= p.T) {
#pragma unroll
      for (int i = 0; i < KCH; ++i) dma16(src + koff[i], dst + i * kTileWaves * 1024);
    } else {   // rows past the end re-read the last one
#pragma unroll
      for (int i = 0; i < KCH; ++i) {
        int row, ck;
        KTile::slot_chunk((i * kTileWaves + wave) * 64 + lane, row, ck);
        dma16(src + static_cast<uint32_t>(min(row, p.T - 1 - k0) * kstride + ck * 16), dst + i * kTileWaves * 1024);
      }
    }
  };
  v8 vreg[FB];
  auto load_values = [&](int kt) {
    const TV* src = vbase + static_cast<int64_t>(kt) * 32 * p.D;
#pragma unroll
    for (int f = 0; f < FB; ++f) vreg[f] = load8(src + f * 16 * 32);
  };

  // Queries (rows past the end repeat the last one), then the first tiles.
  q8 qf[QPW][KS];
  int qrow[QPW];
#pragma unroll
  for (int i = 0; i < QPW; ++i) {
    qrow[i] = q0 + (qg * QPW + i) * 16 + c;
    const TQ* src = qbase + static_cast<int64_t>(min(qrow[i], p.T - 1)) * p.qk_stride_t + 8 * g;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) qf[i][kk] = load8(src + kk * 32);
  }
  load_keys(kt0);
  load_keys(kt0 + 1);
  // Nothing that uses a loaded value moves above the loads' issue.
  __builtin_amdgcn_sched_barrier(0);
  wait_vmem();
  float sc = scalar_value(scale_raw, p.scales_dtype);   // may be negative: only |q . k| is bounded
  if (p.flags & kAttnScalesAreLog) sc = expf(fminf(fmaxf(sc, kLogScaleMin), kLogScaleMax));
  sc *= p.scale_mult * kLog2e;

  int kfrag[KS < 4 ? KS : 4];
#pragma unroll
  for (int k = 0; k < (KS < 4 ? KS : 4); ++k) kfrag[k] = KTile::base(c, g, k) + kg * KPW * KTile::ROW_BLOCK;
  // Scores of tile kt: lane (c, g) element e of block (i, kb) is
  // key key_of(kt, kb, e) for query qrow[i].
  auto scores = [&](int kt, f32x4 (&st)[QPW][KPW]) {
    const char* tile = lds + (kt & 1) * KTile::BYTES;
#pragma unroll
    for (int i = 0; i < QPW; ++i)
#pragma unroll
      for (int kb = 0; kb < KPW; ++kb) st[i][kb] = zero4();
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
#pragma unroll
      for (int kb = 0; kb < KPW; ++kb) {
        const q8 a = lds_v8<TQ>(tile + kfrag[kk & 3] + 256 * (kk >> 2) + kb * KTile::ROW_BLOCK);
#pragma unroll
        for (int i = 0; i < QPW; ++i) st[i][kb] = Elem<TQ>::mma(a, qf[i][kk], st[i][kb]);
      }
    }
    // Four fragments stay in flight ahead of their MFMAs (left to itself the
    // compiler reads one, waits, and multiplies).
    constexpr int FR = KS * KPW, AHEAD = FR < 4 ? FR : 4;
    __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
    for (int n = 0; n < FR - AHEAD; ++n) {
      __builtin_amdgcn_sched_group_barrier(0x008, QPW, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, AHEAD * QPW, 0);
  };
  auto key_of = [&](int kt, int kb, int e) {
    const int blk = kg * KPW + kb;
    return kt * KT + 32 * (blk >> 1) + 8 * g + 4 * (blk & 1) + e;
  };
  // Steps that hold no masked key for any query of the tile need no mask.
  auto needs_mask = [&](int kt) { return (causal && kt * KT + KT - 1 > q0) || kt * KT + KT > p.T; };
  auto visible = [&](int key, int i) { return key < p.T && (!causal || key <= qrow[i]); };

  f32x4 acc[FB][QB];
#pragma unroll
  for (int f = 0; f < FB; ++f)
#pragma unroll
    for (int i = 0; i < QB; ++i) acc[f][i] = zero4();
  float l_part[QPW];
#pragma unroll
  for (int i = 0; i < QPW; ++i) l_part[i] = 0.f;

  // The fixed reference bound * sc when every probability then stays in
  // bf16's range, else each row's maximum from a pass over the keys.
  const bool fixed = p.score_bound > 0.f && std::is_same<TV, __bf16>::value && 2.f * p.score_bound * fabsf(sc) <= 120.f;
  float xs[QPW], ref[QPW];   // a row's reference, and what is added to its scaled scores
#pragma unroll
  for (int i = 0; i < QPW; ++i) {
    xs[i] = p.score_bound * fabsf(sc);
    ref[i] = -xs[i];
  }
  if (!fixed) {
    float mx[QPW];
#pragma unroll
    for (int i = 0; i < QPW; ++i) mx[i] = -INFINITY;
    for (int kt = kt0; kt < kt1; ++kt) {
      wait_vmem();
      lds_barrier();
      if (kt > kt0) load_keys(kt + 1);
      f32x4 st[QPW][KPW];
      scores(kt, st);
#pragma unroll
      for (int i = 0; i < QPW; ++i)
#pragma unroll
        for (int kb = 0; kb < KPW; ++kb)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (visible(key_of(kt, kb, e), i)) mx[i] = fmaxf(mx[i], st[i][kb][e] * sc);
    }
    float* xch = reinterpret_cast<float*>(lds + OFF_X);
#pragma unroll
    for (int i = 0; i < QPW; ++i) {
      const float m = group_max(mx[i]);
      if (g == 0) xch[kg * QT + (qg * QPW + i) * 16 + c] = m;
    }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < QPW; ++i) {
      float m = -INFINITY;
#pragma unroll
      for (int w = 0; w < NKG; ++w) m = fmaxf(m, xch[w * QT + (qg * QPW + i) * 16 + c]);
      xs[i] = m;
      ref[i] = m == -INFINITY ? 0.f : -m;
    }
    // The pipeline restarts at the first tile (every wave is past its reads
    // of both key buffers; the barrier below is past the exchange's).
    wait_vmem();
    load_keys(kt0);
    load_keys(kt0 + 1);
    wait_vmem();
  }

  // Scores of tile kt, turned into probabilities in its P buffer.
  auto probabilities = [&](int kt) {
    char* dst = lds + OFF_P + (kt & 1) * PBYTES;
    f32x4 pr[QPW][KPW];
    scores(kt, pr);
#pragma unroll
    for (int i = 0; i < QPW; ++i)
#pragma unroll
      for (int kb = 0; kb < KPW; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e) pr[i][kb][e] = __builtin_amdgcn_exp2f(__builtin_fmaf(pr[i][kb][e], sc, ref[i]));
    if (needs_mask(kt)) {
#pragma unroll
      for (int i = 0; i < QPW; ++i)
#pragma unroll
        for (int kb = 0; kb < KPW; ++kb)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (!visible(key_of(kt, kb, e), i)) pr[i][kb][e] = 0.f;
    }
#pragma unroll
    for (int i = 0; i < QPW; ++i) {
#pragma unroll
      for (int kb = 0; kb < KPW; ++kb) l_part[i] += (pr[i][kb][0] + pr[i][kb][1]) + (pr[i][kb][2] + pr[i][kb][3]);
      // B operand of the query block: 16 bytes per lane, key half kb.
      if constexpr (KPW == 2) {
        *reinterpret_cast<v8*>(dst + ((qg * QPW + i) * 64 + lane) * 16) = pack_blocked<TV>(pr[i][0], pr[i][1]);
      } else {
        typename Elem<TV>::v4 h;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = static_cast<TV>(pr[i][0][e]);
        *reinterpret_cast<typename Elem<TV>::v4*>(dst + ((qg * QPW + i) * 64 + lane) * 16 + kg * 8) = h;
      }
    }
  };
  // O^T += V^T(kt) P^T(kt).
  auto multiply = [&](int kt) {
    const char* pb = lds + OFF_P + (kt & 1) * PBYTES + lane * 16;
#pragma unroll
    for (int i = 0; i < QB; ++i) {
      const v8 pf = lds_v8<TV>(pb + i * 1024);
#pragma unroll
      for (int f = 0; f < FB; ++f) acc[f][i] = Elem<TV>::mma(vreg[f], pf, acc[f][i]);
    }
    constexpr int FR = QB, AHEAD = 3;
    __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
    for (int n = 0; n < FR - AHEAD; ++n) {
      __builtin_amdgcn_sched_group_barrier(0x008, FB, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, AHEAD * FB, 0);
  };

  lds_barrier();   // keys of kt0 and kt0 + 1
  load_values(kt0);
  __builtin_amdgcn_sched_barrier(0);
  probabilities(kt0);

  // Step kt finds P(kt) and the keys of kt + 1 in LDS; the key buffer of kt
  // and the P buffer of kt - 1 are free.  The key loads land behind the
  // step's products; the value loads of kt + 1 follow them.
  for (int kt = kt0; kt + 1 < kt1; ++kt) {
    lds_barrier();
    load_keys(kt + 2);
    __builtin_amdgcn_sched_barrier(0);
    multiply(kt);
    wait_vmem();
    load_values(kt + 1);
    __builtin_amdgcn_sched_barrier(0);
    probabilities(kt + 1);
    __builtin_amdgcn_sched_barrier(0);
  }
  lds_barrier();
  multiply(kt1 - 1);

  // Row sums over the waves along the keys, then the outputs: lane (c, g)
  // holds features ds0 + 16 (wave FB + f) + 4g + r of query q0 + 16 i + c.
  float* xch = reinterpret_cast<float*>(lds + OFF_X);
  lds_barrier();
#pragma unroll
  for (int i = 0; i < QPW; ++i) {
    const float l = group_sum(l_part[i]);
    if (g == 0) xch[kg * QT + (qg * QPW + i) * 16 + c] = l;
  }
  lds_barrier();
  const bool partial = tile_pieces(it.qt, p.piece_group, p.n_pieces) > 1;
  char* slot = nullptr;
  if (partial) {
    slot = p.part + (static_cast<int64_t>(b * p.n_slices + slice) * p.items +
                     tile_slot(it.qt, it.piece, p.piece_group, p.n_pieces)) * piece_slot_bytes(QT, DS, p.piece_es);
    if (kg == 0 && g == 0) {
      float* stats = reinterpret_cast<float*>(slot + static_cast<int64_t>(QT) * DS * p.piece_es);
#pragma unroll
      for (int i = 0; i < QPW; ++i) {
        const int ql = (qg * QPW + i) * 16 + c;
        float l = 0.f;
#pragma unroll
        for (int w = 0; w < NKG; ++w) l += xch[w * QT + ql];
        stats[ql] = xs[i];
        stats[QT + ql] = l;
      }
    }
  }
  const int es = partial ? p.piece_es : (p.flags & kAttnOutF32) ? 4 : 2;
#pragma unroll
  for (int i = 0; i < QB; ++i) {
    float l = 0.f;
#pragma unroll
    for (int k = 0; k < NKG; ++k) l += xch[k * QT + i * 16 + c];
    const float w = 1.f / (l > 0.f ? l : 1.f);
    const int tq = q0 + i * 16 + c;
    const int64_t at = partial ? static_cast<int64_t>(i * 16 + c) * DS + wave * FB * 16
                               : b * p.out_stride_b + static_cast<int64_t>(tq) * p.out_stride_t + ds0 + wave * FB * 16;
    char* dst = (partial ? slot : static_cast<char*>(p.out)) + at * es;
    if (!partial && tq >= p.T) continue;
#pragma unroll
    for (int f = 0; f < FB; ++f) store_features<TV>(dst + (f * 16 + 4 * g) * es, es, acc[f][i] * w);
  }
}

// Merge of a query tile's pieces: O = sum 2^(m_c - M) l_c o_c / sum 2^(m_c - M) l_c
// per row.
template <typename TV, int DS, int PE>
__global__ __launch_bounds__(256) void attention_tile_merge_kernel(TileParams p) {
  // Eight features per lane; a wave takes 512 / DS rows at a time, RW times.
  constexpr int QT = kTileQueries, LPR = DS / 8, RPP = 64 / LPR, RW = 2, AHEAD = 2;
  static_assert(LPR <= 64, "a row fits a wave");
  const int qt = static_cast<int>(blockIdx.y);
  const int first = tile_slot(qt, 0, p.piece_group, p.n_pieces);
  const int n = tile_pieces(qt, p.piece_group, p.n_pieces);
  if (n == 1) return;
  const int b = static_cast<int>(blockIdx.x) / p.n_slices;
  const int ds0 = (static_cast<int>(blockIdx.x) - b * p.n_slices) * DS;
  const int lane = lane_id();
  const int d8 = (lane % LPR) * 8;
  const int r0 = (static_cast<int>(blockIdx.z) * 4 + uniform_wave()) * RW * RPP + lane / LPR;
  const int64_t bytes = piece_slot_bytes(QT, DS, PE);
  const char* base = p.part + (static_cast<int64_t>(blockIdx.x) * p.items + first) * bytes;
  float M[RW], den[RW], o[RW][8];
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    M[r] = -INFINITY;
    den[r] = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[r][e] = 0.f;
  }
  for (int y = 0; y < n; y += AHEAD) {
    // The loads of AHEAD pieces fly together (past the last piece its own are
    // repeated and dropped).
    float m[AHEAD][RW], l[AHEAD][RW];
    u32x4 v[AHEAD][RW][PE / 2];
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) {
      const char* pc = base + min(y + k, n - 1) * bytes;
      const float* stats = reinterpret_cast<const float*>(pc + static_cast<int64_t>(QT) * DS * PE);
#pragma unroll
      for (int r = 0; r < RW; ++r) {
        const int row = r0 + r * RPP;
        m[k][r] = stats[row];
        l[k][r] = stats[QT + row];
#pragma unroll
        for (int h = 0; h < PE / 2; ++h) v[k][r][h] = load16B(pc + (static_cast<int64_t>(row) * DS + d8) * PE + 16 * h);
      }
    }
#pragma unroll
    for (int k = 0; k < AHEAD; ++k)
#pragma unroll
      for (int r = 0; r < RW; ++r) {
        // A piece with every key of the row masked has the sum 0; a NaN sum is
        // a NaN score and goes on to the output, as it does without a split.
        if (y + k >= n || l[k][r] == 0.f) continue;
        const float Mn = fmaxf(M[r], m[k][r]);
        const float f_old = M[r] == -INFINITY ? 0.f : exp2f(M[r] - Mn);
        const float wl = exp2f(m[k][r] - Mn) * l[k][r];
        den[r] = den[r] * f_old + wl;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float x;
          if constexpr (PE == 4) {
            x = __uint_as_float(v[k][r][e >> 2][e & 3]);
          } else {
            x = static_cast<float>(__builtin_bit_cast(typename Elem<TV>::v8, v[k][r][0])[e]);
          }
          o[r][e] = o[r][e] * f_old + x * wl;
        }
        M[r] = Mn;
      }
  }
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    const int tq = qt * QT + r0 + r * RPP;
    if (tq >= p.T) continue;
    const float w = den[r] == 0.f ? 0.f : 1.f / den[r];
    const int es = (p.flags & kAttnOutF32) ? 4 : 2;
    char* dst = static_cast<char*>(p.out) +
                (b * p.out_stride_b + static_cast<int64_t>(tq) * p.out_stride_t + ds0 + d8) * es;
    if (es == 4) {
      *reinterpret_cast<f32x4*>(dst) = f32x4{o[r][0], o[r][1], o[r][2], o[r][3]} * w;
      *reinterpret_cast<f32x4*>(dst + 16) = f32x4{o[r][4], o[r][5], o[r][6], o[r][7]} * w;
    } else {
      typename Elem<TV>::v8 h;
#pragma unroll
      for (int e = 0; e < 8; ++e) h[e] = static_cast<TV>(o[r][e] * w);
      // 16-bit outputs and their strides may be 8-byte aligned only.
      const u32x4 bits = __builtin_bit_cast(u32x4, h);
      *reinterpret_cast<u32x2*>(dst) = u32x2{bits[0], bits[1]};
      *reinterpret_cast<u32x2*>(dst + 8) = u32x2{bits[2], bits[3]};
    }
  }
}

namespace {

constexpr int64_t kTileCUs = 256;

// What a launch needs: value slice width and the split of its work.
struct TilePlan {
  bool fits;
  int ds, piece_group, n_pieces, piece_len, items, piece_es;
  int64_t part_bytes;
};

TilePlan plan_tile(int64_t B, int64_t S, int64_t T, int64_t D, int64_t W, bool causal, int out_es) {
  TilePlan t{};
  // Sequences long enough to give every piece a run of key tiles.
  if (S != 1 || D % 256 || !(W == 256 || W == 512) || T < (W == 512 ? 1024 : 2048)) return t;
  t.fits = true;
  // Value slices as wide as the registers allow: the scores are formed once
  // per slice.
  t.ds = W == 256 && D % 512 == 0 ? 512 : 256;
  const int64_t n_qt = (T + kTileQueries - 1) / kTileQueries, slices = D / t.ds;
  t.items = static_cast<int>(n_qt);
  t.n_pieces = 1;
  t.piece_len = static_cast<int>((T + kTileKeys - 1) / kTileKeys);
  // Key ranges are split when the heaviest query tile holds well over an even
  // share of all steps.
  const int64_t per = kTileQueries / kTileKeys;   // key tiles a causal query tile adds
  const int64_t n_last = t.piece_len;
  const int64_t all = causal ? per * n_qt * (n_qt + 1) / 2 : n_qt * n_last;
  const int64_t share = std::max<int64_t>(16, B * slices * all / kTileCUs);
  if (n_last <= share + share / 2) return t;
  if (causal) {
    // The shortest pieces that keep the items within one round of CUs.
    auto items = [&](int64_t group) { return tile_slot(static_cast<int>(n_qt), 0, static_cast<int>(group), 1); };
    int64_t group = std::max<int64_t>(1, share / per);
    while (group < n_qt && B * slices * items(group) > kTileCUs) ++group;
    if (group < n_qt) {
      t.piece_group = static_cast<int>(group);
      t.piece_len = static_cast<int>(group * per);
      t.items = static_cast<int>(items(group));
    }
  } else {
    // The fewest pieces with the shortest rounds of CUs: a few workgroups past
    // a round cost a whole one (bf16, 256-wide scores, 3 x 2500 tokens, D 256: five
    // pieces, 300 workgroups, 57 us; four, 240 workgroups, 40 us).
    double best = 0;
    for (int64_t pieces = 1; pieces <= (n_last + share - 1) / share; ++pieces) {
      const int64_t len = (n_last + pieces - 1) / pieces, n = (n_last + len - 1) / len;
      const double steps = dealt_steps(B, slices, n_qt * n, kTileCUs / kXcds, static_cast<double>(len) + kLaunchSteps, 0);
      if (pieces > 1 && steps >= best) continue;
      best = steps;
      t.piece_len = static_cast<int>(len);
      t.n_pieces = static_cast<int>(n);
      t.items = static_cast<int>(n_qt * n);
    }
  }
  if (t.items == n_qt) return t;
  // Pieces are fp32, unless the general kernel would split this call's keys
  // too and round its pieces to the output's 16 bits.  Their error against 64
  // bits is then the same (bf16, causal: 1 x 8192 tokens 2.35e-3 there, 2.38e-3
  // here; 4 x 2048 2.40e-3 both); where it does not split, 16-bit pieces would add
  // a rounding (2 x 2500 without a mask 2.36e-3 there, 2.89e-3 with them).
  t.piece_es = out_es == 2 && plan_attention(B, S, T, D, W, false, causal, true, 2).part_bytes > 0 ? 2 : 4;
  t.part_bytes = B * slices * t.items * piece_slot_bytes(kTileQueries, t.ds, t.piece_es);
  return t;
}

// As attention_general_us, fitted to the same shapes.
double tile_us(const TilePlan& t, int64_t B, int64_t T, int64_t D, int64_t W, bool causal, bool fixed) {
  const double step = W == 512 ? (fixed ? 1.47 : 2.26) : t.ds == 512 ? (fixed ? 1.26 : 1.85) : (fixed ? 1.03 : 1.53);
  const int64_t n_qt = (T + kTileQueries - 1) / kTileQueries;
  const double fall = causal && t.items == n_qt ? kTileQueries / kTileKeys : 0;
  const double steps = dealt_steps(B, D / t.ds, t.items, kTileCUs / kXcds, t.piece_len + kLaunchSteps, fall);
  if (t.part_bytes == 0) return (fixed ? 6 : 1) + step * steps;
  const double start = W == 512 ? 8.5 : t.ds == 512 ? 13 : 10, per_mb = W == 512 ? 0.30 : t.ds == 512 ? 0.15 : 0.25;
  return start + per_mb * 1e-6 * static_cast<double>(t.part_bytes) + step * steps;
}

// Whether this kernel beats the general one, by the predicted times of both.
// It forms the scores fewer times, but the general kernel's smaller query tiles
// fill the chip better in some calls, above all where its value slices are as
// wide (us, bf16, here / there: 4 x 5000 causal, 256-wide scores, D 768 269 / 245;
// 1 x 2048 without a mask, D 512 37.6 / 33.3; but 1 x 8192 causal 76 / 93).  With row
// maxima (fp16 values, or no bound) it forms them twice, and the general one
// rescales as it goes: fp16, 1 x 8192 causal 98 / 121 at 256-wide scores, 234 / 206 at
// 512-wide.  A bf16 call with a bound runs fixed exponents up to a gamma of about
// 41 and maxima past it, which only the device knows: it has to win with the
// one and not lose 10 % with the other.  Over the shapes that the constants
// were fitted to, the slowest choices are 6 % over the general kernel's time (a
// few with fp16 values or no bound up to 12 %), where taking every call was up
// to 62 %.
bool tile_wins(const TilePlan& t, int64_t B, int64_t T, int64_t D, int64_t W, bool causal, int out_es, bool bf16,
               bool bounded) {
  auto ratio = [&](AttnExponents mode) {
    return tile_us(t, B, T, D, W, causal, mode == AttnExponents::kFixed) /
           attention_general_us(B, T, D, W, causal, out_es, mode);
  };
  if (!bf16) return ratio(AttnExponents::kMaximaF16) < 1;
  if (!bounded) return ratio(AttnExponents::kMaximaBf16) < 1;
  // The prediction for 512-wide scores is on the high side.
  return ratio(AttnExponents::kFixed) < (W == 512 ? 1.05 : 1) && ratio(AttnExponents::kMaximaBf16) < 1.1;
}

template <typename TV, int W, int DS>
void launch_tile_k(const AttentionArgs& a, const TilePlan& t, const TileParams& p, hipStream_t s) {
  hipLaunchKernelGGL((attention_tile_kernel<TV, W, DS>), dim3(static_cast<unsigned>(a.B * p.n_slices * p.items)),
                     dim3(kTileWaves * 64), 0, s, p);
  if (t.part_bytes == 0) return;
  const dim3 merge(static_cast<unsigned>(a.B * p.n_slices), static_cast<unsigned>(p.n_qt),
                   static_cast<unsigned>(kTileQueries / (8 * (512 / DS))));
  if (t.piece_es == 4) hipLaunchKernelGGL((attention_tile_merge_kernel<TV, DS, 4>), merge, dim3(256), 0, s, p);
  else hipLaunchKernelGGL((attention_tile_merge_kernel<TV, DS, 2>), merge, dim3(256), 0, s, p);
}

template <typename TV>
void launch_tile_t(const AttentionArgs& a, const TilePlan& t, const TileParams& p, hipStream_t s) {
  if (a.RP == 512) launch_tile_k<TV, 512, 256>(a, t, p, s);
  else if (t.ds == 512) launch_tile_k<TV, 256, 512>(a, t, p, s);
  else launch_tile_k<TV, 256, 256>(a, t, p, s);
}

}  // namespace

int64_t attention_tile_bytes(int64_t B, int64_t S, int64_t T, int64_t D, int64_t RP, bool causal, int es) {
  const TilePlan t = plan_tile(B, S, T, D, RP, causal, es);
  if (t.part_bytes == 0) return 0;
  const bool taken = tile_wins(t, B, T, D, RP, causal, es, true, true) || tile_wins(t, B, T, D, RP, causal, es, true, false) ||
                     tile_wins(t, B, T, D, RP, causal, es, false, false);
  return taken ? t.part_bytes : 0;
}

bool launch_attention_tile(const AttentionArgs& a, void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  const int es = (a.flags & kAttnOutF32) ? 4 : 2;
  // Key offsets inside a tile are 32-bit.
  if (a.qk_dtype != kF16 || a.qk_stride_t * 2 * kTileKeys > INT32_MAX) return false;
  const TilePlan t = plan_tile(a.B, a.S, a.T, a.D, a.RP, a.flags & kAttnCausal, es);
  if (!t.fits || t.part_bytes > workspace_bytes) return false;
  if (!tile_wins(t, a.B, a.T, a.D, a.RP, a.flags & kAttnCausal, es, a.v_dtype == kBF16, a.score_bound > 0.f)) return false;
  if (static_cast<int64_t>(a.B) * (a.D / t.ds) * t.items > INT32_MAX) return false;
  TileParams p{};
  p.q = a.q;
  p.k = a.k;
  p.qk_stride_b = a.qk_stride_b;
  p.qk_stride_t = a.qk_stride_t;
  p.vt = a.vt;
  p.vt_stride_b = a.vt_stride_b;
  p.T = a.T;
  p.D = a.D;
  p.n_qt = (a.T + kTileQueries - 1) / kTileQueries;
  p.n_slices = a.D / t.ds;
  p.items = t.items;
  p.piece_group = t.piece_group;
  p.n_pieces = t.n_pieces;
  p.piece_len = t.piece_len;
  p.piece_es = t.piece_es;
  p.part = static_cast<char*>(workspace);
  p.scales = a.scales;
  p.scales_dtype = a.scales_dtype;
  p.scale_mult = a.scale_mult;
  p.flags = a.flags;
  p.score_bound = a.score_bound;
  p.out = a.out;
  p.out_stride_b = a.out_stride_b;
  p.out_stride_t = a.out_stride_t;
  if (a.v_dtype == kBF16) launch_tile_t<__bf16>(a, t, p, stream);
  else launch_tile_t<_Float16>(a, t, p, stream);
  return true;
}

}  // namespace da
