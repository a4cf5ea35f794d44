// dense_attn.hip -- threshold-masked attention on MFMA tiles with fp32
// probabilities (gfx950): fp32 inputs, and 16-bit inputs below the length at
// which tile_attn.hip takes over.
//
// Same result as sparse_attn.hip (reference dsa_attention.py:234-324), to the
// rounding of its fp32 sums.  The per-query gathers pull every selected K/V
// row for every query (B = 8, T = 1024, HQ = 8, D = 64, k = 64 in fp32: 2.1 GB
// through the CUs' load units, which issue one wave load per ~15 cycles); the
// staged kernel reads each key once per 64 queries but spends ~25 dependent
// VALU instructions on every selected pair.  Here, as in tile_attn.hip, a
// block of 128 queries of one head computes the causal triangle densely on
// the matrix cores with the selection as a bitmask, and the operands that the
// matrix cores have no fp32-rate type for are split into 16-bit pieces whose
// products are exact and summed in fp32:
//   fp32 K, V   two f16 pieces each (23 bits), made once per call by
//               prepare_kernel into the workspace; Q's in registers.
//               S = Kl.Qh + Kh.Ql + Kh.Qh,  O = Vl.Ph + Vh.Pl + Vh.Ph
//   f16 inputs  S as is; P in two f16 pieces:   O = V.Pl + V.Ph
//   bf16 inputs S as is; P in three bf16 pieces (24 bits, exact):
//               O = V.P3 + V.P2 + V.P1
// Scales are powers of two, so exact: a Q row, a head's 64-key tile of K or V
// and, where P takes f16 pieces, a query's probabilities in a tile are scaled
// to put their largest in [2^14, 2^15).  (The scale of the probabilities is a
// multiplication apart from the exponent: added to exp2's argument, 14 would
// cost it four bits for the largest keys.)  A tile's products are summed apart
// and added to O with the scales undone.
//
// Two f16 pieces hold 23 bits down to 2^-15 of what the scale is taken from and
// an absolute error of 2^-39 of it below.  So a probability far below its tile's
// largest loses bits, which matters where the large ones meet a V of next to
// nothing (a key that takes up the attention without adding to it): the result
// is off by at most 2^-32 of sum_tiles (largest p of the tile) (largest |V| of
// the tile) over the normaliser (f16: of the largest |V| of all tiles, no less).
// Rows whose largest output is less than 2^-13 of that are left to redo_kernel,
// so the pieces cost no row more than 2^-19 of its largest output, and most of
// them less than the rounding of fp32 sums (T = 1500, k = 256 fp32, one key with V
// = 0 at a logit 10 above the rest: relative error against float64 4.1e-7, the
// gathers' 7.1e-7; from 12 above on such rows are gathered.  N(0, 1) operands:
// 1.9e-7 against 3.9e-7).
//
// One pass over the scores first (prepare_kernel) writes the selection as one
// bit per pair, unless the select has done so.  Last, redo_kernel gathers
// (attn_tile.h, on the bitmask) the rows the pieces could not carry: those with a
// non-finite result that selected something or below that bound, and the
// 128-query tiles that read a K or V tile non-finite or beyond the scales.  Rows
// that select nothing get 0/0 = NaN, as the reference.
//
// What bounds the dense kernel at D = 64 fp32: per wave and 64-key tile 96
// MFMAs (1536 cycles), ~350 VALU instructions (36 of them exp2 at a quarter of
// the rate, ~1800 cycles) and 42 KB of LDS reads; one SIMD's two waves overlap
// the first two only in part (about 5600 cycles for two tiles, MFMA busy 41%).  B = 4, T = 4096,
// HQ = 8, k = 256 fp32: 253 us in all (prepare 48, 25 where the select has written
// the bitmask; dense 192-200, redo 4.5) against 0.44 ms staged, relative error
// against float64 2.1e-7 against 3.7e-7.
// B = 2, T = 3001, HQ = 16, D = 128, k = 300 f16: 141 us against 862 gathered.
#include <algorithm>
#include <type_traits>

#include "attn_tile.h"
#include "dsa_launch.h"
#include "tile_common.h"

namespace dsa {
namespace {

struct DenseArgs {
  const void* Q;
  const void* K;  // fp32: the high pieces
  const void* V;
  int64_t K_lo;   // fp32: bytes from the high to the low pieces
  int64_t V_lo;
  int64_t B;
  int T;
  int HQ;
  float scale_log2;
  float* out;
  const uint64_t* mask;  // [B*T][W]
  uint32_t* flags;       // [B][128-query tiles][4][HQ]: 32 queries' bits, redo this row
  const uint32_t* kmax;  // fp32: largest |K| bits per [B][HQ][64-key tile]
  const uint32_t* vmax;
};

constexpr uint32_t kBadTile = 0xffffffffu;  // kmax / vmax of a tile the pieces cannot carry

// ---------------------------------------------------------------------------
// One launch prepares the dense kernel's operands, HBM-bound throughout.
//
// Blocks below nconv (fp32 only) turn 64 keys of one head of K and V into f16
// pieces, laid out [B][HQ][T][D], at the scale of the tile's largest
// magnitude (held in registers between the maximum and the conversion), and
// record that magnitude.
//
// The others (none if the select has written the mask: scores null) write the
// selection bitmask: one wave per row, rows longest first, each causal score
// read once (nontemporal, 16 loads in flight per lane), as selection_mask_kernel
// (tile_attn.hip) does.
// ---------------------------------------------------------------------------
struct PrepareArgs {
  const float* scores;
  int64_t ld;
  const float* thr;
  int64_t B;
  int T;
  int HQ;
  const float* K;
  const float* V;
  uint16_t* pieces;  // Kh, Kl, Vh, Vl, `plane` elements apart
  int64_t plane;
  uint32_t* kmax;
  uint32_t* vmax;
  uint32_t nconv;
  uint64_t* mask;
};

template <int D>
__device__ __forceinline__ void convert_tile(const float* __restrict__ X, int64_t b, int h, int tile,
                                             int T, int HQ, uint16_t* __restrict__ hi,
                                             uint16_t* __restrict__ lo, uint32_t* __restrict__ maxbits,
                                             uint32_t* wmax) {
  constexpr int NC = D / 32;  // 8-element chunks per thread (64 rows of D / 256 threads)
  const int tid = threadIdx.x;
  const int64_t bh = b * HQ + h;
  float x[NC][8];
  uint32_t mx = 0u;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int u = tid + 256 * i;
    const int t = min(tile * 64 + u / (D / 8), T - 1);
    load_f32<8>(X + ((b * T + t) * HQ + h) * static_cast<int64_t>(D) + 8 * (u % (D / 8)), x[i]);
  }
#pragma unroll
  for (int i = 0; i < NC; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = max(mx, __float_as_uint(x[i][e]) & 0x7fffffffu);
  mx = wave_extreme_u32<true>(mx);
  if ((tid & 63) == 0) wmax[tid >> 6] = mx;
  block_sync_lds();
  mx = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
  int sh;
  const bool ok = split_scale(mx, sh);
  if (tid == 0) maxbits[bh * ((T + 63) / 64) + tile] = ok ? mx : kBadTile;
  const float sc = ok ? pow2f(sh) : 0.f;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int u = tid + 256 * i;
    const int t = tile * 64 + u / (D / 8);
    if (t >= T) continue;
    uint4 hv, lv;
    split_pair(x[i][0] * sc, x[i][1] * sc, hv.x, lv.x);
    split_pair(x[i][2] * sc, x[i][3] * sc, hv.y, lv.y);
    split_pair(x[i][4] * sc, x[i][5] * sc, hv.z, lv.z);
    split_pair(x[i][6] * sc, x[i][7] * sc, hv.w, lv.w);
    const int64_t to = (bh * T + t) * D + 8 * (u % (D / 8));
    *reinterpret_cast<uint4*>(hi + to) = hv;
    *reinterpret_cast<uint4*>(lo + to) = lv;
  }
}

// D = 0: 16-bit inputs (bitmask only).
template <int D>
__global__ __launch_bounds__(256) void prepare_kernel(PrepareArgs a) {
  const int T = a.T;
  if constexpr (D > 0) {
    __shared__ uint32_t wmax[2][4];
    if (blockIdx.x < a.nconv) {
      const int h = static_cast<int>(blockIdx.x % static_cast<uint32_t>(a.HQ));
      const uint32_t bt = blockIdx.x / static_cast<uint32_t>(a.HQ);
      const int tile = static_cast<int>(bt / static_cast<uint32_t>(a.B));
      const int64_t b = bt % static_cast<uint32_t>(a.B);
      convert_tile<D>(a.K, b, h, tile, T, a.HQ, a.pieces, a.pieces + a.plane, a.kmax, wmax[0]);
      convert_tile<D>(a.V, b, h, tile, T, a.HQ, a.pieces + 2 * a.plane, a.pieces + 3 * a.plane,
                      a.vmax, wmax[1]);
      return;
    }
  }
  const int lane = lane_id();
  const int64_t idx = static_cast<int64_t>(blockIdx.x - (D > 0 ? a.nconv : 0u)) * 4 + (threadIdx.x >> 6);
  if (idx >= a.B * T) return;  // whole waves
  const int64_t b = idx % a.B;
  const int t = T - 1 - static_cast<int>(idx / a.B);
  const int64_t row = b * T + t;
  const float th = a.thr[row];
  const float* __restrict__ srow = a.scores + row * a.ld;
  const int W = (T + 63) / 64;
  uint64_t* __restrict__ mrow = a.mask + row * W;
  const int nw = min(W, ((t | 127) >> 6) + 1);
  constexpr int U = 16;  // loads in flight per lane
  for (int c = 0; c < nw; c += 64) {
    const int nu = min(64, nw - c);
    uint64_t mine = 0;
    for (int u = 0; u < nu; u += U) {
      float v[U];
#pragma unroll
      for (int e = 0; e < U; ++e)  // in the row; read once: nontemporal
        v[e] = __builtin_nontemporal_load(srow + min(64 * (c + u + e) + lane, t));
#pragma unroll
      for (int e = 0; e < U; ++e) {
        const uint64_t bits = ballot(64 * (c + u + e) + lane <= t && v[e] >= th);
        mine = (lane == u + e) ? bits : mine;
      }
    }
    if (lane < nu) mrow[c + lane] = mine;
  }
}

// ---------------------------------------------------------------------------
// The dense kernel.  Block, wave and lane layout are tile_attn.hip's: 4 waves
// of 32 queries, S^T = K.Q^T then O^T = V^T.P^T with P^T straight from the S^T
// registers, K/V tiles copied HBM -> LDS one tile ahead into double buffers,
// the mask words one tile ahead in registers.  KT keys per tile: 64, or 32 for
// fp32 rows of 128, whose four 16-bit planes of 64 keys would leave room for
// one block per CU.
// ---------------------------------------------------------------------------
template <typename Tag>
struct Pieces {  // pieces of K/V/Q, and of P
  static constexpr bool kF32 = __is_same(Tag, F32);
  static constexpr int X = kF32 ? 2 : 1;
  static constexpr int P = __is_same(Tag, BF16) ? 3 : 2;
  static constexpr bool kApart = P == 2;  // tiles summed apart, P scaled per tile
  using Half = std::conditional_t<__is_same(Tag, BF16), BF16, F16>;
};

template <typename Tag, int D>
constexpr int dense_kt() { return __is_same(Tag, F32) && D == 128 ? 32 : 64; }

//
// KS = 2: a block's keys are split over two groups of four waves, which take
// alternate key tiles of the same 128 queries and merge their sums at the
// end.  A wave's step over a tile is one serial chain (copy, products,
// softmax, products: ~5200 cycles at D = 64 fp32 whether its SIMD holds one
// wave or two), so a launch of few blocks ends with its longest block's chain;
// two groups halve it, at the same waves per SIMD (one block per CU).
template <typename Tag, int D, int KS>
__global__ __launch_bounds__(kNT * KS, 2) void dense_attn_kernel(DenseArgs a) {
  constexpr int KT = dense_kt<Tag, D>();
  using PC = Pieces<Tag>;
  using M = Mfma16x16x32<typename PC::Half>;
  using L = TileLds<D, KT>;
  constexpr bool F = PC::kF32;
  constexpr bool AP = PC::kApart;
  constexpr int NX = PC::X, NP = PC::P;
  constexpr int NJ = KT / 16;   // 16-key tiles
  constexpr int NJJ = KT / 32;  // P fragments (32 keys each)
  constexpr int NKS = D / 32;   // k-steps of the first product
  constexpr int NDT = D / 16;   // 16-dim output tiles
  // 16-key tiles whose K fragments are read at once, and 16-dim output tiles
  // whose V fragments are (twice: the next ones are on their way): 64 and 32
  // registers, at D = 128 32 and 32 (sums apart: 16).
  constexpr int KF = D == 128 ? 8 : 16;
  constexpr int KJ = NJ * NKS * NX <= KF ? NJ : KF / (NKS * NX);
  constexpr int VG = (AP && D == 128 ? 4 : 8) / (NJJ * NX);
  constexpr int GB = NX * L::BYTES;  // bytes of a group's K (or V) tile
  __shared__ __align__(16) uint8_t k0[KS * GB], k1[KS * GB], v0[KS * GB], v1[KS * GB];
  // bias of the four keys a nibble of a mask word covers (tile_attn.hip), at
  // LDS address 0
  __shared__ __align__(1024) float btab[64];
  __shared__ uint32_t vtop;  // f16: largest |V| bits the block has seen

  const int tid = threadIdx.x;
  const int kg = KS == 2 ? __builtin_amdgcn_readfirstlane(tid >> 8) : 0;  // key group
  const int wave = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);         // in its group
  const int lane = lane_id();
  const int g = lane >> 4, c16 = lane & 15;
  const int T = a.T;
  const int HQ = a.HQ;
  if (tid < 64) btab[tid] = (((tid >> 2) >> (tid & 3)) & 1) ? 0.f : -__builtin_huge_valf();
  if (tid == 0) vtop = 0u;
  const DSA_LDS uint8_t* const btabl = (const DSA_LDS uint8_t*)btab;

  // Block -> (tile, batch, head): tiles longest first, then batch, head fastest.
  const int ntile = (T + kTQ - 1) / kTQ;
  const int64_t per_tile = a.B * HQ;
  const uint32_t bid = blockIdx.x;
  const int tile = ntile - 1 - static_cast<int>(bid / per_tile);
  const int64_t bh = bid % per_tile;
  const int64_t b = bh / HQ;
  const int h = static_cast<int>(bh % HQ);
  const int t0 = tile * kTQ;
  const int tw = t0 + 32 * wave;  // first query of this wave
  const int s_hi = min(T, t0 + kTQ);
  const int nkt = (s_hi + KT - 1) / KT;
  uint32_t* const flag = a.flags + (b * ntile + tile) * 4 * HQ + h;  // a wave's: HQ apart

  const int n64 = (T + 63) / 64;
  const uint32_t* const kmx = F ? a.kmax + bh * n64 : nullptr;
  const int64_t rowE = static_cast<int64_t>(HQ) * D;  // elements per Q/K/V row
  // The pieces are laid out [B][HQ][T][D]: a tile is one contiguous run.
  const uint32_t rowbytes = F ? 2u * D : static_cast<uint32_t>(rowE) * 2u;
  const int64_t kv0 = F ? bh * T * static_cast<int64_t>(D) : b * T * rowE + static_cast<int64_t>(h) * D;
  const char* const kbase = static_cast<const char*>(a.K) + kv0 * 2;
  const char* const vbase = static_cast<const char*>(a.V) + kv0 * 2;

  // Loop-invariant copy offsets of this wave's chunks within a tile.
  constexpr int PW = L::BYTES / 1024 / (kNT / kWave);
  uint32_t koff[PW], voff[PW];
#pragma unroll
  for (int i = 0; i < PW; ++i) {
    const int P = (wave * PW + i) * 64 + lane;
    const int r = P / L::NCH, pc = P % L::NCH;
    koff[i] = static_cast<uint32_t>(r) * rowbytes + 16u * static_cast<uint32_t>(pc ^ L::swz_k(r));
    voff[i] = static_cast<uint32_t>(r) * rowbytes + 16u * static_cast<uint32_t>(pc ^ L::swz_v(r));
  }
  auto copy_k = [&](int s, DSA_LDS uint8_t* dst) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NX; ++p)
      dma_tile<PW>(tile_rsrc(kbase + p * a.K_lo, s, T, rowbytes), koff, dst + p * L::BYTES, wave);
  };
  auto copy_v = [&](int s, DSA_LDS uint8_t* dst) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NX; ++p)
      dma_tile<PW>(tile_rsrc(vbase + p * a.V_lo, s, T, rowbytes), voff, dst + p * L::BYTES, wave);
  };
  DSA_LDS uint8_t* const kl0 = (DSA_LDS uint8_t*)k0 + kg * GB;
  DSA_LDS uint8_t* const kl1 = (DSA_LDS uint8_t*)k1 + kg * GB;
  DSA_LDS uint8_t* const vl0 = (DSA_LDS uint8_t*)v0 + kg * GB;
  DSA_LDS uint8_t* const vl1 = (DSA_LDS uint8_t*)v1 + kg * GB;
  copy_k(kg * KT, kl0);
  copy_v(kg * KT, vl0);

  // Q^T fragments: qf[p][qt][ks] = piece p of Q[query tw+16qt+c16][dims 32ks+8g .. +8].
  u32x4 qf[NX][2][NKS];
  int tq[2];
  uint32_t soff[2];
  float cq[2];  // softmax scale in log2 units, over the Q row's scale
  const int W = (T + 63) / 64;
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    tq[qt] = tw + 16 * qt + c16;
    const int tl = min(tq[qt], T - 1);
    soff[qt] = static_cast<uint32_t>(tl - t0) * static_cast<uint32_t>(W) * 8u;
    cq[qt] = a.scale_log2;
    if constexpr (F) {
      const float* Qr = static_cast<const float*>(a.Q) + (b * T + tl) * rowE + static_cast<int64_t>(h) * D;
      float x[NKS][8];
      uint32_t mx = 0u;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        load_f32<8>(Qr + 32 * ks + 8 * g, x[ks]);
#pragma unroll
        for (int e = 0; e < 8; ++e) mx = max(mx, __float_as_uint(x[ks][e]) & 0x7fffffffu);
      }
      mx = max_xor32_u32(max_xor16_u32(mx));  // over the row's four lanes
      int sh;
      // a row the pieces cannot carry becomes NaN and is redone
      const bool ok = split_scale(mx, sh);
      const float sc = ok ? pow2f(sh) : __builtin_nanf("");
      cq[qt] *= ok ? pow2f(-sh) : 1.f;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          uint32_t hw, lw;
          split_pair(x[ks][2 * e] * sc, x[ks][2 * e + 1] * sc, hw, lw);
          qf[0][qt][ks][e] = hw;
          qf[NX - 1][qt][ks][e] = lw;
        }
    } else {
      const uint16_t* Qr = static_cast<const uint16_t*>(a.Q) + (b * T + tl) * rowE + static_cast<int64_t>(h) * D;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
        qf[0][qt][ks] = *reinterpret_cast<const u32x4*>(Qr + 32 * ks + 8 * g);
    }
  }

  float m[2] = {-__builtin_huge_valf(), -__builtin_huge_valf()};
  float lpart[2] = {0.f, 0.f};  // this lane's part of the normaliser, fp32
  // fp32: sum over the tiles of their largest p times their largest |V|
  [[maybe_unused]] float esum[2] = {0.f, 0.f};
  f32x4 o[NDT][2];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) o[dt][qt] = f32x4{0.f, 0.f, 0.f, 0.f};

  int kofs[NKS], vofs[NDT];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) kofs[ks] = c16 * (2 * D) + 16 * ((4 * ks + g) ^ L::swz_k(c16));
  {
    const int vr = 4 * g + (c16 >> 2);
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
      vofs[dt] = vr * (2 * D) + 16 * ((2 * dt + ((c16 & 3) >> 1)) ^ L::swz_v(vr)) + 8 * (c16 & 1);
  }

  // Mask bits of this wave's queries in tile kt: KT bits each, one buffer
  // load per query tile against a resource over the block's rows from the
  // tile's first word on.
  using word = std::conditional_t<KT == 64, uint64_t, uint32_t>;
  const char* const sblk = reinterpret_cast<const char*>(a.mask + (b * T + t0) * W);
  const uint64_t sbytes = static_cast<uint64_t>(T - t0) * static_cast<uint64_t>(W) * 8u;
  // fp32: the tile's largest |K| and |V| come with them (a load of their own
  // inside the products would make the compiler wait for the copies too).
  const __amdgpu_buffer_rsrc_t kxrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint32_t*>(kmx), 0, F ? n64 * 4 : 0, 0x00020000);
  const __amdgpu_buffer_rsrc_t vxrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint32_t*>(F ? a.vmax + bh * n64 : nullptr), 0, F ? n64 * 4 : 0, 0x00020000);
  auto load_words = [&](int kt, word (&mw)[2], uint32_t (&xb)[2]) __attribute__((always_inline)) {
    const uint64_t w0b = static_cast<uint64_t>(kt) * sizeof(word);
    const uint64_t rem = sbytes - w0b;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(sblk + w0b), 0, rem > 0xffffffffull ? -1 : static_cast<int>(static_cast<uint32_t>(rem)),
        0x00020000);
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      if constexpr (KT == 64)
        mw[qt] = __builtin_bit_cast(uint64_t, buffer_load_f32x2(rs, static_cast<int>(soff[qt]), 0, 0));
      else
        mw[qt] = __float_as_uint(buffer_load_f32(rs, static_cast<int>(soff[qt]), 0, 0));
    }
    if constexpr (F) {
      xb[0] = __float_as_uint(buffer_load_f32(kxrs, ((kt * KT) >> 6) * 4, 0, 0));
      xb[1] = __float_as_uint(buffer_load_f32(vxrs, ((kt * KT) >> 6) * 4, 0, 0));
    }
  };

  auto compute = [&](const uint32_t (&xb)[2], const word (&mwc)[2], const DSA_LDS uint8_t* kl,
                     const DSA_LDS uint8_t* vl) __attribute__((always_inline)) {
    // S^T from the bias of each key's bit (0 or -inf)
    f32x4 st[NJ][2];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      const word w = mwc[qt] >> (4 * g);
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const uint32_t hw = static_cast<uint32_t>(KT == 64 ? static_cast<uint64_t>(w) >> (32 * (j >> 1)) : w);
        const uint32_t nib = (hw >> (16 * (j & 1))) & 15u;
        st[j][qt] = *reinterpret_cast<const DSA_LDS f32x4*>(btabl + 16 * nib);
      }
    }
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int jp = 0; jp < NJ; jp += KJ) {
      u32x4 ka[NX][KJ][NKS];
#pragma unroll
      for (int p = 0; p < NX; ++p)
#pragma unroll
        for (int jj = 0; jj < KJ; ++jj)
#pragma unroll
          for (int ks = 0; ks < NKS; ++ks)
            ka[p][jj][ks] = *reinterpret_cast<const DSA_LDS u32x4*>(kl + p * L::BYTES + kofs[ks] +
                                                                   16 * (jp + jj) * (2 * D));
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (F) {  // the small terms first
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
          for (int jj = 0; jj < KJ; ++jj)
#pragma unroll
            for (int qt = 0; qt < 2; ++qt)
              st[jp + jj][qt] = M::run(ka[NX - 1][jj][ks], qf[0][qt][ks], st[jp + jj][qt]);
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
          for (int jj = 0; jj < KJ; ++jj)
#pragma unroll
            for (int qt = 0; qt < 2; ++qt)
              st[jp + jj][qt] = M::run(ka[0][jj][ks], qf[NX - 1][qt][ks], st[jp + jj][qt]);
      }
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
        for (int jj = 0; jj < KJ; ++jj)
#pragma unroll
          for (int qt = 0; qt < 2; ++qt)
            st[jp + jj][qt] = M::run(ka[0][jj][ks], qf[0][qt][ks], st[jp + jj][qt]);
    }
    __builtin_amdgcn_s_setprio(0);
    // The first V fragments arrive while the softmax runs.
    u32x4 vf[2][NX][VG][NJJ];
    auto read_v = [&](int dg, int buf) __attribute__((always_inline)) {
#pragma unroll
      for (int p = 0; p < NX; ++p)
#pragma unroll
        for (int d = 0; d < VG; ++d)
#pragma unroll
          for (int jj = 0; jj < NJJ; ++jj) {
            const DSA_LDS uint8_t* va = vl + p * L::BYTES + vofs[dg + d] + 32 * jj * (2 * D);
            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((DSA_LDS s16x4*)va);
            const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((DSA_LDS s16x4*)(va + 16 * (2 * D)));
            const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
            vf[buf][p][d][jj] = u32x4{l2.x, l2.y, h2.x, h2.y};
          }
    };
    __builtin_amdgcn_sched_barrier(0);
    read_v(0, 0);
    __builtin_amdgcn_sched_barrier(0);

    // Online softmax per query, log2 domain; a running max that moves only
    // past 2^8.  Unselected entries are -inf + logit: where a lane sees NaN
    // (a non-finite logit), the wave masks its entries exactly.
    float mxm[2];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      mxm[qt] = -__builtin_huge_valf();
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) mxm[qt] = __builtin_elementwise_maximum(mxm[qt], st[j][qt][r]);
    }
    if (ballot(__builtin_isnan(mxm[0]) | __builtin_isnan(mxm[1])) != 0) {
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
        mxm[qt] = -__builtin_huge_valf();
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const word w = mwc[qt] >> (4 * g);
            const uint32_t hw = static_cast<uint32_t>(KT == 64 ? static_cast<uint64_t>(w) >> (32 * (j >> 1)) : w);
            const uint32_t keep =
                static_cast<uint32_t>(static_cast<int32_t>(hw << (31 - (16 * (j & 1) + r))) >> 31);
            const float x = st[j][qt][r];
            st[j][qt][r] = __uint_as_float((__float_as_uint(x) & keep) | (0xff800000u & ~keep));
            mxm[qt] = fmaxf(mxm[qt], st[j][qt][r]);
          }
      }
    }
    float kx = 1.f;  // the K tile's inverse scale
    if constexpr (F) {
      int ksh;
      (void)split_scale(xb[0], ksh);
      kx = pow2f(-ksh);
    }
    [[maybe_unused]] float vx = 1.f;  // the V tile's inverse scale
    if constexpr (F) {
      int vsh;
      (void)split_scale(xb[1], vsh);
      vx = pow2f(-vsh);
    }
    u32x4 pf[NP][2][NJJ];
    bool grow = false;
    float alpha[2];
    [[maybe_unused]] float back[2];  // undoes the scales of P and V
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      const float cs = F ? cq[qt] * kx : cq[qt];
      float mx = mxm[qt];
      {
        const auto r16 =
            __builtin_amdgcn_permlane16_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mx = __builtin_elementwise_maximum(__uint_as_float(r16[0]), __uint_as_float(r16[1]));
        const auto r32 =
            __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mx = __builtin_elementwise_maximum(__uint_as_float(r32[0]), __uint_as_float(r32[1]));
      }
      const float m_blk = mx * cs;
      const bool up = m_blk > m[qt] + 8.f;
      const float m_new = up ? m_blk : m[qt];
      alpha[qt] = up ? exp2f(m[qt] - m_new) : 1.f;  // m = -inf: alpha = 0 on an empty O
      grow |= up && (m[qt] != -__builtin_huge_valf());
      m[qt] = m_new;
      const float m_use = (m_new == -__builtin_huge_valf()) ? 0.f : m_new;
      float p[NJ][4];
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          p[j][r] = __builtin_amdgcn_exp2f(fmaf(st[j][qt][r], cs, -m_use));
      float ls = 0.f;
#pragma unroll
      for (int j = 0; j < NJ; ++j) ls += (p[j][0] + p[j][1]) + (p[j][2] + p[j][3]);
      lpart[qt] = fmaf(lpart[qt], alpha[qt], ls);
      if constexpr (AP) {
        // pm: the largest p, by the operations that made it.  Tiles 2^-107 below
        // the running max share a scale (their products leave fp32's range).
        const float pm = __builtin_amdgcn_exp2f(fmaf(mx, cs, -m_use));
        const uint32_t eb = max(__float_as_uint(pm) >> 23, 20u);
        const float pc = __uint_as_float((268u - eb) << 23);
        back[qt] = __uint_as_float((eb - 14u) << 23) * vx;
        if constexpr (F) esum[qt] = fmaf(esum[qt], alpha[qt], pm * __uint_as_float(xb[1]));
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) p[j][r] *= pc;
      }
#pragma unroll
      for (int jj = 0; jj < NJJ; ++jj)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = p[2 * jj + (e >> 1)][2 * (e & 1)], y = p[2 * jj + (e >> 1)][2 * (e & 1) + 1];
          if constexpr (NP == 2) {
            uint32_t hw, lw;
            split_pair(x, y, hw, lw);
            pf[0][qt][jj][e] = hw;
            pf[1][qt][jj][e] = lw;
          } else {
            // bf16 pieces by truncation: 8 + 8 + 8 bits, exact
            const uint32_t xb = __float_as_uint(x), yb = __float_as_uint(y);
            const float x1 = x - __uint_as_float(xb & 0xffff0000u);
            const float y1 = y - __uint_as_float(yb & 0xffff0000u);
            const uint32_t x1b = __float_as_uint(x1), y1b = __float_as_uint(y1);
            const float x2 = x1 - __uint_as_float(x1b & 0xffff0000u);
            const float y2 = y1 - __uint_as_float(y1b & 0xffff0000u);
            pf[0][qt][jj][e] = __builtin_amdgcn_perm(yb, xb, 0x07060302u);
            pf[1][qt][jj][e] = __builtin_amdgcn_perm(y1b, x1b, 0x07060302u);
            pf[NP - 1][qt][jj][e] =
                __builtin_amdgcn_perm(__float_as_uint(y2), __float_as_uint(x2), 0x07060302u);
          }
        }
    }
    if (ballot(grow) != 0) {
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int qt = 0; qt < 2; ++qt)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[dt][qt][r] *= alpha[qt];
    }

    // O^T += V^T . P^T, the small terms first.  The next group's fragments are
    // on their way while a group's products run.
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int dg = 0; dg < NDT; dg += VG) {
      if (dg + VG < NDT) {
        read_v(dg + VG, (dg / VG + 1) & 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      const u32x4(&vg)[NX][VG][NJJ] = vf[(dg / VG) & 1];
      if constexpr (AP) {
        // Summed apart also means one rounding at O's magnitude per tile
        // instead of one per MFMA.
        f32x4 t[VG][2];
#pragma unroll
        for (int d = 0; d < VG; ++d)
#pragma unroll
          for (int qt = 0; qt < 2; ++qt) t[d][qt] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto sum = [&](int pv, int pp) __attribute__((always_inline)) {
#pragma unroll
          for (int jj = 0; jj < NJJ; ++jj)
#pragma unroll
            for (int d = 0; d < VG; ++d)
#pragma unroll
              for (int qt = 0; qt < 2; ++qt)
                t[d][qt] = M::run(vg[pv][d][jj], pf[pp][qt][jj], t[d][qt]);
        };
        if constexpr (F) sum(NX - 1, 0);
        sum(0, NP - 1);
        sum(0, 0);
#pragma unroll
        for (int d = 0; d < VG; ++d)
#pragma unroll
          for (int qt = 0; qt < 2; ++qt)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              o[dg + d][qt][r] = fmaf(t[d][qt][r], back[qt], o[dg + d][qt][r]);
      } else {
#pragma unroll
        for (int p = NP - 1; p >= 0; --p)
#pragma unroll
          for (int jj = 0; jj < NJJ; ++jj)
#pragma unroll
            for (int d = 0; d < VG; ++d)
#pragma unroll
              for (int qt = 0; qt < 2; ++qt)
                o[dg + d][qt] = M::run(vg[0][d][jj], pf[p][qt][jj], o[dg + d][qt]);
      }
    }
    __builtin_amdgcn_s_setprio(0);
  };

  // f16: the largest and lowest V of this thread's share of the tiles seen, read
  // behind a tile's products (before them it holds up the K fragments: 9 us of
  // the 117 at B = 2, T = 3001, HQ = 16, D = 128 against 2.5).
  typedef _Float16 h16x2 __attribute__((ext_vector_type(2)));
  [[maybe_unused]] h16x2 vhi = {0, 0}, vlo = {0, 0};
  [[maybe_unused]] auto see_v = [&](const DSA_LDS uint8_t* vl) __attribute__((always_inline)) {
    constexpr int N = L::BYTES / 16 / kNT;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const u32x4 x = *reinterpret_cast<const DSA_LDS u32x4*>(vl + (i * kNT + (tid & (kNT - 1))) * 16);
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        const h16x2 y = __builtin_bit_cast(h16x2, x[e]), z = __builtin_bit_cast(h16x2, x[e + 1]);
        vhi = __builtin_elementwise_maximum(__builtin_elementwise_maximum(vhi, y), z);
        vlo = __builtin_elementwise_minimum(__builtin_elementwise_minimum(vlo, y), z);
      }
    }
  };

  // Per tile: the next tile's copy and mask words go out first (in that
  // order: the barrier waits for the copy only), then the products.
  constexpr int NSL = F ? 4 : 2;  // loads behind a tile's copy
  word mw[2];
  uint32_t xb[2] = {0u, 0u};
  auto step = [&](int kt, DSA_LDS uint8_t* kc, DSA_LDS uint8_t* vc, DSA_LDS uint8_t* kn,
                  DSA_LDS uint8_t* vn) __attribute__((always_inline)) {
    const word mwc[2] = {mw[0], mw[1]};
    const uint32_t xc[2] = {xb[0], xb[1]};
    const bool act = kt < nkt && ballot((mw[0] | mw[1]) != 0) != 0;
    const bool more = kt + KS < nkt;
    if (more) {
      copy_k((kt + KS) * KT, kn);
      copy_v((kt + KS) * KT, vn);
      __builtin_amdgcn_sched_barrier(0);
      load_words(kt + KS, mw, xb);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (act) compute(xc, mwc, kc, vc);
    if constexpr (AP && !F) {
      if (kt < nkt) see_v(vc);
    }
    if (more) wait_dma_keep<NSL>();
    else wait_dma_keep<0>();
    block_sync_lds();
  };
  // Left to redo_kernel: tiles with a key whose K or V the pieces cannot carry.
  if constexpr (F) {
    uint32_t bad = 0u;
    for (int i = lane; i < (s_hi + 63) / 64; i += kWave)
      bad |= (kmx[i] == kBadTile || a.vmax[bh * n64 + i] == kBadTile) ? 1u : 0u;
    if (__builtin_amdgcn_readfirstlane(ballot(bad != 0u) != 0u)) {  // the same in every wave
      wait_dma_keep<0>();  // the first tile's copy writes this block's LDS
      if (tid < 4) flag[tid * HQ] = 0xffffffffu;
      return;
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  load_words(kg, mw, xb);
  __builtin_amdgcn_sched_barrier(0);
  wait_dma_keep<NSL>();
  block_sync_lds();
  const int nstep = (nkt + KS - 1) / KS;
  int i = 0;
  for (; i + 1 < nstep; i += 2) {
    step(i * KS + kg, kl0, vl0, kl1, vl1);
    step((i + 1) * KS + kg, kl1, vl1, kl0, vl0);
  }
  if (i < nstep) step(i * KS + kg, kl0, vl0, kl1, vl1);

  // The second group hands its sums to the first through the tile buffers:
  // O tile dt of query tile qt in buffer qt + 2 (dt % 2), [slot][lane] floats,
  // the running max behind the even tiles, the normaliser and esum behind the odd.
  if constexpr (KS == 2) {
    constexpr int NS = NDT * 2 + 2;  // slots per wave and buffer
    static_assert(NS * 4 * 256 <= KS * GB, "the partial sums fit the tile buffers");
    DSA_LDS float* const buf[4] = {(DSA_LDS float*)k0 + wave * NS * 64 + lane,
                                   (DSA_LDS float*)k1 + wave * NS * 64 + lane,
                                   (DSA_LDS float*)v0 + wave * NS * 64 + lane,
                                   (DSA_LDS float*)v1 + wave * NS * 64 + lane};
    if (kg == 1) {
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
          for (int r = 0; r < 4; ++r) buf[qt + 2 * (dt & 1)][((dt >> 1) * 4 + r) * 64] = o[dt][qt][r];
        buf[qt][(NS - 2) * 64] = m[qt];
        buf[qt + 2][(NS - 2) * 64] = lpart[qt];
        if constexpr (F) buf[qt + 2][(NS - 1) * 64] = esum[qt];
      }
    }
    block_sync_lds();
    if (kg == 0) {
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
        const float m1 = buf[qt][(NS - 2) * 64], l1 = buf[qt + 2][(NS - 2) * 64];
        const float mn = fmaxf(m[qt], m1);
        const float mu = mn == -__builtin_huge_valf() ? 0.f : mn;
        const float a0 = exp2f(m[qt] - mu), a1 = exp2f(m1 - mu);
        lpart[qt] = fmaf(lpart[qt], a0, l1 * a1);
        if constexpr (F) esum[qt] = fmaf(esum[qt], a0, buf[qt + 2][(NS - 1) * 64] * a1);
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            o[dt][qt][r] = fmaf(o[dt][qt][r], a0, buf[qt + 2 * (dt & 1)][((dt >> 1) * 4 + r) * 64] * a1);
      }
    }
  }

  // O = O^T / l, lane l: query tq[qt], dims 16dt + 4g .. +3.
  // f16: the largest |V| of all tiles, whose sums of p are at least their largest
  [[maybe_unused]] float vcap = 0.f;
  if constexpr (AP && !F) {
    const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_elementwise_maximum(vhi, -vlo));
    const uint32_t v = wave_extreme_u32<true>(max(w & 0xffffu, w >> 16));
    if (lane == 0) atomicMax(&vtop, v);
    block_sync_lds();
    vcap = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(vtop)));
  }
  uint32_t redo = 0u;  // the wave's 32 queries
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    bool bad = false;
    const float l = sum_xor32(sum_xor16(lpart[qt]));
    const float inv = 1.f / l;  // l == 0 only if nothing passed: NaN, as the reference
    if (kg == 0 && tq[qt] < T) {
      float* orow = a.out + ((b * T + tq[qt]) * HQ + h) * static_cast<int64_t>(D);
      uint32_t mxb = 0u;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) {
        float4 v;
        v.x = o[dt][qt][0] * inv;
        v.y = o[dt][qt][1] * inv;
        v.z = o[dt][qt][2] * inv;
        v.w = o[dt][qt][3] * inv;
        mxb = max(max(mxb, __float_as_uint(v.x) & 0x7fffffffu), __float_as_uint(v.y) & 0x7fffffffu);
        mxb = max(max(mxb, __float_as_uint(v.z) & 0x7fffffffu), __float_as_uint(v.w) & 0x7fffffffu);
        *reinterpret_cast<float4*>(orow + 16 * dt + 4 * g) = v;
      }
      bad |= mxb >= 0x7f800000u && l != 0.f;
      if constexpr (AP) {
        mxb = max_xor32_u32(max_xor16_u32(mxb));  // over the query's four lanes
        bad |= __uint_as_float(mxb) < (F ? esum[qt] * inv : vcap) * 0x1p-13f;  // false for NaN
      }
    }
    uint64_t any = ballot(bad);  // lanes c16, c16 + 16, .. hold query c16
    any |= any >> 32;
    any |= any >> 16;
    redo |= static_cast<uint32_t>(any & 0xffffu) << (16 * qt);
  }
  if (kg == 0 && lane == 0) flag[wave * HQ] = redo;
}

// ---------------------------------------------------------------------------
// The gathers of attn_tile.h on the bitmask, for the rows left to them: a wave
// per query (and head chunk), as sparse_attn.hip has it, that leaves at once
// where, as nearly always, none of the row's heads is flagged.  With every row
// flagged it is the gathers' time on top of the dense kernel's (B = 4, T = 4096,
// HQ = 8, D = 64, k = 256 fp32: 0.99 ms in all, the gathers 0.75; f16 B = 2, T =
// 3001, HQ = 16, D = 128, k = 300: 0.99 and 0.86; eight waves per 128 queries and
// whole tiles flagged took 2.07 and 4.88 ms, and 0.5 and 1.08 where one row was).
// With none flagged the launch takes 4.5 us, 1 to 2 more than with those fewer
// blocks.  Blocks of eight waves: up to 1 us more; waves that stay for several
// rows: 2 more (their index arithmetic), and no faster with every row flagged.
// ---------------------------------------------------------------------------
struct RedoArgs {
  const uint64_t* mask;
  const uint32_t* flags;
  const void* Q;
  const void* K;
  const void* V;
  int64_t B;
  int T;
  int HQ, D;
  float scale_log2;
  float* out;
  int HQc;     // heads per chunk
  int nchunk;  // HQ / HQc
};

constexpr int kRedoQ = 4;

template <typename Tag, int E>
__global__ __launch_bounds__(64 * kRedoQ) void redo_kernel(RedoArgs a) {
  using raw = typename Tag::raw;
  constexpr bool PAIR = __is_same(Tag, F32) && E == 2;
  __shared__ __align__(16) int lists[kRedoQ][kListCap];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = lane_id();
  const int T = a.T;
  const int ntile = (T + kTQ - 1) / kTQ;
  // blocks in chunk, batch, longest-rows-first order (32-bit: the grid is)
  uint32_t i = blockIdx.x, chunk = 0u, bb = 0u;
  if (a.nchunk > 1) {
    chunk = i % static_cast<uint32_t>(a.nchunk);
    i /= static_cast<uint32_t>(a.nchunk);
  }
  if (a.B > 1) {
    bb = i % static_cast<uint32_t>(a.B);
    i /= static_cast<uint32_t>(a.B);
  }
  const int64_t b = bb;
  const int t = ((T + kRedoQ - 1) / kRedoQ - 1 - static_cast<int>(i)) * kRedoQ + wave;
  if (t >= T) return;
  const uint32_t* fl = a.flags + ((b * ntile + t / kTQ) * 4 + (t % kTQ) / 32) * a.HQ;
  uint32_t rows = 0u;
  for (int h = lane; h < a.HQ; h += kWave) rows |= fl[h];
  if (ballot((rows >> (t % 32)) & 1u) == 0u) return;
  const int64_t E64 = static_cast<int64_t>(a.HQ) * a.D;
  const int64_t c0 = static_cast<int64_t>(chunk) * a.HQc * a.D;  // chunk's first element
  const raw* Q = static_cast<const raw*>(a.Q) + b * T * E64 + c0;
  const raw* K = static_cast<const raw*>(a.K) + b * T * E64 + c0;
  const raw* V = static_cast<const raw*>(a.V) + b * T * E64 + c0;
  const int W = (T + 63) / 64;
  int* list = lists[wave];
  const int64_t qrow = b * T + t;
  const uint8_t* mrow = reinterpret_cast<const uint8_t*>(a.mask + qrow * W);
  // keys s0 .. s0 + 511 of the row: lane l's byte holds keys s0 + 8l .. + 7
  // (bits of keys past t are 0 in the words that hold them)
  auto segment = [&](int s0) {
    const int sb = s0 + 8 * lane;
    uint32_t bits = sb <= t ? mrow[sb >> 3] : 0u;
    const int cnt = __popc(bits);
    const int incl = wave_inclusive_sum(cnt);
    int p = incl - cnt;
    while (bits != 0u) {
      list[p++] = sb + __ffs(static_cast<int>(bits)) - 1;
      bits &= bits - 1u;
    }
    return wave_read_lane(incl, kWave - 1);
  };
  if constexpr (PAIR)
    attend_query_pair_on(Q, K, V, t, a.D, a.scale_log2, segment, list, a.out + qrow * E64);
  else
    attend_query_on<Tag, E, E>(Q, K, V, t, a.HQc, a.D, a.D, a.scale_log2, segment, list,
                               a.out + qrow * E64 + c0, nullptr, static_cast<int>(E64),
                               static_cast<int>(E64));
}

// Two key groups per block while every block has a CU to itself or shares it
// with one other (they end with their longest block: B = 4, T = 2048, HQ = 8,
// D = 64 fp32, 512 blocks, 98 us against 108); past that two independent
// blocks per CU overlap one's products with the other's softmax, which a
// block's own groups, tied by its barriers, do not (B = 4, T = 4096, 1024
// blocks, 252 us against 294; f16 D = 128, 768 blocks, 142 against 159).
template <typename Tag, int D>
hipError_t launch_dense(const DenseArgs& a, hipStream_t stream) {
  const int64_t nblk = a.B * a.HQ * ((a.T + kTQ - 1) / kTQ);
  const dim3 grid(static_cast<unsigned>(nblk));
  if (nblk <= 2 * static_cast<int64_t>(device_cus()))
    hipLaunchKernelGGL((dense_attn_kernel<Tag, D, 2>), grid, dim3(2 * kNT), 0, stream, a);
  else
    hipLaunchKernelGGL((dense_attn_kernel<Tag, D, 1>), grid, dim3(kNT), 0, stream, a);
  return hipGetLastError();
}

template <typename Tag>
hipError_t dispatch_dense(const DenseArgs& a, int D, hipStream_t stream) {
  if (D == 64) return launch_dense<Tag, 64>(a, stream);
  if (D == 128) return launch_dense<Tag, 128>(a, stream);
  return hipErrorInvalidValue;
}

template <typename Tag>
hipError_t dispatch_redo(const RedoArgs& a, int E, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(a.B * ((a.T + kRedoQ - 1) / kRedoQ) * a.nchunk));
#define DSA_REDO_CASE(e) \
  case e: hipLaunchKernelGGL((redo_kernel<Tag, e>), grid, dim3(64 * kRedoQ), 0, stream, a); break;
  switch (E) {
    DSA_REDO_CASE(1)
    DSA_REDO_CASE(2)
    DSA_REDO_CASE(4)
    DSA_REDO_CASE(8)
    DSA_REDO_CASE(16)
    case 32:
      if constexpr (!__is_same(Tag, F32)) {
        hipLaunchKernelGGL((redo_kernel<Tag, 32>), grid, dim3(64 * kRedoQ), 0, stream, a);
        break;
      }
      return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
#undef DSA_REDO_CASE
  return hipGetLastError();
}

template <int D>
hipError_t launch_prepare(PrepareArgs a, hipStream_t stream) {
  a.nconv = D > 0 ? static_cast<uint32_t>(a.B * ((a.T + 63) / 64) * a.HQ) : 0u;
  const int64_t nblk = a.nconv + (a.scores != nullptr ? (a.B * a.T + 3) / 4 : 0);
  if (nblk == 0) return hipSuccess;
  hipLaunchKernelGGL((prepare_kernel<D>), dim3(static_cast<unsigned>(nblk)), dim3(256), 0, stream, a);
  return hipGetLastError();
}

struct Layout {
  int64_t flags, kmax, vmax, pieces, plane, total;  // byte offsets; plane in elements
};
Layout dense_layout(int dtype, int64_t B, int64_t T, int HQ, int D) {
  auto up = [](int64_t n) { return (n + 255) / 256 * 256; };
  const int64_t n64 = (T + 63) / 64;
  Layout l{};
  l.flags = up(B * T * n64 * 8);  // behind the bitmask
  l.kmax = l.flags + up(B * ((T + kTQ - 1) / kTQ) * 4 * HQ * 4);
  l.total = l.kmax;
  if (dtype == 0) {
    l.vmax = l.kmax + up(B * HQ * n64 * 4);
    l.pieces = l.vmax + up(B * HQ * n64 * 4);
    l.plane = up(B * T * HQ * static_cast<int64_t>(D) * 2) / 2;
    l.total = l.pieces + 4 * l.plane * 2;
  }
  return l;
}

}  // namespace

bool dense_attn_supported(int dtype, int64_t T, int HQ, int DQ, int DV) {
  if (dtype < 0 || dtype > 2 || DQ != DV || (DQ != 64 && DQ != 128)) return false;
  if (T < 1 || T > (int64_t{1} << 20)) return false;  // 128 mask rows: 32-bit byte offsets
  return sparse_attn_supported(dtype, HQ, DQ, DV);
}

int64_t dense_attn_workspace(int dtype, int64_t B, int64_t T, int HQ, int D) {
  return dense_layout(dtype, B, T, HQ, D).total;
}

hipError_t launch_dense_attn(const float* scores, int64_t ld, const float* thr, const void* Q,
                             const void* K, const void* V, int dtype, int64_t B, int64_t T, int HQ,
                             int D, float scale, float* out, void* ws, hipStream_t stream) {
  if (B == 0 || T == 0) return hipSuccess;
  const Layout l = dense_layout(dtype, B, T, HQ, D);
  char* base = static_cast<char*>(ws);
  uint64_t* mask = reinterpret_cast<uint64_t*>(base);
  uint32_t* flags = reinterpret_cast<uint32_t*>(base + l.flags);
  uint32_t* kmax = dtype == 0 ? reinterpret_cast<uint32_t*>(base + l.kmax) : nullptr;
  uint32_t* vmax = dtype == 0 ? reinterpret_cast<uint32_t*>(base + l.vmax) : nullptr;
  uint16_t* pieces = dtype == 0 ? reinterpret_cast<uint16_t*>(base + l.pieces) : nullptr;
  const PrepareArgs pa{scores, ld, thr, B, static_cast<int>(T), HQ, static_cast<const float*>(K),
                       static_cast<const float*>(V), pieces, l.plane, kmax, vmax, 0u, mask};
  hipError_t e;
  if (dtype != 0) e = launch_prepare<0>(pa, stream);
  else if (D == 64) e = launch_prepare<64>(pa, stream);
  else e = launch_prepare<128>(pa, stream);
  if (e != hipSuccess) return e;
  const float scale_log2 = scale * 1.4426950408889634f;
  const DenseArgs a{Q,
                    dtype == 0 ? static_cast<const void*>(pieces) : K,
                    dtype == 0 ? static_cast<const void*>(pieces + 2 * l.plane) : V,
                    l.plane * 2,
                    l.plane * 2,
                    B,
                    static_cast<int>(T),
                    HQ,
                    scale_log2,
                    out,
                    mask,
                    flags,
                    kmax,
                    vmax};
  if (dtype == 0) e = dispatch_dense<F32>(a, D, stream);
  else if (dtype == 1) e = dispatch_dense<BF16>(a, D, stream);
  else e = dispatch_dense<F16>(a, D, stream);
  if (e != hipSuccess) return e;
  int nchunk = 1;  // as sparse_attn.hip splits wide rows
  while (static_cast<int64_t>(HQ) * D / nchunk > static_cast<int64_t>(kWave) * (dtype == 0 ? 16 : 32))
    nchunk *= 2;
  const RedoArgs ra{mask, flags, Q, K, V, B, static_cast<int>(T), HQ, D, scale_log2, out,
                      HQ / nchunk, nchunk};
  const int E = HQ / nchunk * D / kWave;
  if (dtype == 0) return dispatch_redo<F32>(ra, E, stream);
  if (dtype == 1) return dispatch_redo<BF16>(ra, E, stream);
  return dispatch_redo<F16>(ra, E, stream);
}

// Which kernel suits a shape whose queries select about top_k keys (0:
// unknown).  Estimated times in us on this chip's measured rates:
//   gathers: cycles of a CU per gathered (query, key) pair, all heads, by bytes
//     of a K row -- 24 at 512 (two keys per load), 50 at 1 KiB, 86 at 2 KiB,
//     265 at 4 KiB (groups of two keys) -- over the CUs, plus the score rows
//     at ~3 TB/s;
//   dense: 0.4 cycles per (query, key, head) over the CUs, plus half the
//     longest block's chain where two key groups share a block (1.3 us per 64
//     keys), the scores and K / V through prepare_kernel at 5.5 TB/s, and 15
//     for the launches' fixed parts.
// (B = 4, T = 2048, HQ = 8, D = 64 fp32: k = 128 95 us dense against 168
// gathered, k = 64 93 / 98, k = 32 93 / 59; bf16 k = 128 69 / 93, k = 32 66 /
// 32.)  Where top_k is unknown the dense kernel takes only the shapes the
// staged kernel would have had, which streams every key whatever is selected
// (B = 4, T = 4096, HQ = 8, D = 64: 360-450 us at any k against 253), with
// enough blocks that it wins at any k (B = 1, T = 4096: 123 us against 94 at
// k = 16).
AttnPick pick_sparse_attn(int dtype, int64_t B, int64_t T, int HQ, int DQ, int DV, int64_t top_k) {
  if (!dense_attn_supported(dtype, T, HQ, DQ, DV) || sparse_attn_uses_tiles(dtype, T, HQ, DQ, DV))
    return AttnPick::kThreshold;
  const double cus = device_cus();
  if (cus <= 0) return AttnPick::kThreshold;
  const bool staged = staged_attn_auto(dtype, B, T, HQ, DQ, DV, true) && staged_attn_fits(T, T);
  const double blocks = static_cast<double>(B) * HQ * ((T + kTQ - 1) / kTQ);
  if (top_k <= 0) return staged && blocks >= 4 * cus ? AttnPick::kDense : AttnPick::kThreshold;
  const double es = dtype == 0 ? 4 : 2, row = HQ * DQ * es;
  const double pairs = static_cast<double>(B) * T * (T + 1) / 2, k = static_cast<double>(std::min(top_k, T));
  const double sel = static_cast<double>(B) * (k * T - k * k / 2);
  const double per = row <= 512 ? 24 : row <= 1024 ? 50 : row <= 2048 ? 86 : 265 * row / 4096;
  const double mhz = 2100 * cus;
  const double gather = sel * per / mhz + pairs * 4 / 3e6 + 5;
  const double chain = 1.3 * (static_cast<double>(T) / 64);
  const double bytes = pairs * 4 + (dtype == 0 ? 4.0 * B * T * row : 0.0);
  const double dense = std::max(pairs * HQ * (DQ == 128 ? 0.8 : 0.4) / mhz, chain / 2) +
                       (blocks <= 2 * cus ? chain / 2 : 0.0) + bytes / 5.5e6 + 15;
  if (dense < 0.9 * gather) return AttnPick::kDense;
  if (!staged) return AttnPick::kThreshold;
  return gather < dense ? AttnPick::kGather : AttnPick::kDense;
}

}  // namespace dsa
