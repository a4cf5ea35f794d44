// forward.cpp -- the split forward as one host call: indexer -> per-row select
// -> sparse attention on one stream, over one workspace (host code only; the
// kernels are the stages' own).
//
// Replaces dsa_attention_split_triton (reference dsa_attention.py:327-345).
// Called stage by stage from Python the three stages cost ~40 us of host time,
// more than their kernels take on short sequences; this call costs what one
// stage does.
#include <algorithm>

#include "dsa_launch.h"

namespace dsa {
namespace {

struct SplitLayout {
  int64_t thr, att, total;  // byte offsets: scores, then thresholds, then the attention's workspace
};

int64_t up256(int64_t n) { return (n + 255) / 256 * 256; }

// Workspace of the attention stage: the tile kernel's bitmask, the dense
// kernel's workspace, or the staged kernel's.
int64_t attention_bytes(int dtype, int64_t B, int64_t T, int HQ, int DQ, int DV, int64_t k) {
  if (sparse_attn_uses_tiles(dtype, T, HQ, DQ, DV)) return B * T * ((T + 63) / 64) * 8;
  switch (pick_sparse_attn(dtype, B, T, HQ, DQ, DV, k)) {
    case AttnPick::kDense: return dense_attn_workspace(dtype, B, T, HQ, DQ);
    case AttnPick::kGather: return 0;
    default: return sparse_attn_workspace_bytes(false, dtype, B, T, HQ, DQ, DV, T);
  }
}

SplitLayout split_layout(int dtype, int64_t B, int64_t T, int HQ, int DQ, int DV, int64_t k) {
  SplitLayout l;
  l.thr = up256(B * T * T * 4);
  l.att = l.thr + up256(B * T * 4);
  l.total = l.att + up256(std::max<int64_t>(0, attention_bytes(dtype, B, T, HQ, DQ, DV, k)));
  return l;
}

}  // namespace

int64_t split_workspace(int dtype, int64_t B, int64_t T, int HQ, int DQ, int DV, int64_t k) {
  return split_layout(dtype, B, T, HQ, DQ, DV, k).total;
}

// Whether the split forward is expected to beat the fused kernel (where both
// exist).  Measured, us fused / split:
//   - attention that the dense kernel takes: T = 731, B = 12, HI = 16, DI = 64,
//     HQ = 4, D = 128 fp32 242 / 111; below T = 512 its launches do not pay
//     (T = 256, B = 32 bf16 41 / 43);
//   - DI = 128, whose fused instance holds one wave per SIMD: T = 512, B = 4,
//     HI = 64 bf16 69 / 37, T = 224, B = 27, HI = 4 39 / 33; short ones are
//     launch-bound (T = 106, B = 22 20 / 24);
//   - T >= 900, where a fused block's score rows leave one block per CU, unless
//     the call is small: T = 2048, B = 4, HI = 8, DI = 64, k = 16 bf16 111 / 58,
//     T = 1900, B = 22, HI = 16, DI = 32 fp32 1040 / 594, T = 1024, B = 2, HI =
//     8, DI = 64 fp32 68 / 55, but T = 2048, B = 2, HI = 4, DI = 32 62 / 69;
//   - everything else fused: T = 512, B = 16, HI = 4, DI = 32 fp32 25 / 35, T =
//     697, B = 19, HI = 16, DI = 32 bf16 100 / 118.
// Below forward_split_min_T never; a caller may ask that first.
int64_t forward_split_min_T(int DI) { return DI >= 128 ? 200 : 512; }

bool forward_uses_split(int dtype, int64_t B, int64_t T, int HI, int DI, int HQ, int DQ, int DV,
                        int64_t k) {
  if (T < forward_split_min_T(DI)) return false;
  const double work = static_cast<double>(B) * T * T * HI * DI;
  if (T >= 512 && pick_sparse_attn(dtype, B, T, HQ, DQ, DV, k) == AttnPick::kDense) return true;
  if (DI >= 128 && work >= 6e8) return true;
  return T >= 900 && work >= (HI * DI >= 512 ? 1e9 : 2e9);
}

hipError_t launch_split(const void* qi, const void* ki, const void* wi, int idx_dtype, const void* Q,
                        const void* K, const void* V, int dtype, int64_t B, int64_t T, int HI, int DI,
                        int HQ, int DQ, int DV, int k, float scale, float* out, void* ws,
                        hipStream_t stream) {
  const SplitLayout l = split_layout(dtype, B, T, HQ, DQ, DV, k);
  char* base = static_cast<char*>(ws);
  float* scores = reinterpret_cast<float*>(base);
  float* thr = reinterpret_cast<float*>(base + l.thr);
  void* att = base + l.att;
  const int64_t att_bytes = l.total - l.att;
  hipError_t e = launch_indexer(qi, ki, wi, idx_dtype, B, T, HI, DI, static_cast<int64_t>(HI) * DI, DI,
                                HI, scores, T, 0, stream);
  if (e != hipSuccess) return e;
  if (sparse_attn_uses_tiles(dtype, T, HQ, DQ, DV)) {
    // the select writes the selection bitmask the tile kernel reads
    uint64_t* mask = static_cast<uint64_t*>(att);
    const int64_t W = (T + 63) / 64;
    e = launch_topk_mask(scores, B, T, T, k, thr, mask, W, stream);
    if (e != hipSuccess) return e;
    return launch_tile_attn_mask(mask, W, Q, K, V, dtype, B, T, HQ, DQ, scale, out, stream);
  }
  const AttnPick pick = pick_sparse_attn(dtype, B, T, HQ, DQ, DV, k);
  if (pick == AttnPick::kDense && T <= 4096) {
    // the select holds the row in registers and writes the bitmask from there
    // (the dense kernel's workspace begins with it).  Longer rows leave it to
    // prepare_kernel, though the bracket select's bitmask costs less than that
    // second read of the scores there too (B = 2, k = 256: T = 5000 8 us against
    // 19, T = 8192 17 against 45).
    e = launch_topk_mask(scores, B, T, T, k, thr, static_cast<uint64_t*>(att), (T + 63) / 64, stream);
    if (e != hipSuccess) return e;
    return launch_dense_attn(nullptr, T, thr, Q, K, V, dtype, B, T, HQ, DQ, scale, out, att, stream);
  }
  e = launch_topk(scores, B * T, T, T, k, T, thr, nullptr, stream);
  if (e != hipSuccess) return e;
  switch (pick) {
    case AttnPick::kDense:
      return launch_dense_attn(scores, T, thr, Q, K, V, dtype, B, T, HQ, DQ, scale, out, att, stream);
    case AttnPick::kGather:
      return launch_sparse_attn_gather(scores, T, thr, Q, K, V, dtype, B, T, HQ, DQ, DV, scale, out,
                                       stream);
    default:
      return launch_sparse_attn(scores, T, thr, Q, K, V, dtype, B, T, HQ, DQ, DV, scale, out,
                                att_bytes > 0 ? att : nullptr, att_bytes, stream);
  }
}

}  // namespace dsa
