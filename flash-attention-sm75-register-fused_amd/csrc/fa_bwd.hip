// Fused attention backward for gfx950: grid plan and instance selection.
// The kernels are in fa_bwd_kernel.h, instantiated per head dimension and
// mask mode in fa_bwd_d{64,128}{,_mask}.hip.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "fa_internal.h"

namespace fa {

// The split gives every key block ceil(S / T) pieces of its S steps, T being
// the longest piece allowed.  One dK/dV workgroup fills a CU, so with one
// workgroup per key block a launch of few (batch, KV head) units or few keys
// leaves CUs idle, and its time is its longest block's (causal: block 0's)
// chain of steps: B=4 Hq=14 Hkv=2 N=2048 d=64 causal is 128 blocks of up to 224
// steps where 60 per CU would do.  T minimises an estimate of the launch in
// steps: with at most one piece per CU its longest piece, else the mean load
// of a CU and half a piece for the uneven end (equal pieces: whole rounds),
// and kPieceSteps per piece (its prologue and epilogue, one idle period, its
// partials' trip to memory) and kMergeSteps for the merge launch.  Fitted to
// 16 shapes timed at up to 11 values of T each on MI355X; the choice is
// within 7% of the fastest T on all of them (backward call, T = none ->
// chosen, bf16): B=4 Hq=14 Hkv=2 N=2048 d64 causal 254 -> 147 us, B=1 Hq=14
// Hkv=2 N=4096 d64 causal 443 -> 152 us, N=1024 118 -> 42 us, B=1 Hq=32 Hkv=8
// d128 causal N=1024 117 -> 65 us, N=4096 545 -> 480 us, B=1 Hq=64 Hkv=8
// N=2048 d128 full 500 -> 418 us.  Where the unsplit launch already fills the
// GPU a split loses (B=1 Hq=32 Hkv=8 N=8192 d128 causal 1605 -> 1658-1790 us,
// B=4 H=8 N=2048 d64 causal 85 -> 95-112 us, B=4 H=12 N=1024 d64 full 69 -> 80
// us): it must be estimated kMinGain faster to be taken, and to save kMinSaved
// steps (about a microsecond each), since the merge launch costs the host 3 us
// (B=1 H=12 N=1114 d64 full, 4 steps saved: 40.3 us unsplit, 42.0 split).
constexpr int kPieceSteps = 8;
constexpr int kMergeSteps = 5;
constexpr int kMinPiece = 8;  // shortest T considered (T = 4 on the N=1024 shape below: 45 us)
constexpr double kMinGain = 1.08;
constexpr int kMinSaved = 8;
constexpr int kMaxPiecesPerCu = 4;  // bounds the partials: 134 MB at head_dim 128 on 256 CUs

int64_t plan_bwd_split(const BwdArgs& a, int batch, int head_dim, bool causal, BwdSplit& s) {
  s.pieces = 0;
  s.merged = 0;
  const int64_t key_blocks = ((int64_t)a.nk + kBwdBlockKeys - 1) / kBwdBlockKeys;
  if (key_blocks > kBwdMaxSplitBlocks) return 0;
  const int nkb = (int)key_blocks;
  const int64_t units = (int64_t)batch * (a.hq / a.group);
  const int cus = resident_fused_workgroups() / 2;
  const int64_t qtiles = ((int64_t)a.n + kBwdStatsTile - 1) / kBwdStatsTile;
  // Equal blocks run in whole rounds; under a mask their steps are an upper
  // bound and the rounds are not whole (B=1 H=8 N=6016 d128, causal mask: 376
  // blocks split for their rounds 467 us, unsplit 426).
  int64_t steps[kBwdMaxSplitBlocks], longest = 0, shortest = INT64_MAX, sum = 0;
  for (int kb = 0; kb < nkb; ++kb) {
    const int64_t q_first =
        causal ? std::min(qtiles, std::max<int64_t>(0, (int64_t)kb * kBwdBlockKeys - a.diag) /
                                      kBwdStatsTile)
               : 0;
    steps[kb] = a.group * (qtiles - q_first);
    longest = std::max(longest, steps[kb]);
    shortest = std::min(shortest, steps[kb]);
    sum += steps[kb];
  }
  const bool equal = longest == shortest && a.mbits == nullptr;
  const double load = (double)sum * units / cus;  // steps per CU
  // No split can be estimated below a CU's mean load: most launches that fill
  // the GPU end here.
  const int64_t rounds = (nkb * units + cus - 1) / cus;
  const double one_each =
      equal
          ? (double)((longest + kPieceSteps) * rounds)
          : std::max((double)longest + kPieceSteps, load + (double)kPieceSteps * nkb * units / cus);
  if ((std::max(load, (double)kMinPiece) + kPieceSteps + kMergeSteps) * kMinGain > one_each)
    return 0;
  auto pieces_of = [](int64_t st, int64_t t) { return std::max<int64_t>(1, (st + t - 1) / t); };
  double best = 0;
  int64_t best_t = 0;
  for (const int parts : {2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32, 40, 48, 64}) {
    const int64_t t = (longest + parts - 1) / parts;
    if (t < kMinPiece) break;
    int64_t count = 0;
    for (int kb = 0; kb < nkb; ++kb) count += pieces_of(steps[kb], t);
    const int64_t total = count * units;
    if (count > kBwdMaxPieces || total > (int64_t)kMaxPiecesPerCu * cus) break;
    double est = (double)t + kPieceSteps;
    if (total > cus) {
      if (equal)
        est *= (double)((total + cus - 1) / cus);
      else
        est = std::max(est, load + (double)kPieceSteps * total / cus +
                                0.5 * (double)sum / count);
    }
    if (best_t == 0 || est + kMergeSteps < best) {
      best = est + kMergeSteps;
      best_t = t;
    }
  }
  if (best_t == 0 || best * kMinGain > one_each || best + kMinSaved > one_each) return 0;
  int64_t n[kBwdMaxSplitBlocks];
  int first = 0;
  for (int kb = 0; kb < nkb; ++kb) {
    n[kb] = pieces_of(steps[kb], best_t);
    s.first[kb] = (uint16_t)first;
    first += (int)n[kb];
    if (n[kb] > 1) s.merge[s.merged++] = (uint8_t)kb;
  }
  s.first[nkb] = (uint16_t)first;
  // The longest pieces first: short ones fill the end of the launch.
  int order[kBwdMaxSplitBlocks];
  for (int kb = 0; kb < nkb; ++kb) order[kb] = kb;
  std::stable_sort(order, order + nkb,
                   [&](int x, int y) { return steps[x] * n[y] > steps[y] * n[x]; });
  for (int i = 0; i < nkb; ++i)
    for (int64_t piece = 0; piece < n[order[i]]; ++piece)
      s.item[s.pieces++] = (uint16_t)(order[i] | (int)piece << 8);
  return units * s.pieces * 2 * kBwdBlockKeys * head_dim * (int64_t)sizeof(float);
}

int launch_backward(const BwdArgs& args, const BwdSplit& split, int batch, int head_dim,
                    bool causal, bool bf16, hipStream_t stream) {
  BwdArgs a = args;
  a.qtiles = (a.n + kBwdStatsTile - 1) / kBwdStatsTile;
  a.units = batch * (a.hq / a.group);
  a.num_qblocks = (a.n + kBwdBlockRows - 1) / kBwdBlockRows;
  a.items = batch * a.hq * a.num_qblocks;
  a.xcds = plan_xcds(a, a.units, a.items);
  a.pair_half = 0;
  a.mwords = (a.nk + 63) / 64;
  const bool mask = a.mbits != nullptr;
  if (head_dim == 128) {
    if (mask) {
      if (bf16) launch_bwd<128, true, true>(a, split, batch, causal, stream);
      else launch_bwd<128, false, true>(a, split, batch, causal, stream);
    } else {
      if (bf16) launch_bwd<128, true, false>(a, split, batch, causal, stream);
      else launch_bwd<128, false, false>(a, split, batch, causal, stream);
    }
  } else {
    if (mask) {
      if (bf16) launch_bwd<64, true, true>(a, split, batch, causal, stream);
      else launch_bwd<64, false, true>(a, split, batch, causal, stream);
    } else {
      if (bf16) launch_bwd<64, true, false>(a, split, batch, causal, stream);
      else launch_bwd<64, false, false>(a, split, batch, causal, stream);
    }
  }
  return 0;
}

}  // namespace fa
