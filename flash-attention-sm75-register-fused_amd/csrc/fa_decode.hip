// Split-K forward for few query rows per K/V head (KV-cache decode).
//
// When heads_q / heads_kv * seq_len <= 32, all query rows that read one
// (batch, KV head) -- the "unit" -- fit the 32 query columns of one MFMA
// tile, and the work is streaming K and V once from HBM: the path is
// HBM-bound (2 * Nk * D * 2 bytes per unit against 4 * rows * Nk * D FLOP).
// The 128-row prefill kernel would read K/V once per query head and leave
// most of its rows empty, so this path reorganises the work:
//
//   * grid = units x splits: split s of a unit takes key tiles
//     [s * chunk, (s + 1) * chunk) of 32 keys; the four waves of a workgroup
//     take every fourth tile of the chunk and run independently (no
//     workgroup barrier inside the loop): K straight from HBM into VGPRs as
//     the MFMA A operand, V through a per-wave, double-buffered LDS tile
//     (direct-to-LDS loads, read back transposed with ds_read_b64_tr_b16);
//   * the four waves' (max, sum, O) merge through LDS at the end;
//   * with one split the workgroup writes O (and LSE) directly; otherwise it
//     writes an fp32 partial (unnormalised O, running max in log2 units, sum)
//     to the caller's workspace, and the unit's last workgroup to finish
//     merges them (MERGE) or, where they are many bytes, fa_decode_combine
//     (for many splits, fa_decode_combine_wide) does in a second launch.
//
// Small launches (a 128-row prefill grid of at most kSmallLaunchItems
// workgroups, e.g. one head of 512 rows) take the same path with the query
// rows of each (batch, KV head) in blocks of 32: a unit is then one such
// block, and its keys are split over workgroups like a decode unit's, so the
// launch spreads over many CUs instead of running a few long key chains.
//
// The MFMA formulation, the LDS tile layout, the online-softmax numerics and
// the lazy rescale are those of the prefill kernel (fa_fwd.hip): S^T = K Q^T
// with one query per lane, P kept in registers as the B operand of
// O^T = V^T P^T.  Query column c of unit (b, hkv, row block rb) is row
// r = 32 rb + c of the (batch, KV head): query head hkv * group + r / Nq,
// query index r % Nq.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <chrono>

#include "fa_internal.h"

#include "fa_kernel_common.h"

namespace fa {
namespace {

constexpr int kDecTile = 32;       // keys per wave tile

typedef unsigned v4u __attribute__((ext_vector_type(4)));

// Per-wave V tile: 32 rows of D halves with no padding (a direct load costs
// its wave about the same per instruction whatever it moves, so padding
// lanes were a third of the loads at head_dim 64, a fifth at 128).  Only the
// transposing V reads touch this tile, and each reads the same 64 bytes of
// rows 4k..4k+3 (and 4k+8..): chunk c of row r is stored at c ^ swz(r) so
// that those four rows land in four disjoint 64-byte windows of the 256-byte
// bank sweep -- at head_dim 64 (128-byte rows) rows 4k and 4k+2 differ in
// chunk bit 2 (dense_swizzle, as the prefill kernel's dense tiles), at 128
// (256-byte rows, one sweep each) chunk bits 2-3 take the row's position in
// its group of four.  swz(r + 16) = swz(r), so the two 16-key halves share a
// base; the XOR reaches chunk bit 2, so each 32-dim output tile has its own.
template <int D>
struct DecLds {
  static constexpr int Pitch = D;                      // halves per row
  static constexpr int Tile = kDecTile * Pitch;        // halves per V tile
  static constexpr int Segs = Tile * 2 / 1024;         // 1 KB direct-load segments
  static_assert(Tile * 2 % 1024 == 0, "V tile must be whole segments");
  static __device__ __forceinline__ int swz(int r) {
    if constexpr (D == 64) return dense_swizzle(r);
    else return (r & 3) << 2;
  }
};

// s_waitcnt with only vmcnt constrained (gfx9 encoding: vmcnt[3:0] and
// vmcnt[5:4] at bits 15:14, expcnt 7, lgkmcnt 15), followed by a compiler
// memory barrier: the waitcnt intrinsic does not touch memory as far as the
// compiler knows, so without it the LDS reads that depend on the wait could
// be hoisted above it.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
  asm volatile("" ::: "memory");
}

// Cache policy of the in-kernel merge's accesses: sc1, coherent over the
// device's L2s.
constexpr int kCoherent = 16;
// 16-byte partials a merging thread has in flight at once.
constexpr int kMergeLoads = 8;
// Units with at most this many bytes of partial O are merged by the split-K
// kernel itself: it saves the second launch (3.1 us of host time, and 0-0.5
// us on the GPU: Hq=14 Hkv=2 d64 4097 keys 9.0 -> 8.6 us back to back, 11.0 ->
// 8.7 through the SDPA patch, where the host is the limit).  One workgroup
// reads a unit's partials at about 50 bytes/ns, so larger ones go to the
// combine kernels' many (Hq=32 Hkv=8 8 rows 2048 keys d128, 128 KB: 14.8 us
// merged here, 11.1 by the combine kernel; 64 KB within 0.7 us either way).
constexpr int kMergeMaxBytes = 64 << 10;
// ... and at head_dim 64 not where many units of many splits fill the GPU:
// every CU then ends with a merge of short partials, which the next launch
// cannot overlap (B=2 Hq=8 Hkv=8 4096 keys d64, 16 units of 16 splits: 9.5
// merged here, 8.8 by the combine kernel; B=16 H=1 16384 keys 16.9 and 16.1;
// 8 splits, B=4 H=8 4096 keys, 11.5 and 11.6).  Row blocks, whose units are
// many as well, up to 5 splits and 48 KB (8 splits of 32 columns at head_dim 64,
// 8 heads 128 x 2600 11.3 merged here and 10.2, 6 splits 11.3 and 11.0, 5 11.7
// and 11.9; head_dim 128, 4 splits, 8 heads 256 x 2600 17.8 and 17.3, 3 24.6
// and 25.0).
constexpr int kMergeMaxSplits64 = 8;
constexpr int kMergeFewWgs = 128;
constexpr int kMergeMaxBlockBytes = 48 << 10, kMergeMaxBlockSplits = 5;
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));

// The max that a merge of splits takes the others relative to.  Where it is -inf
// every split so far saw no key, with sum and O zero, or only NaN scores, with
// both NaN.  Relative to 0 the weight of either is 2^-inf = 0, which leaves the
// zeros and keeps the NaN (such splits left out, a query with a NaN in it gave
// zeros where an unsplit call gives NaN).
__device__ __forceinline__ float finite_max(float m) { return m == -__builtin_inff() ? 0.0f : m; }

// Normalises and stores 4 dimensions of query column c of row block rb of
// (batch, KV head) bh from the splits' merged max (log2 units), sum and O,
// and the row's LSE once.  Columns past the last row are not stored.
template <int D, bool BF16>
__device__ __forceinline__ void store_merged(const DecArgs& d, int bh, int rb, int c, int dim,
                                             float m, float l, v4f o) {
  const FwdArgs& a = d.f;
  const int hkv_count = a.hq / a.group;
  const int b = bh / hkv_count;
  const int hkv = bh - b * hkv_count;
  const int r = rb * kDecodeMaxRows + c;
  if (r >= d.total_rows) return;
  const int g = r / a.n;
  const int qi = r - g * a.n;
  const int hq = hkv * a.group + g;
  const float inv = (l > 0.0f) ? (1.0f / l) : 0.0f;
  half4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = Elem<BF16>::round(o[e] * inv);
  *(half4*)(a.o + b * a.osb + hq * a.osh + (int64_t)qi * a.osn + dim) = v;
  if (a.lse != nullptr && dim == 0) {
    const float m_use = (m == -__builtin_inff()) ? 0.0f : m;
    a.lse[((int64_t)b * a.hq + hq) * a.n + qi] =
        (m_use + __builtin_log2f(l)) * 0.69314718055994530942f;
  }
}

// MASK_MODE: 0 no explicit mask, 1 mask bits (one 32-bit word per row and
// tile), 2 key-padding bytes (fa_fwd_params.mask_keys: one byte per key, the
// same for every row of the batch; a ballot over the tile's 32 bytes forms
// the word).  MERGE: the unit's last workgroup merges its splits (an instance
// of its own: with that code in it the others' tile loop ran up to 13%
// slower, one head of 256 rows of 8 at head_dim 64 5.0 -> 5.6 us).
template <int D, bool CAUSAL, int MASK_MODE, bool BF16, bool MERGE>
__global__ void __launch_bounds__(kThreads, 2) fa_decode_kernel(const DecArgs d) {
  constexpr bool MASK = MASK_MODE != 0;
  constexpr bool KEY_BYTES = MASK_MODE == 2;
  const FwdArgs& a = d.f;
  using L = DecLds<D>;
  using E = Elem<BF16>;
  constexpr int KK = D / 16;   // 16-wide contraction steps of S^T
  constexpr int MT = D / 32;   // 32-row output tiles of O^T
  constexpr int NPV = 2 * MT;  // P V MFMAs per 32-key tile
  constexpr int SEGS = L::Segs;

  // Per-wave V tiles: wave w uses [w * Tile, (w + 1) * Tile) of each array.
  __shared__ __attribute__((aligned(1024))) _Float16 v_lds0[kWaves * L::Tile];
  __shared__ __attribute__((aligned(1024))) _Float16 v_lds1[kWaves * L::Tile];
  // Each wave's running max and row sums for the final merge (its O goes to
  // its two V tiles, which it fills exactly: MT 32 x 32 float tiles).
  __shared__ float ml_lds[kWaves * 128];
  static_assert(MT / 2 * 16 * 64 * 4 <= L::Tile * 2, "O of a wave fits its V tiles");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  // Wave-uniform (in a scalar register): the per-wave buffer windows and LDS
  // destinations derived from it must be scalar, or every direct load would
  // become a loop over the distinct values of the wave.
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hi = lane >> 5;
  const int ql = lane & 31;
  const int grp = lane >> 4;
  const int gi = lane & 15;

  const int unit = (int)blockIdx.x / d.splits;
  const int split = (int)blockIdx.x - unit * d.splits;
  const int hkv_count = a.hq / a.group;
  const int bh = unit / d.row_blocks;  // (batch, KV head)
  const int rb = unit - bh * d.row_blocks;
  const int b = bh / hkv_count;
  const int hkv = bh - b * hkv_count;
  const int nq = a.n;
  const int NK = a.nk;

  // This lane's query column: row r of the (batch, KV head).
  const int r = rb * kDecodeMaxRows + ql;
  const bool row_ok = ql < d.rows && r < d.total_rows;
  const int g = r / nq;
  const int qi = r - g * nq;
  const int hq = hkv * a.group + g;
  // Smallest query index of the block's rows (wave-uniform): causal tiles
  // past it + diag need the per-element mask.
  const int r0 = rb * kDecodeMaxRows;
  const int r_last = min(d.total_rows, r0 + kDecodeMaxRows) - 1;
  const bool one_head = r0 / nq == r_last / nq;
  const int qi_lo = one_head ? r0 % nq : 0;
  // Largest query index of the block's rows: under causal masking no row of
  // the unit sees a key past qi_hi + diag, so tiles past it are skipped.
  const int qi_hi = one_head ? r_last % nq : nq - 1;
  const int unit_tiles =
      CAUSAL ? min(d.tiles, max(0, (qi_hi + a.diag + kDecTile) / kDecTile)) : d.tiles;

  half8 qf[KK];
  if (row_ok) {
    const _Float16* qp = a.q + b * a.qsb + hq * a.qsh + (int64_t)qi * a.qsn + 8 * hi;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) qf[kk] = *(const half8*)(qp + 16 * kk);
  } else {
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) qf[kk] = (half8)(_Float16)0;
  }
  if (a.negate_q) {
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) qf[kk] = negate16(qf[kk]);
  }

  // Tiles of this split, and this wave's share (every fourth one).
  const int t_begin = split * d.chunk_tiles;
  const int t_end = min(t_begin + d.chunk_tiles, unit_tiles);
  const int nt_w = t_end - t_begin > wave ? (t_end - t_begin - wave + kWaves - 1) / kWaves : 0;
  const int key0 = t_begin * kDecTile;
  const _Float16* Kp = a.k + b * a.ksb + hkv * a.ksh;
  const _Float16* Vp = a.v + b * a.vsb + hkv * a.vsh;

  // Loads of tile it are issued whether or not the tile exists (`valid`);
  // a missing tile reads through an empty window (zeros, no memory traffic),
  // so every iteration has the same loads in flight and one vmcnt value
  // serves all of them (a conditional load would make the compiler wait
  // for the worst case and serialise the prefetch).
  // K operand of tile it: key row (tile key base + ql), dims 16 kk + 8 hi;
  // rows past the last key read as zeros.
  const int k_rows_left = NK - key0;
  const int k_bytes = k_rows_left > 0 ? k_rows_left * (int)a.ksn * 2 : 0;
  auto load_k = [&](int it, half8 (&kf)[KK], bool valid) {
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(Kp + (int64_t)key0 * a.ksn, valid ? k_bytes : 0);
    const int key = (wave + kWaves * it) * kDecTile + ql;
    const int voff = key * (int)a.ksn * 2 + 16 * hi;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
      kf[kk] = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(rk, voff + 32 * kk, 0, 0));
  };

  // V direct loads: segment s, lane l covers tile bytes [1024 s + 16 l, +16).
  int goff_v[SEGS];
#pragma unroll
  for (int s = 0; s < SEGS; ++s) {
    const int pos = s * 1024 + 16 * lane;
    const int row = pos / (2 * L::Pitch);
    const int within = pos - row * (2 * L::Pitch);
    const int c = (within >> 4) ^ L::swz(row);
    goff_v[s] = (int)(row * a.vsn * 2) + 16 * c;
  }
  auto load_v = [&](int it, _Float16* tile, bool valid) {
    const int kb = key0 + (wave + kWaves * it) * kDecTile;
    const int rows_left = valid ? NK - kb : 0;
    const __amdgpu_buffer_rsrc_t rv =
        make_rsrc(Vp + (int64_t)kb * a.vsn, rows_left > 0 ? rows_left * (int)a.vsn * 2 : 0);
    // Non-temporal: every V row is read once (measured +13-17% on the
    // long-context shapes; the K loads, 32 rows x 32 bytes per instruction,
    // stay cached so that the other half of each line hits).
#pragma unroll
    for (int s = 0; s < SEGS; ++s) direct_load16_nt(rv, (lds_void*)(tile + s * 512), goff_v[s]);
  };
  _Float16* const my_v0 = v_lds0 + wave * L::Tile;
  _Float16* const my_v1 = v_lds1 + wave * L::Tile;

  // MASK: this lane's mask row read as 32-bit words (word t: keys of 32-key
  // tile t), through a buffer window over batch b's rows so the load is the
  // same kind as the K and V loads (their completion order is then the
  // issue order, which the vmcnt wait below relies on).  KEY_BYTES: byte
  // (tile * 32 + ql) of batch b's key row instead, one load per step too,
  // through a window that ends at the last key (keys past it read as 0).
  __amdgpu_buffer_rsrc_t rmask;
  int m_voff = 0;
  if (KEY_BYTES) {
    const int64_t span = NK > 0 ? (int64_t)(NK - 1) * a.mksk + 1 : 0;
    rmask = make_rsrc(a.mkeys + b * a.mksb, (int)min(span, (int64_t)INT32_MAX));
    m_voff = ql * (int)a.mksk;
  } else if (MASK) {
    const int hq_c = row_ok ? hq : hkv * a.group;
    const int qi_c = row_ok ? qi : 0;
    const int64_t words = (NK + 63) / 64;
    const int64_t span =
        ((int64_t)(hkv * a.group + a.group - 1) * a.msh + (int64_t)(nq - 1) * a.msq + words) * 8;
    rmask = make_rsrc(a.mbits + b * a.msb, (int)min(span, (int64_t)INT32_MAX));
    m_voff = (int)((hq_c * a.msh + qi_c * a.msq) * 8);
  }
  auto load_mask = [&](int it, bool valid) -> uint32_t {
    const int tile = valid ? t_begin + wave + kWaves * it : t_begin;
    if constexpr (KEY_BYTES)
      return __builtin_amdgcn_raw_buffer_load_b8(rmask, m_voff + tile * kDecTile * (int)a.mksk,
                                                 0, 0);
    return __builtin_amdgcn_raw_buffer_load_b32(rmask, m_voff + 4 * tile, 0, 0);
  };

  // Per-lane bases of the transposing V reads: rows 16ks + 4hi + gi/4
  // (+8), dims 32mt + 16(grp&1) + 4(gi&3), one pair of bases per mt.
  const int v_row = 4 * hi + (gi >> 2);
  const int v_c = 2 * (grp & 1) + ((gi & 3) >> 1);
  int v_base0[MT], v_base1[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    v_base0[mt] = v_row * L::Pitch + 8 * ((v_c + 4 * mt) ^ L::swz(v_row)) + 4 * (gi & 1);
    v_base1[mt] = (v_row + 8) * L::Pitch + 8 * ((v_c + 4 * mt) ^ L::swz(v_row + 8)) + 4 * (gi & 1);
  }
  auto read_v = [&](const _Float16* Vs, int v) -> half8 {
    const int ks = v / MT, mt = v % MT;
    const int imm = 16 * ks * L::Pitch;
    const half4 lo = ds_read_tr16(Vs + v_base0[mt] + imm);
    const half4 hi4 = ds_read_tr16(Vs + v_base1[mt] + imm);
    return __builtin_shufflevector(lo, hi4, 0, 1, 2, 3, 4, 5, 6, 7);
  };

  float16v oacc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) oacc[mt] = (float16v)0.0f;
  float m_run = -__builtin_inff();
  float l_run = 0.0f;
  const float c2 = a.c;
  const int diag_row = qi + a.diag;  // causal: keys <= diag_row are visible

  half8 kA[KK], kB[KK];

  // The word of a tile from what load_mask returned (bit k: key 32 t + k
  // visible): key bytes (lanes l and l + 32 hold key 32 t + l) give it as the
  // low half of a ballot; mask bits are the lane's word itself.
  auto word_of = [&](uint32_t raw) -> uint32_t {
    if constexpr (KEY_BYTES) return (uint32_t)__builtin_amdgcn_ballot_w64(raw != 0);
    else return raw;
  };
  // Whether no lane (query row) sees a key of a tile: its K and V are then
  // not read (an empty window: zeros, no memory traffic) and its scores are
  // all masked, so it adds exactly nothing.  Padded batches skip their
  // padding this way.
  auto hidden = [&](uint32_t w) -> bool { return __builtin_amdgcn_ballot_w64(w != 0) == 0; };

  // One tile: S, softmax, P V.  The loads of the next tile are issued first.
  // MASK: mw and w_next are the words of tiles it and it + 1; raw2 is what
  // load_mask returned for tile it + 2 (issued a step ago), and tile it + 3's
  // mask load goes to raw3.  Returns tile it + 2's word, formed after this
  // step's V wait, when raw2 has landed: every mask load is issued two steps
  // before its tile's K and V loads, so deciding whether they are needed
  // never waits.
  auto step = [&](int it, half8 (&kc)[KK], half8 (&kn)[KK], _Float16* vc, _Float16* vn,
                  uint32_t mw, uint32_t w_next, uint32_t raw2, uint32_t& raw3) -> uint32_t {
    const bool has_next = it + 1 < nt_w;
    const bool skip_next = MASK && hidden(w_next);
    if (MASK) raw3 = load_mask(it + 3, it + 3 < nt_w);
    load_k(it + 1, kn, has_next && !skip_next);
    load_v(it + 1, vn, has_next && !skip_next);
    float16v s = (float16v)0.0f;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
      s = E::mfma(kc[kk], qf[kk], s);

    const int kstart = key0 + (wave + kWaves * it) * kDecTile;
    bool need_mask =
        (kstart + kDecTile > NK) || (CAUSAL && kstart + kDecTile - 1 > qi_lo + a.diag);
    if (MASK) need_mask = need_mask || __builtin_amdgcn_ballot_w64(~mw != 0) != 0;
    if (need_mask) {
      const uint32_t mws = mw >> (4 * hi);  // bit 8 (i / 4) + i % 4: element i
      static_for<16>([&](auto i_c) {
        constexpr int i = decltype(i_c)::value;
        const int key = kstart + 8 * (i >> 2) + 4 * hi + (i & 3);
        bool masked = key >= NK || (CAUSAL && key > diag_row);
        if (MASK) masked = masked || ((mws >> (8 * (i >> 2) + (i & 3))) & 1) == 0;
        if (masked) s[i] = -__builtin_inff();
      });
    }
    float mx = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
    mx = halves_max(mx);
    const bool grow = (mx - m_run) * c2 > kRescaleLog2;
    if (__builtin_amdgcn_ballot_w64(grow) != 0) {
      const float m_new = fmaxf(m_run, mx);
      const float m_use = (m_new == -__builtin_inff()) ? 0.0f : m_new;
      const float alpha =
          (m_run == -__builtin_inff()) ? 0.0f : __builtin_amdgcn_exp2f((m_run - m_use) * c2);
      l_run *= alpha;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) oacc[mt] *= alpha;
      m_run = m_new;
    }
    const float mc = ((m_run == -__builtin_inff()) ? 0.0f : m_run) * c2;
    uint4v pf[2];  // P operands as 32-bit lanes (pairs written whole)
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
      const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], c2, -mc));
      const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i + 1], c2, -mc));
      const half2v pr = E::pack(p0, p1);
      pf[i >> 3][(i & 7) >> 1] = __builtin_bit_cast(unsigned, pr);
      l_run = E::sum2(pr, l_run);
    }
    // V of this tile has landed once only the next tile's loads are pending
    // (loads complete in order).
    wait_vmcnt<KK + SEGS + (MASK ? 1 : 0)>();
    const uint32_t w_next2 = MASK ? word_of(raw2) : ~0u;
    half8 vf[NPV];
#pragma unroll
    for (int v = 0; v < NPV; ++v) vf[v] = read_v(vc, v);
#pragma unroll
    for (int v = 0; v < NPV; ++v) {
      const int ks = v / MT, mt = v % MT;
      oacc[mt] = E::mfma(vf[v], __builtin_bit_cast(half8, pf[ks]), oacc[mt]);
    }
    return w_next2;
  };

  if (nt_w > 0) {
    // Every step issues one mask load (MASK), then K and V of its next tile;
    // the prologue issues the masks of tiles 0, 1 and 2, then K and V of tile
    // 0 (read whether hidden or not: deciding would wait for its mask first).
    uint32_t raw0 = 0u, raw1 = 0u, rawA = 0u, rawB = 0u, wc = ~0u, wn = ~0u;
    if (MASK) {
      raw0 = load_mask(0, true);
      raw1 = load_mask(1, 1 < nt_w);
      rawB = load_mask(2, 2 < nt_w);
    }
    load_k(0, kA, true);
    load_v(0, my_v0, true);
    if (MASK) {
      wc = word_of(raw0);
      wn = word_of(raw1);
    }
    int it = 0;
    for (; it + 1 < nt_w; it += 2) {
      uint32_t w2 = step(it, kA, kB, my_v0, my_v1, wc, wn, rawB, rawA);
      wc = wn;
      wn = w2;
      w2 = step(it + 1, kB, kA, my_v1, my_v0, wc, wn, rawA, rawB);
      wc = wn;
      wn = w2;
    }
    if (it < nt_w) step(it, kA, kB, my_v0, my_v1, wc, wn, rawB, rawA);
  }

  // ---- merge the four waves through LDS (the V tiles are free now) --------
  // The last step's loads of a tile that does not exist are still in flight:
  // drain them, or their zeros could land in LDS after the merge writes.
  wait_vmcnt<0>();
  const float l_tot = halves_sum(l_run);
  __syncthreads();
  {
    float* o_lo = (float*)(v_lds0 + wave * L::Tile);
    float* o_hi = (float*)(v_lds1 + wave * L::Tile);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      float* dst = (mt < MT / 2 ? o_lo : o_hi) + (mt % (MT / 2)) * 16 * 64;
#pragma unroll
      for (int i = 0; i < 16; ++i) dst[i * 64 + lane] = oacc[mt][i];
    }
    float* ml = ml_lds + wave * 128;
    ml[lane] = m_run;
    ml[64 + lane] = l_tot;
  }
  __syncthreads();
  // Wave mt merges output tile mt (at head_dim 64 waves 2 and 3 have none, and
  // go on only for the splits' merge).
  if (!MERGE && wave >= MT) return;
  const int mt = wave < MT ? wave : 0;
  float m_w[kWaves], M = -__builtin_inff();
#pragma unroll
  for (int u = 0; u < kWaves; ++u) {
    const float* ml = ml_lds + u * 128;
    m_w[u] = ml[lane];
    M = fmaxf(M, m_w[u]);
  }
  float Ltot = 0.0f;
  float o[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) o[i] = 0.0f;
#pragma unroll
  for (int u = 0; u < kWaves; ++u) {
    const float f = (m_w[u] == -__builtin_inff()) ? 0.0f : __builtin_amdgcn_exp2f((m_w[u] - M) * c2);
    const float* base = (const float*)((mt < MT / 2 ? v_lds0 : v_lds1) + u * L::Tile) +
                        (mt % (MT / 2)) * 16 * 64;
    const float* ml = ml_lds + u * 128;
    Ltot += f * ml[64 + lane];
#pragma unroll
    for (int i = 0; i < 16; ++i) o[i] += f * base[i * 64 + lane];
  }
  const bool mine = row_ok && wave < MT;
  if (!MERGE && !mine) return;
  if (!MERGE && d.splits == 1) {
    const float inv = (Ltot > 0.0f) ? (1.0f / Ltot) : 0.0f;
    _Float16* op = a.o + b * a.osb + hq * a.osh + (int64_t)qi * a.osn + 32 * mt + 4 * hi;
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      half4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = E::round(o[4 * g4 + e] * inv);
      *(half4*)(op + 8 * g4) = v;
    }
    if (a.lse != nullptr && mt == 0 && hi == 0) {
      const float m_use = (M == -__builtin_inff()) ? 0.0f : M;
      a.lse[((int64_t)b * a.hq + hq) * nq + qi] =
          (m_use * c2 + __builtin_log2f(Ltot)) * 0.69314718055994530942f;
    }
    return;
  }
  const float M2 = (M == -__builtin_inff()) ? M : M * c2;  // log2 units
  if constexpr (!MERGE) {  // a combine kernel merges the splits
    const int64_t p = ((int64_t)unit * d.splits + split) * d.rows + ql;
    float* po = d.part_o + p * D + 32 * mt + 4 * hi;
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      float4 v = {o[4 * g4], o[4 * g4 + 1], o[4 * g4 + 2], o[4 * g4 + 3]};
      *(float4*)(po + 8 * g4) = v;
    }
    if (mt == 0 && hi == 0) {
      d.part_ml[2 * p] = M2;
      d.part_ml[2 * p + 1] = Ltot;
    }
    return;
  }

  if constexpr (MERGE) {
    // ---- merge of the unit's splits by the last workgroup to finish ----------
    // Every partial and flag goes through device-coherent accesses (the sc1
    // bit: stores write through to memory, loads do not take a line another
    // XCD's L2 may have left stale), so no cache has to be written back or
    // invalidated: a release fence here would write back the XCD's whole L2
    // (20-35% of a call, measured).  A workgroup's partials are acknowledged
    // before it sets its flag, and its flag before it reads the others', so of
    // any two workgroups of a unit at least one sees the other's flag set, and
    // the last flag to be set is set by a workgroup that sees them all.  Two that
    // both see all of them merge the same partials in the same order and store
    // the same values.
    const int unit_ml = unit * d.splits * d.rows;  // first (split, row) record of the unit
    const __amdgpu_buffer_rsrc_t rp = make_rsrc(d.part_o + (int64_t)unit_ml * D, d.splits * d.rows * D * 4);
    const __amdgpu_buffer_rsrc_t rl = make_rsrc(d.part_ml + (int64_t)unit_ml * 2, d.splits * d.rows * 8);
    const __amdgpu_buffer_rsrc_t rf = make_rsrc(d.flags + (int64_t)unit * d.splits, d.splits * 8);
    if (mine) {
      const int rec = split * d.rows + ql;
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const v4f v = {o[4 * g4], o[4 * g4 + 1], o[4 * g4 + 2], o[4 * g4 + 3]};
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, v), rp,
                                               (rec * D + 32 * mt + 4 * hi + 8 * g4) * 4, 0, kCoherent);
      }
      if (mt == 0 && hi == 0)
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v2f{M2, Ltot}), rl, rec * 8, 0,
                                              kCoherent);
    }
    wait_vmcnt<0>();
    __syncthreads();
    if (tid == 0) {
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, d.mark), rf, split * 8, 0, kCoherent);
      wait_vmcnt<0>();
    }
    __syncthreads();
    bool set = true;  // one flag per thread (at most kThreads splits)
    if (tid < d.splits)
      set = __builtin_bit_cast(uint64_t, __builtin_amdgcn_raw_buffer_load_b64(rf, tid * 8, 0, kCoherent)) ==
            d.mark;
    if (!__syncthreads_and(set)) return;

    // Thread (grp, item): 4 dimensions of one query column (item = column *
    // D / 4 + dimension / 4), splits grp, grp + groups, ...; the groups' states
    // meet in LDS.  More than kThreads items: one group, items in turns.
    const int items = d.rows * (D / 4);
    const int groups = max(1, min(kThreads / items, d.splits));
    const int grp_m = groups > 1 ? tid / items : 0;
    float* const xm = ml_lds;              // [group][item] max, then sum (kThreads each)
    float4* const xo = (float4*)v_lds0;    // [group][item] O
    static_assert(kThreads * 16 <= kWaves * L::Tile * 2, "the merge's states fit the V tiles");
    // NI items at once (kThreads apart), so that a thread with several has all
    // their loads in flight together.
    auto merge = [&](int it0, auto ni_c) {
      constexpr int NI = decltype(ni_c)::value;
      constexpr int BATCH = kMergeLoads / NI;
      float m_acc[NI], l_acc[NI];
      v4f o_acc[NI];
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        m_acc[i] = -__builtin_inff();
        l_acc[i] = 0.0f;
        o_acc[i] = (v4f)0.0f;
      }
      for (int s0 = grp_m; s0 < d.splits; s0 += BATCH * groups) {
        v4f os[NI][BATCH];
        v2f ml[NI][BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
#pragma unroll
          for (int i = 0; i < NI; ++i) {
            // Splits past the last read zeros beyond the windows (their max is
            // replaced below).
            const int it = it0 + i * kThreads;
            const int rec = (s0 + u * groups) * d.rows + it / (D / 4);
            ml[i][u] =
                __builtin_bit_cast(v2f, __builtin_amdgcn_raw_buffer_load_b64(rl, rec * 8, 0, kCoherent));
            os[i][u] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(
                                                   rp, (rec * D + 4 * (it % (D / 4))) * 4, 0, kCoherent));
          }
        }
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          float m_new = m_acc[i];
#pragma unroll
          for (int u = 0; u < BATCH; ++u) {
            if (s0 + u * groups >= d.splits) ml[i][u][0] = -__builtin_inff();
            m_new = fmaxf(m_new, ml[i][u][0]);
          }
          const float m_use = finite_max(m_new);
          const float alpha = __builtin_amdgcn_exp2f(m_acc[i] - m_use);
          l_acc[i] *= alpha;
          o_acc[i] *= alpha;
#pragma unroll
          for (int u = 0; u < BATCH; ++u) {
            const float w = __builtin_amdgcn_exp2f(ml[i][u][0] - m_use);
            l_acc[i] += w * ml[i][u][1];
            o_acc[i] += w * os[i][u];
          }
          m_acc[i] = m_new;
        }
      }
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int it = it0 + i * kThreads;
        if (groups > 1) {
          xm[tid] = m_acc[i];
          xm[kThreads + tid] = l_acc[i];
          xo[tid] = __builtin_bit_cast(float4, o_acc[i]);
        } else {
          store_merged<D, BF16>(d, bh, rb, it / (D / 4), 4 * (it % (D / 4)), m_acc[i], l_acc[i], o_acc[i]);
        }
      }
    };
    int it = tid - grp_m * items;
    if (grp_m < groups) {
      for (; it + kThreads < items; it += 2 * kThreads) merge(it, std::integral_constant<int, 2>{});
      if (it < items) merge(it, std::integral_constant<int, 1>{});
    }
    if (groups == 1) return;
    __syncthreads();
    if (tid >= items) return;
    float Mg = xm[tid];
    for (int q = 1; q < groups; ++q) Mg = fmaxf(Mg, xm[q * items + tid]);
    float lg = 0.0f;
    v4f og = {0.0f, 0.0f, 0.0f, 0.0f};
    const float Mg_use = finite_max(Mg);
    for (int q = 0; q < groups; ++q) {
      const float w = __builtin_amdgcn_exp2f(xm[q * items + tid] - Mg_use);
      lg += w * xm[kThreads + q * items + tid];
      og += w * __builtin_bit_cast(v4f, xo[q * items + tid]);
    }
    store_merged<D, BF16>(d, bh, rb, tid / (D / 4), 4 * (tid % (D / 4)), Mg, lg, og);
  }
}

// Merges the splits of one (unit, query column) with 256 threads:
// O = sum_s 2^(m_s - M) O_s / sum_s 2^(m_s - M) l_s, M = max_s m_s.
// Thread (grp, dim) of the 256 / D groups of D threads takes every
// (256 / D)-th split from grp: it loads the (max, sum) records and its
// dimension of the partial O of four splits at a time, all independent of
// each other, and folds them into its own running (max, sum, O) as the
// prefill kernel folds key tiles; the groups' states merge once through
// LDS.  One round trip to memory per four splits and one barrier: the
// partials come from other XCDs' caches or HBM, so a merge that waits for
// the maxima before it asks for the sums and the O values pays that latency
// three times.
constexpr int kCombineThreads = 256;
constexpr int kMaxSplits = 1024;  // splits per unit (the plan's bound)

template <int D, bool BF16>
__global__ void __launch_bounds__(kCombineThreads) fa_decode_combine(const DecArgs d) {
  const FwdArgs& a = d.f;
  constexpr int GROUPS = kCombineThreads / D;
  __shared__ float m_grp[GROUPS], l_grp[GROUPS];
  __shared__ float o_grp[GROUPS][D];
  const int tid = threadIdx.x;
  const int unit = (int)blockIdx.x / d.rows;
  const int c = (int)blockIdx.x - unit * d.rows;  // query column of the unit
  const int hkv_count = a.hq / a.group;
  const int bh = unit / d.row_blocks;
  const int rb = unit - bh * d.row_blocks;
  const int b = bh / hkv_count;
  const int hkv = bh - b * hkv_count;
  const int r = rb * kDecodeMaxRows + c;
  if (r >= d.total_rows) return;  // whole workgroup: columns past the last row
  const int g = r / a.n;
  const int qi = r - g * a.n;
  const int hq = hkv * a.group + g;
  const int64_t p0 = (int64_t)unit * d.splits * d.rows + c;  // split s: p0 + s * rows
  const int S = d.splits;

  const int dim = tid % D;
  const int grp = tid / D;
  constexpr float kNegInf = -__builtin_inff();
  // Running state of this thread's splits: max (log2 units), sum, O[dim]
  // relative to that max (finite_max).  A split that saw no key has max -inf and
  // adds nothing; while every split so far is such, the state stays (-inf, 0, 0).
  float m_run = kNegInf, l_run = 0.0f, o_run = 0.0f;
  auto fold = [&](int n, const float* ms, const float* ls, const float* os) {
    float m_new = m_run;
    for (int u = 0; u < n; ++u) m_new = fmaxf(m_new, ms[u]);
    const float m_use = finite_max(m_new);
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
    l_run *= alpha;
    o_run *= alpha;
    for (int u = 0; u < n; ++u) {
      const float w = __builtin_amdgcn_exp2f(ms[u] - m_use);
      l_run += w * ls[u];
      o_run += w * os[u];
    }
    m_run = m_new;
  };
  int s = grp;
  for (; s + 3 * GROUPS < S; s += 4 * GROUPS) {
    float ms[4], ls[4], os[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t p = p0 + (int64_t)(s + u * GROUPS) * d.rows;
      ms[u] = d.part_ml[2 * p];
      ls[u] = d.part_ml[2 * p + 1];
      os[u] = d.part_o[p * D + dim];
    }
    fold(4, ms, ls, os);
  }
  for (; s < S; s += GROUPS) {
    const int64_t p = p0 + (int64_t)s * d.rows;
    const float ms = d.part_ml[2 * p], ls = d.part_ml[2 * p + 1], os = d.part_o[p * D + dim];
    fold(1, &ms, &ls, &os);
  }
  if (dim == 0) {
    m_grp[grp] = m_run;
    l_grp[grp] = l_run;
  }
  o_grp[grp][dim] = o_run;
  __syncthreads();
  if (grp != 0) return;
  float M = m_grp[0];
#pragma unroll
  for (int q = 1; q < GROUPS; ++q) M = fmaxf(M, m_grp[q]);
  float o = 0.0f, Ltot = 0.0f;
  const float m_use = finite_max(M);
#pragma unroll
  for (int q = 0; q < GROUPS; ++q) {
    const float w = __builtin_amdgcn_exp2f(m_grp[q] - m_use);
    o += w * o_grp[q][dim];
    Ltot += w * l_grp[q];
  }
  const float inv = (Ltot > 0.0f) ? (1.0f / Ltot) : 0.0f;
  a.o[b * a.osb + hq * a.osh + (int64_t)qi * a.osn + dim] = Elem<BF16>::round(o * inv);
  if (a.lse != nullptr && dim == 0) {
    a.lse[((int64_t)b * a.hq + hq) * a.n + qi] =
        (m_use + __builtin_log2f(Ltot)) * 0.69314718055994530942f;
  }
}

// Launches whose threads would each walk more than a few batches of splits
// in fa_decode_combine (split count times head_dim at least
// kWideCombineMin; e.g. one KV head of 65536 keys at 256 splits, whose
// combine took 23 us that way) take this variant: one workgroup per (unit,
// query column, 32 dimensions), 256 threads = 32 split groups x 8 lanes, lane
// i taking dimensions 4i..4i+3 of the chunk (a float4 of each split's
// partial O) and group g the splits g, g + 32, ... with up to 8 loads in
// flight per thread; the groups' states merge once through LDS.  For few
// splits its many small workgroups cost more than they save (a 16-column
// GQA decode with 4 splits: 14% slower), hence the threshold.
constexpr int kWideLanes = 8;                              // float4 lanes: 32 dims
constexpr int kWideGroups = kCombineThreads / kWideLanes;  // split groups
constexpr int kWideBatch = 8;                              // splits in flight per thread
constexpr int kWideCombineMin = 4096;                      // splits * head_dim

template <int D, bool BF16>
__global__ void __launch_bounds__(kCombineThreads) fa_decode_combine_wide(const DecArgs d) {
  const FwdArgs& a = d.f;
  constexpr int CHUNKS = D / (4 * kWideLanes);
  __shared__ float m_grp[kWideGroups], l_grp[kWideGroups];
  __shared__ float4 o_grp[kWideGroups][kWideLanes];
  const int tid = threadIdx.x;
  const int chunk = (int)blockIdx.x % CHUNKS;
  const int uc = (int)blockIdx.x / CHUNKS;
  const int unit = uc / d.rows;
  const int c = uc - unit * d.rows;  // query column of the unit
  const int hkv_count = a.hq / a.group;
  const int bh = unit / d.row_blocks;
  const int rb = unit - bh * d.row_blocks;
  const int b = bh / hkv_count;
  const int hkv = bh - b * hkv_count;
  const int r = rb * kDecodeMaxRows + c;
  if (r >= d.total_rows) return;  // whole workgroup: columns past the last row
  const int g = r / a.n;
  const int qi = r - g * a.n;
  const int hq = hkv * a.group + g;
  const int64_t p0 = (int64_t)unit * d.splits * d.rows + c;  // split s: p0 + s * rows
  const int S = d.splits;

  const int lane = tid % kWideLanes;
  const int grp = tid / kWideLanes;
  const int dim0 = 4 * (chunk * kWideLanes + lane);
  constexpr float kNegInf = -__builtin_inff();
  // Running state as in fa_decode_combine, for 4 dimensions.
  float m_run = kNegInf, l_run = 0.0f;
  float o_run[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int s = grp; s < S; s += kWideBatch * kWideGroups) {
    float ms[kWideBatch], ls[kWideBatch];
    float4 os[kWideBatch];
    int n = 0;  // splits of this batch (a prefix of the 8)
#pragma unroll
    for (int u = 0; u < kWideBatch; ++u) {
      const int su = s + u * kWideGroups;
      if (su < S) {
        const int64_t p = p0 + (int64_t)su * d.rows;
        const float2 ml = *(const float2*)(d.part_ml + 2 * p);
        ms[u] = ml.x;
        ls[u] = ml.y;
        os[u] = *(const float4*)(d.part_o + p * D + dim0);
        n = u + 1;
      }
    }
    float m_new = m_run;
#pragma unroll
    for (int u = 0; u < kWideBatch; ++u)
      if (u < n) m_new = fmaxf(m_new, ms[u]);
    const float m_use = finite_max(m_new);
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
    l_run *= alpha;
#pragma unroll
    for (int e = 0; e < 4; ++e) o_run[e] *= alpha;
#pragma unroll
    for (int u = 0; u < kWideBatch; ++u) {
      if (u < n) {
        const float w = __builtin_amdgcn_exp2f(ms[u] - m_use);
        l_run += w * ls[u];
        o_run[0] += w * os[u].x;
        o_run[1] += w * os[u].y;
        o_run[2] += w * os[u].z;
        o_run[3] += w * os[u].w;
      }
    }
    m_run = m_new;
  }
  if (lane == 0) {
    m_grp[grp] = m_run;
    l_grp[grp] = l_run;
  }
  o_grp[grp][lane] = float4{o_run[0], o_run[1], o_run[2], o_run[3]};
  __syncthreads();
  if (grp != 0) return;
  float M = m_grp[0];
#pragma unroll
  for (int q = 1; q < kWideGroups; ++q) M = fmaxf(M, m_grp[q]);
  float o[4] = {0.0f, 0.0f, 0.0f, 0.0f}, Ltot = 0.0f;
  const float m_use = finite_max(M);
#pragma unroll 8
  for (int q = 0; q < kWideGroups; ++q) {
    const float w = __builtin_amdgcn_exp2f(m_grp[q] - m_use);
    const float4 oq = o_grp[q][lane];
    o[0] += w * oq.x;
    o[1] += w * oq.y;
    o[2] += w * oq.z;
    o[3] += w * oq.w;
    Ltot += w * l_grp[q];
  }
  const float inv = (Ltot > 0.0f) ? (1.0f / Ltot) : 0.0f;
  half4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = Elem<BF16>::round(o[e] * inv);
  *(half4*)(a.o + b * a.osb + hq * a.osh + (int64_t)qi * a.osn + dim0) = v;
  if (a.lse != nullptr && chunk == 0 && lane == 0) {
    a.lse[((int64_t)b * a.hq + hq) * a.n + qi] =
        (m_use + __builtin_log2f(Ltot)) * 0.69314718055994530942f;
  }
}

template <bool BF16>
void launch_decode_typed(const DecArgs& d, const DecodePlan& pl, int head_dim, bool causal,
                         hipStream_t stream) {
  const dim3 grid((unsigned)((int64_t)pl.units * pl.splits));
#define FA_DEC(DD, C, M) \
  if (d.flags != nullptr)                                                                         \
    hipLaunchKernelGGL((fa_decode_kernel<DD, C, M, BF16, true>), grid, dim3(kThreads), 0, stream, d); \
  else                                                                                            \
    hipLaunchKernelGGL((fa_decode_kernel<DD, C, M, BF16, false>), grid, dim3(kThreads), 0, stream, d)
#define FA_DEC_M(DD, C)                            \
  if (d.f.mkeys != nullptr) { FA_DEC(DD, C, 2); }      \
  else if (d.f.mbits != nullptr) { FA_DEC(DD, C, 1); } \
  else { FA_DEC(DD, C, 0); }
  if (head_dim == 128) {
    if (causal) { FA_DEC_M(128, true); } else { FA_DEC_M(128, false); }
  } else {
    if (causal) { FA_DEC_M(64, true); } else { FA_DEC_M(64, false); }
  }
#undef FA_DEC_M
#undef FA_DEC
  if (pl.splits > 1 && d.flags == nullptr) {
    const bool wide = pl.splits * head_dim >= kWideCombineMin;
    const dim3 cgrid((unsigned)((int64_t)pl.units * pl.rows * (wide ? head_dim / 32 : 1)));
#define FA_CMB(DD)                                                                          \
  if (wide)                                                                                 \
    hipLaunchKernelGGL((fa_decode_combine_wide<DD, BF16>), cgrid, dim3(kCombineThreads), 0, \
                       stream, d);                                                          \
  else                                                                                      \
    hipLaunchKernelGGL((fa_decode_combine<DD, BF16>), cgrid, dim3(kCombineThreads), 0, stream, d)
    if (head_dim == 128) { FA_CMB(128); } else { FA_CMB(64); }
#undef FA_CMB
  }

}

}  // namespace

namespace {

__global__ void fa_clear_flags(uint64_t* flags, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) flags[i] = 0;
}

// A mark no other call of this process has used: a counter from a random
// start, so that what else the workspace may hold does not equal it either.
uint64_t fresh_mark() {
  static std::atomic<uint64_t> next{[] {
    // splitmix64 of the clock and this object's address
    uint64_t x = (uint64_t)std::chrono::steady_clock::now().time_since_epoch().count() +
                 0x9e3779b97f4a7c15ull * (uint64_t)(uintptr_t)&fa_clear_flags;
    x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
    x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
    return (x ^ (x >> 31)) | 1u;
  }()};
  return next.fetch_add(2, std::memory_order_relaxed);
}
constexpr uint64_t kCapturedMark = 2;  // calls under capture (fresh marks are odd)


}  // namespace

bool decode_eligible(const FwdArgs& a, int batch) {
  const bool decode = (int64_t)a.group * a.n <= kDecodeMaxRows;
  const int64_t prefill_items = (int64_t)batch * a.hq * ((a.n + 127) / 128);
  if (!decode && prefill_items > kSmallLaunchItems) return false;
  if (a.mbits != nullptr) {
    // The split-K kernel reads one batch's mask rows through a single 32-bit
    // buffer window (byte offsets up to this span); a call whose mask strides
    // span more runs on the prefill kernel, which reads the words through
    // 64-bit addresses.
    const int64_t words = ((int64_t)a.nk + 63) / 64;
    const int64_t span =
        ((int64_t)(a.hq - 1) * a.msh + (int64_t)(a.n - 1) * a.msq + words) * 8;
    if (span > (int64_t)INT32_MAX) return false;
  }
  // Key bytes: 32-bit offsets up to one tile past the last key.
  if (a.mkeys != nullptr && ((int64_t)a.nk + 64) * a.mksk > (int64_t)INT32_MAX) return false;
  return true;
}

namespace {

// How many workgroups share a unit's keys.  A workgroup (four waves, one tile
// of 32 keys each in flight) streams K and V at about 50 bytes/ns at head_dim
// 128 (16 KB per tile) and half that at 64, so few workgroups are slow and the
// split spreads a unit over CUs; the merge costs 1-3 us.  Timed on MI355X,
// bfloat16, us per call:
//  * few tiles run as one split: decode at head_dim 128 up to 15 (Hq=32 Hkv=8
//    385 keys 8.6 against 9.4 for 3 splits, 16 sequences 448 keys 9.4 and 10.4),
//    at 64 up to 20 (Hq=14 Hkv=2 512 keys 5.9 against 7.7 for 4 splits), 28 for
//    more than 64 units (8 x 12 heads 704 keys 7.7 and 9.4, 896 keys 8.6 and
//    9.7; 16 x 8 heads 918 keys 9.2 and 9.3, 1078 keys 10.0 and 9.8); row
//    blocks (32 columns, a longer merge) up to 36 at head_dim 64 and 28 at 128
//    (one head of 1024 rows d64 8.2 against 8.8; 8 heads 448 x 896 d128 14.1 and
//    14.6, 448 x 960 15.7 and 14.8), and at 64 up to 64 where they could only
//    be halved (4 heads of 1024 rows 9.6 against 10.3);
//  * a split has at least four tiles, one per wave; at head_dim 64, of fewer than
//    eight there are at most 16, or 8 where a unit is one row or 16 would not be
//    merged in the kernel (16 splits against one per eight tiles at 65-125 tiles:
//    Hq=14 Hkv=2 7.9-8.2 and 8.2-8.5, 4 sequences 8.1-8.3 and 8.3-8.8; 8 splits
//    against 16 at 44-64 tiles: 2 x 8 heads 8.1-8.4 and 8.9, one head level;
//    4097 keys 8.4 for 15 splits, 8.7 for 17, 9.0 for 32); row blocks eight
//    (one head of 1024 rows d128 16.1 -> 12.9, 4 heads 300 x 2000 29.6 -> 16.2);
//  * the workgroups fill whole rounds of CUs: rounding the split count up
//    put two workgroups on some CUs and one on others, and the launch took
//    as long as two (B=3 Hq=32 Hkv=8 9000 keys d128: 264 workgroups 31.7,
//    240 22.6; B=12 8192 keys 288 workgroups 92.5, 192 70.2).  Where one round
//    leaves more than a seventh of the CUs idle, two rounds' worth (two
//    workgroups of a CU run together) if that fills them better: the latter
//    480 workgroups 67.4, B=20 Hq=8 3000 keys d128 160 workgroups 48.2, 480
//    44.3.
constexpr int kDecMinTiles = 4, kMinTiles = 8;
constexpr int kBlockLongTiles = 64;
constexpr int kTargetWgs = 256;  // one workgroup per CU

// (`most`: splits the workspace has room for.)
int plan_splits(const DecodePlan& pl, int head_dim, int64_t most) {
  const bool blocks = pl.row_blocks > 1;
  const bool many = 4 * pl.units > kTargetWgs;  // fewer than four splits a unit in one round
  const int no_split =
      blocks ? (head_dim == 64 ? 36 : 28) : head_dim == 64 ? (many ? 28 : 20) : 15;
  if (pl.tiles <= no_split) return 1;
  int limit = pl.tiles / (blocks ? kMinTiles : kDecMinTiles);
  if (!blocks && head_dim == 64) {
    const bool one_row = pl.rows == 1;
    const int most_short = one_row || 16 * pl.units > kMergeFewWgs ? 8 : 16;
    limit = std::max(std::min(limit, most_short), (pl.tiles + (one_row ? 7 : 0)) / kMinTiles);
  }
  int splits = std::max(1, kTargetWgs / pl.units);
  if (blocks) {
    if (pl.tiles > kBlockLongTiles)  // one block per CU, a long range each: halve it
      splits = std::max(splits, std::min(2, (kTargetWgs + pl.units - 1) / pl.units));
    else if (head_dim == 64 && std::min<int64_t>(splits, most) < 4)
      splits = 1;
  } else {
    const int two = 2 * kTargetWgs / pl.units;
    if (7 * splits * pl.units < 6 * kTargetWgs && two * pl.units > 9 * splits * pl.units / 4)
      splits = two;
  }
  splits = std::min(std::min(splits, kMaxSplits), limit);
  return (int)std::max<int64_t>(1, std::min<int64_t>(splits, most));
}

}  // namespace

DecodePlan plan_decode(const FwdArgs& a, int batch, int head_dim, bool causal,
                       int64_t workspace_bytes) {
  DecodePlan pl;
  pl.total_rows = a.group * a.n;
  pl.rows = std::min(pl.total_rows, kDecodeMaxRows);
  pl.row_blocks = (pl.total_rows + kDecodeMaxRows - 1) / kDecodeMaxRows;
  pl.units = batch * (a.hq / a.group) * pl.row_blocks;
  // Keys any query row can see.
  int64_t nk_eff = a.nk;
  if (causal) nk_eff = std::min<int64_t>(a.nk, std::max<int64_t>(0, (int64_t)a.n + a.diag));
  pl.tiles = (int)((nk_eff + kDecTile - 1) / kDecTile);
  // One split's partials and its mark (merge in the split-K kernel).  A
  // workspace with room for fewer splits than the GPU wants gets those; one with
  // room for the partials alone, the combine kernel.
  const int64_t record = (int64_t)pl.units * pl.rows * (head_dim + 2) * 4;
  const int64_t mark = (int64_t)pl.units * 8;
  const int splits = plan_splits(pl, head_dim, workspace_bytes / record);
  pl.chunk_tiles = std::max(1, (pl.tiles + splits - 1) / splits);
  pl.splits = std::max(1, (pl.tiles + pl.chunk_tiles - 1) / pl.chunk_tiles);
  const int64_t partial_o = (int64_t)pl.splits * pl.rows * head_dim * 4;
  pl.merge_in_kernel =
      pl.splits > 1 && pl.splits <= kThreads && pl.splits * (record + mark) <= workspace_bytes;
  if (pl.row_blocks > 1)
    pl.merge_in_kernel = pl.merge_in_kernel && partial_o <= kMergeMaxBlockBytes &&
                         pl.splits <= kMergeMaxBlockSplits;
  else
    pl.merge_in_kernel = pl.merge_in_kernel && partial_o <= kMergeMaxBytes &&
                         (head_dim != 64 || pl.splits <= kMergeMaxSplits64 ||
                          (int64_t)pl.units * pl.splits <= kMergeFewWgs);
  pl.workspace_bytes =
      pl.splits > 1 ? pl.splits * (record + (pl.merge_in_kernel ? mark : 0)) : 0;
  return pl;
}

int launch_decode_forward(const FwdArgs& a, const DecodePlan& pl, int head_dim, bool causal,
                          void* workspace, hipStream_t stream) {
  DecArgs d;
  d.f = a;
  d.rows = pl.rows;
  d.total_rows = pl.total_rows;
  d.row_blocks = pl.row_blocks;
  d.splits = pl.splits;
  d.chunk_tiles = pl.chunk_tiles;
  d.tiles = pl.tiles;
  d.part_o = static_cast<float*>(workspace);
  d.part_ml = pl.splits > 1
                  ? d.part_o + (int64_t)pl.units * pl.splits * pl.rows * head_dim
                  : nullptr;
  d.flags = nullptr;
  d.mark = kCapturedMark;
  if (pl.merge_in_kernel) {
    d.flags = reinterpret_cast<uint64_t*>(d.part_ml + (int64_t)pl.units * pl.splits * pl.rows * 2);
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    const hipError_t e = hipStreamIsCapturing(stream, &capture);
    if (e != hipSuccess) (void)hipGetLastError();  // not this call's error
    if (e == hipSuccess && capture == hipStreamCaptureStatusNone) {
      d.mark = fresh_mark();
    } else {
      const int64_t n = (int64_t)pl.units * pl.splits;
      hipLaunchKernelGGL(fa_clear_flags, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream,
                         d.flags, n);
    }
  }
  if (a.bf16)
    launch_decode_typed<true>(d, pl, head_dim, causal, stream);
  else
    launch_decode_typed<false>(d, pl, head_dim, causal, stream);
  return 0;
}

}  // namespace fa
