// Paged causal GQA attention for gfx950: a window of L query tokens per
// sequence over its paged K/V (a prompt, a chunk of one, or a verify window).
//
// The reference masks a multi-token window explicitly (k_pos <= q_pos,
// runtime/layer_runner.py:166-177) over the concatenated pages.  Query token t
// of the window sits at position S - L + t and sees the S - L + t + 1 first
// tokens of its sequence.
//
// What bounds it: matrix work, 4 * NQ * D flops per (query, visible key).  The
// (query token, head of the group) pairs of one (sequence, kv head) segment are
// the rows of the products, so every head of a GQA group shares the K/V tiles;
// a workgroup of NW wavefronts takes 32 * NW consecutive rows and walks the
// 64-key tiles its last row sees.  Per tile and wavefront, on
// v_mfma_f32_32x32x16_bf16 with the wavefront's 32 rows as the N dimension:
//   scores^T[64 keys][32 rows] = K . Q^T      A = K rows (LDS), B = q (registers)
//   out^T[D dims][32 rows]    += V^T . P^T    A = V^T rows (LDS), B = P (registers)
// A lane holds one row's scores, so the softmax needs one exchange with lane
// l ^ 32 per tile and no LDS, and rescaling is one factor per lane.  The key
// rows of the score operand are permuted (key_of_row) so that the scores of a
// lane are, in order, the 8 consecutive keys its P^T operand needs.
//
// K tiles are token-major and V tiles transposed in the pool already, both in
// contiguous 64 * D-byte blocks of 32 tokens; they go straight into LDS
// (buffer_load ... lds, 1 KiB each), double-buffered, one barrier per tile,
// chunk-swizzled through the per-lane source offsets so that the operand reads
// spread over all banks (no conflicts counted).
//
// Per tile a wavefront needs 1,024 cycles of MFMA (D = 128) and about as many of
// exponentials and conversions.  So the scores run one tile ahead: the MFMAs of
// tile t + 1 interleave with the exponentials of tile t, and P.V of tile t with
// the maximum of tile t + 1.  What else it took, in a chunk of 2,011 queries over
// 6,007 tokens (32/8 heads, D = 128; every query its own row of the decode kernel:
// 5,520 us): eight wavefronts, scores and softmax in turn 220 us; loads issued
// between the MFMAs and pool blocks looked up 64 at a time, one per lane (a
// scalar lookup per tile cost 800 cycles of latency) 203 us; four wavefronts, so
// that two workgroups per CU do not wait at each other's barriers, 198 us; tiles
// on the diagonal in a loop of their own, which frees the first one of their
// registers, 187 us; long and short row tiles paired on the CUs 182 us (176 on
// another box, 940 TFLOP/s; a large bf16 library product reaches 1,290 here).
//
// Windows whose rows do not fill the chip are split over keys as well; the
// splits leave (m, l, o) in fp32 and gqa_prefill_combine_kernel merges them.
#include "common.h"

#include <cfloat>
#include <type_traits>

namespace voom {
namespace {

constexpr int kBlk = 32;        // tokens of a K/V block in the pool
constexpr int kKeys = 64;       // keys per tile
constexpr int kRows = 32;       // rows of a wavefront
constexpr int NW = 4;           // wavefronts of a workgroup
constexpr int kAhead = 4;       // operand reads ahead of the MFMAs

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

struct PrefillArgs {
  const uint16_t* q;       // [B, NQ, L, D]
  const uint16_t* k_pool;
  const uint16_t* v_pool;
  const int32_t* table;    // [B, max_pages]
  uint16_t* out;           // [B, L, NQ, D]
  float* part_o;           // [B * NKV * R, splits, D]
  float* part_ml;          // [B * NKV * R, splits, 2]
  int NQ, NKV, G, L, S, max_pages, pt_shift, num_slots;
  int R;          // rows of a segment: L * G, (token, head) with the head fastest
  int row_tiles;  // workgroups along R
  int splits;     // key splits
  int work;       // B * NKV * row_tiles * splits
  int per_xcd;    // work items per XCD
  int xcd_cus;    // CUs per XCD
  // |softmax scale| in log2 units, > 0.  The sign is applied to q (q_flip =
  // 0x80008000), a scale of 0 by clearing q but for infinities and NaN (q_zero,
  // scale 1).
  float scale;
  uint32_t q_flip;
  bool q_zero;
};

// Key (0..31 of a block) that row r of the score tile holds: lane half h then
// has keys 8h..8h+7 in its first eight accumulators and 16+8h.. in the others.
__device__ __forceinline__ int key_of_row(int r) {
  return 16 * (r >> 4) + 8 * ((r >> 2) & 1) + 4 * ((r >> 3) & 1) + (r & 3);
}

// Chunk c (16 bytes) of K row r sits at c ^ k_swizzle(r): 16 consecutive keys
// then read one chunk from 16 different 16-byte columns.
template <int D>
__device__ __forceinline__ int k_swizzle(int r) {
  return D == 128 ? (r & 15) : ((r >> 1) & 7);
}

template <int D>
__global__ __launch_bounds__(NW * kWave) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gqa_prefill_kernel(PrefillArgs a) {
  constexpr int kBlkElems = kBlk * D;          // elements of one K or V block
  constexpr int kPieces = kBlkElems / 512;     // 1 KiB loads per block
  constexpr int kLoads = 4 * kPieces / NW;     // loads per wavefront and tile
  constexpr int kCpr = D / 8;                  // 16-byte chunks of a K row
  constexpr int KS = D / 16;                   // k-steps of the scores
  constexpr int DT = D / 32;                   // dim tiles of out^T
  // masks of __builtin_amdgcn_sched_group_barrier
  constexpr int kValu = 0x002, kMfma = 0x008, kVmemRead = 0x020, kDsRead = 0x100, kTrans = 0x400;
  static_assert(kLoads * NW == 4 * kPieces, "loads split evenly over the wavefronts");
  // K block 0, K block 1, V^T block 0, V^T block 1.  Two distinct objects, so
  // that reads of one provably miss the other's pending direct-to-LDS loads.
  __shared__ __attribute__((aligned(1024))) uint16_t tile_a[4 * kBlkElems];
  __shared__ __attribute__((aligned(1024))) uint16_t tile_b[4 * kBlkElems];

  // Consecutive work items of one XCD are row tiles of the same segment (its
  // K/V stay in that XCD's L2), the longest first.  Where all of them run at
  // once, at most two per CU, the second of a CU is as short as the first is long.
  const int bid = static_cast<int>(blockIdx.x);
  int at = bid >> 3;
  if (at >= a.xcd_cus && a.per_xcd <= 2 * a.xcd_cus) at = a.per_xcd - 1 - (at - a.xcd_cus);
  const int wk = (bid & 7) * a.per_xcd + at;
  if (wk >= a.work) return;
  const int per_seg = a.row_tiles * a.splits;
  const int seg = wk / per_seg;
  const int in_seg = wk - seg * per_seg;
  const int rt = a.row_tiles - 1 - in_seg / a.splits;
  const int split = in_seg % a.splits;
  const int b = seg / a.NKV;
  const int kvh = seg - b * a.NKV;

  const int lane = threadIdx.x & (kWave - 1);
  const int w = uniform(threadIdx.x / kWave) & (NW - 1);
  const int l32 = lane & 31;
  const int lh = lane >> 5;

  // This lane's row (rows past the segment repeat its last one and are not
  // stored), the keys it sees, and the fewest and most of the wavefront.
  const int row = rt * (NW * kRows) + w * kRows + l32;
  const bool row_ok = row < a.R;
  const int rc = row_ok ? row : a.R - 1;
  const int tok = rc / a.G;
  const int head = kvh * a.G + (rc - tok * a.G);
  const int vis = a.S - a.L + tok + 1;
  const int vis_lo = uniform(vis);
  const int vis_hi = __builtin_amdgcn_readlane(vis, 31);
  int last = rt * (NW * kRows) + NW * kRows - 1;
  last = last < a.R ? last : a.R - 1;
  const int n_tiles = (a.S - a.L + last / a.G + 1 + kKeys - 1) / kKeys;
  const int t_lo = static_cast<int>(static_cast<long long>(split) * n_tiles / a.splits);
  const int t_hi = static_cast<int>(static_cast<long long>(split + 1) * n_tiles / a.splits);

  // Q^T operand: lane (row l32, half lh) holds q[16 s + 8 lh .. + 8]
  u32x4 qop[KS];
  auto load_q = [&]() {
    const uint16_t* qh = a.q + ((static_cast<size_t>(b) * a.NQ + head) * a.L + tok) * D + 8 * lh;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      qop[s] = *reinterpret_cast<const u32x4*>(qh + 16 * s);
#pragma unroll
      for (int i = 0; i < 4; ++i) qop[s][i] ^= a.q_flip;
    }
    if (a.q_zero) {
#pragma unroll
      for (int s = 0; s < KS; ++s) {
#pragma unroll
        for (int i = 0; i < 4; ++i) qop[s][i] = nan_bf16(qop[s][i]);
      }
    }
  };

  // Pool blocks (K and V alike, in units of 32 tokens of one kv head) of the
  // sequence's 32-token blocks win .. win + 63, one per lane; blocks past the
  // last token repeat it (their keys are masked).
  const int32_t* trow = a.table + static_cast<size_t>(b) * a.max_pages;
  const int sub_shift = a.pt_shift - 5;
  const int last_blk = (a.S - 1) / kBlk;
  int win = -kWave;
  int blocks = 0;
  auto fill_window = [&](int bi) {
    win = bi;
    const int mine = bi + lane < last_blk ? bi + lane : last_blk;
    const int page = mine >> sub_shift;
    int slot = trow[page];
    if (static_cast<unsigned>(slot) >= static_cast<unsigned>(a.num_slots)) slot = 0;
    blocks = ((slot * a.NKV + kvh) << sub_shift) + (mine - (page << sub_shift));
    wait_vmem_all();  // here, not at the readlanes below on every tile
  };
  // Stage t holds K of tile t + 1 (the scores run one tile ahead of P.V) and
  // V^T of tile t.  Its pieces of 1 KiB, 4 * kPieces of them, go piece p to
  // wavefront p % NW.  stage_blocks looks the pool blocks up (V's are K's of the
  // stage before), load_piece issues load i of this wavefront.
  int kblk0 = 0, kblk1 = 0, vblk0 = 0, vblk1 = 0;
  auto stage_blocks = [&](int t) {
    const int bi = 2 * t + 2;
    if (bi >= win + kWave) fill_window(bi);  // bi is even: so is the window's start
    vblk0 = kblk0;
    vblk1 = kblk1;
    kblk0 = __builtin_amdgcn_readlane(blocks, bi - win);
    kblk1 = __builtin_amdgcn_readlane(blocks, bi - win + 1);
  };
  auto load_piece = [&](int i, uint16_t* dst) {
    const int p = w + NW * i;
    const int blk = p / kPieces;
    const int sub = p % kPieces;
    const bool is_v = blk >= 2;
    const int j = blk & 1;
    // (sums, not a choice between variables, which would become one of addresses)
    const unsigned src = uniform((is_v ? vblk0 + 0 : kblk0 + 0) * (1 - j) +
                                 (is_v ? vblk1 + 0 : kblk1 + 0) * j);
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>((is_v ? a.v_pool : a.k_pool) + static_cast<size_t>(src) * kBlkElems),
        static_cast<short>(0), kBlkElems * 2, 0x00020000);
    const int krow = sub * (kWave / kCpr) + lane / kCpr;
    const int ksrc = krow * (D * 2) + 16 * ((lane % kCpr) ^ k_swizzle<D>(krow));
    const int vrow = sub * 16 + (lane >> 2);
    const int vsrc = vrow * (kBlk * 2) + 16 * ((lane & 3) ^ ((lane >> 4) & 3));
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)(dst + p * 512), 16, is_v ? vsrc : ksrc,
                                             0, 0, 0);
  };
  auto load_stage = [&](int t, uint16_t* dst) {
    stage_blocks(t);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) load_piece(i, dst);
  };

  // Per-lane LDS byte addresses of the operands.  K: row key_of_row(l32),
  // chunk 2 s + lh.  V^T: dim row 32 dt + l32, chunk 2 ks + lh of its block.
  const int key = key_of_row(l32);
  const int k_lane = key * (D * 2) + 16 * (lh ^ k_swizzle<D>(key));
  int v_lane[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
    v_lane[ks] = l32 * (kBlk * 2) + 16 * ((2 * ks + lh) ^ ((l32 >> 2) & 3));

  f32x16 acc[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) acc[d] = f32x16{};
  // Reference maximum, log2 units; the same in both halves.  Never -inf: keys of
  // score -inf (masked or not) then have P = 0 also where nothing else came before.
  float m = -FLT_MAX;
  float l = 0.f;        // over this lane's keys

  typedef f32x16 Scores[2];  // 32-key blocks of a tile; accumulator i of block
                             // j: key 32 j + 16 (i / 8) + 8 lh + i % 8
  // Keys of tile t that this lane's row does not see score -inf.
  auto mask_scores = [&](int t, Scores& sc) {
    const int lim = vis - t * kKeys - 8 * lh;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        sc[j][i] = 32 * j + 16 * (i >> 3) + (i & 7) < lim ? sc[j][i] : -INFINITY;
    }
  };
  auto max_of = [&](const Scores& sc) {
    float mx = fmaxf(sc[0][0], sc[1][0]);
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(fmaxf(mx, sc[0][i]), sc[1][i]);
    return mx;
  };
  // Raises the reference maxima to a tile's (mx: this lane's, in raw scores)
  // before its P is formed.  The asm keeps the rescaling inside the branch.
  auto raise = [&](float mx) {
    mx = fmaxf(mx, __shfl_xor(mx, 32)) * a.scale;
    if (__builtin_amdgcn_ballot_w64(mx > m) == 0) return;
    const float mn = fmaxf(m, mx);
    float alpha = fast_exp2(m - mn);
    asm volatile("" : "+v"(alpha));
    m = mn;
    l *= alpha;
#pragma unroll
    for (int d = 0; d < DT; ++d) acc[d] *= alpha;
  };
  // K operand i of the scores (i = 2 s + j: k-step s, block j), V operand i of
  // P.V (i = (2 j + ks) * DT + d)
  auto read_k = [&](const uint16_t* tile, int i) {
    return *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(tile) +
                                           (i & 1) * (kBlkElems * 2) + (k_lane ^ (32 * (i >> 1))));
  };
  auto read_v = [&](const uint16_t* tile, int i) {
    const int j = i / (2 * DT), ks = (i / DT) & 1, d = i % DT;
    return *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(tile) +
                                           (2 + j) * (kBlkElems * 2) + d * (32 * kBlk * 2) +
                                           v_lane[ks]);
  };

  auto first_scores = [&](const uint16_t* tile, Scores& sc) {
#pragma unroll
    for (int j = 0; j < 2; ++j) sc[j] = f32x16{};
#pragma unroll
    for (int i = 0; i < 2 * KS; ++i) {
      sc[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          __builtin_bit_cast(bf16x8, read_k(tile, i)), __builtin_bit_cast(bf16x8, qop[i >> 1]),
          sc[i & 1], 0, 0, 0);
    }
  };
  // Bits of the V operand's dwords (16-key step jk of tile t) that hold tokens
  // of the sequence.
  auto tail_mask = [&](int t, int jk, uint32_t (&keep)[4]) {
    const int lim = a.S - t * kKeys - 16 * jk - 8 * lh;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      keep[e] = (2 * e < lim ? 0xffffu : 0u) | (2 * e + 1 < lim ? 0xffff0000u : 0u);
  };
  // One of P's pairs, into the operand layout; the normaliser sums the bf16
  // weights that the MFMA consumes.
  auto form_p = [&](int e, const Scores& sc, float mref, u32x4 (&pk)[2][2]) {
    const int j = e >> 3, n = 2 * (e & 7);
    const uint32_t p2 = pack_bf16x2(fast_exp2(__builtin_fmaf(sc[j][n], a.scale, -mref)),
                                    fast_exp2(__builtin_fmaf(sc[j][n + 1], a.scale, -mref)));
    pk[j][n >> 3][(n & 7) >> 1] = p2;
    l = sum_bf16x2(p2, l);
  };

  // Tile t where every row of the wavefront sees all of tiles t and t + 1:
  // scores of tile t + 1 on the matrix cores while the vector units form P of
  // tile t, then P.V of tile t while they find the maximum of tile t + 1.  The
  // next stage's loads go out one by one between the MFMAs.
  auto whole_tile = [&](const uint16_t* tile, uint16_t* next, const Scores& sc, Scores& nx) {
    const float mref = m;
    u32x4 pk[2][2];
    u32x4 ring[kAhead];
#pragma unroll
    for (int j = 0; j < 2; ++j) nx[j] = f32x16{};
#pragma unroll
    for (int i = 0; i < kAhead; ++i) ring[i] = read_k(tile, i);
    __builtin_amdgcn_sched_group_barrier(kDsRead, kAhead, 0);
#pragma unroll
    for (int i = 0; i < 2 * KS; ++i) {
      nx[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          __builtin_bit_cast(bf16x8, ring[i % kAhead]), __builtin_bit_cast(bf16x8, qop[i >> 1]),
          nx[i & 1], 0, 0, 0);
      __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
      if (i + kAhead < 2 * KS) {
        ring[i % kAhead] = read_k(tile, i + kAhead);
        __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 0);
      }
      if (i * kLoads / (2 * KS) != (i + 1) * kLoads / (2 * KS)) {
        load_piece(i * kLoads / (2 * KS), next);
        __builtin_amdgcn_sched_group_barrier(kVmemRead, 1, 0);
      }
#pragma unroll
      for (int e = i * 16 / (2 * KS); e < (i + 1) * 16 / (2 * KS); ++e) {
        form_p(e, sc, mref, pk);
        __builtin_amdgcn_sched_group_barrier(kValu, 2, 0);
        __builtin_amdgcn_sched_group_barrier(kTrans, 2, 0);
        __builtin_amdgcn_sched_group_barrier(kValu, 2, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kAhead; ++i) ring[i] = read_v(tile, i);
    __builtin_amdgcn_sched_group_barrier(kDsRead, kAhead, 1);
    float mx = fmaxf(nx[0][0], nx[1][0]);
#pragma unroll
    for (int i = 0; i < 4 * DT; ++i) {
      const int j = i / (2 * DT), ks = (i / DT) & 1, d = i % DT;
      acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ring[i % kAhead]),
                                                       __builtin_bit_cast(bf16x8, pk[j][ks]),
                                                       acc[d], 0, 0, 0);
      __builtin_amdgcn_sched_group_barrier(kMfma, 1, 1);
      if (i + kAhead < 4 * DT) {
        ring[i % kAhead] = read_v(tile, i + kAhead);
        __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 1);
      }
#pragma unroll
      for (int e = i * 16 / (4 * DT); e < (i + 1) * 16 / (4 * DT); ++e) {
        if (e == 0) continue;
        mx = fmaxf(fmaxf(mx, nx[0][e]), nx[1][e]);
        __builtin_amdgcn_sched_group_barrier(kValu, 1, 1);
      }
    }
    raise(mx);
  };

  // Any tile t that some row of the wavefront sees: its scores are in sc, which
  // then takes those of tile t + 1 if a row sees that too.
  auto edge_tile = [&](int t, const uint16_t* tile, Scores& sc) {
    const float mref = m;
    u32x4 pk[2][2];
#pragma unroll
    for (int e = 0; e < 16; ++e) form_p(e, sc, mref, pk);
    // Tokens past the sequence's end are garbage and are cut out of V^T.  Keys
    // past a row's own position have P = 0 in that row, but 0 times a NaN or an
    // infinity is NaN: `finite` ends up with a zero half if V holds one.
    u16x2 finite = {0xffff, 0xffff};
#pragma unroll
    for (int jk = 0; jk < 4; ++jk) {
      uint32_t keep[4];
      tail_mask(t, jk, keep);
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        const u32x4 vv = read_v(tile, jk * DT + d);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          finite = __builtin_elementwise_min(
              finite, __builtin_bit_cast(u16x2, ~(vv[e] & keep[e]) & 0x7f807f80u));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // read V^T again below instead of holding all of it across the branch
    asm volatile("" ::: "memory");
    if (__builtin_amdgcn_ballot_w64(finite[0] == 0 || finite[1] == 0) == 0) {
#pragma unroll
      for (int jk = 0; jk < 4; ++jk) {
        uint32_t keep[4];
        tail_mask(t, jk, keep);
#pragma unroll
        for (int d = 0; d < DT; ++d) {
          u32x4 vv = read_v(tile, jk * DT + d);
#pragma unroll
          for (int e = 0; e < 4; ++e) vv[e] &= keep[e];
          acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              __builtin_bit_cast(bf16x8, vv), __builtin_bit_cast(bf16x8, pk[jk >> 1][jk & 1]),
              acc[d], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      // Key by key: V^T with one key's column alone times P^T, added only to
      // the rows that see the key.
#pragma unroll
      for (int jk = 0; jk < 4; ++jk) {
#pragma unroll 1
        for (int k = 0; k < 16; ++k) {
          const int kt = t * kKeys + 16 * jk + k;
          if (kt >= a.S) break;
          const bool sees = kt < vis;
          const int slot = lh == (k >> 3) ? (k & 7) : -1;
#pragma unroll
          for (int d = 0; d < DT; ++d) {
            u32x4 vv = read_v(tile, jk * DT + d);
#pragma unroll
            for (int e = 0; e < 4; ++e)
              vv[e] &= (slot == 2 * e ? 0xffffu : 0u) | (slot == 2 * e + 1 ? 0xffff0000u : 0u);
            const f32x16 one = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                __builtin_bit_cast(bf16x8, vv), __builtin_bit_cast(bf16x8, pk[jk >> 1][jk & 1]),
                f32x16{}, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[d][e] += sees ? one[e] : 0.f;
            __builtin_amdgcn_sched_barrier(0);  // one product in registers at a time
          }
        }
      }
    }
    if (t + 1 < t_hi && (t + 1) * kKeys < vis_hi) {
      first_scores(tile, sc);
      mask_scores(t + 1, sc);
      raise(max_of(sc));
    }
  };

  Scores sc_a, sc_b;
  // Stage t has landed for every wavefront and the other buffer is no longer read.
  auto landed = [&]() {
    wait_vmem_all();
    lds_barrier();
  };
  if (t_lo < t_hi) {
    // K of the first tile, then (in flight while it is scored) the first stage
    stage_blocks(t_lo - 1);
#pragma unroll
    for (int i = 0; i < kLoads / 2; ++i) load_piece(i, tile_b);
    load_q();
    load_stage(t_lo, tile_a);
    static_assert(kLoads == 8 || kLoads == 4, "the wait below counts the first stage's loads");
    // gfx9 encoding: vmcnt kLoads, expcnt 7, lgkmcnt 15
    if constexpr (kLoads == 8) __builtin_amdgcn_s_waitcnt(0x0F78);
    else __builtin_amdgcn_s_waitcnt(0x0F74);
    lds_barrier();
    first_scores(tile_b, sc_a);
    mask_scores(t_lo, sc_a);
    raise(max_of(sc_a));
  }
  // Pairs of tiles that every row of the wavefront sees whole, the tile after
  // them included (its scores run ahead), then the rest.  Wavefronts leave the
  // first loop at different tiles; all pass one barrier per tile.
  int t = t_lo;
  for (; t + 2 < t_hi && (t + 3) * kKeys <= vis_lo; t += 2) {
    landed();
    stage_blocks(t + 1);
    whole_tile(tile_a, tile_b, sc_a, sc_b);
    landed();
    stage_blocks(t + 2);
    whole_tile(tile_b, tile_a, sc_b, sc_a);
  }
  for (; t < t_hi; t += 2) {
    landed();
    if (t + 1 < t_hi) load_stage(t + 1, tile_b);
    if (t * kKeys < vis_hi) edge_tile(t, tile_a, sc_a);
    if (t + 1 >= t_hi) break;
    landed();
    if (t + 2 < t_hi) load_stage(t + 2, tile_a);
    if ((t + 1) * kKeys < vis_hi) edge_tile(t + 1, tile_b, sc_a);
  }

  const float lt = l + __shfl_xor(l, 32);
  if (!row_ok) return;
  if (a.splits == 1) {
    const float inv = 1.f / lt;
    uint16_t* o = a.out + ((static_cast<size_t>(b) * a.L + tok) * a.NQ + head) * D + 4 * lh;
#pragma unroll
    for (int d = 0; d < DT; ++d) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        *reinterpret_cast<u32x2*>(o + 32 * d + 8 * i) =
            u32x2{pack_bf16x2(acc[d][4 * i] * inv, acc[d][4 * i + 1] * inv),
                  pack_bf16x2(acc[d][4 * i + 2] * inv, acc[d][4 * i + 3] * inv)};
      }
    }
    return;
  }
  const size_t p = (static_cast<size_t>(seg) * a.R + row) * a.splits + split;
  float* o = a.part_o + p * D + 4 * lh;
#pragma unroll
  for (int d = 0; d < DT; ++d) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      *reinterpret_cast<f32x4*>(o + 32 * d + 8 * i) =
          f32x4{acc[d][4 * i], acc[d][4 * i + 1], acc[d][4 * i + 2], acc[d][4 * i + 3]};
    }
  }
  if (lh == 0) {
    a.part_ml[p * 2 + 0] = m;
    a.part_ml[p * 2 + 1] = lt;
  }
}

// One wavefront per row: merges its key splits (at most 64) into the output.
constexpr int kMaxSplits = 64;
constexpr int kCombineWaves = 4;

template <int D>
__global__ __launch_bounds__(kCombineWaves * kWave) void gqa_prefill_combine_kernel(PrefillArgs a,
                                                                                    int rows) {
  constexpr int DPL = D / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int task = blockIdx.x * kCombineWaves + uniform(threadIdx.x / kWave);
  if (task >= rows) return;
  const int seg = task / a.R;
  const int row = task - seg * a.R;
  const int b = seg / a.NKV;
  const int kvh = seg - b * a.NKV;
  const int tok = row / a.G;
  const int head = kvh * a.G + (row - tok * a.G);
  const size_t p0 = static_cast<size_t>(task) * a.splits;
  const float2* ml2 = reinterpret_cast<const float2*>(a.part_ml);
  const bool live = lane < a.splits;
  const float2 ml = ml2[p0 + (live ? lane : 0)];
  const float M = wave_max_uniform(live ? ml.x : -INFINITY);
  // (a split that holds no visible key of the row left m = -FLT_MAX, l = 0)
  const float wt = live ? fast_exp2(ml.x - M) : 0.f;
  const float inv = 1.f / wave_sum_uniform(live ? ml.y * wt : 0.f);
  float acc[DPL] = {};
  const float* po = a.part_o + p0 * D + lane * DPL;
  for (int s0 = 0; s0 < a.splits; s0 += 8) {
    float v[8][DPL];  // eight rows in flight
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int s = s0 + u < a.splits ? s0 + u : a.splits - 1;
#pragma unroll
      for (int d = 0; d < DPL; ++d) v[u][d] = po[static_cast<size_t>(s) * D + d];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (s0 + u >= a.splits) break;
      const float ws = __builtin_bit_cast(
          float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wt), s0 + u));
#pragma unroll
      for (int d = 0; d < DPL; ++d) acc[d] += v[u][d] * ws;
    }
  }
  uint16_t* o = a.out + ((static_cast<size_t>(b) * a.L + tok) * a.NQ + head) * D + lane * DPL;
#pragma unroll
  for (int d = 0; d < DPL; ++d) o[d] = f2bf(acc[d] * inv);
}

// How a window is cut: row tiles and key splits.
struct PrefillPlan {
  int row_tiles, splits;
};

// Row tiles that leave CUs idle are split over keys (key_splits), with at least
// four 64-key tiles each.  Two workgroups per CU from the start are slower (a
// split's fixed cost: 4 queries over 16,384 tokens, 32/8 heads: 39 against 30 us;
// 1,024 over 1,024: 38 against 28 us); from one per CU on, splitting no longer
// gains (2,011 over 6,007: 204 against 183 us).  Two tiles per split win at 512
// over 512 with 9/3 heads of 64 (13.2 against 14.5 us) and lose at 2 over 4,000
// (19.8 against 16.4 us).
PrefillPlan plan_prefill(int B, int NKV, int G, int L, int S) {
  const long long R = static_cast<long long>(L) * G;
  const long long segs = static_cast<long long>(B) * NKV;
  PrefillPlan p;
  p.row_tiles = static_cast<int>((R + NW * kRows - 1) / (NW * kRows));
  const long long wgs = segs * p.row_tiles;
  const int tiles = (S + kKeys - 1) / kKeys;
  long long s = key_splits(wgs, device_cu_count());
  if (s > tiles / 4) s = tiles / 4;
  if (s > kMaxSplits) s = kMaxSplits;
  p.splits = s < 1 ? 1 : static_cast<int>(s);
  return p;
}

size_t o_bytes(const PrefillPlan& p, long long rows, int D) {
  return (static_cast<size_t>(rows) * p.splits * D * sizeof(float) + 255) & ~size_t(255);
}

bool prefill_shape_ok(int batch, int num_q_heads, int num_kv_heads, int head_dim, int window,
                      int seq_len) {
  return batch > 0 && num_kv_heads > 0 && num_q_heads > 0 && num_q_heads % num_kv_heads == 0 &&
         num_q_heads / num_kv_heads <= 16 && (head_dim == 64 || head_dim == 128) && window > 0 &&
         window <= seq_len && seq_len < (1 << 30) &&
         static_cast<long long>(batch) * num_q_heads * window < (1LL << 30);
}

}  // namespace
}  // namespace voom

using namespace voom;

extern "C" size_t voom_paged_gqa_prefill_workspace_bytes(int batch, int num_q_heads,
                                                         int num_kv_heads, int head_dim,
                                                         int window, int seq_len) {
  if (!prefill_shape_ok(batch, num_q_heads, num_kv_heads, head_dim, window, seq_len)) return 0;
  const int G = num_q_heads / num_kv_heads;
  const PrefillPlan p = plan_prefill(batch, num_kv_heads, G, window, seq_len);
  if (p.splits == 1) return 0;
  const long long rows = static_cast<long long>(batch) * num_q_heads * window;
  return o_bytes(p, rows, head_dim) + static_cast<size_t>(rows) * p.splits * 2 * sizeof(float);
}

extern "C" int voom_paged_gqa_prefill(const void* q, const void* k_pool, const void* v_pool,
                                      const int32_t* block_table, void* out, void* workspace,
                                      size_t ws_bytes, int batch, int num_q_heads,
                                      int num_kv_heads, int head_dim, int page_tokens,
                                      int max_pages, int num_slots, int window, int seq_len,
                                      float scale, hipStream_t stream) {
  const char* who = "paged_gqa_prefill";
  VOOM_REQUIRE(q && k_pool && v_pool && block_table && out, "%s: null pointer argument", who);
  VOOM_REQUIRE(num_slots > 0, "%s: empty page pool", who);
  VOOM_REQUIRE(prefill_shape_ok(batch, num_q_heads, num_kv_heads, head_dim, window, seq_len),
               "%s: unsupported geometry (batch %d, heads %d/%d, head_dim %d, window %d of %d)", who,
               batch, num_q_heads, num_kv_heads, head_dim, window, seq_len);
  VOOM_REQUIRE(is_pow2(page_tokens) && page_tokens >= 32 && page_tokens <= 4096,
               "%s: page_tokens %d must be a power of two in [32, 4096]", who, page_tokens);
  VOOM_REQUIRE(max_pages > 0 && static_cast<long long>(max_pages) * page_tokens >= seq_len,
               "%s: %d tokens do not fit the block table", who, seq_len);
  VOOM_REQUIRE(reinterpret_cast<uintptr_t>(q) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(k_pool) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(v_pool) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(out) % 8 == 0,
               "%s: q and pools must be 16-byte aligned", who);
  const int G = num_q_heads / num_kv_heads;
  const PrefillPlan p = plan_prefill(batch, num_kv_heads, G, window, seq_len);
  const long long rows = static_cast<long long>(batch) * num_q_heads * window;
  const size_t need = voom_paged_gqa_prefill_workspace_bytes(batch, num_q_heads, num_kv_heads,
                                                             head_dim, window, seq_len);
  VOOM_REQUIRE(need == 0 || (workspace != nullptr && ws_bytes >= need &&
                             reinterpret_cast<uintptr_t>(workspace) % 16 == 0),
               "%s: workspace %zu bytes < required %zu (16-byte aligned)", who, ws_bytes, need);
  PrefillArgs a;
  a.q = static_cast<const uint16_t*>(q);
  a.k_pool = static_cast<const uint16_t*>(k_pool);
  a.v_pool = static_cast<const uint16_t*>(v_pool);
  a.table = block_table;
  a.out = static_cast<uint16_t*>(out);
  a.part_o = static_cast<float*>(workspace);
  a.part_ml = need ? reinterpret_cast<float*>(static_cast<char*>(workspace) +
                                              o_bytes(p, rows, head_dim))
                   : nullptr;
  a.NQ = num_q_heads;
  a.NKV = num_kv_heads;
  a.G = G;
  a.L = window;
  a.S = seq_len;
  a.max_pages = max_pages;
  a.pt_shift = ilog2(page_tokens);
  a.num_slots = num_slots;
  a.R = window * G;
  a.row_tiles = p.row_tiles;
  a.splits = p.splits;
  a.work = batch * num_kv_heads * p.row_tiles * p.splits;
  a.per_xcd = (a.work + 7) / 8;
  a.xcd_cus = device_cu_count() / 8;
  a.scale = scale == 0.f ? 1.f : fabsf(scale) * 1.4426950408889634f;
  a.q_zero = scale == 0.f;
  a.q_flip = scale < 0.f ? 0x80008000u : 0u;
  const dim3 grid(static_cast<unsigned>(8 * a.per_xcd));
  const dim3 block(NW * kWave);
  if (head_dim == 128) hipLaunchKernelGGL(gqa_prefill_kernel<128>, grid, block, 0, stream, a);
  else hipLaunchKernelGGL(gqa_prefill_kernel<64>, grid, block, 0, stream, a);
  int rc = VOOM_LAUNCH_CHECK("paged_gqa_prefill: kernel launch");
  if (rc || p.splits == 1) return rc;
  const dim3 cgrid(static_cast<unsigned>((rows + kCombineWaves - 1) / kCombineWaves));
  const dim3 cblock(kCombineWaves * kWave);
  if (head_dim == 128)
    hipLaunchKernelGGL(gqa_prefill_combine_kernel<128>, cgrid, cblock, 0, stream, a,
                       static_cast<int>(rows));
  else
    hipLaunchKernelGGL(gqa_prefill_combine_kernel<64>, cgrid, cblock, 0, stream, a,
                       static_cast<int>(rows));
  return VOOM_LAUNCH_CHECK("paged_gqa_prefill: combine launch");
}
