// Position-free paged attention for gfx950.
//
// Restates the reference's position_free_paged_attention (runtime/
// pic_attention.py:22-232): keys are stored *before* RoPE in physical pages
// [pages, NKV, BLOCK, D] (V in the same layout), a block table maps the
// logical sequence to pages (a page id may repeat: that is the sharing
// primitive), and every key is rotated at its logical position while the
// attention runs.  Per the reference:
//   q      [B, NQ, TQ, D]  already rotated, element type T (bf16, fp16, fp32)
//   key k  rotated with cos/sin tables [max_pos, D/2] (fp32 or T; NeoX
//          rotate-half) in fp32 and rounded to T before the dot product
//          (:81-90)
//   mask   a key attends iff k_positions[k] <= q_positions[tq]     (:57-58)
//   out    softmax(q.k * scale) . v, zeros when no key is visible   (:117-128)
// Like the Metal kernel, any number of queries and any GQA group is served.
//
// Two attention kernels leave split partials (m, l, o) that pf_reduce_kernel
// merges:
//   pf_attention_kernel  bf16 and fp16 pages, D in {64, 128}: MFMA.  Segments are
//                        (batch row, kv head); 16 (head, query) columns of a
//                        segment form the N dimension of one MFMA tile, so each
//                        key byte is read once for all of them.
//   pf_generic_kernel    fp32 pages and every other head dim (any multiple of
//                        32 up to 256): fp32 VALU over LDS-staged 32-key
//                        blocks, no rounding of P.
// A segment with more columns than one pass holds (16 for the MFMA kernel,
// 4096 / D for the generic one) runs as several column passes.  The passes of
// one piece of work are launched next to each other on the same XCD, so the
// second pass reads the pages from that XCD's L2.
// Many columns over 16-bit pages take a route of their own (pf_stage_kernel,
// pf_window_kernel, below), from where window_pays says.
//
// MFMA kernel, per 32-key block a wavefront:
//   - looks up the 32 page rows and positions (one key per lane),
//   - loads its K rows as MFMA A operands (16 bytes per lane per k-step),
//     rotates them in registers -- dims d and d + D/2 sit in k-steps s and
//     s + D/64 of the same lane -- and rounds them to the element type,
//   - scores^T[key][column] = K_rot . Q^T with v_mfma_f32_16x16x32_{bf16,f16},
//   - stages the 32 V rows in its own LDS slice and reads V^T operands back
//     with ds_read_b64_tr_b16, so out^T += V^T . P^T needs no V^T storage.
// The two 16-key score tiles leave lane (column j, group g) holding keys
// 4g + r and 16 + 4g + r; the transposed V reads address exactly those rows,
// so P^T is used straight from the score registers.
#include "common.h"

#include <float.h>
#include <limits.h>

namespace voom {
namespace {

constexpr int kKeys = 32;  // keys per block
constexpr int kCols = 16;  // MFMA N: (head, query) columns of one pass
constexpr float kLog2e = 1.4426950408889634f;

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;

// ---- element types (the VOOM_DTYPE_* codes) --------------------------------
struct EBf16 {
  typedef uint16_t raw;
  __device__ static float load(const raw* p) { return bf2f(*p); }
  __device__ static float round(float x) { return bf2f(f2bf(x)); }
  __device__ static void store4(raw* p, f32x4 v) {
    *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
  }
};
struct EF16 {
  typedef uint16_t raw;
  __device__ static float h2f(uint16_t h) {
    return static_cast<float>(__builtin_bit_cast(_Float16, h));
  }
  __device__ static uint16_t f2h(float x) {  // round to nearest even
    return __builtin_bit_cast(uint16_t, static_cast<_Float16>(x));
  }
  __device__ static float load(const raw* p) { return h2f(*p); }
  __device__ static float round(float x) { return h2f(f2h(x)); }
  __device__ static void store4(raw* p, f32x4 v) {
    const uint32_t w0 = f2h(v[0]) | (static_cast<uint32_t>(f2h(v[1])) << 16);
    const uint32_t w1 = f2h(v[2]) | (static_cast<uint32_t>(f2h(v[3])) << 16);
    *reinterpret_cast<uint2*>(p) = make_uint2(w0, w1);
  }
};
struct EF32 {
  typedef float raw;
  __device__ static float load(const raw* p) { return *p; }
  __device__ static float round(float x) { return x; }
  __device__ static void store4(raw* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }
};

// 16-bit element types on the matrix cores.  widen / narrow convert two packed
// values; weights() packs two or four softmax weights for P . V in kParts operands
// and returns their sum: bf16 weights are rounded to bf16 and summed as rounded.
// fp16 weights are two fp16 halves, hi + lo, both rounded to nearest: within 2^-24
// of a weight near 1 (an ulp of fp32), as good as the fp32 weights of the generic
// kernel; they are summed in fp32.  An infinite or NaN V needs the weight in one
// piece (0 times infinity is NaN), see odd_halves.
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

typedef float f32x16 __attribute__((ext_vector_type(16)));

template <typename E> struct Mma;
template <> struct Mma<EBf16> {
  static constexpr int kParts = 1;
  static constexpr float kPScale = 1.f;
  __device__ __forceinline__ static f32x16 mma32(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  __device__ __forceinline__ static float weights(float p0, float p1, uint32_t (&w)[kParts],
                                                  float l) {
    w[0] = pack_bf16x2(p0, p1);
    return sum_bf16x2(w[0], l);
  }
  __device__ __forceinline__ static f32x4 mma16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  __device__ __forceinline__ static f32x2 widen(uint32_t x) {
    return f32x2{__builtin_bit_cast(float, x << 16), __builtin_bit_cast(float, x & 0xffff0000u)};
  }
  __device__ __forceinline__ static uint32_t narrow(float a, float b) { return pack_bf16x2(a, b); }
  __device__ __forceinline__ static float weights(const float (&p)[4], uint32_t (&w)[kParts][2]) {
    w[0][0] = pack_bf16x2(p[0], p[1]);
    w[0][1] = pack_bf16x2(p[2], p[3]);
    const f32x2 x = widen(w[0][0]), y = widen(w[0][1]);
    return x[0] + x[1] + y[0] + y[1];
  }
};
template <> struct Mma<EF16> {
  static constexpr int kParts = 2;
  // Weights are scaled by kPScale, so that the halves of small ones do not fall
  // into fp16's subnormals; l carries the same factor.  (Multiplied: added to the
  // exponent instead, 12 would cost a weight near 1 three bits.)
  static constexpr float kPScale = 4096.f;
  // p0, p1 >= 0 as hi + lo: hi to nearest, the exact rest to nearest
  // (v_cvt_pk_f16_f32, v_fma_mix: four operations).
  __device__ __forceinline__ static void split(float p0, float p1, uint32_t (&w)[kParts]) {
    w[0] = narrow(p0, p1);
    const f16x2 hi = __builtin_bit_cast(f16x2, w[0]);
    w[1] = narrow(__builtin_fmaf(static_cast<float>(hi[0]), -1.f, p0),
                  __builtin_fmaf(static_cast<float>(hi[1]), -1.f, p1));
  }
  __device__ __forceinline__ static f32x16 mma32(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  __device__ __forceinline__ static float weights(float p0, float p1, uint32_t (&w)[kParts],
                                                  float l) {
    split(p0, p1, w);
    return l + (p0 + p1);
  }
  __device__ __forceinline__ static f32x4 mma16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  __device__ __forceinline__ static f32x2 widen(uint32_t x) {
    return __builtin_convertvector(__builtin_bit_cast(f16x2, x), f32x2);
  }
  __device__ __forceinline__ static uint32_t narrow(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, f16x2));
  }
  __device__ __forceinline__ static float weights(const float (&p)[4], uint32_t (&w)[kParts][2]) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      uint32_t x[kParts];
      split(p[2 * i], p[2 * i + 1], x);
      w[0][i] = x[0];
      w[1][i] = x[1];
    }
    return p[0] + p[1] + p[2] + p[3];
  }
};

// fp16 V with infinities or NaN: hi * inf + lo * inf is NaN where lo is 0 or
// negative.  Such values count apart from the others, under whole_weight: 1 for any
// positive weight, else the weight (0 or NaN).
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t odd_halves(uint32_t x) {
  return ((x & 0x7c00u) == 0x7c00u ? 0xffffu : 0u) |
         ((x & 0x7c000000u) == 0x7c000000u ? 0xffff0000u : 0u);
}
__device__ __forceinline__ u32x4 finite_part(u32x4 v) {
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] &= ~odd_halves(v[e]);
  return v;
}
__device__ __forceinline__ float whole_weight(float p) { return p > 0.f ? 1.f : p; }
// A zero half once some value so far was infinite or NaN (two operations a pair).
__device__ __forceinline__ u16x2 note_odd(u32x4 v, u16x2 seen) {
#pragma unroll
  for (int e = 0; e < 4; ++e)
    seen = __builtin_elementwise_min(seen, __builtin_bit_cast(u16x2, ~v[e] & 0x7c007c00u));
  return seen;
}

// Four consecutive table entries as loaded (raw) and as fp32 (cvt): the MFMA
// kernel keeps the raw chunk in registers while it is in flight and converts
// it when it is stored to LDS.
template <typename TT> struct TabChunk;
template <> struct TabChunk<EF32> {
  typedef f32x4 raw;
  __device__ static raw load(const void* base, size_t off) {
    return *reinterpret_cast<const f32x4*>(static_cast<const float*>(base) + off);
  }
  __device__ static f32x4 cvt(raw r) { return r; }
};
template <> struct TabChunk<EBf16> {
  typedef u32x2 raw;
  __device__ static raw load(const void* base, size_t off) {
    return *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(base) + off);
  }
  __device__ static f32x4 cvt(raw r) {
    return f32x4{__builtin_bit_cast(float, r[0] << 16),
                 __builtin_bit_cast(float, r[0] & 0xffff0000u),
                 __builtin_bit_cast(float, r[1] << 16),
                 __builtin_bit_cast(float, r[1] & 0xffff0000u)};
  }
};

template <> struct TabChunk<EF16> {
  typedef u32x2 raw;
  __device__ static raw load(const void* base, size_t off) {
    return *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(base) + off);
  }
  __device__ static f32x4 cvt(raw r) {
    const f32x2 a = Mma<EF16>::widen(r[0]), b = Mma<EF16>::widen(r[1]);
    return f32x4{a[0], a[1], b[0], b[1]};
  }
};

struct PfArgs {
  const void* q;             // [B, NQ, TQ, D]
  const void* k_pages;       // [P, NKV, BLOCK, D]
  const void* v_pages;       // [P, NKV, BLOCK, D]
  const int32_t* table;      // [ceil(TK / BLOCK)]
  const int32_t* k_pos;      // [TK]
  const int32_t* q_pos;      // [TQ]
  const void* cos_t;         // [max_pos, D/2]
  const void* sin_t;         // [max_pos, D/2]
  float* part_o;             // [B * NKV * splits, NCP, D]
  float* part_ml;            // [B * NKV * splits, NCP, 2]
  int B, NQ, TQ, NKV, G, D, BLOCK, P, TK, max_pos, splits;
  int NC;      // columns of a segment: G * TQ
  int ncg;     // columns per pass
  int passes;  // ceil(NC / ncg)
  int NCP;     // passes * ncg: partial rows per (segment, split)
  int nwork;   // workgroups of one pass
  float scale, scale_log2e;
};

// Work item and column pass of this workgroup.  With several passes, the
// passes of one work item get consecutive groups of eight workgroup ids at
// the same position in the group, i.e. the same XCD at about the same time
// (workgroups go to the XCDs round-robin), so every pass after the first
// reads the pages from that XCD's L2.  Ids past the last work item return
// false (a whole workgroup, before any barrier).
__device__ __forceinline__ bool pf_work(const PfArgs& a, int& w, int& pass) {
  const int bid = static_cast<int>(blockIdx.x);
  if (a.passes == 1) {
    w = bid;
    pass = 0;
    return true;
  }
  const int r = bid >> 3;
  pass = r % a.passes;
  w = (r / a.passes) * 8 + (bid & 7);
  return w < a.nwork;
}

// Table entry and raw logical position of key `key` (one per lane).  The
// loads are unconditional -- a key past the end reads entry 0, so a wavefront
// issues the same number of loads every block -- and only the loads: the
// arithmetic on them waits for pf_key_finish, so a wait for these loads never
// covers loads issued after them.  Requires TK > 0.
__device__ __forceinline__ void pf_key_load(const PfArgs& a, int key, int& page, int& pos) {
  const int k = key < a.TK ? key : 0;
  page = a.table[k / a.BLOCK];
  pos = a.k_pos[k];
}

// Page row of `key` for kv head `kvh` (split in 32-bit halves for the
// cross-lane reads) and its position clamped into the tables.  A key past the
// end gets row 0 and position 0; page ids out of range read page 0.
__device__ __forceinline__ void pf_key_finish(const PfArgs& a, int kvh, int key, int page,
                                              int pos, int& row_lo, int& row_hi, int& kpos) {
  long long row = 0;
  kpos = 0;
  if (key < a.TK) {
    const int blk = key / a.BLOCK;
    page = static_cast<unsigned>(page) < static_cast<unsigned>(a.P) ? page : 0;
    row = (static_cast<long long>(page) * a.NKV + kvh) * a.BLOCK + (key - blk * a.BLOCK);
    kpos = pos < 0 ? 0 : (pos >= a.max_pos ? a.max_pos - 1 : pos);
  }
  row_lo = static_cast<int>(row & 0xffffffff);
  row_hi = static_cast<int>(row >> 32);
}

__device__ __forceinline__ long long pf_row_of(int row_lo, int row_hi, int src) {
  return (static_cast<long long>(__shfl(row_hi, src)) << 32) |
         static_cast<unsigned>(__shfl(row_lo, src));
}

// One workgroup per (batch row, split, group of HW kv heads, column pass);
// wavefront w takes kv head HW * group + w.  All HW wavefronts walk the same
// key blocks, so a block's cos/sin rows are loaded once per workgroup into a
// shared LDS tile (double-buffered, one barrier per block) while every
// wavefront keeps its own K rows in registers and stages its own V rows in a
// private LDS slice.  Block i + 1's K and V rows, and its cos/sin rows, are in
// flight while block i is computed; table entries are fetched two blocks
// ahead.  Partials are indexed (segment * splits + split, pass * 16 + column).
// (With 2 or 1 wavefronts per workgroup each thread stages 4-8x the cos/sin
// chunks of the 8-wavefront shape; those variants get the whole register file.)
template <int D, int HW, typename E, typename TT>
__global__ __launch_bounds__(HW * kWave) __attribute__((amdgpu_waves_per_eu(HW >= 4 ? 2 : 1)))
void pf_attention_kernel(PfArgs a) {
  typedef Mma<E> MM;
  constexpr int KS = D / 32;     // k-steps of the score MFMA
  constexpr int HS = D / 64;     // k-steps in one rotary half
  constexpr int DT = D / 16;     // dim tiles of out^T
  constexpr int kVRow = D + 8;   // LDS row stride of the staged V rows (elements)
  constexpr int kVLoads = kKeys * D / 8 / kWave;  // 16-byte V chunks per lane
  constexpr int CPR = D / 8;     // 4-entry chunks in one cos (or sin) row of D/2 entries
  constexpr int kCsPerThread = kKeys * 2 * CPR / (HW * kWave);
  static_assert(kCsPerThread * HW * kWave == kKeys * 2 * CPR, "cos/sin tile split");
  typedef TabChunk<TT> TC;
  __shared__ __attribute__((aligned(16))) uint16_t v_stage[HW][kKeys * kVRow];
  // [buffer][key][cos, sin][chunk]: chunk c of key r sits at c ^ (r % CPR), so
  // the 16 lanes that read one chunk of 16 different keys hit distinct banks
  __shared__ f32x4 cs_stage[2][kKeys][2][CPR];

  int w, pass;
  if (!pf_work(a, w, pass)) return;
  const uint16_t* q16 = static_cast<const uint16_t*>(a.q);
  const uint16_t* kpg = static_cast<const uint16_t*>(a.k_pages);
  const uint16_t* vpg = static_cast<const uint16_t*>(a.v_pages);
  const int lane = threadIdx.x & (kWave - 1);
  const int wl = uniform(threadIdx.x / kWave);
  const int groups = a.NKV / HW;
  const int kg = w % groups;
  const int rest = w / groups;
  const int split = rest % a.splits;
  const int b = rest / a.splits;
  const int kvh = kg * HW + wl;
  const int seg = b * a.NKV + kvh;
  const size_t pidx = static_cast<size_t>(seg) * a.splits + split;
  const int nb = (a.TK + kKeys - 1) / kKeys;
  const int blo = static_cast<int>(static_cast<long long>(split) * nb / a.splits);
  const int bhi = static_cast<int>(static_cast<long long>(split + 1) * nb / a.splits);

  const int i16 = lane & 15;
  const int g = lane >> 4;
  const int col = pass * kCols + i16;  // (head, query) column of the segment
  const bool col_ok = col < a.NC;
  const int cj = col_ok ? col / a.TQ : 0;      // head within the group
  const int ctq = col_ok ? col - cj * a.TQ : 0;  // query
  const int qpos = a.q_pos[ctq];
  const int klane = lane & 31;  // the key this lane looks up (lanes 32..63 mirror)
  uint16_t* vs = v_stage[wl];

  // Q^T operand: lane (column i16, group g) holds q[head][tq][32s + 8g .. +8]
  u32x4 qop[KS];
  {
    const uint16_t* qh =
        q16 + ((static_cast<size_t>(b) * a.NQ + kvh * a.G + cj) * a.TQ + ctq) * D;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const u32x4 z = {0u, 0u, 0u, 0u};
      qop[s] = col_ok ? *reinterpret_cast<const u32x4*>(qh + 32 * s + 8 * g) : z;
    }
  }

  // K and V rows are read once per call: non-temporal loads (measured 37.7 ->
  // 36.7 us per call at 32,768 keys).
  auto load_k = [&](int rlo, int rhi, u32x4 (&kk)[2][KS]) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const uint16_t* krow = kpg + pf_row_of(rlo, rhi, 16 * t + i16) * D;
#pragma unroll
      for (int s = 0; s < KS; ++s)
        kk[t][s] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(krow + 32 * s + 8 * g));
    }
  };
  auto load_v = [&](int rlo, int rhi, u32x4 (&vv)[kVLoads]) {
#pragma unroll
    for (int u = 0; u < kVLoads; ++u) {
      const int c = u * kWave + lane;
      const int r = c / (D / 8);
      const int cc = c - r * (D / 8);
      vv[u] = __builtin_nontemporal_load(
          reinterpret_cast<const u32x4*>(vpg + pf_row_of(rlo, rhi, r) * D + 8 * cc));
    }
  };
  // V rows, coalesced 16-byte chunks, into this wave's LDS slice
  auto store_v = [&](const u32x4 (&vv)[kVLoads]) {
#pragma unroll
    for (int u = 0; u < kVLoads; ++u) {
      const int c = u * kWave + lane;
      const int r = c / (D / 8);
      const int cc = c - r * (D / 8);
      *reinterpret_cast<u32x4*>(vs + r * kVRow + 8 * cc) = vv[u];
    }
  };
  // this thread's share of a block's cos/sin rows: chunk id -> (key, table, chunk)
  auto load_cs = [&](int kp, typename TC::raw (&cr)[kCsPerThread]) {
#pragma unroll
    for (int i = 0; i < kCsPerThread; ++i) {
      const int cid = static_cast<int>(threadIdx.x) + i * HW * kWave;
      const int key = cid / (2 * CPR);
      const int tab = (cid / CPR) & 1;
      const int ch = cid & (CPR - 1);
      const int p = __shfl(kp, key);
      cr[i] = TC::load(tab ? a.sin_t : a.cos_t, static_cast<size_t>(p) * (D / 2) + 4 * ch);
    }
  };
  auto store_cs = [&](int buf, const typename TC::raw (&cr)[kCsPerThread]) {
#pragma unroll
    for (int i = 0; i < kCsPerThread; ++i) {
      const int cid = static_cast<int>(threadIdx.x) + i * HW * kWave;
      const int key = cid / (2 * CPR);
      const int tab = (cid / CPR) & 1;
      const int ch = cid & (CPR - 1);
      cs_stage[buf][key][tab][ch ^ (key & (CPR - 1))] = TC::cvt(cr[i]);
    }
  };

  f32x4 acc[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY;
  float l_lane = 0.f;

  // ---- prologue: block blo resident (K in registers; V and cos/sin in
  //      LDS), block blo + 1's table entries loaded ----
  // rows / table position / position for the mask of block bi.  (bf16 pages
  // mask by the position clamped into the tables, fp16 pages by the given one.)
  int rA_lo = 0, rA_hi = 0, kA = 0, mA = 0;
  int pgB = 0, psB = 0;               // raw table entry / position of block bi + 1
  u32x4 kc[2][KS];  // K rows of block bi (block bi + 1's once scored)
  if (blo < bhi) {
    int pg, ps;
    pf_key_load(a, blo * kKeys + klane, pg, ps);
    pf_key_finish(a, kvh, blo * kKeys + klane, pg, ps, rA_lo, rA_hi, kA);
    mA = MM::kParts == 2 ? ps : kA;
    pf_key_load(a, blo + 1 < bhi ? (blo + 1) * kKeys + klane : a.TK, pgB, psB);
    typename TC::raw c0[kCsPerThread];
    u32x4 v0[kVLoads];
    load_cs(kA, c0);
    load_v(rA_lo, rA_hi, v0);
    load_k(rA_lo, rA_hi, kc);
    store_cs(blo & 1, c0);
    store_v(v0);
  }
  // nothing of the prologue stays in flight into the loop, so the loop's
  // waits count only its own loads
  wait_vmem_all();
  lds_barrier();

  for (int bi = blo; bi < bhi; ++bi) {
    const bool more = bi + 1 < bhi;
    // ---- issue: table entries two ahead, then block bi + 1's rows.  Every
    //      load issues every block; past the split's end they read key
    //      row 0 / table entry 0 (one cache line), so the wait counts stay
    //      exact ----
    int pgC, psC;
    pf_key_load(a, bi + 2 < bhi ? (bi + 2) * kKeys + klane : a.TK, pgC, psC);
    int rB_lo, rB_hi, kB;
    pf_key_finish(a, kvh, more ? (bi + 1) * kKeys + klane : a.TK, pgB, psB, rB_lo, rB_hi,
                  kB);
    const int mB = MM::kParts == 2 ? psB : kB;
    u32x4 vn[kVLoads];
    typename TC::raw cn[kCsPerThread];
    // cos/sin and V now (they are waited for at the end of this block); K
    // once this block's keys are scored and their registers are free
    load_cs(kB, cn);
    load_v(rB_lo, rB_hi, vn);
    int kp[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int r = 0; r < 4; ++r) kp[t][r] = __shfl(mA, 16 * t + 4 * g + r);
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- rotate the keys in registers, score the two 16-key tiles ----
    const int buf = bi & 1;
    f32x4 sc[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int key = 16 * t + i16;
      const int sw = key & (CPR - 1);
#pragma unroll
      for (int s = 0; s < HS; ++s) {
        const int c0 = 8 * s + 2 * g;
        const f32x4 cA = cs_stage[buf][key][0][c0 ^ sw];
        const f32x4 cB = cs_stage[buf][key][0][(c0 + 1) ^ sw];
        const f32x4 sA = cs_stage[buf][key][1][c0 ^ sw];
        const f32x4 sB = cs_stage[buf][key][1][(c0 + 1) ^ sw];
        u32x4 lo_out, hi_out;
#pragma unroll
        for (int wv = 0; wv < 4; ++wv) {
          const f32x2 av = MM::widen(kc[t][s][wv]);
          const f32x2 bv = MM::widen(kc[t][s + HS][wv]);
          float ra[2], rb[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int e = 2 * wv + h;
            const float c = e < 4 ? cA[e] : cB[e - 4];
            const float sv = e < 4 ? sA[e] : sB[e - 4];
            ra[h] = av[h] * c - bv[h] * sv;
            rb[h] = bv[h] * c + av[h] * sv;
          }
          lo_out[wv] = MM::narrow(ra[0], ra[1]);
          hi_out[wv] = MM::narrow(rb[0], rb[1]);
        }
        kc[t][s] = lo_out;
        kc[t][s + HS] = hi_out;
      }
      f32x4 acc_s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        acc_s = MM::mma16(kc[t][s], qop[s], acc_s);
      }
      sc[t] = acc_s;
    }
    load_k(rB_lo, rB_hi, kc);

    // ---- mask, online softmax; lane (column i16, group g) holds keys
    //      16t + 4g + r ----
    float x[2][4];
    float mb = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kk = 16 * t + 4 * g + r;
        const bool vis = col_ok && bi * kKeys + kk < a.TK && kp[t][r] <= qpos;
        x[t][r] = vis ? sc[t][r] * a.scale_log2e : -INFINITY;
        mb = fmaxf(mb, x[t][r]);
      }
    }
    mb = wave_max_across_groups(mb);
    const float m_new = fmaxf(m_run, mb);
    const float alpha = m_new == m_run ? 1.f : fast_exp2(m_run - m_new);
    m_run = m_new;
    u32x4 pk[MM::kParts];
    float ps = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float p[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        p[r] = x[t][r] == -INFINITY ? 0.f : fast_exp2(x[t][r] - m_new) * MM::kPScale;
      uint32_t pw[MM::kParts][2];
      ps += MM::weights(p, pw);
#pragma unroll
      for (int part = 0; part < MM::kParts; ++part) {
        pk[part][2 * t] = pw[part][0];
        pk[part][2 * t + 1] = pw[part][1];
      }
    }
    l_lane = l_lane * alpha + ps;

    // ---- out^T[dims][columns] += V^T . P^T ----
#pragma unroll
    for (int d = 0; d < DT; ++d) acc[d] *= alpha;
    // lane i16 of group g addresses key row 4g + i16/4 (and +16) at dims
    // 16dt + 4*(i16%4): after the transpose lane l holds keys 4g..4g+3 (and
    // 16 + 4g..) of dim 16dt + l%16
    const uint16_t* vb = vs + (4 * g + (i16 >> 2)) * kVRow + 4 * (i16 & 3);
    auto read_v = [&](int d) {
      const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(vb + 16 * d));
      const bf16x4 hi =
          __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(vb + 16 * kVRow + 16 * d));
      return __builtin_bit_cast(u32x4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      const u32x4 av = read_v(d);
#pragma unroll
      for (int part = 0; part < MM::kParts; ++part) acc[d] = MM::mma16(av, pk[part], acc[d]);
    }

    // ---- block bi + 1's V rows into the slice once this block's reads of
    //      it are done, its cos/sin into the other buffer; after the barrier
    //      every wave has finished with this block's tiles ----
    if (more) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      store_v(vn);
      store_cs(buf ^ 1, cn);
    }
    lds_barrier();
    rA_lo = rB_lo;
    rA_hi = rB_hi;
    kA = kB;
    mA = mB;
    pgB = pgC;
    psB = psC;
  }

  if constexpr (MM::kParts == 2) {
    // An infinite or NaN V leaves nothing finite in its dim whatever its weight, but
    // possibly the wrong one of them: the keys' infinities once more, under whole
    // weights and the scores as above.  Rare and key by key.
    float any = 0.f;
#pragma unroll
    for (int d = 0; d < DT; ++d) {
#pragma unroll
      for (int r = 0; r < 4; ++r) any = __builtin_fmaf(acc[d][r], 0.f, any);
    }
    // (a NaN among the weights makes the whole row NaN: nothing to look for)
    if (__builtin_amdgcn_ballot_w64(any != 0.f && l_lane * 0.f == 0.f) != 0) {
      f32x4 odd[DT] = {};
      for (int key = blo * kKeys; key < min(bhi * kKeys, a.TK); ++key) {
        int pg, ps, rlo, rhi, kp;
        pf_key_load(a, key, pg, ps);
        pf_key_finish(a, kvh, key, pg, ps, rlo, rhi, kp);
        const size_t at = static_cast<size_t>(pf_row_of(rlo, rhi, lane)) * D;
        u32x2 vv[DT];
        uint32_t here = 0;
#pragma unroll
        for (int d = 0; d < DT; ++d) {
          vv[d] = *reinterpret_cast<const u32x2*>(vpg + at + 16 * d + 4 * g);
          here |= odd_halves(vv[d][0]) | odd_halves(vv[d][1]);
        }
        if (__builtin_amdgcn_ballot_w64(here != 0) == 0) continue;
        float s = 0.f;
#pragma unroll
        for (int st = 0; st < HS; ++st) {
          const int dim = 32 * st + 8 * g;
          const u32x4 lo = *reinterpret_cast<const u32x4*>(kpg + at + dim);
          const u32x4 hi = *reinterpret_cast<const u32x4*>(kpg + at + dim + D / 2);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const size_t to = static_cast<size_t>(kp) * (D / 2) + dim + 4 * (e >> 1);
            const f32x4 c = TC::cvt(TC::load(a.cos_t, to)), sn = TC::cvt(TC::load(a.sin_t, to));
            const f32x2 x = MM::widen(lo[e]), y = MM::widen(hi[e]);
            const f32x2 qa = MM::widen(qop[st][e]), qb = MM::widen(qop[st + HS][e]);
            const int n = 2 * (e & 1);
            const f32x2 ra = MM::widen(MM::narrow(x[0] * c[n] - y[0] * sn[n],
                                                  x[1] * c[n + 1] - y[1] * sn[n + 1]));
            const f32x2 rb = MM::widen(MM::narrow(y[0] * c[n] + x[0] * sn[n],
                                                  y[1] * c[n + 1] + x[1] * sn[n + 1]));
            s += ra[0] * qa[0] + ra[1] * qa[1] + rb[0] * qb[0] + rb[1] * qb[1];
          }
        }
        s = wave_sum_across_groups(s) * a.scale_log2e;
        const bool sees = ps <= qpos;
        const float wt = s == -INFINITY ? 0.f : whole_weight(fast_exp2(s - m_run));
#pragma unroll
        for (int d = 0; d < DT; ++d) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const f32x2 v = MM::widen(vv[d][r >> 1] & odd_halves(vv[d][r >> 1]));
            odd[d][r] += sees && v[r & 1] != 0.f ? wt * v[r & 1] : 0.f;
          }
        }
      }
#pragma unroll
      for (int d = 0; d < DT; ++d) {
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[d][r] = odd[d][r] != 0.f ? odd[d][r] : acc[d][r];
      }
    }
  }

  const float l_tot = wave_sum_across_groups(l_lane);
  if (col_ok) {
    const size_t row = pidx * a.NCP + col;
    float* po = a.part_o + row * D + 4 * g;
#pragma unroll
    for (int d = 0; d < DT; ++d) *reinterpret_cast<f32x4*>(po + 16 * d) = acc[d];
    if (g == 0) {
      a.part_ml[row * 2 + 0] = m_run;
      a.part_ml[row * 2 + 1] = l_tot;
    }
  }
}

// ---- generic kernel ---------------------------------------------------------
constexpr int kGenThreads = 256;
constexpr int kGenAcc = 16;                     // output values per thread
constexpr int kGenOut = kGenThreads * kGenAcc;  // columns * D of one pass
constexpr int kGenMaxD = 256;

// LDS of the generic kernel, in 4-byte words, for head dim D and ncg columns.
struct GenLds {
  int kr, vr, qs, ss, mcol, lcol, acol, qp, kpv, kpt, krow;  // word offsets
  int words;
};
__host__ __device__ inline GenLds gen_lds(int D, int ncg) {
  GenLds s;
  s.kr = 0;                              // [32][D + 4] rotated keys, rounded to T
  s.vr = s.kr + kKeys * (D + 4);         // [32][D]
  s.qs = s.vr + kKeys * D;               // [ncg][D] q * scale
  s.ss = s.qs + ncg * D;                 // [ncg][32] scores (log2 units), then P
  s.mcol = s.ss + ncg * kKeys;           // [ncg] running maximum
  s.lcol = s.mcol + ncg;                 // [ncg] running sum
  s.acol = s.lcol + ncg;                 // [ncg] this block's rescale
  s.qp = s.acol + ncg;                   // [ncg] query position (INT_MIN: no column)
  s.kpv = s.qp + ncg;                    // [32] key position for the mask
  s.kpt = s.kpv + kKeys;                 // [32] key position clamped into the tables
  s.krow = (s.kpt + kKeys + 1) & ~1;     // [32] int64 page rows
  s.words = s.krow + 2 * kKeys;
  return s;
}

// One workgroup of 256 threads per (batch row, kv head, split, column pass).
// Per 32-key block: thread t < 32 resolves key t's page row and position; the
// keys are rotated in fp32, rounded to T and staged in LDS with the V rows
// (one pair of rotary dims per thread step, coalesced over dims); every score
// is an fp32 dot product over LDS (thread = (key, column)); each half-wave
// runs one column's online-softmax step; then thread t owns output values
// t + 256 i (i < 16) of the pass's [columns][D] block and adds P . V over the
// 32 keys.  P stays fp32, as in the reference kernel.
template <typename E, typename TT>
__global__ __launch_bounds__(kGenThreads) void pf_generic_kernel(PfArgs a) {
  extern __shared__ __attribute__((aligned(16))) float gsm[];
  int w, pass;
  if (!pf_work(a, w, pass)) return;
  typedef typename E::raw R;
  typedef typename TT::raw TR;
  const int D = a.D;
  const int H = D / 2;
  const int KR = D + 4;
  const int ncg = a.ncg;
  const GenLds L = gen_lds(D, ncg);
  float* kr = gsm + L.kr;
  float* vr = gsm + L.vr;
  float* qs = gsm + L.qs;
  float* ss = gsm + L.ss;
  float* mcol = gsm + L.mcol;
  float* lcol = gsm + L.lcol;
  float* acol = gsm + L.acol;
  int* qp = reinterpret_cast<int*>(gsm + L.qp);
  int* kpv = reinterpret_cast<int*>(gsm + L.kpv);
  int* kpt = reinterpret_cast<int*>(gsm + L.kpt);
  long long* krow = reinterpret_cast<long long*>(gsm + L.krow);

  const R* qg = static_cast<const R*>(a.q);
  const R* kpg = static_cast<const R*>(a.k_pages);
  const R* vpg = static_cast<const R*>(a.v_pages);
  const TR* cos_t = static_cast<const TR*>(a.cos_t);
  const TR* sin_t = static_cast<const TR*>(a.sin_t);
  const int t = threadIdx.x;
  const int kvh = w % a.NKV;
  const int rest = w / a.NKV;
  const int split = rest % a.splits;
  const int b = rest / a.splits;
  const size_t pidx = static_cast<size_t>(b * a.NKV + kvh) * a.splits + split;
  const int nb = (a.TK + kKeys - 1) / kKeys;
  const int blo = static_cast<int>(static_cast<long long>(split) * nb / a.splits);
  const int bhi = static_cast<int>(static_cast<long long>(split + 1) * nb / a.splits);
  const int n0 = pass * ncg;
  const int ncols = min(ncg, a.NC - n0);

  for (int e = t; e < ncg * D; e += kGenThreads) {
    const int c = e / D;
    const int d = e - c * D;
    float v = 0.f;
    if (c < ncols) {
      const int n = n0 + c;
      const int j = n / a.TQ;
      const int tq = n - j * a.TQ;
      v = E::load(qg + ((static_cast<size_t>(b) * a.NQ + kvh * a.G + j) * a.TQ + tq) * D + d) *
          a.scale;
    }
    qs[e] = v;
  }
  for (int c = t; c < ncg; c += kGenThreads) {
    mcol[c] = -INFINITY;
    lcol[c] = 0.f;
    qp[c] = c < ncols ? a.q_pos[(n0 + c) % a.TQ] : INT_MIN;
  }
  float acc[kGenAcc];
#pragma unroll
  for (int i = 0; i < kGenAcc; ++i) acc[i] = 0.f;

  for (int bi = blo; bi < bhi; ++bi) {
    __syncthreads();  // the previous block's LDS reads are done
    if (t < kKeys) {
      const int key = bi * kKeys + t;
      long long row = 0;
      int pv = INT_MAX, pt = 0;
      if (key < a.TK) {
        const int blk = key / a.BLOCK;
        int page = a.table[blk];
        page = static_cast<unsigned>(page) < static_cast<unsigned>(a.P) ? page : 0;
        row = (static_cast<long long>(page) * a.NKV + kvh) * a.BLOCK + (key - blk * a.BLOCK);
        pv = a.k_pos[key];
        pt = pv < 0 ? 0 : (pv >= a.max_pos ? a.max_pos - 1 : pv);
      }
      krow[t] = row;
      kpv[t] = pv;
      kpt[t] = pt;
    }
    __syncthreads();
    for (int p = t; p < kKeys * H; p += kGenThreads) {
      const int key = p / H;
      const int d = p - key * H;
      const R* kk = kpg + krow[key] * D;
      const float x = E::load(kk + d);
      const float y = E::load(kk + d + H);
      const size_t to = static_cast<size_t>(kpt[key]) * H + d;
      const float c = TT::load(cos_t + to);
      const float s = TT::load(sin_t + to);
      kr[key * KR + d] = E::round(x * c - y * s);
      kr[key * KR + d + H] = E::round(y * c + x * s);
    }
    for (int e = t; e < kKeys * D; e += kGenThreads) {
      const int key = e / D;
      vr[e] = E::load(vpg + krow[key] * D + (e - key * D));
    }
    __syncthreads();
    {
      const int sk = t & (kKeys - 1);
      const f32x4* kq = reinterpret_cast<const f32x4*>(kr + sk * KR);
      const bool key_ok = bi * kKeys + sk < a.TK;
      for (int c = t / kKeys; c < ncg; c += kGenThreads / kKeys) {
        const f32x4* qq = reinterpret_cast<const f32x4*>(qs + c * D);
        float s = 0.f;
        for (int d4 = 0; d4 < D / 4; ++d4) {
          const f32x4 x = kq[d4];
          const f32x4 y = qq[d4];
          s = fmaf(x[0], y[0], s);
          s = fmaf(x[1], y[1], s);
          s = fmaf(x[2], y[2], s);
          s = fmaf(x[3], y[3], s);
        }
        ss[c * kKeys + sk] = key_ok && kpv[sk] <= qp[c] ? s * kLog2e : -INFINITY;
      }
    }
    __syncthreads();
    {
      const int l32 = t & (kKeys - 1);
      for (int c = t / kKeys; c < ncg; c += kGenThreads / kKeys) {
        const float x = ss[c * kKeys + l32];
        float mx = x;
#pragma unroll
        for (int o = kKeys / 2; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, kKeys));
        const float mo = mcol[c];
        const float mn = fmaxf(mo, mx);
        const float p = x == -INFINITY ? 0.f : fast_exp2(x - mn);
        ss[c * kKeys + l32] = p;
        float sum = p;
#pragma unroll
        for (int o = kKeys / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o, kKeys);
        if (l32 == 0) {
          const float al = mn == mo ? 1.f : fast_exp2(mo - mn);
          acol[c] = al;
          lcol[c] = lcol[c] * al + sum;
          mcol[c] = mn;
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kGenAcc; ++i) {
      const int e = t + kGenThreads * i;
      if (e < ncg * D) {
        const int c = e / D;
        const int d = e - c * D;
        const f32x4* pc = reinterpret_cast<const f32x4*>(ss + c * kKeys);
        float s = acc[i] * acol[c];
#pragma unroll
        for (int k4 = 0; k4 < kKeys / 4; ++k4) {
          const f32x4 pp = pc[k4];
          s = fmaf(pp[0], vr[(4 * k4 + 0) * D + d], s);
          s = fmaf(pp[1], vr[(4 * k4 + 1) * D + d], s);
          s = fmaf(pp[2], vr[(4 * k4 + 2) * D + d], s);
          s = fmaf(pp[3], vr[(4 * k4 + 3) * D + d], s);
        }
        acc[i] = s;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kGenAcc; ++i) {
    const int e = t + kGenThreads * i;
    if (e < ncols * D) {
      const int c = e / D;
      a.part_o[(pidx * a.NCP + n0 + c) * D + (e - c * D)] = acc[i];
    }
  }
  for (int c = t; c < ncols; c += kGenThreads) {
    a.part_ml[(pidx * a.NCP + n0 + c) * 2 + 0] = mcol[c];
    a.part_ml[(pidx * a.NCP + n0 + c) * 2 + 1] = lcol[c];
  }
}

// One workgroup per (segment, column, 32-dim slice of the output row): its
// kRedWaves wavefronts each merge a contiguous share of the segment's split
// partials, then wave 0 merges their states and writes the slice of
// out[b][head][tq][:] (zeros when no key was visible).  Spreading a row over
// D/32 workgroups spreads the partial reads over that many more CUs.  Lane
// (r, j) of a wavefront reads dims 4j..4j+3 of the slice for split r of each
// group of kRedRows consecutive splits; a batch of kRedIters groups is loaded
// before its first use (one memory round trip), and the batch maximum
// rescales the running state.  A split with no visible key left m = -inf and
// weighs 0.
constexpr int kRedWaves = 4;
constexpr int kRedDims = 32;                  // output dims per workgroup
constexpr int kRedCols = kRedDims / 4;        // lanes across one slice (float4 each)
constexpr int kRedRows = kWave / kRedCols;    // splits per wave-wide load
constexpr int kRedIters = 8;                  // wave-wide loads per batch

template <typename E>
__global__ __launch_bounds__(kRedWaves * kWave) void pf_reduce_kernel(PfArgs a,
                                                                      typename E::raw* out) {
  __shared__ float st_ml[kRedWaves][2];
  __shared__ __attribute__((aligned(16))) f32x4 st_o[kRedWaves][kRedCols];
  const int D = a.D;
  const int slices = D / kRedDims;
  const int lane = threadIdx.x & (kWave - 1);
  const int wl = uniform(threadIdx.x / kWave);
  const int slice = blockIdx.x % slices;
  const int task = blockIdx.x / slices;
  const int seg = task / a.NC;
  const int n = task - seg * a.NC;
  const int r = lane / kRedCols;
  const int j = lane - r * kRedCols;
  const int s0 = static_cast<int>(static_cast<long long>(wl) * a.splits / kRedWaves);
  const int cnt = static_cast<int>(static_cast<long long>(wl + 1) * a.splits / kRedWaves) - s0;
  const size_t first = static_cast<size_t>(seg) * a.splits + s0;
  const float2* ml2 = reinterpret_cast<const float2*>(a.part_ml);
  const int dim0 = slice * kRedDims + 4 * j;

  float M = -INFINITY;
  float L = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int i0 = 0; i0 < cnt; i0 += kRedRows * kRedIters) {
    float2 ml[kRedIters];
    f32x4 o[kRedIters];
#pragma unroll
    for (int u = 0; u < kRedIters; ++u) {
      const int i = i0 + u * kRedRows + r;
      const size_t p = (first + (i < cnt ? i : cnt - 1)) * a.NCP + n;
      ml[u] = ml2[p];
      o[u] = *reinterpret_cast<const f32x4*>(a.part_o + p * D + dim0);
    }
    // everything above issues before the first use
    __builtin_amdgcn_sched_barrier(0);
    float Mc = -INFINITY;
#pragma unroll
    for (int u = 0; u < kRedIters; ++u) {
      const bool live = i0 + u * kRedRows + r < cnt;
      if (live) Mc = fmaxf(Mc, ml[u].x);
    }
    Mc = wave_max_uniform(Mc);  // DPP moves + v_readlane, no LDS crossbar trips
    const float Mn = fmaxf(M, Mc);
    if (Mn == -INFINITY) continue;  // wave-uniform: nothing visible yet
    const float rescale = M == -INFINITY ? 0.f : fast_exp2(M - Mn);
    float Lc = 0.f;
    acc *= rescale;
#pragma unroll
    for (int u = 0; u < kRedIters; ++u) {
      const bool live = i0 + u * kRedRows + r < cnt && ml[u].x != -INFINITY;
      const float w = live ? fast_exp2(ml[u].x - Mn) : 0.f;
      acc += o[u] * w;
      Lc += ml[u].y * w;
    }
    // each split's l is held by all kRedCols lanes of its row: count lane j == 0
    Lc = wave_sum_uniform(j == 0 ? Lc : 0.f);
    L = L * rescale + Lc;
    M = Mn;
  }
  // Past the last split a lane reads that split's row once more, with weight 0: an
  // infinity there has become NaN, so once more without those rows (rare).
  float any = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) any = __builtin_fmaf(acc[e], 0.f, any);
  if (__builtin_amdgcn_ballot_w64(any != 0.f) != 0) {
    acc = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int i = r; i < cnt; i += kRedRows) {
      const size_t p = (first + i) * a.NCP + n;
      const float w = ml2[p].x == -INFINITY ? 0.f : fast_exp2(ml2[p].x - M);
      acc += *reinterpret_cast<const f32x4*>(a.part_o + p * D + dim0) * w;
    }
  }
  // rows of one wave share M: the lanes of a column sum their rows
#pragma unroll
  for (int x = kRedCols; x < kWave; x <<= 1) {
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] += __shfl_xor(acc[e], x);
  }
  if (lane == 0) {
    st_ml[wl][0] = M;
    st_ml[wl][1] = L;
  }
  if (r == 0) st_o[wl][j] = acc;
  __syncthreads();
  if (wl != 0 || r != 0) return;
  float Mt = -INFINITY;
#pragma unroll
  for (int k = 0; k < kRedWaves; ++k) Mt = fmaxf(Mt, st_ml[k][0]);
  float Lt = 0.f;
  f32x4 res = {0.f, 0.f, 0.f, 0.f};
  if (Mt != -INFINITY) {
#pragma unroll
    for (int k = 0; k < kRedWaves; ++k) {
      const float mk = st_ml[k][0];
      const float wk = mk == -INFINITY ? 0.f : fast_exp2(mk - Mt);
      Lt += st_ml[k][1] * wk;
      res += st_o[k][j] * wk;
    }
  }
  const float inv = Lt > 0.f ? 1.f / Lt : 0.f;
  const int b = seg / a.NKV;
  const int kvh = seg - b * a.NKV;
  const int hj = n / a.TQ;
  const int tq = n - hj * a.TQ;
  E::store4(out + ((static_cast<size_t>(b) * a.NQ + kvh * a.G + hj) * a.TQ + tq) * D + dim0,
            res * inv);
}

// ---- windows: many columns over 16-bit pages ----------------------------------
// A segment with many (query, head) columns is bound by matrix work, and the
// passes of pf_attention_kernel rotate every key again for each 16 columns.  So
// pf_stage_kernel first gathers the pages once, rotates the keys, and leaves
// contiguous 32-key blocks in the workspace, K [32][D] and V^T [D][32], with the
// positions for the mask; pf_window_kernel then runs 64-key tiles of them against
// 32 rows per wavefront, as gqa_prefill_kernel does over pages of rotated keys:
// the rows of a kv head are its (batch row, query, head of the group) columns,
// scores^T and out^T on 32x32x16 MFMAs, P^T in registers, the scores one tile
// ahead of P . V, operands straight into LDS, one barrier per tile.  250 queries
// over 8,003 keys (28q/4kv, D = 128): fp16 3,866 us in the generic kernel, 446 in
// pf_attention_kernel's 110 passes, 72 here (11 of them staging, 5 the merge of its
// splits); bf16 449 and 60 us.
constexpr int kWinWaves = 4;
constexpr int kWinRows = 32;                       // rows of a wavefront
constexpr int kWinTile = kWinWaves * kWinRows;     // rows of a workgroup
constexpr int kWinKeys = 64;                       // keys of a tile
constexpr int kWinAhead = 4;                       // operand reads ahead of the MFMAs
constexpr int kWinMaxSplits = 64;

struct WinArgs {
  PfArgs p;
  uint16_t* k_blk;      // [NKV, nblk, 32, D]
  uint16_t* v_blk;      // [NKV, nblk, D, 32]
  int32_t* pos;         // [nblk * 32] positions for the mask (INT_MAX past the last key)
  int2* span;           // [nblk] smallest and largest of them
  int32_t* odd;         // [NKV, nblk] fp16: whether V holds an infinity or a NaN
  int nblk;             // 32-key blocks, even
  int R;                // rows of a kv head: B * TQ * G, the head fastest
  int row_tiles, splits;
  int work, per_xcd, xcd_cus;
  float scale;          // |softmax scale| in log2 units, > 0; its sign is applied to q
  uint32_t q_keep, q_flip;
};

// Workgroup (blk, kvh): one 32-key block.
template <int D, typename E, typename TT>
__global__ __launch_bounds__(256) void pf_stage_kernel(WinArgs w) {
  typedef Mma<E> MM;
  typedef TabChunk<TT> TC;
  constexpr int kPairs = kKeys * D / 16;   // (8 dims, their rotary partners) of a key
  constexpr int kChunks = kKeys * D / 8;   // 16-byte chunks of V
  constexpr int kVs = D + 8;
  __shared__ long long row[kKeys];
  __shared__ int at[kKeys];
  __shared__ __attribute__((aligned(16))) uint16_t vs[kKeys * kVs];
  const PfArgs& a = w.p;
  const int t = threadIdx.x;
  const int blk = blockIdx.x / a.NKV;
  const int kvh = blockIdx.x - blk * a.NKV;
  if (t < kKeys) {
    const int key = blk * kKeys + t;
    long long r = -1;
    int p = 0, m = INT_MAX;
    if (key < a.TK) {
      const int tb = key / a.BLOCK;
      int page = a.table[tb];
      page = static_cast<unsigned>(page) < static_cast<unsigned>(a.P) ? page : 0;
      r = (static_cast<long long>(page) * a.NKV + kvh) * a.BLOCK + (key - tb * a.BLOCK);
      const int raw = a.k_pos[key];
      p = raw < 0 ? 0 : (raw >= a.max_pos ? a.max_pos - 1 : raw);
      m = MM::kParts == 2 ? raw : p;  // as pf_attention_kernel masks
    }
    row[t] = r;
    at[t] = p;
    if (kvh == 0) {
      w.pos[blk * kKeys + t] = m;
      int lo = m, hi = m;
#pragma unroll
      for (int o = kKeys / 2; o > 0; o >>= 1) {
        lo = min(lo, __shfl_xor(lo, o, kKeys));
        hi = max(hi, __shfl_xor(hi, o, kKeys));
      }
      if (t == 0) w.span[blk] = make_int2(lo, hi);
    }
  }
  __syncthreads();
  const uint16_t* kp = static_cast<const uint16_t*>(a.k_pages);
  const uint16_t* vp = static_cast<const uint16_t*>(a.v_pages);
  const size_t out = (static_cast<size_t>(kvh) * w.nblk + blk) * (kKeys * D);
  u16x2 seen = {0xffff, 0xffff};
  for (int i = t; i < kChunks; i += 256) {
    const int key = i / (D / 8), c = i % (D / 8);
    const u32x4 z = {0u, 0u, 0u, 0u};
    u32x4 v = row[key] < 0 ? z : __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(
                                     vp + row[key] * D + 8 * c));
    if constexpr (MM::kParts == 2) {
      seen = note_odd(v, seen);
      v = finite_part(v);  // pf_window_kernel's add_odd brings the others
    }
    *reinterpret_cast<u32x4*>(vs + key * kVs + 8 * c) = v;
  }
  for (int i = t; i < kPairs; i += 256) {
    const int key = i / (D / 16), c = i % (D / 16);
    const uint16_t* kr = kp + (row[key] < 0 ? 0 : row[key]) * D + 8 * c;
    const u32x4 x = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(kr));
    const u32x4 y = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(kr + D / 2));
    const size_t to = static_cast<size_t>(at[key]) * (D / 2) + 8 * c;
    const f32x4 c0 = TC::cvt(TC::load(a.cos_t, to)), c1 = TC::cvt(TC::load(a.cos_t, to + 4));
    const f32x4 s0 = TC::cvt(TC::load(a.sin_t, to)), s1 = TC::cvt(TC::load(a.sin_t, to + 4));
    u32x4 lo, hi;
#pragma unroll
    for (int wv = 0; wv < 4; ++wv) {
      const f32x2 av = MM::widen(x[wv]), bv = MM::widen(y[wv]);
      float ra[2], rb[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int e = 2 * wv + h;
        const float cv = e < 4 ? c0[e] : c1[e - 4];
        const float sv = e < 4 ? s0[e] : s1[e - 4];
        ra[h] = av[h] * cv - bv[h] * sv;
        rb[h] = bv[h] * cv + av[h] * sv;
      }
      lo[wv] = MM::narrow(ra[0], ra[1]);
      hi[wv] = MM::narrow(rb[0], rb[1]);
    }
    if (row[key] < 0) lo = hi = u32x4{0u, 0u, 0u, 0u};
    uint16_t* o = w.k_blk + out + key * D + 8 * c;
    *reinterpret_cast<u32x4*>(o) = lo;
    *reinterpret_cast<u32x4*>(o + D / 2) = hi;
  }
  if constexpr (MM::kParts == 2) {
    const int odd = __syncthreads_or(seen[0] == 0 || seen[1] == 0);
    if (t == 0) w.odd[kvh * w.nblk + blk] = odd;
  } else {
    __syncthreads();
  }
  for (int i = t; i < kChunks; i += 256) {
    const int d = i >> 2, c = i & 3;
    u32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = vs[(8 * c + 2 * e) * kVs + d] |
             (static_cast<uint32_t>(vs[(8 * c + 2 * e + 1) * kVs + d]) << 16);
    *reinterpret_cast<u32x4*>(w.v_blk + out + d * kKeys + 8 * c) = v;
  }
}

// Key (0..31 of a block) that row r of the score tile holds: lane half h then
// has keys 8h..8h+7 in its first eight accumulators and 16+8h.. in the others,
// which is the order its P^T operand needs.
__device__ __forceinline__ int win_key_of_row(int r) {
  return 16 * (r >> 4) + 8 * ((r >> 2) & 1) + 4 * ((r >> 3) & 1) + (r & 3);
}
// Chunk c (16 bytes) of K row r sits at c ^ win_k_swizzle(r) in LDS.
template <int D>
__device__ __forceinline__ int win_k_swizzle(int r) {
  return D == 128 ? (r & 15) : ((r >> 1) & 7);
}

template <int D, typename E>
__global__ __launch_bounds__(kWinWaves * kWave) __attribute__((amdgpu_waves_per_eu(2, 2)))
void pf_window_kernel(WinArgs wa, uint16_t* out) {
  typedef Mma<E> MM;
  typedef __attribute__((address_space(3))) void lds_void;
  constexpr int NW = kWinWaves;
  constexpr int kBlkElems = kKeys * D;
  constexpr int kPieces = kBlkElems / 512;  // 1 KiB loads per block
  constexpr int kLoads = 4 * kPieces / NW;  // per wavefront and stage
  constexpr int kCpr = D / 8;               // 16-byte chunks of a K row
  constexpr int KS = D / 16;
  constexpr int DT = D / 32;
  constexpr int kA = kWinAhead;
  // masks of __builtin_amdgcn_sched_group_barrier
  constexpr int kValu = 0x002, kMfma = 0x008, kVmemRead = 0x020, kDsRead = 0x100, kTrans = 0x400;
  static_assert(kPieces >= NW && (kLoads == 8 || kLoads == 4), "loads of a stage");
  // K block 0, K block 1, V^T block 0, V^T block 1; two distinct objects, so that
  // reads of one provably miss the other's pending direct-to-LDS loads
  __shared__ __attribute__((aligned(1024))) uint16_t tile_a[4 * kBlkElems];
  __shared__ __attribute__((aligned(1024))) uint16_t tile_b[4 * kBlkElems];
  const PfArgs& a = wa.p;

  // as in gqa_prefill_kernel: consecutive work items of one XCD share a kv head
  const int bid = static_cast<int>(blockIdx.x);
  int slot = bid >> 3;
  if (slot >= wa.xcd_cus && wa.per_xcd <= 2 * wa.xcd_cus)
    slot = wa.per_xcd - 1 - (slot - wa.xcd_cus);
  const int wk = (bid & 7) * wa.per_xcd + slot;
  if (wk >= wa.work) return;
  const int per_seg = wa.row_tiles * wa.splits;
  const int kvh = wk / per_seg;
  const int in_seg = wk - kvh * per_seg;
  const int rt = wa.row_tiles - 1 - in_seg / wa.splits;
  const int split = in_seg % wa.splits;

  const int lane = threadIdx.x & (kWave - 1);
  const int w = uniform(threadIdx.x / kWave) & (NW - 1);
  const int l32 = lane & 31;
  const int lh = lane >> 5;

  // this lane's row: (batch row, query, head)
  const int row = rt * kWinTile + w * kWinRows + l32;
  const bool row_ok = row < wa.R;
  const int rc = row_ok ? row : wa.R - 1;
  const int bt = rc / a.G;
  const int b = bt / a.TQ;
  const int tq = bt - b * a.TQ;
  const size_t qrow =
      (static_cast<size_t>(b) * a.NQ + kvh * a.G + (rc - bt * a.G)) * a.TQ + tq;
  const int qpos = a.q_pos[tq];
  int q_lo = qpos, q_hi = qpos;  // of the wavefront's rows
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) {
    q_lo = min(q_lo, __shfl_xor(q_lo, o));
    q_hi = max(q_hi, __shfl_xor(q_hi, o));
  }
  // keys end (for this workgroup) with the last block that one of its rows sees
  int n_tiles;
  {
    int top = INT_MIN;
#pragma unroll
    for (int i = 0; i < kWinTile / kWave; ++i) {
      const int r = min(rt * kWinTile + i * kWave + lane, wa.R - 1);
      top = max(top, a.q_pos[(r / a.G) % a.TQ]);
    }
    int last = -1;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) top = max(top, __shfl_xor(top, o));
    for (int i = lane; i < wa.nblk; i += kWave) {
      if (i * kKeys < a.TK && wa.span[i].x <= top) last = i;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) last = max(last, __shfl_xor(last, o));
    n_tiles = uniform(last + 2) >> 1;
  }
  const int t_lo = static_cast<int>(static_cast<long long>(split) * n_tiles / wa.splits);
  const int t_hi = static_cast<int>(static_cast<long long>(split + 1) * n_tiles / wa.splits);
  // whether V of this workgroup's blocks 2 t_lo + lane, + 64 .. had infinities or NaN
  const int32_t* odd = wa.odd + static_cast<size_t>(kvh) * wa.nblk;
  int odd_blocks = 0;
  if (MM::kParts == 2 && 2 * t_lo + lane < 2 * t_hi) odd_blocks = odd[2 * t_lo + lane];

  u32x4 qop[KS];
  auto load_q = [&]() {
    const uint16_t* qh = static_cast<const uint16_t*>(a.q) + qrow * D + 8 * lh;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      qop[s] = *reinterpret_cast<const u32x4*>(qh + 16 * s);
#pragma unroll
      for (int i = 0; i < 4; ++i) qop[s][i] = (qop[s][i] & wa.q_keep) ^ wa.q_flip;
    }
  };

  // Per tile of win .. win + 63, one bit each: every row of the wavefront sees
  // all its keys; some row sees one.
  int win = 0;
  unsigned long long whole_bits = 0, seen_bits = 0;
  auto look_ahead = [&](int t) {
    win = t;
    const int mine = t + lane;
    int2 s0 = make_int2(INT_MAX, INT_MAX), s1 = s0;
    if (2 * mine < wa.nblk) {
      s0 = wa.span[2 * mine];
      s1 = wa.span[2 * mine + 1];
    }
    whole_bits = __builtin_amdgcn_ballot_w64((mine + 1) * kWinKeys <= a.TK && s0.y <= q_lo &&
                                             s1.y <= q_lo);
    seen_bits = __builtin_amdgcn_ballot_w64(mine * kWinKeys < a.TK && (s0.x <= q_hi || s1.x <= q_hi));
    wait_vmem_all();
  };
  auto whole = [&](int t) { return ((whole_bits >> (t - win)) & 1) != 0; };
  auto seen = [&](int t) { return ((seen_bits >> (t - win)) & 1) != 0; };

  // Stage t holds K of tile t + 1 and V^T of tile t.
  const uint16_t* kseg = wa.k_blk + static_cast<size_t>(kvh) * wa.nblk * kBlkElems;
  const uint16_t* vseg = wa.v_blk + static_cast<size_t>(kvh) * wa.nblk * kBlkElems;
  auto load_piece = [&](int i, int t, uint16_t* dst) {
    const int p = w + NW * i;
    const int j = (p / kPieces) & 1;
    const int sub = p % kPieces;
    const bool is_v = i >= kLoads / 2;
    const uint16_t* base =
        (is_v ? vseg + static_cast<size_t>(max(t, 0)) * (2 * kBlkElems)
              : kseg + static_cast<size_t>(min(t + 1, t_hi - 1)) * (2 * kBlkElems)) +
        j * kBlkElems;
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(base), static_cast<short>(0), kBlkElems * 2, 0x00020000);
    const int krow = sub * (kWave / kCpr) + lane / kCpr;
    const int ksrc = krow * (D * 2) + 16 * ((lane % kCpr) ^ win_k_swizzle<D>(krow));
    const int vrow = sub * 16 + (lane >> 2);
    const int vsrc = vrow * (kKeys * 2) + 16 * ((lane & 3) ^ ((lane >> 4) & 3));
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)(dst + p * 512), 16, is_v ? vsrc : ksrc,
                                             0, 0, 0);
  };
  auto load_stage = [&](int t, uint16_t* dst) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) load_piece(i, t, dst);
  };

  const int key = win_key_of_row(l32);
  const int k_lane = key * (D * 2) + 16 * (lh ^ win_k_swizzle<D>(key));
  int v_lane[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
    v_lane[ks] = l32 * (kKeys * 2) + 16 * ((2 * ks + lh) ^ ((l32 >> 2) & 3));

  f32x16 acc[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) acc[d] = f32x16{};
  // never -inf, as in gqa_prefill_kernel: keys of score -inf have P = 0
  float m = -FLT_MAX;
  float l = 0.f;

  typedef f32x16 Scores[2];  // accumulator i of block j: key 32 j + 16 (i / 8) + 8 lh + i % 8
  auto mask_scores = [&](int t, Scores& sc) {
    const int32_t* kp = wa.pos + t * kWinKeys + 8 * lh;
#pragma unroll
    for (int jk = 0; jk < 4; ++jk) {
      const int4 p0 = *reinterpret_cast<const int4*>(kp + 16 * jk);
      const int4 p1 = *reinterpret_cast<const int4*>(kp + 16 * jk + 4);
      const int ps[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
      const int lim = a.TK - t * kWinKeys - 16 * jk - 8 * lh;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float x = sc[jk >> 1][8 * (jk & 1) + i];
        sc[jk >> 1][8 * (jk & 1) + i] = i < lim && ps[i] <= qpos ? x : -INFINITY;
      }
    }
  };
  auto max_of = [&](const Scores& sc) {
    float mx = fmaxf(sc[0][0], sc[1][0]);
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(fmaxf(mx, sc[0][i]), sc[1][i]);
    return mx;
  };
  auto raise = [&](float mx) {
    mx = fmaxf(mx, __shfl_xor(mx, 32)) * wa.scale;
    if (__builtin_amdgcn_ballot_w64(mx > m) == 0) return;
    const float mn = fmaxf(m, mx);
    float alpha = fast_exp2(m - mn);
    asm volatile("" : "+v"(alpha));  // keeps the rescaling inside the branch
    m = mn;
    l *= alpha;
#pragma unroll
    for (int d = 0; d < DT; ++d) acc[d] *= alpha;
  };
  auto read_k = [&](const uint16_t* tile, int i) {  // i = 2 s + j
    return *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(tile) +
                                           (i & 1) * (kBlkElems * 2) + (k_lane ^ (32 * (i >> 1))));
  };
  auto read_v = [&](const uint16_t* tile, int i) {  // i = (2 j + ks) * DT + d
    const int j = i / (2 * DT), ks = (i / DT) & 1, d = i % DT;
    return *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(tile) +
                                           (2 + j) * (kBlkElems * 2) + d * (32 * kKeys * 2) +
                                           v_lane[ks]);
  };
  auto first_scores = [&](const uint16_t* tile, Scores& sc) {
#pragma unroll
    for (int j = 0; j < 2; ++j) sc[j] = f32x16{};
#pragma unroll
    for (int i = 0; i < 2 * KS; ++i) sc[i & 1] = MM::mma32(read_k(tile, i), qop[i >> 1], sc[i & 1]);
  };
  typedef u32x4 Weights[MM::kParts][4];  // P^T operands of the four 16-key steps
  auto form_p = [&](int e, const Scores& sc, float mref, Weights& pk) {
    const int j = e >> 3, n = 2 * (e & 7);
    uint32_t pw[MM::kParts];
    l = MM::weights(fast_exp2(__builtin_fmaf(sc[j][n], wa.scale, -mref)) * MM::kPScale,
                    fast_exp2(__builtin_fmaf(sc[j][n + 1], wa.scale, -mref)) * MM::kPScale, pw, l);
#pragma unroll
    for (int part = 0; part < MM::kParts; ++part)
      pk[part][2 * j + (n >> 3)][(n & 7) >> 1] = pw[part];
  };

  // Tile t where every row of the wavefront sees all of tiles t and t + 1.
  auto whole_tile = [&](int t, const uint16_t* tile, uint16_t* next, const Scores& sc,
                        Scores& nx) {
    const float mref = m;
    Weights pk;
    u32x4 ring[kA];
#pragma unroll
    for (int j = 0; j < 2; ++j) nx[j] = f32x16{};
#pragma unroll
    for (int i = 0; i < kA; ++i) ring[i] = read_k(tile, i);
    __builtin_amdgcn_sched_group_barrier(kDsRead, kA, 0);
#pragma unroll
    for (int i = 0; i < 2 * KS; ++i) {
      nx[i & 1] = MM::mma32(ring[i % kA], qop[i >> 1], nx[i & 1]);
      __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
      if (i + kA < 2 * KS) {
        ring[i % kA] = read_k(tile, i + kA);
        __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 0);
      }
      if (i * kLoads / (2 * KS) != (i + 1) * kLoads / (2 * KS)) {
        load_piece(i * kLoads / (2 * KS), t + 1, next);
        __builtin_amdgcn_sched_group_barrier(kVmemRead, 1, 0);
      }
#pragma unroll
      for (int e = i * 16 / (2 * KS); e < (i + 1) * 16 / (2 * KS); ++e) {
        form_p(e, sc, mref, pk);
        __builtin_amdgcn_sched_group_barrier(kValu, 2, 0);
        __builtin_amdgcn_sched_group_barrier(kTrans, 2, 0);
        __builtin_amdgcn_sched_group_barrier(kValu, MM::kParts == 2 ? 10 : 2, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kA; ++i) ring[i] = read_v(tile, i);
    __builtin_amdgcn_sched_group_barrier(kDsRead, kA, 1);
    float mx = fmaxf(nx[0][0], nx[1][0]);
#pragma unroll
    for (int i = 0; i < 4 * DT; ++i) {
#pragma unroll
      for (int part = 0; part < MM::kParts; ++part)
        acc[i % DT] = MM::mma32(ring[i % kA], pk[part][i / DT], acc[i % DT]);
      __builtin_amdgcn_sched_group_barrier(kMfma, MM::kParts, 1);
      if (i + kA < 4 * DT) {
        ring[i % kA] = read_v(tile, i + kA);
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

  // Any tile t: its scores are in sc, which then takes those of tile t + 1.
  auto edge_tile = [&](int t, const uint16_t* tile, Scores& sc) {
    if (seen(t)) {
      const float mref = m;
      Weights pk;
#pragma unroll
      for (int e = 0; e < 16; ++e) form_p(e, sc, mref, pk);
#pragma unroll
      for (int i = 0; i < 4 * DT; ++i) {
        const u32x4 vv = read_v(tile, i);
#pragma unroll
        for (int part = 0; part < MM::kParts; ++part)
          acc[i % DT] = MM::mma32(vv, pk[part][i / DT], acc[i % DT]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (t + 1 < t_hi && seen(t + 1)) {
      first_scores(tile, sc);
      mask_scores(t + 1, sc);
      raise(max_of(sc));
    }
  };

  // Infinities and NaN in V of key kt, under the whole weights of the rows that see
  // it: V from the pages (the staged V holds the finite values), the key's score
  // once more.  Rare; key by key, since two tiles' worth of operands would cost the
  // loops above their registers.
  auto add_odd = [&](int kt) {
    const int tb = kt / a.BLOCK;
    int page = a.table[tb];
    page = static_cast<unsigned>(page) < static_cast<unsigned>(a.P) ? page : 0;
    const size_t row = (static_cast<size_t>(page) * a.NKV + kvh) * a.BLOCK + (kt - tb * a.BLOCK);
    const uint16_t* vr = static_cast<const uint16_t*>(a.v_pages) + row * D;
    uint32_t any = 0;
#pragma unroll
    for (int i = 0; i < D / kWave; ++i) any |= odd_halves(vr[i * kWave + lane]);
    if (__builtin_amdgcn_ballot_w64(any != 0) == 0) return;
    const uint16_t* kr = kseg + static_cast<size_t>(kt) * D + 8 * lh;  // (blocks are contiguous)
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const u32x4 kk = *reinterpret_cast<const u32x4*>(kr + 16 * i);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const f32x2 x = MM::widen(kk[e]), y = MM::widen(qop[i][e]);
        s = __builtin_fmaf(x[1], y[1], __builtin_fmaf(x[0], y[0], s));
      }
    }
    s += __shfl_xor(s, 32);
    const float wt = whole_weight(fast_exp2(__builtin_fmaf(s, wa.scale, -m)));
    const bool sees = wa.pos[kt] <= qpos;
#pragma unroll
    for (int d = 0; d < DT; ++d) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const u32x2 x = *reinterpret_cast<const u32x2*>(vr + 32 * d + 8 * i + 4 * lh);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t pair = x[e >> 1];
          const f32x2 v = MM::widen(pair & odd_halves(pair));
          acc[d][4 * i + e] += sees && v[e & 1] != 0.f ? wt * v[e & 1] : 0.f;
        }
      }
    }
  };

  Scores sc_a, sc_b;
  auto landed = [&]() {
    wait_vmem_all();
    lds_barrier();
  };
  if (t_lo < t_hi) {
    look_ahead(t_lo);
#pragma unroll
    for (int i = 0; i < kLoads / 2; ++i) load_piece(i, t_lo - 1, tile_b);
    load_q();
    load_stage(t_lo, tile_a);
    // the first tile's K has landed (gfx9 encoding: vmcnt kLoads, lgkmcnt 15)
    if constexpr (kLoads == 8) __builtin_amdgcn_s_waitcnt(0x0F78);
    else __builtin_amdgcn_s_waitcnt(0x0F74);
    lds_barrier();
    if (seen(t_lo)) {
      first_scores(tile_b, sc_a);
      mask_scores(t_lo, sc_a);
      raise(max_of(sc_a));
    }
  }
  for (int t = t_lo; t < t_hi;) {
    // pairs of tiles that are whole, the one after them (whose scores run
    // ahead) too; otherwise a pair of any kind
    while (t + 2 < t_hi && t - win < 60 && ((whole_bits >> (t - win)) & 7) == 7) {
      landed();
      whole_tile(t, tile_a, tile_b, sc_a, sc_b);
      landed();
      whole_tile(t + 1, tile_b, tile_a, sc_b, sc_a);
      t += 2;
    }
    landed();
    if (t - win >= 60) look_ahead(t);
    if (t + 1 < t_hi) load_stage(t + 1, tile_b);
    edge_tile(t, tile_a, sc_a);
    if (t + 1 >= t_hi) break;
    landed();
    if (t + 2 < t_hi) load_stage(t + 2, tile_a);
    edge_tile(t + 1, tile_b, sc_a);
    t += 2;
  }

  if constexpr (MM::kParts == 2) {
    for (int i = 2 * t_lo + kWave + lane; i < 2 * t_hi; i += kWave) odd_blocks |= odd[i];
  }
  if (MM::kParts == 2 && __builtin_amdgcn_ballot_w64(odd_blocks != 0) != 0) {
    for (int blk = 2 * t_lo; blk < 2 * t_hi; ++blk) {
      if (uniform(odd[blk]) == 0 || uniform(wa.span[blk].x) > q_hi) continue;
      for (int kt = blk * kKeys; kt < min((blk + 1) * kKeys, a.TK); ++kt) add_odd(kt);
    }
  }

  const float lt = l + __shfl_xor(l, 32);
  if (!row_ok) return;
  if (wa.splits == 1) {
    const float inv = lt > 0.f ? 1.f / lt : 0.f;
    uint16_t* o = out + qrow * D + 4 * lh;
#pragma unroll
    for (int d = 0; d < DT; ++d) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        E::store4(o + 32 * d + 8 * i, f32x4{acc[d][4 * i], acc[d][4 * i + 1], acc[d][4 * i + 2],
                                            acc[d][4 * i + 3]} * inv);
    }
    return;
  }
  const size_t p = (static_cast<size_t>(kvh) * wa.R + row) * wa.splits + split;
  float* o = a.part_o + p * D + 4 * lh;
#pragma unroll
  for (int d = 0; d < DT; ++d) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<f32x4*>(o + 32 * d + 8 * i) =
          f32x4{acc[d][4 * i], acc[d][4 * i + 1], acc[d][4 * i + 2], acc[d][4 * i + 3]};
  }
  if (lh == 0) {
    a.part_ml[p * 2 + 0] = m;
    a.part_ml[p * 2 + 1] = lt;
  }
}

// One wavefront per row: merges its key splits (at most 64) into the output.
template <int D, typename E>
__global__ __launch_bounds__(256) void pf_window_combine_kernel(WinArgs wa, uint16_t* out,
                                                                int rows) {
  constexpr int kLanes = D / 4;           // lanes across a row, four dims each
  constexpr int kSide = kWave / kLanes;   // splits side by side
  const PfArgs& a = wa.p;
  const int lane = threadIdx.x & (kWave - 1);
  const int task = blockIdx.x * 4 + uniform(threadIdx.x / kWave);
  if (task >= rows) return;
  const int kvh = task / wa.R;
  const int row = task - kvh * wa.R;
  const int bt = row / a.G;
  const int b = bt / a.TQ;
  const size_t p0 = static_cast<size_t>(task) * wa.splits;
  const bool live = lane < wa.splits;
  const float2 ml = reinterpret_cast<const float2*>(a.part_ml)[p0 + (live ? lane : 0)];
  const float M = wave_max_uniform(live ? ml.x : -INFINITY);
  // (a split that holds no visible key of the row left m = -FLT_MAX, l = 0)
  const float wt = live ? fast_exp2(ml.x - M) : 0.f;
  const float lt = wave_sum_uniform(live ? ml.y * wt : 0.f);
  const int c = lane % kLanes, side = lane / kLanes;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < wa.splits; s0 += 4 * kSide) {
    f32x4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int s = min(s0 + u * kSide + side, wa.splits - 1);
      v[u] = *reinterpret_cast<const f32x4*>(a.part_o + (p0 + s) * D + 4 * c);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int s = s0 + u * kSide + side;
      const float ws = __shfl(wt, s & (kWave - 1));
      if (s < wa.splits) acc += v[u] * ws;
    }
  }
#pragma unroll
  for (int x = kLanes; x < kWave; x <<= 1) {
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] += __shfl_xor(acc[e], x);
  }
  if (side != 0) return;
  const float inv = lt > 0.f ? 1.f / lt : 0.f;
  const size_t qrow =
      (static_cast<size_t>(b) * a.NQ + kvh * a.G + (row - bt * a.G)) * a.TQ + (bt - b * a.TQ);
  E::store4(out + qrow * D + 4 * c, acc * inv);
}

template <int D, typename E, typename TT>
void launch_pf_attention(int hw, dim3 grid, dim3 block, hipStream_t stream, const PfArgs& a) {
  switch (hw) {
    case 8: hipLaunchKernelGGL((pf_attention_kernel<D, 8, E, TT>), grid, block, 0, stream, a); break;
    case 4: hipLaunchKernelGGL((pf_attention_kernel<D, 4, E, TT>), grid, block, 0, stream, a); break;
    case 2: hipLaunchKernelGGL((pf_attention_kernel<D, 2, E, TT>), grid, block, 0, stream, a); break;
    default: hipLaunchKernelGGL((pf_attention_kernel<D, 1, E, TT>), grid, block, 0, stream, a); break;
  }
}
template <typename E>
void launch_pf_attention_e(int D, bool f32_tab, int hw, dim3 grid, dim3 block, hipStream_t stream,
                           const PfArgs& a) {
  if (D == 128) {
    if (f32_tab) launch_pf_attention<128, E, EF32>(hw, grid, block, stream, a);
    else launch_pf_attention<128, E, E>(hw, grid, block, stream, a);
  } else {
    if (f32_tab) launch_pf_attention<64, E, EF32>(hw, grid, block, stream, a);
    else launch_pf_attention<64, E, E>(hw, grid, block, stream, a);
  }
}

// How one call is cut: which kernel, columns per pass, passes, splits and the
// workspace it needs.  voom_position_free_workspace_bytes and the call share
// it, so the two always agree.
struct PfPlan {
  bool mfma;
  int hw;      // kv heads per workgroup (MFMA kernel)
  int ncg, passes, ncp, splits;
  bool window;            // the window kernels
  int row_tiles, nblk;
  size_t o_bytes;         // the partial outputs' bytes (the statistics follow)
  size_t stage_at, pos_at, span_at, odd_at;  // window: the staged blocks in the workspace
  size_t ws_bytes;
};

// kv heads of one workgroup of pf_attention_kernel.
int heads_per_workgroup(int NKV) {
  return NKV % 8 == 0 ? 8 : NKV % 4 == 0 ? 4 : NKV % 2 == 0 ? 2 : 1;
}

// Columns from which staging the pages pays.  The staged route takes about 21 us and
// 1.2 us per 2^19 elements of K (a pass over the pages, launches and fill), hardly
// growing with the columns; the page-walking one is short for few columns and grows
// by a rotation of every key per 16 of them, at a rate of its own in each variant
// (head dim, kv heads per workgroup).  So per variant: `least` columns however many
// keys, and `extra` / e more with e = elements / 2^19, without which the walk is over
// before the staged route's fixed part; eight heads of 128, whose workgroups just
// fill the CUs at 64 columns, stay with the walk there from e = 8 on (`slope` 1: one
// column more per e up to 16).  Measured with either route at 1,128 points of 10 head
// geometries, 300 to 40,000 keys and 40 to 1,000 columns, bf16, walking / staged, us:
// 9q/3kv, D = 64, 5,000 keys: 99 columns 20.1 / 23.1, 177 columns 24.4 / 24.8; 28q/4kv,
// D = 128, 3,000 keys: 63 columns 21.9 / 26.2, 98 columns 28.7 / 27.4; 32q/8kv, 1,500
// keys: 56 columns 20.7 / 21, 64 columns 24.5 / 21.9; 4q/2kv, D = 64, 12,000 keys: 120
// columns 19.8 / 26.8, 200 columns 28 / 26.
struct StageRule {
  int least, extra, slope;
};
constexpr StageRule kStageRules[2][4] = {
    // kv heads per workgroup: 1, 2, 4, 8
    {{48, 140, 0}, {110, 300, 0}, {72, 70, 0}, {65, 60, 0}},  // D = 64
    {{48, 110, 0}, {65, 110, 0}, {56, 110, 0}, {56, 17, 1}},  // D = 128
};
// The staged copy of K and V is scratch of the call, so it is bounded: past
// kWinMaxStage (262,144 keys of 8 heads of 128) the pages are walked.
constexpr long long kWinMaxStage = 1LL << 30;
bool window_pays(long long cols, int TK, int NKV, int D) {
  const long long elems = static_cast<long long>(TK) * NKV * D;
  const StageRule r = kStageRules[D == 128][ilog2(heads_per_workgroup(NKV))];
  const long long e = elems >> 19;
  const long long least = r.least + r.slope * (e < 16 ? e : 16);
  return 4 * elems <= kWinMaxStage && cols >= least &&
         (cols - least) * elems >= static_cast<long long>(r.extra) << 19;
}

size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

PfPlan pf_plan(int B, int NQ, int TQ, int NKV, int D, int TK, int dtype, int num_splits) {
  PfPlan p = {};
  const int NC = NQ / NKV * TQ;
  const int nb = (TK + kKeys - 1) / kKeys;
  p.mfma = dtype != VOOM_DTYPE_F32 && (D == 64 || D == 128);
  p.window = p.mfma && window_pays(static_cast<long long>(B) * NC, TK, NKV, D);
  if (p.window) {
    const long long R = static_cast<long long>(B) * NC;
    p.row_tiles = static_cast<int>((R + kWinTile - 1) / kWinTile);
    p.nblk = (nb + 1) & ~1;
    long long s = num_splits > 0 ? num_splits
                                 : key_splits(static_cast<long long>(NKV) * p.row_tiles,
                                              device_cu_count());
    if (num_splits <= 0 && s > p.nblk / 8) s = p.nblk / 8;  // four 64-key tiles each
    if (s > kWinMaxSplits) s = kWinMaxSplits;
    p.splits = s < 1 ? 1 : static_cast<int>(s);
    const size_t rows = p.splits > 1 ? static_cast<size_t>(NKV) * R * p.splits : 0;
    p.o_bytes = align256(rows * D * sizeof(float));
    p.stage_at = p.o_bytes + align256(rows * 2 * sizeof(float));
    const size_t blocks = static_cast<size_t>(NKV) * p.nblk;
    p.pos_at = p.stage_at + blocks * 2 * kKeys * D * sizeof(uint16_t);
    p.span_at = p.pos_at + align256(static_cast<size_t>(p.nblk) * kKeys * sizeof(int32_t));
    p.odd_at = p.span_at + align256(static_cast<size_t>(p.nblk) * sizeof(int2));
    p.ws_bytes = p.odd_at + align256(blocks * sizeof(int32_t));
    return p;
  }
  p.hw = heads_per_workgroup(NKV);
  p.ncg = p.mfma ? kCols : (NC < kGenOut / D ? NC : kGenOut / D);
  p.passes = (NC + p.ncg - 1) / p.ncg;
  p.ncp = p.passes * p.ncg;
  // default: 8 wavefronts per CU for the MFMA kernel, 2 workgroups of 4
  // wavefronts per CU for the generic one
  const long long target = p.mfma ? 8LL * device_cu_count() : 2LL * device_cu_count();
  const long long per = static_cast<long long>(B) * NKV * p.passes;
  long long s = num_splits > 0 ? num_splits : (target + per - 1) / per;
  if (s > nb) s = nb;
  p.splits = s < 1 ? 1 : static_cast<int>(s);
  const size_t rows = static_cast<size_t>(B) * NKV * p.splits * p.ncp;
  p.o_bytes = align256(rows * D * sizeof(float));
  p.ws_bytes = p.o_bytes + rows * 2 * sizeof(float);
  return p;
}

// Stages the pages and runs the window kernels (a.part_* set).
template <int D, typename E>
int launch_pf_window(const PfPlan& p, const PfArgs& a, char* ws, bool f32_tab, void* out,
                     hipStream_t stream) {
  WinArgs w;
  w.p = a;
  const size_t blocks = static_cast<size_t>(a.NKV) * p.nblk;
  w.k_blk = reinterpret_cast<uint16_t*>(ws + p.stage_at);
  w.v_blk = w.k_blk + blocks * kKeys * D;
  w.pos = reinterpret_cast<int32_t*>(ws + p.pos_at);
  w.span = reinterpret_cast<int2*>(ws + p.span_at);
  w.odd = reinterpret_cast<int32_t*>(ws + p.odd_at);
  w.nblk = p.nblk;
  w.R = a.B * a.NC;
  w.row_tiles = p.row_tiles;
  w.splits = p.splits;
  w.work = a.NKV * p.row_tiles * p.splits;
  w.per_xcd = (w.work + 7) / 8;
  w.xcd_cus = device_cu_count() / 8;
  w.scale = a.scale == 0.f ? 1.f : fabsf(a.scale_log2e);
  w.q_keep = a.scale == 0.f ? 0u : 0xffffffffu;
  w.q_flip = a.scale < 0.f ? 0x80008000u : 0u;
  const dim3 grid(static_cast<unsigned>(p.nblk) * a.NKV);
  if (f32_tab) hipLaunchKernelGGL((pf_stage_kernel<D, E, EF32>), grid, dim3(256), 0, stream, w);
  else hipLaunchKernelGGL((pf_stage_kernel<D, E, E>), grid, dim3(256), 0, stream, w);
  hipLaunchKernelGGL((pf_window_kernel<D, E>), dim3(8u * static_cast<unsigned>(w.per_xcd)),
                     dim3(kWinWaves * kWave), 0, stream, w, static_cast<uint16_t*>(out));
  int rc = VOOM_LAUNCH_CHECK("position_free_attention: window launch");
  if (rc || p.splits == 1) return rc;
  const int rows = a.NKV * w.R;
  hipLaunchKernelGGL((pf_window_combine_kernel<D, E>), dim3(static_cast<unsigned>((rows + 3) / 4)),
                     dim3(256), 0, stream, w, static_cast<uint16_t*>(out), rows);
  return VOOM_LAUNCH_CHECK("position_free_attention: combine launch");
}

bool pf_dtype_ok(int dt) {
  return dt == VOOM_DTYPE_BF16 || dt == VOOM_DTYPE_F16 || dt == VOOM_DTYPE_F32;
}

// Launches the generic kernel with `lds` bytes of dynamic LDS (up to 85 KB at
// head_dim 256), raising the kernel's dynamic-LDS limit first when the
// request is above the 64 KB default.
template <typename E, typename TT>
int launch_pf_generic_tt(dim3 grid, size_t lds, hipStream_t stream, const PfArgs& a) {
  if (lds > 65536) {
    const int rc = check_hip(
        hipFuncSetAttribute(reinterpret_cast<const void*>(&pf_generic_kernel<E, TT>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)),
        "position_free_attention: dynamic LDS limit");
    if (rc) return rc;
  }
  hipLaunchKernelGGL((pf_generic_kernel<E, TT>), grid, dim3(kGenThreads), lds, stream, a);
  return VOOM_LAUNCH_CHECK("position_free_attention: kernel launch");
}

template <typename E>
int launch_pf_generic(int table_dtype, dim3 grid, size_t lds, hipStream_t stream,
                      const PfArgs& a) {
  return table_dtype == VOOM_DTYPE_F32 ? launch_pf_generic_tt<E, EF32>(grid, lds, stream, a)
                                       : launch_pf_generic_tt<E, E>(grid, lds, stream, a);
}

}  // namespace
}  // namespace voom

using namespace voom;

extern "C" size_t voom_position_free_workspace_bytes(int batch, int num_q_heads, int num_queries,
                                                     int num_kv_heads, int head_dim,
                                                     int num_keys, int dtype, int num_splits) {
  if (batch <= 0 || num_q_heads <= 0 || num_queries <= 0 || num_kv_heads <= 0 ||
      num_q_heads % num_kv_heads || head_dim <= 0 || head_dim % 32 || head_dim > kGenMaxD ||
      num_keys < 0 || !pf_dtype_ok(dtype))
    return 0;
  return pf_plan(batch, num_q_heads, num_queries, num_kv_heads, head_dim, num_keys, dtype,
                 num_splits)
      .ws_bytes;
}

extern "C" int voom_position_free_attention(
    const void* q, const void* k_pages, const void* v_pages, const int32_t* block_table,
    const int32_t* key_positions, const int32_t* query_positions, const void* cos_table,
    const void* sin_table, void* out, void* workspace, size_t ws_bytes, int batch,
    int num_q_heads, int num_queries, int num_kv_heads, int head_dim, int block_size,
    int num_pages, int num_keys, int max_position, int dtype, int table_dtype, float scale,
    int num_splits, hipStream_t stream) {
  const char* who = "position_free_attention";
  VOOM_REQUIRE(q && k_pages && v_pages && out && workspace && query_positions && cos_table &&
                   sin_table,
               "%s: null pointer argument", who);
  VOOM_REQUIRE(num_keys == 0 || (block_table && key_positions), "%s: null key arrays", who);
  VOOM_REQUIRE(batch > 0 && num_queries > 0 && num_kv_heads > 0 && num_q_heads > 0 &&
                   num_q_heads % num_kv_heads == 0,
               "%s: unsupported head or position geometry", who);
  VOOM_REQUIRE(head_dim > 0 && head_dim % 32 == 0 && head_dim <= kGenMaxD,
               "%s: head_dim %d unsupported (a multiple of 32 up to %d)", who, head_dim,
               kGenMaxD);
  VOOM_REQUIRE(pf_dtype_ok(dtype), "%s: unsupported element type code %d", who, dtype);
  VOOM_REQUIRE(table_dtype == VOOM_DTYPE_F32 || table_dtype == dtype,
               "%s: RoPE cache must be FP32 or match the Q/K/V dtype", who);
  VOOM_REQUIRE(block_size > 0 && num_pages > 0 && num_keys >= 0 && num_keys <= (1 << 30) &&
                   max_position > 0,
               "%s: bad page or position geometry", who);
  const PfPlan p = pf_plan(batch, num_q_heads, num_queries, num_kv_heads, head_dim, num_keys,
                           dtype, num_splits);
  VOOM_REQUIRE(ws_bytes >= p.ws_bytes, "%s: workspace %zu bytes < required %zu", who, ws_bytes,
               p.ws_bytes);
  VOOM_REQUIRE(reinterpret_cast<uintptr_t>(q) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(k_pages) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(v_pages) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(cos_table) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(sin_table) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(workspace) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(out) % 16 == 0,
               "%s: tensors must be 16-byte aligned", who);
  const int G = num_q_heads / num_kv_heads;
  const long long NC = static_cast<long long>(G) * num_queries;
  const long long segs = static_cast<long long>(batch) * num_kv_heads;
  const long long nwork = p.window ? static_cast<long long>(num_kv_heads) * p.row_tiles * p.splits
                                   : segs * p.splits / (p.mfma ? p.hw : 1);
  const long long grid_x =
      p.window || p.passes == 1 ? nwork : (nwork + 7) / 8 * 8 * p.passes;
  VOOM_REQUIRE(NC < (1LL << 24) && grid_x < (1LL << 30) && segs * NC * (head_dim / 32) < (1LL << 31),
               "%s: grid too large", who);

  PfArgs a;
  a.q = q;
  a.k_pages = k_pages;
  a.v_pages = v_pages;
  a.table = block_table;
  a.k_pos = key_positions;
  a.q_pos = query_positions;
  a.cos_t = cos_table;
  a.sin_t = sin_table;
  a.part_o = static_cast<float*>(workspace);
  a.part_ml = reinterpret_cast<float*>(static_cast<char*>(workspace) + p.o_bytes);
  a.B = batch;
  a.NQ = num_q_heads;
  a.TQ = num_queries;
  a.NKV = num_kv_heads;
  a.G = G;
  a.D = head_dim;
  a.BLOCK = block_size;
  a.P = num_pages;
  a.TK = num_keys;
  a.max_pos = max_position;
  a.splits = p.splits;
  a.NC = static_cast<int>(NC);
  a.ncg = p.ncg;
  a.passes = p.passes;
  a.NCP = p.ncp;
  a.nwork = static_cast<int>(nwork);
  a.scale = scale;
  a.scale_log2e = scale * kLog2e;
  const dim3 grid(static_cast<unsigned>(grid_x));
  int rc;
  if (p.window) {
    char* ws = static_cast<char*>(workspace);
    const bool f32_tab = table_dtype == VOOM_DTYPE_F32;
    if (dtype == VOOM_DTYPE_BF16)
      return head_dim == 128 ? launch_pf_window<128, EBf16>(p, a, ws, f32_tab, out, stream)
                             : launch_pf_window<64, EBf16>(p, a, ws, f32_tab, out, stream);
    return head_dim == 128 ? launch_pf_window<128, EF16>(p, a, ws, f32_tab, out, stream)
                           : launch_pf_window<64, EF16>(p, a, ws, f32_tab, out, stream);
  }
  if (p.mfma) {
    const dim3 block(static_cast<unsigned>(p.hw * kWave));
    const bool f32_tab = table_dtype == VOOM_DTYPE_F32;
    if (dtype == VOOM_DTYPE_BF16)
      launch_pf_attention_e<EBf16>(head_dim, f32_tab, p.hw, grid, block, stream, a);
    else
      launch_pf_attention_e<EF16>(head_dim, f32_tab, p.hw, grid, block, stream, a);
    rc = VOOM_LAUNCH_CHECK("position_free_attention: kernel launch");
  } else {
    const size_t lds = static_cast<size_t>(gen_lds(head_dim, p.ncg).words) * 4;
    if (dtype == VOOM_DTYPE_F32) rc = launch_pf_generic<EF32>(table_dtype, grid, lds, stream, a);
    else if (dtype == VOOM_DTYPE_F16) rc = launch_pf_generic<EF16>(table_dtype, grid, lds, stream, a);
    else rc = launch_pf_generic<EBf16>(table_dtype, grid, lds, stream, a);
  }
  if (rc) return rc;
  const dim3 grid_red(static_cast<unsigned>(segs * NC * (head_dim / kRedDims)));
  const dim3 block_red(kRedWaves * kWave);
  if (dtype == VOOM_DTYPE_F32) {
    hipLaunchKernelGGL(pf_reduce_kernel<EF32>, grid_red, block_red, 0, stream, a,
                       static_cast<float*>(out));
  } else if (dtype == VOOM_DTYPE_F16) {
    hipLaunchKernelGGL(pf_reduce_kernel<EF16>, grid_red, block_red, 0, stream, a,
                       static_cast<uint16_t*>(out));
  } else {
    hipLaunchKernelGGL(pf_reduce_kernel<EBf16>, grid_red, block_red, 0, stream, a,
                       static_cast<uint16_t*>(out));
  }
  return VOOM_LAUNCH_CHECK("position_free_attention: reduce launch");
}
