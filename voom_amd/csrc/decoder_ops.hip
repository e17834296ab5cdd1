// Fused per-token ops of the config-1 decoder harness (a Llama-style block
// around the paged attention), so that one decode step is a short chain of
// launches: the residual add + RMSNorm, RoPE of q and k together with the
// split of the fused qkv projection into the attention layouts, SwiGLU, and
// the one-token projections (GEMV, optionally with SwiGLU fused).
// They restate the block math of runtime/layer_runner.py (rms_norm :263,309,
// rope :99-103, _silu_mul :43-46 and :188) with Hugging Face LlamaForCausalLM's
// cast order -- the reference its parity tests use:
//   rms_norm:  y = bf16(w * bf16(x * rsqrt(mean(x^2) + eps)))   stats in fp32
//   rope:      rotate-half, fp32 products from fp32 cos/sin tables, bf16 out
//   swiglu:    bf16(bf16(g / (1 + exp(-g))) * u)
// All memory-bound; each kernel reads and writes its rows once.
#include "common.h"

namespace voom {
namespace {

constexpr int kRowThreads = 256;

// bf16(a + d) of two 16-byte chunks.
__device__ __forceinline__ u32x4 sum_chunks(u32x4 a, u32x4 d) {
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float lo = bf2f(static_cast<uint16_t>(a[w] & 0xffffu)) +
                     bf2f(static_cast<uint16_t>(d[w] & 0xffffu));
    const float hi = bf2f(static_cast<uint16_t>(a[w] >> 16)) +
                     bf2f(static_cast<uint16_t>(d[w] >> 16));
    a[w] = pack_bf16x2(lo, hi);
  }
  return a;
}

// 16-byte chunk at col of bf16(x + delta) (of x alone without delta).
__device__ __forceinline__ u32x4 add_chunk(const uint16_t* __restrict__ x,
                                           const uint16_t* __restrict__ delta, int col) {
  const u32x4 a = *reinterpret_cast<const u32x4*>(x + col);
  return delta ? sum_chunks(a, *reinterpret_cast<const u32x4*>(delta + col)) : a;
}

// Sum of squares of one chunk's 8 values added to ss, in element order with
// explicit fused multiply-adds.  The row statistics of every kernel here are
// built the same way -- lane l of one wavefront takes chunks l, l + 64, ...
// in order, then the lanes are summed by wave_sum_uniform (and
// 1 / sqrt(ss / hidden + eps)) -- so a fused normalisation is bit-identical
// to add_rms_norm_kernel's.
__device__ __forceinline__ float chunk_sumsq(u32x4 a, float ss) {
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float lo = bf2f(static_cast<uint16_t>(a[w] & 0xffffu));
    const float hi = bf2f(static_cast<uint16_t>(a[w] >> 16));
    ss = __builtin_fmaf(lo, lo, ss);
    ss = __builtin_fmaf(hi, hi, ss);
  }
  return ss;
}
__device__ __forceinline__ float rms_inv(float ss_lane, int hidden, float eps) {
  const float ss = wave_sum_uniform(ss_lane);
  return 1.f / sqrtf(ss / static_cast<float>(hidden) + eps);
}
// bf16(w * bf16(v * inv)) for one chunk, as packed bf16.
__device__ __forceinline__ u32x4 norm_chunk(u32x4 a, u32x4 wv, float inv) {
  u32x4 o;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float n0 = bf2f(f2bf(bf2f(static_cast<uint16_t>(a[w] & 0xffffu)) * inv));
    const float n1 = bf2f(f2bf(bf2f(static_cast<uint16_t>(a[w] >> 16)) * inv));
    o[w] = pack_bf16x2(bf2f(static_cast<uint16_t>(wv[w] & 0xffffu)) * n0,
                       bf2f(static_cast<uint16_t>(wv[w] >> 16)) * n1);
  }
  return o;
}

// One workgroup per row of `hidden` bf16 values (hidden % 8 == 0, <= 8192).
// With delta, the row first becomes bf16(x + delta) and is written back.
// Wavefront 0 computes the row statistics in the canonical order above.
__global__ __launch_bounds__(kRowThreads) void add_rms_norm_kernel(
    uint16_t* __restrict__ x, const uint16_t* __restrict__ delta,
    const uint16_t* __restrict__ weight, uint16_t* __restrict__ out, int hidden, float eps) {
  __shared__ float s_inv;
  const size_t row = blockIdx.x;
  uint16_t* xr = x + row * hidden;
  const uint16_t* dr = delta ? delta + row * hidden : nullptr;
  uint16_t* orow = out + row * hidden;
  const int chunks = hidden / 8;
  if (threadIdx.x < kWave) {
    float ss = 0.f;
    for (int c = threadIdx.x; c < chunks; c += kWave) ss = chunk_sumsq(add_chunk(xr, dr, 8 * c), ss);
    const float inv = rms_inv(ss, hidden, eps);
    if (threadIdx.x == 0) s_inv = inv;
  }
  __syncthreads();  // every read of the unmodified row is done
  const float inv = s_inv;
  for (int c = threadIdx.x; c < chunks; c += kRowThreads) {
    const u32x4 a = add_chunk(xr, dr, 8 * c);
    if (dr) *reinterpret_cast<u32x4*>(xr + 8 * c) = a;
    const u32x4 wv = *reinterpret_cast<const u32x4*>(weight + 8 * c);
    *reinterpret_cast<u32x4*>(orow + 8 * c) = norm_chunk(a, wv, inv);
  }
}

// qkv [B * L, (nq + 2 nkv) * hd] -> q [B, nq, L, hd], k and v [B, nkv, L, hd];
// q and k rotated (rotate-half) with the fp32 tables cos/sin [L, hd]
// (cos[i] = cos[i + hd/2]).  One thread per (row, head, dim pair).
__global__ __launch_bounds__(kRowThreads) void rope_split_kernel(
    const uint16_t* __restrict__ qkv, const float* __restrict__ cos_t,
    const float* __restrict__ sin_t, uint16_t* __restrict__ q, uint16_t* __restrict__ k,
    uint16_t* __restrict__ v, int B, int L, int nq, int nkv, int hd) {
  const int half = hd / 2;
  const int heads = nq + 2 * nkv;
  const long long idx = static_cast<long long>(blockIdx.x) * kRowThreads + threadIdx.x;
  const long long total = static_cast<long long>(B) * L * heads * half;
  if (idx >= total) return;
  const int i = static_cast<int>(idx % half);
  const long long rh = idx / half;
  const int h = static_cast<int>(rh % heads);
  const int row = static_cast<int>(rh / heads);
  const int b = row / L;
  const int l = row - b * L;
  const uint16_t* src = qkv + (static_cast<size_t>(row) * heads + h) * hd;
  const float x1 = bf2f(src[i]);
  const float x2 = bf2f(src[i + half]);
  uint16_t* dst;
  if (h < nq) {
    dst = q + ((static_cast<size_t>(b) * nq + h) * L + l) * hd;
  } else if (h < nq + nkv) {
    dst = k + ((static_cast<size_t>(b) * nkv + (h - nq)) * L + l) * hd;
  } else {
    dst = v + ((static_cast<size_t>(b) * nkv + (h - nq - nkv)) * L + l) * hd;
    dst[i] = src[i];
    dst[i + half] = src[i + half];
    return;
  }
  {
    // x * cos + rotate_half(x) * sin with each product and the sum rounded as
    // separate fp32 ops (no fused multiply-add), as torch evaluates it
#pragma clang fp contract(off)
    const float c0 = cos_t[static_cast<size_t>(l) * hd + i];
    const float s0 = sin_t[static_cast<size_t>(l) * hd + i];
    const float c1 = cos_t[static_cast<size_t>(l) * hd + i + half];
    const float s1 = sin_t[static_cast<size_t>(l) * hd + i + half];
    const float a0 = x1 * c0;
    const float b0 = -x2 * s0;
    const float a1 = x2 * c1;
    const float b1 = x1 * s1;
    dst[i] = f2bf(a0 + b0);
    dst[i + half] = f2bf(a1 + b1);
  }
}

// gate_up [rows, 2 I] (gate first) -> out [rows, I]; 8 values per thread.
__global__ __launch_bounds__(kRowThreads) void silu_mul_kernel(
    const uint16_t* __restrict__ gate_up, uint16_t* __restrict__ out, int rows, int inter) {
  const long long idx = static_cast<long long>(blockIdx.x) * kRowThreads + threadIdx.x;
  const int per_row = inter / 8;
  if (idx >= static_cast<long long>(rows) * per_row) return;
  const int row = static_cast<int>(idx / per_row);
  const int c = static_cast<int>(idx - static_cast<long long>(row) * per_row) * 8;
  const uint16_t* gr = gate_up + static_cast<size_t>(row) * 2 * inter;
  const u32x4 g = *reinterpret_cast<const u32x4*>(gr + c);
  const u32x4 u = *reinterpret_cast<const u32x4*>(gr + inter + c);
  u32x4 o;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    float r[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float gv = bf2f(static_cast<uint16_t>(e ? g[w] >> 16 : g[w] & 0xffffu));
      const float uv = bf2f(static_cast<uint16_t>(e ? u[w] >> 16 : u[w] & 0xffffu));
      const float s = bf2f(f2bf(gv / (1.f + expf(-gv))));
      r[e] = s * uv;
    }
    o[w] = pack_bf16x2(r[0], r[1]);
  }
  *reinterpret_cast<u32x4*>(out + static_cast<size_t>(row) * inter + c) = o;
}

// One-token projection: y[r] = bf16(sum_k W[r][k] x[k]) with W [N, K] bf16
// row-major (a torch Linear weight), x [K], fp32 sums.  Decode runs these at
// one row of activations, where a GEMM tiling reads the weights at a fraction
// of the bandwidth; here each wavefront takes 4 weight rows, every lane holds
// KC 16-byte chunks of x (chunks lane, lane + 64, ...) in registers and reads
// the same chunks of its 4 rows (coalesced 1 KB per row per step, all 4 x KC
// loads in flight, non-temporal: each weight byte is used once per token),
// and the 4 dot products are summed across the lanes.
// SWIGLU: W is the fused [gate; up] weight [2I, K] and y [I] is
// bf16(bf16(silu(g)) * u) with g, u the bf16-rounded projections of rows r
// and I + r -- the projection followed by silu_mul_kernel's math; a wave then
// takes 2 gate and the 2 matching up rows.
// The projection input of one lane: chunks lane, lane + 64, ... of x (and of
// delta and ln when the residual-add + RMSNorm prologue is on).  The raw
// loads are issued first, then the weight loads, then the input is finished
// while the weights are still in flight: the prologue costs no second memory
// round trip.
template <int KC>
struct GemvInput {
  u32x4 x[KC], d[KC], ln[KC];
};

template <int KC, bool NORM>
__device__ __forceinline__ void gemv_fetch_x(const uint16_t* __restrict__ x,
                                             const uint16_t* __restrict__ delta,
                                             const uint16_t* __restrict__ ln, int chunks, int lane,
                                             GemvInput<KC>& in) {
  // every lane loads (lanes past the row reread its last chunk and are
  // masked later): straight-line loads let the compiler wait for exactly
  // the ones it needs
  const uint16_t* d = delta ? delta : x;
#pragma unroll
  for (int j = 0; j < KC; ++j) {
    const int c = min(lane + kWave * j, chunks - 1);
    in.x[j] = *reinterpret_cast<const u32x4*>(x + 8 * c);
    if (NORM) {
      in.d[j] = *reinterpret_cast<const u32x4*>(d + 8 * c);
      in.ln[j] = *reinterpret_cast<const u32x4*>(ln + 8 * c);
    }
  }
}

// Plain (ln == nullptr): the input is x.  Otherwise it is add_rms_norm_kernel's
// output, bit for bit: v = bf16(x + delta) (x without delta), input =
// bf16(ln * bf16(v * rsqrt(mean(v^2) + eps))), with v also stored to x_out
// (when given) by one wavefront of the grid.
template <int KC, bool NORM>
__device__ __forceinline__ void gemv_finish_x(const GemvInput<KC>& in, bool has_delta, float eps,
                                              uint16_t* __restrict__ x_out, bool writer, int k,
                                              int lane, float (&xv)[KC][8]) {
  const int chunks = k / 8;
  u32x4 v[KC];
#pragma unroll
  for (int j = 0; j < KC; ++j) {
    v[j] = lane + kWave * j < chunks ? in.x[j] : u32x4{0u, 0u, 0u, 0u};
    if (NORM) {
      // the sum is formed either way and selected: a branch here lets the
      // compiler sink the delta loads into it, behind a wait for the weights
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float lo = bf2f(static_cast<uint16_t>(v[j][w] & 0xffffu)) +
                         bf2f(static_cast<uint16_t>(in.d[j][w] & 0xffffu));
        const float hi = bf2f(static_cast<uint16_t>(v[j][w] >> 16)) +
                         bf2f(static_cast<uint16_t>(in.d[j][w] >> 16));
        const uint32_t sum = pack_bf16x2(lo, hi);
        v[j][w] = has_delta ? sum : v[j][w];
      }
    }
  }
  if (NORM) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < KC; ++j) {
      if (lane + kWave * j < chunks) ss = chunk_sumsq(v[j], ss);
    }
    const float inv = rms_inv(ss, k, eps);
#pragma unroll
    for (int j = 0; j < KC; ++j) {
      const int c = lane + kWave * j;
      if (c < chunks) {
        if (writer && x_out) *reinterpret_cast<u32x4*>(x_out + 8 * c) = v[j];
        v[j] = norm_chunk(v[j], in.ln[j], inv);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < KC; ++j) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      xv[j][2 * e] = bf2f(static_cast<uint16_t>(v[j][e] & 0xffffu));
      xv[j][2 * e + 1] = bf2f(static_cast<uint16_t>(v[j][e] >> 16));
    }
  }
}

// Loads of 4 weight rows (non-temporal: each weight byte is read once per
// token).
template <int KC>
__device__ __forceinline__ void gemv_fetch_w(const uint16_t* __restrict__ w, const int (&rows)[4],
                                             int k, int chunks, int lane, u32x4 (&wv)[4][KC]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint16_t* wr = w + static_cast<size_t>(rows[i]) * k;
#pragma unroll
    for (int j = 0; j < KC; ++j) {
      const int c = min(lane + kWave * j, chunks - 1);  // see gemv_fetch_x
      wv[i][j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wr + 8 * c));
    }
  }
}

// Dot products of the 4 weight rows with x, summed over the wave (every lane
// gets the 4 sums); chunks past the row (lane + 64 j >= chunks) add nothing.
template <int KC>
__device__ __forceinline__ void gemv_dot4(const u32x4 (&wv)[4][KC], const float (&xv)[KC][8],
                                          int chunks, int lane, float (&acc)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < KC; ++j) {
      if (lane + kWave * j >= chunks) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s += bf2f(static_cast<uint16_t>(wv[i][j][e] & 0xffffu)) * xv[j][2 * e];
        s += bf2f(static_cast<uint16_t>(wv[i][j][e] >> 16)) * xv[j][2 * e + 1];
      }
    }
    acc[i] = wave_sum_uniform(s);
  }
}

// One wavefront's projection of rows[0..3]: input fetch, weight fetch, input
// finish, dot products.
template <int KC, bool NORM>
__device__ __forceinline__ void gemv_rows(const uint16_t* __restrict__ w,
                                          const uint16_t* __restrict__ x,
                                          const uint16_t* __restrict__ delta,
                                          const uint16_t* __restrict__ ln, float eps,
                                          uint16_t* __restrict__ x_out, bool writer,
                                          const int (&rows)[4], int k, int lane,
                                          float (&acc)[4]) {
  const int chunks = k / 8;
  GemvInput<KC> in;
  gemv_fetch_x<KC, NORM>(x, delta, ln, chunks, lane, in);
  u32x4 wv[4][KC];
  gemv_fetch_w<KC>(w, rows, k, chunks, lane, wv);
  float xv[KC][8];
  gemv_finish_x<KC, NORM>(in, delta != nullptr, eps, x_out, writer, k, lane, xv);
  gemv_dot4<KC>(wv, xv, chunks, lane, acc);
}

template <int KC, bool SWIGLU, bool NORM>
__global__ __launch_bounds__(kRowThreads) void gemv_kernel(
    const uint16_t* __restrict__ w, const uint16_t* __restrict__ x,
    const uint16_t* __restrict__ delta, const uint16_t* __restrict__ ln, float eps,
    uint16_t* __restrict__ x_out, uint16_t* __restrict__ y, int n, int k) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = blockIdx.x * (kRowThreads / kWave) + (threadIdx.x / kWave);
  // rows of this wave: plain 4r..4r+3; SwiGLU gate 2r, 2r+1 and up n + 2r, n + 2r + 1
  // (rows past the end read row `first` again; their sums are not stored)
  const int first = SWIGLU ? 2 * wave : 4 * wave;
  if (first >= n) return;
  int rows[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int local = SWIGLU ? (i & 1) : i;
    const int r = first + local < n ? first + local : first;
    rows[i] = SWIGLU && i >= 2 ? n + r : r;
  }
  float acc[4];
  gemv_rows<KC, NORM>(w, x, delta, ln, eps, x_out, wave == 0, rows, k, lane, acc);
  if (lane == 0) {
    if (SWIGLU) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (first + i < n) {
          const float g = bf2f(f2bf(acc[i]));
          const float u = bf2f(f2bf(acc[2 + i]));
          const float sg = bf2f(f2bf(g / (1.f + expf(-g))));
          y[first + i] = f2bf(sg * u);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (first + i < n) y[first + i] = f2bf(acc[i]);
      }
    }
  }
}

// The fused qkv projection of one decode token [(nq + 2 nkv) hd, k] . x, the
// RoPE of its q and k heads and the page write of k and v: wave w of head h
// takes rows d, d + 1, d + hd/2, d + hd/2 + 1 of the head (d = 2 (w % (hd/4))),
// so both halves of each rotated pair are in the wave.  The projection is
// rounded to bf16 before the rotation and the rotation rounds each product
// and the sum (rope_split_kernel's formula), so q, k and v are bit-identical
// to the projection, voom_rope_split and voom_append_kv in sequence.  k and v
// land at position *pos of the sequence through its block-table row, in the
// pool layouts of voom_append_kv.
template <int KC, bool NORM>
__global__ __launch_bounds__(kRowThreads) void qkv_rope_append_kernel(
    const uint16_t* __restrict__ w, const uint16_t* __restrict__ x,
    const uint16_t* __restrict__ delta, const uint16_t* __restrict__ ln, float eps,
    uint16_t* __restrict__ x_out,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t, uint16_t* __restrict__ q,
    uint16_t* __restrict__ k_pool, uint16_t* __restrict__ v_pool,
    const int32_t* __restrict__ table_row, const int32_t* __restrict__ pos_ptr, int nq, int nkv,
    int hd, int k, int pt_shift, int max_pages, int num_slots, int rope_rows) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = blockIdx.x * (kRowThreads / kWave) + (threadIdx.x / kWave);
  const int half = hd / 2;
  const int per_head = half / 2;
  const int h = wave / per_head;
  if (h >= nq + 2 * nkv) return;
  const int d = 2 * (wave - h * per_head);
  const int rows[4] = {h * hd + d, h * hd + d + 1, h * hd + d + half, h * hd + d + half + 1};
  float acc[4];
  gemv_rows<KC, NORM>(w, x, delta, ln, eps, x_out, wave == 0, rows, k, lane, acc);
  if (lane >= 2) return;
  // lane e handles dims d + e and d + e + half
  const float x1 = bf2f(f2bf(acc[lane]));
  const float x2 = bf2f(f2bf(acc[2 + lane]));
  const int i = d + lane;
  uint16_t o1, o2;
  if (h < nq + nkv) {
#pragma clang fp contract(off)
    if (rope_rows > 0) {  // tables: the row of the token's position (clamped)
      const int r = min(max(*pos_ptr, 0), rope_rows - 1);
      cos_t += static_cast<size_t>(r) * hd;
      sin_t += static_cast<size_t>(r) * hd;
    }
    const float a0 = x1 * cos_t[i];
    const float b0 = -x2 * sin_t[i];
    const float a1 = x2 * cos_t[i + half];
    const float b1 = x1 * sin_t[i + half];
    o1 = f2bf(a0 + b0);
    o2 = f2bf(a1 + b1);
  } else {
    o1 = f2bf(x1);
    o2 = f2bf(x2);
  }
  if (h < nq) {
    q[static_cast<size_t>(h) * hd + i] = o1;
    q[static_cast<size_t>(h) * hd + i + half] = o2;
    return;
  }
  const int pos = *pos_ptr;
  if (pos < 0) return;
  const int page = pos >> pt_shift;
  if (page >= max_pages) return;
  const int slot = table_row[page];
  if (static_cast<unsigned>(slot) >= static_cast<unsigned>(num_slots)) return;
  const int off = pos & ((1 << pt_shift) - 1);
  const bool is_k = h < nq + nkv;
  const int kvh = is_k ? h - nq : h - nq - nkv;
  const size_t head_page = static_cast<size_t>(slot) * nkv + kvh;
  if (is_k) {
    uint16_t* kr = k_pool + ((head_page << pt_shift) + off) * hd;
    kr[i] = o1;
    kr[i + half] = o2;
  } else {
    const int vb_shift = pt_shift < 5 ? pt_shift : 5;
    const size_t blk = (head_page << (pt_shift - vb_shift)) + (off >> vb_shift);
    const int col = off & ((1 << vb_shift) - 1);
    v_pool[((blk * hd + i) << vb_shift) + col] = o1;
    v_pool[((blk * hd + i + half) << vb_shift) + col] = o2;
  }
}

// Greedy sampling key of one bf16 logit: larger keys are larger logits, and
// among equal logits the lower index; -0 counts as +0 and every NaN as the
// largest value, as torch.argmax orders them.
__device__ __forceinline__ uint64_t logit_key(uint16_t bits, int idx) {
  if ((bits & 0x7fffu) == 0) bits = 0;
  if ((bits & 0x7f80u) == 0x7f80u && (bits & 0x7fu)) bits = 0x7fc0u;
  const uint32_t f = static_cast<uint32_t>(bits) << 16;
  const uint32_t ordered = f ^ ((f >> 31) ? 0xffffffffu : 0x80000000u);
  return (static_cast<uint64_t>(ordered) << 32) | (0xffffffffu - static_cast<uint32_t>(idx));
}

// The lm_head projection of one row with its argmax: each wavefront projects
// 4 vocabulary rows (the GEMV above, optional final-norm prologue), keys its
// bf16 logits and the workgroup's best key goes to keys[blockIdx.x].  No
// logits are stored.
template <int KC, bool NORM>
__global__ __launch_bounds__(kRowThreads) void gemv_argmax_kernel(
    const uint16_t* __restrict__ w, const uint16_t* __restrict__ x,
    const uint16_t* __restrict__ delta, const uint16_t* __restrict__ ln, float eps,
    uint64_t* __restrict__ keys, int n, int k) {
  __shared__ uint64_t s_key[kRowThreads / kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wib = threadIdx.x / kWave;
  const int first = 4 * (blockIdx.x * (kRowThreads / kWave) + wib);
  uint64_t best = 0;  // below every real key
  if (first < n) {  // uniform over the wavefront
    int rows[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) rows[i] = first + i < n ? first + i : first;
    float acc[4];
    gemv_rows<KC, NORM>(w, x, delta, ln, eps, nullptr, false, rows, k, lane, acc);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (first + i < n) {
        const uint64_t key = logit_key(f2bf(acc[i]), first + i);
        best = key > best ? key : best;
      }
    }
  }
  if (lane == 0) s_key[wib] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t m = s_key[0];
#pragma unroll
    for (int i = 1; i < kRowThreads / kWave; ++i) m = s_key[i] > m ? s_key[i] : m;
    keys[blockIdx.x] = m;
  }
}

// One workgroup: the best of nkeys keys; its index goes to token[0] and,
// when given, token_copy[0].
__global__ __launch_bounds__(kRowThreads) void argmax_finish_kernel(
    const uint64_t* __restrict__ keys, int nkeys, int64_t* __restrict__ token,
    int64_t* __restrict__ token_copy) {
  __shared__ uint64_t s_key[kRowThreads];
  constexpr int kPer = 16;  // loads in flight per thread
  uint64_t m = 0;
  for (int base = 0; base < nkeys; base += kPer * kRowThreads) {
    uint64_t v[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int i = base + j * kRowThreads + threadIdx.x;
      v[j] = i < nkeys ? keys[i] : 0;
    }
#pragma unroll
    for (int j = 0; j < kPer; ++j) m = v[j] > m ? v[j] : m;
  }
  s_key[threadIdx.x] = m;
  __syncthreads();
  for (int h = kRowThreads / 2; h >= 1; h >>= 1) {
    if (threadIdx.x < h) {
      const uint64_t o = s_key[threadIdx.x + h];
      if (o > s_key[threadIdx.x]) s_key[threadIdx.x] = o;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const int64_t idx = static_cast<int64_t>(0xffffffffu - static_cast<uint32_t>(s_key[0]));
    token[0] = idx;
    if (token_copy) token_copy[0] = idx;
  }
}

template <bool SWIGLU, bool NORM>
void launch_gemv_kc(int kc, dim3 grid, const uint16_t* w, const uint16_t* x, const uint16_t* delta,
                    const uint16_t* ln, float eps, uint16_t* x_out, uint16_t* y, int n, int k,
                    hipStream_t stream) {
#define VOOM_GEMV(KC_)                                                                       \
  hipLaunchKernelGGL((gemv_kernel<KC_, SWIGLU, NORM>), grid, dim3(kRowThreads), 0, stream, w, x, \
                     delta, ln, eps, x_out, y, n, k)
  switch (kc) {
    case 1: VOOM_GEMV(1); break;
    case 2: VOOM_GEMV(2); break;
    case 3: VOOM_GEMV(3); break;
    default: VOOM_GEMV(4); break;
  }
#undef VOOM_GEMV
}

template <bool SWIGLU>
int launch_gemv(const uint16_t* w, const uint16_t* x, const uint16_t* delta, const uint16_t* ln,
                float eps, uint16_t* x_out, uint16_t* y, int n, int k, hipStream_t stream) {
  const int rows_per_wave = SWIGLU ? 2 : 4;
  const long long waves = (static_cast<long long>(n) + rows_per_wave - 1) / rows_per_wave;
  const dim3 grid(static_cast<unsigned>((waves + kRowThreads / kWave - 1) / (kRowThreads / kWave)));
  const int kc = (k / 8 + kWave - 1) / kWave;
  if (ln)
    launch_gemv_kc<SWIGLU, true>(kc, grid, w, x, delta, ln, eps, x_out, y, n, k, stream);
  else
    launch_gemv_kc<SWIGLU, false>(kc, grid, w, x, delta, ln, eps, x_out, y, n, k, stream);
  return VOOM_LAUNCH_CHECK("gemv: kernel launch");
}

// Projections of several rows (a prompt, a batch of tokens): y = x . W^T with
// the decode kernels' fusions around it -- the residual add + RMSNorm of the
// rows in front and SwiGLU (kSwiglu) or RoPE and the page write of k and v
// (kRope) behind, or neither (kPlain).  A prompt of a small model is bound by its
// launches, not by its sums (a 512-row projection with k 576 and n 960 is 0.2 us
// of matrix work), so the aim is few launches, each one memory round trip deep:
//   a workgroup takes 32 rows and NW wavefronts of 16-column weight tiles (two
//   tiles for the pairs of SwiGLU and RoPE).  Its rows and each wavefront's first
//   2 SC k-steps of weights are put in flight together, straight into registers;
//   the rows are normed, LPR lanes a row, and left in LDS, and the MFMAs take the
//   weights as A and the rows as B: a lane ends with four adjacent columns of one
//   row, and a pair's two halves are in one lane.
// The rows are prepared again by each column group; that is 37 KB of reads that
// hit L2, against a launch.  Column groups go round the XCDs, so each weight
// crosses into one L2 only.  512 rows (k 576): qkv with its norm, RoPE and page
// write 13.1 us, gate/up with norm and SwiGLU 15.8, 576 columns 6.7, and down
// (k 1536) 11.2; as separate launches around library products a 30-layer prompt of
// 512 tokens took 5.6 ms, so 2.3, and one of 64 tokens 5.2, so 2.0, both then
// bound by the host.
enum RowsMode { kPlain, kSwiglu, kRope };
constexpr int kRowsTile = 32;   // rows of one workgroup
constexpr int kRowsUnit = 256;  // k of one LDS size class

struct RowsArgs {
  const uint16_t* x;
  const uint16_t* delta;
  const uint16_t* ln;
  uint16_t* x_out;
  const uint16_t* w;
  uint16_t* y;  // q in kRope
  int rows, n, k;
  int tiles;       // 16-column tiles (kSwiglu, kRope: tile pairs)
  int groups;      // column groups: of NW tiles
  int row_groups;  // groups of kRowsTile rows
  float eps;
  // kRope
  const float* cos_t;
  const float* sin_t;
  uint16_t* k_pool;
  uint16_t* v_pool;
  const int32_t* table;
  int L, start, nq, nkv, hd, pt_shift, max_pages, num_slots;
};

// Sum over each aligned group of LPR (8 or 16) lanes, the same value in all.
template <int LPR>
__device__ __forceinline__ float group_sum(float v) {
  v += dpp_move<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  v += dpp_move<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  v += dpp_move<0x141>(v);  // row_half_mirror
  if (LPR == 16) v += dpp_move<0x140>(v);  // row_mirror
  return v;
}

__device__ __forceinline__ uint16_t swiglu_bf16(float gate, float up) {
  const float g = bf2f(f2bf(gate));
  const float s = bf2f(f2bf(g / (1.f + expf(-g))));
  return f2bf(s * bf2f(f2bf(up)));
}

// Dims d .. d + 3 and d + half .. of head h of one row: rotated (q, k) and
// written to q or through the block table to the pools.
__device__ __forceinline__ void store_rope(const RowsArgs& a, int row, int h, int d, f32x4 lo,
                                           f32x4 hi) {
  const int half = a.hd / 2;
  const int b = row / a.L;
  const int l = row - b * a.L;
  uint16_t o1[4], o2[4];
  if (h < a.nq + a.nkv) {
#pragma clang fp contract(off)
    const float* cr = a.cos_t + static_cast<size_t>(l) * a.hd + d;
    const float* sr = a.sin_t + static_cast<size_t>(l) * a.hd + d;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x1 = bf2f(f2bf(lo[e]));
      const float x2 = bf2f(f2bf(hi[e]));
      const float a0 = x1 * cr[e];
      const float b0 = -x2 * sr[e];
      const float a1 = x2 * cr[half + e];
      const float b1 = x1 * sr[half + e];
      o1[e] = f2bf(a0 + b0);
      o2[e] = f2bf(a1 + b1);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o1[e] = f2bf(lo[e]);
      o2[e] = f2bf(hi[e]);
    }
  }
  const u32x2 p1 = {o1[0] | static_cast<uint32_t>(o1[1]) << 16,
                    o1[2] | static_cast<uint32_t>(o1[3]) << 16};
  const u32x2 p2 = {o2[0] | static_cast<uint32_t>(o2[1]) << 16,
                    o2[2] | static_cast<uint32_t>(o2[3]) << 16};
  if (h < a.nq) {
    uint16_t* qr = a.y + ((static_cast<size_t>(b) * a.nq + h) * a.L + l) * a.hd + d;
    *reinterpret_cast<u32x2*>(qr) = p1;
    *reinterpret_cast<u32x2*>(qr + half) = p2;
    return;
  }
  const int pos = a.start + l;
  const int page = pos >> a.pt_shift;
  if (page >= a.max_pages) return;
  const int slot = a.table[static_cast<size_t>(b) * a.max_pages + page];
  if (static_cast<unsigned>(slot) >= static_cast<unsigned>(a.num_slots)) return;
  const int off = pos & ((1 << a.pt_shift) - 1);
  const bool is_k = h < a.nq + a.nkv;
  const int kvh = is_k ? h - a.nq : h - a.nq - a.nkv;
  const size_t head_page = static_cast<size_t>(slot) * a.nkv + kvh;
  if (is_k) {
    uint16_t* kr = a.k_pool + ((head_page << a.pt_shift) + off) * a.hd + d;
    *reinterpret_cast<u32x2*>(kr) = p1;
    *reinterpret_cast<u32x2*>(kr + half) = p2;
  } else {
    const int vb_shift = a.pt_shift < 5 ? a.pt_shift : 5;
    const size_t blk = (head_page << (a.pt_shift - vb_shift)) + (off >> vb_shift);
    const int col = off & ((1 << vb_shift) - 1);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      a.v_pool[((blk * a.hd + d + e) << vb_shift) + col] = o1[e];
      a.v_pool[((blk * a.hd + d + half + e) << vb_shift) + col] = o2[e];
    }
  }
}

template <int CH, int MODE, int NW>
__global__ __launch_bounds__(kWave* NW) void linear_rows_kernel(RowsArgs a) {
  constexpr bool NORM = MODE != kPlain;
  constexpr int T = MODE == kPlain ? 1 : 2;    // weight tiles of a wavefront
  constexpr int SC = MODE == kPlain ? 12 : 6;  // k-steps of one register buffer
  constexpr int LPR = kWave * NW / kRowsTile;  // lanes of one row
  constexpr int CPL = kRowsUnit / 8 * CH / LPR;  // 16-byte chunks of one lane
  // 16 bytes past whole 512-byte units: an odd multiple of 16 bytes between rows,
  // so the 16 rows of a fragment lie on different LDS banks
  constexpr int STRIDE = kRowsUnit * CH + 8;
  __shared__ __align__(16) uint16_t lds[kRowsTile * STRIDE];
  // workgroup i: XCD i % 8 takes column groups i % 8, i % 8 + 8, ...
  const int xcd = blockIdx.x & 7;
  const int idx = blockIdx.x >> 3;
  const int group = uniform(xcd + 8 * (idx / a.row_groups));
  const int row0 = uniform(kRowsTile * (idx % a.row_groups));
  if (group >= a.groups) return;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = uniform(threadIdx.x / kWave);

  // this lane's chunks of its row (a row past the end repeats the last one, a
  // chunk past the row its last; neither is stored)
  const int chunks = a.k / 8;
  const int local = (kWave / LPR) * wave + lane / LPR;
  const int c0 = lane % LPR;
  const size_t at = static_cast<size_t>(min(row0 + local, a.rows - 1)) * a.k;
  u32x4 v[CPL], d[NORM ? CPL : 1];
  const uint16_t* dsrc = NORM && a.delta ? a.delta : a.x;
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
    const int c = min(c0 + LPR * j, chunks - 1);
    v[j] = *reinterpret_cast<const u32x4*>(a.x + at + 8 * c);
    if (NORM) d[j] = *reinterpret_cast<const u32x4*>(dsrc + at + 8 * c);
  }

  const int i16 = lane & 15;
  const int kq = 8 * (lane >> 4);
  const int steps = a.k / 32;
  const int tile = uniform(NW * group + wave);
  // wavefronts past the last tile read it again and store nothing
  const int t = min(tile, a.tiles - 1);
  int col[T];  // first column of each tile
  int head = 0, dim = 0;
  if (MODE == kPlain) {
    col[0] = 16 * t;
  } else if (MODE == kSwiglu) {
    col[0] = 16 * t;
    col[T - 1] = a.n + 16 * t;
  } else {
    const int per_head = a.hd / 32;
    head = t / per_head;
    dim = 16 * (t - head * per_head);
    col[0] = head * a.hd + dim;
    col[T - 1] = col[0] + a.hd / 2;
  }
  const uint16_t* wr[T];
#pragma unroll
  for (int j = 0; j < T; ++j) {
    const int last = MODE == kRope ? col[j] + 15 : (j + 1) * a.n - 1;
    wr[j] = a.w + static_cast<size_t>(min(col[j] + i16, last)) * a.k + kq;
  }
  auto load = [&](int s0, u32x4 (&wq)[T][SC]) {
#pragma unroll
    for (int i = 0; i < SC; ++i) {
      const int s = min(s0 + i, steps - 1);
#pragma unroll
      for (int j = 0; j < T; ++j) wq[j][i] = *reinterpret_cast<const u32x4*>(wr[j] + 32 * s);
    }
  };
  u32x4 wa[T][SC], wb[T][SC];
  load(0, wa);
  load(SC, wb);
  asm volatile("" ::: "memory");  // the weights stay in flight under the norm

  float inv = 1.f;
  if (NORM) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      if (LPR * j >= chunks) continue;
      const u32x4 sum = sum_chunks(v[j], d[NORM ? j : 0]);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[j][e] = a.delta ? sum[e] : v[j][e];
      if (c0 + LPR * j < chunks) ss = chunk_sumsq(v[j], ss);
    }
    inv = 1.f / sqrtf(group_sum<LPR>(ss) / static_cast<float>(a.k) + a.eps);
  }
  const bool writer = NORM && a.x_out != nullptr && group == 0 && row0 + local < a.rows;
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
    const int c = c0 + LPR * j;
    if (c < chunks) {
      if (writer) *reinterpret_cast<u32x4*>(a.x_out + at + 8 * c) = v[j];
      if (NORM) v[j] = norm_chunk(v[j], *reinterpret_cast<const u32x4*>(a.ln + 8 * c), inv);
      *reinterpret_cast<u32x4*>(lds + local * STRIDE + 8 * c) = v[j];
    }
  }
  lds_barrier();

  f32x4 acc[2][T];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int j = 0; j < T; ++j) acc[m][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto product = [&](int s0, const u32x4 (&wq)[T][SC]) {
#pragma unroll
    for (int i = 0; i < SC; ++i) {
      if (s0 + i < steps) {
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const bf16x8 xr = *reinterpret_cast<const bf16x8*>(lds + (16 * m + i16) * STRIDE +
                                                             32 * (s0 + i) + kq);
#pragma unroll
          for (int j = 0; j < T; ++j)
            acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8, wq[j][i]), xr, acc[m][j], 0, 0, 0);
        }
      }
    }
  };
  for (int s0 = 0; s0 < steps; s0 += 2 * SC) {
    product(s0, wa);
    if (s0 + SC >= steps) break;
    if (s0 + 2 * SC < steps) load(s0 + 2 * SC, wa);
    product(s0 + SC, wb);
    if (s0 + 3 * SC < steps) load(s0 + 3 * SC, wb);
  }
  if (tile >= a.tiles) return;
  // lane (row i16 of its half): columns 4 (lane / 16) .. + 3 of the tile
  const int sub = 4 * (lane >> 4);
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const int row = row0 + 16 * m + i16;
    if (row >= a.rows) continue;
    if (MODE == kRope) {
      store_rope(a, row, head, dim + sub, acc[m][0], acc[m][T - 1]);
    } else if (col[0] + sub < a.n) {
      u32x2 o;
      if (MODE == kSwiglu) {
        uint16_t s[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = swiglu_bf16(acc[m][0][e], acc[m][T - 1][e]);
        o = u32x2{s[0] | static_cast<uint32_t>(s[1]) << 16,
                  s[2] | static_cast<uint32_t>(s[3]) << 16};
      } else {
        o = u32x2{pack_bf16x2(acc[m][0][0], acc[m][0][1]),
                  pack_bf16x2(acc[m][0][2], acc[m][0][3])};
      }
      *reinterpret_cast<u32x2*>(a.y + static_cast<size_t>(row) * a.n + col[0] + sub) = o;
    }
  }
}

template <int MODE>
int launch_rows(const char* who, RowsArgs& a, hipStream_t stream) {
  // The widest form prepares its rows half as often with eight wavefronts (3072
  // columns: 18.1 us with four, 15.8 with eight); the narrow ones would leave most
  // CUs idle (960 columns: 13.1 and 16.1 us; 576 columns, k 1536: 11.2 and 15.9).
  constexpr int NW = MODE == kSwiglu ? 8 : 4;
  a.groups = (a.tiles + NW - 1) / NW;
  a.row_groups = (a.rows + kRowsTile - 1) / kRowsTile;
  const long long grid = 8LL * ((a.groups + 7) / 8) * a.row_groups;
  VOOM_REQUIRE(grid < (1LL << 31), "%s: too many rows", who);
#define VOOM_ROWS(CH_)                                                                           \
  case CH_:                                                                                      \
    hipLaunchKernelGGL((linear_rows_kernel<CH_, MODE, NW>), dim3(static_cast<unsigned>(grid)), \
                       dim3(kWave * NW), 0, stream, a);                                         \
    break
  switch ((a.k + kRowsUnit - 1) / kRowsUnit) {
    VOOM_ROWS(1);
    VOOM_ROWS(2);
    VOOM_ROWS(3);
    VOOM_ROWS(4);
    VOOM_ROWS(5);
    VOOM_ROWS(6);
    VOOM_ROWS(7);
    VOOM_ROWS(8);
  }
#undef VOOM_ROWS
  return VOOM_LAUNCH_CHECK("linear_rows: kernel launch");
}

}  // namespace
}  // namespace voom

using namespace voom;

namespace {
// Shared checks of the residual-add + RMSNorm prologue arguments.
int check_norm_prologue(const char* who, const void* x, const void* delta, const void* ln_weight,
                        const void* x_out) {
  VOOM_REQUIRE(ln_weight != nullptr || (delta == nullptr && x_out == nullptr),
               "%s: delta and x_out need ln_weight", who);
  VOOM_REQUIRE(x_out == nullptr || (x_out != x && x_out != delta),
               "%s: x_out must not alias x or delta", who);
  VOOM_REQUIRE(reinterpret_cast<uintptr_t>(delta) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(ln_weight) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(x_out) % 16 == 0,
               "%s: delta, ln_weight and x_out must be 16-byte aligned", who);
  return 0;
}
}  // namespace

extern "C" int voom_qkv_rope_append(const void* w_qkv, const void* x, const void* delta,
                                    const void* ln_weight, float eps, void* x_out,
                                    const float* cos_row, const float* sin_row, void* q,
                                    void* k_pool, void* v_pool, const int32_t* table_row,
                                    const int32_t* position, int num_q_heads, int num_kv_heads,
                                    int head_dim, int k, int page_tokens, int max_pages,
                                    int num_slots, int rope_rows, hipStream_t stream) {
  const char* who = "qkv_rope_append";
  VOOM_REQUIRE(w_qkv && x && cos_row && sin_row && q && k_pool && v_pool && table_row && position,
               "%s: null pointer argument", who);
  if (int rc = check_norm_prologue(who, x, delta, ln_weight, x_out)) return rc;
  VOOM_REQUIRE(num_q_heads > 0 && num_kv_heads > 0 && head_dim > 0 && head_dim % 4 == 0,
               "%s: bad head geometry", who);
  VOOM_REQUIRE(k > 0 && k % 8 == 0 && k <= 8 * kWave * 4,
               "%s: k %d must be a positive multiple of 8 up to %d", who, k, 8 * kWave * 4);
  VOOM_REQUIRE(is_pow2(page_tokens) && page_tokens <= 4096 && max_pages > 0 && num_slots > 0,
               "%s: bad page geometry", who);
  VOOM_REQUIRE(rope_rows >= 0, "%s: rope_rows must be >= 0", who);
  VOOM_REQUIRE(reinterpret_cast<uintptr_t>(w_qkv) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(x) % 16 == 0,
               "%s: weight and x must be 16-byte aligned", who);
  const long long waves = static_cast<long long>(num_q_heads + 2 * num_kv_heads) * (head_dim / 4);
  const dim3 grid(static_cast<unsigned>((waves + kRowThreads / kWave - 1) / (kRowThreads / kWave)));
  const int kc = (k / 8 + kWave - 1) / kWave;
  const auto* wq = static_cast<const uint16_t*>(w_qkv);
  const auto* xv = static_cast<const uint16_t*>(x);
  auto* qo = static_cast<uint16_t*>(q);
  auto* kp = static_cast<uint16_t*>(k_pool);
  auto* vp = static_cast<uint16_t*>(v_pool);
  const auto* dv = static_cast<const uint16_t*>(delta);
  const auto* lw = static_cast<const uint16_t*>(ln_weight);
  auto* xo = static_cast<uint16_t*>(x_out);
  const int pts = ilog2(page_tokens);
#define VOOM_QRA_N(KC_, NORM_)                                                             \
  hipLaunchKernelGGL((qkv_rope_append_kernel<KC_, NORM_>), grid, dim3(kRowThreads), 0, stream, \
                     wq, xv, dv, lw, eps, xo, cos_row, sin_row, qo, kp, vp, table_row,         \
                     position, num_q_heads, num_kv_heads, head_dim, k, pts, max_pages,         \
                     num_slots, rope_rows)
#define VOOM_QRA(KC_)      \
  if (lw)                  \
    VOOM_QRA_N(KC_, true); \
  else                     \
    VOOM_QRA_N(KC_, false)
  switch (kc) {
    case 1: VOOM_QRA(1); break;
    case 2: VOOM_QRA(2); break;
    case 3: VOOM_QRA(3); break;
    default: VOOM_QRA(4); break;
  }
#undef VOOM_QRA
#undef VOOM_QRA_N
  return VOOM_LAUNCH_CHECK("qkv_rope_append: kernel launch");
}

extern "C" int voom_gemv_bf16(const void* weight, const void* x, void* y, int n, int k,
                              int swiglu, hipStream_t stream) {
  return voom_add_rms_norm_gemv(x, nullptr, nullptr, 0.f, nullptr, weight, y, n, k, swiglu,
                                stream);
}

extern "C" int voom_add_rms_norm_gemv(const void* x, const void* delta, const void* ln_weight,
                                      float eps, void* x_out, const void* weight, void* y, int n,
                                      int k, int swiglu, hipStream_t stream) {
  const char* who = "gemv_bf16";
  VOOM_REQUIRE(weight && x && y, "%s: null pointer argument", who);
  if (int rc = check_norm_prologue(who, x, delta, ln_weight, x_out)) return rc;
  VOOM_REQUIRE(n > 0 && k > 0 && k % 8 == 0 && k <= 8 * kWave * 4,
               "%s: k %d must be a positive multiple of 8 up to %d", who, k, 8 * kWave * 4);
  VOOM_REQUIRE(n < (1 << 28), "%s: n %d too large", who, n);
  VOOM_REQUIRE(reinterpret_cast<uintptr_t>(weight) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(y) % 2 == 0,
               "%s: weight and x must be 16-byte aligned", who);
  const auto* w = static_cast<const uint16_t*>(weight);
  const auto* xv = static_cast<const uint16_t*>(x);
  auto* yv = static_cast<uint16_t*>(y);
  const auto* dv = static_cast<const uint16_t*>(delta);
  const auto* lw = static_cast<const uint16_t*>(ln_weight);
  auto* xo = static_cast<uint16_t*>(x_out);
  return swiglu ? launch_gemv<true>(w, xv, dv, lw, eps, xo, yv, n, k, stream)
                : launch_gemv<false>(w, xv, dv, lw, eps, xo, yv, n, k, stream);
}

namespace {
int prepare_rows(const char* who, const void* x, const void* delta, const void* ln_weight,
                 float eps, void* x_out, const void* weight, void* y, long long rows, int k,
                 RowsArgs& a) {
  VOOM_REQUIRE(weight && x && y, "%s: null pointer argument", who);
  if (int rc = check_norm_prologue(who, x, delta, ln_weight, x_out)) return rc;
  VOOM_REQUIRE(k > 0 && k % 32 == 0 && k <= 8 * kWave * 4,
               "%s: k %d must be a positive multiple of 32 up to %d", who, k, 8 * kWave * 4);
  VOOM_REQUIRE(rows > 0 && rows < (1LL << 24), "%s: bad row count", who);
  VOOM_REQUIRE(reinterpret_cast<uintptr_t>(weight) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(y) % 16 == 0,
               "%s: weight, x and the output must be 16-byte aligned", who);
  a = RowsArgs{};
  a.x = static_cast<const uint16_t*>(x);
  a.delta = static_cast<const uint16_t*>(delta);
  a.ln = static_cast<const uint16_t*>(ln_weight);
  a.x_out = static_cast<uint16_t*>(x_out);
  a.w = static_cast<const uint16_t*>(weight);
  a.y = static_cast<uint16_t*>(y);
  a.rows = static_cast<int>(rows);
  a.k = k;
  a.eps = eps;
  return VOOM_OK;
}
}  // namespace

extern "C" int voom_linear_rows(const void* x, const void* weight, void* y, int rows, int n, int k,
                                hipStream_t stream) {
  const char* who = "linear_rows";
  RowsArgs a;
  if (int rc = prepare_rows(who, x, nullptr, nullptr, 0.f, nullptr, weight, y, rows, k, a))
    return rc;
  VOOM_REQUIRE(n > 0 && n % 8 == 0 && n < (1 << 28), "%s: n %d must be a positive multiple of 8",
               who, n);
  a.n = n;
  a.tiles = (n + 15) / 16;
  return launch_rows<kPlain>(who, a, stream);
}

extern "C" int voom_norm_swiglu_rows(const void* x, const void* delta, const void* ln_weight,
                                     float eps, void* x_out, const void* weight, void* y, int rows,
                                     int n, int k, hipStream_t stream) {
  const char* who = "norm_swiglu_rows";
  RowsArgs a;
  VOOM_REQUIRE(ln_weight != nullptr, "%s: null pointer argument", who);
  if (int rc = prepare_rows(who, x, delta, ln_weight, eps, x_out, weight, y, rows, k, a)) return rc;
  VOOM_REQUIRE(n > 0 && n % 8 == 0 && n < (1 << 28), "%s: n %d must be a positive multiple of 8",
               who, n);
  a.n = n;
  a.tiles = (n + 15) / 16;
  return launch_rows<kSwiglu>(who, a, stream);
}

extern "C" int voom_qkv_rope_append_rows(const void* w_qkv, const void* x, const void* delta,
                                         const void* ln_weight, float eps, void* x_out,
                                         const float* cos_table, const float* sin_table, void* q,
                                         void* k_pool, void* v_pool, const int32_t* block_table,
                                         int batch, int seq, int start, int num_q_heads,
                                         int num_kv_heads, int head_dim, int k, int page_tokens,
                                         int max_pages, int num_slots, hipStream_t stream) {
  const char* who = "qkv_rope_append_rows";
  RowsArgs a;
  VOOM_REQUIRE(ln_weight && cos_table && sin_table && k_pool && v_pool && block_table,
               "%s: null pointer argument", who);
  VOOM_REQUIRE(batch > 0 && seq > 0, "%s: bad geometry", who);
  if (int rc = prepare_rows(who, x, delta, ln_weight, eps, x_out, w_qkv, q,
                            static_cast<long long>(batch) * seq, k, a))
    return rc;
  VOOM_REQUIRE(num_q_heads > 0 && num_kv_heads > 0 && num_q_heads < (1 << 14) &&
                   num_kv_heads < (1 << 14) && head_dim > 0 && head_dim <= 1024 &&
                   head_dim % 32 == 0,
               "%s: bad head geometry (head_dim a multiple of 32)", who);
  VOOM_REQUIRE(is_pow2(page_tokens) && page_tokens <= 4096 && max_pages > 0 && num_slots > 0,
               "%s: bad page geometry", who);
  VOOM_REQUIRE(start >= 0 && static_cast<long long>(start) + seq < (1LL << 31),
               "%s: bad start %d", who, start);
  VOOM_REQUIRE(reinterpret_cast<uintptr_t>(k_pool) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(v_pool) % 16 == 0,
               "%s: pools must be 16-byte aligned", who);
  a.n = (num_q_heads + 2 * num_kv_heads) * head_dim;
  a.tiles = (num_q_heads + 2 * num_kv_heads) * (head_dim / 32);
  a.cos_t = cos_table;
  a.sin_t = sin_table;
  a.k_pool = static_cast<uint16_t*>(k_pool);
  a.v_pool = static_cast<uint16_t*>(v_pool);
  a.table = block_table;
  a.L = seq;
  a.start = start;
  a.nq = num_q_heads;
  a.nkv = num_kv_heads;
  a.hd = head_dim;
  a.pt_shift = ilog2(page_tokens);
  a.max_pages = max_pages;
  a.num_slots = num_slots;
  return launch_rows<kRope>(who, a, stream);
}

extern "C" int voom_lm_head_argmax(const void* x, const void* delta, const void* ln_weight,
                                   float eps, const void* weight, int n, int k, void* workspace,
                                   size_t ws_bytes, int64_t* token, int64_t* token_copy,
                                   hipStream_t stream) {
  const char* who = "lm_head_argmax";
  VOOM_REQUIRE(x && weight && workspace && token, "%s: null pointer argument", who);
  if (int rc = check_norm_prologue(who, x, delta, ln_weight, nullptr)) return rc;
  VOOM_REQUIRE(n > 0 && n < (1 << 28) && k > 0 && k % 8 == 0 && k <= 8 * kWave * 4,
               "%s: k %d must be a positive multiple of 8 up to %d", who, k, 8 * kWave * 4);
  VOOM_REQUIRE(reinterpret_cast<uintptr_t>(weight) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(workspace) % 8 == 0,
               "%s: weight and x must be 16-byte aligned, workspace 8-byte", who);
  const int rows_per_block = 4 * (kRowThreads / kWave);
  const int blocks = (n + rows_per_block - 1) / rows_per_block;
  VOOM_REQUIRE(ws_bytes >= static_cast<size_t>(blocks) * 8, "%s: workspace needs %d bytes", who,
               blocks * 8);
  const auto* w = static_cast<const uint16_t*>(weight);
  const auto* xv = static_cast<const uint16_t*>(x);
  const auto* dv = static_cast<const uint16_t*>(delta);
  const auto* lw = static_cast<const uint16_t*>(ln_weight);
  auto* keys = static_cast<uint64_t*>(workspace);
  const int kc = (k / 8 + kWave - 1) / kWave;
#define VOOM_GA(KC_, NORM_)                                                                   \
  hipLaunchKernelGGL((gemv_argmax_kernel<KC_, NORM_>), dim3(blocks), dim3(kRowThreads), 0,      \
                     stream, w, xv, dv, lw, eps, keys, n, k)
#define VOOM_GA_KC(KC_) \
  if (lw)               \
    VOOM_GA(KC_, true); \
  else                  \
    VOOM_GA(KC_, false)
  switch (kc) {
    case 1: VOOM_GA_KC(1); break;
    case 2: VOOM_GA_KC(2); break;
    case 3: VOOM_GA_KC(3); break;
    default: VOOM_GA_KC(4); break;
  }
#undef VOOM_GA_KC
#undef VOOM_GA
  if (int rc = VOOM_LAUNCH_CHECK("lm_head_argmax: projection launch")) return rc;
  hipLaunchKernelGGL(argmax_finish_kernel, dim3(1), dim3(kRowThreads), 0, stream, keys, blocks,
                     token, token_copy);
  return VOOM_LAUNCH_CHECK("lm_head_argmax: finish launch");
}

extern "C" int voom_add_rms_norm(void* x, const void* delta, const void* weight, void* out,
                                 int rows, int hidden, float eps, hipStream_t stream) {
  const char* who = "add_rms_norm";
  VOOM_REQUIRE(x && weight && out, "%s: null pointer argument", who);
  VOOM_REQUIRE(rows > 0 && hidden > 0 && hidden % 8 == 0 && hidden <= 8192,
               "%s: hidden %d must be a multiple of 8 up to 8192", who, hidden);
  VOOM_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(weight) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(out) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(delta) % 16 == 0,
               "%s: tensors must be 16-byte aligned", who);
  hipLaunchKernelGGL(add_rms_norm_kernel, dim3(static_cast<unsigned>(rows)), dim3(kRowThreads),
                     0, stream, static_cast<uint16_t*>(x), static_cast<const uint16_t*>(delta),
                     static_cast<const uint16_t*>(weight), static_cast<uint16_t*>(out), hidden,
                     eps);
  return VOOM_LAUNCH_CHECK("add_rms_norm: kernel launch");
}

extern "C" int voom_rope_split(const void* qkv, const float* cos_table, const float* sin_table,
                               void* q, void* k, void* v, int batch, int seq, int num_q_heads,
                               int num_kv_heads, int head_dim, hipStream_t stream) {
  const char* who = "rope_split";
  VOOM_REQUIRE(qkv && cos_table && sin_table && q && k && v, "%s: null pointer argument", who);
  VOOM_REQUIRE(batch > 0 && seq > 0 && num_q_heads > 0 && num_kv_heads > 0 && head_dim > 0 &&
                   head_dim % 2 == 0,
               "%s: bad geometry", who);
  const long long total =
      static_cast<long long>(batch) * seq * (num_q_heads + 2 * num_kv_heads) * (head_dim / 2);
  VOOM_REQUIRE(total < (1LL << 40), "%s: too large", who);
  hipLaunchKernelGGL(rope_split_kernel,
                     dim3(static_cast<unsigned>((total + kRowThreads - 1) / kRowThreads)),
                     dim3(kRowThreads), 0, stream, static_cast<const uint16_t*>(qkv), cos_table,
                     sin_table, static_cast<uint16_t*>(q), static_cast<uint16_t*>(k),
                     static_cast<uint16_t*>(v), batch, seq, num_q_heads, num_kv_heads, head_dim);
  return VOOM_LAUNCH_CHECK("rope_split: kernel launch");
}

extern "C" int voom_silu_mul(const void* gate_up, void* out, int rows, int intermediate,
                             hipStream_t stream) {
  const char* who = "silu_mul";
  VOOM_REQUIRE(gate_up && out, "%s: null pointer argument", who);
  VOOM_REQUIRE(rows > 0 && intermediate > 0 && intermediate % 8 == 0,
               "%s: intermediate %d must be a positive multiple of 8", who, intermediate);
  VOOM_REQUIRE(reinterpret_cast<uintptr_t>(gate_up) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(out) % 16 == 0,
               "%s: tensors must be 16-byte aligned", who);
  const long long total = static_cast<long long>(rows) * (intermediate / 8);
  hipLaunchKernelGGL(silu_mul_kernel,
                     dim3(static_cast<unsigned>((total + kRowThreads - 1) / kRowThreads)),
                     dim3(kRowThreads), 0, stream, static_cast<const uint16_t*>(gate_up),
                     static_cast<uint16_t*>(out), rows, intermediate);
  return VOOM_LAUNCH_CHECK("silu_mul: kernel launch");
}
