// Draft decode attention over the working cache's capacity view.
//
// Counterpart of DiffSpecDraftCache.forward_attention's linear path:
// diffspec/runtime.py:2024-2077 (CPU loop) and :2079-2134 (one batched NPU
// fused-attention call over the [slot, head, token_budget, head_dim] view with
// per-row valid lengths).  For each row r with slot s and local position p:
//   working_key[s, :, p] = key[r], working_value[s, :, p] = value[r],
//   working_lens[s] = p + 1,
//   out[r, h] = softmax(scale * q[r, h] . K[s, h / G, 0..p]) V[s, h / G, 0..p]
// in fp32, and out rows past the batch are zero.
//
// Work split (draft_attention_kernel; larger batches run
// attention_stream_kernel, see there): one workgroup per (row, KV head, block
// of up to 16 query heads of that KV head's group, span of tokens).  Each of its 4 waves walks
// 16-token tiles of its quarter of the span:
//   scores  S[t][g] = K[t] . Q[g]     one 16x16x32 bf16/fp16 MFMA per 32 of
//                                     head_dim, K as the A operand (lane owns
//                                     token t = lane % 16), Q as B (lane owns
//                                     query g = lane % 16);
//   softmax online per query g (lane column), rows of the S tile are tokens
//                                     4 * (lane / 16) + i;
//   output  O^T[d][g] += V^T[d][t] P^T[t][g]   the same MFMA over the 32
//                                     tokens of two tiles, P split into an
//                                     upper and a lower 16-bit part (two MFMAs
//                                     per head_dim block): the k-slot (lane /
//                                     16, e) is token 4 * (lane / 16) + e % 4 of
//                                     tile e / 4, so the B operand is the
//                                     lane's own probabilities; head_dim column
//                                     m of block j is d = out_dim(m, j) (J = D /
//                                     16 blocks), so the A operand is the
//                                     elements of V's row that lane column m
//                                     loads, and each lane ends with D / 4
//                                     outputs of query g.
// Probabilities are fp32 (the reference's softmax is fp32 and multiplies fp32
// V) and enter the products to within 2^-14.  The four waves merge in LDS.  A
// row that fits one span writes its output directly; in a longer row every
// span writes its partial (running max, sum and unnormalised output, fp32)
// with device-scope stores, waits for their acknowledgement and counts itself
// on the row's counter, and the one that counts last merges the spans in
// index order and resets the counter.
//
// Every workgroup stores a "seen" word (tag << 32, tag = launch epoch + 1)
// once it has read its position; the grid's last workgroup waits for all of
// them, writes working_lens[slot] = position + 1 and advances the epoch,
// which keeps graph replays and workspace reuse safe.  Positions may
// therefore come from working_lens itself.  It only waits for workgroups of
// lower index, which are dispatched before it, so the wait ends whether or
// not the grid is resident at once; it is bounded all the same.  The new
// token's K/V is read from the input rows (its working-cache slot is written
// by the same launch).  Barriers in this kernel are LDS-only but for the wait
// for a partial's stores: loads stay in flight behind them.
#include "ds355_common.h"

namespace ds355 {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kThreadsA = 256;
constexpr int kWavesA = kThreadsA / 64;
constexpr int kTileT = 16;        // tokens per MFMA tile
constexpr int kGroupQ = 16;       // query heads per workgroup (MFMA N)
constexpr int kGroupS = 8;      // other spans merged per round trip
constexpr uint32_t kSpinA = 1u << 20;
constexpr float kLog2e = 1.44269504088896340736f;

// Workspace layout (bytes): a 256-byte header (epoch, status); a fixed
// region of kMaxUnits 32-bit span counters, one per (row, KV head, query
// block), 0 between launches (a shape-independent place, so a launch of
// another shape never reads other words as counters); one tagged "seen"
// word per workgroup of the pending rows (64-bit, tag << 32 | value, so a
// launch of another shape finds only older tags); then the fp32 partial
// results of every span.
constexpr int kMaxUnits = 65536;
constexpr size_t kCounterBytes = kMaxUnits * sizeof(uint32_t);
enum { kHdrEpoch = 0, kHdrStatus = 2, kHdrGiveUp = 3 };  // kHdrGiveUp: set by the owner, the wait ends at once
constexpr size_t kHeaderBytes = 256;
constexpr uint32_t kStatusPosition = 1;  // a row's slot or position was out of range
constexpr uint32_t kStatusExpired = 2;   // the last workgroup stopped waiting for the others

template <int D>
struct AttnShape {
  static constexpr int kTiles = D <= 128 ? 4 : 2;          // tiles per wave
  static constexpr int kSpan = kWavesA * kTiles * kTileT;  // tokens per workgroup
  static constexpr int kSteps = D / 32;                    // score MFMAs per tile
  static constexpr int kJ = D / 16;                        // output column blocks
  static constexpr int kRow = D + 4;                       // partial floats per query: D outputs, max, sum, 2 pad
};

struct AttnArgs {
  const void* q;
  int64_t q_row, q_head;
  const void* k_in;
  int64_t k_row, k_head;
  const void* v_in;
  int64_t v_row, v_head;
  void* out;
  int64_t o_row, o_head;
  void* work_k;
  void* work_v;
  int32_t* working_lens;
  const int32_t* slots;
  const int32_t* positions;
  int rows, out_rows, num_slots, hq, hkv, group, qblocks, budget, splits;
  float scale;
  uint32_t* header;
  uint64_t* seen;
  uint32_t* counters;  // [rows * hkv * qblocks] spans done this launch
  float* partials;     // [rows * hkv * qblocks][splits][kGroupQ][kRow]
};

template <int DT>
__device__ __forceinline__ f32x4 mfma_scores(u32x4 a, u32x4 b, f32x4 c);
template <>
__device__ __forceinline__ f32x4 mfma_scores<DS_BF16>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mfma_scores<DS_FP16>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                0, 0, 0);
}

__device__ __forceinline__ u32x4 load16(const uint16_t* p) { return *reinterpret_cast<const u32x4*>(p); }

// Working rows are read in whole 128-byte lines.  The A operand of the score
// MFMAs wants 64 bytes of each of 16 tokens (lane quad * 16 + col: token col,
// 16-byte slice quad).  Loads 2 p and 2 p + 1 of a tile therefore take line p
// of tokens 0-7 and of tokens 8-15: lane (quad, col) holds slice quad + 4 (col
// / 8) of token (col % 8) + 8 (i % 2), and swap_lines exchanges halves between
// lanes col and col ^ 8.  attention_stream_kernel loads them non-temporally
// (a bare read loop on this card: 5.95 TB/s cached or in half lines, 6.7-6.9
// TB/s so), also where the batch would fit the 256 MB last-level cache: four
// draft steps over one cache that starts in HBM, us each, non-temporal /
// cached, rows of 1987 tokens (4 heads x 128, 4 MB a row): 17 rows 22.8 / 22.8,
// 24 23.9 / 26.3, 32 28.5 / 31.6, 48 38.4 / 42.0, 60 44.9 / 50.2 (the same cache
// read over and over: 21.0 / 20.8, 22.4 / 23.2, 26.7 / 27.3, 36.3 / 35.8, 43.5 /
// 42.5).  The one-shot kernel, on one round, loads them cached: 16 rows 16.3 us,
// non-temporal 16.9; a 16-row draft cycle 180.7 against 182.2.
constexpr int kPolicyNt = 2;
__device__ __forceinline__ int line_token(int col, int i) { return (col & 7) + 8 * (i & 1); }
__device__ __forceinline__ int line_elem(int quad, int col, int i) { return 8 * quad + 32 * (col >> 3) + 64 * (i >> 1); }
constexpr int kRowRor8 = 0x128;  // DPP: lane c of a 16-lane row reads lane c ^ 8
__device__ __forceinline__ void swap_lines(u32x4& a, u32x4& b) {
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const int x = static_cast<int>(a[w]), y = static_cast<int>(b[w]);
    a[w] = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(x, y, kRowRor8, 0xf, 0xc, false));
    b[w] = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(y, x, kRowRor8, 0xf, 0x3, false));
  }
}

// p = hi + lo in the cache dtype (16-bit words).  bf16: hi is p cut to its
// top 16 bits (exact), lo the remainder p - hi (exact in fp32) cut the same
// way, so |p - hi - lo| < 2^-14 |p|.  fp16: hi is p rounded to fp16, lo the
// fp16 rounding of p - hi.
template <int DT>
__device__ __forceinline__ void split_prob(float p, uint32_t& hi, uint32_t& lo) {
  if constexpr (DT == DS_BF16) {
    const uint32_t bits = __float_as_uint(p);
    const float h = __uint_as_float(bits & 0xffff0000u);
    hi = bits >> 16;
    lo = __float_as_uint(p - h) >> 16;
  } else {
    const _Float16 h = static_cast<_Float16>(p);
    hi = __builtin_bit_cast(uint16_t, h);
    lo = __builtin_bit_cast(uint16_t, static_cast<_Float16>(p - static_cast<float>(h)));
  }
}

// The J = D / 16 elements of a V row that lane column m reads, as J / 2 words:
// J m .. J m + J - 1 for J <= 8 (16 lanes cover the row); for J = 16 8 m .. 8 m
// + 7 of each half of the row, so that either load of 16 lanes covers whole
// lines.  out_dim is the head_dim index of element j.
template <int J>
__device__ __forceinline__ constexpr int v_elem(int m) { return (J < 8 ? J : 8) * m; }
template <int J>
__device__ __forceinline__ constexpr int out_dim(int m, int j) { return v_elem<J>(m) + (j & 7) + (j >> 3) * 128; }
template <int J>
__device__ __forceinline__ void load_words(const uint16_t* p, uint32_t (&w)[J / 2]) {
  if constexpr (J == 4) {
    const u32x2 v = *reinterpret_cast<const u32x2*>(p);
    w[0] = v.x; w[1] = v.y;
  } else {
#pragma unroll
    for (int h = 0; h < J / 8; ++h) {
      const u32x4 v = load16(p + 128 * h);
      w[4 * h] = v.x; w[4 * h + 1] = v.y; w[4 * h + 2] = v.z; w[4 * h + 3] = v.w;
    }
  }
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// 16-byte accesses with the device-scope cache policy (sc1), through a raw
// buffer resource over one row's partials.
typedef __amdgpu_buffer_rsrc_t Rsrc16;
constexpr int kPolicySc1 = 16;
__device__ __forceinline__ Rsrc16 make_rsrc16(const void* base, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), 0x00020000);
}
__device__ __forceinline__ void store16_sc1(Rsrc16 r, int voff, int soff, f32x4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, voff, soff, kPolicySc1);
}
__device__ __forceinline__ f32x4 load16_sc1(Rsrc16 r, int voff, int soff) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, kPolicySc1));
}
__device__ __forceinline__ f32x2 load8_sc1(Rsrc16 r, int voff, int soff) {
  return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, kPolicySc1));
}

// The same through a buffer resource, non-temporally.
template <int J>
__device__ __forceinline__ void load_words_buf(Rsrc16 r, int voff, int soff, uint32_t (&w)[J / 2]) {
  if constexpr (J == 4) {
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, kPolicyNt);
    w[0] = v.x; w[1] = v.y;
  } else {
#pragma unroll
    for (int h = 0; h < J / 8; ++h) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, voff + 256 * h, soff, kPolicyNt);
      w[4 * h] = v.x; w[4 * h + 1] = v.y; w[4 * h + 2] = v.z; w[4 * h + 3] = v.w;
    }
  }
}

__device__ __forceinline__ uint64_t tagged(uint32_t tag, float v) {
  return (static_cast<uint64_t>(tag) << 32) | __float_as_uint(v);
}

__device__ __forceinline__ void raise_status(const AttnArgs& a, uint32_t bit) {
  __hip_atomic_fetch_or(a.header + kHdrStatus, bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Waits until a workgroup's seen word carries this launch's tag.  The wait is
// bounded: after one expiry the thread stops waiting (status bit set).
__device__ __forceinline__ void await_seen(const AttnArgs& a, const uint64_t* p, uint32_t tag, bool& expired) {
  uint32_t spins = 0;
  for (uint64_t v = coherent_load(p); static_cast<uint32_t>(v >> 32) != tag; v = coherent_load(p)) {
    if (expired) return;
    if (++spins > kSpinA) {
      raise_status(a, kStatusExpired);
      expired = true;
      return;
    }
    __builtin_amdgcn_s_sleep(2);
  }
}

// Zero out[row, head0 .. head0 + count) (padding rows and rows with a bad position).
template <int D>
__device__ __forceinline__ void zero_heads(const AttnArgs& a, int row, int head0, int count) {
  uint16_t* o = static_cast<uint16_t*>(a.out) + static_cast<int64_t>(row) * a.o_row;
  const int chunks = count * (D / 8);
  for (int c = threadIdx.x; c < chunks; c += kThreadsA) {
    const int g = c / (D / 8), e = c % (D / 8);
    *reinterpret_cast<u32x4*>(o + static_cast<int64_t>(head0 + g) * a.o_head + 8 * e) = u32x4{0, 0, 0, 0};
  }
}

// A wave's 32 tokens (two 16-token tiles): K rows for the score MFMAs, V rows
// for the output.
template <int D>
struct KTiles {
  u32x4 k[2][AttnShape<D>::kSteps];
};
template <int D>
struct VTiles {
  uint32_t v[2][4][AttnShape<D>::kJ / 2];
};

// A wave's running softmax state: lane (quad, col) holds query col's max and
// sum (the sum over its own rows only) and D / 4 unnormalised outputs.
template <int D>
struct Running {
  f32x4 acc[AttnShape<D>::kJ];
  float m, l;
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int j = 0; j < AttnShape<D>::kJ; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    m = -INFINITY;
    l = 0.f;
  }
};

// Scores of the wave's 32 tokens: lane (quad, col) holds query col's scores
// of tokens 4 * quad + i of each tile.
template <int DT, int D>
__device__ __forceinline__ void pair_scores(const KTiles<D>& T, const u32x4 (&qv)[AttnShape<D>::kSteps],
                                            f32x4 (&sc)[2]) {
  sc[0] = f32x4{0.f, 0.f, 0.f, 0.f};
  sc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < AttnShape<D>::kSteps; i += 2) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u32x4 k0 = T.k[h][i], k1 = T.k[h][i + 1];
      swap_lines(k0, k1);
      sc[h] = mfma_scores<DT>(k0, qv[i], sc[h]);
      sc[h] = mfma_scores<DT>(k1, qv[i + 1], sc[h]);
    }
  }
}

// Online softmax and output of the 32 tokens tb .. tb + 31 (n valid tokens in
// all).  The output MFMAs are 16x16x32 in the cache dtype with A = V^T and
// B = P^T: k-slot (lane / 16, e) is token 4 * (lane / 16) + (e & 3) of tile
// e / 4, i.e. the rows of the lane's own score tiles, and head_dim column m of
// block j is out_dim(m, j), so both operands are in the lane's registers.  P
// is split into an upper part (its fp32 value cut to the dtype) and the dtype
// rounding of the exact remainder; two MFMAs per block keep the products
// within 2^-14 of fp32 probabilities (see split_prob).
template <int DT, int D>
__device__ __forceinline__ void pair_output(const VTiles<D>& T, const f32x4 (&sc)[2], Running<D>& run, int tb, int n,
                                            int quad, float c) {
  constexpr int J = AttnShape<D>::kJ;
  float x[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[i] = (tb + 4 * quad + i < n) ? sc[0][i] * c : -INFINITY;
    x[4 + i] = (tb + kTileT + 4 * quad + i < n) ? sc[1][i] * c : -INFINITY;
  }
  float tmax = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
  tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
  tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
  const float mn = fmaxf(run.m, tmax);
  const float alpha = fast_exp2(run.m - mn);
  float p[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) p[e] = fast_exp2(x[e] - mn);
  run.l = run.l * alpha + (((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7])));
  run.m = mn;
#pragma unroll
  for (int j = 0; j < J; ++j) run.acc[j] *= alpha;
  u32x4 phi, plo;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    uint32_t h0, h1, l0, l1;
    split_prob<DT>(p[2 * w], h0, l0);
    split_prob<DT>(p[2 * w + 1], h1, l1);
    phi[w] = h0 | (h1 << 16);
    plo[w] = l0 | (l1 << 16);
  }
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;  // high or low halves
    const int w = j >> 1;
    u32x4 av;
    av[0] = __builtin_amdgcn_perm(T.v[0][1][w], T.v[0][0][w], sel);
    av[1] = __builtin_amdgcn_perm(T.v[0][3][w], T.v[0][2][w], sel);
    av[2] = __builtin_amdgcn_perm(T.v[1][1][w], T.v[1][0][w], sel);
    av[3] = __builtin_amdgcn_perm(T.v[1][3][w], T.v[1][2][w], sel);
    run.acc[j] = mfma_scores<DT>(av, phi, run.acc[j]);
    run.acc[j] = mfma_scores<DT>(av, plo, run.acc[j]);
  }
}

// LDS of one workgroup's merge: the waves' running max, sum and unnormalised
// outputs.
template <int D>
struct MergeShared {
  alignas(16) float acc[kWavesA][kGroupQ][D + 4];
  float m[kWavesA][kGroupQ];
  float l[kWavesA][kGroupQ];
};

// The waves' states of `gcount` queries go to LDS as they are (then a barrier).
template <int D>
__device__ __forceinline__ void waves_to_lds(MergeShared<D>& sh, const Running<D>& run, int wave, int quad, int col,
                                             int gcount) {
  constexpr int J = AttnShape<D>::kJ;
  float l = run.l;
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (col >= gcount) return;
  if (quad == 0) {
    sh.m[wave][col] = run.m;
    sh.l[wave][col] = l;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int j = 0; j < J; ++j) sh.acc[wave][col][out_dim<J>(4 * quad + i, j)] = run.acc[j][i];
  }
}

// The workgroup's (max, sum, outputs e .. e + 3) of query g: the waves in
// wave order, common max, rescaled sums.
template <int D>
__device__ __forceinline__ f32x4 span_item(const MergeShared<D>& sh, int g, int e, float& mx, float& total_l) {
  mx = sh.m[0][g];
#pragma unroll
  for (int w = 1; w < kWavesA; ++w) mx = fmaxf(mx, sh.m[w][g]);
  total_l = 0.f;
  f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < kWavesA; ++w) {
    const float f = fast_exp2(sh.m[w][g] - mx);
    total_l += sh.l[w][g] * f;
    const f32x4 x = *reinterpret_cast<const f32x4*>(&sh.acc[w][g][e]);
    v = w == 0 ? x * f : v + x * f;
  }
  return v;
}

template <int DT>
__device__ __forceinline__ void store_out(const AttnArgs& a, int row, int head, int e, f32x4 v, float inv) {
  uint16_t* o = static_cast<uint16_t*>(a.out) + row * a.o_row + head * a.o_head + e;
  const uint32_t w0 = static_cast<uint32_t>(Elem<DT>::store(v[0] * inv)) |
                      (static_cast<uint32_t>(Elem<DT>::store(v[1] * inv)) << 16);
  const uint32_t w1 = static_cast<uint32_t>(Elem<DT>::store(v[2] * inv)) |
                      (static_cast<uint32_t>(Elem<DT>::store(v[3] * inv)) << 16);
  *reinterpret_cast<u32x2*>(o) = u32x2{w0, w1};
}

// The workgroup's result of `gcount` queries, written out normalised.
template <int DT, int D>
__device__ __forceinline__ void write_outputs(const AttnArgs& a, const MergeShared<D>& sh, int row, int head0,
                                              int gcount, int tid) {
  constexpr int kChunks = D / 4;
  for (int item = tid; item < gcount * kChunks; item += kThreadsA) {
    const int g = item / kChunks, e = 4 * (item % kChunks);
    float mx, total_l;
    const f32x4 v = span_item<D>(sh, g, e, mx, total_l);
    store_out<DT>(a, row, head0 + g, e, v, 1.f / total_l);
  }
}

// One more span joins a query's running (max, sum, outputs): the spans of a
// row are merged in index order by this one expression, whichever workgroup
// and kernel does it, so a row's result depends on that row alone.
struct Merged {
  float m = -INFINITY, l = 0.f;
  f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
  __device__ __forceinline__ void add(float m_s, float l_s, f32x4 v_s) {
    const float gm = fmaxf(m, m_s);
    const float r1 = fast_exp2(m - gm);
    const float r2 = fast_exp2(m_s - gm);
    l = l * r1 + l_s * r2;
    v = v * r1 + v_s * r2;
    m = gm;
  }
};

// Item (query g, outputs e .. e + 3) of a partial at `off` (bytes, the same
// for all lanes) of the partials, with device-scope stores.  Row g of a
// partial: D outputs, then (max, sum, 0, 0).
template <int D>
__device__ __forceinline__ void store_partial(Rsrc16 prs, int off, int g, int e, float m, float l, f32x4 v) {
  using S = AttnShape<D>;
  store16_sc1(prs, (g * S::kRow + e) * 4, off, v);
  if (e == 0) store16_sc1(prs, (g * S::kRow + D) * 4, off, f32x4{m, l, 0.f, 0.f});
}

// A unit done by several workgroups: this one waits until its partials'
// stores are acknowledged, then counts itself on the unit's counter.  True
// for the one that counts last of `parts`: the others' stores are complete
// before their counts, so it can read them without waiting, and it resets
// the counter for the next launch.
__device__ __forceinline__ bool count_part(const AttnArgs& a, int unit, int parts, int* s_last, int tid) {
  // Device-scope write-throughs: once this thread's are acknowledged they are
  // visible to every workgroup.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    const uint32_t prev =
        __hip_atomic_fetch_add(a.counters + unit, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *s_last = prev == static_cast<uint32_t>(parts - 1) ? 1 : 0;
    if (*s_last) coherent_store(a.counters + unit, 0u);
  }
  lds_barrier();
  return *s_last != 0;
}

// Merge of a unit's `parts` partials in index order (so the result does not
// depend on arrival order); part i is at place_of(i) (bytes, the same for all lanes), part `own` is
// this workgroup's, from own_item(item, max, sum) (none if negative).  The
// others' words of kGroupS parts are requested at once.
template <int DT, int D, typename PlaceOf, typename OwnItem>
__device__ __forceinline__ void merge_partials(const AttnArgs& a, Rsrc16 prs, int row, int head0, int gcount,
                                               int parts, int own, int tid, PlaceOf place_of, OwnItem own_item) {
  using S = AttnShape<D>;
  constexpr int kChunks = D / 4;
  for (int item = tid; item < gcount * kChunks; item += kThreadsA) {
    const int g = item / kChunks;
    const int e = 4 * (item % kChunks);
    Merged run;
    for (int s0 = 0; s0 < parts; s0 += kGroupS) {
      const int cnt = min(kGroupS, parts - s0);
      f32x4 pv[kGroupS];
      f32x2 pml[kGroupS];
#pragma unroll
      for (int u = 0; u < kGroupS; ++u) {
        const int sp = s0 + u;
        if (u < cnt && sp != own) {
          const int at = place_of(sp);
          pv[u] = load16_sc1(prs, (g * S::kRow + e) * 4, at);
          pml[u] = load8_sc1(prs, (g * S::kRow + D) * 4, at);
        }
      }
#pragma unroll
      for (int u = 0; u < kGroupS; ++u) {
        const int sp = s0 + u;
        if (u >= cnt) break;
        float m_s, l_s;
        f32x4 a_s;
        if (sp == own) {
          a_s = own_item(item, m_s, l_s);
        } else {
          m_s = pml[u][0];
          l_s = pml[u][1];
          a_s = pv[u];
        }
        run.add(m_s, l_s, a_s);
      }
    }
    store_out<DT>(a, row, head0 + g, e, run.v, 1.f / run.l);
  }
}

// The new token's K/V rows of one (row, KV head) go into the working cache
// (workgroups of this launch read the input rows in their place).
template <int D>
__device__ __forceinline__ void write_token(const AttnArgs& a, int64_t work_base, int pos, const uint16_t* kin,
                                            const uint16_t* vin, int tid) {
  if (tid < D / 4) {
    const int e = tid % (D / 8);
    const bool is_v = tid >= D / 8;
    uint16_t* dst = static_cast<uint16_t*>(is_v ? a.work_v : a.work_k) + work_base + static_cast<int64_t>(pos) * D;
    *reinterpret_cast<u32x4*>(dst + 8 * e) = load16((is_v ? vin : kin) + 8 * e);
  }
}

// Run by the grid's last workgroup at its end: once every workgroup of the
// pending rows has stored its seen word (all of them have lower indices and
// were dispatched before this one), each row's working length becomes
// position + 1 and the epoch advances.  If that wait expires (on any thread),
// a workgroup may still have its position to read: the working lengths stay
// as they are.  The epoch advances all the same, or the next launch would
// take this one's seen words for its own.
__device__ __forceinline__ void publish(const AttnArgs& a, uint32_t tag, int seen_words) {
  __shared__ int s_expired[kWavesA];
  bool expired = coherent_load(a.header + kHdrGiveUp) != 0u;
  if (expired && threadIdx.x == 0) raise_status(a, kStatusExpired);
  for (int b = threadIdx.x; b < seen_words; b += kThreadsA) {
    if (b != static_cast<int>(blockIdx.x)) await_seen(a, a.seen + b, tag, expired);
  }
  const bool wave_expired = __any(expired);
  if ((threadIdx.x & 63) == 0) s_expired[threadIdx.x >> 6] = wave_expired ? 1 : 0;
  lds_barrier();
  int give_up = 0;
#pragma unroll
  for (int w = 0; w < kWavesA; ++w) give_up |= s_expired[w];
  for (int r = threadIdx.x; r < a.rows; r += kThreadsA) {
    const int slot = a.slots[r];
    int pos = -1;
    if (slot >= 0 && slot < a.num_slots) pos = a.positions ? a.positions[r] : a.working_lens[slot];
    if (pos < 0 || pos >= a.budget) raise_status(a, kStatusPosition);
    else if (give_up == 0) a.working_lens[slot] = pos + 1;
  }
  if (threadIdx.x == 0 && a.rows > 0) coherent_store(a.header + kHdrEpoch, tag);
}

template <int DT, int D>
__global__ __launch_bounds__(kThreadsA, 2) void draft_attention_kernel(AttnArgs a) {
  using S = AttnShape<D>;
  constexpr int J = S::kJ;
  __shared__ MergeShared<D> sh;
  __shared__ int s_last;
  __shared__ int s_pos;
  __shared__ uint32_t s_tag;

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int col = lane & 15;
  const int quad = lane >> 4;
  int b = blockIdx.x;
  const int split = b % a.splits;
  b /= a.splits;
  const int qb = b % a.qblocks;
  b /= a.qblocks;
  const int kvh = b % a.hkv;
  const int row = b / a.hkv;
  const int g0 = qb * kGroupQ;
  const int gcount = min(kGroupQ, a.group - g0);
  const int head0 = kvh * a.group + g0;

  // Thread 0 reads the launch epoch (tag = epoch + 1) and, for a pending
  // row, the row's position (scalar loads), then stores this workgroup's
  // tagged "seen" word.  The grid's last workgroup waits for every seen word
  // before it advances working_lens and the epoch, so no workgroup reads
  // either after they change.  No atomics: every word has one writer.
  const bool real = row < a.rows;
  const int slot = real ? scalar_load(a.slots + row) : -1;
  const bool slot_ok = slot >= 0 && slot < a.num_slots;
  if (threadIdx.x == 0) {
    const uint32_t epoch = static_cast<uint32_t>(scalar_load(reinterpret_cast<const int32_t*>(a.header + kHdrEpoch)));
    int pos = -1;
    if (real && slot_ok) pos = a.positions ? scalar_load(a.positions + row) : scalar_load(a.working_lens + slot);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    s_pos = (pos >= 0 && pos < a.budget) ? pos : -1;
    s_tag = epoch + 1;
    if (real) coherent_store(a.seen + blockIdx.x, tagged(epoch + 1, 0.f));
  }

  const int64_t work_base = (static_cast<int64_t>(slot_ok ? slot : 0) * a.hkv + kvh) * a.budget * D;
  const uint16_t* kw = static_cast<const uint16_t*>(a.work_k) + work_base;
  const uint16_t* vw = static_cast<const uint16_t*>(a.work_v) + work_base;
  const uint16_t* kin = static_cast<const uint16_t*>(a.k_in) + row * a.k_row + kvh * a.k_head;
  const uint16_t* vin = static_cast<const uint16_t*>(a.v_in) + row * a.v_row + kvh * a.v_head;
  const int t0 = split * S::kSpan + wave * S::kTiles * kTileT;

  // Loads of the 32 tokens from tb on, from the working rows only (rows clamped to the
  // cache); the rows from the position on are fixed up once it is known.
  auto load_rows = [&](KTiles<D>& K, VTiles<D>& V, int tb) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < S::kSteps; ++i) {
        const int t = min(tb + h * kTileT + line_token(col, i), a.budget - 1);
        K.k[h][i] = load16(kw + static_cast<int64_t>(t) * D + line_elem(quad, col, i));
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = min(tb + h * kTileT + 4 * quad + r, a.budget - 1);
        load_words<J>(vw + static_cast<int64_t>(t) * D + v_elem<J>(col), V.v[h][r]);
      }
    }
  };
  // The first pair of the wave's tiles and this row's input K / V slices are
  // requested before the position arrives (the position is a second
  // dependent load after the slot).  Every address is valid whatever the
  // position: working rows below the cache capacity and the input row.
  KTiles<D> k0, k1;
  VTiles<D> v0, v1;
  u32x4 kin_s[S::kSteps / 2];  // the lane's slice of each line
  uint32_t vin_s[J / 2];
  const bool early = real && slot_ok && t0 < a.budget;
  if (early) {
    load_rows(k0, v0, t0);
#pragma unroll
    for (int i = 0; i < S::kSteps; i += 2) kin_s[i / 2] = load16(kin + line_elem(quad, col, i));
    load_words<J>(vin + v_elem<J>(col), vin_s);
  }
  lds_barrier();
  const int pos = s_pos;
  const uint32_t tag = s_tag;
  const bool valid = pos >= 0;
  const int n = valid ? pos + 1 : 0;
  const int active = valid ? (n + S::kSpan - 1) / S::kSpan : 1;
  auto finish = [&]() {
    if (blockIdx.x == gridDim.x - 1) publish(a, tag, a.rows * a.hkv * a.qblocks * a.splits);
  };

  if (!real) {  // padding row: zero once
    if (split == 0) zero_heads<D>(a, row, head0, gcount);
    finish();
    return;
  }
  if (split >= active) {
    finish();
    return;
  }
  if (!valid) {  // bad slot or position: zero output, touch nothing else
    zero_heads<D>(a, row, head0, gcount);
    finish();
    return;
  }

  // Query block as the B operand of the score MFMAs: lane (quad, col) holds
  // q[head0 + col][32 i + 8 quad .. + 8]; columns past the group are zero.
  // Every load of the main loop is unconditional (addresses clamped to valid
  // rows, results masked by value), so the compiler can keep the next tile's
  // loads in flight while the current tile is computed.
  u32x4 qv[S::kSteps];
  {
    const int qcol = min(col, gcount - 1);
    const uint16_t* qp = static_cast<const uint16_t*>(a.q) + row * a.q_row + (head0 + qcol) * a.q_head + 8 * quad;
#pragma unroll
    for (int i = 0; i < S::kSteps; ++i) {
      const u32x4 v = load16(qp + 32 * i);
      qv[i] = col < gcount ? v : u32x4{0, 0, 0, 0};
    }
  }

  Running<D> run;
  run.clear();
  const float c = a.scale * kLog2e;

  // Rows at or past n read row n - 1 = pos (the new token's input row): a
  // valid, finite row whose scores are masked to -inf below.
  auto row_ptr = [&](const uint16_t* work, const uint16_t* in, int t) {
    return t >= pos ? in : work + static_cast<int64_t>(t) * D;
  };
  auto load_pair = [&](KTiles<D>& K, VTiles<D>& V, int tb) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < S::kSteps; ++i) {
        K.k[h][i] = load16(row_ptr(kw, kin, tb + h * kTileT + line_token(col, i)) + line_elem(quad, col, i));
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        load_words<J>(row_ptr(vw, vin, tb + h * kTileT + 4 * quad + r) + v_elem<J>(col), V.v[h][r]);
      }
    }
  };
  // A pair loaded from the working rows: the position's row becomes the
  // input row, later rows of V become zeros (their probabilities are 0, and
  // stale cache words may not be finite; K rows there only feed masked
  // scores).
  auto fix_pair = [&](KTiles<D>& K, VTiles<D>& V, int tb) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < S::kSteps; ++i) {
        if (tb + h * kTileT + line_token(col, i) == pos) K.k[h][i] = kin_s[i / 2];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = tb + h * kTileT + 4 * quad + r;
#pragma unroll
        for (int w = 0; w < J / 2; ++w) V.v[h][r][w] = t == pos ? vin_s[w] : (t > pos ? 0u : V.v[h][r][w]);
      }
    }
  };
  auto compute_pair = [&](const KTiles<D>& K, const VTiles<D>& V, int tb) {
    f32x4 sc[2];
    pair_scores<DT, D>(K, qv, sc);
    pair_output<DT, D>(V, sc, run, tb, n, quad, c);
  };

  // The first pair came from the working rows and is fixed up here; the
  // second pair is requested now, before the first is computed (the
  // scheduling barrier keeps the compiler from sinking the loads next to
  // their use); a pair wholly past n is loaded (cache hits on row pos) but
  // not computed.
  if (t0 < n) {
    fix_pair(k0, v0, t0);
    if constexpr (S::kTiles == 4) {
      load_pair(k1, v1, t0 + 2 * kTileT);
      __builtin_amdgcn_sched_barrier(0);
      compute_pair(k0, v0, t0);
      if (t0 + 2 * kTileT < n) compute_pair(k1, v1, t0 + 2 * kTileT);
    } else {
      compute_pair(k0, v0, t0);
    }
  }

  if (qb == 0 && split == pos / S::kSpan) write_token<D>(a, work_base, pos, kin, vin, threadIdx.x);
  waves_to_lds<D>(sh, run, wave, quad, col, gcount);
  lds_barrier();
  if (active == 1) {
    write_outputs<DT, D>(a, sh, row, head0, gcount, threadIdx.x);
    finish();
    return;
  }

  // Several spans: the one that counts last merges the row's partials.
  const int unit = (row * a.hkv + kvh) * a.qblocks + qb;
  constexpr int kPartBytes = kGroupQ * S::kRow * 4;
  const Rsrc16 prs = make_rsrc16(a.partials + static_cast<int64_t>(unit) * a.splits * kGroupQ * S::kRow,
                                 static_cast<int64_t>(a.splits) * kPartBytes);
  for (int item = threadIdx.x; item < gcount * (D / 4); item += kThreadsA) {
    const int g = item / (D / 4), e = 4 * (item % (D / 4));
    float mx, total_l;
    const f32x4 v = span_item<D>(sh, g, e, mx, total_l);
    store_partial<D>(prs, split * kPartBytes, g, e, mx, total_l, v);
  }
  if (count_part(a, unit, active, &s_last, threadIdx.x)) {
    merge_partials<DT, D>(
        a, prs, row, head0, gcount, active, split, threadIdx.x, [](int sp) { return sp * kPartBytes; },
        [&](int item, float& m, float& l) { return span_item<D>(sh, item / (D / 4), 4 * (item % (D / 4)), m, l); });
  }
  finish();
}

// ---- Batches of more than one round of spans --------------------------------
// The same attention with the work dealt evenly.  Bound by HBM reads; one
// workgroup per span lost to it on large batches: every workgroup pays its
// own ramp, wave merge and partial, rows' empty spans are launched too, and
// the last round of workgroups is partly empty.
//   - The spans of every (row, KV head, query block) unit are numbered unit
//     by unit (a prefix sum over the rows' positions, in LDS), and each
//     resident workgroup takes one contiguous range, so all end together
//     whatever the rows' lengths.
//   - Within a unit a wave requests the next 32 tokens' K as soon as the score
//     MFMAs have read the current K, and the next V after the output MFMAs.
//   - Each span is computed and merged over the waves as the one-shot kernel
//     does it, and the spans join in index order (Merged): a row's bits are
//     the same in either kernel, whatever the other rows are and wherever the
//     ranges end.
//   - A unit inside one range is finished in place.  A unit cut by range
//     ends (a range has two such units at most) leaves its first range's sum
//     and the later ranges' spans as partials, and the workgroup that counts
//     last on it continues the sum.
// us on 57 rows of 300-3970 tokens (64/8 heads x 128, fp16) / 64 rows of 1987
// (32/4 x 128) / 16 rows of 1984-3990 (32/8 x 256) / 48 rows of 984-1990
// (32/8 x 64); bandwidth of the last line 5.6, 6.1, 5.3 and 4.4 TB/s:
//   one workgroup per span, cached half lines             184 / 63 / 130 / 43.5
//   cut at any 128 tokens, one partial per range (a row's
//     rounding then depends on the other rows)            98 / 42.7 / 70 / 30.1
//   whole spans, later ranges' spans stored one by one    97 / 43.4 / 79 / 34.5
//   held in LDS and stored when the unit ends, kept       96 / 43.0 / 74 / 33.8
// The stores are what the later ranges' spans cost (without them 90 / - / 71 /
// 30.8; writes at about 1% of the read bytes).  2 workgroups per CU at
// head_dim 64 (1: 39); 1 else, where 4 waves x 16 KB in flight per CU already
// fill the memory queue.
template <int D>
struct StreamShape {
  static constexpr int kPerCu = D == 64 ? 2 : 1;            // workgroups per CU
  static constexpr int kHeld = (D == 64 ? 40 : 64) * 1024;  // LDS bytes of held span results
  // Spans above which the batch is streamed: about one round of one-shot
  // workgroups (4 per CU at head_dim 64, 2 at 128).  us, one-shot against
  // streamed, at 512 spans of head_dim 128: 16.6 / 17.2 (16 rows of 1987
  // tokens), 14.4 / 17.2 (64 rows of 184-487); 576: 21.8 / 22.5; 768: 26.9 /
  // 24.1 (1987 tokens), 22.7 / 17.9 (100-1987).  Head_dim 64, 1152 spans:
  // 19.9 / 22.5 (36 x 1987); 1280: 18.9 / 18.3 (100-1987), 22.6 / 23.9 (20 x
  // 4032); 1472: 26.1 / 26.7; 1536: 26.4 / 26.6 (1987); 1792: 30.2 / 28.0; 4096:
  // 53.3 / 41.1 (1000-1987).  Head_dim 256, 320 spans: 21.5 / 20.7; 384: 18.0 /
  // 19.3 (12 x 950), 27.4 / 24.9 (3 x 4032); 576: 28.5 / 27.7; 1024: 43.5 / 32.5.
  static constexpr int kOneRound = D == 64 ? 1536 : (D == 128 ? 576 : 256);
};

struct Ranges {  // workgroup w < used takes spans [start(w), start(w + 1))
  int base, rem, used;
  __device__ __forceinline__ int start(int w) const { return w * base + min(w, rem); }
  __device__ __forceinline__ int owner(int x) const {
    const int wide = rem * (base + 1);
    return __builtin_amdgcn_readfirstlane(x < wide ? x / (base + 1) : rem + (x - wide) / base);
  }
};

template <int DT, int D>
__global__ __launch_bounds__(kThreadsA, StreamShape<D>::kPerCu) void attention_stream_kernel(AttnArgs a) {
  using S = AttnShape<D>;
  constexpr int J = S::kJ;
  constexpr int kPairs = S::kTiles / 2;  // 32-token pairs of a wave's quarter of a span
  constexpr int kChunks = D / 4;
  constexpr int kItems = kGroupQ * kChunks / kThreadsA;  // merge items per thread
  __shared__ MergeShared<D> sh;
  __shared__ f32x4 s_held[StreamShape<D>::kHeld / sizeof(f32x4)];  // span results not stored yet
  __shared__ int s_prefix[kMaxRows + 1];  // spans of one unit of each row, exclusive prefix
  __shared__ int s_pos[kMaxRows];
  __shared__ int s_slot[kMaxRows];
  __shared__ int s_scratch[4];
  __shared__ int s_last;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15;
  const int quad = lane >> 4;
  const int units_row = a.hkv * a.qblocks;

  const uint32_t tag =
      static_cast<uint32_t>(scalar_load(reinterpret_cast<const int32_t*>(a.header + kHdrEpoch))) + 1u;
  build_row_prefix(a.rows, s_prefix, s_scratch, [&](int r) {
    const int slot = a.slots[r];
    int pos = -1;
    if (slot >= 0 && slot < a.num_slots) pos = a.positions ? a.positions[r] : a.working_lens[slot];
    if (pos >= a.budget) pos = -1;
    s_pos[r] = max(pos, -1);
    s_slot[r] = slot;
    return pos >= 0 ? (pos + S::kSpan) / S::kSpan : 0;
  });
  // Every thread's reads of the positions and the epoch have landed (the
  // prefix's barriers waited for them): the workgroup's seen word may go out.
  if (threadIdx.x == 0 && a.rows > 0) coherent_store(a.seen + blockIdx.x, tagged(tag, 0.f));

  // Padding rows and rows with a bad slot or position are zero.
  for (int r = blockIdx.x; r < a.out_rows; r += gridDim.x) {
    if (r >= a.rows || s_pos[r] < 0) zero_heads<D>(a, r, 0, a.hq);
  }

  const int total = __builtin_amdgcn_readfirstlane(s_prefix[a.rows]) * units_row;
  Ranges st;
  st.used = min(static_cast<int>(gridDim.x), max(1, total));
  st.base = __builtin_amdgcn_readfirstlane(total / st.used);
  st.rem = total - st.base * st.used;
  const int w = blockIdx.x;
  const int first = w < st.used ? st.start(w) : 0;
  const int end = w < st.used ? st.start(w + 1) : 0;

  // One unit: row, KV head, query block and its spans [s0, s0 + count).
  struct Unit {
    int row, kvh, qb, s0, count, pos;
    int64_t work;  // element offset of the working rows
  };
  int row_hint = 0;
  auto unit_at = [&](int s) {
    int lo = row_hint, hi = a.rows - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (s_prefix[mid] * units_row <= s) lo = mid; else hi = mid - 1;
    }
    Unit u;
    u.row = __builtin_amdgcn_readfirstlane(lo);
    row_hint = u.row;
    u.pos = __builtin_amdgcn_readfirstlane(s_pos[u.row]);
    u.count = (u.pos + S::kSpan) / S::kSpan;
    const int base = __builtin_amdgcn_readfirstlane(s_prefix[u.row]) * units_row;
    const int k = __builtin_amdgcn_readfirstlane((s - base) / u.count);
    u.s0 = base + k * u.count;
    u.kvh = __builtin_amdgcn_readfirstlane(k / a.qblocks);
    u.qb = k - u.kvh * a.qblocks;
    const int slot = __builtin_amdgcn_readfirstlane(s_slot[u.row]);
    u.work = (static_cast<int64_t>(slot) * a.hkv + u.kvh) * a.budget * D;
    // Made scalar: quotients are computed in vector registers, and a buffer
    // resource held there costs a loop over the lanes at every load.
    u.s0 = __builtin_amdgcn_readfirstlane(u.s0);
    u.count = __builtin_amdgcn_readfirstlane(u.count);
    u.qb = __builtin_amdgcn_readfirstlane(u.qb);
    u.work = uniform64(u.work);
    return u;
  };
  // This wave's quarter of span s starts at token_of(u, s).
  auto token_of = [&](const Unit& u, int s) { return (s - u.s0) * S::kSpan + wave * (S::kTiles * kTileT); };
  auto kin_of = [&](const Unit& u) { return static_cast<const uint16_t*>(a.k_in) + u.row * a.k_row + u.kvh * a.k_head; };
  auto vin_of = [&](const Unit& u) { return static_cast<const uint16_t*>(a.v_in) + u.row * a.v_row + u.kvh * a.v_head; };
  // Loads of the 32 tokens from tb on: buffer loads whose resource ends at the
  // position, so rows from there on are zeros and cost nothing.  One path for
  // every tile: with a branch here the compiler sees a path on which V was not
  // requested after K, and its waits for K wait for V too.
  const int k_lane = (line_token(col, 0) * D + line_elem(quad, col, 0)) * 2;
  const int v_lane = (4 * quad * D + v_elem<J>(col)) * 2;
  auto tile_rows = [&](const void* work, const Unit& u, int t) {  // (made scalar: see unit_at)
    const int bytes = __builtin_amdgcn_readfirstlane(min(max(u.pos - t, 0), kTileT) * D * 2);
    return make_rsrc16(static_cast<const uint16_t*>(work) + uniform64(u.work + static_cast<int64_t>(t) * D), bytes);
  };
  auto load_k = [&](KTiles<D>& T, const Unit& u, int tb) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const Rsrc16 r = tile_rows(a.work_k, u, tb + h * kTileT);
#pragma unroll
      for (int i = 0; i < S::kSteps; ++i) {
        T.k[h][i] = __builtin_amdgcn_raw_buffer_load_b128(r, k_lane + 16 * (i & 1) * D + 128 * (i >> 1), 0, kPolicyNt);
      }
    }
  };
  auto load_v = [&](VTiles<D>& T, const Unit& u, int tb) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const Rsrc16 r = tile_rows(a.work_v, u, tb + h * kTileT);
#pragma unroll
      for (int i = 0; i < 4; ++i) load_words_buf<J>(r, v_lane + i * D * 2, 0, T.v[h][i]);
    }
  };
  // The position's row is the new token's input row: the lane's slices of it,
  // loaded with the unit's queries, go into the tile that holds the position.
  u32x4 kin_s[S::kSteps / 2];
  uint32_t vin_s[J / 2];
  auto fix_k = [&](KTiles<D>& T, int at) {  // at = position - first token of the pair
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < S::kSteps; ++i) {
        if (h * kTileT + line_token(col, i) == at) T.k[h][i] = kin_s[i / 2];
      }
    }
  };
  auto fix_v = [&](VTiles<D>& T, int at) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int w = 0; w < J / 2; ++w) T.v[h][i][w] = h * kTileT + 4 * quad + i == at ? vin_s[w] : T.v[h][i][w];
      }
    }
  };
  u32x4 qv[S::kSteps];
  auto load_q = [&](const Unit& u) {  // columns past the unit's queries hold its last one and are not read out
    const int g0 = u.qb * kGroupQ, gcount = min(kGroupQ, a.group - g0);
    const uint16_t* qp = static_cast<const uint16_t*>(a.q) + u.row * a.q_row +
                         (u.kvh * a.group + g0 + min(col, gcount - 1)) * a.q_head + 8 * quad;
#pragma unroll
    for (int i = 0; i < S::kSteps; ++i) qv[i] = load16(qp + 32 * i);
#pragma unroll
    for (int i = 0; i < S::kSteps; i += 2) kin_s[i / 2] = load16(kin_of(u) + line_elem(quad, col, i));
    load_words<J>(vin_of(u) + v_elem<J>(col), vin_s);
  };

  constexpr int kPartBytes = kGroupQ * S::kRow * 4;
  const float c = a.scale * kLog2e;
  for (int s = first; s < end;) {
    const Unit u = unit_at(s);
    const int unit_end = u.s0 + u.count;
    const int stop = min(unit_end, end);  // this range's spans of the unit: [s, stop)
    const bool head = __builtin_amdgcn_readfirstlane(s == u.s0 ? 1 : 0) != 0;
    const int n = u.pos + 1;
    const int g0 = u.qb * kGroupQ, gcount = min(kGroupQ, a.group - g0);
    const int head0 = u.kvh * a.group + g0;
    const int unit = (u.row * a.hkv + u.kvh) * a.qblocks + u.qb;
    const Rsrc16 prs = make_rsrc16(a.partials + static_cast<int64_t>(unit) * a.splits * kGroupQ * S::kRow,
                                   static_cast<int64_t>(a.splits) * kPartBytes);
    // The unit's first range merges its spans in sum.  A later range holds
    // each span's result in LDS, every thread its own items, and stores them
    // when the unit (or the room) ends: a store among the loads delays the
    // span.
    Merged sum[kItems];
    const int entries = gcount * (kChunks + 1);  // per held span: the outputs, then each query's (max, sum)
    const int room = (StreamShape<D>::kHeld / static_cast<int>(sizeof(f32x4))) / entries;
    int held = 0, held_at = s - u.s0;  // spans held, the first one's index in the unit
    auto store_held = [&]() {
      for (int h = 0; h < held; ++h) {
        const int place = __builtin_amdgcn_readfirstlane((held_at + h) * kPartBytes);
        for (int item = threadIdx.x; item < gcount * kChunks; item += kThreadsA) {
          const int g = item / kChunks, e = 4 * (item % kChunks);
          const f32x4 ml = s_held[h * entries + gcount * kChunks + g];
          store_partial<D>(prs, place, g, e, ml[0], ml[1], s_held[h * entries + item]);
        }
      }
      held_at += held;
      held = 0;
    };
    KTiles<D> K;
    VTiles<D> V;
    load_q(u);
    load_k(K, u, token_of(u, s));
    load_v(V, u, token_of(u, s));
    Running<D> run;
    run.clear();
    int tb = token_of(u, s), p = 0;
    // One pair; MORE: the next one's loads are issued on the way (on every
    // path: see load_k).
    auto pair = [&](auto more) {
      constexpr bool MORE = decltype(more)::value;
      const bool span_end = !MORE || p == kPairs - 1;
      const int next = span_end ? token_of(u, s + 1) : tb + 2 * kTileT;
      const int at = __builtin_amdgcn_readfirstlane(u.pos - tb);
      const bool holds_pos = at >= 0 && at < 2 * kTileT;  // wave-uniform
      f32x4 sc[2];
      if (holds_pos) fix_k(K, at);
      pair_scores<DT, D>(K, qv, sc);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (MORE) load_k(K, u, next);
      __builtin_amdgcn_sched_barrier(0);
      if (tb < n) {
        if (holds_pos) fix_v(V, at);
        pair_output<DT, D>(V, sc, run, tb, n, quad, c);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (MORE) load_v(V, u, next);
      tb = next;
      ++p;
      if (!span_end) return;
      lds_barrier();  // every wave has read the previous span's states
      waves_to_lds<D>(sh, run, wave, quad, col, gcount);
      lds_barrier();
#pragma unroll
      for (int i = 0; i < kItems; ++i) {
        const int item = threadIdx.x + i * kThreadsA;
        if (item < gcount * kChunks) {
          const int g = item / kChunks, e = 4 * (item % kChunks);
          float mx, total_l;
          const f32x4 v = span_item<D>(sh, g, e, mx, total_l);
          if (head) {
            sum[i].add(mx, total_l, v);
          } else {
            s_held[held * entries + item] = v;
            if (e == 0) s_held[held * entries + gcount * kChunks + g] = f32x4{mx, total_l, 0.f, 0.f};
          }
        }
      }
      if (!head && ++held == room) store_held();
      run.clear();
      ++s;
      p = 0;
    };
    for (int left = (stop - s) * kPairs; left > 1; --left) pair(std::true_type{});
    pair(std::false_type{});
    if (u.qb == 0 && stop == unit_end) write_token<D>(a, u.work, u.pos, kin_of(u), vin_of(u), threadIdx.x);
    if (head && stop == unit_end) {
#pragma unroll
      for (int i = 0; i < kItems; ++i) {
        const int item = threadIdx.x + i * kThreadsA;
        if (item < gcount * kChunks) {
          store_out<DT>(a, u.row, head0 + item / kChunks, 4 * (item % kChunks), sum[i].v, 1.f / sum[i].l);
        }
      }
      continue;
    }
    // A unit cut by range ends: its first range's sum is the first part, the
    // later ranges' spans the others.  The first range is mostly the last to
    // end (it meets the unit at its end, the others at their start): it looks
    // whether all others have counted before it stores anything.
    const int w0 = st.owner(u.s0);
    const int ranges = st.owner(unit_end - 1) - w0 + 1;
    const int skip = __builtin_amdgcn_readfirstlane(st.start(w0 + 1) - u.s0 - 1);  // spans of the sum besides span 0
    bool last = false;
    if (head) {
#pragma unroll
      for (int i = 0; i < kItems; ++i) {  // (nothing is held in a first range)
        const int item = threadIdx.x + i * kThreadsA;
        if (item < gcount * kChunks) {
          s_held[item] = sum[i].v;
          if (item % kChunks == 0) s_held[gcount * kChunks + item / kChunks] = f32x4{sum[i].m, sum[i].l, 0.f, 0.f};
        }
      }
      if (threadIdx.x == 0) {
        s_last = coherent_load(a.counters + unit) == static_cast<uint32_t>(ranges - 1) ? 1 : 0;
        if (s_last != 0) coherent_store(a.counters + unit, 0u);
      }
      lds_barrier();
      last = __builtin_amdgcn_readfirstlane(s_last) != 0;
      if (!last) held = 1;
    }
    if (!last) {
      store_held();
      last = count_part(a, unit, ranges, &s_last, threadIdx.x);
    }
    if (last) {
      merge_partials<DT, D>(
          a, prs, u.row, head0, gcount, u.count - skip, head ? 0 : -1, threadIdx.x,
          [skip](int i) { return (i == 0 ? 0 : i + skip) * kPartBytes; },
          [&](int item, float& m, float& l) {
            const f32x4 ml = s_held[gcount * kChunks + item / kChunks];
            m = ml[0];
            l = ml[1];
            return s_held[item];
          });
    }
  }
  if (blockIdx.x == gridDim.x - 1) publish(a, tag, gridDim.x);
}

template <int DT, int D>
int launch_attention(hipStream_t stream, const AttnArgs& a) {
  const int64_t spans = static_cast<int64_t>(a.rows) * a.hkv * a.qblocks * a.splits;
  // (32-bit span numbers and byte offsets within a unit's rows.)
  if (spans > StreamShape<D>::kOneRound && spans < (int64_t{1} << 30) && static_cast<int64_t>(a.budget) * D * 2 < INT32_MAX) {
    // (One seen word per workgroup, out of the workspace's one per span.)
    const int64_t grid = std::min<int64_t>(static_cast<int64_t>(StreamShape<D>::kPerCu) * device_cu_count(), spans);
    attention_stream_kernel<DT, D><<<static_cast<unsigned>(grid), kThreadsA, 0, stream>>>(a);
    return check_launch("ds_draft_attention");
  }
  const int64_t grid = static_cast<int64_t>(a.out_rows) * a.hkv * a.qblocks * a.splits;
  draft_attention_kernel<DT, D><<<static_cast<unsigned>(grid), kThreadsA, 0, stream>>>(a);
  return check_launch("ds_draft_attention");
}

int span_for(int head_dim) { return head_dim <= 128 ? kWavesA * 4 * kTileT : kWavesA * 2 * kTileT; }

size_t seen_bytes(size_t wgs) { return (wgs * sizeof(uint64_t) + 255) / 256 * 256; }

size_t attention_workspace_bytes(int rows, int num_q_heads, int num_kv_heads, int head_dim, int token_budget) {
  if (rows <= 0 || num_q_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 || token_budget <= 0) return 0;
  if (num_q_heads % num_kv_heads) return 0;
  const int group = num_q_heads / num_kv_heads;
  const int qblocks = (group + kGroupQ - 1) / kGroupQ;
  const int splits = (token_budget + span_for(head_dim) - 1) / span_for(head_dim);
  const size_t units = static_cast<size_t>(rows) * num_kv_heads * qblocks;
  const size_t wgs = units * splits;
  return kHeaderBytes + kCounterBytes + seen_bytes(wgs) + wgs * kGroupQ * (head_dim + 4) * sizeof(float);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int draft_attention_impl(hipStream_t stream, int dtype, const void* query, int64_t q_row, int64_t q_head,
                         const void* key, int64_t k_row, int64_t k_head, const void* value, int64_t v_row,
                         int64_t v_head, void* out, int64_t o_row, int64_t o_head, void* working_key,
                         void* working_value, int32_t* working_lens, const int32_t* slots,
                         const int32_t* positions, int rows, int out_rows, int num_slots, int num_q_heads,
                         int num_kv_heads, int head_dim, int token_budget, float scale, void* workspace,
                         size_t workspace_bytes) {
  DS_REQUIRE(rows >= 0 && out_rows >= rows, "output rows must cover the pending rows");
  DS_REQUIRE(num_slots > 0 && token_budget > 0 && head_dim > 0, "working cache shape must be positive");
  DS_REQUIRE(num_q_heads > 0 && num_kv_heads > 0 && num_q_heads % num_kv_heads == 0,
             "query heads must be a positive multiple of KV heads");
  DS_REQUIRE(rows <= num_slots, "more pending rows than working-cache slots");
  DS_SUPPORTED(dtype == DS_BF16 || dtype == DS_FP16, "draft attention runs on BF16 or FP16 tensors");
  DS_SUPPORTED(head_dim == 64 || head_dim == 128 || head_dim == 256, "draft attention head_dim must be 64, 128 or 256");
  DS_SUPPORTED(out_rows <= kMaxRows, "at most %d output rows per launch (got %d)", kMaxRows, out_rows);
  const int group = num_q_heads / num_kv_heads;
  const int qblocks = (group + kGroupQ - 1) / kGroupQ;
  DS_SUPPORTED(static_cast<int64_t>(out_rows) * num_kv_heads * qblocks <= kMaxUnits,
               "at most %d (row, KV head, 16-query block) units per launch", kMaxUnits);
  if (out_rows == 0) return clear_error();
  DS_REQUIRE(query && out && (rows == 0 || (key && value && working_key && working_value && working_lens && slots)),
             "null tensor pointer");
  DS_REQUIRE(workspace, "draft attention needs a workspace");
  const size_t need = attention_workspace_bytes(rows > 0 ? rows : 1, num_q_heads, num_kv_heads, head_dim,
                                                token_budget);
  DS_REQUIRE(workspace_bytes >= need, "attention workspace too small: %zu bytes, need %zu", workspace_bytes, need);
  DS_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 255u) == 0, "workspace must be 256-byte aligned");
  // 16-byte vector accesses: every row and head start must be 16-byte aligned.
  DS_REQUIRE(aligned16(query) && aligned16(out) && q_row % 8 == 0 && q_head % 8 == 0 && o_row % 8 == 0 &&
                 o_head % 8 == 0,
             "query and output rows and heads must start on 16-byte boundaries");
  DS_REQUIRE(rows == 0 || (aligned16(key) && aligned16(value) && aligned16(working_key) &&
                           aligned16(working_value) && k_row % 8 == 0 && k_head % 8 == 0 && v_row % 8 == 0 &&
                           v_head % 8 == 0),
             "key, value and working caches must start rows and heads on 16-byte boundaries");

  AttnArgs a{};
  a.q = query; a.q_row = q_row; a.q_head = q_head;
  a.k_in = key; a.k_row = k_row; a.k_head = k_head;
  a.v_in = value; a.v_row = v_row; a.v_head = v_head;
  a.out = out; a.o_row = o_row; a.o_head = o_head;
  a.work_k = working_key; a.work_v = working_value;
  a.working_lens = working_lens; a.slots = slots; a.positions = positions;
  a.rows = rows; a.out_rows = out_rows; a.num_slots = num_slots;
  a.hq = num_q_heads; a.hkv = num_kv_heads; a.group = group; a.qblocks = qblocks;
  a.budget = token_budget;
  a.splits = (token_budget + span_for(head_dim) - 1) / span_for(head_dim);
  a.scale = scale;
  char* ws = static_cast<char*>(workspace);
  a.header = reinterpret_cast<uint32_t*>(ws);
  const size_t units = static_cast<size_t>(rows) * num_kv_heads * qblocks;
  a.counters = reinterpret_cast<uint32_t*>(ws + kHeaderBytes);
  a.seen = reinterpret_cast<uint64_t*>(ws + kHeaderBytes + kCounterBytes);
  a.partials = reinterpret_cast<float*>(ws + kHeaderBytes + kCounterBytes + seen_bytes(units * a.splits));

#define DS_ATTN_CASE(DTV, DV) \
  if (dtype == DTV && head_dim == DV) return launch_attention<DTV, DV>(stream, a);
  DS_ATTN_CASE(DS_BF16, 64) DS_ATTN_CASE(DS_BF16, 128) DS_ATTN_CASE(DS_BF16, 256)
  DS_ATTN_CASE(DS_FP16, 64) DS_ATTN_CASE(DS_FP16, 128) DS_ATTN_CASE(DS_FP16, 256)
#undef DS_ATTN_CASE
  return set_error(DS_ERR_UNSUPPORTED, "unsupported draft attention shape");
}

}  // namespace
}  // namespace ds355

extern "C" size_t ds_draft_attention_workspace_bytes(int batch_rows, int num_q_heads, int num_kv_heads,
                                                     int head_dim, int token_budget) {
  return ds355::attention_workspace_bytes(batch_rows, num_q_heads, num_kv_heads, head_dim, token_budget);
}

extern "C" int ds_draft_attention(ds_stream_t stream, int dtype, const void* query, int64_t q_row_stride,
                                  int64_t q_head_stride, const void* key, int64_t k_row_stride,
                                  int64_t k_head_stride, const void* value, int64_t v_row_stride,
                                  int64_t v_head_stride, void* out, int64_t o_row_stride, int64_t o_head_stride,
                                  void* working_key, void* working_value, int32_t* working_lens,
                                  const int32_t* slots, const int32_t* positions, int rows, int out_rows,
                                  int num_slots, int num_q_heads, int num_kv_heads, int head_dim, int token_budget,
                                  float scale, void* workspace, size_t workspace_bytes) {
  return ds355::draft_attention_impl(reinterpret_cast<hipStream_t>(stream), dtype, query, q_row_stride,
                                     q_head_stride, key, k_row_stride, k_head_stride, value, v_row_stride,
                                     v_head_stride, out, o_row_stride, o_head_stride, working_key, working_value,
                                     working_lens, slots, positions, rows, out_rows, num_slots, num_q_heads,
                                     num_kv_heads, head_dim, token_budget, scale, workspace, workspace_bytes);
}
