// Shared kernel parameters and helpers of the flash-spacetime HIP library.
#pragma once

#include "fst_device.h"
#include "../../include/flash_spacetime.h"

namespace fst {

// Event layout shared by every kernel: padded [B, H, L, X] with seqlens, or
// packed [T, H, X] with cu_seqlens (forward.py:247-255, _tiles.py:80-117).
// Padded events may also be stored token-major, [B, L, H, X] (vectors
// [B, L, H]): the layout a [B, L, H*D] projection has before its heads are
// split, so the heads-first views a model passes are read in place.
struct EventSpec {
  const int32_t* lens;    // seqlens [B] (padded) or the work list's sanitised cu_seqlens [B+1] (packed)
  const int32_t* blkcum;  // [B+1] prefix sums of row blocks per event
  const int32_t* perm;    // [B] events by decreasing length (the tile kernels' schedules)
  const int32_t* scum;    // [B+1] packed: prefix sums of row blocks in perm order; padded: null
  // [8 ceil(B / 8) + 1] padded: prefix sums of the valid (not padding-only)
  // 16-row tiles over the events in XCD order (entry x S + j: XCD x's j-th
  // event, S = ceil(B / 8)), for tile_block's padding-last schedule; or null.
  const int32_t* vp;
  const float4* pos4;     // [B*L] or [T] (x, y, z, t) fp32
  const int32_t* status;  // the work list's verdict on the call's lengths: 0 = well formed (or null)
  int B, H, L, T, packed;
  int tokmajor;           // rows of one token's heads are adjacent (packed, or padded token-major)
  int xmul;               // 3: q, k, v (and dq, dk, dv) interleaved per token as [.., 3, H, X]; else 1
  int max_len;            // longest event whose rows of all heads span less than 2^31 bytes
  // No work list: lens are the caller's (the raw cu_seqlens when packed) and
  // every workgroup forms the lists it needs itself (InlineList); blkcum,
  // perm, scum, vp and status are null. Calls of up to kInlineEvents events
  // (fst_capi.hip: inline_list).
  int inl;
};

// tile0: the event's first block in the work list (blkcum[b]); bad: the
// call's packed offsets are malformed.
struct EventBlock {
  int b, blk, len, tok0, tile0;
  bool bad;
};

// Row addressing of one event. Offsets are in elements of a row of width X.
struct RowAddr {
  long base_row;  // row index of (token 0, head 0)
  long hs, ts;    // row strides of head and token
  long pos_base;
  __device__ __forceinline__ long vec(int h, int i) const { return base_row + h * hs + i * ts; }
  __device__ __forceinline__ long off(int h, int i, int width) const { return vec(h, i) * width; }
  __device__ __forceinline__ float4 pos(const float4* p4, int i) const { return p4[pos_base + i]; }
};

// Token range of event b, clamped into the tensor: padded lengths to [0, L],
// packed offsets to [0, T] and non-decreasing. The packed offsets the
// kernels read are the work list's sanitised copy (running maximum of the
// caller's offsets, clamped to [0, T]), so events never overlap and their
// row blocks never outnumber the per-tile slots sized from T.
__device__ __forceinline__ void event_range(const EventSpec& ev, int b, int& tok0, int& len) {
  if (ev.packed) {
    int a = ev.lens[b], e = ev.lens[b + 1];
    a = a < 0 ? 0 : (a > ev.T ? ev.T : a);
    e = e < a ? a : (e > ev.T ? ev.T : e);
    tok0 = a;
    len = e - a;
  } else {
    const int l = ev.lens[b];
    tok0 = 0;
    len = l < 0 ? 0 : (l > ev.L ? ev.L : l);
  }
}

// Whether the kernels refuse event eb and write NaN into its rows instead of
// computing: the call's packed offsets were malformed (the work list found
// cu_seqlens[0] != 0, a decreasing offset, or cu_seqlens[B] > T, and ran on
// sanitised offsets so that no access leaves the tensors), or the event's
// rows of all heads span 2^31 bytes or more, past the 32-bit byte offsets of
// the buffer loads (which would read zeros there).
__device__ __forceinline__ bool event_refused(const EventSpec& ev, const EventBlock& eb) {
  return eb.bad || (ev.status && *ev.status != 0) || eb.len > ev.max_len;
}

// NaN into rows [r0, r1) of every head of a refused event: out (rows of
// width X, addressed by ra) and vec (per-row scalars addressed by rv, when
// not null).
template <typename T, int X>
__device__ void fill_rows_nan(const RowAddr& ra, const RowAddr& rv, int r0, int r1, int H, int tid, int nthreads,
                              T* out, float* vec) {
  if (r1 <= r0) return;
  const int nr = r1 - r0;
  for (int idx = tid; idx < H * nr * X; idx += nthreads) {
    const int c = idx % X, r = (idx / X) % nr, h = idx / (X * nr);
    out[ra.off(h, r0 + r, X) + c] = (T)__builtin_nanf("");
  }
  if (vec)
    for (int idx = tid; idx < H * nr; idx += nthreads) vec[rv.vec(idx / nr, r0 + idx % nr)] = __builtin_nanf("");
}

// Largest i in [0, n) with key(i) <= t, for key nondecreasing in i and
// key(0) <= t. Each round the wave reads 64 evenly spaced entries of the
// range left (one load per lane) and the count of those at or below t
// (a ballot) narrows it to one gap: one round for n <= 64, two for n <= 4096,
// where a binary search would chain log2 n dependent loads. The result is
// the same in every lane of the wave.
template <typename F>
__device__ __forceinline__ int wave_last_le(int n, int t, F key) {
  const int lane = threadIdx.x & 63;
  int lo = 0, len = n;
  while (len > 1) {
    const int step = (len + 63) >> 6;
    const int i = lo + lane * step;
    const bool le = i < lo + len && key(i) <= t;
    const int c = __builtin_popcountll(__builtin_amdgcn_ballot_w64(le));
    const int nlo = lo + (c - 1) * step;
    len = min(step, lo + len - nlo);
    lo = nlo;
  }
  return __builtin_amdgcn_readfirstlane(lo);
}

// Inclusive scan over the wave's lanes in six DPP steps (row shifts, then the
// row broadcasts); id is op's identity.
template <typename Op>
__device__ __forceinline__ int wave_scan(int x, int id, Op op) {
  x = op(x, __builtin_amdgcn_update_dpp(id, x, 0x111, 0xf, 0xf, false));  // row_shr:1
  x = op(x, __builtin_amdgcn_update_dpp(id, x, 0x112, 0xf, 0xf, false));
  x = op(x, __builtin_amdgcn_update_dpp(id, x, 0x114, 0xf, 0xf, false));
  x = op(x, __builtin_amdgcn_update_dpp(id, x, 0x118, 0xf, 0xf, false));
  x = op(x, __builtin_amdgcn_update_dpp(id, x, 0x142, 0xa, 0xf, false));  // row_bcast:15
  x = op(x, __builtin_amdgcn_update_dpp(id, x, 0x143, 0xc, 0xf, false));  // row_bcast:31
  return x;
}

// The work list of a call of at most kInlineEvents events, formed by each
// wave for itself: lane i holds event i. Sanitised token ranges, block counts
// and the offsets' verdict are those worklist_kernel writes. The wave's own
// list takes two loads, some forty vector instructions and, for the schedules,
// a rank per event (three instructions an event; ranking and summing the
// blocks before each event took ten, and three waves a SIMD run it: forward of
// 64 events of up to 192 tokens, H = 12, D = C = 32, bf16 33.8 us, with the list
// 31.6).
constexpr int kInlineEvents = 64;
struct InlineList {
  int tok0, len, nblk, incl;  // this lane's event; incl: blocks of events 0 .. lane
  bool bad;
  __device__ __forceinline__ InlineList(const EventSpec& ev, int rows) {
    const int lane = threadIdx.x & 63;
    const bool in = lane < ev.B;
    bad = false;
    if (ev.packed) {
      const int lo = in ? ev.lens[lane] : 0, hi = in ? ev.lens[lane + 1] : 0;
      bad = __builtin_amdgcn_ballot_w64(in && ((lane == 0 && lo != 0) || hi < lo || (lane == ev.B - 1 && hi > ev.T))) != 0;
      // Running maximum of the offsets, from 0, clamped to [0, T].
      const int top = wave_scan(lo, 0, [](int a, int c) { return a > c ? a : c; });
      tok0 = min(max(top, 0), ev.T);
      len = in ? min(max(max(top, hi), 0), ev.T) - tok0 : 0;
    } else {
      const int l = in ? ev.lens[lane] : 0;
      tok0 = 0;
      len = l < 0 ? 0 : (l > ev.L ? ev.L : l);
    }
    // Padded events always get one block so that their padding rows are zeroed.
    nblk = !in ? 0 : (len > 0 ? (len + rows - 1) / rows : (ev.packed ? 0 : 1));
    incl = wave_scan(nblk, 0, [](int a, int c) { return a + c; });
  }
  // Position of this lane's event by decreasing length (ties by index): the
  // count of larger keys among the first B, eight to a step (lanes past the
  // events hold the lowest key; their own rank is B).
  __device__ __forceinline__ int rank(int B) const {
    const int lane = threadIdx.x & 63;
    const int key = lane < B ? (min(len, (1 << 25) - 1) << 6) | (63 - lane) : -1;
    int r = 0;
    for (int j = 0; j < B; j += 8)
#pragma unroll
      for (int i = 0; i < 8; ++i) r += __builtin_amdgcn_readlane(key, j + i) > key ? 1 : 0;
    return r;
  }
  // Blocks of the event in position `lane` of the order that rank() gives (0
  // past the events).
  __device__ __forceinline__ int by_rank(int r) const { return __builtin_amdgcn_ds_permute(r << 2, nblk); }
  // Lane b's event as eb.
  __device__ __forceinline__ void event(int b, EventBlock& eb) const {
    eb.b = b;
    eb.tok0 = __builtin_amdgcn_readlane(tok0, b);
    eb.len = __builtin_amdgcn_readlane(len, b);
    eb.tile0 = __builtin_amdgcn_readlane(incl, b) - __builtin_amdgcn_readlane(nblk, b);
    eb.bad = bad;
  }
};
__device__ __forceinline__ int wave_sum_scan(int x) {
  return wave_scan(x, 0, [](int a, int c) { return a + c; });
}
// The lane a ballot names (one bit set).
__device__ __forceinline__ int ballot_lane(bool hit) { return __builtin_ctzll(__builtin_amdgcn_ballot_w64(hit)); }

// Work item of workgroup w: the event whose blocks (of `rows` rows) hold w.
__device__ __forceinline__ bool locate_block(const EventSpec& ev, int rows, int w, EventBlock& eb) {
  if (ev.inl) {
    const InlineList il(ev, rows);
    const bool hit = w < il.incl && w >= il.incl - il.nblk;
    if (__builtin_amdgcn_ballot_w64(hit) == 0) return false;
    il.event(ballot_lane(hit), eb);
    eb.blk = w - eb.tile0;
    return true;
  }
  if (w >= ev.blkcum[ev.B]) return false;
  const int32_t* bc = ev.blkcum;
  const int lo = wave_last_le(ev.B, w, [&](int i) { return bc[i]; });
  eb.b = lo;
  eb.tile0 = ev.blkcum[lo];
  eb.blk = w - eb.tile0;
  eb.bad = false;
  event_range(ev, lo, eb.tok0, eb.len);
  return true;
}

__device__ __forceinline__ RowAddr row_addr(const EventSpec& ev, const EventBlock& eb) {
  RowAddr r;
  if (ev.packed) {
    r.base_row = (long)eb.tok0 * ev.H;
    r.hs = 1;
    r.ts = ev.H;
    r.pos_base = eb.tok0;
  } else if (ev.tokmajor) {
    r.base_row = (long)eb.b * ev.L * ev.H;
    r.hs = 1;
    r.ts = ev.H;
    r.pos_base = (long)eb.b * ev.L;
  } else {
    r.base_row = (long)eb.b * ev.H * ev.L;
    r.hs = ev.L;
    r.ts = 1;
    r.pos_base = (long)eb.b * ev.L;
  }
  return r;
}

// Register load of a four-wave bf16 rows-kernel lane, in the units of
// (HP / 4) D + 3 C: at 160 and more such instances spill, and the rows kernel
// runs eight waves instead (which needs HP % 8 == 0).
__host__ __device__ constexpr int rows_wave_load(int HP, int D, int C) { return (HP / 4) * D + 3 * C; }

// Row addressing of q, k, v, dq, dk and dv. With the operands interleaved
// per token (one [.., 3, H, D] projection output), a token's q heads are
// followed by its k heads and v heads: the token stride is three times that
// of out, grad_out and the per-row vectors, and k, v start H D elements
// after q.
__device__ __forceinline__ RowAddr row_addr_x(const EventSpec& ev, const EventBlock& eb) {
  RowAddr r = row_addr(ev, eb);
  if (ev.xmul > 1) {
    r.base_row *= ev.xmul;
    r.ts *= ev.xmul;
  }
  return r;
}

struct FwdParams {
  EventSpec ev;
  int H, flags;
  float scale;
  const void *q, *k, *v;
  const float* weight;  // [D, C]
  const float* bias;    // [D] or null
  void* out;
  float* lse;
  FreqTable freq;
};

struct BwdParams {
  EventSpec ev;     // rows-kernel work list in ev.blkcum
  const int32_t* blkcum_cols;  // cols-kernel work list
  const int32_t* scum_cols;    // its packed schedule (row blocks in ev.perm order); padded: null
  int H, flags;
  float scale;
  const void *q, *k, *v, *dout;
  const float* weight;  // [D, C]
  const float* bias;    // [D] or null
  const float* lse;     // [rows]
  const void* out;      // the forward's output, laid out as dout (nullable; bf16 rows kernel)
  // scratch written by the rows kernel, read by the cols kernel
  void* u;              // [rows, C] T
  void* wt;             // [rows, C] T
  void* qt;             // [rows, D] T: bf16(q * scale) (written by the bf16 rows kernel)
  float* dob;           // [rows]
  float* dsum;          // [rows]
  // [rows] the rows kernel's sum of P per row, Z, for the cols kernel's P / Z:
  // bf16, the log2-domain LSE of the normalised P, lse log2(e) + log2 Z;
  // float32, log2 Z alone (at logits of O(1e4) the sum would round away the
  // correction, so the float32 cols kernel subtracts it after the exponent's
  // fma).
  float* lse_z;
  float* dw_part;       // [blocks, D, C]
  float* db_part;       // [blocks, D]
  // outputs
  void *dq, *dk, *dv;
  float* rowsum;        // nullable
  float* dweight;
  float* dbias;         // nullable
  FreqTable freq;
  // dW / db summed by the first red_blocks workgroups of the cols launch
  // (reduce_block) over red_seg runs of the rows kernel's red_rows-row blocks;
  // 0: by a launch of their own.
  int red_blocks, red_seg, red_rows, red_lg;
};

// dW / db from the per-block partials of the rows kernel, in two fixed-order
// stages so the result does not depend on scheduling: stage 1 sums runs of
// kRedSeg consecutive blocks per column (coalesced over the columns), stage
// 2 sums the run totals in four interleaved sums added in order.
constexpr int kRedSeg = 64;

// Blocks of the call's work list (of `rows` rows).
__device__ __forceinline__ int total_blocks(const EventSpec& ev, int rows) {
  if (!ev.inl) return ev.blkcum[ev.B];
  return __builtin_amdgcn_readlane(InlineList(ev, rows).incl, 63);
}

// Blocks [64 s, 64 s + 64) of column col, in order.
__device__ __forceinline__ float run_sum(const float* part, int nblk, int ncol, int s, int col) {
  const long w0 = (long)s * kRedSeg;
  const long w1 = w0 + kRedSeg < nblk ? w0 + kRedSeg : nblk;
  float acc = 0.f;
#pragma unroll 8
  for (long w = w0; w < w1; ++w) acc += part[w * ncol + col];
  return acc;
}

__device__ __forceinline__ void store_dw(float acc, int e, int DC, float* dw, float* db) {
  if (e < DC)
    dw[e] = acc;
  else if (db)
    db[e - DC] = acc;
}

// Both stages by the first workgroups of the cols kernel's launch, for at most
// kRedFold runs (1024 blocks): a thread per run and column, 2^red_lg columns a
// workgroup (64 for up to 4 runs, 32 for up to 8, else 16: every run is summed
// at once and a workgroup is 256 threads), the run totals exchanged through
// LDS and added in the two-launch order (bit for bit the same sums). It runs
// beside the cols tiles, and the launch it saves is 6 us of kernel and the gap
// before it on calls whose kernels take 15 to 60 us. Whole backward, bf16,
// D = 32, C = 16, 4 / 12 heads: 16 events of 64 tokens 23.7 -> 18.7 / 29.3 ->
// 24.5 us, 48 of 192 57.4 -> 52.2 / 90.1 -> 84.6, 256 of 64 48.2 -> 46.1 /
// 77.4 -> 73.1 (64 columns a workgroup at 16 runs, four runs one after the
// other: 55.2 / 75.9). With more runs the two launches spread them over more
// workgroups. part: 1 KB of LDS.
constexpr int kRedFold = 16;
template <int DC, int D>
__device__ void reduce_block(const BwdParams& prm, int tid, float* part) {
  const int lg = prm.red_lg, nc = 1 << lg, c = tid & (nc - 1), s = tid >> lg;
  const int e = (blockIdx.x << lg) + c;
  const bool ok = e < DC + D;
  const int nblk = total_blocks(prm.ev, prm.red_rows);  // by whole waves
  if (tid < 256)
    part[tid] = ok && s < prm.red_seg && (prm.flags & (FST_ATTN_BIAS | FST_ACT_BIAS))
                    ? run_sum(prm.dw_part, nblk, DC + D, s, e)
                    : 0.f;
  __syncthreads();
  if (s != 0 || !ok) return;
  float q4[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    q4[q] = 0.f;
    for (int k = q; k < prm.red_seg; k += 4) q4[q] += part[(k << lg) + c];
  }
  store_dw(((q4[0] + q4[1]) + q4[2]) + q4[3], e, DC, prm.dweight, prm.dbias);
}

template <typename T>
struct VecOf;
template <>
struct VecOf<bf16> {
  typedef bf16x8 type;
  static __device__ __forceinline__ bf16x8 zero() {
    bf16x8 z;
#pragma unroll
    for (int e = 0; e < 8; ++e) z[e] = (bf16)0.f;
    return z;
  }
};
template <>
struct VecOf<float> {
  typedef f32x4 type;
  static __device__ __forceinline__ f32x4 zero() { return zero4(); }
};

__device__ __forceinline__ float exp2f_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// Completion of this wave's outstanding buffer loads (including loads into
// LDS), ordered against every later memory access of the wave.
__device__ __forceinline__ void wait_vmem() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Four consecutive output elements from an fp32 quad.
template <typename T>
__device__ __forceinline__ void store4(T* p, const f32x4& v);
template <>
__device__ __forceinline__ void store4<bf16>(bf16* p, const f32x4& v) {
  bf16x4 o;
#pragma unroll
  for (int r = 0; r < 4; ++r) o[r] = (bf16)v[r];
  *reinterpret_cast<bf16x4*>(p) = o;
}
template <>
__device__ __forceinline__ void store4<float>(float* p, const f32x4& v) {
  *reinterpret_cast<f32x4*>(p) = v;
}

// ---------------------------------------------------------------------------
// Channel operand of the u.E / w~.E contractions (K = C). Slot r of lane
// group g in channel tile ct is channel 16ct + 4g + r -- the C layout of a
// 16x16 fp32 MFMA tile -- so U computed on the MFMA feeds the next one
// directly. bf16 contracts each tile with one 16x16x16 step; fp32 with four
// 16x16x4 steps (step r covers channels 16ct + r + {0, 4, 8, 12}).
// ---------------------------------------------------------------------------
template <typename T, int C>
struct CFrag;

template <int C>
struct CFrag<bf16, C> {
  bf16x4 v[C / 16];
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int ct = 0; ct < C / 16; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[ct][r] = (bf16)0.f;
  }
  __device__ __forceinline__ void load(const bf16* p, int g) {
#pragma unroll
    for (int ct = 0; ct < C / 16; ++ct) v[ct] = *reinterpret_cast<const bf16x4*>(p + 16 * ct + 4 * g);
  }
  __device__ __forceinline__ void from_acc(const f32x4* acc) {
#pragma unroll
    for (int ct = 0; ct < C / 16; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[ct][r] = (bf16)acc[ct][r];
  }
};

template <int C>
struct CFrag<float, C> {
  f32x4 v[C / 16];
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int ct = 0; ct < C / 16; ++ct) v[ct] = zero4();
  }
  __device__ __forceinline__ void load(const float* p, int g) {
#pragma unroll
    for (int ct = 0; ct < C / 16; ++ct) v[ct] = *reinterpret_cast<const f32x4*>(p + 16 * ct + 4 * g);
  }
  __device__ __forceinline__ void from_acc(const f32x4* acc) {
#pragma unroll
    for (int ct = 0; ct < C / 16; ++ct) v[ct] = acc[ct];
  }
};

// The float32 embedding of one pair formed straight in the channel layout of
// CFrag (lane group g: channels 16 ct + 4 g + r), with write_embedding's
// arithmetic: channel c < C / 2 is the sine of frequency c, channel C / 2 + c
// its cosine. With C a multiple of 32 a lane's channels are the sines and
// cosines of the same C / 8 frequencies.
template <int C>
__device__ __forceinline__ CFrag<float, C> embed_cfrag(float4 pi, float4 pj, const FreqTable& ft, int g) {
  static_assert(C % 32 == 0, "each lane holds the sine and cosine of its frequencies");
  constexpr int FT = C / 32;  // sine channel tiles
  const double x = pair_angle_f64(pi, pj);
  CFrag<float, C> e;
#pragma unroll
  for (int ct = 0; ct < FT; ++ct)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int f = 16 * ct + 4 * g + r;
      const double rev = x * ((double)ft.ghi[f] + (double)ft.glo[f]);
      const float rr = (float)(rev - __builtin_floor(rev));
      e.v[ct][r] = __builtin_amdgcn_sinf(rr);
      e.v[FT + ct][r] = __builtin_amdgcn_cosf(rr);
    }
  return e;
}

template <int C>
__device__ __forceinline__ f32x4 mma_c(const CFrag<bf16, C>& a, const CFrag<bf16, C>& b, f32x4 c) {
#pragma unroll
  for (int ct = 0; ct < C / 16; ++ct) c = mfma_x16(a.v[ct], b.v[ct], c);
  return c;
}
template <int C>
__device__ __forceinline__ f32x4 mma_c(const CFrag<float, C>& a, const CFrag<float, C>& b, f32x4 c) {
#pragma unroll
  for (int ct = 0; ct < C / 16; ++ct)
#pragma unroll
    for (int r = 0; r < 4; ++r) c = mfma_f32(a.v[ct][r], b.v[ct][r], c);
  return c;
}

// Projection of one row's heads onto the channels, in fp32 MFMA:
//   acc[ct] = (x_row[h] * mult) @ W[:, 16ct..16ct+15]  as U^T[c, h]
// lane (g, n = h) ends with channels 16ct + 4g + r. Step s contracts
// d = (D/4) g + s (lane group g holds a contiguous quarter of the row).
// x_row points at head 0 of the row; hstride = element stride between heads.
template <typename T, int D, int C>
__device__ __forceinline__ void project_row(const T* x_row, long hstride, bool valid, float mult,
                                            const float* __restrict__ W, int g, int n, f32x4* acc) {
  constexpr int Q = D / 4;
  float xv[Q];
  if (valid) {
    const T* p = x_row + n * hstride + Q * g;
#pragma unroll
    for (int s = 0; s < Q; ++s) xv[s] = (float)p[s] * mult;
  } else {
#pragma unroll
    for (int s = 0; s < Q; ++s) xv[s] = 0.f;
  }
#pragma unroll
  for (int ct = 0; ct < C / 16; ++ct) {
    f32x4 a = zero4();
#pragma unroll
    for (int s = 0; s < Q; ++s) a = mfma_f32(W[(Q * g + s) * C + 16 * ct + n], xv[s], a);
    acc[ct] = a;
  }
}

// Pair embedding of one (row i, key j) into an LDS row: channel f is
// sin(x_ij f_f), channel C/2 + f is cos(x_ij f_f) (reference.py:75-84 order).
// bf16 kernels evaluate the angle in fp32 (the result is rounded to bf16);
// fp32 kernels evaluate angle and argument reduction in binary64. With
// SPLIT > 1, SPLIT lanes share the pair: this one writes the frequencies
// [part F / SPLIT, (part + 1) F / SPLIT) and their cosines.
template <typename T, int C, int SPLIT = 1>
__device__ __forceinline__ void write_embedding(T* erow, float4 pi, float4 pj, const FreqTable& ft, int part = 0) {
  constexpr int F = C / 2, FP = F / SPLIT;
  static_assert(FP % 4 == 0, "each lane writes whole groups of four frequencies");
  const int f0 = SPLIT == 1 ? 0 : part * FP;
  float sv[FP], cv[FP];
  if constexpr (is_bf16<T>::value) {
    const float x = pair_angle(pi, pj);
#pragma unroll
    for (int f = 0; f < FP; ++f)
      sincos_rev<false>(x, ft.ghi[f0 + f], ft.glo[f0 + f], (ft.reduce_mask >> (f0 + f)) & 1u, sv[f], cv[f]);
  } else {
    const double x = pair_angle_f64(pi, pj);
#pragma unroll
    for (int f = 0; f < FP; ++f) {
      const double rev = x * ((double)ft.ghi[f0 + f] + (double)ft.glo[f0 + f]);
      const float r = (float)(rev - __builtin_floor(rev));
      sv[f] = __builtin_amdgcn_sinf(r);
      cv[f] = __builtin_amdgcn_cosf(r);
    }
  }
  if constexpr (is_bf16<T>::value) {
#pragma unroll
    for (int f = 0; f < FP; f += 4) {
      bf16x4 a, b;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        a[e] = (bf16)sv[f + e];
        b[e] = (bf16)cv[f + e];
      }
      *reinterpret_cast<bf16x4*>(erow + f0 + f) = a;
      *reinterpret_cast<bf16x4*>(erow + F + f0 + f) = b;
    }
  } else {
#pragma unroll
    for (int f = 0; f < FP; f += 4) {
      *reinterpret_cast<f32x4*>(erow + f0 + f) = f32x4{sv[f], sv[f + 1], sv[f + 2], sv[f + 3]};
      *reinterpret_cast<f32x4*>(erow + F + f0 + f) = f32x4{cv[f], cv[f + 1], cv[f + 2], cv[f + 3]};
    }
  }
}

// Lane assignment of a wave's embeddings: NP (row, key) pairs of a chunk
// per wave. NP >= 64: EPL pairs per lane, lane l taking key l % KC of rows
// l / KC + (64 / KC) k; NP < 64 (a divisor of 64): SPLIT = 64 / NP lanes
// per pair, each writing 1 / SPLIT of the frequencies.
template <int NP>
struct EmbedLanes {
  static constexpr bool OK = NP % 64 == 0 || 64 % NP == 0;
  static constexpr int EPL = NP >= 64 ? NP / 64 : 1;
  static constexpr int SPLIT = NP >= 64 ? 1 : 64 / NP;
  // pair slot and frequency part of a lane
  static __device__ __forceinline__ int slot(int lane) { return SPLIT == 1 ? lane : lane % NP; }
  static __device__ __forceinline__ int part(int lane) { return SPLIT == 1 ? 0 : lane / NP; }
};

// Zero the outputs of padding rows [max(row0, len), end) of a padded event,
// where end is the block's last row, or L for the event's last block
// (pad-row contract: forward.py:19-22, 288-304). Rows of out are addressed
// by ra, those of vec_out by rv.
template <typename T>
__device__ __forceinline__ void zero_pad_rows(const EventSpec& ev, const EventBlock& eb, const RowAddr& ra,
                                              const RowAddr& rv, int row0, int rows, int width, int tid,
                                              int nthreads, T* out, float* vec_out, int vec_count) {
  if (ev.packed) return;
  const int nblk = eb.len > 0 ? (eb.len + rows - 1) / rows : 1;
  const int first = row0 > eb.len ? row0 : eb.len;
  const int end = (eb.blk == nblk - 1) ? ev.L : (row0 + rows < ev.L ? row0 + rows : ev.L);
  if (first >= end) return;
  const int nrows = end - first;
  const int total = ev.H * nrows * width;
  for (int idx = tid; idx < total; idx += nthreads) {
    const int c = idx % width;
    const int r = (idx / width) % nrows;
    const int h = idx / (width * nrows);
    out[ra.off(h, first + r, width) + c] = (T)0.f;
  }
  if (vec_out)
    for (int idx = tid; idx < ev.H * nrows * vec_count; idx += nthreads) {
      const int r = (idx / vec_count) % nrows;
      const int h = idx / (vec_count * nrows);
      vec_out[rv.vec(h, first + r) * vec_count + idx % vec_count] = 0.f;
    }
}

// Forward dispatch per (dtype, D), one translation unit each
// (fst_fwd_inst.hip). With query set, only reports the rows per workgroup
// of the kernel that (HP, C) selects (0 = unsupported) in *rows.
// fwd_plans_* reports the FST_PLAN_FWD_* bits compiled for (HP, C).
#define FST_DECL_FWD(NAME)                                                                                       \
  int fwd_dispatch_##NAME(const FwdParams& prm, int HP, int C, hipStream_t stream, int grid, bool query, int* rows); \
  int fwd_plans_##NAME(int HP, int C);
FST_DECL_FWD(bf16_16)
FST_DECL_FWD(bf16_32)
FST_DECL_FWD(bf16_48)
FST_DECL_FWD(bf16_64)
FST_DECL_FWD(f32_16)
FST_DECL_FWD(f32_32)
FST_DECL_FWD(f32_48)
FST_DECL_FWD(f32_64)
#undef FST_DECL_FWD

// Backward dispatch per (dtype, D) (fst_bwd_inst.hip). which = 0: rows
// kernel, 1: cols kernel. With query set, reports rows (or keys) per
// workgroup in *rows (0 = unsupported). bwd_plans_* reports the
// FST_PLAN_ROWS_* / FST_PLAN_COLS_* bits compiled for (HP, C).
#define FST_DECL_BWD(NAME)                                                                                   \
  int bwd_dispatch_##NAME(const BwdParams& prm, int which, int HP, int C, hipStream_t stream, int grid, bool query, \
                          int* rows);                                                                        \
  int bwd_plans_##NAME(int HP, int C);
FST_DECL_BWD(bf16_16)
FST_DECL_BWD(bf16_32)
FST_DECL_BWD(bf16_48)
FST_DECL_BWD(bf16_64)
FST_DECL_BWD(f32_16)
FST_DECL_BWD(f32_32)
FST_DECL_BWD(f32_48)
FST_DECL_BWD(f32_64)
#undef FST_DECL_BWD

// ---------------------------------------------------------------------------
// Plan requests of the first-generation kernels (fst_forward.hip,
// fst_backward.hip), which come in (NW, NS) splits: NW waves per 16-row tile
// (16 * 4 / NW rows or keys per four-wave workgroup; NW = 8 is one 16-row
// tile in an eight-wave workgroup) and 16 * NS keys (or rows) per chunk.
// ---------------------------------------------------------------------------
// (NW, NS) of a plan request for a family of configurations F<NW, NS>
// (nw, ns = 0: not requested), as 10 NW + NS, or 0 when nothing fits.
// Preference: the most waves per 16-row tile first (on gfx950 the 16-row
// workgroups run about twice as fast as 64-row ones, e.g. 2.8 against 5.3
// ms for the float32 forward at B=256, L=768, H=12, D=32, C=16: more waves
// share the tile's work and each holds less), then ns_first keys (or rows)
// per chunk.
template <template <int, int> class F>
constexpr int pick_split(int nw, int ns, int ns_first = 2) {
  const bool fits[4][2] = {{F<8, 1>::FITS, F<8, 2>::FITS}, {F<4, 1>::FITS, F<4, 2>::FITS},
                           {F<2, 1>::FITS, F<2, 2>::FITS}, {F<1, 1>::FITS, F<1, 2>::FITS}};
  const int nws[4] = {8, 4, 2, 1};
  for (int w = 0; w < 4; ++w) {
    if (nw && nws[w] != nw) continue;
    // The eight-wave plan bits stand for even splits; the uneven one is a
    // static choice only.
    if (nw == 8 && !F<8, 1>::HS::EVEN) continue;
    for (int k = 0; k < 2; ++k) {
      const int s = k == 0 ? ns_first : 3 - ns_first;
      if (ns && s != ns) continue;
      if (fits[w][s - 1]) return 10 * nws[w] + s;
    }
  }
  return 0;
}

// The requested (nw, ns) of the plan bits in flags, for the groups starting
// at bit t (three tile-height bits) and bit k (two key-chunk bits).
// t: bit index of the T16 / T32 / T64 triple; w8: bit index of the
// eight-wave 16-row tile.
__host__ __device__ inline int plan_nw(int flags, int t, int w8) {
  return (flags >> w8) & 1 ? 8
                           : ((flags >> t) & 1 ? 4 : ((flags >> (t + 1)) & 1 ? 2 : ((flags >> (t + 2)) & 1 ? 1 : 0)));
}
__host__ __device__ inline int plan_ns(int flags, int k) { return (flags >> k) & 1 ? 1 : ((flags >> (k + 1)) & 1 ? 2 : 0); }
constexpr int bit_index(int b) { return b <= 1 ? 0 : 1 + bit_index(b >> 1); }

// Heads of a 16-row tile's NW waves: ceil(HP / NW) a wave, one fewer from wave
// NBIG on where NW does not divide HP (eight waves of 12 heads: 2 and 1; waves
// w and w + 4 share a SIMD, so every SIMD serves three). Twelve heads over four
// waves kept the float32 kernels at one wave per SIMD (311 to 411 registers a
// lane at D = 32, C = 16); over eight they run two: H = 12, D = 32, C = 16, B = 32,
// L = 768, lengths U{16..768}: forward 0.457 -> 0.414 ms, rows 0.795 -> 0.638,
// cols 1.004 -> 0.683; every width forward -13 to -30 %, rows -9 to -32 %, cols
// -24 to -34 % (but those two that keep four waves, bwd_launch_t).
template <int HP, int NW>
struct HeadSplit {
  static constexpr int HW = (HP + NW - 1) / NW, NBIG = HP - NW * (HW - 1);
  static constexpr bool EVEN = HP % NW == 0, OK = EVEN || (NW == 8 && HP == 12);
  // Head hl of wave ws, or one past every head.
  static __device__ __forceinline__ int head(int ws, int hl) {
    if constexpr (EVEN) return ws * HW + hl;
    if (ws < NBIG) return ws * HW + hl;
    return hl < HW - 1 ? NBIG * HW + (ws - NBIG) * (HW - 1) + hl : HP;
  }
};

// The plan bits of a (NW, NS) family: a tile-height bit for each NW and a
// key-chunk bit for each NS that fits with some value of the other.
template <template <int, int> class F>
constexpr int split_plans(int t16, int k16, int w8) {
  int bits = 0;
  const int nws[3] = {4, 2, 1};
  for (int w = 0; w < 3; ++w)
    if (pick_split<F>(nws[w], 0)) bits |= t16 << w;
  if (pick_split<F>(8, 0)) bits |= w8;
  for (int s = 1; s <= 2; ++s)
    if (pick_split<F>(0, s)) bits |= k16 << (s - 1);
  return bits;
}

}  // namespace fst
