// Chunked gated delta rule forward for gfx950 (fp32 arithmetic, MFMA).
//
// Computes what transformers' torch_chunk_gated_delta_rule computes for the
// decider's linear-attention layers (called at ref: src/decider/packed_conv.py:55-59
// with use_qk_l2norm_in_kernel=True; transformers modeling_qwen3_5.py:249-328),
// per value head h (key head h / (Hv/Hk), the repeat_interleave mapping):
//
//   q, k <- l2norm(q), l2norm(k) on the bf16 rows, each step rounded to bf16
//   q <- q * scale;  per 64-token chunk: gc = cumsum(g),  D_ij = e^{gc_i - gc_j} (j <= i)
//   L = strictly-lower(beta_i k_i.k_j D_ij),  T = (I + L)^-1
//   u = T (beta v),  w = T (beta e^{gc} k),   A = (q k^T) o D (j <= i)
//   across chunks, state S [dk, dv] (zero or the initial state):
//     v' = u - w S;  o = (q e^{gc}) S + A v';  S <- e^{gc_last} S + (k e^{gc_last - gc})^T v'
//
// Packed requests (cu_seqlens) are chunked per request and each request starts
// from its own state, so no state crosses a request boundary.
//
// Up to four launches, all on the caller's stream, intermediates in a
// caller-provided workspace (fd_gated_delta_workspace_bytes):
//   1. gd_chunk_table — packed requests only, one workgroup: chunk -> (first
//      row, length), request -> first chunk, the requests longest first.  A
//      padded batch needs no table.
//   2. gd_prep_kernel — one workgroup per (chunk, value head), chunk-parallel:
//      l2norm, cumsum, the Gram and q.k tiles on bf16 MFMA (the normalised q/k
//      are bf16 values, so these products are exact before fp32 accumulation),
//      then u and w as the solutions of (I + L) x = rhs by forward substitution,
//      one right-hand-side column per thread (256 columns: 128 of u, 128 of w),
//      in four 16-row blocks; each finished block is stored while the next runs.
//   3. gd_state_kernel — one workgroup per (request, value head, 16 value
//      columns): the only sequential part.  Each state column evolves on its
//      own, so the 128 value columns split over 8 workgroups.  Four wavefronts
//      run the chain: the state slice lives in their registers, and the
//      operands of the chunks two ahead are loaded straight into registers
//      (three register sets) while the current chunk runs; two barriers per
//      chunk.  Four more wavefronts, one per SIMD beside the chain's, compute
//      each chunk's output o = scale e^{gc} (q S_chunk) + A v' for the
//      slice's columns from the state and v' planes the chain leaves in LDS,
//      so neither the chunk-start states nor v' go through HBM.
//      All products run on bf16 MFMA over exact bf16 splits of the fp32 operands.
//   4. fd_gated_rmsnorm_fwd's kernel — with the layer's gated RMSNorm
//      (fd_gated_delta_norm_fwd) only: the output rows, written to the
//      workspace, normalised into the caller's output.
// The intermediates sit in the workspace in the order their consumer's MFMA
// operands are loaded (one wavefront load = 1-2 KiB contiguous).  The MFMA
// lane layout (v_mfma_f32_16x16x32_bf16): lane l supplies A[l%16][8(l/16)+j]
// and B[8(l/16)+j][l%16] for j = 0..7 of each 32-step; D[4(l/16)+r][l%16].
#include <mutex>
#include <type_traits>

#include "fd_common.h"

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

namespace {

constexpr int kC = 64;                 // tokens per chunk
constexpr int kD = 128;                // head_k_dim == head_v_dim
constexpr int kSlice = 16;             // value columns per state workgroup
constexpr int kSlices = kD / kSlice;   // state workgroups per (request, head)
constexpr int kThreads = 256;
// A's three planes in a chunk of GdArgs::aq (see aq_offset)
constexpr int kAqPlane = 5 * 64 * 8 + 64;  // elements per plane (a multiple of 128 bytes)
constexpr int kAqChunk = kC * kC * 2;      // elements per chunk
// The order of packed requests lies behind the planes, an entry per chunk, so that it
// takes no room of its own and the no-allocation scratch, a fixed size, takes every
// call it took without it.  There are at least as many chunks as requests.
constexpr int kOrderStep = kAqChunk / 2;   // int32 entries
static_assert(3 * kAqPlane + 2 <= kAqChunk, "A's planes and an entry of the order fit in the space of the fp32 matrix");

struct GdArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const float* g;
  const void* beta;
  uint16_t* o;
  const float* s0;   // [N, Hv, Dk, Dv] or null
  float* sN;         // [N, Hv, Dk, Dv] or null
  int32_t* row0;     // [nc]  first packed row of each chunk
  int32_t* len;      // [nc]  valid rows of each chunk (0 = unused)
  int32_t* first;    // [N+1] first chunk of each request
  // requests, longest first: entry i at i * kOrderStep, behind A's planes in chunk i of aq.  (Formed
  // from aq instead of held here, every call took 0.2 us longer: the arguments behind it then straddle
  // one more line of the scalar loads at a workgroup's start.)
  int32_t* order;
  float* gc;         // [Hv, nc, 3, 64]: e^{gc_t}, e^{gl - gc_t}, then e^{gl} 64 times (gl = gc of the last row)
  // q and A are stored in the state pass's output-wavefront operand order
  // (lane = 16 * g4 + c16): every load there reads 1-2 KiB contiguous
  uint16_t* qn;      // [Hv, nc, rt 4, st 4, lane 64, 8] bf16: q[16rt + c16][32st + 8g4 + e]
  // w, k^T and u are stored in the state pass's operand order: every load of a
  // wavefront there reads 1 KiB contiguous (lane = 16 * g4 + c16, see gd_state_kernel)
  uint16_t* kn;      // [Hv, nc, wv 4, m 2, st 2, lane 64, 8] bf16: k^T[32wv + 16m + c16][32st + 8g4 + e]
  uint16_t* w;       // [Hv, nc, plane 3, wv 4, st 4, lane 64, 8] bf16: w_x[16wv + c16][32st + 8g4 + e],
                     // w split exactly into hi + mid + lo planes
  float* u;          // [Hv, nc, js 8, wv 4, lane 64, r 4]: u[16wv + 4g4 + r][16js + c16]
  uint16_t* aq;      // [Hv, nc, kAqChunk] bf16: planes hi, mid, lo (an exact split) of A[16rt + c16][32st + 8g4 + e],
                     // e = 0..7 at aq_offset(rt, st, lane) of each plane
  int hk, hv, nc, nseq;
  int varlen, seq_len, nct;  // packed requests (table) or a padded batch of nct chunks per sequence
  int beta_f32, l2norm;
  float scale;
};

// round to bf16 and back (v_cvt_pk_bf16_f32, round to nearest even)
__device__ __forceinline__ float bf16r(float x) { return fd_lo(fd_pack2(x, 0.0f)); }

__device__ __forceinline__ f32x4_t mfma_f32(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x4_t mfma_bf16(uint4 a, uint4 b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                 c, 0, 0, 0);
}

// x == hi + mid + lo exactly (each a bf16; the two differences are exact in fp32),
// so a product with a bf16 value is three exact bf16 products accumulated in fp32.
// The conversions are v_cvt_pk_bf16_f32 (round to nearest even).
// four fp32 values -> three planes of four bf16 each (8 bytes per plane)
__device__ __forceinline__ void split3x4(const float* x, uint2& hi, uint2& mid, uint2& lo) {
  const uint32_t h01 = fd_pack2(x[0], x[1]), h23 = fd_pack2(x[2], x[3]);
  const float r[4] = {x[0] - fd_lo(h01), x[1] - fd_hi(h01), x[2] - fd_lo(h23), x[3] - fd_hi(h23)};
  const uint32_t m01 = fd_pack2(r[0], r[1]), m23 = fd_pack2(r[2], r[3]);
  const uint32_t l01 = fd_pack2(r[0] - fd_lo(m01), r[1] - fd_hi(m01));
  const uint32_t l23 = fd_pack2(r[2] - fd_lo(m23), r[3] - fd_hi(m23));
  hi = make_uint2(h01, h23);
  mid = make_uint2(m01, m23);
  lo = make_uint2(l01, l23);
}

// eight fp32 values -> three planes of eight bf16 (16 bytes per plane)
__device__ __forceinline__ void split3x8(f32x4_t v0, f32x4_t v1, uint4& hi, uint4& mid, uint4& lo) {
  const float va[4] = {v0[0], v0[1], v0[2], v0[3]};
  const float vb[4] = {v1[0], v1[1], v1[2], v1[3]};
  uint2 ha, ma, la, hb, mb, lb;
  split3x4(va, ha, ma, la);
  split3x4(vb, hb, mb, lb);
  hi = make_uint4(ha.x, ha.y, hb.x, hb.y);
  mid = make_uint4(ma.x, ma.y, mb.x, mb.y);
  lo = make_uint4(la.x, la.y, lb.x, lb.y);
}

__device__ __forceinline__ void unpack8(uint4 raw, float* x) {
  const uint32_t wd[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[2 * i] = fd_lo(wd[i]);
    x[2 * i + 1] = fd_hi(wd[i]);
  }
}

__device__ __forceinline__ uint4 pack8(const float* x) {
  uint4 r;
  r.x = fd_pack2(x[0], x[1]);
  r.y = fd_pack2(x[2], x[3]);
  r.z = fd_pack2(x[4], x[5]);
  r.w = fd_pack2(x[6], x[7]);
  return r;
}

// transformers' l2norm on a bf16 row of 128 held by 16 consecutive lanes (8
// values each): x*x rounded to bf16, summed in fp32 (lane chunk order, then an
// xor butterfly over the 16 lanes), the sum, sum + eps and 1/sqrt each rounded
// to bf16, then x * inv rounded to bf16.  Every lane of the wavefront must call it.
__device__ __forceinline__ uint4 l2norm_row8(uint4 raw) {
  float x[8];
  unpack8(raw, x);
  float s = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) s = s + bf16r(x[e] * x[e]);
  s = fd_xor_sum_down<16>(s);
  const float e = bf16r(bf16r(s) + 1e-6f);
  const float inv = bf16r(1.0f / __builtin_sqrtf(e));
  float y[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) y[i] = x[i] * inv;
  return pack8(y);
}

// ---------------------------------------------------------------------------
// 1. chunk table (packed requests, one workgroup): the first chunk of every
// request by a scan of their chunk counts, then every chunk's request by a
// binary search, one chunk per thread (a thread per request that walked the
// request's chunks took 12.8 us for requests of up to 8002 tokens; this takes 4.6).
// `order` lists the requests longest first, so that the state pass starts the
// longest chains first (by counting, up to kTableThreads requests; more keep
// their own order: their chains are many and short).
constexpr int kTableThreads = 1024;

__device__ __forceinline__ int request_rows(const int32_t* cu, int s, int total, int* start) {
  *start = min(max(cu[s], 0), total);
  return min(max(cu[s + 1], *start), total) - *start;
}

__global__ __launch_bounds__(kTableThreads) void gd_chunk_table(const int32_t* __restrict__ cu, int total, GdArgs a) {
  __shared__ int wave_total[kTableThreads / 64];
  __shared__ int first[kTableThreads], chunks[kTableThreads];
  const int t = threadIdx.x;
  const int nseq = a.nseq;
  int carry = 0;
  for (int base = 0; base < nseq; base += kTableThreads) {
    const int s = base + t;
    int start = 0;
    const int n = s < nseq ? (request_rows(cu, s, total, &start) + kC - 1) / kC : 0;
    int incl = n;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int up = __shfl_up(incl, off);
      if ((t & 63) >= off) incl += up;
    }
    if ((t & 63) == 63) wave_total[t >> 6] = incl;
    __syncthreads();
    int before = carry, block_total = 0;
#pragma unroll
    for (int w = 0; w < kTableThreads / 64; ++w) {
      if (w < (t >> 6)) before += wave_total[w];
      block_total += wave_total[w];
    }
    const int f = before + incl - n;
    if (s < nseq) a.first[s] = f;
    first[t] = s < nseq ? f : a.nc;
    chunks[t] = n;
    carry += block_total;
    __syncthreads();
    // the chunks of these requests: the last request of the block whose first chunk is <= c
    // (an empty request shares its first chunk with the next one)
    const int here = min(kTableThreads, nseq - base);
    const int c_end = min(carry, a.nc);
    for (int c = carry - block_total + t; c < c_end; c += kTableThreads) {
      int lo = 0, hi = here;
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (first[mid] <= c) lo = mid; else hi = mid;
      }
      int r0;
      const int rows = request_rows(cu, base + lo, total, &r0);
      const int j = c - first[lo];
      a.row0[c] = r0 + j * kC;
      a.len[c] = min(kC, rows - j * kC);
    }
    if (nseq <= kTableThreads) {
      if (s < nseq) {
        int rank = 0;
        for (int o = 0; o < nseq; ++o) rank += chunks[o] > n || (chunks[o] == n && o < s);
        a.order[static_cast<size_t>(rank) * kOrderStep] = s;
      }
    } else if (s < nseq) {
      a.order[static_cast<size_t>(s) * kOrderStep] = s;
    }
    __syncthreads();
  }
  if (t == 0) a.first[nseq] = carry;
  for (int c = carry + t; c < a.nc; c += kTableThreads) {
    a.row0[c] = 0;
    a.len[c] = 0;
  }
}

// ---------------------------------------------------------------------------
// chunk and request ranges: from the table for packed requests, by arithmetic
// for a padded batch (no table launch)
__device__ __forceinline__ void chunk_rows(const GdArgs& a, int c, int* r0, int* len) {
  if (a.varlen) {
    *r0 = a.row0[c];
    *len = a.len[c];
  } else {
    const int s = c / a.nct;
    const int j = c - s * a.nct;
    *r0 = s * a.seq_len + j * kC;
    *len = min(kC, a.seq_len - j * kC);
  }
}

__device__ __forceinline__ void request_chunks(const GdArgs& a, int s, int* first, int* last) {
  if (a.varlen) {
    *first = a.first[s];
    *last = min(a.first[s + 1], a.nc);
  } else {
    *first = s * a.nct;
    *last = (s + 1) * a.nct;
  }
}

// ---------------------------------------------------------------------------
// 2. per-chunk preparation
constexpr int kRowK = kD + 8;    // bf16 row stride of the row-major q/k/v tiles (272 B)
constexpr int kRowF = kC + 4;    // fp32 row stride of the 64x64 tiles (272 B)
constexpr int kPrepK = 0;                                   // bf16 [64][kRowK]
constexpr int kPrepQ = kPrepK + kC * kRowK * 2;             // bf16 [64][kRowK]; then A, fp32 [64][kRowF]
constexpr int kPrepV = kPrepQ + kC * kRowK * 2;             // bf16 [64][kRowK]
constexpr int kPrepL = kPrepV + kC * kRowK * 2;             // fp32 [64][kRowF]
constexpr int kPrepG = kPrepL + kC * kRowF * 4;             // fp32 [64]  gc
constexpr int kPrepB = kPrepG + kC * 4;                     // fp32 [64]  beta
constexpr int kPrepBG = kPrepB + kC * 4;                    // fp32 [64]  beta e^gc
constexpr int kPrepBytes = kPrepBG + kC * 4;
static_assert(kC * kRowF * 4 <= kC * kRowK * 2, "A takes the place of the q tile");

// A's planes in the state pass's output-wavefront operand order: five slots of 64
// lanes x 8 elements and one lane's zeros.  A is lower triangular: rows 0..31 have no
// tile st = 1, and the upper lanes (8g4 >= 16) of tiles (0,0) and (2,1) are zero, so
// the two share slot 0 and their upper lanes read the zeros.  (1,0) (2,0) (3,0) and
// (3,1) take the slots 1..4.
__device__ __forceinline__ int aq_offset(int rt, int st, int lane) {
  if (rt == 2 * st) return (lane < 32 ? st * 32 + lane : 5 * 64) * 8;
  return ((st == 0 ? rt : 4) * 64 + lane) * 8;
}

// Inside a 16-row block the solve reads row m of the transposed L tile in 4-wide
// pieces starting at (m + 1) & ~3, for m = 0..14: 36 reads, piece k at (tri_m(k), tri_i0(k)).
constexpr int kTriReads = 36;
constexpr int kTriWin = 8;
// rows 0-2 have 4 pieces, rows 3-6 three, rows 7-10 two, rows 11-14 one
constexpr int tri_m(int k) {
  return k < 12 ? k / 4 : k < 24 ? 3 + (k - 12) / 3 : k < 32 ? 7 + (k - 24) / 2 : 11 + (k - 32);
}
constexpr int tri_i0(int k) {
  return k < 12 ? 4 * (k % 4) : k < 24 ? 4 + 4 * ((k - 12) % 3) : k < 32 ? 8 + 4 * ((k - 24) % 2) : 12;
}
static_assert(tri_m(kTriReads - 1) == 14 && tri_i0(kTriReads - 1) == 12 && tri_m(11) == 2 && tri_i0(11) == 12 &&
                  tri_m(12) == 3 && tri_i0(12) == 4 && tri_m(24) == 7 && tri_i0(25) == 12 && tri_m(32) == 11,
              "36 pieces in the inner solve of a 16-row block");

// One workgroup per (chunk, value head).  u = T (beta v) and w = T (beta e^gc k)
// are the solutions of (I + L) x = rhs; thread j < 128 solves for column j of
// u, thread 128 + j for column j of w, by forward substitution with the rows of
// L read from LDS (every lane reads the same address: broadcast).
// BETA_F32: beta is fp32 (else bf16).
template <bool BETA_F32>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) void gd_prep_kernel(GdArgs a) {
  const int h = blockIdx.x % a.hv;
  const int c = blockIdx.x / a.hv;
  int r0, L;
  chunk_rows(a, c, &r0, &L);
  if (L <= 0) return;
  const int hk = h / (a.hv / a.hk);
  const size_t hc = static_cast<size_t>(h) * a.nc + c;

  __shared__ __attribute__((aligned(16))) unsigned char smem[kPrepBytes];
  uint16_t* sK = reinterpret_cast<uint16_t*>(smem + kPrepK);
  uint16_t* sQ = reinterpret_cast<uint16_t*>(smem + kPrepQ);
  uint16_t* sV = reinterpret_cast<uint16_t*>(smem + kPrepV);
  float* sL = reinterpret_cast<float*>(smem + kPrepL);
  float* sG = reinterpret_cast<float*>(smem + kPrepG);
  float* sB = reinterpret_cast<float*>(smem + kPrepB);
  float* sBG = reinterpret_cast<float*>(smem + kPrepBG);

  const int tid = threadIdx.x;
  const int wv = tid >> 6;
  const int l = tid & 63;
  const int g4 = l >> 4;
  const int c16 = l & 15;

  // q, k, v rows: 16 lanes per row, 8 values (16 bytes) per lane
  const size_t qk_row = static_cast<size_t>(a.hk) * kD;
  const size_t v_row = static_cast<size_t>(a.hv) * kD;
  uint16_t* gq = a.qn + hc * kC * kD;
  // g and beta of row l (padded rows carry g = beta = 0; wave 0 uses them), loaded
  // first and by every wave, with no branch to convert in: wave 0 runs the cumsum
  // below while the q, k, v rows are in flight
  const size_t gidx = static_cast<size_t>(r0 + (l < L ? l : 0)) * a.hv + h;
  const float graw = a.g[gidx];
  float braw;
  if constexpr (BETA_F32)
    braw = static_cast<const float*>(a.beta)[gidx];
  else
    braw = fd_bf16_to_f32(static_cast<const uint16_t*>(a.beta)[gidx]);
  __builtin_amdgcn_sched_barrier(0);
  // every load of the block is issued before any is used (rows past the chunk's
  // end re-read its first row and are zeroed below)
  uint4 rq[4], rk[4], rv[4];
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const int row = it * 16 + wv * 4 + g4;
    const size_t grow = static_cast<size_t>(r0 + (row < L ? row : 0));
    rq[it] = *reinterpret_cast<const uint4*>(a.q + grow * qk_row + hk * kD + c16 * 8);
    rk[it] = *reinterpret_cast<const uint4*>(a.k + grow * qk_row + hk * kD + c16 * 8);
    rv[it] = *reinterpret_cast<const uint4*>(a.v + grow * v_row + h * kD + c16 * 8);
  }
  // g (inclusive cumsum over the chunk) and beta
  if (wv == 0) {
    float gv = l < L ? graw : 0.0f;
    const float bv = l < L ? braw : 0.0f;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float up = __shfl_up(gv, off);
      if (l >= off) gv = gv + up;
    }
    sG[l] = gv;
    sB[l] = bv;
    const float eg = expf(gv);
    sBG[l] = bv * eg;
    const float gl = __shfl(gv, kC - 1);
    float* gx = a.gc + hc * 3 * kC;
    gx[l] = eg;
    gx[kC + l] = expf(gl - gv);
    gx[2 * kC + l] = expf(gl);  // in every place: the state pass copies the block whole
  }
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const int row = it * 16 + wv * 4 + g4;
    const uint4 zero = make_uint4(0, 0, 0, 0);
    uint4 q4 = row < L ? rq[it] : zero;
    uint4 k4 = row < L ? rk[it] : zero;
    const uint4 v4 = row < L ? rv[it] : zero;
    if (a.l2norm) {
      q4 = l2norm_row8(q4);
      k4 = l2norm_row8(k4);
    }
    *reinterpret_cast<uint4*>(sQ + row * kRowK + c16 * 8) = q4;
    *reinterpret_cast<uint4*>(sK + row * kRowK + c16 * 8) = k4;
    *reinterpret_cast<uint4*>(sV + row * kRowK + c16 * 8) = v4;
    *reinterpret_cast<uint4*>(gq + (((row >> 4) * 4 + (c16 >> 2)) * 64 + 16 * (c16 & 3) + (row & 15)) * 8) = q4;
  }
  __syncthreads();

  // Gram (k.k) and q.k lower 32x32 tiles on bf16 MFMA (waves 0-2)
  float* sA = reinterpret_cast<float*>(smem + kPrepQ);
  const int I = wv == 0 ? 0 : 1;
  const int J = wv == 2 ? 1 : 0;
  f32x16_t accG = {};
  f32x16_t accA = {};
  if (wv < 3) {
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int kc = 16 * s + 8 * (l >> 5);
      const bf16x8_t ak = *reinterpret_cast<const bf16x8_t*>(sK + (32 * I + (l & 31)) * kRowK + kc);
      const bf16x8_t aq = *reinterpret_cast<const bf16x8_t*>(sQ + (32 * I + (l & 31)) * kRowK + kc);
      const bf16x8_t bk = *reinterpret_cast<const bf16x8_t*>(sK + (32 * J + (l & 31)) * kRowK + kc);
      accG = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ak, bk, accG, 0, 0, 0);
      accA = __builtin_amdgcn_mfma_f32_32x32x16_bf16(aq, bk, accA, 0, 0, 0);
    }
  }
  __syncthreads();  // the q tile is free: A takes its place
  if (wv < 3) {
    const int j = 32 * J + (l & 31);
    const float gj = sG[j];
    // gc and beta of the lane's 16 rows 32I + 8q + 4(l/32) + e, read before any is
    // used, and the decays computed for every row and then selected: a branch per
    // row would serialise the 16 LDS round trips
    f32x4_t gi[4], bi[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      gi[q] = *reinterpret_cast<const f32x4_t*>(sG + 32 * I + 8 * q + 4 * (l >> 5));
      bi[q] = *reinterpret_cast<const f32x4_t*>(sB + 32 * I + 8 * q + 4 * (l >> 5));
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int i = 32 * I + (r >> 2) * 8 + (l >> 5) * 4 + (r & 3);
      const float e = expf(gi[r >> 2][r & 3] - gj);
      const float dec = i >= j ? e : 0.0f;
      sL[j * kRowF + i] = i > j ? (bi[r >> 2][r & 3] * accG[r]) * dec : 0.0f;  // transposed: sL[j][i] = L[i][j]
      sA[i * kRowF + j] = i >= j ? (a.scale * accA[r]) * dec : 0.0f;
    }
  }
  __syncthreads();
  // A's planes in operand order, row block wv: through LDS a lane stores 16 bytes
  // per plane (straight from the accumulators it would be 2)
  {
    for (int st = 0; st <= (wv >> 1); ++st) {
      uint16_t* ga = a.aq + hc * kAqChunk + aq_offset(wv, st, l);  // upper lanes of a shared tile store the zeros
      const float* src_a = sA + (16 * wv + c16) * kRowF + 32 * st + 8 * g4;
      const f32x4_t v0 = *reinterpret_cast<const f32x4_t*>(src_a);
      const f32x4_t v1 = *reinterpret_cast<const f32x4_t*>(src_a + 4);
      uint4 hi, mid, lo;
      split3x8(v0, v1, hi, mid, lo);
      *reinterpret_cast<uint4*>(ga) = hi;
      *reinterpret_cast<uint4*>(ga + kAqPlane) = mid;
      *reinterpret_cast<uint4*>(ga + 2 * kAqPlane) = lo;
    }
  }

  // forward substitution (I + L) x = rhs, one column per thread (wave wv owns the 64
  // columns of its lanes), in four blocks of 16 rows:
  //  - inside a block, right-looking on the thread's column: once x_m is final every
  //    later row of the block takes -L[i][m] x_m (column m of L is row m of the
  //    transposed tile, read as broadcasts);
  //  - after a block, every remaining row takes -L[rest, block] X_block on fp32 MFMA
  //    (v_mfma_f32_16x16x4f32), the operands and results passing through a
  //    wave-private LDS area (the wave's own 64 columns: no barrier).
  const bool is_w = tid >= kD;   // waves 2, 3
  const int j = tid & (kD - 1);
  const uint16_t* src = is_w ? sK : sV;
  float x[kC];
  uint32_t kbits[kC / 2];
#pragma unroll
  for (int i = 0; i < kC; ++i) {
    const uint32_t bits = src[i * kRowK + j];
    if (i & 1)
      kbits[i >> 1] |= bits << 16;
    else
      kbits[i >> 1] = bits;
    x[i] = (is_w ? sBG[i] : sB[i]) * fd_bf16_to_f32(bits);
  }
  if (is_w) {
    // normalised k^T in the state pass's operand order: row dk = j, the 8 tokens
    // 32st + 8g4 .. +7 of lane 16g4 + (j % 16) (16 lanes write 256 B contiguous);
    // stored before the substitution so that its registers are free there
    uint16_t* kt = a.kn + hc * kC * kD;
    const int kwv = j >> 5, km = (j >> 4) & 1, kc16 = j & 15;
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int i = 4 * (4 * st + g);  // kbits index of token 32st + 8g
        *reinterpret_cast<uint4*>(kt + ((((kwv * 2 + km) * 2 + st) * 64) + 16 * g + kc16) * 8) =
            make_uint4(kbits[i], kbits[i + 1], kbits[i + 2], kbits[i + 3]);
      }
  }
  __syncthreads();  // every wave has read its right-hand sides: the q/k/v tiles are free
  float* wl = reinterpret_cast<float*>(smem) + wv * (48 * 64);  // 12 KiB per wave
  uint16_t* gw = a.w + hc * 3 * kC * kD;
  float* gu = a.u + hc * kC * kD;
  // the four blocks, each with its block index a compile-time constant (a loop
  // this size is beyond the unroller's limit)
  auto block = [&](auto bc) __attribute__((always_inline)) {
    constexpr int b = decltype(bc)::value;
    constexpr int b0 = 16 * b;
    // the block's 36 reads of L pieces pass through a window of kTriWin registers,
    // each issued kTriWin steps before its FMAs, so the LDS latency is not paid per
    // read (x[i] still takes its updates in increasing m)
    f32x4_t lwin[kTriWin];
#pragma unroll
    for (int k = 0; k < kTriWin; ++k)
      lwin[k] = *reinterpret_cast<const f32x4_t*>(sL + (b0 + tri_m(k)) * kRowF + b0 + tri_i0(k));
#pragma unroll
    for (int k = 0; k < kTriReads; ++k) {
      const int m = b0 + tri_m(k), i0 = b0 + tri_i0(k);
      const f32x4_t lv = lwin[k % kTriWin];
      const float xm = x[m];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i0 + e > m) x[i0 + e] = fmaf(-lv[e], xm, x[i0 + e]);
      if (k + kTriWin < kTriReads)
        lwin[k % kTriWin] = *reinterpret_cast<const f32x4_t*>(sL + (b0 + tri_m(k + kTriWin)) * kRowF + b0 +
                                                               tri_i0(k + kTriWin));
      __builtin_amdgcn_sched_barrier(0);
    }
    // X_block (16 rows of the wave's 64 columns) -> LDS [16][64]
#pragma unroll
    for (int k = 0; k < 16; ++k) wl[k * 64 + l] = x[b0 + k];
    // These 16 rows of u or w are final: store them now, in the state pass's
    // operand order, so the writes drain while the later blocks run.
    if (is_w) {
      // w piece (row 16b + lane%16, columns 32c + 8(lane/16) .. +7) as three exact bf16 planes;
      // this wave holds the column groups c = 2(wv-2), 2(wv-2)+1
#pragma unroll
      for (int ch = 0; ch < 2; ++ch) {
        const int q = (b << 8) | ((2 * (wv - 2) + ch) << 6) | l;
        const float* src_row = wl + (l & 15) * 64 + 32 * ch + 8 * (l >> 4);
        const f32x4_t v0 = *reinterpret_cast<const f32x4_t*>(src_row);
        const f32x4_t v1 = *reinterpret_cast<const f32x4_t*>(src_row + 4);
        uint4 hi, mid, lo;
        split3x8(v0, v1, hi, mid, lo);
        *reinterpret_cast<uint4*>(gw + q * 8) = hi;
        *reinterpret_cast<uint4*>(gw + kC * kD + q * 8) = mid;
        *reinterpret_cast<uint4*>(gw + 2 * kC * kD + q * 8) = lo;
      }
    } else {
      // u piece (rows 16b + 4(lane/16) .. +3, column 16g + lane%16) in fp32;
      // this wave holds the column groups g = 4wv .. 4wv+3
#pragma unroll
      for (int cg = 0; cg < 4; ++cg) {
        const int q = ((4 * wv + cg) << 8) | (b << 6) | l;
        const float* src_col = wl + 4 * (l >> 4) * 64 + 16 * cg + (l & 15);
        const f32x4_t v = {src_col[0], src_col[64], src_col[128], src_col[192]};
        *reinterpret_cast<f32x4_t*>(gu + q * 4) = v;
      }
    }
    if constexpr (b == 3) return;
    // C[rest rows][64 columns] = L[rest, block] X_block: rest row tile rt (16 rows), column tile t
    constexpr int kMaxRt = 3;
    const int nrt = 3 - b;
    float bx[4][4];  // B[k = 4s + l/16][n = 16t + l%16]
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int st = 0; st < 4; ++st) bx[t][st] = wl[(4 * st + (l >> 4)) * 64 + 16 * t + (l & 15)];
    f32x4_t acc[kMaxRt][4];
#pragma unroll
    for (int rt = 0; rt < kMaxRt; ++rt) {
      if (rt >= nrt) break;
      float al[4];  // A[i = l%16][k = l/16 + 4s] = L[b0 + 16 + 16rt + l%16][b0 + 4s + l/16]
#pragma unroll
      for (int st = 0; st < 4; ++st) al[st] = sL[(b0 + 4 * st + (l >> 4)) * kRowF + b0 + 16 + 16 * rt + (l & 15)];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        acc[rt][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int st = 0; st < 4; ++st) acc[rt][t] = mfma_f32(al[st], bx[t][st], acc[rt][t]);
      }
    }
    // C -> LDS [rest rows][64], then every lane subtracts its own column
#pragma unroll
    for (int rt = 0; rt < kMaxRt; ++rt) {
      if (rt >= nrt) break;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) wl[(16 * rt + 4 * (l >> 4) + r) * 64 + 16 * t + (l & 15)] = acc[rt][t][r];
    }
#pragma unroll
    for (int i = b0 + 16; i < kC; ++i) x[i] = x[i] - wl[(i - b0 - 16) * 64 + l];
  };
  block(std::integral_constant<int, 0>{});
  block(std::integral_constant<int, 1>{});
  block(std::integral_constant<int, 2>{});
  block(std::integral_constant<int, 3>{});
}

// ---------------------------------------------------------------------------
// 3. sequential state pass over the chunks of one request, with the chunks' outputs
//
// Both products of a chunk run on v_mfma_f32_16x16x32_bf16 with the fp32
// operands split exactly into bf16 planes (x = hi + mid + lo): w S keeps six of
// the nine plane products (hi.hi, hi.mid, mid.hi, hi.lo, mid.mid, lo.hi; the
// rest are below 2^-24 relative), k^T v' (k is a bf16 value) keeps all three.
// The lane layout is that of the fp32 MFMA (A[l%16][k], B[k][l%16],
// D[4(l/16)+r][l%16]) with the 8 consecutive reduction indices 8(l/16)..+7 of
// each 32-step in a lane.
constexpr int kRowSB = kD + 8;   // bf16 row stride of a transposed state plane (272 B)
constexpr int kRowVB = kC + 8;   // bf16 row stride of a transposed v' plane (144 B)

constexpr int kStateThreads = 512;

// PREFETCH: the output wavefronts fetch the operands into L2 ahead of the loads.
template <bool PREFETCH>
__global__ __launch_bounds__(kStateThreads) void gd_state_kernel(GdArgs a) {
  // Block b runs on XCD b % 8.  The 8 column slices of one head (which read the
  // same w / k / q / A tiles) go to one XCD and share its L2; the heads of one
  // request go round the XCDs, and the longest requests come first.  (A
  // contiguous range of heads per XCD left the 8002-token request of four on two
  // XCDs, two rounds of it: state pass 541 -> 297 us.)
  const int unit = blockIdx.x / (8 * kSlices) * 8 + blockIdx.x % 8;
  if (unit >= a.nseq * a.hv) return;
  const int js = blockIdx.x / 8 % kSlices;
  const int h = unit % a.hv;
  const int sq = a.varlen ? a.order[static_cast<size_t>(unit / a.hv) * kOrderStep] : unit / a.hv;
  int first, last;
  request_chunks(a, sq, &first, &last);

  __shared__ __attribute__((aligned(16))) uint16_t sS[3][kSlice * kRowSB];   // state planes [col][dk]
  __shared__ __attribute__((aligned(16))) uint16_t sVd[3][kSlice * kRowVB];  // e^{gl - gc} v' planes [col][t]
  __shared__ __attribute__((aligned(16))) uint16_t sVp[3][kSlice * kRowVB];  // v' planes [col][t]
  __shared__ __attribute__((aligned(16))) float sE[2][3 * kC];               // a chunk's exponentials (GdArgs::gc)

  const int tid = threadIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63;
  const int g4 = l >> 4;
  const int c16 = l & 15;
  const int col = kSlice * js + c16;  // value column owned in the C layout
  const size_t state_base = (static_cast<size_t>(sq) * a.hv + h) * kD * kD;

  if (wv < 4) {
    // ---- the state chain (wavefront wv: v' rows 16wv .. +15, state rows 32wv .. +31)
    // state slice in the C layout (fp32): S[m][r] = S[dk = 32wv + 16m + 4g4 + r][col]
    float S[2][4];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        S[m][r] = a.s0 ? a.s0[state_base + static_cast<size_t>(32 * wv + 16 * m + 4 * g4 + r) * kD + col] : 0.0f;

    // operands of one chunk, loaded straight into registers two chunks ahead;
    // three register sets rotate (the loop body is unrolled by three) and every
    // load is issued unconditionally (past the last chunk it re-reads the last one)
    struct ChunkRegs {
      uint4 w[3][4];  // plane x, step s: w_x[16wv + c16][32s + 8g4 .. +7]      (A of w S)
      uint4 k[2][2];  // tile m, step s: k^T[32wv + 16m + c16][32s + 8g4 .. +7]  (A of k^T v')
      f32x4_t u;      // u[16wv + 4g4 + r][col]                                 (C layout)
    };
    // The chunk to load next: uniform pointers that advance by a chunk, and stay on
    // the request's last one.  (Addresses formed from the chunk index cost each part
    // of the loads several 64-bit scalar multiplies, in line with the chain.)
    const size_t hc0 = static_cast<size_t>(h) * a.nc + first;
    const uint16_t* pw = a.w + hc0 * 3 * kC * kD;
    const uint16_t* pk = a.kn + hc0 * kC * kD;
    const float* pu = a.u + hc0 * kC * kD;
    int at = first;
    const int lane_op = (wv * 4 * 64 + l) * 8, lane_u = ((js * 4 + wv) * 64 + l) * 4;
    // Its 17 operand loads: 4 x + st plane x of w, 12 + 2 m + st k^T, then u.
    constexpr int kOps = 17;
    auto load_op = [&](ChunkRegs& R, int i) {
      if (i < 12) {
        R.w[i >> 2][i & 3] = *reinterpret_cast<const uint4*>(pw + (i >> 2) * kC * kD + lane_op + (i & 3) * 64 * 8);
      } else if (i < 16) {
        R.k[(i >> 1) & 1][i & 1] = *reinterpret_cast<const uint4*>(pk + lane_op + (i & 3) * 64 * 8);
      } else {
        R.u = *reinterpret_cast<const f32x4_t*>(pu + lane_u);
      }
    };
    auto next_chunk = [&]() {
      if (at + 1 < last) {
        ++at;
        pw += 3 * kC * kD;
        pk += kC * kD;
        pu += kC * kD;
      }
    };
    auto load_ops = [&](ChunkRegs& R, int i0, int i1) {
#pragma unroll
      for (int i = i0; i < i1; ++i) load_op(R, i);
    };

    // One chunk.  The loads of the chunk two ahead into P are spread over the step:
    // before the barriers, where the wavefront waits anyway, and one behind each
    // group of MFMAs.  The CU returns at most 64 B per cycle to all eight wavefronts
    // (the data return unit is busy 75 % of the pass), so a load issued with others
    // waits about 100 cycles in line; behind MFMAs that wait is theirs.
    // sched_barrier keeps each in place.  Spread so, the loads cost nothing: what
    // sets the step are the LDS reads of the planes after its two barriers, 72 KB
    // here and 66 KB by the output wavefronts (B=1, T=2048, copies for timing only,
    // pass 40.5 us: no global loads at all 41.4; no plane reads here 38.4, by the
    // outputs 37.0, by neither 27.9; no output work 37.4).
    int par = 0;  // the chunk's buffer of exponentials
    auto step = [&](const ChunkRegs& R, ChunkRegs& P) {
      // state at the chunk start: bf16 planes to LDS (B of w S and of the output's q S)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const int dk = 32 * wv + 16 * m + 4 * g4;
        uint2 ph, pm, pl;
        split3x4(S[m], ph, pm, pl);
        *reinterpret_cast<uint2*>(sS[0] + c16 * kRowSB + dk) = ph;
        *reinterpret_cast<uint2*>(sS[1] + c16 * kRowSB + dk) = pm;
        *reinterpret_cast<uint2*>(sS[2] + c16 * kRowSB + dk) = pl;
      }
      __builtin_amdgcn_sched_barrier(0);
      load_ops(P, 0, 4);
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();

      // v' = u - w S for rows 16wv..16wv+15 of this slice
      f32x4_t acc0 = {};
      f32x4_t acc1 = {};
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const int off = c16 * kRowSB + 32 * st + 8 * g4;
        const uint4 sh = *reinterpret_cast<const uint4*>(sS[0] + off);
        const uint4 sm = *reinterpret_cast<const uint4*>(sS[1] + off);
        const uint4 sl = *reinterpret_cast<const uint4*>(sS[2] + off);
        acc0 = mfma_bf16(R.w[0][st], sh, acc0);
        acc1 = mfma_bf16(R.w[0][st], sm, acc1);
        acc0 = mfma_bf16(R.w[1][st], sh, acc0);
        acc1 = mfma_bf16(R.w[0][st], sl, acc1);
        acc0 = mfma_bf16(R.w[1][st], sm, acc0);
        acc1 = mfma_bf16(R.w[2][st], sh, acc1);
        load_op(P, 4 + st);
        __builtin_amdgcn_sched_barrier(0);
      }
      const f32x4_t dec = *reinterpret_cast<const f32x4_t*>(sE[par] + kC + 16 * wv + 4 * g4);
      const float egl = sE[par][2 * kC];
      par ^= 1;
      f32x4_t vnew;
      float vdec[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        vnew[r] = R.u[r] - (acc0[r] + acc1[r]);
        vdec[r] = vnew[r] * dec[r];
      }
      {
        const int off = c16 * kRowVB + 16 * wv + 4 * g4;
        uint2 ph, pm, pl;
        split3x4(vdec, ph, pm, pl);
        *reinterpret_cast<uint2*>(sVd[0] + off) = ph;
        *reinterpret_cast<uint2*>(sVd[1] + off) = pm;
        *reinterpret_cast<uint2*>(sVd[2] + off) = pl;
        // v'[t][col] planes for the output wavefronts
        const float vv[4] = {vnew[0], vnew[1], vnew[2], vnew[3]};
        split3x4(vv, ph, pm, pl);
        *reinterpret_cast<uint2*>(sVp[0] + off) = ph;
        *reinterpret_cast<uint2*>(sVp[1] + off) = pm;
        *reinterpret_cast<uint2*>(sVp[2] + off) = pl;
      }
      __builtin_amdgcn_sched_barrier(0);
      load_ops(P, 8, 12);
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();

      // S <- e^{gl} S + k^T (e^{gl - gc} v'), dk rows 32wv..32wv+31
      f32x4_t st0 = {S[0][0] * egl, S[0][1] * egl, S[0][2] * egl, S[0][3] * egl};
      f32x4_t st1 = {S[1][0] * egl, S[1][1] * egl, S[1][2] * egl, S[1][3] * egl};
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const int off = c16 * kRowVB + 32 * st + 8 * g4;
        const uint4 dh = *reinterpret_cast<const uint4*>(sVd[0] + off);
        const uint4 dm = *reinterpret_cast<const uint4*>(sVd[1] + off);
        const uint4 dl = *reinterpret_cast<const uint4*>(sVd[2] + off);
        st0 = mfma_bf16(R.k[0][st], dh, st0);
        st1 = mfma_bf16(R.k[1][st], dh, st1);
        load_op(P, 12 + 2 * st);
        __builtin_amdgcn_sched_barrier(0);
        st0 = mfma_bf16(R.k[0][st], dm, st0);
        st1 = mfma_bf16(R.k[1][st], dm, st1);
        load_op(P, 13 + 2 * st);
        __builtin_amdgcn_sched_barrier(0);
        st0 = mfma_bf16(R.k[0][st], dl, st0);
        st1 = mfma_bf16(R.k[1][st], dl, st1);
        if (st == 1) load_op(P, 16);
        __builtin_amdgcn_sched_barrier(0);
      }
      next_chunk();
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        S[0][r] = st0[r];
        S[1][r] = st1[r];
      }
      // no third barrier: the next writes of sS follow this step's second
      // barrier, and the next writes of sVd and sVp follow the next step's first
    };

    if (first < last) {
      ChunkRegs A, B, Cr;
      load_ops(A, 0, kOps);
      next_chunk();
      load_ops(B, 0, kOps);
      next_chunk();
      for (int c = first; c < last; c += 3) {
        step(A, Cr);
        if (c + 1 < last) step(B, A);
        if (c + 2 < last) step(Cr, B);
      }
    }

    if (a.sN != nullptr) {
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          a.sN[state_base + static_cast<size_t>(32 * wv + 16 * m + 4 * g4 + r) * kD + col] = S[m][r];
    }
  } else {
    // ---- the chunk outputs (wavefront wv: rows 16rt .. +15 of every chunk)
    //   o[t][col] = scale e^{gc_t} (q S_chunk)[t][col] + (A v')[t][col]
    // q S takes the three products of the bf16 q with the state planes the
    // chain wrote; A v' six of the nine plane products of exact three-plane
    // splits of the fp32 A and v'.
    const int rt = wv - 4;
    const size_t o_row = static_cast<size_t>(a.hv) * kD;
    struct OutRegs {
      uint4 q[4];       // q[16rt + c16][32st + 8g4 .. +7]
      uint4 a[2][3];    // plane x of A[16rt + c16][32st + 8g4 .. +7]; st = 1 for rt >= 2 only
      f32x4_t e;        // wavefront rt = 0: the chunk's exponentials 4l .. 4l + 3, for every wavefront
    };
    // the chunk to load next, as the chain's
    const size_t hc0 = static_cast<size_t>(h) * a.nc + first;
    const uint16_t* pq = a.qn + hc0 * kC * kD;
    const uint16_t* pa = a.aq + hc0 * kAqChunk;
    const float* pg = a.gc + hc0 * 3 * kC;
    int at = first;
    const int lane_q = (rt * 4 * 64 + l) * 8, lane_e = 4 * min(l, 3 * kC / 4 - 1);
    const int lane_a[2] = {aq_offset(rt, 0, l), aq_offset(rt, 1, l)};
    // its 11 loads: 0 .. 3 q, 4 .. 9 the A planes, 10 the exponentials
    auto load_op = [&](OutRegs& R, int i) {
      if (i < 4) {
        R.q[i] = *reinterpret_cast<const uint4*>(pq + lane_q + i * 64 * 8);
      } else if (i < 10) {
        if (i < 7 || rt >= 2)
          R.a[(i - 4) / 3][(i - 4) % 3] = *reinterpret_cast<const uint4*>(pa + lane_a[(i - 4) / 3] + (i - 4) % 3 * kAqPlane);
      } else if (rt == 0) {
        R.e = *reinterpret_cast<const f32x4_t*>(pg + lane_e);
      }
    };
    auto next_chunk = [&]() {
      if (at + 1 < last) {
        ++at;
        pq += kC * kD;
        pa += kAqChunk;
        pg += 3 * kC;
      }
    };
    auto load_out = [&](OutRegs& R) {
#pragma unroll
      for (int i = 0; i < 11; ++i) load_op(R, i);
      next_chunk();
    };
    // L2 prefetch: the operands of the chunk four ahead, one 4-byte load
    // of each 128-byte line; the 32 output wavefronts of a head's slices take a share
    // each, and a lane keeps one line's address.
    const char* pf_line = nullptr;
    int pf_step = 0, pf_left = 0;  // chunks from pf_line's to the request's last
    if constexpr (PREFETCH) {
      constexpr int kRegions = 6;
      constexpr int kBytes[kRegions] = {3 * kC * kD * 2, kC * kD * 2, kC * kD * 4, kC * kD * 2, 3 * kAqPlane * 2, 3 * kC * 4};
      constexpr int kStep[kRegions] = {3 * kC * kD * 2, kC * kD * 2, kC * kD * 4, kC * kD * 2, kAqChunk * 2, 3 * kC * 4};
      constexpr int kLines = (kBytes[0] + kBytes[1] + kBytes[2] + kBytes[3] + kBytes[4] + kBytes[5]) / 128;
      constexpr int kShare = (kLines + 4 * kSlices - 1) / (4 * kSlices);
      static_assert(kShare <= 64, "one line per lane");
      const void* const base[kRegions] = {a.w, a.kn, a.u, a.qn, a.aq, a.gc};
      const int line = l < kShare ? (js * 4 + rt) * kShare + l : kLines;
      int begin = 0;
#pragma unroll
      for (int r = 0; r < kRegions; ++r) {
        if (line >= begin && line < begin + kBytes[r] / 128) {
          pf_line = static_cast<const char*>(base[r]) + hc0 * kStep[r] + (line - begin) * 128;
          pf_step = kStep[r];
          pf_left = last - 1 - first;
        }
        begin += kBytes[r] / 128;
      }
    }
    auto prefetch = [&]() {
      int v = 0;
      if (pf_left >= 0 && pf_line != nullptr) v = *reinterpret_cast<const int*>(pf_line);
      pf_line += pf_step;
      --pf_left;
      return v;
    };
    int pf_value = 0;
    // the request's rows: chunk c of it holds rows [row, min(row + 64, row_end)), row
    // advancing with c
    int row = 0, row_end = 0;
    if (first < last) {
      int tail_row, tail_len;
      chunk_rows(a, first, &row, &tail_len);
      chunk_rows(a, last - 1, &tail_row, &tail_len);
      row_end = tail_row + tail_len;
    }
    uint16_t* po = a.o + static_cast<size_t>(row) * o_row + h * kD;  // uniform: the lane's part is lane_o
    const int lane_row = 16 * rt + 4 * g4 + 2 * (l & 1);  // of the two rows this lane stores
    const int lane_o = lane_row * a.hv * kD + (col & ~1);
    // The barriers match the chain's step: the first finds the chunk-start
    // state planes in sS, the second the v' planes in sVp.  The chain waits here
    // for these wavefronts as much as they for it, so what they need not do is not
    // done: A comes split from prep, the zero half of its upper rows is skipped, a
    // chunk's rows follow from the last's, every LDS read of a phase is issued before
    // its MFMAs (a dependent chain) and one load of the chunk two ahead behind each
    // of those (B=1, T=2048: state pass 46.8 -> 42 us, prep 24.6 -> 25.4; 64 requests
    // of 64 tokens: 164 -> 148 us for the call).
    int par = 0;  // the chunk's buffer of exponentials
    auto out_step = [&](const OutRegs& R, const OutRegs& N, OutRegs& P) {
      __syncthreads();
      f32x4_t acc1 = {};
      uint4 sp[4][3];
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int x = 0; x < 3; ++x) sp[st][x] = *reinterpret_cast<const uint4*>(sS[x] + c16 * kRowSB + 32 * st + 8 * g4);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int st = 0; st < 4; ++st) {
#pragma unroll
        for (int x = 0; x < 3; ++x) {
          acc1 = mfma_bf16(R.q[st], sp[st][x], acc1);
          if (st * 3 + x < 11) load_op(P, st * 3 + x);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      next_chunk();
      if constexpr (PREFETCH) {
        asm volatile("" ::"v"(pf_value));  // the last step's line, long arrived
        pf_value = prefetch();
      }
      __syncthreads();
      f32x4_t acc2 = {};
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        if (st == 1 && rt < 2) break;  // A is lower triangular: zero right of column 31 in rows 0..31
        const int off = c16 * kRowVB + 32 * st + 8 * g4;
        const uint4 b0 = *reinterpret_cast<const uint4*>(sVp[0] + off);
        const uint4 b1 = *reinterpret_cast<const uint4*>(sVp[1] + off);
        const uint4 b2 = *reinterpret_cast<const uint4*>(sVp[2] + off);
        acc2 = mfma_bf16(R.a[st][0], b0, acc2);
        acc2 = mfma_bf16(R.a[st][0], b1, acc2);
        acc2 = mfma_bf16(R.a[st][1], b0, acc2);
        acc2 = mfma_bf16(R.a[st][0], b2, acc2);
        acc2 = mfma_bf16(R.a[st][1], b1, acc2);
        acc2 = mfma_bf16(R.a[st][2], b0, acc2);
      }
      const f32x4_t eg = *reinterpret_cast<const f32x4_t*>(sE[par] + 16 * rt + 4 * g4);
      par ^= 1;
      if (rt == 0) *reinterpret_cast<f32x4_t*>(sE[par] + lane_e) = N.e;  // read after the next step's first barrier
      float val[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) val[r] = (a.scale * eg[r]) * acc1[r] + acc2[r];
      // lanes 2i and 2i + 1 (columns c, c + 1) swap two of their four rows, so that each
      // stores two rows of a column pair
      const uint32_t p01 = fd_pack2(val[0], val[1]), p23 = fd_pack2(val[2], val[3]);
      const bool odd = l & 1;
      const uint32_t own = odd ? p23 : p01;
      const uint32_t other = static_cast<uint32_t>(
          __builtin_amdgcn_mov_dpp(static_cast<int>(odd ? p01 : p23), 0xB1, 0xF, 0xF, false));  // quad_perm [1,0,3,2]
      const uint32_t c0 = odd ? other : own, c1 = odd ? own : other;
      const uint32_t lo = (c0 & 0xffffu) | (c1 << 16), hi = (c0 >> 16) | (c1 & 0xffff0000u);
      if (row + kC <= row_end) {  // uniform: every row of the chunk is valid
        *reinterpret_cast<uint32_t*>(po + lane_o) = lo;
        *reinterpret_cast<uint32_t*>(po + lane_o + a.hv * kD) = hi;
      } else {
        if (row + lane_row < row_end) *reinterpret_cast<uint32_t*>(po + lane_o) = lo;
        if (row + lane_row + 1 < row_end) *reinterpret_cast<uint32_t*>(po + lane_o + a.hv * kD) = hi;
      }
      row += kC;
      po += kC * o_row;
    };

    if (first < last) {
      OutRegs A, B, Cr;
      load_out(A);
      load_out(B);
      if constexpr (PREFETCH) {  // the loads above are chunks 0 and 1, the steps fetch chunk 4 on
        pf_line += 2 * pf_step;
        pf_left -= 2;
        const int v2 = prefetch();
        pf_value = prefetch();
        asm volatile("" ::"v"(v2));
      }
      if (rt == 0) *reinterpret_cast<f32x4_t*>(sE[0] + lane_e) = A.e;
      for (int c = first; c < last; c += 3) {
        out_step(A, B, Cr);
        if (c + 1 < last) out_step(B, Cr, A);
        if (c + 2 < last) out_step(Cr, A, B);
      }
    }
  }
}

// Byte offsets of the workspace regions: the chunk table, the per-(head, chunk)
// intermediates GdArgs describes, and `ob`, the raw bf16 output rows
// [tokens, Hv, 128] that the gated norm reads (fd_gated_delta_norm_fwd only).
struct GdLayout {
  size_t row0, len, first, gc, qn, kn, w, u, aq, ob, total;
};

GdLayout gd_layout(int64_t nc, int64_t hv, int64_t nseq, int64_t tokens) {
  auto al = [](size_t x) { return (x + 255) & ~static_cast<size_t>(255); };
  const size_t hc = static_cast<size_t>(hv) * static_cast<size_t>(nc);
  GdLayout L;
  size_t off = 0;
  L.row0 = off;
  off = al(off + static_cast<size_t>(nc) * 4);
  L.len = off;
  off = al(off + static_cast<size_t>(nc) * 4);
  L.first = off;
  off = al(off + static_cast<size_t>(nseq + 1) * 4);
  L.gc = off;
  off = al(off + hc * 3 * kC * 4);
  L.qn = off;
  off = al(off + hc * kC * kD * 2);
  L.kn = off;
  off = al(off + hc * kC * kD * 2);
  L.w = off;
  off = al(off + hc * 3 * kC * kD * 2);
  L.u = off;
  off = al(off + hc * kC * kD * 4);
  L.aq = off;
  off = al(off + hc * kAqChunk * 2);
  L.ob = off;
  off = al(off + static_cast<size_t>(tokens) * hv * kD * 2);
  L.total = off;
  return L;
}

// chunks and requests of a launch; false if the sizes are out of range
bool gd_counts(int batch, int seq_len, int n_seqs, bool varlen, int64_t* nc, int64_t* nseq) {
  if (batch < 0 || seq_len < 0) return false;
  const int64_t total = static_cast<int64_t>(batch) * seq_len;
  if (total >= (1LL << 31)) return false;
  if (varlen) {
    if (n_seqs < 1 || batch != 1) return false;
    *nseq = n_seqs;
    *nc = (total + kC - 1) / kC + n_seqs;
  } else {
    *nseq = batch;
    *nc = static_cast<int64_t>(batch) * ((seq_len + kC - 1) / kC);
  }
  return true;
}

}  // namespace

extern "C" FD_API int64_t fd_gated_delta_workspace_bytes(int batch, int seq_len, int v_heads, int head_k_dim,
                                                         int head_v_dim, int n_seqs) {
  if (v_heads <= 0 || head_k_dim != kD || head_v_dim != kD) return FD_ERR_UNSUPPORTED;
  int64_t nc = 0, nseq = 0;
  if (!gd_counts(batch, seq_len, n_seqs, n_seqs > 0, &nc, &nseq)) return FD_ERR_INVALID_ARGUMENT;
  return static_cast<int64_t>(gd_layout(nc, v_heads, nseq, static_cast<int64_t>(batch) * seq_len).total);
}

namespace {

struct GdNorm {
  const void* z;
  int64_t z_ts, z_hs;
  const void* w;
  int w_dtype;
  float eps;
};

int gd_run(const void* q, const void* k, const void* v, const float* g, const void* beta, void* out,
           const float* initial_state, float* final_state, void* workspace, int64_t workspace_bytes, int batch,
           int seq_len, int k_heads, int v_heads, int head_k_dim, int head_v_dim, float scale, int beta_dtype,
           int l2norm_qk, const int32_t* cu_seqlens, int n_seqs, void* stream, const GdNorm* norm) {
  FD_REQUIRE(q && k && v && g && beta && out && workspace, FD_ERR_INVALID_ARGUMENT,
             "fd_gated_delta_fwd: q, k, v, g, beta, out and workspace must be non-null");
  FD_REQUIRE(k_heads > 0 && v_heads > 0 && v_heads % k_heads == 0, FD_ERR_INVALID_ARGUMENT,
             "fd_gated_delta_fwd: v_heads (%d) must be a positive multiple of k_heads (%d)", v_heads, k_heads);
  FD_REQUIRE(head_k_dim == kD && head_v_dim == kD, FD_ERR_UNSUPPORTED,
             "fd_gated_delta_fwd: head_k_dim and head_v_dim must be 128 (got %d, %d)", head_k_dim, head_v_dim);
  FD_REQUIRE(beta_dtype == FD_DTYPE_BF16 || beta_dtype == FD_DTYPE_F32, FD_ERR_INVALID_ARGUMENT,
             "fd_gated_delta_fwd: beta_dtype must be FD_DTYPE_BF16 or FD_DTYPE_F32");
  FD_REQUIRE(scale > 0.0f && scale < 1e30f, FD_ERR_INVALID_ARGUMENT, "fd_gated_delta_fwd: scale must be positive");
  FD_REQUIRE(fd_aligned16(q) && fd_aligned16(k) && fd_aligned16(v) && fd_aligned16(out) && fd_aligned16(workspace),
             FD_ERR_ALIGNMENT, "fd_gated_delta_fwd: q, k, v, out and workspace must be 16-byte aligned");
  FD_REQUIRE((reinterpret_cast<uintptr_t>(g) & 3u) == 0 && (reinterpret_cast<uintptr_t>(beta) & 1u) == 0 &&
                 (beta_dtype != FD_DTYPE_F32 || (reinterpret_cast<uintptr_t>(beta) & 3u) == 0),
             FD_ERR_ALIGNMENT, "fd_gated_delta_fwd: g and beta must be aligned to their element size");
  const bool varlen = cu_seqlens != nullptr;
  if (varlen) {
    FD_REQUIRE(batch == 1, FD_ERR_INVALID_ARGUMENT, "fd_gated_delta_fwd: cu_seqlens requires batch == 1 (got %d)",
               batch);
    FD_REQUIRE(n_seqs >= 1, FD_ERR_INVALID_ARGUMENT, "fd_gated_delta_fwd: n_seqs must be >= 1 with cu_seqlens");
  }
  int64_t nc = 0, nseq = 0;
  FD_REQUIRE(gd_counts(batch, seq_len, n_seqs, varlen, &nc, &nseq), FD_ERR_INVALID_ARGUMENT,
             "fd_gated_delta_fwd: batch and seq_len must be >= 0 with batch * seq_len < 2^31");
  FD_REQUIRE(nc * v_heads < (1LL << 31) && (nseq * v_heads + 7) * kSlices < (1LL << 31), FD_ERR_INVALID_ARGUMENT,
             "fd_gated_delta_fwd: problem too large");
  if (nseq == 0) return FD_OK;  // empty batch: nothing to launch
  const int64_t total = static_cast<int64_t>(batch) * seq_len;
  // the gated norm runs over total * v_heads rows (checked here so nothing is launched if it cannot)
  FD_REQUIRE(norm == nullptr || total * v_heads < (1LL << 31), FD_ERR_INVALID_ARGUMENT,
             "fd_gated_delta_norm_fwd: problem too large (batch * seq_len * v_heads must be < 2^31)");
  const GdLayout lay = gd_layout(nc, v_heads, nseq, total);
  FD_REQUIRE(workspace_bytes >= static_cast<int64_t>(lay.total), FD_ERR_INVALID_ARGUMENT,
             "fd_gated_delta_fwd: workspace too small (%lld bytes, need %lld)",
             static_cast<long long>(workspace_bytes), static_cast<long long>(lay.total));

  unsigned char* ws = static_cast<unsigned char*>(workspace);
  GdArgs a;
  a.q = static_cast<const uint16_t*>(q);
  a.k = static_cast<const uint16_t*>(k);
  a.v = static_cast<const uint16_t*>(v);
  a.g = g;
  a.beta = beta;
  // with the gated norm the raw output rows go to the workspace and the norm writes `out`
  a.o = norm ? reinterpret_cast<uint16_t*>(ws + lay.ob) : static_cast<uint16_t*>(out);
  a.s0 = initial_state;
  a.sN = final_state;
  a.row0 = reinterpret_cast<int32_t*>(ws + lay.row0);
  a.len = reinterpret_cast<int32_t*>(ws + lay.len);
  a.first = reinterpret_cast<int32_t*>(ws + lay.first);
  a.gc = reinterpret_cast<float*>(ws + lay.gc);
  a.qn = reinterpret_cast<uint16_t*>(ws + lay.qn);
  a.kn = reinterpret_cast<uint16_t*>(ws + lay.kn);
  a.w = reinterpret_cast<uint16_t*>(ws + lay.w);
  a.u = reinterpret_cast<float*>(ws + lay.u);
  a.aq = reinterpret_cast<uint16_t*>(ws + lay.aq);
  a.order = reinterpret_cast<int32_t*>(a.aq + 3 * kAqPlane);
  a.hk = k_heads;
  a.hv = v_heads;
  a.nc = static_cast<int>(nc);
  a.nseq = static_cast<int>(nseq);
  a.varlen = varlen;
  a.seq_len = seq_len;
  a.nct = (seq_len + kC - 1) / kC;
  a.beta_f32 = beta_dtype == FD_DTYPE_F32;
  a.l2norm = l2norm_qk != 0;
  a.scale = scale;

  hipStream_t s = static_cast<hipStream_t>(stream);
  if (varlen)
    hipLaunchKernelGGL(gd_chunk_table, dim3(1), dim3(kTableThreads), 0, s, cu_seqlens, static_cast<int>(total), a);
  if (nc > 0) {
    if (a.beta_f32)
      hipLaunchKernelGGL(gd_prep_kernel<true>, dim3(static_cast<unsigned>(nc * v_heads)), dim3(kThreads), 0, s, a);
    else
      hipLaunchKernelGGL(gd_prep_kernel<false>, dim3(static_cast<unsigned>(nc * v_heads)), dim3(kThreads), 0, s, a);
  }
  const int64_t units = (nseq * v_heads + 7) / 8 * 8;  // (request, head) units, rounded up to the XCDs
  // Intermediates that do not fit the 256 MB memory-side cache beside q, k, v and the
  // output come from HBM, too late for loads two chunks ahead: long chains then fetch
  // four chunks ahead into L2.  The line, 208 MiB = 218 MB, lies between the sizes that
  // gain and lose (B=1, 16 heads: T=8192, 270 MB, 339 -> 282 us; T=7000, 232 MB, 248 ->
  // 230; T=6000, 198 MB, 191.9 -> 188.8; T=4096, 135 MB, 123.6 -> 129.1; B=4, T=2048,
  // 270 MB, 236 -> 217).  Short chains pay for it (40 requests of 10 to 200 tokens: 164
  // -> 177 us), so the requests must have 24 chunks on average: the host knows no more
  // of packed lengths.  One long request among many short ones runs without it.
  const dim3 state_grid(static_cast<unsigned>(units * kSlices));
  if (lay.ob > 208LL << 20 && nc >= 24 * nseq)
    hipLaunchKernelGGL(gd_state_kernel<true>, state_grid, dim3(kStateThreads), 0, s, a);
  else
    hipLaunchKernelGGL(gd_state_kernel<false>, state_grid, dim3(kStateThreads), 0, s, a);
  const int rc = fd_check_launch("fd_gated_delta_fwd");
  if (rc != FD_OK || norm == nullptr || total == 0) return rc;
  // the layer's gated RMSNorm over the raw output rows (one row per token and value head)
  return fd_gated_rmsnorm_fwd(a.o, norm->z, norm->z_ts, norm->z_hs, v_heads, norm->w, norm->w_dtype, out,
                              total * v_heads, kD, norm->eps, stream);
}

}  // namespace

// ---------------------------------------------------------------------------
// Static device scratch of fd_gated_delta_fwd_noalloc: the workspace of callers
// that cannot allocate (HIP graph capture, serving loops).  Every GPU the
// library runs on holds its own copy for the life of the process.  Host code
// never passes `scratch` itself to a kernel (in host code the name is a
// host-side stand-in, not a device address): it uses the address that
// hipGetSymbolAddress returns once per device.
static __device__ __align__(256) unsigned char scratch[FD_GD_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the device `stream` belongs to (the current
// device for the null stream), looked up on that device's first call.
int scratch_address(hipStream_t stream, void** out) {
  int dev = -1;
  if (stream != nullptr) {
    FD_REQUIRE(hipStreamGetDevice(stream, &dev) == hipSuccess, FD_ERR_LAUNCH,
               "fd_gated_delta_fwd_noalloc: cannot query the stream's device");
  } else {
    FD_REQUIRE(hipGetDevice(&dev) == hipSuccess, FD_ERR_LAUNCH, "fd_gated_delta_fwd_noalloc: no current device");
  }
  FD_REQUIRE(dev >= 0 && dev < kMaxDevices, FD_ERR_UNSUPPORTED, "fd_gated_delta_fwd_noalloc: device %d out of range",
             dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    int cur = -1;
    FD_REQUIRE(hipGetDevice(&cur) == hipSuccess, FD_ERR_LAUNCH, "fd_gated_delta_fwd_noalloc: no current device");
    if (cur != dev) FD_REQUIRE(hipSetDevice(dev) == hipSuccess, FD_ERR_LAUNCH,
                               "fd_gated_delta_fwd_noalloc: cannot select device %d", dev);
    void* p = nullptr;
    const hipError_t err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (cur != dev) (void)hipSetDevice(cur);
    FD_REQUIRE(err == hipSuccess && p != nullptr, FD_ERR_LAUNCH,
               "fd_gated_delta_fwd_noalloc: hipGetSymbolAddress of the scratch failed: %s", hipGetErrorString(err));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return FD_OK;
}

}  // namespace

extern "C" FD_API int fd_gated_delta_fwd(const void* q, const void* k, const void* v, const float* g,
                                         const void* beta, void* out, const float* initial_state,
                                         float* final_state, void* workspace, int64_t workspace_bytes, int batch,
                                         int seq_len, int k_heads, int v_heads, int head_k_dim, int head_v_dim,
                                         float scale, int beta_dtype, int l2norm_qk, const int32_t* cu_seqlens,
                                         int n_seqs, void* stream) {
  return gd_run(q, k, v, g, beta, out, initial_state, final_state, workspace, workspace_bytes, batch, seq_len,
                k_heads, v_heads, head_k_dim, head_v_dim, scale, beta_dtype, l2norm_qk, cu_seqlens, n_seqs, stream,
                nullptr);
}

extern "C" FD_API int fd_gated_delta_norm_fwd(const void* q, const void* k, const void* v, const float* g,
                                              const void* beta, const void* z, int64_t z_token_stride,
                                              int64_t z_head_stride, const void* norm_weight, int norm_weight_dtype,
                                              float norm_eps, void* out, const float* initial_state,
                                              float* final_state, void* workspace, int64_t workspace_bytes,
                                              int batch, int seq_len, int k_heads, int v_heads, int head_k_dim,
                                              int head_v_dim, float scale, int beta_dtype, int l2norm_qk,
                                              const int32_t* cu_seqlens, int n_seqs, void* stream) {
  FD_REQUIRE(z && norm_weight, FD_ERR_INVALID_ARGUMENT, "fd_gated_delta_norm_fwd: z and norm_weight must be non-null");
  FD_REQUIRE(norm_weight_dtype == FD_DTYPE_BF16 || norm_weight_dtype == FD_DTYPE_F32, FD_ERR_INVALID_ARGUMENT,
             "fd_gated_delta_norm_fwd: norm_weight_dtype must be FD_DTYPE_BF16 or FD_DTYPE_F32");
  FD_REQUIRE(norm_eps >= 0.0f, FD_ERR_INVALID_ARGUMENT, "fd_gated_delta_norm_fwd: norm_eps must be >= 0");
  FD_REQUIRE(fd_aligned16(z) && z_token_stride % 8 == 0 && z_head_stride % 8 == 0 && z_head_stride >= kD &&
                 z_token_stride >= static_cast<int64_t>(v_heads) * z_head_stride,
             FD_ERR_ALIGNMENT,
             "fd_gated_delta_norm_fwd: z must be 16-byte aligned with strides that are multiples of 8 covering "
             "[v_heads, 128]");
  FD_REQUIRE((reinterpret_cast<uintptr_t>(norm_weight) & (norm_weight_dtype == FD_DTYPE_F32 ? 3u : 1u)) == 0,
             FD_ERR_ALIGNMENT, "fd_gated_delta_norm_fwd: norm_weight must be aligned to its element size");
  const GdNorm norm{z, z_token_stride, z_head_stride, norm_weight, norm_weight_dtype, norm_eps};
  return gd_run(q, k, v, g, beta, out, initial_state, final_state, workspace, workspace_bytes, batch, seq_len,
                k_heads, v_heads, head_k_dim, head_v_dim, scale, beta_dtype, l2norm_qk, cu_seqlens, n_seqs, stream,
                &norm);
}

extern "C" FD_API int fd_gated_delta_fwd_noalloc(const void* q, const void* k, const void* v, const float* g,
                                                 const void* beta, void* out, const float* initial_state,
                                                 float* final_state, int batch, int seq_len, int k_heads,
                                                 int v_heads, int head_k_dim, int head_v_dim, float scale,
                                                 int beta_dtype, int l2norm_qk, const int32_t* cu_seqlens,
                                                 int n_seqs, void* stream) {
  const int64_t need = fd_gated_delta_workspace_bytes(batch, seq_len, v_heads, head_k_dim, head_v_dim,
                                                      cu_seqlens != nullptr ? n_seqs : 0);
  if (need < 0) {
    return fd_set_error(static_cast<int>(need), "fd_gated_delta_fwd_noalloc: unsupported sizes (batch %d, seq_len %d, "
                        "v_heads %d, head dims %d/%d, n_seqs %d)", batch, seq_len, v_heads, head_k_dim, head_v_dim,
                        n_seqs);
  }
  FD_REQUIRE(need <= FD_GD_SCRATCH_BYTES, FD_ERR_UNSUPPORTED,
             "fd_gated_delta_fwd_noalloc: these sizes need %lld bytes of workspace, more than the %lld-byte "
             "static scratch (call fd_gated_delta_fwd with a workspace instead)",
             static_cast<long long>(need), static_cast<long long>(FD_GD_SCRATCH_BYTES));
  void* ws = nullptr;
  const int rc = scratch_address(static_cast<hipStream_t>(stream), &ws);
  if (rc != FD_OK) return rc;
  return gd_run(q, k, v, g, beta, out, initial_state, final_state, ws, FD_GD_SCRATCH_BYTES, batch, seq_len, k_heads,
                v_heads, head_k_dim, head_v_dim, scale, beta_dtype, l2norm_qk, cu_seqlens, n_seqs, stream, nullptr);
}
