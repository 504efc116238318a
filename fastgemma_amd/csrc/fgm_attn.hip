// fgm_attn.hip -- int8-KV attention on gfx950: fgm_attend_q8_heads /
// fgm_attend_q8_row (ops.c:353-877), the transposed V store (ops.c:653-657)
// and the forward pass's KV append (forward.rs:515-548).
//
// One call is one launch for short rows (see the single-launch path below),
// else:
//  1. the scores s = ((float)(K.q) * qscale) * kscale for every (row, head,
//     slot).  The per-head int8 query (amax, 127 / amax, round to nearest even,
//     clamp +-127; ops.c:417-433); K.q is an exact int32 on the i8 matrix
//     instructions, equal to the reference's biased vpdpbusd sum minus its
//     correction.  Rows by themselves: attn_scores_kernel (heads x slots);
//     tiles of rows: attn_quant_q_kernel, then attn_scores_tile_kernel.
//  2. attn_softmax_kernel, one workgroup per (row, head): the maximum, the
//     exponentials (exp512_ps restated for the 16-wide chunks, a correctly
//     rounded exp for the n % 16 tail), the reference's summation order (16
//     lane sums in chunk order, GCC's reduce tree, the tail in order), then
//     the 16-bit weights iw = (int)fma((e * inv) * vs, 65535 / wmax, 0.5)
//     clamped to [0, 65535], written by slot as two byte planes.
//  3. the weighted sum over slots of iw v, against the transposed V cache:
//     attn_pv_kernel (rows by themselves) or attn_pv_tile_kernel;
//  4. attn_final_kernel where step 3 left partial sums or a row counts slots
//     twice: out = (float)(sum) * (wmax / 65535) (integer addition is
//     order-free, so the chunking changes nothing).
// Scores, weights and V are walked by cache slot, in the order that they lie
// in memory; only the softmax maps slots to positions.  Two byte planes hold
// a 16-bit weight exactly: with the sign bit of both bytes flipped they are
// the signed digits of iw - 32896 = 256 hi + lo, so
//   sum iw v = 256 sum hi v + sum lo v + 32896 sum v
// where the last sum is over every slot of the domain, the same for all rows
// (a slot outside a row's range has iw = 0), modulo 2^32 as the reference's
// int32 lanes.  Where a wrapped ring's two four-slot-aligned runs share a
// group (ops.c:605-631 walks each run's span in turn), its slots count twice:
// the final step adds them once more.
// Everything that is not integer arithmetic follows the reference's
// operation order, so outputs equal its bytes.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>

#include "fgm_common.h"
#include "fgm_kernels.h"

namespace {

// max over each row of 16 lanes
FGM_DEV float row16_max(float v) {
  v = __builtin_fmaxf(v, row_ror<8>(v));
  v = __builtin_fmaxf(v, row_ror<4>(v));
  v = __builtin_fmaxf(v, row_ror<2>(v));
  return __builtin_fmaxf(v, row_ror<1>(v));
}

// max over the wave, in every lane (DPP row broadcasts: no LDS round trips)
FGM_DEV float wave_max(float v) {
  v = row16_max(v);
  auto bcast = [&](auto ctrl) {
    const int i = __float_as_int(v);
    v = __builtin_fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(i, i, decltype(ctrl)::value, 0xF, 0xF, false)));
  };
  bcast(std::integral_constant<int, 0x142>{});  // lane 15 of each row to the next row
  bcast(std::integral_constant<int, 0x143>{});  // lane 31 to the upper half
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// max of three without the quieting of signalling NaNs (results of arithmetic
// are never signalling)
FGM_DEV float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// max over the workgroup; `red` holds one float per wave; every thread gets it
FGM_DEV float block_max(float v, float* red) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) red[w] = v;
  __syncthreads();
  float m = red[0];
  for (int i = 1; i < nw; i++) m = __builtin_fmaxf(m, red[i]);
  return m;
}

// One row's (or row tile's) view of its sequence: cache, attended range (of a
// tile: the union of its rows') and slot domain.
struct Geo {
  const int8_t* kc;
  const float* ks;
  const int8_t* vc;
  const float* vs;
  int k_len, ring, n;
  int s0;                           // slot of the range's first position
  int lo0, hi1;                     // slots [lo0, hi1) lie in both spans (none when lo0 >= hi1)
  int dom_lo, dom_steps, nst1, gap; // slot domain of P.V: see AttnSpan
  int r0, nr;                       // the tile's rows [r0, r0 + nr)

  __device__ int slot_of(int u) const {  // position u of the range, u < n
    const int s = s0 + u;
    return ring && s >= ring ? s - ring : s;
  }
  // u of the position held in slot s of the range, outside [0, n) if none
  __device__ int pos_of(int s) const {
    if (ring && s >= ring) return -1;
    const int u = s - s0;
    return u < 0 ? u + ring : u;
  }
  __device__ bool twice(int s) const { return s >= lo0 && s < hi1; }
  // first slot of a 64-slot step, of a group of four slots of the domain
  __device__ int dom_slot(int step) const { return dom_lo + 64 * step + (step >= nst1 ? gap : 0); }
  __device__ int dom_slot4(int qd) const { return dom_lo + 4 * qd + ((qd >> 4) >= nst1 ? gap : 0); }
  // offset of slot s in the domain
  __device__ int dom_off(int s) const {
    const int d = s - dom_lo;
    return d >= 64 * nst1 + gap ? d - gap : d;
  }
};

typedef const __attribute__((address_space(4))) AttnArgs* KernArgs;

// Index of the sequence that item x (a row or a tile) belongs to.  One
// sequence, or one row each, need no look at the table (a dependent fetch of
// the arguments less).
FGM_DEV int seq_of(const AttnArgs& a, const int* first, int x) {
  if (a.one_row) return x;
  if (a.nseq == 1) return 0;
  int i = 0;
#pragma unroll
  for (int j = 1; j < FGM_ATTN_MAX_SEQ; j++) i += x >= first[j];
  return __builtin_amdgcn_readfirstlane(i);
}

// The union of the ranges of rows [dr, dr + nr) of sequence i (a uniform
// index into the kernel argument itself).
FGM_DEV Geo seq_geo(const AttnArgs& a, int i, int dr, int nr) {
  const auto& s = ((KernArgs)__builtin_amdgcn_kernarg_segment_ptr())->seq[i];
  Geo g;
  g.kc = s.kc, g.ks = s.ks, g.vc = s.vc, g.vs = s.vs, g.k_len = s.k_len, g.ring = s.ring;
  g.r0 = s.row0 + dr, g.nr = nr;
  const int en = s.pos0 + dr + 1, st = attn_start(en, s.lo, a.window);
  // the slot of the sequence's first row's start is known: no division
  // unless the rows run past the ring
  int s0 = s.slot0 + (st - s.st0);
  if (g.ring && s0 >= g.ring) s0 = s0 < 2 * g.ring ? s0 - g.ring : s0 % g.ring;
  const AttnSpan sp = attn_span(st, en + nr - 1, g.ring, s0);
  g.n = sp.n, g.s0 = s0;
  g.lo0 = sp.lo0, g.hi1 = sp.hi1;
  g.dom_lo = sp.dom_lo, g.dom_steps = sp.dom_steps, g.nst1 = sp.nst1, g.gap = sp.gap;
  return g;
}

FGM_DEV Geo row_geo(const AttnArgs& a, int r) {
  const int i = seq_of(a, a.row0, r);
  return seq_geo(a, i, r - ((KernArgs)__builtin_amdgcn_kernarg_segment_ptr())->seq[i].row0, 1);
}

FGM_DEV Geo tile_geo(const AttnArgs& a, int t) {
  const int i = seq_of(a, a.tile0, t);
  const KernArgs ka = (KernArgs)__builtin_amdgcn_kernarg_segment_ptr();
  const int dr = (t - ka->tile0[i]) * a.rt;
  return seq_geo(a, i, dr, min(a.rt, ka->seq[i].nrows - dr));
}

// Byte address of the weights of pair (row, head) in its tile: a 64-slot step
// is [half step of 32 slots][plane hi, lo][pair][32 bytes], so that an MFMA
// operand of 32 pairs is one contiguous KB.  *plane: bytes from the hi to the
// lo plane; half steps are 2 planes apart, steps 4.
FGM_DEV int8_t* planes(const AttnArgs& a, const Geo& T, int r, int g, int hl, int* plane) {
  const int grp = a.nh / a.kvh;
  *plane = T.nr * grp * 32;
  return a.wpl + ((size_t)g * a.m + T.r0) * grp * a.cap * 128 + ((r - T.r0) * grp + hl) * 32;
}

// The reference's sum of exponentials over the 16-wide chunks, for lanes
// 0..15 of one wave (lane j: c = row j of the transposed row, e[16 t + j] at
// c[t], 16 readable floats past nt): lane j sums its column in chunk order,
// reads two groups ahead, then _mm512_reduce_add_ps on DPP row rotations.
FGM_DEV float chunk_sum16(const float* c, int nt) {
  float acc = 0.0f;
  float4 P[4], Q[4];
  auto rd = [&](float4* p, int t0) {
#pragma unroll
    for (int q = 0; q < 4; q++) p[q] = *(const float4*)(c + t0 + 4 * q);
  };
  auto add = [&](const float4* p) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      acc = acc + p[q].x;
      acc = acc + p[q].y;
      acc = acc + p[q].z;
      acc = acc + p[q].w;
    }
  };
  int t = 0;
  rd(P, 0);
  for (; t + 32 <= nt; t += 32) {
    rd(Q, t + 16);
    __builtin_amdgcn_sched_barrier(0);
    add(P);
    __builtin_amdgcn_sched_barrier(0);
    rd(P, t + 32);
    __builtin_amdgcn_sched_barrier(0);
    add(Q);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (t + 16 <= nt) {
    add(P);
    t += 16;
  }
  for (; t < nt; t++) acc = acc + c[t];
  acc = acc + row_ror<8>(acc);
  acc = acc + row_ror<4>(acc);
  acc = acc + row_ror<2>(acc);
  return acc + row_ror<1>(acc);
}

// --------------------------------------------------- 1. scores, single rows
// grid (score chunks, m * kvh), 256 threads; wave w takes the 16-slot tiles
// w, w + 4, ... of the workgroup's steps.  K is read 64 bytes a row and
// instruction, the next tile in flight while one multiplies.
template <int KS>  // head_dim / 64
__global__ __launch_bounds__(256) void attn_scores_kernel(const AttnArgs a) {
  constexpr int HD = KS * 64, QROW = HD + 16;  // padded LDS row: conflict-free fragment reads
  __shared__ __attribute__((aligned(16))) int8_t qq[16 * QROW];
  __shared__ float qsc[16];
  const int r = blockIdx.y / a.kvh, g = blockIdx.y - r * a.kvh;
  const Geo G = row_geo(a, r);
  const int d_beg = (int)blockIdx.x * 64 * a.p1_steps;
  const int d_end = min(d_beg + 64 * a.p1_steps, 64 * G.dom_steps);
  if (d_beg >= d_end) return;
  const int grp = a.nh / a.kvh;
  const int hb = max(a.h0, g * grp), he = min(a.h1, (g + 1) * grp);
  if (hb >= he) return;
  const int lane = threadIdx.x & 63, w = wave_id();

  const int kvd = a.kvh * HD;
  const __amdgpu_buffer_rsrc_t rk = make_rsrc(G.kc, (uint32_t)((size_t)G.k_len * kvd));
  const __amdgpu_buffer_rsrc_t rks = make_rsrc(G.ks, (uint32_t)G.k_len * 4u);
  float* srow = a.sc + (size_t)r * a.nh * (64 * a.cap);
  auto load = [&](v4i* B, int& kscale, int d0) {
    const int slot = G.dom_slot4(d0 >> 2) + (lane & 15);
    const uint32_t base =
        slot < G.k_len ? (uint32_t)slot * (uint32_t)kvd + (uint32_t)(g * HD + 16 * (lane >> 4)) : FGM_OOB;
#pragma unroll
    for (int kk = 0; kk < KS; kk++) B[kk] = buf_load_b128(rk, base, 64 * kk);
    kscale = buf_load_b32(rks, slot < G.k_len ? 4u * (uint32_t)slot : FGM_OOB, 0);
  };
  v4i B0[KS], B1[KS];
  int ks0 = 0, ks1 = 0;
  int d0 = d_beg + 16 * w;
  if (d0 < d_end) load(B0, ks0, d0);
  if (d0 + 64 < d_end) load(B1, ks1, d0 + 64);

  // per-head int8 query, one wave per head row; rows past the group are zero
  for (int hl = w; hl < 16; hl += 4) {
    const int h = g * grp + hl;
    const bool live = hl < grp && h >= hb && h < he;
    float x[KS];
    float amax = 0.0f;
#pragma unroll
    for (int kk = 0; kk < KS; kk++) {
      x[kk] = live ? a.q[((size_t)r * a.nh + h) * HD + 64 * kk + lane] : 0.0f;
      amax = __builtin_fmaxf(amax, __builtin_fabsf(x[kk]));
    }
    amax = wave_max(amax);
    const float qinv = amax > 0.0f ? 127.0f / amax : 0.0f;
#pragma unroll
    for (int kk = 0; kk < KS; kk++) {
      const float v = __builtin_amdgcn_fmed3f(__builtin_rintf(x[kk] * qinv), -127.0f, 127.0f);
      qq[hl * QROW + 64 * kk + lane] = (int8_t)(int)v;
    }
    if (lane == 0) qsc[hl] = amax / 127.0f;
  }
  __syncthreads();

  // A: lane row lane % 16 (head), bytes 16 (lane / 16) .. of each 64-dim step
  v4i A[KS];
#pragma unroll
  for (int kk = 0; kk < KS; kk++)
    A[kk] = *(const v4i*)(qq + (lane & 15) * QROW + 64 * kk + 16 * (lane >> 4));
  auto tile = [&](const v4i* B, int kscale, int d) {
    v4i acc = {0, 0, 0, 0};
#pragma unroll
    for (int kk = 0; kk < KS; kk++) acc = mfma16(A[kk], B[kk], acc);
    // D: lane, register i -> head row 4 (lane / 16) + i, slot lane % 16
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int hl = 4 * (lane >> 4) + i, h = g * grp + hl;
      if (hl < grp && h >= hb && h < he)
        srow[(size_t)h * (64 * a.cap) + d + (lane & 15)] = ((float)acc[i] * qsc[hl]) * __int_as_float(kscale);
    }
  };
  for (; d0 < d_end; d0 += 128) {
    tile(B0, ks0, d0);
    if (d0 + 64 >= d_end) break;
    if (d0 + 128 < d_end) load(B0, ks0, d0 + 128);
    tile(B1, ks1, d0 + 64);
    if (d0 + 192 < d_end) load(B1, ks1, d0 + 192);
  }
}

// ---------------------------------------------------- 1. scores, row tiles
// The int8 query of every (row, head), one wave each: into the partial sums'
// place (free until P.V), its scale into wq's (free until the softmax).
__global__ __launch_bounds__(256) void attn_quant_q_kernel(const float* q, int8_t* q8, float* qsc, int count, int hd) {
  const int lane = threadIdx.x & 63, i = blockIdx.x * 4 + wave_id();
  if (i >= count) return;
  float x[8];
  float amax = 0.0f;
#pragma unroll
  for (int kk = 0; kk < 8; kk++) {
    x[kk] = 64 * kk < hd ? q[(size_t)i * hd + 64 * kk + lane] : 0.0f;
    amax = __builtin_fmaxf(amax, __builtin_fabsf(x[kk]));
  }
  amax = wave_max(amax);
  const float qinv = amax > 0.0f ? 127.0f / amax : 0.0f;
#pragma unroll
  for (int kk = 0; kk < 8; kk++) {
    const float v = __builtin_amdgcn_fmed3f(__builtin_rintf(x[kk] * qinv), -127.0f, 127.0f);
    if (64 * kk < hd) q8[(size_t)i * hd + 64 * kk + lane] = (int8_t)(int)v;
  }
  if (lane == 0) qsc[i] = amax / 127.0f;
}

typedef int v16i __attribute__((ext_vector_type(16)));

// grid (score chunks, ntiles * kvh), 256 threads: the 128 (row, head) pairs of
// a tile x the slots of p1_steps steps on v_mfma_i32_32x32x32_i8, wave w the
// pairs 32 w ...  A wave keeps its queries (32 x hd bytes) in registers; K
// goes through LDS in stages of 32 slots, a ring of three filled by 1 KB
// LDS-DMA units (two stages ahead), so the four waves share each byte of K
// and a row's K is read once per tile instead of once per row.  LDS rows are
// hd bytes; their 16-byte chunks are permuted (chunk ^ slot % 8 inside each
// 128-byte line, by the DMA's source address), so that the fragment reads hit
// every bank.  Bound by the scores' stores (67 MB at 256 rows x 8 heads x 8192
// positions, head_dim 512: 129 us with every row reading K for itself, 21 us
// as tiles, beside 4.5 us for the queries).
template <int KS>
__global__ __launch_bounds__(256, 2) void attn_scores_tile_kernel(const AttnArgs a) {
  constexpr int HD = KS * 64, SWZ = KS % 2 ? 3 : 7;
  constexpr int UPW = (2 * KS + 3) / 4, STAGE = UPW * 4096, NSTORE = 16;
  constexpr int MAXP = 8;  // steps per workgroup, at most
  __shared__ __attribute__((aligned(1024))) int8_t ring[3 * STAGE];
  __shared__ float ksl[64 * MAXP];
  const int t = blockIdx.y / a.kvh, g = blockIdx.y - t * a.kvh;
  const Geo T = tile_geo(a, t);
  const int step0 = (int)blockIdx.x * a.p1_steps, nsteps = min(a.p1_steps, T.dom_steps - step0);
  if (nsteps <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
  const int grp = a.nh / a.kvh, pairs = T.nr * grp;
  const int kvd = a.kvh * HD;
  const v4i rk = rsrc_words(T.kc, (uint32_t)((size_t)T.k_len * kvd));
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) int8_t*)ring;
  // DMA unit 4 j + w of a stage: 64 chunks from chunk 64 (4 j + w) of the
  // stage's LDS image on; the lane's chunk there is chunk p of slot sl
  uint32_t src[UPW];
#pragma unroll
  for (int j = 0; j < UPW; j++) {
    const int c = 64 * (4 * j + w) + lane, sl = c / (4 * KS), p = c - sl * (4 * KS);
    src[j] = (uint32_t)sl * (uint32_t)kvd + (uint32_t)(g * HD + 16 * (p ^ (sl & SWZ)));
    if (sl >= 32) src[j] = FGM_OOB;
  }
  const int nst = 2 * nsteps;
  auto issue = [&](int s) {
    const uint32_t at = (uint32_t)(T.dom_slot(step0 + (s >> 1)) + 32 * (s & 1)) * (uint32_t)kvd;
    const uint32_t to = lds0 + (uint32_t)(s % 3) * STAGE + 1024u * w;
#pragma unroll
    for (int j = 0; j < UPW; j++) dma16(rk, to + 4096u * j, src[j] == FGM_OOB ? FGM_OOB : src[j] + at, 0);
  };
  issue(0);
  issue(1);
  // the wave's queries: lane row lane % 32, bytes 32 kk + 16 (lane / 32) ...
  const int c32 = lane & 31, half = lane >> 5;
  auto pair_row = [&](int mr) {  // (row, head) index of pair mr of the tile
    const int rr = mr / grp;
    return (T.r0 + rr) * a.nh + g * grp + (mr - rr * grp);
  };
  const int8_t* q8 = (const int8_t*)a.part;
  const int mine = min(32 * w + c32, pairs - 1);
  const int8_t* qp = q8 + (size_t)pair_row(mine) * HD + 16 * half;
  v4i A[2 * KS];
#pragma unroll
  for (int kk = 0; kk < 2 * KS; kk++) A[kk] = *(const v4i*)(qp + 32 * kk);
  // D: register i of a lane is pair 32 w + 8 (i / 4) + 4 half + i % 4, slot c32
  float qs[16];
  int prow[16];
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int mr = min(32 * w + 8 * (i >> 2) + 4 * half + (i & 3), pairs - 1);
    prow[i] = pair_row(mr);
    qs[i] = a.wq[prow[i]];
  }
  for (int i = tid; i < 64 * nsteps; i += 256) {
    const int slot = T.dom_slot4((64 * step0 + i) >> 2) + (i & 3);
    ksl[i] = slot < T.k_len ? T.ks[slot] : 0.0f;
  }
  const bool full = 32 * w + 32 <= pairs, some = 32 * w < pairs;
  const size_t stride = (size_t)64 * a.cap;
  // LDS addresses of the four chunk pairs of a 128-byte line
  int fr[4];
#pragma unroll
  for (int j = 0; j < 4; j++) fr[j] = c32 * HD + 16 * (((2 * j) ^ half) ^ (c32 & SWZ));
  wait_vm<0>();
  for (int s = 0; s < nst; s++) {
    // Stage s was requested two stages ago; since then the wave has issued
    // stage s + 1 (UPW loads) and, when all its pairs exist, the 16 stores of
    // stages s - 2 and s - 1 each.  Stages 0 and 1 are already here.
    if (s >= 2) {
      if (!full) wait_vm<0>();
      else if (s + 1 < nst) wait_vm<2 * NSTORE + UPW>();
      else wait_vm<2 * NSTORE>();
    }
    __syncthreads();
    if (s + 2 < nst) issue(s + 2);
    if (!some) continue;
    const int8_t* img = ring + (s % 3) * STAGE;
    v16i acc = {};
#pragma unroll
    for (int kk = 0; kk < 2 * KS; kk++) {
      const v4i b = *(const v4i*)(img + fr[kk & 3] + 128 * (kk >> 2));
      acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[kk], b, acc, 0, 0, 0);
    }
    const float ksc = ksl[32 * s + c32];
    float* to = a.sc + 64 * step0 + 32 * s + c32;
    if (full) {
#pragma unroll
      for (int i = 0; i < 16; i++) to[(size_t)prow[i] * stride] = ((float)acc[i] * qs[i]) * ksc;
    } else {
#pragma unroll
      for (int i = 0; i < 16; i++)
        if (32 * w + 8 * (i >> 2) + 4 * half + (i & 3) < pairs)
          to[(size_t)prow[i] * stride] = ((float)acc[i] * qs[i]) * ksc;
    }
  }
}

// ---------------------------------------------------- 2. softmax, weights
// grid (m * (h1 - h0)), T threads.  A thread owns NQ groups of four slots,
// tid + T j, from the load of their scores to the store of their weights: all
// loads are in flight at once, and only the exponentials go through LDS, for
// the ordered sum: e[16 c + j] at lds[j * S + c] (S = 4 mod 64, >= n / 16 +
// 16), then the reduction slots.  A few rows are one dependent chain (8 rows x
// 8 heads x 8192 positions: 15.2 us walking LDS, 9.5 us from registers); many
// wait for their own barriers, loads and ordered sum about half the time
// (2048 pairs x 8192: 72 us walking LDS, 42 us from registers with three
// workgroups per CU and 54 VALU instructions a slot; 35 us with four, the V
// scales loaded after the exponentials, and fewer instructions).  Four leave 64
// registers, of which NQ = 4 is 13 short and NQ = 3 three: 56 and 16 bytes of
// scratch a lane.
// The row stride of the transposed exponentials, for the kernels and for the
// LDS that their launches ask for.
__host__ __device__ inline int exp_stride(int n) { return (((n + 15) >> 4) + 16 + 63) / 64 * 64 + 4; }

template <int NQ, int T_>  // up to 512 threads, NQ <= 4: 32 waves per CU (64 registers)
__global__ __launch_bounds__(T_, T_ <= 512 && NQ <= 4 ? 8 : 4) void attn_softmax_kernel(const AttnArgs a) {
  extern __shared__ float lds[];
  const int nhr = a.h1 - a.h0;
  // consecutive (row, head) pairs on one XCD: they share lines of the weights
  int b = blockIdx.x;
  if ((gridDim.x & 7) == 0) b = (b & 7) * (gridDim.x >> 3) + (b >> 3);
  const int r = b / nhr, h = a.h0 + (b - r * nhr);
  const int grp = a.nh / a.kvh, g = h / grp, hl = h - g * grp;
  const int si = seq_of(a, a.row0, r);
  const KernArgs ka = (KernArgs)__builtin_amdgcn_kernarg_segment_ptr();
  const int dr = r - ka->seq[si].row0;
  const Geo G = seq_geo(a, si, dr, 1);
  Geo T = G;  // the domain: the row tile's
  if (a.rt > 1) {
    const int t0 = dr / a.rt * a.rt;
    T = seq_geo(a, si, t0, min(a.rt, ka->seq[si].nrows - t0));
  }
  const int tid = threadIdx.x, lane = tid & 63, nt = blockDim.x, nw = nt >> 6, w = wave_id();
  const int n = max(G.n, 0), n16 = n & ~15, S = exp_stride(n);
  float* red = lds + 16 * S;
  const float* scr = a.sc + ((size_t)r * a.nh + h) * (64 * a.cap);
  const __amdgpu_buffer_rsrc_t rvs = make_rsrc(G.vs, (uint32_t)G.k_len * 4u);
  const int nq = 16 * T.dom_steps;

  // A wave's 64 groups j are 256 consecutive domain offsets.  Where all of
  // them hold positions of the row before its n % 16 tail (uc: the chunk of 16
  // of the first; it starts at r0 % 16, the same for all j that count here),
  // nothing has to be masked, and an LDS index is one addition.  Elsewhere,
  // slots outside the range take part in nothing: their score is -inf, their
  // V scale and so their weight 0, and their exponential goes to a place that
  // nobody reads.
  const int DUMP = 16 * S + 24;
  float e[NQ][4];
  int vs[NQ][4], uc[NQ], r0 = -1;
#pragma unroll
  for (int j = 0; j < NQ; j++) {
    const int q0 = 64 * w + nt * j, f = T.dom_slot4(q0), l = T.dom_slot4(q0 + 63) + 3;
    const int uf = G.pos_of(f), ul = G.pos_of(l);
    const bool full = l - f == 255 && q0 + 64 <= nq && uf >= 0 && ul == uf + 255 && ul < n16 &&
                      (r0 < 0 || r0 == (uf & 15));
    if (full) r0 = uf & 15;
    uc[j] = full ? uf >> 4 : -1;
    const int qd = tid + nt * j, s4 = T.dom_slot4(qd);
    if (full) {
      const float4 v = *(const float4*)(scr + 4 * qd);
      e[j][0] = v.x, e[j][1] = v.y, e[j][2] = v.z, e[j][3] = v.w;
    } else {
      float4 v = {0, 0, 0, 0};
      if (qd < nq) v = *(const float4*)(scr + 4 * qd);
      e[j][0] = v.x, e[j][1] = v.y, e[j][2] = v.z, e[j][3] = v.w;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const bool ok = qd < nq && (unsigned)G.pos_of(s4 + i) < (unsigned)n;
        e[j][i] = ok ? e[j][i] : -INFINITY;
      }
    }
  }
  float mx = -INFINITY;
#pragma unroll
  for (int j = 0; j < NQ; j++) mx = max3(max3(mx, e[j][0], e[j][1]), e[j][2], e[j][3]);
  mx = block_max(mx, red);
  // LDS indices of the groups' slots from the first full chunk on
  int at0[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int u = r0 + 4 * lane + i;
    at0[i] = (u & 15) * S + (u >> 4);
  }
  uint64_t tl = 0;  // this thread's slots in the tail
#pragma unroll
  for (int j = 0; j < NQ; j++) {
    if (uc[j] >= 0) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        e[j][i] = exp16(e[j][i] - mx);
        lds[at0[i] + uc[j]] = e[j][i];
      }
      const v4i x = buf_load_b128(rvs, 4u * (uint32_t)T.dom_slot4(tid + nt * j), 0);
#pragma unroll
      for (int i = 0; i < 4; i++) vs[j][i] = x[i];
    } else {
      const int qd = tid + nt * j, s4 = T.dom_slot4(qd);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int u = G.pos_of(s4 + i);
        const float x = e[j][i] - mx;
        const bool ok = qd < nq && (unsigned)u < (unsigned)n;
        const int at = ok ? (u & 15) * S + (u >> 4) : DUMP;
        vs[j][i] = buf_load_b32(rvs, ok ? 4u * (uint32_t)(s4 + i) : FGM_OOB, 0);
        e[j][i] = exp16(x);
        // the tail: shifted scores, for lanes 0..15 to exponentiate
        const bool t = ok && u >= n16;
        lds[at] = t ? x : e[j][i];
        tl |= (uint64_t)t << (4 * j + i);
      }
    }
  }
  __syncthreads();
  if (tid < 16) {
    float t = 0.0f;
    if (n16 + tid < n) t = (float)exp((double)lds[tid * S + (n16 >> 4)]);
    float sum = chunk_sum16(lds + tid * S, n16 >> 4);
    for (int u = 0; u < n - n16; u++) sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t), u));
    if (n16 + tid < n) lds[tid * S + (n16 >> 4)] = t;
    if (tid == 0) red[nw] = 1.0f / sum;
  }
  __syncthreads();
  const float inv = red[nw];
  if (tl) {
#pragma unroll
    for (int j = 0; j < NQ; j++)
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (tl >> (4 * j + i) & 1)
          e[j][i] = lds[(G.pos_of(T.dom_slot4(tid + nt * j) + i) & 15) * S + (n16 >> 4)];
  }
  // weights (e * inv) * vs (the V scales in flight since the exponentials),
  // and their maximum
  float wm = 0.0f;
#pragma unroll
  for (int j = 0; j < NQ; j++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      e[j][i] = (e[j][i] * inv) * __int_as_float(vs[j][i]);
      if (i & 1) wm = max3(wm, e[j][i - 1], e[j][i]);
    }
  wm = block_max(wm, red);
  const bool some = wm > 0.0f;
  const float wq_inv = some ? 65535.0f / wm : 0.0f;
  int plane;
  int8_t* wp = planes(a, T, r, g, hl, &plane);
  wp += (size_t)(tid >> 3) * (2 * plane) + 4 * (tid & 7);
#pragma unroll
  for (int j = 0; j < NQ; j++) {
    if (tid + nt * j >= nq) continue;
    uint32_t q[4];
#pragma unroll
    for (int i = 0; i < 4; i++)  // an empty row's weights are NaN: 0 too
      q[i] = (uint32_t)min(max((int)__builtin_fmaf(e[j][i], wq_inv, 0.5f), 0), 65535);
    // the bytes of the four weights, high and low, with flipped sign bits
    const uint32_t q01 = q[0] | q[1] << 16, q23 = q[2] | q[3] << 16;
    int8_t* p = wp + (size_t)(nt >> 3) * (2 * plane) * j;
    *(uint32_t*)p = __builtin_amdgcn_perm(q23, q01, 0x07050301u) ^ 0x80808080u;
    *(uint32_t*)(p + plane) = __builtin_amdgcn_perm(q23, q01, 0x06040200u) ^ 0x80808080u;
  }
  if (tid == 0) a.wq[r * a.nh + h] = some ? wm / 65535.0f : 0.0f;
}

// ------------------------------------------------------------------ 3. P.V
constexpr uint32_t IW_BIAS = 32896u;  // 256 * 128 + 128: see the planes above

constexpr int ONES = 0x01010101;
FGM_DEV int dot4(int x, int y, int c) { return __builtin_amdgcn_sdot4(x, y, c, false); }

// Single rows.  grid (hd / (16 DPL), m * kvh, p3_chunks), 64 NW threads:
// workgroup (x, y, z) takes the dims [16 DPL x, + 16 DPL) and the steps
// [p3_steps z, + p3_steps) of the row's domain, wave w the steps w, w + NW,
// ...; lane (c, q4) loads the 4 DPL bytes [DPL dims][4 slots] of dims DPL c ..
// and slot groups 4 q4 + r, r = 0..3: register q of the four loads is one MFMA
// B operand (column c = dim DPL c + q).  The A operand's rows are the heads'
// hi planes (0..7) and lo planes (8..15), with more than eight heads one
// operand each.  PF steps are in flight, without branches around the loads
// (past the last step they read nothing), so that the waits count them.
// Sixteen waves so that one workgroup covers all of K where 256 or more run:
// the sums stay in the workgroup and need no further launch.  DPL = 1 (64-byte
// pieces of V's lines; consecutive workgroups, which share them, go to one
// XCD) where 32-dim workgroups would leave CUs idle.  8 rows x 8192 slots at
// head_dim 512: 14.7 us and 4.9 us for the partial sums' launch with 4-byte
// loads in 2048 workgroups, 12.4 us as 128 workgroups of 32 dims with a branch
// around each load, 2.2 us less so (the whole call 36.3 -> 34.0 us; 37.0 with
// 128 workgroups and no branches, eight steps in flight as four).
template <bool TWO, int DPL>  // TWO: more than eight heads
__global__ __launch_bounds__(TWO ? 512 : 1024) void attn_pv_kernel(const AttnArgs a) {
  constexpr int NW = TWO ? 8 : 16, ND = 16 * DPL, PF = 4;
  __shared__ __attribute__((aligned(16))) int32_t red[NW][17][ND];
  const int nx = gridDim.x, total = nx * gridDim.y;
  int id = blockIdx.x + nx * blockIdx.y;
  if ((total & 7) == 0) id = (id & 7) * (total >> 3) + (id >> 3);
  const int rg = id / nx, r = rg / a.kvh, g = rg - r * a.kvh;
  const Geo G = row_geo(a, r);
  const int grp = a.nh / a.kvh;
  const int hb = max(a.h0, g * grp), he = min(a.h1, (g + 1) * grp);
  if (hb >= he) return;
  const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
  const int kvd = a.kvh * a.hd, d0 = ND * (id - rg * nx);
  const int c16 = lane & 15, q4 = lane >> 4;
  const int first = (int)blockIdx.z * a.p3_steps, last = min(first + a.p3_steps, G.dom_steps);
  int plane;
  const int8_t* wp = planes(a, G, r, g, 0, &plane);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(wp, (uint32_t)(4 * plane) * (uint32_t)G.dom_steps);
  const int hl = TWO ? c16 : c16 & 7;
  const uint32_t wat = (uint32_t)(32 * hl + (TWO ? 0 : plane * (c16 >> 3)) + (q4 >> 1) * 2 * plane + 16 * (q4 & 1));
  const __amdgpu_buffer_rsrc_t rv = make_rsrc(G.vc, (uint32_t)((size_t)((G.k_len + 3) >> 2) * kvd * 4));
  const uint32_t vat = ((uint32_t)(4 * q4) * (uint32_t)kvd + (uint32_t)(g * a.hd + d0 + DPL * c16)) * 4u;
  v4i D0[DPL], D1[DPL];
  int sv[DPL];
#pragma unroll
  for (int q = 0; q < DPL; q++) D0[q] = D1[q] = v4i{0, 0, 0, 0}, sv[q] = 0;
  v4i A[PF][TWO ? 2 : 1];
  int V[PF][4][DPL];
  auto load = [&](int i, int step) {
    const bool ok = step < last;
    const uint32_t wo = ok && hl < grp ? wat + (uint32_t)step * (uint32_t)(4 * plane) : FGM_OOB;
    const uint32_t vo = ok ? vat + (uint32_t)(G.dom_slot(step) >> 2) * (uint32_t)(kvd * 4) : FGM_OOB;
    A[i][0] = buf_load_b128(rw, wo, 0);
    if constexpr (TWO) A[i][1] = buf_load_b128(rw, wo + (uint32_t)plane, 0);
#pragma unroll
    for (int rr = 0; rr < 4; rr++) {
      if constexpr (DPL == 1) {
        V[i][rr][0] = buf_load_b32(rv, vo + (uint32_t)(rr * kvd * 4), 0);
      } else {
        const v2i x = buf_load_b64(rv, vo + (uint32_t)(rr * kvd * 4), 0);
        V[i][rr][0] = x[0], V[i][rr][DPL - 1] = x[1];
      }
    }
  };
  auto mul = [&](int i, int step) {
    const int ones = step < last ? ONES : 0;
#pragma unroll
    for (int q = 0; q < DPL; q++) {
      const v4i b = {V[i][0][q], V[i][1][q], V[i][2][q], V[i][3][q]};
      D0[q] = mfma16(A[i][0], b, D0[q]);
      if constexpr (TWO) D1[q] = mfma16(A[i][TWO ? 1 : 0], b, D1[q]);
#pragma unroll
      for (int rr = 0; rr < 4; rr++) sv[q] = dot4(b[rr], ones, sv[q]);
    }
  };
#pragma unroll
  for (int i = 0; i < PF; i++) load(i, first + w + NW * i);
#pragma unroll 1
  for (int step = first + w; step < last; step += PF * NW) {
#pragma unroll
    for (int i = 0; i < PF; i++) {
      mul(i, step + i * NW);
      load(i, step + (PF + i) * NW);
    }
  }
#pragma unroll
  for (int q = 0; q < DPL; q++) {
    sv[q] += __shfl_xor(sv[q], 16, 64);
    sv[q] += __shfl_xor(sv[q], 32, 64);
  }
  // rows 0..15: heads' sums 256 hi (+ lo), or hi and lo of eight; row 16: sum v
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int row = 4 * q4 + i;
#pragma unroll
    for (int q = 0; q < DPL; q++)
      red[w][row][DPL * c16 + q] = TWO ? (int)(((uint32_t)D0[q][i] << 8) + (uint32_t)D1[q][i])
                                       : (int)(row < 8 ? (uint32_t)D0[q][i] << 8 : (uint32_t)D0[q][i]);
  }
#pragma unroll
  for (int q = 0; q < DPL; q++)
    if (q4 == 0) red[w][16][DPL * c16 + q] = sv[q];
  __syncthreads();
  for (int idx = tid; idx < grp * ND; idx += 64 * NW) {
    const int hr = idx / ND, d = idx % ND, h = g * grp + hr;
    if (h < hb || h >= he) continue;
    uint32_t t = 0;
#pragma unroll 4
    for (int i = 0; i < NW; i++)
      t += (uint32_t)red[i][hr][d] + (TWO ? 0u : (uint32_t)red[i][8 + hr][d]) + IW_BIAS * (uint32_t)red[i][16][d];
    const size_t row = (size_t)r * a.nh + h;
    if (a.p3_chunks == 1 && !a.dup)
      a.out[row * a.hd + d0 + d] = (float)(int32_t)t * a.wq[row];
    else
      a.part[(row * a.p3_chunks + blockIdx.z) * a.hd + d0 + d] = (int32_t)t;
  }
}

// Row tiles.  grid (hd / 256 rounded up, ntiles * kvh, p3_chunks), 64 * 4 NG
// threads (NG = 2, or 1 for head_dim <= 128): the 128 pairs of a tile x 128 NG
// dims x the chunk's steps on v_mfma_i32_32x32x32_i8.  Wave (mg, ng) takes
// the pairs 32 mg ... and the dims 128 ng ..., with both planes' sums in
// registers.  Half steps of 32 slots go through LDS, a ring of NS filled by
// 1 KB LDS-DMA units: the planes of 32 pairs each, and V's rows of eight slot
// groups.  A fragments are 16 bytes of a pair's 32, B fragments the 16 bytes
// [4 dims][4 slots] of a group, as above (column c = dim 4 c + q).  sum v: wave
// mg adds up the half steps mg, mg + 4, ...
// 256 rows x 8 heads x 8192 slots at head_dim 512: 93 us with every row
// reading V for itself and three 7-bit planes; 40 us as tiles with the
// operands loaded from L1 to registers (48 KB a half step and CU, 768 cycles
// of L1 under 512 of the matrix cores), 37 us through LDS, both in four chunks
// (128 workgroups); 28.5 us in eight.
template <int NG>
__global__ __launch_bounds__(256 * NG, 2) void attn_pv_tile_kernel(const AttnArgs a) {
  constexpr int NW = 4 * NG, UNITS = 8 + 4 * NG, UPW = UNITS / NW, NS = 5, STAGE = UNITS * 1024;
  static_assert(UPW * NW == UNITS, "units per wave");
  __shared__ __attribute__((aligned(1024))) int8_t ring[NS * STAGE];
  __shared__ __attribute__((aligned(16))) int svl[NG][4][32][4];
  const int t = blockIdx.y / a.kvh, g = blockIdx.y - t * a.kvh;
  const Geo T = tile_geo(a, t);
  const int lane = threadIdx.x & 63, w = wave_id(), mg = w & 3, ng = w >> 2;
  const int grp = a.nh / a.kvh, pairs = T.nr * grp;
  const int kvd = a.kvh * a.hd, dwg = (int)blockIdx.x * 128 * NG, d0 = dwg + 128 * ng;
  const int c32 = lane & 31, half = lane >> 5;
  const int first = 2 * (int)blockIdx.z * a.p3_steps, last = min(first + 2 * a.p3_steps, 2 * T.dom_steps);
  int plane;
  const int8_t* wp = planes(a, T, T.r0, g, 0, &plane);
  const v4i rw = rsrc_words(wp, (uint32_t)plane * 4u * (uint32_t)T.dom_steps);
  const v4i rv = rsrc_words(T.vc, (uint32_t)((size_t)((T.k_len + 3) >> 2) * kvd * 4));
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) int8_t*)ring;
  // DMA unit u = w + NW i of a half step: planes (u / 4) of the pairs 32 (u %
  // 4) ... (past the tile's pairs: zeros), or V group rows, NG a unit
  uint32_t src[UPW];
#pragma unroll
  for (int i = 0; i < UPW; i++) {
    const int u = w + NW * i;
    if (u < 8) {
      const int o = (u & 3) * 1024 + 16 * lane;
      src[i] = o < plane ? (uint32_t)((u >> 2) * plane + o) : FGM_OOB;
    } else {
      const int row = NG == 2 ? u - 8 : 2 * (u - 8) + half, o = NG == 2 ? 16 * lane : 16 * c32;
      src[i] = ((uint32_t)row * (uint32_t)kvd + (uint32_t)(g * a.hd + dwg)) * 4u + (uint32_t)o;
    }
  }
  auto issue = [&](int hs, int slot) {
    const uint32_t gi = (uint32_t)(T.dom_slot(hs >> 1) >> 2) + 8u * (hs & 1);
    const uint32_t av = gi * (uint32_t)kvd * 4u, aw = (uint32_t)hs * 2u * (uint32_t)plane;
    const uint32_t to = lds0 + (uint32_t)slot * STAGE + 1024u * w;
#pragma unroll
    for (int i = 0; i < UPW; i++) {
      if (w + NW * i < 8)
        dma16(rw, to + 1024u * NW * i, src[i] == FGM_OOB ? FGM_OOB : src[i] + aw, 0);
      else
        dma16(rv, to + 1024u * NW * i, src[i] + av, 0);
    }
  };
  v16i H[4], L[4];
  int sv[4] = {0, 0, 0, 0};
#pragma unroll
  for (int q = 0; q < 4; q++) H[q] = L[q] = v16i{};
  const int8_t* fa = ring + mg * 1024 + 32 * c32 + 16 * half;
  const int8_t* fb = ring + 8192 + (NG * 512) * 4 * half + 512 * ng + 16 * c32;
  auto mul = [&](int hs, int slot) {
    const v4i A0 = *(const v4i*)(fa + slot * STAGE), A1 = *(const v4i*)(fa + slot * STAGE + 4096);
    v4i V[4];
#pragma unroll
    for (int rr = 0; rr < 4; rr++) V[rr] = *(const v4i*)(fb + slot * STAGE + NG * 512 * rr);
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const v4i b = {V[0][q], V[1][q], V[2][q], V[3][q]};
      H[q] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A0, b, H[q], 0, 0, 0);
      L[q] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A1, b, L[q], 0, 0, 0);
    }
    if ((hs & 3) == mg) {
#pragma unroll
      for (int q = 0; q < 4; q++)
#pragma unroll
        for (int rr = 0; rr < 4; rr++) sv[q] = dot4(V[rr][q], ONES, sv[q]);
    }
  };
#pragma unroll
  for (int i = 0; i < NS - 1; i++)
    if (first + i < last) issue(first + i, i);
  // Half step hs is in slot (hs - first) % NS.  When its turn comes, the wave
  // has issued at most NS - 2 later ones; the barrier then shows every wave's
  // part, and that all are done with half step hs - 1, whose slot is refilled.
  int hs = first;
#pragma unroll 1
  while (hs < last) {
#pragma unroll
    for (int i = 0; i < NS; i++) {
      if (hs < last) {
        if (hs + NS - 2 < last) wait_vm<(NS - 2) * UPW>();
        else wait_vm<0>();
        __syncthreads();
        if (hs + NS - 1 < last) issue(hs + NS - 1, (i + NS - 1) % NS);
        mul(hs, i);
      }
      hs++;
    }
  }
#pragma unroll
  for (int q = 0; q < 4; q++) sv[q] += __shfl_xor(sv[q], 32, 64);
  if (half == 0) *(v4i*)svl[ng][mg][c32] = v4i{sv[0], sv[1], sv[2], sv[3]};
  __syncthreads();
  if (d0 + 4 * c32 >= a.hd) return;
  v4i bias;
#pragma unroll
  for (int q = 0; q < 4; q++)
    bias[q] = (int)(IW_BIAS * ((uint32_t)svl[ng][0][c32][q] + (uint32_t)svl[ng][1][c32][q] +
                               (uint32_t)svl[ng][2][c32][q] + (uint32_t)svl[ng][3][c32][q]));
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int mr = 32 * mg + 8 * (i >> 2) + 4 * half + (i & 3);
    if (mr >= pairs) continue;
    const int rr = mr / grp, h = g * grp + (mr - rr * grp);
    if (h < a.h0 || h >= a.h1) continue;
    const size_t row = (size_t)(T.r0 + rr) * a.nh + h;
    v4i v;
#pragma unroll
    for (int q = 0; q < 4; q++)
      v[q] = (int)(((uint32_t)H[q][i] << 8) + (uint32_t)L[q][i] + (uint32_t)bias[q]);
    if (a.p3_chunks == 1 && !a.dup) {
      const float s = a.wq[row];
      float* o = a.out + row * a.hd + d0 + 4 * c32;
#pragma unroll
      for (int q = 0; q < 4; q++) o[q] = (float)v[q] * s;
    } else {
      *(v4i*)(a.part + (row * a.p3_chunks + blockIdx.z) * a.hd + d0 + 4 * c32) = v;
    }
  }
}

// ---------------------------------------------------------------- 4. final
// grid (m * (h1 - h0)), hd / 4 threads (a multiple of 16), four dims each: the
// chunks' partial sums, plus once more the slots that the row counts twice.
__global__ __launch_bounds__(128) void attn_final_kernel(const AttnArgs a) {
  const int nhr = a.h1 - a.h0;
  const int r = blockIdx.x / nhr, h = a.h0 + ((int)blockIdx.x - r * nhr);
  const int d = 4 * threadIdx.x;
  const size_t row = (size_t)r * a.nh + h;
  const int32_t* part = a.part + row * a.p3_chunks * a.hd + d;
  uint32_t t[4] = {0, 0, 0, 0};
#pragma unroll 4
  for (int c = 0; c < a.p3_chunks; c++) {
    const v4i v = *(const v4i*)(part + (size_t)c * a.hd);
#pragma unroll
    for (int q = 0; q < 4; q++) t[q] += (uint32_t)v[q];
  }
  if (a.dup) {
    const int grp = a.nh / a.kvh, g = h / grp, hl = h - g * grp;
    const int si = seq_of(a, a.row0, r);
    const KernArgs ka = (KernArgs)__builtin_amdgcn_kernarg_segment_ptr();
    const int dr = r - ka->seq[si].row0;
    const Geo G = seq_geo(a, si, dr, 1);
    const int t0 = dr / a.rt * a.rt;
    const Geo T = seq_geo(a, si, t0, min(a.rt, ka->seq[si].nrows - t0));
    int plane;
    const int8_t* wp = planes(a, T, r, g, hl, &plane);
    const int kvd = a.kvh * a.hd;
    for (int s = G.lo0; s < min(G.hi1, G.ring); s++) {
      const int o = T.dom_off(s);
      const int8_t* p = wp + (size_t)(o >> 5) * (2 * plane) + (o & 31);
      const uint32_t iw = 256u * (uint8_t)(p[0] ^ 0x80) + (uint8_t)(p[plane] ^ 0x80);
      const int8_t* v = G.vc + ((size_t)(s >> 2) * kvd + g * a.hd + d) * 4 + (s & 3);
#pragma unroll
      for (int q = 0; q < 4; q++) t[q] += iw * (uint32_t)(int32_t)v[4 * q];
    }
  }
  float* o = a.out + row * a.hd + d;
  const float s = a.wq[row];
#pragma unroll
  for (int q = 0; q < 4; q++) o[q] = (float)(int32_t)t[q] * s;
}

// ------------------------------------------------------ single-launch path
// Rows of at most FUSED_MAX_N positions and kv groups of at most 8 query
// heads: one workgroup per (row, kv head, hpw of its query heads) does all
// four steps above with the same arithmetic, the scores, exponentials and
// weight planes in LDS and the P.V sums in registers -- one launch instead of
// four (sliding-window layers, short contexts).  A launch of a few rows is one
// dependent chain (arguments, K, softmax, P.V, each a few hundred
// instructions, fetched cold), so its heads are dealt to separate workgroups
// until they fill the chip (each reads the K and V of its kv head again, from
// the L2 of its XCD), and the softmax runs one position per lane in loops that
// are not unrolled.  8 rows x 8 heads x 512 positions at head_dim 256: 22.8 us
// with the eight heads in one workgroup of eight waves, 11.4 us split and
// walked this way; 256 rows (every head in one workgroup of sixteen waves)
// 22.2 -> 15.0 us.  Of the 11.4, 2.2 us pass before the wait for the first
// K and query bytes ends, 2 us more in that wait.  grid (HS, m * kvh) flattened with the row fastest (the
// workgroups of one row land on one XCD when the rows are a multiple of 8);
// 64 NW threads; dynamic LDS:
//   qq [16][hd + 16] int8 | qsc, wqs [16] f32 | smax [8][16] f32 | wred [16] f32 |
//   E [hpw][16][S] f32 (per head, e[16 c + j] at [j][c]), reused for the
//   int32 P.V sums [NW][3 hpw][64] | planes [blocks][3 hpw][16] int8 + one row pad.
constexpr int FUSED_MAX_N = 1024, FUSED_MAX_GRP = 8;
// most waves of a workgroup: sixteen while a tile's registers leave room for
// four waves per SIMD
constexpr int fused_max_waves(int hd) { return hd <= 256 ? 16 : 8; }

__host__ __device__ inline size_t fused_e_bytes(int nw, int hpw, int max_n) {
  const size_t e = (size_t)hpw * 16 * exp_stride(max_n) * 4, red = (size_t)nw * 3 * hpw * 64 * 4;
  return e > red ? e : red;
}
// the last block's operand reads run to row 31 of 16 bytes
inline size_t fused_lds(int nw, int hd, int hpw, int max_n, int steps) {
  return (size_t)16 * (hd + 16) + (32 + 128 + 16) * 4 + fused_e_bytes(nw, hpw, max_n) +
         (size_t)steps * 4 * 48 * hpw + 32 * 16;
}

template <int KS, int NW>
__global__ __launch_bounds__(64 * NW) void attn_fused_kernel(const AttnArgs a) {
  constexpr int HD = KS * 64, QROW = HD + 16;
  constexpr int NSL = NW / KS;  // slot slices of the P.V product
  extern __shared__ __attribute__((aligned(16))) char sm[];
  const int rows = a.m * a.kvh, hs = blockIdx.x / rows, rg = blockIdx.x - hs * rows;
  const int r = rg / a.kvh, g = rg - r * a.kvh;
  const Geo G = row_geo(a, r);
  const int grp = a.nh / a.kvh, hpw = a.hpw;
  // heads [hf, hf + nhl) of this workgroup; of them [h0, h1) are computed
  const int hf = g * grp + hs * hpw, nhl = min(hpw, grp - hs * hpw);
  const int hb = max(a.h0, hf), he = min(a.h1, hf + nhl);
  if (hb >= he) return;
  const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
  const int n = max(G.n, 0), n16 = n & ~15, S = exp_stride(n);
  int8_t* qq = (int8_t*)sm;
  float* qsc = (float*)(sm + 16 * QROW);
  float* wqs = qsc + 16;    // per head: wmax / 65535, 0 = zero output
  float* smax = wqs + 16;   // [head][wave]: the maximum score
  float* wred = smax + 128; // per wave: the maximum weight of its head
  float* E = wred + 16;
  int8_t* PL = (int8_t*)E + fused_e_bytes(NW, hpw, a.max_n);  // three 7-bit planes, iw = a 2^14 + b 2^7 + c
  const int kvd = a.kvh * HD;
  const int c16 = lane & 15, q4 = lane >> 4;

  // ---- K: position tiles of 16, wave w the tiles w, w + NW, ...; the first
  // two in flight while the query is quantised
  const __amdgpu_buffer_rsrc_t rk = make_rsrc(G.kc, (uint32_t)((size_t)G.k_len * kvd));
  const __amdgpu_buffer_rsrc_t rks = make_rsrc(G.ks, (uint32_t)G.k_len * 4u);
  auto load = [&](v4i* B, int& kscale, int u0) {
    const int u = u0 + c16;
    const int slot = G.slot_of(u);
    const uint32_t base = u < n ? (uint32_t)slot * (uint32_t)kvd + (uint32_t)(g * HD + 16 * q4) : FGM_OOB;
    kscale = buf_load_b32(rks, u < n ? 4u * (uint32_t)slot : FGM_OOB, 0);
#pragma unroll
    for (int kk = 0; kk < KS; kk++) B[kk] = buf_load_b128(rk, base, 64 * kk);
  };
  v4i B0[KS], B1[KS];
  int ks0 = 0, ks1 = 0;
  int u0 = 16 * w;
  // the int8 query, one wave per head; the rows of A past nhl hold whatever
  // LDS held, and so do the scores' rows that nobody reads
  for (int hl = w; hl < nhl; hl += NW) {
    const float* qp = a.q + ((size_t)r * a.nh + hf + hl) * HD + lane;
    float x[KS];
    float amax = 0.0f;
#pragma unroll
    for (int kk = 0; kk < KS; kk++) x[kk] = qp[64 * kk];
    if (u0 < n && hl == w) load(B0, ks0, u0);
#pragma unroll
    for (int kk = 0; kk < KS; kk++) amax = __builtin_fmaxf(amax, __builtin_fabsf(x[kk]));
    amax = wave_max(amax);
    const float qinv = amax > 0.0f ? 127.0f / amax : 0.0f;
#pragma unroll
    for (int kk = 0; kk < KS; kk++) {
      const float v = __builtin_amdgcn_fmed3f(__builtin_rintf(x[kk] * qinv), -127.0f, 127.0f);
      qq[hl * QROW + 64 * kk + lane] = (int8_t)(int)v;
    }
    if (lane == 0) qsc[hl] = amax / 127.0f;
  }
  if (w >= nhl && u0 < n) load(B0, ks0, u0);
  if (u0 + 16 * NW < n) load(B1, ks1, u0 + 16 * NW);

  // ---- V: wave w takes the 64-dim block w % KS and the 64-slot steps w / KS,
  // + NSL, ...; lane (c, q4) loads the 16 bytes [4 dims][4 slots] of dims
  // 4 c .. 4 c + 3 and slot groups 4 q4 + r, r = 0..3: register q of the four
  // loads is one MFMA B operand (column c = dim 4 c + q).  The first steps do
  // not depend on the weights: in flight through scores and softmax.
  const int db = w % KS, sl = w / KS;
  const int steps = sl < NSL ? G.dom_steps : 0;
  const __amdgpu_buffer_rsrc_t rv = make_rsrc(G.vc, (uint32_t)((size_t)((G.k_len + 3) >> 2) * kvd * 4));
  auto loadv = [&](v4i* V, int step) {
    const int gi = (G.dom_slot(step) >> 2) + 4 * q4;
    const uint32_t at = ((uint32_t)gi * (uint32_t)kvd + (uint32_t)(g * HD + 64 * db + 4 * c16)) * 4u;
#pragma unroll
    for (int rr = 0; rr < 4; rr++) V[rr] = buf_load_b128(rv, at, (uint32_t)(rr * kvd * 4));
  };
  v4i V0[4], V1[4];
  if (sl < steps) loadv(V0, sl);
  __syncthreads();

  // ---- scores; each head's maximum is taken on the way to LDS
  float hmax[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
  {
    float qs4[4];
#pragma unroll
    for (int i = 0; i < 4; i++) qs4[i] = qsc[4 * q4 + i];
    auto tile = [&](const v4i* B, int ksc, int ut) {
      v4i acc = {0, 0, 0, 0};
#pragma unroll
      for (int kk = 0; kk < KS; kk++)
        acc = mfma16(*(const v4i*)(qq + c16 * QROW + 64 * kk + 16 * q4), B[kk], acc);
      const int u = ut + c16;
      const float kscale = __int_as_float(ksc);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int hl = 4 * q4 + i;
        if (u < n && hl < nhl) {
          const float s = ((float)acc[i] * qs4[i]) * kscale;
          hmax[i] = __builtin_fmaxf(hmax[i], s);
          E[(size_t)hl * 16 * S + (u & 15) * S + (u >> 4)] = s;
        }
      }
    };
#pragma unroll 1
    for (; u0 < n; u0 += 32 * NW) {
      tile(B0, ks0, u0);
      if (u0 + 16 * NW >= n) break;
      if (u0 + 32 * NW < n) load(B0, ks0, u0 + 32 * NW);
      tile(B1, ks1, u0 + 16 * NW);
      if (u0 + 48 * NW < n) load(B1, ks1, u0 + 48 * NW);
    }
  }
  if (sl + NSL < steps) loadv(V1, sl + NSL);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float m = row16_max(hmax[i]);
    if (c16 == 0 && 4 * q4 + i < nhl) smax[16 * (4 * q4 + i) + w] = m;
  }

  // ---- softmax: WPH waves per head, one slot (position) per lane
  const int WPH = NW / hpw, hw = w / WPH, sub = w - hw * WPH, first = 64 * sub + lane;
  const bool mine = hw < nhl && hf + hw >= hb && hf + hw < he;
  float* Eh = E + (size_t)hw * 16 * S;
  const __amdgpu_buffer_rsrc_t rvs = make_rsrc(G.vs, (uint32_t)G.k_len * 4u);
  // the first position's V scale is in flight through the exponentials
  const int vs0 = buf_load_b32(rvs, first < n ? 4u * (uint32_t)G.slot_of(first) : FGM_OOB, 0);
  __syncthreads();
  if (mine) {
    const float mx = row16_max(c16 < NW ? smax[16 * hw + c16] : -INFINITY);
#pragma unroll 1
    for (int u = first; u < n; u += 64 * WPH) {
      float* p = Eh + (u & 15) * S + (u >> 4);
      const float x = *p - mx;
      *p = u < n16 ? exp16(x) : (float)exp((double)x);
    }
  }
  __syncthreads();
  float wm = 0.0f, inv = 0.0f;
  if (mine) {
    // every wave of the head makes the reference's sum: lanes 0..15 in chunk
    // order, GCC's reduce tree, the tail in order
    float sum = 0.0f;
    if (lane < 16) sum = chunk_sum16(Eh + lane * S, n16 >> 4);
    sum = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(sum)));
#pragma unroll 1
    for (int u = n16; u < n; u++) sum += Eh[(u & 15) * S + (u >> 4)];
    inv = 1.0f / sum;
    int vs = vs0;
#pragma unroll 1
    for (int u = first; u < n; u += 64 * WPH) {
      wm = __builtin_fmaxf(wm, (Eh[(u & 15) * S + (u >> 4)] * inv) * __int_as_float(vs));
      if (u + 64 * WPH < n) vs = buf_load_b32(rvs, 4u * (uint32_t)G.slot_of(u + 64 * WPH), 0);
    }
    wm = wave_max(wm);
    if (lane == 0) wred[w] = wm;
  }
  // the planes of the slots that hold no position are zero
  for (int i = tid; i < G.dom_steps * 4 * 3 * hpw; i += 64 * NW) ((v4i*)PL)[i] = v4i{0, 0, 0, 0};
  __syncthreads();

  // ---- weight planes by slot
  if (mine) {
    wm = row16_max(c16 < WPH ? wred[hw * WPH + c16] : 0.0f);
    const bool pos = wm > 0.0f;
    const float wq_inv = 65535.0f / wm;
    if (sub == 0 && lane == 0) wqs[hw] = pos ? wm / 65535.0f : 0.0f;
    int vs = vs0;
#pragma unroll 1
    for (int u = first; pos && u < n; u += 64 * WPH) {
      const float wt = (Eh[(u & 15) * S + (u >> 4)] * inv) * __int_as_float(vs);
      int q = (int)__builtin_fmaf(wt, wq_inv, 0.5f);
      q = q > 65535 ? 65535 : (q < 0 ? 0 : q);
      const int s = G.slot_of(u), d = G.dom_off(s);
      q <<= G.twice(s) ? 1 : 0;
      int8_t* p = PL + (size_t)(d >> 4) * (48 * hpw) + hw * 16 + (d & 15);
      p[0] = (int8_t)(q >> 14);
      p[16 * hpw] = (int8_t)((q >> 7) & 127);
      p[32 * hpw] = (int8_t)(q & 127);
      if (u + 64 * WPH < n) vs = buf_load_b32(rvs, 4u * (uint32_t)G.slot_of(u + 64 * WPH), 0);
    }
  }
  __syncthreads();

  // ---- P.V: the A operand's rows are (plane, head), 3 hpw of them in one
  // operand or two; sums over the wave's steps in registers
  v4i D0[4], D1[4];
#pragma unroll
  for (int q = 0; q < 4; q++) D0[q] = D1[q] = v4i{0, 0, 0, 0};
  const bool two = 3 * hpw > 16;
  auto mulv = [&](const v4i* V, int step) {
    const int8_t* wp = PL + (size_t)(4 * step + q4) * (48 * hpw) + c16 * 16;
    const v4i A0 = *(const v4i*)wp;
#pragma unroll
    for (int q = 0; q < 4; q++) D0[q] = mfma16(A0, v4i{V[0][q], V[1][q], V[2][q], V[3][q]}, D0[q]);
    if (two) {
      const v4i A1 = *(const v4i*)(wp + 256);
#pragma unroll
      for (int q = 0; q < 4; q++) D1[q] = mfma16(A1, v4i{V[0][q], V[1][q], V[2][q], V[3][q]}, D1[q]);
    }
  };
#pragma unroll 1
  for (int st = sl; st < steps; st += 2 * NSL) {
    mulv(V0, st);
    if (st + NSL >= steps) break;
    if (st + 2 * NSL < steps) loadv(V0, st + 2 * NSL);
    mulv(V1, st + NSL);
    if (st + 3 * NSL < steps) loadv(V1, st + 3 * NSL);
  }
  // the rows' sums to LDS (in the exponentials' place: all read), one
  // [3 hpw][64] block per wave
  int32_t* red = (int32_t*)E;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int row = 4 * q4 + i;
    if (row < 3 * hpw) *(v4i*)(red + ((size_t)w * 3 * hpw + row) * 64 + 4 * c16) = v4i{D0[0][i], D0[1][i], D0[2][i], D0[3][i]};
    if (row + 16 < 3 * hpw)
      *(v4i*)(red + ((size_t)w * 3 * hpw + row + 16) * 64 + 4 * c16) = v4i{D1[0][i], D1[1][i], D1[2][i], D1[3][i]};
  }
  __syncthreads();
  // sum iw v = a 2^14 + b 2^7 + c (modulo 2^32, as the reference's int32
  // lanes) over the slices; out = (float)(that) * wmax / 65535
#pragma unroll 1
  for (int idx = tid; idx < nhl * HD; idx += 64 * NW) {
    const int hr = idx / HD, d = idx - hr * HD;
    uint32_t t = 0;
#pragma unroll
    for (int s = 0; s < NSL; s++) {
      const int32_t* p = red + (size_t)(s * KS + (d >> 6)) * 3 * hpw * 64 + hr * 64 + (d & 63);
      t += ((uint32_t)p[0] << 14) + ((uint32_t)p[64 * hpw] << 7) + (uint32_t)p[128 * hpw];
    }
    if (hf + hr >= hb && hf + hr < he)
      a.out[((size_t)r * a.nh + hf + hr) * HD + d] = (float)(int32_t)t * wqs[hr];
  }
}

// Sixteen waves where only one workgroup shares a CU (its LDS is more than half
// of it, or there is one for each) and has several heads' positions to walk;
// else eight: two such workgroups share a CU (at 122 registers it holds sixteen
// waves) and overlap their chains.  Sixteen -> eight waves: 8 heads on 4 kv heads
// of 128, window 64, 256 / 1024 rows 25.6 -> 14.4 / 93.6 -> 45.5 us; 8 on 1 of 64,
// a prompt of 512 rows 23.7 -> 16.7; 8 decode rows, 8 on 1 of 256, window 512
// 12.4 -> 12.0; on the other side, 256 rows of 8 heads on 1, window 1024 at
// head_dim 128 19.4 -> 21.2 and window 512 at 256 17.0 -> 17.3.
int fused_waves(const AttnArgs& a) {
  const int wgs = a.m * a.kvh * ((a.nh / a.kvh + a.hpw - 1) / a.hpw);
  const bool alone = fused_lds(8, a.hd, a.hpw, a.max_n, a.max_steps) > 80 * 1024 ||
                     (wgs <= 256 && a.hpw * a.max_n >= 3000);
  return std::min(alone ? 16 : 8, fused_max_waves(a.hd));
}

template <int KS, int NW>
hipError_t launch_fused(const AttnArgs& a, size_t lds, hipStream_t st) {
  static hipError_t attr = hipFuncSetAttribute((const void*)attn_fused_kernel<KS, NW>,
                                               hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  if (attr != hipSuccess) return attr;
  const int hs = (a.nh / a.kvh + a.hpw - 1) / a.hpw;
  hipLaunchKernelGGL((attn_fused_kernel<KS, NW>), dim3(a.m * a.kvh * hs), dim3(64 * NW), lds, st, a);
  return hipGetLastError();
}

// ----------------------------------------------------------- cache writes
// fgm_store_v_t (ops.c:653-657)
__global__ void store_v_t_kernel(int8_t* vt, const int8_t* src, int n, int slot) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n) vt[((size_t)(slot >> 2) * n + j) * 4 + (slot & 3)] = src[j];
}

// The forward pass's append (forward.rs:515-548): quant_act of each K and V
// row (ops.c:181-204: s = amax == 0 ? 1 : amax / 127, q = cvt(x * (1 / s))
// saturated, the n % 16 tail as lrintf + clamp), K stored in place, V through
// the transposed layout.  grid (m, 2): y = 0 K, 1 V; 256 threads.
constexpr int KV_VMAX = 8;  // row_len <= 4 * 256 * KV_VMAX
__global__ __launch_bounds__(256) void kv_store_kernel(const float* k, const float* v, int rl,
                                                      int8_t* kc, float* ks, int8_t* vt, float* vs,
                                                      int pos0, int ring) {
  __shared__ float red[4];
  const int r = blockIdx.x, isv = blockIdx.y, tid = threadIdx.x;
  const float* src = (isv ? v : k) + (size_t)r * rl;
  const int pos = pos0 + r, slot = ring ? pos % ring : pos;
  float x[KV_VMAX][4];
  float mx = 0.0f;
#pragma unroll
  for (int s = 0; s < KV_VMAX; s++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int c = 4 * (tid + 256 * s) + e;
      x[s][e] = c < rl ? src[c] : 0.0f;
      mx = __builtin_fmaxf(mx, __builtin_fabsf(x[s][e]));
    }
  mx = wave_max(mx);
  if ((tid & 63) == 0) red[tid >> 6] = mx;
  __syncthreads();
  mx = __builtin_fmaxf(__builtin_fmaxf(red[0], red[1]), __builtin_fmaxf(red[2], red[3]));
  const float sc = mx == 0.0f ? 1.0f : mx / 127.0f;
  const float inv = 1.0f / sc;
  const int rv = rl & ~15;
#pragma unroll
  for (int s = 0; s < KV_VMAX; s++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int c = 4 * (tid + 256 * s) + e;
      if (c >= rl) continue;
      const float y = x[s][e] * inv;
      const int8_t q = c < rv ? quant_vec(y) : quant_tail(y);
      if (isv)
        vt[((size_t)(slot >> 2) * rl + c) * 4 + (slot & 3)] = q;
      else
        kc[(size_t)slot * rl + c] = q;
    }
  if (tid == 0) (isv ? vs : ks)[slot] = sc;
}

// f(integral_constant<head_dim / 64>)
template <class F>
hipError_t with_ks(int hd, F&& f) {
  switch (hd / 64) {
    case 1: return f(std::integral_constant<int, 1>{});
    case 2: return f(std::integral_constant<int, 2>{});
    case 3: return f(std::integral_constant<int, 3>{});
    case 4: return f(std::integral_constant<int, 4>{});
    case 5: return f(std::integral_constant<int, 5>{});
    case 6: return f(std::integral_constant<int, 6>{});
    case 7: return f(std::integral_constant<int, 7>{});
    case 8: return f(std::integral_constant<int, 8>{});
    default: return hipErrorInvalidValue;
  }
}

template <int NQ, int T>
hipError_t launch_softmax(const AttnArgs& a, size_t lds, hipStream_t st) {
  static hipError_t attr = hipFuncSetAttribute((const void*)attn_softmax_kernel<NQ, T>,
                                               hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL((attn_softmax_kernel<NQ, T>), dim3(a.m * (a.h1 - a.h0)), dim3(T), lds, st, a);
  return hipGetLastError();
}

// groups of four slots per thread: the smallest instance that covers them
hipError_t launch_softmax(const AttnArgs& a, hipStream_t st) {
  const int quads = 16 * a.tile_steps;
  // with hundreds of (row, head) pairs several workgroups share a CU; a few
  // get the widest workgroups
  const bool many = a.m * (a.h1 - a.h0) >= 256 && quads <= 6 * 512;
  const size_t lds = ((size_t)16 * exp_stride(a.max_n) + 32) * 4;
  // up to 1024 slots: every further wave is launched and waited for without any
  // (window 64, 16 heads of 256 on one kv head: 16 rows 23.3 -> 13.3 us, 256
  // 55.6 -> 37.4; of 64: 1024 rows 131.4 -> 70.2)
  if (quads <= 1 * 256) return launch_softmax<1, 256>(a, lds, st);
  if (many) {
    if (quads <= 1 * 512) return launch_softmax<1, 512>(a, lds, st);
    if (quads <= 2 * 512) return launch_softmax<2, 512>(a, lds, st);
    if (quads <= 3 * 512) return launch_softmax<3, 512>(a, lds, st);
    if (quads <= 4 * 512) return launch_softmax<4, 512>(a, lds, st);
    return launch_softmax<6, 512>(a, lds, st);
  }
  if (quads <= 1 * 1024) return launch_softmax<1, 1024>(a, lds, st);
  if (quads <= 2 * 1024) return launch_softmax<2, 1024>(a, lds, st);
  if (quads <= 3 * 1024) return launch_softmax<3, 1024>(a, lds, st);
  if (quads <= 4 * 1024) return launch_softmax<4, 1024>(a, lds, st);
  if (quads <= 6 * 1024) return launch_softmax<6, 1024>(a, lds, st);
  if (quads <= 9 * 1024) return launch_softmax<9, 1024>(a, lds, st);
  return hipErrorInvalidValue;
}

}  // namespace

size_t fgm_attn_layout(AttnArgs* a, void* base, int m, int nh, int kvh, int hd, int max_span) {
  const int grp = nh / kvh;
  // the domain of a row tile: the union of its rows' ranges, at most
  // max_span + FGM_ATTN_TILE - 1 positions, in two runs of partial steps
  const int cap = (max_span + FGM_ATTN_TILE + 6) / 64 + 4;
  auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
  size_t off = 0;
  const size_t o_sc = off;
  off = al(off + (size_t)m * nh * cap * 64 * 4);
  const size_t o_wpl = off;
  off = al(off + (size_t)m * kvh * grp * cap * 128);
  const size_t o_part = off;
  off = al(off + (size_t)attn_part_rows(m) * nh * hd * 4);
  const size_t o_wq = off;
  off = al(off + (size_t)m * nh * 4);
  if (a && base) {
    char* b = (char*)base;
    a->sc = (float*)(b + o_sc);
    a->cap = cap;
    a->wpl = (int8_t*)(b + o_wpl);
    a->part = (int32_t*)(b + o_part);
    a->wq = (float*)(b + o_wq);
  }
  return off;
}

hipError_t fgm_launch_attn(const AttnArgs& a, hipStream_t st) {
  if (a.m <= 0 || a.h1 <= a.h0) return hipSuccess;
  hipError_t e = hipSuccess;
  // one launch when every row is short and a kv group fits the workgroup;
  // FGM_ATTN_FUSED=0 keeps the longer path (for comparison and tests)
  const int grp = a.nh / a.kvh;
  const char* fz = getenv("FGM_ATTN_FUSED");
  // query heads per workgroup: as few as fill the chip (256 CUs) once
  AttnArgs f = a;
  f.hpw = 1;
  while (f.hpw < grp && a.m * a.kvh * ((grp + f.hpw - 1) / f.hpw) > 256) f.hpw *= 2;
  f.hpw = std::min(f.hpw, grp);
  const int nw = fused_waves(f);
  const size_t flds = fused_lds(nw, a.hd, f.hpw, a.max_n, a.max_steps);
  if (a.max_n <= FUSED_MAX_N && grp <= FUSED_MAX_GRP && !(fz && fz[0] == '0') && flds <= 160 * 1024)
    return with_ks(a.hd, [&](auto ks) {
      constexpr int KS = decltype(ks)::value;
      return nw == 8 ? launch_fused<KS, 8>(f, flds, st) : launch_fused<KS, fused_max_waves(64 * KS)>(f, flds, st);
    });

  const int chunks = (a.tile_steps + a.p1_steps - 1) / a.p1_steps;
  if (a.rt > 1) {
    const int pairs = a.m * a.nh;
    hipLaunchKernelGGL(attn_quant_q_kernel, dim3((pairs + 3) / 4), dim3(256), 0, st, a.q, (int8_t*)a.part, a.wq, pairs,
                       a.hd);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    e = with_ks(a.hd, [&](auto ks) {
      hipLaunchKernelGGL(attn_scores_tile_kernel<decltype(ks)::value>, dim3(chunks, a.ntiles * a.kvh), dim3(256), 0, st,
                         a);
      return hipGetLastError();
    });
  } else {
    e = with_ks(a.hd, [&](auto ks) {
      hipLaunchKernelGGL(attn_scores_kernel<decltype(ks)::value>, dim3(chunks, a.m * a.kvh), dim3(256), 0, st, a);
      return hipGetLastError();
    });
  }
  if (e != hipSuccess) return e;
  if ((e = launch_softmax(a, st)) != hipSuccess) return e;
  if (a.rt > 1) {
    const dim3 grid((a.hd + 255) / 256, a.ntiles * a.kvh, a.p3_chunks);
    if (a.hd > 128)
      hipLaunchKernelGGL(attn_pv_tile_kernel<2>, grid, dim3(512), 0, st, a);
    else
      hipLaunchKernelGGL(attn_pv_tile_kernel<1>, grid, dim3(256), 0, st, a);
  } else {
    const dim3 grid(a.hd / a.p3_dims, a.m * a.kvh, a.p3_chunks);
    if (grp > 8 && a.p3_dims == 16)
      hipLaunchKernelGGL((attn_pv_kernel<true, 1>), grid, dim3(512), 0, st, a);
    else if (grp > 8)
      hipLaunchKernelGGL((attn_pv_kernel<true, 2>), grid, dim3(512), 0, st, a);
    else if (a.p3_dims == 16)
      hipLaunchKernelGGL((attn_pv_kernel<false, 1>), grid, dim3(1024), 0, st, a);
    else
      hipLaunchKernelGGL((attn_pv_kernel<false, 2>), grid, dim3(1024), 0, st, a);
  }
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (a.p3_chunks > 1 || a.dup) {
    hipLaunchKernelGGL(attn_final_kernel, dim3(a.m * (a.h1 - a.h0)), dim3(a.hd / 4), 0, st, a);
    e = hipGetLastError();
  }
  return e;
}

hipError_t fgm_launch_store_v_t(int8_t* vt, const int8_t* src, int n, int slot, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(store_v_t_kernel, dim3((n + 255) / 256), dim3(256), 0, st, vt, src, n, slot);
  return hipGetLastError();
}

hipError_t fgm_launch_kv_store(const float* k, const float* v, int m, int row_len, int8_t* kc,
                               float* ks, int8_t* vt, float* vs, int pos0, int ring, hipStream_t st) {
  if (m <= 0 || row_len <= 0) return hipSuccess;
  if (row_len > 4 * 256 * KV_VMAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL(kv_store_kernel, dim3(m, 2), dim3(256), 0, st, k, v, row_len, kc, ks, vt, vs,
                     pos0, ring);
  return hipGetLastError();
}
