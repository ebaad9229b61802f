// Selective Attention for MI355X (gfx950): selection scan, forward, chunked prefill, backward.
//
// Operator (reference src/selective_attention/kernels.py:61-83, docs/kernel.md:32-46):
//   L_h = s Q_h K_h^T (causal),  S = relu(L_0) on E <= j < r,  F[i,j] = sum_{r<i} S[r,j],
//   O_h = softmax(L_h - F) V_h.
//
// Kernels (all 256 threads = 4 wavefronts of 64; MFMA 32x32 tiles; the attention kernels order
// their workgroups so that each XCD's L2 serves a contiguous range of heads):
//   sel_colsum   head 0, one 32x32 (queries x keys) tile per step: column sums of S per
//                32-query block -> colsum[b][rb][j]
//   sel_scan     exclusive running sum of colsum over query blocks, seeded by the carried
//                per-key state -> carry[b][rb][j], state_out[b][j]
//   fwd          query-parallel. A wavefront owns 32 queries of G heads. Logit tiles are
//                built transposed (keys x queries) so each lane holds one query: the online
//                softmax row statistics stay in-lane, and O^T = V^T P^T takes P straight from
//                the accumulator registers. Head 0's logits are built (queries x keys) instead,
//                so the selection's prefix over queries runs down each lane's registers; F then
//                reaches the softmax layout through the wavefront's LDS rows.
//   bwd_rowprep  row statistics, bounds for the tiles without weight, the exempt keys' gradients
//   bwd_kv       key-parallel. A wavefront owns 32 keys of G heads and sweeps the query tiles
//                last to first, from the last that holds weight for its workgroup's keys. Tiles are (queries x keys), so the selection prefix F and the
//                suffix U = sum_h sum_{i>r} dz_h[i,j] run down registers. dK, dV (and the
//                group's share of head 0's dK) stay in registers; K, V rows sit in LDS. U is
//                checkpointed per query tile for bwd_dq.
//   bwd_dq       query-parallel. A wavefront owns 32 queries and walks the key tiles up to its
//                diagonal, recomputing P, dz and the selection gradient g from the key side's
//                U checkpoints; dQ = dz K takes dz through a per-wavefront LDS tile.
//   bwd_finish   gradient epilogue: scale, add head 0's shares and the exempt keys' partial sums, convert
//                to the output dtype.
// The group holding head 0 folds g = -gate*U into head 0's own dz; every other group stores its
// share of head 0's gradients in a slot of its own, and bwd_finish sums the slots in a fixed order
// (no atomics: the backward is bitwise repeatable).
//
// MFMA operand layouts used throughout (v_mfma_f32_32x32x16_bf16 / v_mfma_f32_32x32x2_f32):
//   C (32x32, 16 fp32 per lane): lane l holds column l%32, rows crow(i, l/32), i = 0..15,
//                                crow(i,h) = 8*(i/4) + 4*h + i%4.
//   A (32xK) / B (Kx32):         lane l holds row (A) / column (B) l%32 and K elements
//                                [KS*step + (KS/2)*h, +KS/2) with KS = 16 (bf16) or 2 (fp32).
// A C-layout tile fed back as a B operand keeps its registers in place; the matching A operand
// is then read with the C layout's row order (ld_perm; bf16 tiles read that way are staged with
// their columns in that order, ColTile::store_crow, so a fragment is one 16-byte read).


#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <limits.h>
#include <math.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "sa_host.h"

namespace {

using namespace sa_host;

typedef __bf16 bf16_t;
typedef bf16_t bf16x8 __attribute__((__vector_size__(8 * sizeof(bf16_t))));
typedef float f32x16 __attribute__((__vector_size__(16 * sizeof(float))));

constexpr float LOG2E = 1.4426950408889634f;

__device__ __forceinline__ int crow(int i, int h) { return 8 * (i >> 2) + 4 * h + (i & 3); }

__device__ __forceinline__ f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.f;
  return z;
}

__device__ __forceinline__ float xor32(float x) { return __shfl_xor(x, 32); }

// The values of lanes 0-31 (lo) and of lanes 32-63 (hi) of the same column, in every lane
// (one v_permlane32_swap).
struct Halves {
  float lo, hi;
};
__device__ __forceinline__ Halves halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(x), __float_as_int(x), false, false);
  return {__int_as_float(r[0]), __int_as_float(r[1])};
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Word 3 of a raw buffer resource on gfx950 (32-bit data format; offsets in bytes, range-checked
// against the resource's byte count: loads past it return zero).
constexpr int RSRC_WORD3 = 0x00020000;

// A 32 x 32 bf16 tile kept transposed in LDS for the transposing read ds_read_b64_tr_b16: rows of
// 32 elements (64 bytes), the 8-byte chunk c of row r stored at chunk c ^ sw(r / 2 mod 8), sw(a) =
// 4 (a mod 2) + a / 2. The read gives lane i of each 16-lane group, element t, the element i % 4
// of the 8 bytes that lane 4t + i/4 of the group addresses (measured on gfx950). The 8-byte
// lane-per-row writes go to the banks 16 lanes at a time (32 banks of 4 bytes, as measured with the
// bank-conflict counter): sixteen consecutive rows then hold one chunk in 16 distinct bank pairs
// (rows of one parity take distinct chunks); a transposing read of four consecutive rows, chunks
// 0-3 or 4-7, finds the two rows of each parity on opposite halves of the row.
__device__ __forceinline__ int trt_off(int r, int c) {
  const int a = (r >> 1) & 7;
  return r * 32 + ((c ^ (((a & 1) << 2) | (a >> 1))) << 2);
}

typedef short short4v __attribute__((ext_vector_type(4)));

// Writes a C-layout tile x (lane = column n, element i = row crow(i, h)) transposed: row n of the
// LDS tile holds column n of x, 4 consecutive rows of x per 8-byte write. LO: the rounding
// residuals x - bf16(x) instead.
template <bool LO>
__device__ __forceinline__ void put_tr(uint16_t* t, const f32x16& x, int n, int h) {
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    typedef bf16_t bf16x4 __attribute__((__vector_size__(4 * sizeof(bf16_t))));
    bf16x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float f = x[4 * a + e];
      v[e] = LO ? (bf16_t)(f - (float)(bf16_t)f) : (bf16_t)f;
    }
    *reinterpret_cast<bf16x4*>(t + trt_off(n, 2 * a + h)) = v;
  }
}

// The A (or B) operand of K step s read from such a tile: lane l gets row l % 32 of the
// untransposed tile, elements 16s + 8(l / 32) + 0..7, in order.
__device__ __forceinline__ bf16x8 get_tr(const uint16_t* t, int lane, int s) {
  const int g = lane >> 4, k = lane & 15;
  const int n0 = 16 * (g & 1), hh = g >> 1;
  bf16x8 f;
#pragma unroll
  for (int hf = 0; hf < 2; ++hf) {
    const int r = 16 * s + 8 * hh + 4 * hf + (k >> 2);
    typedef __attribute__((address_space(3))) short4v* lds_s4;
    const short4v v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(t + trt_off(r, (n0 >> 2) + (k & 3))));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const short x = v[e];
      f[4 * hf + e] = *reinterpret_cast<const bf16_t*>(&x);
    }
  }
  return f;
}

// Element i = s[crow(i, h)]: a C-layout tile whose rows take the values of a 32-entry LDS row
// vector (four 16-byte reads).
__device__ __forceinline__ f32x16 rows16(const float* s, int h) {
  f32x16 r;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const float4 v = *reinterpret_cast<const float4*>(s + 8 * a + 4 * h);
    r[4 * a] = v.x;
    r[4 * a + 1] = v.y;
    r[4 * a + 2] = v.z;
    r[4 * a + 3] = v.w;
  }
  return r;
}

// The wavefront index within the workgroup, as a value the compiler knows is uniform across the
// wavefront (threadIdx.x / 64 is, but divergence analysis cannot see it): tile flags derived from
// it become scalar branches instead of per-lane exec masks.
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// Wavefront-local ordering of LDS traffic (writes by some lanes, reads by others).
__device__ __forceinline__ void lds_wave_sync() {
  __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}
// The same ordering without the wait: the LDS performs one wavefront's operations in issue order,
// so a read issued after a write of the same wavefront sees it, and a later write cannot overtake an
// earlier read; only the compiler must keep the accesses in program order. (The wait drained every
// outstanding LDS read of the wavefront, operand reads of the next product included: measured, the
// query-side backward at C2 runs 1.4% faster without it, all GPU tests unchanged.)
__device__ __forceinline__ void lds_wave_order() { __asm__ volatile("" ::: "memory"); }

// ---------------------------------------------------------------------------------------------
// Operand traits: bf16 storage -> bf16 MFMA; fp32 storage -> fp32 MFMA.

struct OpBF16 {
  typedef uint16_t elem;
  typedef bf16x8 frag;
  static constexpr int KS = 16;
  static constexpr int KPAD = 8;     // LDS row padding (elements) of [rows][D] tiles
  static constexpr int TPAD = 8;     // LDS row padding (elements) of [rows][32] tiles: 80-byte rows,
                                     // 16-byte aligned, distinct banks for 16 rows

  static __device__ __forceinline__ f32x16 mma(frag a, frag b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ frag zero() {
    frag f;
#pragma unroll
    for (int t = 0; t < 8; ++t) f[t] = (bf16_t)0.f;
    return f;
  }
  // Row r of a row-major tile, K elements [16*s + 8*h, +8).
  static __device__ __forceinline__ frag ld_std(const elem* p, int64_t ld, int r, int h, int s) {
    return *reinterpret_cast<const frag*>(p + r * ld + s * 16 + 8 * h);
  }
  // Row r, K elements in C-layout row order for step s -- columns [16s+4h, +4) and [16s+8+4h, +4)
  // -- from a tile whose columns were stored in that order (ColTile::store_crow): one 16-byte read.
  static __device__ __forceinline__ frag ld_perm(const elem* p, int64_t ld, int r, int h, int s) {
    return *reinterpret_cast<const frag*>(p + r * ld + s * 16 + 8 * h);
  }
  // C-layout registers [8s, 8s+8) as an operand (round to nearest even).
  static __device__ __forceinline__ frag from_acc(const f32x16& c, int s) {
    frag f;
#pragma unroll
    for (int t = 0; t < 8; ++t) f[t] = (bf16_t)c[8 * s + t];
    return f;
  }
  // The rounding residual of from_acc: c - bf16(c), itself rounded. hi + lo carries about 16
  // significant bits, so a product taken on both keeps its sum close to fp32.
  static constexpr bool SPLIT = true;
  static __device__ __forceinline__ frag from_acc_lo(const f32x16& c, int s) {
    frag f;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const float x = c[8 * s + t];
      f[t] = (bf16_t)(x - (float)(bf16_t)x);
    }
    return f;
  }
  static __device__ __forceinline__ elem to_elem(float x) {
    bf16_t b = (bf16_t)x;
    return *reinterpret_cast<elem*>(&b);
  }
  static __device__ __forceinline__ elem to_elem_lo(float x) { return to_elem(x - to_float(to_elem(x))); }
  static __device__ __forceinline__ float to_float(elem x) {
    return __uint_as_float(((uint32_t)x) << 16);
  }
  static constexpr int acc_steps = 2;   // C-layout K steps over 32 rows
};

struct OpF32 {
  typedef float elem;
  typedef float frag;
  static constexpr int KS = 2;
  static constexpr int KPAD = 4;
  static constexpr int TPAD = 1;

  static __device__ __forceinline__ f32x16 mma(frag a, frag b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ frag zero() { return 0.f; }
  static __device__ __forceinline__ frag ld_std(const elem* p, int64_t ld, int r, int h, int s) {
    return p[r * ld + 2 * s + h];
  }
  static __device__ __forceinline__ frag ld_perm(const elem* p, int64_t ld, int r, int h, int s) {
    return p[r * ld + crow(s, h)];   // a standard-order tile (ColTile::store_crow stores fp32 as is)
  }
  static __device__ __forceinline__ frag from_acc(const f32x16& c, int s) { return c[s]; }
  static constexpr bool SPLIT = false;   // fp32 operands are exact already
  static __device__ __forceinline__ frag from_acc_lo(const f32x16& c, int s) { return 0.f; }
  static __device__ __forceinline__ elem to_elem(float x) { return x; }
  static __device__ __forceinline__ elem to_elem_lo(float x) { return 0.f; }
  static __device__ __forceinline__ float to_float(elem x) { return x; }
  static constexpr int acc_steps = 16;
};

// Fragment read straight from global memory with a row bound (rows >= nrows read as zero).
template <class OP>
__device__ __forceinline__ typename OP::frag ld_std_bounded(const typename OP::elem* p, int64_t ld,
                                                            int r, int nrows, int h, int s) {
  if (r < nrows) return OP::ld_std(p, ld, r, h, s);
  return OP::zero();
}

// B operand of a key-contracted product taken from a row-major [keys][D] global matrix:
// lane holds rows key0 + KS*s + (KS/2)*h + t, column d. Rows >= nrows read as zero.
template <class OP>
__device__ __forceinline__ typename OP::frag ld_colgather(const typename OP::elem* p, int D, int key0,
                                                          int nrows, int d, int h, int s) {
  typename OP::frag f;
  if constexpr (OP::KS == 16) {
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      int r = key0 + 16 * s + 8 * h + t;
      uint16_t raw = (r < nrows) ? p[(int64_t)r * D + d] : (uint16_t)0;
      f[t] = *reinterpret_cast<bf16_t*>(&raw);
    }
  } else {
    int r = key0 + 2 * s + h;
    f = (r < nrows) ? p[(int64_t)r * D + d] : 0.f;
  }
  return f;
}

// ---------------------------------------------------------------------------------------------
// LDS staging (whole workgroup).

// [32 rows][COLS] tile from a row-major global matrix (row stride gld); rows >= nrows are zero.
template <typename E, int COLS, int SLD>
__device__ __forceinline__ void stage_rows(E* s, const E* g, int64_t gld, int row0, int nrows, int tid) {
  constexpr int EPC = 16 / sizeof(E);
  constexpr int CPR = COLS / EPC;
  constexpr int NCH = TILE * CPR;
  static_assert((SLD * sizeof(E)) % 16 == 0, "row stride must keep 16-byte alignment");
#pragma unroll
  for (int c = tid; c < NCH; c += NTHREADS) {
    const int r = c / CPR, cc = (c % CPR) * EPC;
    uint4 val = make_uint4(0u, 0u, 0u, 0u);
    if (row0 + r < nrows) val = *reinterpret_cast<const uint4*>(g + (int64_t)(row0 + r) * gld + cc);
    *reinterpret_cast<uint4*>(s + r * SLD + cc) = val;
  }
}

// [ROWS][32] tile: columns col0..col0+31 of a row-major global matrix (row stride gld, 16-byte
// aligned rows); columns >= ncols are zero.
template <typename E, int ROWS, int SLD>
__device__ __forceinline__ void stage_cols(E* s, const E* g, int64_t gld, int col0, int ncols, int tid) {
  constexpr int EPC = 16 / sizeof(E);
  constexpr int CPR = TILE / EPC;
  constexpr int NCH = ROWS * CPR;
#pragma unroll
  for (int c = tid; c < NCH; c += NTHREADS) {
    const int r = c / CPR, cc = (c % CPR) * EPC;
    const E* src = g + (int64_t)r * gld + col0 + cc;
    union { uint4 v; E e[EPC]; uint2 h[2]; } u;
    if (col0 + cc + EPC <= ncols) {
      u.v = *reinterpret_cast<const uint4*>(src);
    } else {
#pragma unroll
      for (int e = 0; e < EPC; ++e) u.e[e] = (col0 + cc + e < ncols) ? src[e] : (E)0;
    }
    E* dst = s + r * SLD + cc;
    if constexpr (sizeof(E) == 2) {
      static_assert((SLD * 2) % 8 == 0, "bf16 transposed tiles need 8-byte row alignment");
      reinterpret_cast<uint2*>(dst)[0] = u.h[0];
      reinterpret_cast<uint2*>(dst)[1] = u.h[1];
    } else {
#pragma unroll
      for (int e = 0; e < EPC; ++e) dst[e] = u.e[e];
    }
  }
}

// The dispatcher deals workgroups round-robin to the 8 XCDs, each with its own L2. The selection
// kernels and the generic forward remap the linear workgroup id so that every XCD takes a contiguous
// range of the (head group, block) order instead: the workgroups one L2 serves at a time then belong
// to one or two heads and share that head's tiles (the direct-load forward's order is part_block, the
// backward kernels' work_order_block, below).
constexpr int NXCD = 8;
struct BlockXY {
  int x, y;
};
__device__ __forceinline__ BlockXY xcd_block() {
  const int gx = gridDim.x, n = gx * gridDim.y;
  const int l = blockIdx.x + gx * blockIdx.y;
  const int per = n / NXCD;
  const int m = (l < per * NXCD) ? (l % NXCD) * per + l / NXCD : l;
  return {m % gx, m / gx};
}

// The backward kernels' order: x-major (x the block, whose work falls as x grows; y the head row),
// so the round-robin deal gives every XCD every eighth workgroup of a list sorted by work: each XCD
// runs its share longest first and the XCDs' shares stay even whatever the head count. (With the
// contiguous ranges of xcd_block, 12 heads leave one XCD a third more work than the mean: the
// backward at the reference's 12-head geometry ran as long as at 16 heads.) An XCD still serves
// few heads at a time -- heads i and i + 8 at a multiple of 8 -- whose tiles it shares in its L2.
__device__ __forceinline__ BlockXY work_order_block() {
  const int gy = gridDim.y;
  const int l = blockIdx.x + gridDim.x * blockIdx.y;
  return {l / gy, l % gy};
}

// work_order_block with each XCD's share (every eighth workgroup of the longest-first list, n of
// them) dispatched in a different order when `slots` (the workgroups an XCD runs at once) is
// nonzero: its `slots` longest first, as before, then the shortest third of the rest, shortest
// first, then the middle third, longest first. The dispatcher hands an XCD's next workgroup to
// whichever slot frees first, so with about three workgroups per slot (the 12 heads of the
// reference's model at 16384 tokens) a slot that ran a short first workgroup collects a run of the
// shortest ones before the middle third arrives, and the slots end closer together than with the
// longest-first order, whose third round leaves the spread of the middle third (a list-scheduling
// simulation: 1.03x the balanced share against 1.11x). The query-side kernel takes it (one
// workgroup per CU; the host passes `slots` only in that regime, bwd_snake_slots): at d768 1.28 ->
// 1.18 ms per layer. The key side, two workgroups per CU, keeps the longest-first order: a
// workgroup left alone on its CU speeds up once its CU-mate finishes, which already evens its
// slots (1.20 ms there, three quarters of its 16-head time), and the other order ran it 3% slower.
__device__ __forceinline__ BlockXY work_order_block(int slots) {
  if (slots <= 0) return work_order_block();
  const int gy = gridDim.y, total = gridDim.x * gy;
  const int l = blockIdx.x + gridDim.x * blockIdx.y;
  const int x8 = l % NXCD, p = l / NXCD;             // this XCD's p-th dispatch
  const int n = (total - x8 + NXCD - 1) / NXCD;      // workgroups of this XCD
  int q = p;                                         // rank in the XCD's longest-first list
  if (p >= slots && n > slots) {
    const int rest = n - slots, n_low = rest - rest / 2, pp = p - slots;
    q = (pp < n_low) ? n - 1 - pp : slots + (pp - n_low);
  }
  const int g = q * NXCD + x8;
  return {g / gy, g % gy};
}

// The direct-load forward's order: every XCD takes an equal share of the work from as few head
// groups as that allows, longest first. Each row y (one head group of one sequence, its blocks x
// ordered longest first) is cut into P parts by x mod P, P = 8 / gcd(gy, 8), so that the gy * P
// parts divide evenly over the 8 XCDs; the parts of a row hold nearly equal work. XCD i takes parts
// [i m, i m + m), m = gy P / 8 (one row's worth or a little more), and runs them x-major: block by
// block, longest first. With 6 or 12 rows (the 12 heads of the reference's model, in pairs)
// xcd_block's contiguous ranges give one XCD the long blocks of a row and another its short ones
// (measured: a third more work on the busiest XCD). With gy a multiple of 8 (P = 1) every XCD takes
// whole rows and xcd_block's order, one row after another, is kept: interleaving an XCD's rows
// doubled the forward's HBM fetches at 32 rows (C5's). A grid whose x extent P does not divide falls
// back to xcd_block too.
__device__ __forceinline__ BlockXY part_block() {
  const int gx = gridDim.x, gy = gridDim.y;
  const int P = NXCD >> min(__builtin_ctz((unsigned)gy), 3);   // 8 / gcd(gy, 8)
  if (P == 1 || gx % P != 0) return xcd_block();
  const int m = gy * P / NXCD;
  const int l = blockIdx.x + gx * blockIdx.y;
  const int r = l / NXCD;
  const int part = (l % NXCD) * m + r % m;
  return {part % P + (r / m) * P, part / P};
}

// Unpadded LDS rows of 64 bf16 (eight 16-byte chunks), chunk c of row r stored at chunk position
// (c + r/2) mod 8. A 16-byte read serves 16 lanes per pass from 64 four-byte banks (256 bytes):
// two consecutive 128-byte rows already fall in different halves, and the rotation by r/2 puts the
// eight row pairs of a pass on distinct chunks, so a lane-per-row fragment read (every lane the
// same logical chunk) is conflict-free, as with a padded row stride, without the padding's bytes
// (measured: a rotation by r or an XOR by r mod 8 takes twice the cycles).
__device__ __forceinline__ int swz64(int r, int c) { return r * 64 + (((c + (r >> 1)) & 7) << 3); }

// Unpadded LDS rows of 64 bf16 read both ways: by lane-per-row fragment reads and by transposing
// reads (get_trq). Chunk c of row r is stored at chunk c ^ f(r), f(r) = 2 (r mod 4) ^ (r/4 mod 4).
// A 16-byte read of one chunk by 16 consecutive rows (16 lanes per pass over 64 four-byte banks):
// the eight rows of each parity take eight distinct chunks. A transposing read of four consecutive
// rows, an aligned 32-byte column range of each (16 lanes per pass over 32 banks, or 32 lanes over
// 64 banks reading 64 bytes of each row): f(r) / 2 takes four distinct values on the four rows, and
// rows two apart differ in bit 2 of f, so every pass touches distinct banks.
__device__ __forceinline__ int swzq(int r, int c) { return r * 64 + ((c ^ (((r & 3) << 1) ^ ((r >> 2) & 3))) << 3); }

typedef __attribute__((address_space(3))) void* lds_void_ptr;
// The LDS address of a pointer into a __shared__ variable, as the address-space-3 pointer the direct
// loads take: the low 32 bits of the generic address (a plain cast tests the pointer for null, a
// compare and select on the scalar unit per load).
__device__ __forceinline__ lds_void_ptr lds_ptr(const void* p) { return (lds_void_ptr)(uint32_t)(uintptr_t)p; }

// A buffer resource over `bytes` bytes from p (loads past them read zero).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, RSRC_WORD3);
}

// Direct loads into LDS: one instruction fills 64 consecutive 16-byte slots (1 KB) from the given
// LDS base, lane l slot l (measured lane layout on gfx950); each lane reads the global chunk that
// belongs in its slot, through a buffer resource (the scalar offset counts in the range check,
// measured: rows past the resource load zero). A [32][64] bf16 tile takes four such loads, parts
// m = 0..3.
//   rows64: a [32 rows][64] tile in swz64 layout from rows row0.. of a row-major matrix (row stride
//           ld elements). Slot 64m + l holds row 8m + l/8, stored chunk l mod 8, so logical chunk
//           (l mod 8 - l/16 - 4m) mod 8: c0 = (l mod 8 - l/16) mod 8 for even m, c0 ^ 4 for odd m.
// A wavefront always loads the same part m of every tile, so the lane's offset is chosen once, as a
// value (a per-load choice between two fields compiled into a choice of addresses, which kept the
// pair in scratch memory and made every load wait for a scratch read first).
struct RowsLane {
  int v;   // the lane's byte offset for part m
  __device__ __forceinline__ RowsLane(int ld, int lane, int m) {
    const int c0 = ((lane & 7) - (lane >> 4)) & 7;
    v = ((lane >> 3) * ld + 8 * ((m & 1) ? (c0 ^ 4) : c0)) * 2;
  }
};
__device__ __forceinline__ void g2l_rows64(uint16_t* tile, __amdgpu_buffer_rsrc_t rs, const RowsLane& rl, int ld,
                                           int row0, int m) {   // m: the part rl was made for
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, lds_ptr(tile + 512 * m), 16, rl.v, (row0 + 8 * m) * ld * 2, 0,
                                           0);
}
//   rowsq: a [32 rows][64] tile in swzq layout, as rows64. Slot 64m + l holds row r = 8m + l/8,
//          stored chunk l mod 8, so logical chunk (l mod 8) ^ f(r), f(r) = 2 (l/8 mod 4) ^ (l/32)
//          ^ 2 (m mod 2): c0 = (l mod 8) ^ 2 (l/8 mod 4) ^ l/32 for even m, c0 ^ 2 for odd m.
struct RowsLaneQ {
  int v;   // the lane's byte offset for part m (see RowsLane)
  __device__ __forceinline__ RowsLaneQ(int ld, int lane, int m) {
    const int c0 = (lane & 7) ^ (((lane >> 3) & 3) << 1) ^ (lane >> 5);
    v = ((lane >> 3) * ld + 8 * ((m & 1) ? (c0 ^ 2) : c0)) * 2;
  }
};
__device__ __forceinline__ void g2l_rowsq(uint16_t* tile, __amdgpu_buffer_rsrc_t rs, const RowsLaneQ& rl, int ld,
                                          int row0, int m) {   // m: the part rl was made for
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, lds_ptr(tile + 512 * m), 16, rl.v, (row0 + 8 * m) * ld * 2, 0,
                                           0);
}
// An operand of K step s of a product over the rows of a [32 rows][64] swzq tile Y (Y^T X, or X Y):
// lane l gets column 32 db + l % 32 of the tile, rows 16s + 8(l / 32) + 0..7 in order, or with
// CROW the rows a C-layout tile's fragment holds in the accumulator's row order (X entering from
// registers, OpBF16::from_acc): element e is row crow(8s + e, l / 32) = 16s + 8(e / 4) + 4(l / 32)
// + e % 4. Two transposing reads, four rows each: lane i of a 16-lane group gets, as element t,
// element i % 4 of the 8 bytes that lane 4t + i/4 of the group addresses, so lane k of the group
// addresses row base + k/4, columns 4 (k mod 4) .. +3 of the group's 16 (measured lane layout, see
// get_tr).
template <bool CROW>
__device__ __forceinline__ bf16x8 get_trq(const uint16_t* t, int lane, int db, int s) {
  const int g = lane >> 4, k = lane & 15;
  const int c = 4 * db + 2 * (g & 1) + ((k & 3) >> 1);   // the 16-byte chunk of the lane's 4 columns
  bf16x8 f;
#pragma unroll
  for (int hf = 0; hf < 2; ++hf) {
    const int r = CROW ? 16 * s + 8 * hf + 4 * (g >> 1) + (k >> 2) : 16 * s + 8 * (g >> 1) + 4 * hf + (k >> 2);
    typedef __attribute__((address_space(3))) short4v* lds_s4;
    const short4v v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(t + swzq(r, c) + 4 * (k & 1)));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const short x = v[e];
      f[4 * hf + e] = *reinterpret_cast<const bf16_t*>(&x);
    }
  }
  return f;
}
// the wavefront's outstanding vector-memory operations (the direct loads included) have completed
__device__ __forceinline__ void wait_loads() { __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Register-staged tiles for software pipelining: load() issues a tile's global loads into registers
// (each thread owns PER 16-byte chunks), store() later writes them to LDS, so the loads of the next
// tile are in flight while the current one is computed.

// [32 rows][COLS] of a row-major global matrix (row stride gld); rows >= nrows read as zero: the
// loads go through a buffer resource over the nrows rows (nrows * gld elements below 2 GiB, checked
// by the host), so there is no bound check and the offsets are 32-bit (the lane's own part fixed,
// the tile's in a scalar register).
template <typename E, int COLS>
struct RowTile {
  static constexpr int EPC = 16 / sizeof(E);
  static constexpr int CPR = COLS / EPC;
  static constexpr int NCH = TILE * CPR;
  static constexpr int PER = (NCH + NTHREADS - 1) / NTHREADS;
  uint4 v[PER];
  __device__ __forceinline__ void load(const E* g, int64_t gld, int row0, int nrows, int tid) {
    const int ld = (int)gld;
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)g, 0, nrows * ld * (int)sizeof(E), RSRC_WORD3);
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int c = (tid + p * NTHREADS) % NCH;   // PER * NTHREADS > NCH only for small tiles
      const int r = c / CPR, cc = (c % CPR) * EPC;
      const auto x = __builtin_amdgcn_raw_buffer_load_b128(rs, (r * ld + cc) * (int)sizeof(E),
                                                           row0 * ld * (int)sizeof(E), 0);
      v[p] = make_uint4(x[0], x[1], x[2], x[3]);
    }
  }
  template <int SLD>
  __device__ __forceinline__ void store(E* s, int tid) const {
    static_assert((SLD * sizeof(E)) % 16 == 0, "row stride must keep 16-byte alignment");
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int c = tid + p * NTHREADS;
      const int r = (c % NCH) / CPR, cc = (c % CPR) * EPC;
      if (NCH % NTHREADS == 0 || c < NCH) *reinterpret_cast<uint4*>(s + r * SLD + cc) = v[p];
    }
  }
};

// Columns col0..col0+31 of ROWS rows of one of this library's transposed copies: row stride gld,
// a multiple of 64 elements, zero-filled past the sequence, so every 16-byte chunk is in bounds and
// the load needs no check. Buffer loads as for RowTile: 32-bit offsets, the lane's part fixed.
template <typename E, int ROWS>
struct ColTile {
  static constexpr int EPC = 16 / sizeof(E);
  static constexpr int CPR = TILE / EPC;
  static constexpr int NCH = ROWS * CPR;
  static constexpr int PER = (NCH + NTHREADS - 1) / NTHREADS;
  uint4 v[PER];
  __device__ __forceinline__ void load(const E* g, int64_t gld, int col0, int tid) {
    const int ld = (int)gld;
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)g, 0, ROWS * ld * (int)sizeof(E), RSRC_WORD3);
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int c = (tid + p * NTHREADS) % NCH;
      const int r = c / CPR, cc = (c % CPR) * EPC;
      const auto x = __builtin_amdgcn_raw_buffer_load_b128(rs, (r * ld + cc) * (int)sizeof(E),
                                                           col0 * (int)sizeof(E), 0);
      v[p] = make_uint4(x[0], x[1], x[2], x[3]);
    }
  }
  template <int SLD>
  __device__ __forceinline__ void store(E* s, int tid) const {
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int c = tid + p * NTHREADS;
      const int r = (c % NCH) / CPR, cc = (c % CPR) * EPC;
      if (!(NCH % NTHREADS == 0 || c < NCH)) continue;
      E* dst = s + r * SLD + cc;
      if constexpr (sizeof(E) == 2) {
        static_assert((SLD * 2) % 8 == 0, "bf16 column tiles need 8-byte row alignment");
        reinterpret_cast<uint2*>(dst)[0] = make_uint2(v[p].x, v[p].y);
        reinterpret_cast<uint2*>(dst)[1] = make_uint2(v[p].z, v[p].w);
      } else {
        union { uint4 q; E e[EPC]; } u;
        u.q = v[p];
#pragma unroll
        for (int e = 0; e < EPC; ++e) dst[e] = u.e[e];
      }
    }
  }
  // bf16: the columns of each 16-column block in C-layout row order -- groups of four columns
  // 0, 2, 1, 3 -- so OpBF16::ld_perm reads a fragment with one 16-byte read; fp32 as store().
  template <int SLD>
  __device__ __forceinline__ void store_crow(E* s, int tid) const {
    if constexpr (sizeof(E) != 2) {
      store<SLD>(s, tid);
    } else {
      static_assert((SLD * 2) % 16 == 0, "C-layout-order tiles need 16-byte row alignment");
#pragma unroll
      for (int p = 0; p < PER; ++p) {
        const int c = tid + p * NTHREADS;
        const int r = (c % NCH) / CPR, cc = (c % CPR) * EPC;
        if (!(NCH % NTHREADS == 0 || c < NCH)) continue;
        // cc is a multiple of 8: its groups of four are 2(cc%16)/8 and that + 1, at 0 -> 0, 1 -> 2,
        // 2 -> 1, 3 -> 3
        const int a0 = (cc & 15) >> 2;
        const int a1 = a0 + 1;
        E* row = s + r * SLD + (cc & ~15);
        reinterpret_cast<uint2*>(row + 4 * (((a0 & 1) << 1) | (a0 >> 1)))[0] = make_uint2(v[p].x, v[p].y);
        reinterpret_cast<uint2*>(row + 4 * (((a1 & 1) << 1) | (a1 >> 1)))[0] = make_uint2(v[p].z, v[p].w);
      }
    }
  }
};

// ---------------------------------------------------------------------------------------------
// Lane scans (DPP) across the 32 lanes of each half-wavefront.

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_shift(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xF, true));
}

// Exclusive prefix sums over lanes 0..31 and, separately, 32..63, of 16 values at once, step by step
// across the 16 (each DPP step then has 16 independent instructions and no read-after-write
// hazard waits between them).
__device__ __forceinline__ void excl_scan32x16(f32x16& x) {
  f32x16 s = x;
#pragma unroll
  for (int i = 0; i < 16; ++i) s[i] += dpp_shift<0x111, 0xF>(s[i]);   // row_shr:1
#pragma unroll
  for (int i = 0; i < 16; ++i) s[i] += dpp_shift<0x112, 0xF>(s[i]);   // row_shr:2
#pragma unroll
  for (int i = 0; i < 16; ++i) s[i] += dpp_shift<0x114, 0xF>(s[i]);   // row_shr:4
#pragma unroll
  for (int i = 0; i < 16; ++i) s[i] += dpp_shift<0x118, 0xF>(s[i]);   // row_shr:8
#pragma unroll
  for (int i = 0; i < 16; ++i) s[i] += dpp_shift<0x142, 0xA>(s[i]);   // row_bcast:15 into rows 1, 3
#pragma unroll
  for (int i = 0; i < 16; ++i) x[i] = s[i] - x[i];
}

// Exclusive prefix sum over lanes 0..31 and, separately, 32..63.
__device__ __forceinline__ float excl_scan32(float x) {
  float s = x;
  s += dpp_shift<0x111, 0xF>(s);   // row_shr:1
  s += dpp_shift<0x112, 0xF>(s);   // row_shr:2
  s += dpp_shift<0x114, 0xF>(s);   // row_shr:4
  s += dpp_shift<0x118, 0xF>(s);   // row_shr:8
  s += dpp_shift<0x142, 0xA>(s);   // row_bcast:15 into rows 1 and 3
  return s - x;
}

// ---------------------------------------------------------------------------------------------
// One key block's selection summed over a query block: acc holds the raw logits (queries x keys, C
// layout, lane = key j; element i is the block's query crow(i, h)), relu'd in unscaled logit units
// (relu(s x) = s relu(x), s > 0); on tiles that are not interior, only the pairs with
// exempt <= j < query count: crow(i, 0) > thr, thr = j - (first query of the block) - 4h (32 when j
// is exempt). Queries past the end and keys past the end hold zero rows, so their logits add
// nothing. Summed in a fixed tree order, the wavefront's halves added, times the scale (the same
// value in both lanes of key j). The column-sum and one-pass carry kernels both take it, so their
// sums agree bit for bit.
__device__ __forceinline__ float block_selection_sum(const f32x16& acc, bool interior, int thr, float scale) {
  f32x16 s;
#pragma unroll
  for (int i = 0; i < 16; ++i) s[i] = __builtin_amdgcn_fmed3f(acc[i], 0.f, 3.0e38f);
  if (!interior) {
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = crow(i, 0) > thr ? s[i] : 0.f;
  }
  float p[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) p[i] = s[2 * i] + s[2 * i + 1];
#pragma unroll
  for (int i = 0; i < 4; ++i) p[i] = p[2 * i] + p[2 * i + 1];
  const Halves cs = halves((p[0] + p[1]) + (p[2] + p[3]));
  return (cs.lo + cs.hi) * scale;
}

// ---------------------------------------------------------------------------------------------
// Skipping key tiles that carry no weight. F only grows with the query, so once a key's history has
// outgrown its logit by enough, its softmax weight is an exact fp32 zero for every later query, and so
// are its terms in every sum it enters. For a tile of keys and a block of queries,
//
//     log2 weight <= s log2e (max |q|) (max |k|) - log2e (min F) - (min row maximum so far),
//
// and v_exp_f32 returns exactly zero below -126 (it flushes denormal results). A tile whose bound lies
// below -REACH_ZERO (a margin for the rounding of the bound's own terms; besides, the norms are taken 1%
// high and F a thousandth low) is left out of the sweep: the skipped terms are zeros, so the results keep
// their bits. Nothing is skipped where a zero weight would not give a zero term: a tile with a key or value
// that is not finite, or so large that a product of two rows could overflow, gets the bound infinity,
// and every comparison is written so that a NaN keeps the tile.
// Measured (forward kernel, bf16, D=64, N(0,1) inputs, whose histories grow by 0.4 a query): B=1 H=16
// T=16384 918 -> 97 us, the last 16384 queries of 131072 13.2 -> 0.17 ms, B=2 H=12 T=2048 85 -> 35 us; where
// one pair in a hundred is selected and nothing can be left out: B=2 H=12 T=5003 249 -> 250 us, B=1 H=12
// T=16384 740 -> 751 us, and the key norms add 2 and 6 us to the column sums' launch.
constexpr float REACH_ZERO = 132.f;
constexpr float REACH_WORTH = REACH_ZERO - 16.f;   // a total (log2 units) from which looking for tiles can pay
constexpr float REACH_NORM2 = 1e37f;      // sums of squares at or past this count as not finite
constexpr float REACH_Q = 1.01f * LOG2E;
constexpr float REACH_F = 0.999f * LOG2E;
constexpr int NORM_KEYS = 256;            // keys per workgroup of the norms

// The sum of squares of 8 elements of a row.
template <typename E>
__device__ __forceinline__ float sumsq8(const E* p) {
  float s = 0.f;
  if constexpr (sizeof(E) == 2) {
    const uint4 u = *reinterpret_cast<const uint4*>(p);
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float lo = __uint_as_float(w[i] << 16), hi = __uint_as_float(w[i] & 0xFFFF0000u);
      s = fmaf(lo, lo, s);
      s = fmaf(hi, hi, s);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float4 f = reinterpret_cast<const float4*>(p)[i];
      s = fmaf(f.x, f.x, fmaf(f.y, f.y, fmaf(f.z, f.z, fmaf(f.w, f.w, s))));
    }
  }
  return s;
}

// kn[r][kt] = max |k_j| over the keys of tile kt of head r = b * H + head, infinity when a key or a
// value of the tile is not finite (or too large, REACH_NORM2), and, unread, for the tiles that no query is
// likely to leave out: wanted(kt), asked of the lane half's tile, false (only the time depends on it).
// Workgroup `blk` takes NORM_KEYS keys of head r: a wavefront two tiles, D/8 lanes per row, a tile's loads
// all issued before their use. Bound by HBM (each key and value read once).
template <typename E, int D, class Wanted>
__device__ __forceinline__ void key_norms_block(const E* k, const E* v, const Strides& ks, const Strides& vs, int H,
                                                int Tk, float* kn, int r, int blk, Wanted wanted) {
  constexpr int LPR = D / 8, RPW = 64 / LPR, PASSES = TILE / RPW;
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int NKT = (Tk + TILE - 1) / TILE;
  const E* kh = k + ks.at(r / H, r % H) + (lane % LPR) * 8;
  const E* vh = v + vs.at(r / H, r % H) + (lane % LPR) * 8;
  const int kt0 = blk * (NORM_KEYS / TILE) + wave * 2;
  if (kt0 >= NKT) return;
  const uint64_t want = __ballot(wanted(min(kt0 + (lane >> 5), NKT - 1)));
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int kt = kt0 + u;
    if (kt >= NKT) break;
    if (((want >> (32 * u)) & 1) == 0) {
      if (lane == 0) kn[(int64_t)r * NKT + kt] = INFINITY;
      continue;
    }
    float sk[PASSES], sv[PASSES];
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      const int64_t j = min(kt * TILE + p * RPW + lane / LPR, Tk - 1);   // (the last key again past the end)
      sk[p] = sumsq8(kh + j * ks.row);
      sv[p] = sumsq8(vh + j * vs.row);
    }
    float mx = 0.f;
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
#pragma unroll
      for (int o = LPR / 2; o > 0; o >>= 1) {
        sk[p] += __shfl_xor(sk[p], o);
        sv[p] += __shfl_xor(sv[p], o);
      }
      mx = fmaxf(mx, (sk[p] < REACH_NORM2 && sv[p] < REACH_NORM2) ? sk[p] : INFINITY);
    }
#pragma unroll
    for (int o = LPR; o < 64; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    if (lane == 0) kn[(int64_t)r * NKT + kt] = sqrtf(mx);
  }
}

// The norms in a launch of their own, after the selection: of the tiles whose least total (kt_min) is enough.
template <typename E, int D>
__global__ __launch_bounds__(NTHREADS) void key_norms_kernel(const E* __restrict__ k, const E* __restrict__ v, Strides ks,
                                                             Strides vs, int H, int Tk, float* __restrict__ kn,
                                                             const float* __restrict__ kt_min) {
  const float* totals = kt_min + (int64_t)(blockIdx.y / H) * ((Tk + TILE - 1) / TILE);
  key_norms_block<E, D>(k, v, ks, vs, H, Tk, kn, blockIdx.y, blockIdx.x,
                        [&](int kt) { return totals[kt] * LOG2E > REACH_WORTH; });
}

// The maximum over the 32 lanes of each half-wavefront (those of them that are active).
__device__ __forceinline__ float half_max(float x) {
#pragma unroll
  for (int o = 1; o < 32; o <<= 1) x = fmaxf(x, __shfl_xor(x, o));
  return x;
}

__device__ __forceinline__ uint64_t uniform64(uint64_t x) {
  return ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(x >> 32)) << 32) |
         (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x);
}

// The tiles a workgroup has to visit, newest first, as runs of consecutive tiles: a sweep counts down
// within a run and takes the next one from LDS at its end (a tile list or a bit mask walked in the tile
// loop cost it 2% where nothing is skipped, in scalar instructions and spilled scalar registers).
struct TileRun {
  int hi, lo;
};
constexpr int REACH_RUNS = 64;   // entries of the list

// The set bits of the words (bit i of word w: tile first + 64 w + i), then the tiles below first, as runs
// ending in {-1, INT_MIN}, below which a sweep finds no tile. What the list does not hold -- the tiles below
// first, and whatever is left once it is full -- becomes one run down to tile 0 with REST (for a reader to
// whom a tile too many costs time only: the forward), else an entry {-2, INT_MIN}, at which the reader
// has to look for itself. One wavefront.
template <bool REST>
__device__ __forceinline__ void write_reach_runs(TileRun* runs, const uint64_t* words, int nwords, int first, int lane) {
  int n = 0;
  TileRun open{-1, -1};
  bool more = first > 0;   // (not REST)
  auto add = [&](int hi, int lo) {
    if (open.hi >= 0 && hi == open.lo - 1) {
      open.lo = lo;
      return;
    }
    if (open.hi >= 0) {
      if (lane == 0) runs[n] = open;
      ++n;
    }
    open = {hi, lo};
  };
  int w = nwords;
  while (w > 0) {   // the newest word before w that holds a tile, 64 words at a time
    const int base = max(w - 64, 0);
    const uint64_t some = __ballot(base + lane < w && words[min(base + lane, w - 1)] != 0);
    if (some == 0) {
      w = base;
      continue;
    }
    w = base + 63 - __builtin_clzll(some);
    uint64_t word = uniform64(words[w]);
    while (word != 0) {
      const int bit = 63 - __builtin_clzll(word);
      const uint64_t gaps = ~word << (63 - bit);
      const int len = min(gaps != 0 ? __builtin_clzll(gaps) : 64, bit + 1);
      add(first + 64 * w + bit, first + 64 * w + bit - len + 1);
      word &= (bit - len >= 0) ? (2ull << (bit - len)) - 1 : 0;
      if (n == REACH_RUNS - 2) {   // full, with the open run and the ending
        if constexpr (REST) open.lo = 0;
        else more = true;
        word = 0;
        w = 0;
        first = 0;
      }
    }
  }
  if constexpr (REST) {
    if (first > 0) add(first - 1, 0);
  }
  if (lane == 0) {
    if (open.hi >= 0) runs[n++] = open;
    runs[n] = {!REST && more ? -2 : -1, INT_MIN};
  }
}

// Whether looking for tiles to skip can pay: every key of one of the 64 oldest tiles has received enough by
// the sequence's end. total: this lane's such tile's least selection total (reach_total, loaded before
// the sweep so that it costs no wait). Only the time depends on the answer.
__device__ __forceinline__ float reach_total(const float* kt_min, int ntiles, int lane) {
  return kt_min != nullptr && lane < ntiles ? kt_min[lane] : 0.f;
}
__device__ __forceinline__ bool reach_worth(float total) { return __any(total * LOG2E > REACH_WORTH); }

// Sum of squares of a lane's part of its query row.
template <class OP, int NS>
__device__ __forceinline__ float frag_sumsq(const typename OP::frag (&f)[NS]) {
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    if constexpr (OP::KS == 16) {
#pragma unroll
      for (int e = 0; e < 8; ++e) s = fmaf((float)f[i][e], (float)f[i][e], s);
    } else {
      s = fmaf(f[i], f[i], s);
    }
  }
  return s;
}

// The key tiles below `cut` that a forward workgroup has to visit, as runs (write_reach_runs), once its
// diagonal tiles are behind it: qf the lane's parts of its query of each head, m the query's running
// maximum (log2 units), row whether there is such a query; kn the first head's key norms, the next
// heads' NKT apart; kt_min the least selection total of each tile; crow the carry row of the workgroup's first query block (later
// blocks' histories are no smaller). The tiles below i_lo (exempt keys have no history) are always visited. A lane decides a
// tile by its 128 carry bytes (eight 16-byte loads; past the row's end they read zero, which keeps the
// tile), a wavefront every fourth word of 64 tiles; the tiles older than the words hold are visited.
// All wavefronts of the workgroup; the runs may be read on return.
template <class OP, int G, int NS>
__device__ __forceinline__ void find_reach(const typename OP::frag (&qf)[G][NS], const float (&m)[G], bool row,
                                           float scale, const float* kn, const float* kt_min, int NKT,
                                           const float* crow, int Tk, int cut,
                                           int i_lo, float (*bound)[2 * G], uint64_t* words, TileRun* runs, int lane,
                                           int wave) {
#pragma unroll
  for (int g = 0; g < G; ++g) {
    float qn = frag_sumsq<OP, NS>(qf[g]);
    qn += xor32(qn);
    qn = half_max(qn < REACH_NORM2 ? qn : INFINITY);
    const float ml = -half_max(row ? (m[g] > -3.0e38f ? -m[g] : INFINITY) : -INFINITY);
    if (lane == 0) {
      bound[wave][2 * g] = sqrtf(qn);
      bound[wave][2 * g + 1] = ml;
    }
  }
  __syncthreads();
  float a[G], b[G];   // log2 weight <= a kn + b - F log2e - REACH_ZERO for every query of the workgroup
#pragma unroll
  for (int g = 0; g < G; ++g) {
    float qn = bound[0][2 * g], ml = bound[0][2 * g + 1];
#pragma unroll
    for (int w = 1; w < NWAVES; ++w) {
      qn = fmaxf(qn, bound[w][2 * g]);
      ml = fminf(ml, bound[w][2 * g + 1]);
    }
    a[g] = qn * scale * REACH_Q;
    b[g] = REACH_ZERO - ml;
  }
  const int all = (cut + 63) / 64, nwords = min(all, REACH_MASK_WORDS), first = 64 * (all - nwords);
  const __amdgpu_buffer_rsrc_t rs =
      __builtin_amdgcn_make_buffer_rsrc((void*)crow, 0, (int)((int64_t)Tk * 4), RSRC_WORD3);
  for (int w = wave; w < nwords; w += NWAVES) {
    const int kt = first + 64 * w + lane, ktc = min(kt, cut - 1);
    bool skip = kt >= i_lo && kt < cut;   // every comparison that meets a NaN keeps the tile
    float thr = -INFINITY;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float t = fmaf(a[g], kn[(int64_t)g * NKT + ktc], b[g]);
      skip = skip && t < INFINITY;
      thr = fmaxf(thr, t);
    }
    skip = skip && kt_min[ktc] * REACH_F > thr;   // (its total is at least its history at any query)
    if (__any(skip)) {
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const auto x = __builtin_amdgcn_raw_buffer_load_b128(rs, ktc * (TILE * 4) + 16 * c, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) skip = skip && __uint_as_float(x[e]) * REACH_F > thr;
      }
    }
    const uint64_t bits = __ballot(kt < cut && !skip);
    if (lane == 0) words[w] = bits;
  }
  __syncthreads();
  if (wave == 0) write_reach_runs<true>(runs, words, nwords, first, lane);
  __syncthreads();
}

// ---------------------------------------------------------------------------------------------
// Selection column sums: colsum[b][rb][j] = sum over the queries r of block rb (chunk-relative)
// of S[r, j]. One wavefront per key block (its K rows in registers); a workgroup walks RB query
// blocks, each staged once in LDS for its four wavefronts while the next one loads. The grid's z past the
// sequences takes the key norms (key_norms_block) of all heads along: work of the same launch that the
// forward needs next to the carry, in place of a launch of its own (2-3 us), where the grid has room for them.
constexpr int SEL_RB = 8;   // query blocks per workgroup

template <class OP, int D>
__global__ __launch_bounds__(NTHREADS) void sel_colsum_kernel(
    const typename OP::elem* __restrict__ q, const typename OP::elem* __restrict__ k,
    float* __restrict__ colsum, int H, int Tq, int Tk, Strides qs, Strides ks, int q_off, int exempt, float scale,
    int RB, const typename OP::elem* __restrict__ v, Strides vs, int nseq, float* __restrict__ kn,
    const float* __restrict__ state_in, int64_t state_ld) {
  using elem = typename OP::elem;
  if ((int)blockIdx.z >= nseq) {
    const int nkb = (Tk + NORM_KEYS - 1) / NORM_KEYS;
    const int64_t e = ((int64_t)(blockIdx.z - nseq) * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
    if (e >= (int64_t)nseq * H * nkb) return;
    const int r = (int)(e / nkb);
    // The totals are not known yet. Of a tile before the chunk, what its keys have received is, and with it about
    // what the chunk's queries will add: half as much again per query as so far, to be on the safe side. At head
    // dim 128, where it pays: B=1 H=16, 256 queries over 16384 keys, nothing left out 693 -> 676 us, most left out
    // 74.9 -> 75.2; at 64 (half the bytes) 461 -> 457 and 36.8 -> 38.0.
    key_norms_block<elem, D>(k, v, ks, vs, H, Tk, kn, r, (int)(e % nkb), [&](int kt) {
      const int age = q_off - kt * TILE;   // the queries the tile's first key has seen, and itself
      if (D < 128 || state_in == nullptr || age < NORM_KEYS) return true;
      const float least = -half_max(-state_in[(int64_t)(r / H) * state_ld + kt * TILE + (threadIdx.x & 31)]);
      return least * (1.f + 1.5f * (float)Tq / (float)age) * LOG2E > REACH_WORTH;
    });
    return;
  }
  using frag = typename OP::frag;
  constexpr int NS = D / OP::KS;
  constexpr int LDK = D + OP::KPAD;
  __shared__ __attribute__((aligned(16))) elem sQ[2][TILE * LDK];   // query blocks, double-buffered
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int n = lane & 31, h = lane >> 5;
  const int NKT = (Tk + TILE - 1) / TILE;
  const int NBq = (Tq + TILE - 1) / TILE;
  const int kb = blockIdx.x * NWAVES + wave;   // (a wavefront past the last key block only stages)
  const int b = blockIdx.z;
  const elem* q0 = q + qs.at(b, 0);
  const elem* k0 = k + ks.at(b, 0);
  const int j = kb * TILE + n;
  const int kbase = kb * TILE;

  frag kf[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) kf[s] = ld_std_bounded<OP>(k0, ks.row, kbase + n, Tk, h, s);
  // a tile is interior when every pair passes: keys before every query, not exempt, queries
  // before the end (keys past the end hold zero rows, their sums are never written)
  const int rb0 = blockIdx.y * RB, rb_end = min(NBq, rb0 + RB);
  RowTile<elem, D> nQ;
  if (rb0 < rb_end) {
    nQ.load(q0, qs.row, rb0 * TILE, Tq, tid);
    nQ.template store<LDK>(sQ[0], tid);
  }
  __syncthreads();
  for (int rb = rb0; rb < rb_end; ++rb) {
    const int buf = (rb - rb0) & 1;
    // the next block, into registers, unconditionally (past the end it reads zero rows, unused): a
    // conditional load made the compiler wait for it at the join before this block's products
    nQ.load(q0, qs.row, (rb + 1) * TILE, Tq, tid);
    float cs = 0.f;
    const int qbase = q_off + rb * TILE;   // absolute position of the block's first query
    // the tile holds a selectable pair only if some query is after the first key
    if (kb < NKT && qbase + TILE - 1 > kbase) {
      f32x16 acc = zero16();
#pragma unroll
      for (int s = 0; s < NS; ++s) acc = OP::mma(OP::ld_std(sQ[buf], LDK, n, h, s), kf[s], acc);
      const bool interior = qbase > kbase + TILE - 1 && kbase >= exempt;
      cs = block_selection_sum(acc, interior, j >= exempt ? j - qbase - 4 * h : 32, scale);
    }
    if (kb < NKT && h == 0 && j < Tk) colsum[((int64_t)b * NBq + rb) * Tk + j] = cs;
    if (rb + 1 < rb_end) nQ.template store<LDK>(sQ[buf ^ 1], tid);
    __syncthreads();
  }
}

// carry[b][rb][j] = state_in[b][j] + sum_{rb' < rb} colsum[b][rb'][j] (in place);
// state_out[b][j] = the sum over all blocks. state_in is read for j < q_off only. kt (may be NULL):
// the smallest of them in each key tile (of its 32 keys: a last tile with fewer holds no such figure).
__global__ __launch_bounds__(NTHREADS) void sel_scan_kernel(
    float* __restrict__ carry, const float* state_in, float* state_out, int64_t state_ld,
    int NBq, int Tk, int q_off, float* __restrict__ kt) {
  const int j = blockIdx.x * NTHREADS + threadIdx.x;
  const int b = blockIdx.y;
  if (j >= Tk) return;
  float run = (state_in != nullptr && j < q_off) ? state_in[(int64_t)b * state_ld + j] : 0.f;
  float* col = carry + (int64_t)b * NBq * Tk + j;
  constexpr int U = 16;   // blocks per step: their loads are issued together
  int rb = 0;
  for (; rb + U <= NBq; rb += U) {
    float c[U];
#pragma unroll
    for (int u = 0; u < U; ++u) c[u] = col[(int64_t)(rb + u) * Tk];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      col[(int64_t)(rb + u) * Tk] = run;
      run += c[u];
    }
  }
  for (; rb < NBq; ++rb) {
    const float c = col[(int64_t)rb * Tk];
    col[(int64_t)rb * Tk] = run;
    run += c;
  }
  state_out[(int64_t)b * state_ld + j] = run;
  if (kt) {   // (lanes past the last key have left: a half-wavefront's first lane is never one of them)
    const float mn = -half_max(-run);
    if ((threadIdx.x & 31) == 0) kt[(int64_t)b * ((Tk + TILE - 1) / TILE) + j / TILE] = mn;
  }
}

// The selection carry in one pass, for bf16 storage at head dim 64 when the call has key blocks
// enough for a workgroup per CU (many sequences, as in the per-head mode where every head is its own
// sequence, or a long key range, as in the later chunks of a chunked prefill). grid
// (ceil(NKT/(4 KPW)), nseq): wavefront w owns key blocks (4x + w) KPW + u, u < KPW (their K rows in
// registers, one read of each query fragment serving all of them), and the workgroup walks the
// query blocks from the first that can select one of its keys to the last, each staged once into
// LDS by direct loads issued NBUF - 1 blocks ahead (NBUF buffers, one barrier per block), keeping
// each key's running selection in a register. carry[b][rb][j] is stored on entry to block rb (the
// rows before the first block hold the entering value, state_in or zero, as the scan writes them)
// and state_out[b][j] after the last. Each block's sum is block_selection_sum, as in the column-sum
// kernel, and the sums are added in the scan's order: both paths give the same bits, without the
// column sums' round trip through HBM.
//
// Every block issues the same vector-memory operations -- KPW carry stores through a buffer
// resource (lanes that own no key aim past its end, where the store is dropped) and one query-block
// load (past the last block: zero rows into a buffer nobody reads) -- so a fixed count
// vmcnt((NBUF - 2) (KPW + 1)) at the end of a block waits exactly for the next block's load (the
// counter drains in issue order).
constexpr int SEL_CARRY_KPW = 1;             // key blocks per wavefront
constexpr int SEL_CARRY_NBUF = 4;            // query-block buffers
constexpr int SEL_CARRY_MIN_BLOCKS = 256;    // workgroups below which the two-kernel path runs

__global__ __launch_bounds__(NTHREADS) void sel_carry64_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, float* __restrict__ carry,
    const float* state_in, float* state_out, int64_t state_ld, int Tq, int Tk, Strides qs, Strides ks, int q_off,
    int exempt, float scale, float* __restrict__ kt) {
  using OP = OpBF16;
  using frag = OP::frag;
  constexpr int D = 64, NS = 4, KPW = SEL_CARRY_KPW, NBUF = SEL_CARRY_NBUF, AHEAD = NBUF - 1;
  static_assert(NBUF == 4, "the block loop names four buffers");
  // separate LDS variables, named at compile time, so the compiler knows a block's reads do not
  // touch the buffers the direct loads are filling.
  // Lifetimes (block rb_lo + t lives in buffer t mod 4):
  //   filled: by the direct load g2l_rows64 of every wavefront (a quarter each), for blocks rb_lo,
  //           +1, +2 in the prologue, for block rb + 3 in step t (block rb) -- into the buffer that
  //           held block rb - 1;
  //   drained: by the qa fragment reads of step t only;
  //   separated: the reads of block rb - 1 (step t - 1) from the fill in step t by the end of step
  //           t - 1: lgkmcnt(0) (this wavefront's reads done) and s_barrier (every wavefront's);
  //           the fill of block rb (step t - 3, or the prologue's vmcnt(0)) from its reads by the
  //           vmcnt(4) of step t - 1 (of the 2 per step issued after it, only the last two steps'
  //           may be outstanding) and the same barrier. The peeled last steps keep the count (loads
  //           past the last block read zero rows into buffers nobody reads), and wait_loads() at
  //           the end leaves no load in flight into LDS when the workgroup ends.
  __shared__ __attribute__((aligned(16))) uint16_t sQ0[TILE * D];
  __shared__ __attribute__((aligned(16))) uint16_t sQ1[TILE * D];
  __shared__ __attribute__((aligned(16))) uint16_t sQ2[TILE * D];
  __shared__ __attribute__((aligned(16))) uint16_t sQ3[TILE * D];
  auto sbuf = [&](auto idx) -> uint16_t* {
    constexpr int I = decltype(idx)::value % NBUF;
    if constexpr (I == 0) return sQ0;
    else if constexpr (I == 1) return sQ1;
    else if constexpr (I == 2) return sQ2;
    else return sQ3;
  };
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int n = lane & 31, h = lane >> 5;
  const int NKT = (Tk + TILE - 1) / TILE;
  const int NBq = (Tq + TILE - 1) / TILE;
  const BlockXY bxy = xcd_block();   // each XCD takes whole sequences: their query rows stay in its L2
  const int b = bxy.y;
  const int kb0 = bxy.x * (NWAVES * KPW);
  const uint16_t* q0 = q + qs.at(b, 0);
  const uint16_t* k0 = k + ks.at(b, 0);
  float* plane = carry + (int64_t)b * NBq * Tk;
  const int plane_bytes = NBq * Tk * 4;   // below 2 GiB (the launch checks)
  const __amdgpu_buffer_rsrc_t rs_c = rsrc(plane, plane_bytes);

  // per key block u of the wavefront (blocks past the last one only stage): key j, whether this
  // lane stores key j's values (and the byte offset its stores take: past the plane if not), its
  // K rows, its running selection
  int kb[KPW], jj[KPW], voff[KPW];
  bool owner[KPW];
  frag kf[KPW][NS];
  float run[KPW];
#pragma unroll
  for (int u = 0; u < KPW; ++u) {
    kb[u] = kb0 + wave * KPW + u;
    jj[u] = kb[u] * TILE + n;
    owner[u] = kb[u] < NKT && h == 0 && jj[u] < Tk;
    voff[u] = owner[u] ? jj[u] * 4 : plane_bytes;
#pragma unroll
    for (int s = 0; s < NS; ++s) kf[u][s] = ld_std_bounded<OP>(k0, ks.row, jj[u], Tk, h, s);
    run[u] = (state_in != nullptr && jj[u] < q_off && jj[u] < Tk) ? state_in[(int64_t)b * state_ld + jj[u]] : 0.f;
  }

  // blocks before rb_lo end before the workgroup's first key: no pair of theirs is selectable
  const int lead = kb0 * TILE - q_off;
  const int rb_lo = min(lead > 0 ? lead / TILE : 0, NBq);
#pragma unroll
  for (int u = 0; u < KPW; ++u)
    if (owner[u])
      for (int rb = 0; rb < rb_lo; ++rb) plane[(int64_t)rb * Tk + jj[u]] = run[u];

  const int q_ld = (int)qs.row;
  const __amdgpu_buffer_rsrc_t rs_q = rsrc(q0, (int64_t)Tq * q_ld * 2);   // rows past Tq read zero
  const RowsLane rl_q(q_ld, lane, wave);
  const int nb = NBq - rb_lo;   // blocks walked; block rb_lo + t sits in buffer t mod NBUF
  g2l_rows64(sQ0, rs_q, rl_q, q_ld, rb_lo * TILE, wave);
  g2l_rows64(sQ1, rs_q, rl_q, q_ld, (rb_lo + 1) * TILE, wave);
  g2l_rows64(sQ2, rs_q, rl_q, q_ld, (rb_lo + 2) * TILE, wave);
  wait_loads();
  __syncthreads();

  auto step = [&](int t, auto buf_tag) {
    constexpr int BUF = decltype(buf_tag)::value;
    const int rb = rb_lo + t;
#pragma unroll
    for (int u = 0; u < KPW; ++u)   // the value on entry to the block
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(run[u]), rs_c, voff[u], rb * Tk * 4, 0);
    g2l_rows64(sbuf(std::integral_constant<int, BUF + AHEAD>{}), rs_q, rl_q, q_ld, (rb + AHEAD) * TILE, wave);
    const uint16_t* sQ = sbuf(buf_tag);
    const int qbase = q_off + rb * TILE;
    frag qa[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) qa[s] = *reinterpret_cast<const frag*>(sQ + swz64(n, 2 * s + h));
#pragma unroll
    for (int u = 0; u < KPW; ++u) {
      const int kbase = kb[u] * TILE;
      if (kb[u] < NKT && qbase + TILE - 1 > kbase) {
        f32x16 acc = zero16();
#pragma unroll
        for (int s = 0; s < NS; ++s) acc = OP::mma(qa[s], kf[u][s], acc);
        const bool interior = qbase > kbase + TILE - 1 && kbase >= exempt;
        run[u] += block_selection_sum(acc, interior, jj[u] >= exempt ? jj[u] - qbase - 4 * h : 32, scale);
      }
    }
    // The next block's load is in (the loads and stores issued after it may still run), this
    // block's LDS reads are done, then the barrier: as one asm block, since before a compiler-seen
    // barrier the compiler waits for every direct load into LDS, the ones ahead included.
    __asm__ volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((AHEAD - 1) * (KPW + 1)) : "memory");
  };
  int t = 0;
  for (; t + 3 < nb; t += 4) {
    step(t, std::integral_constant<int, 0>{});
    step(t + 1, std::integral_constant<int, 1>{});
    step(t + 2, std::integral_constant<int, 2>{});
    step(t + 3, std::integral_constant<int, 3>{});
  }
  if (t < nb) step(t, std::integral_constant<int, 0>{});
  if (t + 1 < nb) step(t + 1, std::integral_constant<int, 1>{});
  if (t + 2 < nb) step(t + 2, std::integral_constant<int, 2>{});
  wait_loads();   // nothing may be left in flight into LDS when the workgroup ends
#pragma unroll
  for (int u = 0; u < KPW; ++u) {
    if (owner[u]) state_out[(int64_t)b * state_ld + jj[u]] = run[u];
    if (kt) {
      const float mn = -half_max(owner[u] ? -run[u] : -INFINITY);
      if (lane == 0 && kb[u] < NKT) kt[(int64_t)b * NKT + kb[u]] = mn;
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Forward. grid (ceil(NBq/4), nseq * H/G); wavefront w of block x owns query block
// (gridDim.x-1-x)*4 + w (heavy causal rows launch first) of heads [gi*G, gi*G+G). Key tiles are
// visited newest first, so each row's maximum is usually settled by its diagonal tile and later
// tiles rarely trigger a rescale of the output (skipped when no lane's maximum rises). Tiles whose keys
// carry no weight any more are left out (find_reach). The next tile's K, V^T and carry rows are loaded while the current one is computed (double-buffered LDS).

// Workgroups per CU the forward's register allocation must allow: three at bf16 head dims <= 64
// with one head per wavefront (its LDS fits three), which holds it to 168 registers without spills.
template <class OP, int D, int G>
constexpr int fwd_min_blocks() { return (sizeof(typename OP::elem) == 2 && D <= 64 && G == 1) ? 3 : 1; }

// CV ("contiguous views"): q rows are D apart and its heads Tq * D apart, k rows D apart and its
// heads ks.head apart -- the layout of sa_forward; the view strides are then compile-time facts
// (fewer scalar registers live in the tile loop). Other views take the general instance.
template <class OP, int D, int G, bool CV>
__global__ __launch_bounds__(NTHREADS, (fwd_min_blocks<OP, D, G>())) void fwd_kernel(
    const typename OP::elem* __restrict__ q, const typename OP::elem* __restrict__ k,
    const typename OP::elem* __restrict__ vt, const float* __restrict__ carry,
    float* __restrict__ out, float* __restrict__ rmax, float* __restrict__ rden,
    typename OP::elem* __restrict__ y, Strides ys, int H, int Tq, int Tk, Strides qs, Strides ks, int q_off,
    int64_t ldv, int exempt, float scale, int damp_mode, float train_len, const float* __restrict__ kn,
    const float* __restrict__ kt_min) {
  using elem = typename OP::elem;
  using frag = typename OP::frag;
  constexpr int NS = D / OP::KS;          // MFMA steps over D
  constexpr int DB = D / 32;              // 32-row blocks of D
  constexpr int LDK = D + OP::KPAD;
  constexpr int LDV = TILE + OP::TPAD;
  constexpr int AS = OP::acc_steps;
  constexpr int NH = G + 1;
  constexpr int TILE_BYTES = (NH * TILE * LDK + G * D * LDV) * (int)sizeof(elem);
  // two LDS buffers of the key tiles (the next one is written while this one is read) when they fit
  constexpr int NBUF = (2 * TILE_BYTES <= 120 * 1024) ? 2 : 1;

  __shared__ __attribute__((aligned(16))) elem sK[NBUF][NH][TILE * LDK];
  __shared__ __attribute__((aligned(16))) elem sVt[NBUF][G][D * LDV];
  __shared__ __attribute__((aligned(16))) float sC[NBUF][NWAVES][TILE];   // -carry rows, logit units
  constexpr int LDF = TILE + 4;
  __shared__ __attribute__((aligned(16))) float sF[NWAVES][TILE * LDF];   // each wavefront's F tile
  __shared__ __attribute__((aligned(16))) float sDamp[NWAVES][TILE];      // its queries' damping factors
  __shared__ uint64_t sMask[REACH_MASK_WORDS];    // the tiles to visit, as bits and as runs (find_reach)
  __shared__ TileRun sRuns[REACH_RUNS];
  __shared__ float sBound[NWAVES][2 * G];         // per wavefront and head: max |q|, min row maximum

  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int n = lane & 31, h = lane >> 5;
  const int groups = H / G;
  const BlockXY bxy = xcd_block();
  const int b = bxy.y / groups, gi = bxy.y % groups;
  const int hd0 = gi * G;
  const bool has_h0 = (gi == 0);
  // a one-head group holding head 0 sends that head's whole adjusted logit through LDS, one product per
  // tile instead of two; not at head dim 32 beside other heads, where the host chooses the width per
  // launch and every width is to give the same bits (see fwd64_kernel)
  const bool whole = G == 1 && has_h0 && (D > 32 || H == 1);
  const int NBq = (Tq + TILE - 1) / TILE;
  const int NKT = (Tk + TILE - 1) / TILE;
  const int qsb = gridDim.x - 1 - bxy.x;
  const int rb = qsb * NWAVES + wave;
  const int q_rel = rb * TILE + n;
  const int q_abs = q_off + q_rel;
  const int64_t seq_row = (int64_t)b * H;   // row of head 0 of this sequence
  auto q_head = [&](int hh) -> const elem* {
    if constexpr (CV) return q + (seq_row + hh) * Tq * D;
    else return q + qs.at(b, hh);
  };
  auto k_head = [&](int hh) -> const elem* {
    if constexpr (CV) return k + (seq_row + hh) * ks.head;
    else return k + ks.at(b, hh);
  };
  const int64_t q_ld = CV ? (int64_t)D : (int64_t)qs.row;
  const int64_t k_ld = CV ? (int64_t)D : (int64_t)ks.row;

  auto kt_end_of = [&](int rbw) {
    const int last = q_off + rbw * TILE + TILE - 1;
    return min(last / TILE + 1, NKT);
  };
  const int my_end = (rb < NBq) ? kt_end_of(rb) : 0;
  const int wg_end = kt_end_of(min(qsb * NWAVES + NWAVES - 1, NBq - 1));

  // Q fragments (B operand of K Q^T): lane holds query q_rel.
  frag qf[G][NS];
  frag q0f[NS];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const elem* qh = q_head(hd0 + g);
#pragma unroll
    for (int s = 0; s < NS; ++s) qf[g][s] = ld_std_bounded<OP>(qh, q_ld, q_rel, Tq, h, s);
  }
  if (!has_h0) {
    const elem* qh = q_head(0);
#pragma unroll
    for (int s = 0; s < NS; ++s) q0f[s] = ld_std_bounded<OP>(qh, q_ld, q_rel, Tq, h, s);
  }

  float m[G], l[G];
  f32x16 o[G][DB];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m[g] = -INFINITY;
    l[g] = 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db) o[g][db] = zero16();
  }

  // F is kept negated and in units of the unscaled logit q.k (relu(s x) = s relu(x) for s > 0):
  // the logit product then accumulates onto -F and yields q.k - F/s directly, and the scale (with
  // log2 e) enters once, in the exponent's fma.
  const float sl2 = scale * LOG2E;
  const float neg_inv_scale = -1.f / scale;
  float damp = 1.f;
  if (damp_mode != 0) {
    damp = fminf(1.f, train_len / (float)(q_abs + 1));
    if (damp_mode == 2) damp = sqrtf(damp);
  }
  if (lane < TILE) sDamp[wave][lane] = damp;   // (read after the first barrier)

  // Staging of one key tile: K of the group (+ head 0's), V^T of the group, and the carry rows of
  // the workgroup's four query blocks (threads 0..127: wavefront w's row, key tid % 32).
  RowTile<elem, D> nK[NH];
  ColTile<elem, D> nVt[G];
  const elem* k_rows[NH];   // the key rows of this workgroup's heads (outside the tile loop)
#pragma unroll
  for (int g = 0; g < G; ++g) k_rows[g] = k_head(hd0 + g);
  k_rows[G] = k_head(0);
  const int k_ldi = (int)k_ld;
  float nC = 0.f;
  bool nC_ok = false;
  // (every load is unconditional and the loaded values are first used when stored: the vector-
  // memory counter drains in issue order, so a wait inside the tile for one of them, or at a join
  // after a conditional one, would wait for the whole next tile)
  auto load_tile = [&](int kt) {
    const int kbase = kt * TILE;
    const int w = (tid >> 5) & (NWAVES - 1);
    const int rbw = min(qsb * NWAVES + w, NBq - 1);
    const int jj = kbase + (tid & (TILE - 1));
    nC = carry[((int64_t)b * NBq + rbw) * Tk + min(jj, Tk - 1)];   // scaled (zero past the end) when stored
    nC_ok = jj < Tk;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      nK[g].load(k_rows[g], k_ldi, kbase, Tk, tid);
      nVt[g].load(vt + (seq_row + hd0 + g) * D * ldv, ldv, kbase, tid);
    }
    nK[G].load(k_rows[G], k_ldi, kbase, Tk, tid);   // head 0's rows (its own group's copy unused)
  };
  auto store_tile = [&](int buf) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      nK[g].template store<LDK>(sK[buf][g], tid);
      nVt[g].template store_crow<LDV>(sVt[buf][g], tid);
    }
    if (!has_h0) nK[G].template store<LDK>(sK[buf][G], tid);
    if (tid < NWAVES * TILE) sC[buf][tid >> 5][tid & (TILE - 1)] = nC_ok ? nC * neg_inv_scale : 0.f;
  };

  // The tiles in the order of the sweep: cur, then nxt (negative: none), newest first; those reaching
  // past the workgroup's first query and one more (down to cut) always, the rest as far as their keys
  // carry weight (find_reach)
  const int i_lo = min((exempt + TILE - 1) / TILE, wg_end);
  const int i_hi = max(i_lo, min(min(q_off + qsb * NWAVES * TILE, Tk) / TILE, wg_end));
  const int cut = max(0, i_hi - 1);
  int cur = wg_end - 1, nxt = wg_end - 2, t = 0;
  const float oldest = reach_total(kt_min != nullptr ? kt_min + (int64_t)b * NKT : nullptr, cut, lane);

  // the next key tile is loaded into registers while this one is computed (stored to the other LDS
  // buffer after it)
  load_tile(wg_end - 1);
  store_tile(0);
  __syncthreads();

  // one key tile; INTERIOR: every key of the tile strictly precedes every query of the workgroup,
  // lies before the end and is not exempt, for every wavefront (straight-line code without masks)
  // DAMP: history damping on (a compile-time fact, so the undamped loops carry no branch for it)
  auto tile_step = [&](auto interior_tag, auto damp_tag) __attribute__((always_inline)) {
    constexpr bool INTERIOR = decltype(interior_tag)::value;
    constexpr bool DAMP = decltype(damp_tag)::value;
    const int kt = cur;
    const int buf = NBUF == 2 ? (t & 1) : 0;
    if (nxt >= 0) load_tile(nxt);
    if (kt < my_end) {   // (a wavefront past the last query block has none)
      const int kbase = kt * TILE;
      // edge: some key of the tile does not strictly precede every query of the block, lies past
      // the end or is exempt; interior tiles skip the masks (the selection gate is then the logit's
      // sign alone)
      const bool edge =
          !INTERIOR && ((kbase + TILE - 1 >= q_off + rb * TILE) || (kbase + TILE > Tk) || kbase < exempt);
      // (one body for both kinds of tile within a loop: two copies of its accumulating products
      // would make the compiler copy the output sums between register sets every tile)
      auto body = [&]() {
        // Head 0's logits as (queries x keys), lane = key kbase + n: the selection's running sum
        // over queries then stays within the lane. -F (logit units) = -(the carry at the block's
        // first query + the selection by the block's earlier queries); it returns to the
        // (keys x queries) layout of the softmax through this wavefront's LDS rows.
        f32x16 l0t = zero16();
        {
          const elem* k0s = has_h0 ? sK[buf][0] : sK[buf][G];
#pragma unroll
          for (int s = 0; s < NS; ++s)
            l0t = OP::mma(has_h0 ? qf[0][s] : q0f[s], OP::ld_std(k0s, LDK, n, h, s), l0t);
        }
        {
          f32x16 sel;
#pragma unroll
          // -relu as one v_med3 (fminf on a negated value, or a med3 with an infinite bound, which
          // the compiler folds into fminf, would first be canonicalised)
          for (int i = 0; i < 16; ++i) sel[i] = __builtin_amdgcn_fmed3f(-l0t[i], -3.0e38f, 0.f);
          if (edge) {
            // pairs exempt <= j < r; keys past the end and queries past the end hold zero rows
            const int jk = kbase + n;
            const int thr = jk >= exempt ? jk - (q_off + rb * TILE) - 4 * h : 32;
#pragma unroll
            for (int i = 0; i < 16; ++i) sel[i] = crow(i, 0) > thr ? sel[i] : 0.f;
          }
          float run = sC[buf][wave][n];
          float* fw = sF[wave];
#pragma unroll
          for (int a = 0; a < 4; ++a) {
            const Halves g = halves(((sel[4 * a] + sel[4 * a + 1]) + sel[4 * a + 2]) + sel[4 * a + 3]);
            float p = (h == 0) ? run : run + g.lo;   // rows 8a..8a+3 in the low half, 8a+4.. in the high
            float4 dm = make_float4(1.f, 1.f, 1.f, 1.f);   // the rows' damping factors
            if constexpr (DAMP) dm = *reinterpret_cast<const float4*>(&sDamp[wave][8 * a + 4 * h]);
            const float dmv[4] = {dm.x, dm.y, dm.z, dm.w};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              // (whole: q.k - damp F/s, so its (keys x queries) product is not taken again)
              float f = p;
              if (whole) f = DAMP ? fmaf(dmv[t], p, l0t[4 * a + t]) : p + l0t[4 * a + t];
              fw[crow(4 * a + t, h) * LDF + n] = f;
              p += sel[4 * a + t];
            }
            run = (run + g.lo) + g.hi;
          }
        }
        lds_wave_sync();
        f32x16 fs;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const float4 f4 = *reinterpret_cast<const float4*>(&sF[wave][n * LDF + 8 * a + 4 * h]);
          fs[4 * a] = f4.x;
          fs[4 * a + 1] = f4.y;
          fs[4 * a + 2] = f4.z;
          fs[4 * a + 3] = f4.w;
        }
        if constexpr (DAMP) {
          if (!whole) {
#pragma unroll
            for (int i = 0; i < 16; ++i) fs[i] *= damp;
          }
        }

#pragma unroll
        for (int g = 0; g < G; ++g) {
          f32x16 lg = fs;   // the product accumulates onto -F: lg = q.k - F/s
          if (!whole) {   // (else head 0's came through LDS whole)
#pragma unroll
            for (int s = 0; s < NS; ++s) lg = OP::mma(OP::ld_std(sK[buf][g], LDK, n, h, s), qf[g][s], lg);
          }
          if (edge) {   // keys j = kbase + crow(i, h) <= min(q_abs, Tk - 1)
            const int thr = min(q_abs, Tk - 1) - kbase - 4 * h;
#pragma unroll
            for (int i = 0; i < 16; ++i) lg[i] = crow(i, 0) <= thr ? lg[i] : -INFINITY;
          }
          float zmax = -INFINITY;
#pragma unroll
          for (int i = 0; i < 16; ++i) zmax = fmaxf(zmax, lg[i]);
          const Halves zh = halves(zmax);
          const float m_new = fmaxf(m[g], fmaxf(zh.lo, zh.hi) * sl2);   // log2 units
          if (__any(m_new > m[g])) {   // some row's maximum rose: rescale what was accumulated
            const float alpha = (m_new == -INFINITY) ? 1.f : fast_exp2(m[g] - m_new);
            m[g] = m_new;
            l[g] *= alpha;
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
              for (int i = 0; i < 16; ++i) o[g][db][i] *= alpha;
          }
          const float mu = (m[g] == -INFINITY) ? 0.f : m[g];   // a row with no key yet
          float psum = 0.f;
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const float p = fast_exp2(fmaf(lg[i], sl2, -mu));
            lg[i] = p;
            psum += p;
          }
          l[g] += psum;
          frag pf[AS];
#pragma unroll
          for (int s = 0; s < AS; ++s) pf[s] = OP::from_acc(lg, s);
#pragma unroll
          for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int s = 0; s < AS; ++s)
              o[g][db] = OP::mma(OP::ld_perm(sVt[buf][g], LDV, db * 32 + n, h, s), pf[s], o[g][db]);
        }
      };
      body();
    }
    if constexpr (NBUF == 1) __syncthreads();   // the one buffer is free again
    if (nxt >= 0) store_tile(NBUF == 2 ? buf ^ 1 : 0);
    __syncthreads();
  };
  // key tiles newest first: the diagonals and the sequence end, the interior tiles
  // [i_lo, i_hi), then the tiles holding exempt keys
  auto sweep = [&](auto damp_tag) {
    int run_lo = INT_MIN, run_i = 0;   // the run nxt lies in
    auto shift = [&]() {
      cur = nxt;
      ++t;
      if (__builtin_expect(--nxt < run_lo, 0)) {
        const TileRun r = sRuns[run_i++];
        nxt = __builtin_amdgcn_readfirstlane(r.hi);
        run_lo = __builtin_amdgcn_readfirstlane(r.lo);
      }
    };
    // tiles from cur down to `stop`; those inside a run in a loop of their own, in which the compiler sees that
    // they follow each other (head dim 128, B=1 H=16, 256 queries over 16384 keys, no tile left out: 687 us, 732
    // with every tile's addresses anew)
    auto run = [&](int stop, auto interior_tag) {
      while (cur >= stop) {
        if (nxt == cur - 1) {
          const int lim = max(max(stop, 1), run_lo + 2);
          for (; cur >= lim; --cur, ++t) {
            nxt = cur - 1;
            tile_step(interior_tag, damp_tag);
          }
          nxt = cur - 1;
        }
        if (cur >= stop) {
          tile_step(interior_tag, damp_tag);
          shift();
        }
      }
    };
    for (; cur >= i_hi; shift()) tile_step(std::false_type{}, damp_tag);
    nxt = cut - 1;   // the tiles below cut: all of them, or the runs found
    if (reach_worth(oldest)) {
      find_reach<OP, G, NS>(qf, m, q_rel < Tq, scale, kn + (seq_row + hd0) * NKT, kt_min + (int64_t)b * NKT, NKT,
                            carry + ((int64_t)b * NBq + qsb * NWAVES) * Tk, Tk, cut, i_lo, sBound, sMask, sRuns, lane, wave);
      const TileRun r = sRuns[run_i++];
      nxt = __builtin_amdgcn_readfirstlane(r.hi);
      run_lo = __builtin_amdgcn_readfirstlane(r.lo);
    }
    run(i_lo, std::true_type{});
    for (; cur >= 0; shift()) tile_step(std::false_type{}, damp_tag);
  };
  if (damp_mode != 0) sweep(std::true_type{});
  else sweep(std::false_type{});

  if (rb >= NBq || q_rel >= Tq) return;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const Halves lh = halves(l[g]);
    const float ltot = lh.lo + lh.hi;
    const float inv = 1.f / ltot;
    const int64_t row = (seq_row + hd0 + g) * Tq + q_rel;
    float* orow = out + row * D;
    elem* yrow = y ? y + ys.at(b, hd0 + g) + (int64_t)q_rel * ys.row : nullptr;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        float4 v4 = make_float4(o[g][db][4 * a] * inv, o[g][db][4 * a + 1] * inv,
                                o[g][db][4 * a + 2] * inv, o[g][db][4 * a + 3] * inv);
        const int d = db * 32 + 8 * a + 4 * h;
        *reinterpret_cast<float4*>(orow + d) = v4;
        if (yrow) {
          if constexpr (sizeof(elem) == 2) {
            *reinterpret_cast<uint2*>(yrow + d) = make_uint2(
                (uint32_t)OP::to_elem(v4.x) | ((uint32_t)OP::to_elem(v4.y) << 16),
                (uint32_t)OP::to_elem(v4.z) | ((uint32_t)OP::to_elem(v4.w) << 16));
          } else {
            *reinterpret_cast<float4*>(yrow + d) = v4;
          }
        }
      }
    }
    if (h == 0) {
      rmax[row] = m[g];
      rden[row] = ltot;
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Forward, bf16 storage at head dim 64 with G = 2 heads per wavefront or one (odd head counts, the
// per-head mode, grids that fill the CUs only once: fwd64_group): fwd_kernel's tile work with every
// key tile's operands loaded straight into LDS ahead of use (see bwd_kv64_kernel), and the
// selection one tile ahead of the softmax: while tile t's logit products, softmax and value
// products run, the wavefront also takes head 0's logits of tile t + 1 and turns them into that
// tile's F (through its LDS rows, read at the start of tile t + 1), so each tile is one block of
// independent products and arithmetic the compiler interleaves, with no wait inside it for the F
// round trip. A sequence's only head (G = 1, one head) sends its whole adjusted logits through the
// LDS rows instead (as fwd_kernel does), so it takes one logit product per tile. The K rows of the
// group's heads (swz64) and their V rows (swzq, read transposed by the value products, get_trq)
// load one tile ahead into two buffers; head 0's K rows and each wavefront's carry row two tiles
// ahead into two more; all four are separate LDS variables and the tile loop runs in pairs, so
// every access names its buffer at compile time; one barrier per tile. Two workgroups per CU at
// G = 2, three at G = 1.

template <int G>
struct FwdTileBuf64 {
  __attribute__((aligned(16))) uint16_t k[G][TILE * 64];   // K rows of the group's heads
  __attribute__((aligned(16))) uint16_t v[G][TILE * 64];   // their V rows
};
struct FwdSelBuf64 {
  __attribute__((aligned(16))) uint16_t k0[TILE * 64];      // head 0's K rows
  __attribute__((aligned(16))) float c[NWAVES][64];         // per wavefront: the carry of each key
};

template <bool CV, int G>   // CV: as fwd_kernel; G: heads per wavefront (1 or 2)
__global__ __launch_bounds__(NTHREADS, G == 1 ? 3 : 2) void fwd64_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    const float* __restrict__ carry, float* __restrict__ out, float* __restrict__ rmax, float* __restrict__ rden,
    uint16_t* __restrict__ y, Strides ys, int H, int Tq, int Tk, Strides qs, Strides ks, Strides vs, int q_off,
    int exempt, float scale, int damp_mode, float train_len, const float* __restrict__ kn,
    const float* __restrict__ kt_min) {
  using OP = OpBF16;
  using elem = uint16_t;
  using frag = OP::frag;
  constexpr int D = 64, NS = 4, DB = 2, AS = 2;
  static_assert(G == 1 || G == 2, "one or two heads per wavefront");
  // LDS lifetimes (tile t = key tile wg_end - 1 - t; every fill is a direct load of all four
  // wavefronts, a quarter each, and each tile step ends with wait_loads() -- this wavefront's loads
  // have landed -- and __syncthreads() -- every wavefront's have, and every wavefront is past its
  // reads of the step):
  //   sB0, sB1  tile t's K and V rows, buffer t mod 2. Filled: the prologue (tile 0), tile step
  //             t - 1 (tile t). Drained: tile step t (the logit and value products). Separated:
  //             the last reads of buffer t mod 2 (tile step t - 2) from its fill (tile step t - 1)
  //             by the end of tile step t - 2.
  //   sS0, sS1  tile t's head-0 K rows and each wavefront's carry row, buffer t mod 2. Filled: the
  //             prologue (tiles 0, 1), tile step t - 2 (tile t). Drained: the selection of tile t
  //             (select(), run at the end of tile step t - 1; tile 0's in the sweep's prologue).
  //             Separated: the selection of tile t - 2 (end of tile step t - 3) from the fill in tile
  //             step t - 2 by the end of tile step t - 3; tile 0's selection from tile 2's fill (tile
  //             step 0) by the barrier after it in the sweep's prologue; the fill of tile t (tile
  //             step t - 2) from its selection (end of tile step t - 1) by the end of tile step t - 2.
  //   sF        per wavefront, its F tile: written by select() of tile t + 1 at the end of tile step t
  //             (transposing stores), read at the start of tile step t + 1; the same wavefront's
  //             writes follow its reads of tile t in program order, and the reads of tile t + 1 follow
  //             the writes across the step's barrier.
  //   sDamp     per wavefront, its queries' damping factors: written once before the prologue's
  //             barrier, read only after it.
  //   sBound, sMask, sRuns  written once, in find_reach (after the barrier that ends the last diagonal tile), each
  //             with a barrier between its writes and its reads.
  // (tile t: the t-th tile visited; without skipping it is key tile wg_end - 1 - t)
  __shared__ FwdTileBuf64<G> sB0, sB1;   // tile t's K and V rows in buffer t mod 2
  __shared__ FwdSelBuf64 sS0, sS1;    // tile t's head-0 K rows and carry rows in buffer t mod 2
  constexpr int LDF = TILE + 4;
  __shared__ __attribute__((aligned(16))) float sF[NWAVES][TILE * LDF];   // each wavefront's F tile
  __shared__ __attribute__((aligned(16))) float sDamp[NWAVES][TILE];      // its queries' damping factors
  __shared__ uint64_t sMask[REACH_MASK_WORDS];    // the tiles to visit, as bits and as runs (find_reach)
  __shared__ TileRun sRuns[REACH_RUNS];
  __shared__ float sBound[NWAVES][2 * G];         // per wavefront and head: max |q|, min row maximum

  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int n = lane & 31, h = lane >> 5;
  const int groups = H / G;
  const BlockXY bxy = part_block();
  const int b = bxy.y / groups, gi = bxy.y % groups;
  const int hd0 = gi * G;
  const bool has_h0 = (gi == 0);
  // Head 0's adjusted logits come through LDS whole when it is the sequence's only head (one product
  // per tile instead of two). With other heads beside it, head 0 takes the path of every head (its
  // product accumulating onto -F), so one and two heads per wavefront give the same bits and the
  // host may choose either per launch.
  const bool whole = G == 1 && has_h0 && H == 1;
  const int NBq = (Tq + TILE - 1) / TILE;
  const int NKT = (Tk + TILE - 1) / TILE;
  const int qsb = gridDim.x - 1 - bxy.x;
  const int rb = qsb * NWAVES + wave;
  const int q_rel = rb * TILE + n;
  const int q_abs = q_off + q_rel;
  const int64_t seq_row = (int64_t)b * H;
  auto q_head = [&](int hh) -> const elem* {
    if constexpr (CV) return q + (seq_row + hh) * Tq * D;
    else return q + qs.at(b, hh);
  };
  auto k_head = [&](int hh) -> const elem* {
    if constexpr (CV) return k + (seq_row + hh) * ks.head;
    else return k + ks.at(b, hh);
  };
  const int64_t q_ld = CV ? (int64_t)D : (int64_t)qs.row;
  const int k_ld = CV ? D : (int)ks.row;

  auto kt_end_of = [&](int rbw) {
    const int last = q_off + rbw * TILE + TILE - 1;
    return min(last / TILE + 1, NKT);
  };
  const int my_end = (rb < NBq) ? kt_end_of(rb) : 0;
  const int wg_end = kt_end_of(min(qsb * NWAVES + NWAVES - 1, NBq - 1));

  // Q fragments (B operand of K Q^T): lane holds query q_rel.
  frag qf[G][NS];
  frag q0f[NS];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const elem* qh = q_head(hd0 + g);
#pragma unroll
    for (int s = 0; s < NS; ++s) qf[g][s] = ld_std_bounded<OP>(qh, q_ld, q_rel, Tq, h, s);
  }
  if (!has_h0) {
    const elem* qh = q_head(0);
#pragma unroll
    for (int s = 0; s < NS; ++s) q0f[s] = ld_std_bounded<OP>(qh, q_ld, q_rel, Tq, h, s);
  }

  float m[G], l[G];
  f32x16 o[G][DB];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m[g] = -INFINITY;
    l[g] = 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db) o[g][db] = zero16();
  }
  // F negated, in units of the unscaled logit q.k (see fwd_kernel)
  const float sl2 = scale * LOG2E;
  const float neg_inv_scale = -1.f / scale;
  float damp = 1.f;
  if (damp_mode != 0) {
    damp = fminf(1.f, train_len / (float)(q_abs + 1));
    if (damp_mode == 2) damp = sqrtf(damp);
  }
  if (lane < TILE) sDamp[wave][lane] = damp;   // (read after the first barrier)

  // key-side sources and this lane's parts of the direct loads
  const __amdgpu_buffer_rsrc_t rs_k0 = rsrc(k_head(hd0), (int64_t)Tk * k_ld * 2);
  const __amdgpu_buffer_rsrc_t rs_k1 = rsrc(k_head(hd0 + G - 1), (int64_t)Tk * k_ld * 2);
  const __amdgpu_buffer_rsrc_t rs_kh = rsrc(k_head(0), (int64_t)Tk * k_ld * 2);
  const __amdgpu_buffer_rsrc_t rs_v0 = rsrc(v + vs.at(b, hd0), (int64_t)Tk * vs.row * 2);
  const __amdgpu_buffer_rsrc_t rs_v1 = rsrc(v + vs.at(b, hd0 + G - 1), (int64_t)Tk * vs.row * 2);
  // this wavefront's carry row (its query block's; keys past the end read zero)
  const __amdgpu_buffer_rsrc_t rs_c =
      rsrc(carry + ((int64_t)b * NBq + min(rb, NBq - 1)) * Tk, (int64_t)Tk * 4);
  const RowsLane rl_k(k_ld, lane, wave);
  const RowsLaneQ rl_v(vs.row, lane, wave);

  // key tile kt's K and V rows (into B), and its head-0 K rows and carry rows (into S), by direct
  // loads only
  auto load_tile = [&](int kt, FwdTileBuf64<G>& B) {
    const int kbase = kt * TILE;
    g2l_rows64(B.k[0], rs_k0, rl_k, k_ld, kbase, wave);
    g2l_rowsq(B.v[0], rs_v0, rl_v, vs.row, kbase, wave);
    if constexpr (G == 2) {
      g2l_rows64(B.k[1], rs_k1, rl_k, k_ld, kbase, wave);
      g2l_rowsq(B.v[1], rs_v1, rl_v, vs.row, kbase, wave);
    }
  };
  auto load_sel = [&](int kt, FwdSelBuf64& S) {
    const int kbase = kt * TILE;
    g2l_rows64(S.k0, rs_kh, rl_k, k_ld, kbase, wave);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_c, lds_ptr(S.c[wave]), 4, (kbase + n) * 4, 0, 0, 0);
  };
  auto rfrag = [&](const elem* tile, int s) -> frag {
    return *reinterpret_cast<const frag*>(tile + swz64(n, 2 * s + h));
  };

  // Key tile kt's selection: head 0's logits as (queries x keys), lane = key, so the running sum over
  // queries stays within the lane; -F (logit units) = -(the carry at the block's first query + the
  // selection by the block's earlier queries) goes to this wavefront's LDS rows, where the tile's
  // softmax reads it in the (keys x queries) layout (with `whole`: q.k - damp F/s, damping per row).
  auto select = [&](int kt, const FwdSelBuf64& S, auto damp_tag) {
    constexpr bool DAMP = decltype(damp_tag)::value;
    const int kbase = kt * TILE;
    f32x16 l0t = zero16();
#pragma unroll
    for (int s = 0; s < NS; ++s) l0t = OP::mma(has_h0 ? qf[0][s] : q0f[s], rfrag(S.k0, s), l0t);
    f32x16 sel;
    // -relu as one v_med3 (see fwd_kernel)
#pragma unroll
    for (int i = 0; i < 16; ++i) sel[i] = __builtin_amdgcn_fmed3f(-l0t[i], -3.0e38f, 0.f);
    const bool edge = (kbase + TILE - 1 >= q_off + rb * TILE) || (kbase + TILE > Tk) || kbase < exempt;
    if (edge) {
      // pairs exempt <= j < r; keys past the end and queries past the end hold zero rows
      const int jk = kbase + n;
      const int thr = jk >= exempt ? jk - (q_off + rb * TILE) - 4 * h : 32;
#pragma unroll
      for (int i = 0; i < 16; ++i) sel[i] = crow(i, 0) > thr ? sel[i] : 0.f;
    }
    float run = S.c[wave][n] * neg_inv_scale;
    float* fw = sF[wave];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const Halves g = halves(((sel[4 * a] + sel[4 * a + 1]) + sel[4 * a + 2]) + sel[4 * a + 3]);
      float p = (h == 0) ? run : run + g.lo;
      float4 dm = make_float4(1.f, 1.f, 1.f, 1.f);   // the rows' damping factors
      if constexpr (DAMP && G == 1) dm = *reinterpret_cast<const float4*>(&sDamp[wave][8 * a + 4 * h]);
      const float dmv[4] = {dm.x, dm.y, dm.z, dm.w};
#pragma unroll
      for (int t2 = 0; t2 < 4; ++t2) {
        float f = p;
        if (whole) f = DAMP ? fmaf(dmv[t2], p, l0t[4 * a + t2]) : p + l0t[4 * a + t2];
        fw[crow(4 * a + t2, h) * LDF + n] = f;
        p += sel[4 * a + t2];
      }
      run = (run + g.lo) + g.hi;
    }
  };

  // The tiles in the order of the sweep: cur, then n1 and n2 (-1: none), newest first. Every tile down to
  // `cut` -- those reaching past the workgroup's first query, and two more, so that the loads one and
  // two tiles ahead never run past what is known -- is visited; the rest as far as its keys carry
  // weight, once the row maxima of the diagonal tiles are known (find_reach).
  const int i_lo = min((exempt + TILE - 1) / TILE, wg_end);
  const int i_hi = max(i_lo, min(min(q_off + qsb * NWAVES * TILE, Tk) / TILE, wg_end));
  const int cut = max(0, i_hi - 2);
  int cur = wg_end - 1, n1 = wg_end - 2, n2 = wg_end - 3;
  const float oldest = reach_total(kt_min != nullptr ? kt_min + (int64_t)b * NKT : nullptr, cut, lane);

  // the first tile's operands, head-0 rows and carry of the first two (its F at the sweep's start)
  load_tile(wg_end - 1, sB0);
  load_sel(wg_end - 1, sS0);
  if (wg_end >= 2) load_sel(wg_end - 2, sS1);
  wait_loads();
  __syncthreads();

  // the t-th tile of the sweep, cur (buffer t mod 2, named by ODD); INTERIOR and DAMP as in fwd_kernel
  // (INTERIOR for this tile; the selection of the next one checks its own tile)
  auto tile_step = [&](auto interior_tag, auto damp_tag, auto odd_tag) __attribute__((always_inline)) {
    constexpr bool INTERIOR = decltype(interior_tag)::value;
    constexpr bool DAMP = decltype(damp_tag)::value;
    constexpr bool ODD = decltype(odd_tag)::value;
    FwdTileBuf64<G>& B = ODD ? sB1 : sB0;
    const int kt = cur;
    // free since the last barrier: the other tile buffer, and this parity's head-0 buffer (this tile's
    // rows were used by its selection during the tile before)
    if (n1 >= 0) load_tile(n1, ODD ? sB0 : sB1);
    if (n2 >= 0) load_sel(n2, ODD ? sS1 : sS0);
    if (kt < my_end) {   // (a wavefront past the last query block has none)
      const int kbase = kt * TILE;
      const bool edge =
          !INTERIOR && ((kbase + TILE - 1 >= q_off + rb * TILE) || (kbase + TILE > Tk) || kbase < exempt);
      f32x16 fs;   // -F of this tile, written by its selection
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const float4 f4 = *reinterpret_cast<const float4*>(&sF[wave][n * LDF + 8 * a + 4 * h]);
        fs[4 * a] = f4.x;
        fs[4 * a + 1] = f4.y;
        fs[4 * a + 2] = f4.z;
        fs[4 * a + 3] = f4.w;
      }
      if constexpr (DAMP) {
        if (!whole) {
#pragma unroll
          for (int i = 0; i < 16; ++i) fs[i] *= damp;
        }
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        f32x16 lg = fs;   // the product accumulates onto -F: lg = q.k - F/s
        if (!whole) {
#pragma unroll
          for (int s = 0; s < NS; ++s) lg = OP::mma(rfrag(B.k[g], s), qf[g][s], lg);
        }
        if (edge) {
          const int thr = min(q_abs, Tk - 1) - kbase - 4 * h;
#pragma unroll
          for (int i = 0; i < 16; ++i) lg[i] = crow(i, 0) <= thr ? lg[i] : -INFINITY;
        }
        float zmax = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) zmax = fmaxf(zmax, lg[i]);
        const Halves zh = halves(zmax);
        const float m_new = fmaxf(m[g], fmaxf(zh.lo, zh.hi) * sl2);
        if (__any(m_new > m[g])) {
          const float alpha = (m_new == -INFINITY) ? 1.f : fast_exp2(m[g] - m_new);
          m[g] = m_new;
          l[g] *= alpha;
#pragma unroll
          for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[g][db][i] *= alpha;
        }
        const float mu = (m[g] == -INFINITY) ? 0.f : m[g];
        float psum = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float p = fast_exp2(fmaf(lg[i], sl2, -mu));
          lg[i] = p;
          psum += p;
        }
        l[g] += psum;
        frag pf[AS];
#pragma unroll
        for (int s = 0; s < AS; ++s) pf[s] = OP::from_acc(lg, s);
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int s = 0; s < AS; ++s)
            o[g][db] = OP::mma(get_trq<true>(B.v[g], lane, db, s), pf[s], o[g][db]);
      }
    }
    // the next tile's F (after this tile's reads of the wavefront's F rows, in program order)
    if (n1 >= 0 && n1 < my_end) select(n1, ODD ? sS0 : sS1, damp_tag);
    wait_loads();
    __syncthreads();   // the next tile's operands are in; every wavefront is done with this one
  };
  auto sweep = [&](auto damp_tag) {
    if (wg_end - 1 < my_end) select(wg_end - 1, sS0, damp_tag);   // the first tile's F
    // The first tile step loads tile 2's head-0 K rows into sS0, whose rows every wavefront has
    // just read for that F: all of them must be past their reads first.
    __syncthreads();
    // tiles from cur down to `stop`, in pairs (buffer 0, buffer 1); run_lo, run_i: the run n2 lies in
    bool odd = false;
    int run_lo = INT_MIN, run_i = 0;
    auto shift = [&]() {
      cur = n1;
      n1 = n2;
      if (__builtin_expect(--n2 < run_lo, 0)) {
        const TileRun r = sRuns[run_i++];
        n2 = __builtin_amdgcn_readfirstlane(r.hi);
        run_lo = __builtin_amdgcn_readfirstlane(r.lo);
      }
    };
    auto run = [&](int stop, auto interior_tag) {
      if (odd && cur >= stop) {
        tile_step(interior_tag, damp_tag, std::true_type{});
        shift();
        odd = false;
      }
      while (cur >= stop) {
        tile_step(interior_tag, damp_tag, std::false_type{});
        shift();
        if (cur < stop) {
          odd = true;
          break;
        }
        tile_step(interior_tag, damp_tag, std::true_type{});
        shift();
      }
    };
    run(i_hi, std::false_type{});
    n2 = cut - 1;   // the tiles below cut: all of them, or the runs found
    if (reach_worth(oldest)) {
      find_reach<OP, G, NS>(qf, m, q_rel < Tq, scale, kn + (seq_row + hd0) * NKT, kt_min + (int64_t)b * NKT,
                            NKT, carry + ((int64_t)b * NBq + qsb * NWAVES) * Tk, Tk, cut, i_lo, sBound, sMask, sRuns, lane, wave);
      const TileRun r = sRuns[run_i++];
      n2 = __builtin_amdgcn_readfirstlane(r.hi);
      run_lo = __builtin_amdgcn_readfirstlane(r.lo);
    }
    run(i_lo, std::true_type{});
    run(0, std::false_type{});
  };
  if (damp_mode != 0) sweep(std::true_type{});
  else sweep(std::false_type{});

  if (rb >= NBq || q_rel >= Tq) return;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const Halves lh = halves(l[g]);
    const float ltot = lh.lo + lh.hi;
    const float inv = 1.f / ltot;
    const int64_t row = (seq_row + hd0 + g) * Tq + q_rel;
    float* orow = out + row * D;
    elem* yrow = y ? y + ys.at(b, hd0 + g) + (int64_t)q_rel * ys.row : nullptr;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        float4 v4 = make_float4(o[g][db][4 * a] * inv, o[g][db][4 * a + 1] * inv, o[g][db][4 * a + 2] * inv,
                                o[g][db][4 * a + 3] * inv);
        const int d = db * 32 + 8 * a + 4 * h;
        *reinterpret_cast<float4*>(orow + d) = v4;
        if (yrow)
          *reinterpret_cast<uint2*>(yrow + d) =
              make_uint2((uint32_t)OP::to_elem(v4.x) | ((uint32_t)OP::to_elem(v4.y) << 16),
                         (uint32_t)OP::to_elem(v4.z) | ((uint32_t)OP::to_elem(v4.w) << 16));
      }
    }
    if (h == 0) {
      rmax[row] = m[g];
      rden[row] = ltot;
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Backward preparation, a wavefront per 32 query rows, a workgroup per QSTAT_ROWS rows of one head. Always:
// lse = rmax + log2(rden) and ndbar = -rowsum(dO * O) (negated: the dO.v products accumulate onto it), laid
// out (R, ldt), each head's rows padded to ldt with lse = +inf (P = 0) and ndbar = 0, so a 32-row tile of
// them is always in bounds; D/8 lanes per row, 8 elements each, so a row's loads are contiguous.
//
// With reach.qstat, for the key side's search for the tiles without weight (kv_last_block): the largest
// |q| and the least lse of the workgroup's rows, infinities where a row is not finite or a product with it
// could overflow.
//
// With reach.xk, the gradients of the first xk keys, the exempt ones. They have no history (F = 0), so
// every later query keeps weight on them: the key side would sweep every query tile for those few
// columns, long after its other keys' weights are gone. Here they are one more set of products on the rows
// at hand, which go to the wavefront's LDS tiles for it: P and dz of the 32 first keys (columns from xk on
// masked), dV += P^T dO and dK += dz^T Q with P and dz as split operands (hi + lo, as these sums run over
// every query), the rows taken transposed from LDS. The wavefronts' sums add up in LDS, the workgroups' in
// bwd_finish_kernel, both in a fixed order.
// ONE (xk = 1, the usual number): a matrix product of 32 columns for one key, and the rows' way through LDS for it,
// cost as much again as what they overlapped with. Its logit and dO.v are two more row sums beside -dbar's, and
// each lane adds P dO and dz q of its eight elements in registers.
// Bound by HBM (dO, O and Q once). Measured at B=1 H=16 T=16384 bf16: 25 us with no or one exempt key apart (5.4
// TB/s; one through the matrix products 33), 39 with 16; B=2 H=12 T=2048 9 us (12), fp32 B=1 H=8 T=2048 6 (11.5).

template <class OP, int D, bool ONE>
__global__ __launch_bounds__(NTHREADS, (sizeof(typename OP::elem) == 2 ? (D <= 64 ? 4 : 2) : 1)) void bwd_rowprep_kernel(
    const typename OP::elem* __restrict__ q, const typename OP::elem* __restrict__ k,
    const typename OP::elem* __restrict__ v, const typename OP::elem* __restrict__ dout, Strides qs, Strides ks,
    Strides vs, Strides dos, int H, int T, const float* __restrict__ out, const float* __restrict__ rmax,
    const float* __restrict__ rden, float* __restrict__ lse, float* __restrict__ ndbar, int64_t ldt, float scale,
    BwdReach reach) {
  using elem = typename OP::elem;
  using frag = typename OP::frag;
  constexpr int NS = D / OP::KS, DB = D / 32, AS = OP::acc_steps;
  constexpr int LPR = D / 8, RPW = 64 / LPR, PASSES = TILE / RPW;
  constexpr bool TR = sizeof(elem) == 2 && D == 64;   // rows in swzq, taken transposed by get_trq
  constexpr int LD = TR ? D : D + OP::KPAD;
  static_assert(QSTAT_ROWS == NWAVES * TILE, "a wavefront per row tile");
  constexpr int SUMLD = 2 * D + 4;   // floats of one key's dK and dV (padded: keys on shifted banks)
  union Many {
    elem rows[NWAVES][2][TILE * LD];   // a wavefront's dO rows and Q rows
    float sum[NWAVES][8 * SUMLD];      // then its dK and dV sums of eight keys
  };
  struct Single {
    float sum[NWAVES * RPW][2 * D];           // dK and dV of the key over the rows of one lane group
    float4 part[NTHREADS];                    // then over four of those
  };
  using Shared = typename std::conditional<ONE, Single, Many>::type;
  __shared__ __attribute__((aligned(16))) Shared sh;
  __shared__ __attribute__((aligned(16))) float sRow[NWAVES][2][TILE];   // a wavefront's rows' lse and -dbar
  __shared__ float sStat[NWAVES][2];

  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int n = lane & 31, h = lane >> 5;
  const int r = blockIdx.y, seg = blockIdx.x;
  const int b = r / H, hh = r % H;
  const int xk = ONE ? 1 : reach.xk;
  const int qbase = (seg * NWAVES + wave) * TILE;
  const int part = lane % LPR;
  const bool stats = reach.qstat != nullptr;

  union Row {
    elem e[8];
    uint4 u[sizeof(elem) == 2 ? 1 : 2];
  };
  Row dr[PASSES], qr[PASSES];
  float4 o4[PASSES][2];
  float mv[PASSES], nv[PASSES];
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {   // every load of the tile in flight (the last row again past the end)
    const int row = qbase + p * RPW + lane / LPR;
    const int64_t rr = min(row, T - 1);
    const uint4* ds = reinterpret_cast<const uint4*>(dout + dos.at(b, hh) + rr * dos.row + 8 * part);
    const uint4* qv = reinterpret_cast<const uint4*>(q + qs.at(b, hh) + rr * qs.row + 8 * part);
    const float4* os = reinterpret_cast<const float4*>(out + ((int64_t)r * T + rr) * D + 8 * part);
#pragma unroll
    for (int c = 0; c < (int)(sizeof(elem) / 2); ++c) {
      dr[p].u[c] = ds[c];
      if (ONE || stats) qr[p].u[c] = qv[c];
    }
    o4[p][0] = os[0];
    o4[p][1] = os[1];
    mv[p] = rmax[(int64_t)r * T + rr];
    nv[p] = rden[(int64_t)r * T + rr];
  }
  Row k0, v0;   // ONE: this lane's part of the key and its value
  float dk0[8], dv0[8];
  if constexpr (ONE) {
#pragma unroll
    for (int c = 0; c < (int)(sizeof(elem) / 2); ++c) {
      k0.u[c] = reinterpret_cast<const uint4*>(k + ks.at(b, hh) + 8 * part)[c];
      v0.u[c] = reinterpret_cast<const uint4*>(v + vs.at(b, hh) + 8 * part)[c];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) dk0[e] = dv0[e] = 0.f;
  }
  float qmax = 0.f, lmin = INFINITY;
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    const int rl = p * RPW + lane / LPR, row = qbase + rl;
    const bool ok = row < T;
    const float lv = ok ? mv[p] + __log2f(nv[p]) : INFINITY;
    if (!ok) {   // (zeros)
#pragma unroll
      for (int c = 0; c < (int)(sizeof(elem) / 2); ++c) dr[p].u[c] = qr[p].u[c] = make_uint4(0u, 0u, 0u, 0u);
    }
    const float ov[8] = {o4[p][0].x, o4[p][0].y, o4[p][0].z, o4[p][0].w, o4[p][1].x, o4[p][1].y, o4[p][1].z, o4[p][1].w};
    float acc = 0.f, dd = 0.f, qq = 0.f, qk = 0.f, dov = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float d = OP::to_float(dr[p].e[e]);
      acc += d * ov[e];
      if (ONE || stats) {
        const float x = OP::to_float(qr[p].e[e]);
        dd = fmaf(d, d, dd);
        qq = fmaf(x, x, qq);
        if constexpr (ONE) {
          qk = fmaf(x, OP::to_float(k0.e[e]), qk);
          dov = fmaf(d, OP::to_float(v0.e[e]), dov);
        }
      }
    }
#pragma unroll
    for (int o = LPR / 2; o > 0; o >>= 1) {
      acc += __shfl_xor(acc, o);
      if constexpr (ONE) {
        qk += __shfl_xor(qk, o);
        dov += __shfl_xor(dov, o);
      }
      if (ONE || stats) {
        dd += __shfl_xor(dd, o);
        qq += __shfl_xor(qq, o);
      }
    }
    const float nd = ok ? -acc : 0.f;
    if (part == 0 && row < ldt) {
      lse[(int64_t)r * ldt + row] = lv;
      ndbar[(int64_t)r * ldt + row] = nd;
    }
    if ((ONE || stats) && ok) {
      qmax = fmaxf(qmax, qq < REACH_NORM2 && dd < REACH_NORM2 && fabsf(nd) < REACH_NORM2 ? qq : INFINITY);
      lmin = fminf(lmin, fabsf(lv) < 3.0e38f ? lv : -INFINITY);
    }
    if constexpr (ONE) {   // key 0 precedes every query
      const float pr = fast_exp2(fmaf(qk, scale * LOG2E, -lv)), dz = pr * (dov + nd);
      auto add = [&](float (&sum)[8], float x, const Row& y) {
#pragma unroll
        for (int e = 0; e < 8; ++e) sum[e] = fmaf(x, OP::to_float(y.e[e]), sum[e]);
      };
      if constexpr (OP::SPLIT) {   // hi + lo as in the matrix products (the same results on infinite rows)
        add(dv0, OP::to_float(OP::to_elem(pr)), dr[p]);
        add(dv0, OP::to_float(OP::to_elem_lo(pr)), dr[p]);
        add(dk0, OP::to_float(OP::to_elem(dz)), qr[p]);
        add(dk0, OP::to_float(OP::to_elem_lo(dz)), qr[p]);
      } else {
        add(dv0, pr, dr[p]);
        add(dk0, dz, qr[p]);
      }
    } else if (xk > 0) {
      if (part == 0) {
        sRow[wave][0][rl] = lv;
        sRow[wave][1][rl] = nd;
      }
      elem* dst = &sh.rows[wave][0][TR ? swzq(rl, part) : rl * LD + 8 * part];
#pragma unroll
      for (int c = 0; c < (int)(sizeof(elem) / 2); ++c) {
        reinterpret_cast<uint4*>(dst)[c] = dr[p].u[c];
        reinterpret_cast<uint4*>(dst + TILE * LD)[c] = qr[p].u[c];
      }
    }
  }
  if (!ONE && !stats) return;

#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    qmax = fmaxf(qmax, __shfl_xor(qmax, o));
    lmin = fminf(lmin, __shfl_xor(lmin, o));
  }
  if (lane == 0) {
    sStat[wave][0] = qmax;
    sStat[wave][1] = lmin;
  }
  auto store_stat = [&]() {   // (after a barrier)
    if (tid != 0) return;
    for (int w = 1; w < NWAVES; ++w) {
      qmax = fmaxf(qmax, sStat[w][0]);
      lmin = fminf(lmin, sStat[w][1]);
    }
    reach.qstat[(int64_t)r * reach.nseg + seg] = make_float2(sqrtf(qmax), lmin);
  };
  float4* dst = reinterpret_cast<float4*>(reach.xpart + ((int64_t)r * reach.nseg + seg) * xk * 2 * D);
  if constexpr (ONE) {
    // the key's sums: a lane's rows, then four lane groups at a time, then those
    constexpr int QUADS = 2 * D / 4, SLICES = NTHREADS / QUADS;
    static_assert(NWAVES * RPW == 4 * SLICES, "four lane groups per thread");
    float4* mine = reinterpret_cast<float4*>(sh.sum[wave * RPW + lane / LPR]) + 2 * part;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      mine[c] = make_float4(dk0[4 * c], dk0[4 * c + 1], dk0[4 * c + 2], dk0[4 * c + 3]);
      mine[D / 4 + c] = make_float4(dv0[4 * c], dv0[4 * c + 1], dv0[4 * c + 2], dv0[4 * c + 3]);
    }
    __syncthreads();
    store_stat();
    const int quad = tid % QUADS, slice = tid / QUADS;
    auto add = [](const float4& x, const float4& y) { return make_float4(x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w); };
    float4 x = reinterpret_cast<const float4*>(sh.sum[4 * slice])[quad];
#pragma unroll
    for (int i = 1; i < 4; ++i) x = add(x, reinterpret_cast<const float4*>(sh.sum[4 * slice + i])[quad]);
    sh.part[tid] = x;
    __syncthreads();
    if (slice != 0) return;
#pragma unroll
    for (int i = 1; i < SLICES; ++i) x = add(x, sh.part[i * QUADS + quad]);
    dst[quad] = x;
    return;
  } else {
    f32x16 dkx[DB], dvx[DB];
    if (xk > 0) {
      // the first keys and values (B operands: lane = key), and the rows as A operands (lane = query row). The
      // fp32 products run over the head dim with lane half h at elements [h D/2, (h+1) D/2), so that both load
      // as 16-byte pieces.
      const elem* kh = k + ks.at(b, hh) + (int64_t)min(n, T - 1) * ks.row;   // (columns from xk on are masked)
      const elem* vh = v + vs.at(b, hh) + (int64_t)min(n, T - 1) * vs.row;
      constexpr int PIECES = sizeof(elem) == 2 ? NS : D / 8;
      constexpr int STEP = sizeof(elem) == 2 ? 16 : 4;   // elements between a lane's pieces
      const int at = sizeof(elem) == 2 ? 8 * h : h * (D / 2);
      uint4 kx[PIECES], vx[PIECES];
#pragma unroll
      for (int s = 0; s < PIECES; ++s) {
        kx[s] = *reinterpret_cast<const uint4*>(kh + at + STEP * s);
        vx[s] = *reinterpret_cast<const uint4*>(vh + at + STEP * s);
      }
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        dkx[db] = zero16();
        dvx[db] = zero16();
      }
      lds_wave_sync();
      auto piece = [&](int x, int s) -> uint4 {
        const elem* y = sh.rows[wave][x];
        if constexpr (TR) return *reinterpret_cast<const uint4*>(y + swzq(n, 2 * s + h));
        else return *reinterpret_cast<const uint4*>(y + n * LD + at + STEP * s);
      };
      auto mma_piece = [&](const uint4& a, const uint4& b4, f32x16 c) -> f32x16 {
        if constexpr (sizeof(elem) == 2) {
          return OP::mma(*reinterpret_cast<const frag*>(&a), *reinterpret_cast<const frag*>(&b4), c);
        } else {
          c = OP::mma(__uint_as_float(a.x), __uint_as_float(b4.x), c);
          c = OP::mma(__uint_as_float(a.y), __uint_as_float(b4.y), c);
          c = OP::mma(__uint_as_float(a.z), __uint_as_float(b4.z), c);
          return OP::mma(__uint_as_float(a.w), __uint_as_float(b4.w), c);
        }
      };
      // acc[db] (D x keys) += Y^T X: Y the wavefront's rows, X a (queries x keys) tile
      auto acc_t = [&](f32x16 (&acc)[DB], int which, const f32x16& x) {
        const elem* y = sh.rows[wave][which];
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int s = 0; s < AS; ++s) {
            frag yt;
            if constexpr (TR) {
              yt = get_trq<true>(y, lane, db, s);
            } else if constexpr (sizeof(elem) == 2) {
#pragma unroll
              for (int e = 0; e < 8; ++e) {
                const elem raw = y[(16 * s + 8 * (e >> 2) + 4 * h + (e & 3)) * LD + db * 32 + n];
                yt[e] = *reinterpret_cast<const bf16_t*>(&raw);
              }
            } else {
              yt = y[crow(s, h) * LD + db * 32 + n];
            }
            acc[db] = OP::mma(yt, OP::from_acc(x, s), acc[db]);
            if constexpr (OP::SPLIT) acc[db] = OP::mma(yt, OP::from_acc_lo(x, s), acc[db]);
          }
      };
      f32x16 p = zero16(), dz = rows16(sRow[wave][1], h);
#pragma unroll
      for (int s = 0; s < PIECES; ++s) {
        p = mma_piece(piece(1, s), kx[s], p);
        dz = mma_piece(piece(0, s), vx[s], dz);
      }
      const f32x16 ls = rows16(sRow[wave][0], h);
      const float sl2 = scale * LOG2E;
      const int thr = n < xk ? n - qbase - 4 * h : 32;   // key n <= query qbase + crow(i, h)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        p[i] = crow(i, 0) >= thr ? fast_exp2(fmaf(p[i], sl2, -ls[i])) : 0.f;
        dz[i] = p[i] * dz[i];
      }
      acc_t(dvx, 0, p);
      acc_t(dkx, 1, dz);
    }
    __syncthreads();
    store_stat();
    if (xk == 0) return;
    for (int j0 = 0; j0 < xk; j0 += 8) {   // (every wavefront is past its reads of the rows)
      if (n >= j0 && n < min(j0 + 8, xk)) {
        float* mine = &sh.sum[wave][(n - j0) * SUMLD];
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int a = 0; a < 4; ++a) {
            const int d = db * 32 + 8 * a + 4 * h;
            *reinterpret_cast<float4*>(mine + d) =
                make_float4(dkx[db][4 * a], dkx[db][4 * a + 1], dkx[db][4 * a + 2], dkx[db][4 * a + 3]);
            *reinterpret_cast<float4*>(mine + D + d) =
                make_float4(dvx[db][4 * a], dvx[db][4 * a + 1], dvx[db][4 * a + 2], dvx[db][4 * a + 3]);
          }
      }
      __syncthreads();
      const int quads = min(8, xk - j0) * (2 * D / 4);
      for (int i = tid; i < quads; i += NTHREADS) {
        const int at = (i / (2 * D / 4)) * SUMLD + 4 * (i % (2 * D / 4));
        float4 x = *reinterpret_cast<const float4*>(&sh.sum[0][at]);
#pragma unroll
        for (int w = 1; w < NWAVES; ++w) {
          const float4 y = *reinterpret_cast<const float4*>(&sh.sum[w][at]);
          x = make_float4(x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w);
        }
        dst[j0 * (2 * D / 4) + i] = x;
      }
      __syncthreads();
    }
  }
}

// What a key-side wavefront's search reads first, loaded before its key rows so that the search adds no wait of
// its own to them: the carry of its first round of probes (kv_last_block), and two of the head's row segments
// per lane. (Key side, us, the search's loads behind the key rows / before them: B=1 H=16 T=16384 bf16, most tiles
// left out 185 / 176; B=1 H=12 T=16384, none left out 1371 / 1367; fp32 B=1 H=8 T=2048, none 377 / 371.)
struct KvProbe {
  float f[4];
  float2 q[2];
};
// The query block of a lane group's first probe: the last one, where nothing can be left out all there is to know,
// and, for the usual reach of a few tiles, the blocks 2, 4, ... 128 on.
__device__ __forceinline__ int kv_first_probe(int key0, int i, int NB) {
  return i == 7 ? NB - 1 : min(key0 / TILE + (2 << i), NB - 1);
}
__device__ __forceinline__ KvProbe kv_probe(const BwdReach& reach, int64_t r, const float* carry_b, int T, int NB,
                                            int key0, int lane) {
  KvProbe x{};
  if (reach.qstat) {
    const float* p = carry_b + (int64_t)kv_first_probe(key0, lane >> 3, NB) * T;
#pragma unroll
    for (int e = 0; e < 4; ++e) x.f[e] = p[min(key0 + 4 * (lane & 7) + e, T - 1)];
#pragma unroll
    for (int i = 0; i < 2; ++i) x.q[i] = reach.qstat[r * reach.nseg + min(lane + 64 * i, reach.nseg - 1)];
  }
  return x;
}

// Whether the search can find anything: every key of the wavefront (but those that do not count) has received
// enough before the last query block. Only the time depends on the answer (see reach_worth).
__device__ __forceinline__ bool kv_worth(const KvProbe& x, int key0, int T, int xk, int lane) {
  bool ok = true;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int j = key0 + 4 * (lane & 7) + e;
    ok = ok && (j >= T || j < xk || x.f[e] * LOG2E > REACH_WORTH);
  }
  return __all(lane < 56 || ok);
}

// (Measured, N(0,1) inputs, B=1 H=16 T=16384 bf16: the key side 1560 -> 176 us, the query side 1510 -> 203 us.)
// The last query block on which some key of a wavefront's 32 (from key0) keeps a weight that is not an
// exact zero, of the blocks up to NB - 1 (the key tile's own block at least): a lane group of 8 probes one
// block (4 keys per lane), eight blocks at a time; the history never falls, so the blocks past the last
// one are all without weight. thr: see find_reach, with the head's least lse for the row maxima. Keys
// below xk (their gradients are taken elsewhere) and past the end do not count.
__device__ __forceinline__ int kv_last_block(const KvProbe& first, const float* carry_b, int T, int NB, int key0, int xk,
                                             float thr, int lane) {
  const int part = lane >> 3, j0 = key0 + 4 * (lane & 7);
  auto gone = [&](const float (&f)[4]) {
    bool ok = thr < INFINITY;   // every comparison that meets a NaN keeps the block
#pragma unroll
    for (int e = 0; e < 4; ++e) ok = ok && (j0 + e >= T || j0 + e < xk || f[e] * REACH_F > thr);
    return ok;
  };
  int lo = key0 / TILE, hi = NB;   // lo: kept; hi: without weight (or past the end)
  auto narrow = [&](const float (&f)[4], auto probe) {   // f: the lane's carry at probe(part); probe(i), i = 0..7, ascending
    const uint64_t m = __ballot(gone(f));
    int nlo = lo, nhi = hi;
#pragma unroll
    for (int i = 7; i >= 0; --i) {
      const int p = probe(i);
      if (((m >> (8 * i)) & 0xFF) == 0xFF) nhi = min(nhi, p);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int p = probe(i);
      if (((m >> (8 * i)) & 0xFF) != 0xFF && p < nhi) nlo = max(nlo, p);
    }
    lo = nlo;
    hi = nhi;
  };
  narrow(first.f, [&](int i) { return kv_first_probe(key0, i, NB); });
  if (hi == NB) return NB - 1;
  while (hi - lo > 1) {
    const int from = lo, stride = max(1, (hi - lo) / 9), end = hi - 1;
    auto probe = [&](int i) { return min(from + (i + 1) * stride, end); };
    const float* p = carry_b + (int64_t)probe(part) * T;
    float f[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = p[min(j0 + e, T - 1)];
    narrow(f, probe);
  }
  return lo;
}

// The head's bounds from its row segments: the largest |q| and the least lse. first: two of them per lane.
__device__ __forceinline__ float2 head_qstat(const BwdReach& reach, int64_t r, int lane, const float2 (&first)[2]) {
  float qm = fmaxf(first[0].x, first[1].x), lm = fminf(first[0].y, first[1].y);
  for (int i = lane + 128; i < reach.nseg; i += 64) {
    const float2 x = reach.qstat[r * reach.nseg + i];
    qm = fmaxf(qm, x.x);
    lm = fminf(lm, x.y);
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    qm = fmaxf(qm, __shfl_xor(qm, o));
    lm = fminf(lm, __shfl_xor(lm, o));
  }
  return make_float2(qm, lm);
}

// kv_last_block's threshold of one head for a wavefront's keys: kk, vv the sums of squares of the lane's parts of
// its key and value.
__device__ __forceinline__ float kv_threshold(float kk, float vv, const float2& qstat, float scale) {
  kk += xor32(kk);
  vv += xor32(vv);
  const float kn = sqrtf(half_max(kk < REACH_NORM2 && vv < REACH_NORM2 ? kk : INFINITY));
  const float t = fmaf(qstat.x * scale * REACH_Q, kn, REACH_ZERO - qstat.y);
  return t < INFINITY ? t : INFINITY;   // (a NaN, from 0 * inf, keeps everything)
}

// The query blocks (NB - 1 at most) that a key-side workgroup's sweep starts from, once every wavefront's
// last block is in last[]; the query side finds it in hi, and reads the selection-suffix checkpoints of
// whole groups of eight query blocks: the rows of the sweep's group past its start hold zeros.
__device__ __forceinline__ int kv_sweep_start(const int* last, int NB, int qb_lo, int wave, int lane, int key0, int T,
                                              float* uplane, int* hi) {
  int top = qb_lo + NWAVES - 1;
#pragma unroll
  for (int w = 0; w < NWAVES; ++w) top = max(top, last[w]);
  top = min(__builtin_amdgcn_readfirstlane(top), NB - 1);
  if (wave == 0 && lane == 0) *hi = top;
  const int j = key0 + lane;
  for (int qb = top + 1; qb <= min(top | 7, NB - 1); ++qb)
    if (lane < TILE && j < T) uplane[utri_row(qb) + j] = 0.f;
  return top;
}

// in (R = nseq * H views of T rows, Strides is) -> outT (R, D, ldt), zero past T; a workgroup moves
// a [64 t][D] slab through LDS in 16-byte chunks: row chunks in, then 8 (bf16) or 4 (fp32)
// consecutive t of one d out.
template <typename E, int D>
__global__ __launch_bounds__(NTHREADS) void transpose_kernel(const E* __restrict__ in, E* __restrict__ outT,
                                                             int T, int64_t ldt, Strides is, int H) {
  constexpr int EPC = 16 / (int)sizeof(E);
  constexpr int LDS_LD = D + EPC;   // padded row: 16-byte aligned, rows on shifted banks
  __shared__ __attribute__((aligned(16))) E tile[64 * LDS_LD];
  const int64_t r = blockIdx.y;
  const int t0 = blockIdx.x * 64;
  const E* src = in + is.at(r / H, r % H);
  for (int c = threadIdx.x; c < 64 * D / EPC; c += NTHREADS) {
    const int tt = c / (D / EPC), d0 = (c % (D / EPC)) * EPC;
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    if (t0 + tt < T) v = *reinterpret_cast<const uint4*>(src + (int64_t)(t0 + tt) * is.row + d0);
    *reinterpret_cast<uint4*>(&tile[tt * LDS_LD + d0]) = v;
  }
  __syncthreads();
  E* dst = outT + r * D * ldt;
  for (int c = threadIdx.x; c < D * 64 / EPC; c += NTHREADS) {
    const int d = c % D, tt0 = (c / D) * EPC;
    union {
      uint4 v;
      E e[EPC];
    } u;
#pragma unroll
    for (int e = 0; e < EPC; ++e) u.e[e] = tile[(tt0 + e) * LDS_LD + d];
    if (t0 + tt0 < ldt) *reinterpret_cast<uint4*>(dst + (int64_t)d * ldt + t0 + tt0) = u.v;
  }
}

// The same transpose for 2-byte elements without LDS: a thread moves one 8 x 8 block (8 t, 8 d) --
// eight 16-byte row loads (t past T read as zero), the block transposed in registers (each output
// word joins the same half-word of two rows), eight 16-byte column stores. A wavefront's loads and
// stores cover whole 128-byte segments (eight lanes per row or column).
template <int D>
__global__ __launch_bounds__(NTHREADS) void transpose8_kernel(const uint16_t* __restrict__ in,
                                                              uint16_t* __restrict__ outT, int T, int64_t ldt,
                                                              Strides is, int H) {
  constexpr int CB = D / 8;   // 8-column blocks per row
  const int64_t r = blockIdx.y;
  const int c = threadIdx.x % CB;
  const int64_t t0 = ((int64_t)blockIdx.x * (NTHREADS / CB) + threadIdx.x / CB) * 8;
  if (t0 >= ldt) return;
  const uint16_t* src = in + is.at(r / H, r % H) + 8 * c;
  uint4 v[8];
#pragma unroll
  for (int k = 0; k < 8; ++k)
    v[k] = (t0 + k < T) ? *reinterpret_cast<const uint4*>(src + (t0 + k) * is.row) : make_uint4(0u, 0u, 0u, 0u);
  auto word = [&](int k, int w) -> uint32_t {
    return w == 0 ? v[k].x : (w == 1 ? v[k].y : (w == 2 ? v[k].z : v[k].w));
  };
  uint16_t* dst = outT + r * D * ldt + t0;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    uint32_t o[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const uint32_t lo = word(2 * w, e >> 1), hi = word(2 * w + 1, e >> 1);
      o[w] = (e & 1) ? ((lo >> 16) | (hi & 0xFFFF0000u)) : ((lo & 0xFFFFu) | (hi << 16));
    }
    *reinterpret_cast<uint4*>(dst + (int64_t)(8 * c + e) * ldt) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

// in (R views, Strides is) -> outT (R, D, ldt), ldt a multiple of 64, zero past T.
template <typename E, int D>
void launch_transpose(const E* in, E* outT, int T, int64_t ldt, const Strides& is, int H, int64_t R,
                      hipStream_t st) {
  if constexpr (sizeof(E) == 2) {
    constexpr int rows_per_block = NTHREADS / (D / 8) * 8;
    const dim3 grid((unsigned)cdiv(ldt, rows_per_block), (unsigned)R);
    hipLaunchKernelGGL((transpose8_kernel<D>), grid, dim3(NTHREADS), 0, st, reinterpret_cast<const uint16_t*>(in),
                       reinterpret_cast<uint16_t*>(outT), T, ldt, is, H);
  } else {
    hipLaunchKernelGGL((transpose_kernel<E, D>), dim3((unsigned)cdiv(ldt, 64), (unsigned)R), dim3(NTHREADS), 0, st,
                       in, outT, T, ldt, is, H);
  }
}

// ---------------------------------------------------------------------------------------------
// Backward kernel shapes of the generic instances (every storage type and head dim but bf16 at 64,
// which bwd_kv64_kernel / bwd_dq64_kernel take): each tile is loaded into registers, stored to LDS
// and computed in turn (one LDS buffer), the load latency left to the CU's other workgroup. Both
// sides fit two workgroups per CU at bf16 head dims <= 64: the key side's K and V rows sit in LDS,
// the query side's Q and dO rows and row statistics in registers.
template <class OP, int D>
constexpr int dq_min_blocks() { return (sizeof(typename OP::elem) == 2 && D <= 64) ? 2 : 1; }
template <class OP, int D, int G>
constexpr int kv_min_blocks() { return (sizeof(typename OP::elem) == 2 && D <= 64 && G == 1) ? 2 : 1; }

// ---------------------------------------------------------------------------------------------
// Gradient stores to a caller's view (fp32 or bf16 elements): one element, or four consecutive
// elements of a row (d a multiple of 4; the views' rows start 16-byte aligned).
__device__ __forceinline__ void store_grad1(const GradView& v, int64_t b, int hh, int row, int d, float x) {
  const int64_t o = v.s.at(b, hh) + (int64_t)row * v.s.row + d;
  if (v.f32) static_cast<float*>(v.p)[o] = x;
  else static_cast<uint16_t*>(v.p)[o] = OpBF16::to_elem(x);
}
__device__ __forceinline__ void store_grad4(const GradView& v, int64_t b, int hh, int row, int d, float4 x) {
  const int64_t o = v.s.at(b, hh) + (int64_t)row * v.s.row + d;
  if (v.f32) {
    *reinterpret_cast<float4*>(static_cast<float*>(v.p) + o) = x;
  } else {
    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(v.p) + o) =
        make_uint2((uint32_t)OpBF16::to_elem(x.x) | ((uint32_t)OpBF16::to_elem(x.y) << 16),
                   (uint32_t)OpBF16::to_elem(x.z) | ((uint32_t)OpBF16::to_elem(x.w) << 16));
  }
}

// ---------------------------------------------------------------------------------------------
// Backward helpers on (queries x keys) C-layout tiles: lane n holds key j = key0 + n, rows are the
// queries qbase + crow(i, h), i = 0..15 (h = lane / 32).

// Backward tiles hold (queries x keys) in C layout: lane n is key j, element i is query row
// qbase + crow(i, h). Rows past the sequence end need no mask here: their Q, dO rows are staged as
// zeros and their lse as +inf, so their logits, selection, P and dz are all zero. The remaining
// masks compare the row's offset within its half-wavefront, crow(i, 0), with a per-lane threshold:
//   P, dz:     j <= r  (and j < T)           <=>  crow(i, 0) >= thr_p = j - qbase - 4h  (32 if j >= T)
//   selection: j <  r  (and exempt <= j < T) <=>  crow(i, 0) >  thr_s = j - qbase - 4h  (32 if not)
struct TileMasks {
  int thr_p, thr_s;
  __device__ __forceinline__ TileMasks(int j, int qbase, int T, int exempt, int h, int xk = 0) {
    const int d = j - qbase - 4 * h;
    thr_p = (j < T && j >= xk) ? d : 32;   // (keys below xk: no P, no dz)
    thr_s = (j < T && j >= exempt) ? d : 32;
  }
};

// Head 0's selection on a tile of its raw logits l0 = q.k, in the same unscaled units (relu(s x) =
// s relu(x) for s > 0): sel = relu(l0) where exempt <= j < r < T, and the negated history
// fs[r, j] = nhist - sum of sel over the tile's earlier rows, nhist = -(the selection before the
// tile) / s (the running sum runs down the rows; the half-wavefronts exchange partial sums). A
// logit product accumulating onto fs then yields q.k - F/s. Bit i of gate is sel[i] > 0, the gate
// of the gradient path. `edge` (wave-uniform) marks tiles where some pair fails exempt <= j < r:
// the mask is applied there (every tile when ALWAYS, which costs a few instructions per element
// but no branch).
template <bool ALWAYS>
__device__ __forceinline__ void selection_tile(const f32x16& l0, float nhist, int h, bool edge,
                                               const TileMasks& mk, uint32_t& gate, f32x16& fs) {
  f32x16 sel;
  // relu as one v_med3 (fmaxf on a product's result would first be canonicalised)
#pragma unroll
  for (int i = 0; i < 16; ++i) sel[i] = __builtin_amdgcn_fmed3f(l0[i], 0.f, 3.0e38f);
  if (ALWAYS || edge) {
#pragma unroll
    for (int i = 0; i < 16; ++i) sel[i] = crow(i, 0) > mk.thr_s ? sel[i] : 0.f;
  }
  gate = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) gate |= sel[i] > 0.f ? (1u << i) : 0u;
  float run = nhist;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const Halves g = halves(((sel[4 * a] + sel[4 * a + 1]) + sel[4 * a + 2]) + sel[4 * a + 3]);
    float p = (h == 0) ? run : run - g.lo;   // rows 8a..8a+3 sit in the low half, 8a+4.. in the high
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      fs[4 * a + t] = p;
      p -= sel[4 * a + t];
    }
    run = (run - g.lo) - g.hi;
  }
}

// Selection gradient path: U[r, j] = u_in + sum of z over the tile's later rows, and
// g = -U where the gate is set, else 0. Returns u_in + the sum over the whole tile (U entering the
// tile above). The sum runs negated so the select takes -U without a modifier.
__device__ __forceinline__ float gpath_tile(const f32x16& z, float u_in, uint32_t gate, int h, f32x16& gp) {
  float nrun = -u_in;
#pragma unroll
  for (int a = 3; a >= 0; --a) {
    const Halves g = halves(((z[4 * a + 3] + z[4 * a + 2]) + z[4 * a + 1]) + z[4 * a]);
    float np = (h == 1) ? nrun : nrun - g.hi;
#pragma unroll
    for (int t = 3; t >= 0; --t) {
      const int i = 4 * a + t;
      gp[i] = ((gate >> i) & 1u) ? np : 0.f;
      np -= z[i];
    }
    nrun = (nrun - g.hi) - g.lo;
  }
  return -nrun;
}

// P = exp2(s log2e lg - lse) and dz = P dpb on a tile, lg = q.k - F/s, dpb = dO.v - dbar (the
// product accumulated onto -dbar); lse of the tile's rows comes from LDS (4 consecutive rows per
// float4). Pairs outside j <= r, j < T are zeroed on `edge` tiles (every tile when ALWAYS).
template <bool ALWAYS>
__device__ __forceinline__ void p_dz_tile(const f32x16& lg, const f32x16& dpb, const float* slse, float sl2,
                                          int h, bool edge, const TileMasks& mk, f32x16& pr, f32x16& dz) {
  if constexpr (ALWAYS) {
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const float4 ls = *reinterpret_cast<const float4*>(slse + 8 * a + 4 * h);
      const float lsv[4] = {ls.x, ls.y, ls.z, ls.w};
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int i = 4 * a + t;
        const float p = fast_exp2(fmaf(lg[i], sl2, -lsv[t]));
        pr[i] = crow(i, 0) >= mk.thr_p ? p : 0.f;
        dz[i] = pr[i] * dpb[i];
      }
    }
  } else {
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const float4 ls = *reinterpret_cast<const float4*>(slse + 8 * a + 4 * h);
      const float lsv[4] = {ls.x, ls.y, ls.z, ls.w};
#pragma unroll
      for (int t = 0; t < 4; ++t) pr[4 * a + t] = fast_exp2(fmaf(lg[4 * a + t], sl2, -lsv[t]));
    }
    if (edge) {
#pragma unroll
      for (int i = 0; i < 16; ++i) pr[i] = crow(i, 0) >= mk.thr_p ? pr[i] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) dz[i] = pr[i] * dpb[i];
  }
}

// p_dz_tile with the rows' lse values already in registers (element i: row crow(i, h)).
__device__ __forceinline__ void p_dz_tile_r(const f32x16& lg, const f32x16& dpb, const f32x16& lsev, float sl2,
                                            bool edge, const TileMasks& mk, f32x16& pr, f32x16& dz) {
#pragma unroll
  for (int i = 0; i < 16; ++i) pr[i] = fast_exp2(fmaf(lg[i], sl2, -lsev[i]));
  if (edge) {
#pragma unroll
    for (int i = 0; i < 16; ++i) pr[i] = crow(i, 0) >= mk.thr_p ? pr[i] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) dz[i] = pr[i] * dpb[i];
}

// Whether some value of the wavefront's tile is large enough for the split-operand products (the
// rounding of a bf16 operand then matters beside the others): g sums dz over every later query of
// the group's heads and can outgrow the dz tiles many times. Taken on g, and on head 0's dz + g.
__device__ __forceinline__ bool big_tile(const f32x16& x) {
  bool big = false;
#pragma unroll
  for (int i = 0; i < 16; ++i) big |= fabsf(x[i]) > 0.25f;
  return __any(big);
}

// ---------------------------------------------------------------------------------------------
// Backward, key side. grid (ceil(T/128), nseq * H/G); wavefront w owns keys [x*128 + 32w, +32) of
// heads [gi*G, gi*G+G) and sweeps the query tiles last to first, with K, V and the dK, dV sums in
// registers. The selection suffix U (over this group's heads) is checkpointed on entry to every
// query tile, for the dQ kernel, into row qb (keys j < 32 (qb + 1)) of the (gi, b) plane of ucheck,
// a lower-triangular plane of rows laid end to end (utri_row). Head 0's dK gets g = -gate*U from every
// group: the group holding head 0 folds it into head 0's dz; the others add their share to dk0x.

// CV: every view is the contiguous (nseq, H, T, D) layout of sa_backward (see fwd_kernel).
template <class OP, int D, int G, bool CV>
__global__ __launch_bounds__(NTHREADS, (kv_min_blocks<OP, D, G>())) void bwd_kv_kernel(
    const typename OP::elem* __restrict__ q, const typename OP::elem* __restrict__ k,
    const typename OP::elem* __restrict__ v, const typename OP::elem* __restrict__ qt,
    const typename OP::elem* __restrict__ dout, const typename OP::elem* __restrict__ dot, Strides qs,
    Strides ks, Strides vs, Strides dos, const float* __restrict__ lse, const float* __restrict__ dbar,
    const float* __restrict__ carry, float* __restrict__ ucheck, float* __restrict__ dk0h, float* __restrict__ dk0x,
    GradView dkv, GradView dvv, int nseq, int H, int T, int64_t ldt, int exempt, float scale, BwdReach reach) {
  using elem = typename OP::elem;
  using frag = typename OP::frag;
  constexpr int NS = D / OP::KS;
  constexpr int DB = D / 32;
  constexpr int LDK = D + OP::KPAD;
  constexpr int LDV = TILE + OP::TPAD;
  constexpr int AS = OP::acc_steps;
  constexpr int NH = G + 1;   // staged heads: the group, then head 0 when outside the group
  constexpr int TILE_BYTES = (NH * (TILE * LDK + D * LDV) + G * (TILE * LDK + D * LDV)) * (int)sizeof(elem);

  __shared__ __attribute__((aligned(16))) elem sQ[NH][TILE * LDK];
  __shared__ __attribute__((aligned(16))) elem sQt[NH][D * LDV];
  __shared__ __attribute__((aligned(16))) elem sdO[G][TILE * LDK];
  __shared__ __attribute__((aligned(16))) elem sdOt[G][D * LDV];
  __shared__ __attribute__((aligned(16))) float sLse[G][TILE];
  __shared__ __attribute__((aligned(16))) float sDb[G][TILE];
  // Each wavefront's K and V rows are read from LDS per tile instead of being held in registers,
  // when they fit unpadded (swz64) beside the query tiles in half the CU's LDS: the registers they
  // free let two workgroups share a CU. Head 0's K rows (for a group without head 0) stay in
  // registers.
  constexpr int NKV = 2 * G;   // K, V of each head of the group
  constexpr int OTHER_LDS = TILE_BYTES + 2 * G * TILE * 4;
  constexpr bool KVLDS = sizeof(elem) == 2 && D == 64 && OTHER_LDS + NWAVES * NKV * TILE * D * 2 <= 80 * 1024;
  __shared__ __attribute__((aligned(16))) elem sKV[KVLDS ? NWAVES : 1][KVLDS ? NKV : 1][KVLDS ? TILE * D : 8];

  __shared__ int sLast[NWAVES];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int n = lane & 31, h = lane >> 5;
  const int groups = H / G;
  const BlockXY bxy = work_order_block();
  const int b = bxy.y / groups, gi = bxy.y % groups;
  const int hd0 = gi * G;
  const bool has_h0 = (gi == 0);
  const int NB = (T + TILE - 1) / TILE;
  const int key0 = bxy.x * (NWAVES * TILE) + wave * TILE;
  const int j = key0 + n;
  const int64_t seq_row = (int64_t)b * H;
  // view accessors (CV: the contiguous layout, strides as compile-time facts)
  auto view_head = [&](const elem* base, const Strides& vs_, int hh) -> const elem* {
    if constexpr (CV) return base + (seq_row + hh) * T * D;
    else return base + vs_.at(b, hh);
  };
  auto view_ld = [&](const Strides& vs_) -> int64_t {
    if constexpr (CV) return D;
    else return vs_.row;
  };
  float* uplane = ucheck + ((int64_t)gi * nseq + b) * utri_floats(NB);
  const float* carry_col = carry + (int64_t)b * NB * T + (j < T ? j : 0);

  KvProbe probe[G];   // (the carry is the same for every head)
#pragma unroll
  for (int g = 0; g < G; ++g)
    probe[g] = kv_probe(reach, seq_row + hd0 + g, carry + (int64_t)b * NB * T, T, NB, key0, lane);
  // Key-side operands (B operands: lane = key column): this wavefront's K and V rows of the group
  // and head 0's K rows, in its LDS rows or in registers.
  frag kf[KVLDS ? 1 : G][NS], vf[KVLDS ? 1 : G][NS], k0f[NS];
  if constexpr (KVLDS) {
    constexpr int CPR = D / 8;
    for (int c = lane; c < TILE * CPR; c += 64) {
      const int r = c / CPR, cc = c % CPR;
      const int64_t jr = min(key0 + r, T - 1);
      const bool ok = key0 + r < T;
      auto put = [&](int x, const elem* src, int64_t ld) {
        const uint4 v4 = *reinterpret_cast<const uint4*>(src + jr * ld + cc * 8);
        *reinterpret_cast<uint4*>(&sKV[wave][x][swz64(r, cc)]) =
            make_uint4(ok ? v4.x : 0u, ok ? v4.y : 0u, ok ? v4.z : 0u, ok ? v4.w : 0u);
      };
#pragma unroll
      for (int g = 0; g < G; ++g) {
        put(2 * g, view_head(k, ks, hd0 + g), view_ld(ks));
        put(2 * g + 1, view_head(v, vs, hd0 + g), view_ld(vs));
      }
    }
    if (!has_h0) {
      const elem* kh = view_head(k, ks, 0);
#pragma unroll
      for (int s = 0; s < NS; ++s) k0f[s] = ld_std_bounded<OP>(kh, view_ld(ks), j, T, h, s);
    }
  } else {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const elem* kh = view_head(k, ks, hd0 + g);
      const elem* vh = view_head(v, vs, hd0 + g);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        kf[g][s] = ld_std_bounded<OP>(kh, view_ld(ks), j, T, h, s);
        vf[g][s] = ld_std_bounded<OP>(vh, view_ld(vs), j, T, h, s);
      }
    }
    if (!has_h0) {
      const elem* kh = view_head(k, ks, 0);
#pragma unroll
      for (int s = 0; s < NS; ++s) k0f[s] = ld_std_bounded<OP>(kh, view_ld(ks), j, T, h, s);
    }
  }
  // fragment s of row n (this lane's key) of LDS row block x
  auto kv_lds = [&](int x, int s) -> frag {
    if constexpr (KVLDS) return *reinterpret_cast<const frag*>(&sKV[wave][x][swz64(n, 2 * s + h)]);
    else return OP::zero();
  };
  auto k_frag = [&](int g, int s) -> frag {
    if constexpr (KVLDS) return kv_lds(2 * g, s);
    else return kf[g][s];
  };
  auto v_frag = [&](int g, int s) -> frag {
    if constexpr (KVLDS) return kv_lds(2 * g + 1, s);
    else return vf[g][s];
  };
  // head 0's K: the group's own when it holds head 0 (h0)
  auto k0_frag = [&](bool h0, int s) -> frag {
    if constexpr (KVLDS) {
      return h0 ? kv_lds(0, s) : k0f[s];
    } else {
      return h0 ? kf[0][s] : k0f[s];
    }
  };

  f32x16 dkt[G][DB], dvt[G][DB], dk0t[DB];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      dkt[g][db] = zero16();
      dvt[g][db] = zero16();
    }
#pragma unroll
  for (int db = 0; db < DB; ++db) dk0t[db] = zero16();

  float ucarry = 0.f;
  const float sl2 = scale * LOG2E;
  const float neg_inv_scale = -1.f / scale;
  // query tiles the workgroup visits, last to first: qb_hi down to the first that reaches its keys
  const int qb_lo = bxy.x * NWAVES;
  int qb_hi = NB - 1;   // the first tile of the sweep: later ones hold no weight for the workgroup's keys
  if (reach.qstat) {
    int last = key0 < T ? NB - 1 : 0;
    if (key0 < T && kv_worth(probe[0], key0, T, reach.xk, lane)) {
      if constexpr (KVLDS) lds_wave_sync();   // (the wavefront's own rows)
      float thr = -INFINITY;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        frag kg[NS], vg[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          kg[s] = k_frag(g, s);
          vg[s] = v_frag(g, s);
        }
        const float2 qstat = head_qstat(reach, seq_row + hd0 + g, lane, probe[g].q);
        thr = fmaxf(thr, kv_threshold(frag_sumsq<OP, NS>(kg), frag_sumsq<OP, NS>(vg), qstat, scale));
      }
      last = kv_last_block(probe[0], carry + (int64_t)b * NB * T, T, NB, key0, reach.xk, thr, lane);
    }
    if (lane == 0) sLast[wave] = last;
    __syncthreads();
    qb_hi = kv_sweep_start(sLast, NB, qb_lo, wave, lane, key0, T, uplane,
                           reach.hi + ((int64_t)gi * nseq + b) * reach.nkg + bxy.x);
  }
  const int ntiles = qb_hi - qb_lo + 1;

  // Staging of one query tile: Q, Q^T, dO, dO^T of the group (+ head 0's Q, Q^T), lse, dbar.
  RowTile<elem, D> nQ[NH], ndO[G];
  ColTile<elem, D> nQt[NH], ndOt[G];
  float nLse[G], nDb[G];
  // the query-side rows of this workgroup's heads (computed once, outside the tile loop)
  const elem* q_rows[NH];
  const elem* do_rows[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    q_rows[g] = view_head(q, qs, hd0 + g);
    do_rows[g] = view_head(dout, dos, hd0 + g);
  }
  q_rows[G] = view_head(q, qs, 0);
  const int q_ld = (int)view_ld(qs), do_ld = (int)view_ld(dos);
  auto load_tile = [&](int qb) {
    const int qbase = qb * TILE;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int64_t row = seq_row + hd0 + g;
      nQ[g].load(q_rows[g], q_ld, qbase, T, tid);
      nQt[g].load(qt + row * D * ldt, ldt, qbase, tid);
      ndO[g].load(do_rows[g], do_ld, qbase, T, tid);
      ndOt[g].load(dot + row * D * ldt, ldt, qbase, tid);
      const int r = qbase + (tid & (TILE - 1));   // < ldt: padded rows hold lse = +inf, -dbar = 0
      nLse[g] = lse[row * ldt + r];
      nDb[g] = dbar[row * ldt + r];
    }
    if (!has_h0) {
      nQ[G].load(q_rows[G], q_ld, qbase, T, tid);
      nQt[G].load(qt + seq_row * D * ldt, ldt, qbase, tid);
    }
  };
  auto store_tile = [&]() {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      nQ[g].template store<LDK>(sQ[g], tid);
      nQt[g].template store_crow<LDV>(sQt[g], tid);
      ndO[g].template store<LDK>(sdO[g], tid);
      ndOt[g].template store_crow<LDV>(sdOt[g], tid);
      if (tid < TILE) {
        sLse[g][tid] = nLse[g];
        sDb[g][tid] = nDb[g];
      }
    }
    if (!has_h0) {
      nQ[G].template store<LDK>(sQ[G], tid);
      nQt[G].template store_crow<LDV>(sQt[G], tid);
    }
  };

  // acc[db] (D x keys) += Y^T X: Y a staged transposed LDS tile (rows d, queries in C-layout
  // order), X a C-layout (queries x keys) tile; with split, X also enters as its rounding residual.
  auto acc_t = [&](f32x16 (&acc)[DB], const elem* yt, const f32x16& x, bool split) {
    frag xf[AS];
#pragma unroll
    for (int s = 0; s < AS; ++s) xf[s] = OP::from_acc(x, s);
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int s = 0; s < AS; ++s) acc[db] = OP::mma(OP::ld_perm(yt, LDV, db * 32 + n, h, s), xf[s], acc[db]);
    if constexpr (OP::SPLIT) {
      if (split) {
#pragma unroll
        for (int s = 0; s < AS; ++s) xf[s] = OP::from_acc_lo(x, s);
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int s = 0; s < AS; ++s) acc[db] = OP::mma(OP::ld_perm(yt, LDV, db * 32 + n, h, s), xf[s], acc[db]);
      }
    }
  };

  // Keys below `exempt` are never selected, so they gather attention from every later query and
  // their dV / dK sums run over all of them: their products take the split operands.
  const bool split_keys = key0 < exempt;

  // The tile loop in two instances, for the group holding head 0 and for the others: one loop
  // with a run-time choice between their accumulations makes the compiler copy the sums between
  // register sets every tile.
  auto sweep = [&](auto h0_tag) {
    constexpr bool H0 = decltype(h0_tag)::value;

    // one query tile; INTERIOR: every pair of the tile is unmasked for every wavefront and no key
    // is exempt, so the body is straight-line code without the masks and split products
    auto tile_step = [&](int t, auto interior_tag) {
      constexpr bool INTERIOR = decltype(interior_tag)::value;
      const int qb = qb_hi - t;
      const int qbase = qb * TILE;
      load_tile(qb);
      const float hist = carry_col[(int64_t)qb * T];
      if (t > 0) __syncthreads();   // every wavefront is done with the previous tile
      store_tile();
      __syncthreads();
      if (INTERIOR || qbase + TILE - 1 >= key0) {   // else every query of the tile precedes every key
        if (h == 0 && j < T) uplane[utri_row(qb) + j] = ucarry;   // j < (qb + 1) * TILE here
        // tile body; edge: some pair of the tile is masked (diagonal, sequence end) or exempt
        // (rows past the end and keys past the end need no mask on the key side: the latter's sums
        // stay in their own lanes, which are never written)
        const bool edge = !INTERIOR && ((qbase <= key0 + TILE - 1) || key0 < exempt);
        const bool split = !INTERIOR && split_keys;
        const TileMasks mk(j, qbase, T, exempt, h, reach.xk);
        // (a lambda: inlined late, its loop-invariant parts are not hoisted out of the tile loop,
        // which would hold them in registers across it)
        auto body = [&]() {
          const elem* q0s = H0 ? sQ[0] : sQ[G];
          f32x16 l0 = zero16();
  #pragma unroll
          for (int s = 0; s < NS; ++s) l0 = OP::mma(OP::ld_std(q0s, LDK, n, h, s), k0_frag(H0, s), l0);
          f32x16 fs;
          uint32_t gate;
          selection_tile<false>(l0, (j < T) ? hist * neg_inv_scale : 0.f, h, edge, mk, gate, fs);

          // Per head: P and dz, dV^T += dO^T P, dK^T += Q^T dz; then g from the group's dz sum goes to
          // head 0's dK: added to head 0's own dz when the group holds it, else into dk0t.
          f32x16 dzsum, dz0;
  #pragma unroll
          for (int g = 0; g < G; ++g) {
            f32x16 lg;   // q.k - F/s
            if (H0 && g == 0) {   // head 0 itself: its logits are l0
  #pragma unroll
              for (int i = 0; i < 16; ++i) lg[i] = l0[i] + fs[i];
            } else {
              lg = fs;
  #pragma unroll
              for (int s = 0; s < NS; ++s) lg = OP::mma(OP::ld_std(sQ[g], LDK, n, h, s), k_frag(g, s), lg);
            }
            f32x16 dp = rows16(sDb[g], h);   // dO.v - dbar
  #pragma unroll
            for (int s = 0; s < NS; ++s) dp = OP::mma(OP::ld_std(sdO[g], LDK, n, h, s), v_frag(g, s), dp);
            f32x16 pr, dz;
            p_dz_tile<false>(lg, dp, sLse[g], sl2, h, edge, mk, pr, dz);
            acc_t(dvt[g], sdOt[g], pr, split);
            if (g == 0) {
              dzsum = dz;
            } else {
  #pragma unroll
              for (int i = 0; i < 16; ++i) dzsum[i] += dz[i];
            }
            if (H0 && g == 0) dz0 = dz;   // head 0's dK waits for g
            else acc_t(dkt[g], sQt[g], dz, split);
          }
          f32x16 gp;
          ucarry = gpath_tile(dzsum, ucarry, gate, h, gp);
          if constexpr (H0) {
  #pragma unroll
            for (int i = 0; i < 16; ++i) dz0[i] += gp[i];
            acc_t(dkt[0], sQt[0], dz0, true);
          } else {
            acc_t(dk0t, sQt[G], gp, big_tile(gp));
          }
        };
        body();
      }
    };
    // The last NWAVES tiles hold the wavefronts' diagonals; a workgroup with an exempt key runs
    // every tile with the masks.
    const int n_int = (qb_lo * TILE < exempt) ? 0 : max(ntiles - NWAVES, 0);
    for (int t = 0; t < n_int; ++t) tile_step(t, std::true_type{});
    for (int t = n_int; t < ntiles; ++t) tile_step(t, std::false_type{});
  };
  if (has_h0) sweep(std::true_type{});
  else sweep(std::false_type{});

  if (j >= T || j < reach.xk) return;   // (the first xk keys' gradients: bwd_finish_kernel)
  // dV of every head and dK of heads other than 0 go to the caller's views; head 0's dK to its
  // fp32 sums, where the other groups' shares join it
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int hh = hd0 + g;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const int d = db * 32 + 8 * a + 4 * h;
        const float4 kq = make_float4(dkt[g][db][4 * a] * scale, dkt[g][db][4 * a + 1] * scale,
                                      dkt[g][db][4 * a + 2] * scale, dkt[g][db][4 * a + 3] * scale);
        store_grad4(dvv, b, hh, j, d,
                    make_float4(dvt[g][db][4 * a], dvt[g][db][4 * a + 1], dvt[g][db][4 * a + 2], dvt[g][db][4 * a + 3]));
        if (hh == 0 && H > 1) *reinterpret_cast<float4*>(dk0h + ((int64_t)b * T + j) * D + d) = kq;
        else store_grad4(dkv, b, hh, j, d, kq);
      }
  }
  if (!has_h0) {   // this group's share of head 0's dK, in its own slot (group gi: slot gi - 1)
    float* dst = dk0x + ((int64_t)(gi - 1) * nseq * T + (int64_t)b * T + j) * D;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int a = 0; a < 4; ++a)
        *reinterpret_cast<float4*>(dst + db * 32 + 8 * a + 4 * h) =
            make_float4(dk0t[db][4 * a] * scale, dk0t[db][4 * a + 1] * scale, dk0t[db][4 * a + 2] * scale,
                        dk0t[db][4 * a + 3] * scale);
  }
}

// ---------------------------------------------------------------------------------------------
// Backward, key side, bf16 storage at head dim 64 with one head per wavefront (the instance of
// C2, C3, C4's model and C5): bwd_kv_kernel's tile work, with every query tile's operands loaded
// straight from global memory into LDS one tile ahead -- no staging registers, no load latency at
// the start of a tile, one barrier per tile -- into two buffers of unpadded, swizzled tiles: the Q
// and dO rows (and head 0's Q rows) in swzq layout, read as rows by the logit products and
// transposed (get_trq) by the dK, dV products, so no transposed copies are loaded. The wavefront's
// own K rows sit in registers beside head 0's, its V rows in LDS.

// One tile buffer of bwd_kv64_kernel: the Q, dO and head 0's Q rows (swzq), the rows' lse and
// -dbar (slots 32.. repeat rows 0..31), and per wavefront each lane's carry at the tile's first query.
struct KvTileBuf64 {
  __attribute__((aligned(16))) uint16_t r[3][TILE * 64];
  __attribute__((aligned(16))) float stat[2][64];
  __attribute__((aligned(16))) float hist[NWAVES][64];
};

// CV: every view is the contiguous (nseq, H, T, D) layout of sa_backward. SOLO: one-head sequences
// only (every workgroup runs head 0's loop; the other heads' loop, with its registers for head 0's
// K rows and dK share, is not built).
template <bool CV, bool SOLO>
__global__ __launch_bounds__(NTHREADS, 2) void bwd_kv64_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    const uint16_t* __restrict__ dout, Strides qs, Strides ks, Strides vs, Strides dos,
    const float* __restrict__ lse, const float* __restrict__ dbar, const float* __restrict__ carry,
    float* __restrict__ ucheck, float* __restrict__ dk0h, float* __restrict__ dk0x, GradView dkv, GradView dvv,
    int nseq, int H, int T, int64_t ldt, int exempt, float scale, BwdReach reach) {
  using OP = OpBF16;
  using elem = uint16_t;
  using frag = OP::frag;
  constexpr int D = 64, NS = 4, DB = 2, AS = 2;
  constexpr int TW = TILE * D;   // elements of a [32][64] tile
  // The two tile buffers are separate LDS variables, and the tile loop runs in pairs so that
  // every access names its buffer at compile time: the compiler then knows the direct loads into
  // one buffer do not write what the tile reads from the other, and waits for them only at the end
  // of the tile (a single array indexed by tile parity made it wait before the tile's first read).
  // LDS lifetimes (tile t = query tile qb_hi - t):
  //   sB0, sB1  tile t's Q, dO and head 0's Q rows, its rows' lse and -dbar, each wavefront's carry
  //             row, buffer t mod 2. Filled: by direct loads of all four wavefronts (rows a quarter
  //             each; statistics by wavefronts 0 and 1; each its own carry row), for tile 0 before
  //             the first barrier, for tile t in tile step t - 1. Drained: tile step t only (every
  //             product's fragment reads, rows16 / p_dz_tile of the statistics, the carry value; a
  //             wavefront with no pair in the tile reads nothing but still loads and synchronises).
  //             Separated: each tile step ends with wait_loads() (this wavefront's loads into the
  //             other buffer have landed) and __syncthreads() (every wavefront's have, and every
  //             wavefront is past its reads of this buffer), so the fill in tile step t + 1 of the
  //             buffer tile step t read follows that barrier, and tile step t + 1's reads of the
  //             buffer filled in tile step t follow it too. The last tile step loads nothing.
  //   sV        per wavefront, its own V rows: written once with plain stores before the first
  //             barrier, only read after it.
  __shared__ KvTileBuf64 sB0, sB1;
  __shared__ __attribute__((aligned(16))) elem sV[NWAVES][TW];
  __shared__ int sLast[NWAVES];   // kv_last_block of each wavefront: written and read before the first tile

  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int n = lane & 31, h = lane >> 5;
  const BlockXY bxy = work_order_block();
  const int b = bxy.y / H, hh = bxy.y % H;
  const bool has_h0 = (hh == 0);
  const int NB = (T + TILE - 1) / TILE;
  const int key0 = bxy.x * (NWAVES * TILE) + wave * TILE;
  const int j = key0 + n;
  const int64_t seq_row = (int64_t)b * H;
  auto view_head = [&](const elem* base, const Strides& s_, int hd) -> const elem* {
    if constexpr (CV) return base + (seq_row + hd) * T * D;
    else return base + s_.at(b, hd);
  };
  auto view_ld = [&](const Strides& s_) -> int {
    if constexpr (CV) return D;
    else return (int)s_.row;
  };
  float* uplane = ucheck + ((int64_t)hh * nseq + b) * utri_floats(NB);
  const float* carry_b = carry + (int64_t)b * NB * T;

  const KvProbe probe = kv_probe(reach, seq_row + hh, carry_b, T, NB, key0, lane);
  // B operands (lane = key): the wavefront's K rows and head 0's in registers, its V rows in LDS
  frag kf[NS], k0f[NS];
  {
    const elem* kh = view_head(k, ks, hh);
    const elem* k0 = view_head(k, ks, 0);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      kf[s] = ld_std_bounded<OP>(kh, view_ld(ks), j, T, h, s);
      k0f[s] = has_h0 ? kf[s] : ld_std_bounded<OP>(k0, view_ld(ks), j, T, h, s);
    }
    const elem* vh = view_head(v, vs, hh);
    for (int c = lane; c < TILE * (D / 8); c += 64) {
      const int r = c / (D / 8), cc = c % (D / 8);
      const bool ok = key0 + r < T;
      const uint4 v4 = *reinterpret_cast<const uint4*>(vh + (int64_t)(ok ? key0 + r : 0) * view_ld(vs) + cc * 8);
      *reinterpret_cast<uint4*>(&sV[wave][swzq(r, cc)]) = ok ? v4 : make_uint4(0u, 0u, 0u, 0u);
    }
  }

  // Exempt keys whose gradients are taken apart (j < xk) need no masks in this workgroup's interior tiles:
  // head 0's key is zeroed in their lanes, so their logits select nothing, and their history is taken as
  // beyond any logit, so their P and dz are zeros. (The masks on every tile made the first workgroup of a
  // head, whose sweep is the longest, half again as slow as the others: with 16 exempt keys, B=2 H=12 T=5003,
  // nothing left out, the kernel runs 317 us instead of 342.)
  const bool apart = j < reach.xk;
  if (apart) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      k0f[s] = OP::zero();
      if (has_h0) kf[s] = OP::zero();
    }
  }

  f32x16 dkt[DB], dvt[DB], dk0t[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    dkt[db] = zero16();
    dvt[db] = zero16();
    dk0t[db] = zero16();
  }
  float ucarry = 0.f;
  const float sl2 = scale * LOG2E;
  const float neg_inv_scale = -1.f / scale;
  // fragment s of row n of a swzq tile (A operand: lane = query row; or B: lane = key)
  auto rfrag = [&](const elem* tile, int s) -> frag {
    return *reinterpret_cast<const frag*>(tile + swzq(n, 2 * s + h));
  };
  // query tiles the workgroup visits, last to first: qb_hi (later ones hold no weight for its keys) down
  // to the first that reaches its keys
  const int qb_lo = bxy.x * NWAVES;
  int qb_hi = NB - 1;
  if (reach.qstat) {
    int last = key0 < T ? NB - 1 : 0;
    if (key0 < T && kv_worth(probe, key0, T, reach.xk, lane)) {
      lds_wave_sync();   // the wavefront's V rows
      frag vg[NS];
#pragma unroll
      for (int s = 0; s < NS; ++s) vg[s] = rfrag(sV[wave], s);
      const float2 qstat = head_qstat(reach, seq_row + hh, lane, probe.q);
      const float thr = kv_threshold(frag_sumsq<OP, NS>(kf), frag_sumsq<OP, NS>(vg), qstat, scale);
      last = kv_last_block(probe, carry_b, T, NB, key0, reach.xk, thr, lane);
    }
    if (lane == 0) sLast[wave] = last;
    __syncthreads();
    qb_hi = kv_sweep_start(sLast, NB, qb_lo, wave, lane, key0, T, uplane,
                           reach.hi + ((int64_t)hh * nseq + b) * reach.nkg + bxy.x);
  }
  const int ntiles = qb_hi - qb_lo + 1;

  // operand sources (buffer resources over one head's rows) and this lane's parts of the direct
  // loads
  const int q_ld = view_ld(qs), do_ld = view_ld(dos);
  const __amdgpu_buffer_rsrc_t rs_q = rsrc(view_head(q, qs, hh), (int64_t)T * q_ld * 2);
  const __amdgpu_buffer_rsrc_t rs_do = rsrc(view_head(dout, dos, hh), (int64_t)T * do_ld * 2);
  const __amdgpu_buffer_rsrc_t rs_q0 = rsrc(view_head(q, qs, 0), (int64_t)T * q_ld * 2);
  const __amdgpu_buffer_rsrc_t rs_lse = rsrc(lse + (seq_row + hh) * ldt, ldt * 4);
  const __amdgpu_buffer_rsrc_t rs_ndb = rsrc(dbar + (seq_row + hh) * ldt, ldt * 4);
  const RowsLaneQ rl_q(q_ld, lane, wave), rl_do(do_ld, lane, wave);

  // Everything query tile qb needs, into buffer B, by direct loads only (the tile loop holds no
  // register loads: the vector-memory counter drains in issue order, so waiting for one would wait
  // for the tiles behind it): part `wave` of each operand tile (each wavefront loads a quarter of
  // every tile), the row statistics (wavefronts 0, 1), and each wavefront's carry row of its keys
  // (keys past the end read zero). Tiles load in order, last to first, so the carry row steps back
  // one row per call.
  const float* carry_row = carry_b + (int64_t)qb_hi * T;
  auto load_tile = [&](int qb, KvTileBuf64& B) {
    const int qbase = qb * TILE;
    if (wave == 0)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_lse, lds_ptr(B.stat[0]), 4, (lane & 31) * 4, qbase * 4, 0, 0);
    if (wave == 1)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_ndb, lds_ptr(B.stat[1]), 4, (lane & 31) * 4, qbase * 4, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc(carry_row, (int64_t)T * 4), lds_ptr(B.hist[wave]), 4, j * 4, 0, 0,
                                             0);
    carry_row -= T;
    g2l_rowsq(B.r[0], rs_q, rl_q, q_ld, qbase, wave);
    g2l_rowsq(B.r[1], rs_do, rl_do, do_ld, qbase, wave);
    if (!has_h0) g2l_rowsq(B.r[2], rs_q0, rl_q, q_ld, qbase, wave);
  };
  // the first tile
  load_tile(qb_hi, sB0);
  wait_loads();
  __syncthreads();

  // acc[db] (D x keys) += Y^T X: Y a (queries x D) row tile (swzq, read transposed), X a C-layout
  // (queries x keys) tile; with split, X also enters as its rounding residual.
  auto acc_t = [&](f32x16 (&acc)[DB], const elem* y, const f32x16& x, bool split) {
    frag xf[AS];
#pragma unroll
    for (int s = 0; s < AS; ++s) xf[s] = OP::from_acc(x, s);
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int s = 0; s < AS; ++s) acc[db] = OP::mma(get_trq<true>(y, lane, db, s), xf[s], acc[db]);
    if (split) {
#pragma unroll
      for (int s = 0; s < AS; ++s) xf[s] = OP::from_acc_lo(x, s);
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int s = 0; s < AS; ++s) acc[db] = OP::mma(get_trq<true>(y, lane, db, s), xf[s], acc[db]);
    }
  };

  // Keys below `exempt` are never selected, so they gather attention from every later query and
  // their dV / dK sums run over all of them: their products take the split operands.
  const bool split_keys = key0 < exempt;

  // the tile loop in two instances, for head 0's workgroups and the others (see bwd_kv_kernel)
  auto sweep = [&](auto h0_tag) {
    constexpr bool H0 = decltype(h0_tag)::value;
    // the checkpoint row of tile t's query block (the rows lie end to end, tiles run last to first)
    float* urow = uplane + utri_row(qb_hi);
    // tile t (buffer t mod 2, named by ODD)
    // kind 0: some pairs masked; 1: none; 2: none, with the split products of the tile that holds exempt keys
    auto tile_step = [&](int t, auto kind_tag, auto odd_tag) {
      constexpr int KIND = decltype(kind_tag)::value;
      constexpr bool INTERIOR = KIND != 0;
      constexpr bool ODD = decltype(odd_tag)::value;
      KvTileBuf64& B = ODD ? sB1 : sB0;
      const int qb = qb_hi - t;
      const int qbase = qb * TILE;
      const bool more = t + 1 < ntiles;
      if (more) load_tile(qb - 1, ODD ? sB0 : sB1);   // into the other buffer, free since the last barrier
      if (INTERIOR || qbase + TILE - 1 >= key0) {   // else every query of the tile precedes every key
        if (h == 0 && j < T) urow[j] = ucarry;   // j < (qb + 1) * TILE here
        const bool edge = !INTERIOR && ((qbase <= key0 + TILE - 1) || key0 < exempt);
        const bool split = KIND != 1 && split_keys;
        const TileMasks mk(j, qbase, T, exempt, h, reach.xk);
        auto body = [&]() {
          // (keys past the end read a zero carry through the load's range check)
          const float hist = KIND == 2 && apart ? 1e30f : B.hist[wave][lane];
          const elem* q0s = H0 ? B.r[0] : B.r[2];
          // the four fragments of head 0's Q rows are all requested before the chain of logit
          // products starts, so the chain waits for one LDS latency rather than one per product
          // (the default scheduler otherwise issues each read just before its product)
          frag q0r[NS];
#pragma unroll
          for (int s = 0; s < NS; ++s) q0r[s] = rfrag(q0s, s);
          __builtin_amdgcn_sched_barrier(0);
          f32x16 l0 = zero16();
#pragma unroll
          for (int s = 0; s < NS; ++s) l0 = OP::mma(q0r[s], H0 ? kf[s] : k0f[s], l0);
          f32x16 fs;
          uint32_t gate;
          selection_tile<false>(l0, hist * neg_inv_scale, h, edge, mk, gate, fs);

          f32x16 lg;   // q.k - F/s
          if constexpr (H0) {   // head 0 itself: its logits are l0
#pragma unroll
            for (int i = 0; i < 16; ++i) lg[i] = l0[i] + fs[i];
          } else {
            lg = fs;
#pragma unroll
            for (int s = 0; s < NS; ++s) lg = OP::mma(rfrag(B.r[0], s), kf[s], lg);
          }
          f32x16 dp = rows16(B.stat[1], h);   // dO.v - dbar
#pragma unroll
          for (int s = 0; s < NS; ++s) dp = OP::mma(rfrag(B.r[1], s), rfrag(sV[wave], s), dp);
          f32x16 pr, dz;
          p_dz_tile<false>(lg, dp, B.stat[0], sl2, h, edge, mk, pr, dz);
          acc_t(dvt, B.r[1], pr, split);
          f32x16 gp;
          ucarry = gpath_tile(dz, ucarry, gate, h, gp);
          if constexpr (H0) {   // head 0's dK takes g with its own dz
#pragma unroll
            for (int i = 0; i < 16; ++i) dz[i] += gp[i];
            acc_t(dkt, B.r[0], dz, split || big_tile(dz));
          } else {
            acc_t(dkt, B.r[0], dz, split);
            acc_t(dk0t, B.r[2], gp, big_tile(gp));
          }
        };
        body();
      }
      urow -= 32 * qb;   // utri_row(qb - 1)
      wait_loads();
      __syncthreads();   // the next tile's operands are in; every wavefront is done with this one
    };
    // The last NWAVES tiles hold the wavefronts' diagonals; a workgroup with an exempt key that is not
    // taken apart runs every tile with the masks.
    const bool first = qb_lo * TILE < exempt;
    const int n_int = (first && reach.xk == 0) ? 0 : max(ntiles - NWAVES, 0);
    // tiles [t0, t1) in pairs, even tiles from buffer 0 and odd ones from buffer 1
    auto run = [&](int t0, int t1, auto kind_tag) {
      int t = t0;
      if (t < t1 && (t & 1)) tile_step(t++, kind_tag, std::true_type{});
      for (; t + 1 < t1; t += 2) {
        tile_step(t, kind_tag, std::false_type{});
        tile_step(t + 1, kind_tag, std::true_type{});
      }
      if (t < t1) tile_step(t, kind_tag, std::false_type{});
    };
    if (first) run(0, n_int, std::integral_constant<int, 2>{});
    else run(0, n_int, std::integral_constant<int, 1>{});
    run(n_int, ntiles, std::integral_constant<int, 0>{});
  };
  if (SOLO || has_h0) sweep(std::true_type{});
  else if constexpr (!SOLO) sweep(std::false_type{});

  if (j >= T || j < reach.xk) return;   // (the first xk keys' gradients: bwd_finish_kernel)
  // dV and the dK of heads other than 0 go to the caller's views; head 0's dK to its fp32 sums,
  // where the other heads' shares join it (to its view too when it is the sequence's only head)
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int d = db * 32 + 8 * a + 4 * h;
      const float4 kq = make_float4(dkt[db][4 * a] * scale, dkt[db][4 * a + 1] * scale, dkt[db][4 * a + 2] * scale,
                                    dkt[db][4 * a + 3] * scale);
      store_grad4(dvv, b, hh, j, d, make_float4(dvt[db][4 * a], dvt[db][4 * a + 1], dvt[db][4 * a + 2], dvt[db][4 * a + 3]));
      if (has_h0 && H > 1) *reinterpret_cast<float4*>(dk0h + ((int64_t)b * T + j) * D + d) = kq;
      else store_grad4(dkv, b, hh, j, d, kq);
    }
  if (!has_h0) {   // this head's share of head 0's dK, in its own slot (head hh: slot hh - 1)
    float* dst = dk0x + ((int64_t)(hh - 1) * nseq * T + (int64_t)b * T + j) * D;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int a = 0; a < 4; ++a)
        *reinterpret_cast<float4*>(dst + db * 32 + 8 * a + 4 * h) =
            make_float4(dk0t[db][4 * a] * scale, dk0t[db][4 * a + 1] * scale, dk0t[db][4 * a + 2] * scale,
                        dk0t[db][4 * a + 3] * scale);
  }
}

// ---------------------------------------------------------------------------------------------
// The key tiles that a query-side workgroup has to visit, ascending, from the key side's sweep starts
// (hi, one per four key tiles): those whose sweep reached the workgroup's first query block qb0 -- past
// it their weights and selection suffixes are zeros -- and the tiles of exempt keys, [0, i_lo). As runs of
// groups of four tiles counted from the workgroup's last group (write_reach_runs counts down). No other
// group may be visited: past its sweep's start the key side has written no checkpoint of the suffixes. Where
// the list ends short of the last group (selected and unselected keys in turn over more than 16K keys), the
// walk takes the next groups from hi itself, 64 at a time.
struct QueryWalk {
  const TileRun* runs;
  const int* starts;   // hi
  int first_qb;        // qb0
  int groups, run_to, i;
  bool far;   // the first group is visited for its exempt keys alone
  __device__ __forceinline__ void none() {   // every tile
    runs = nullptr;
    starts = nullptr;
    first_qb = 0;
    groups = 0;
    run_to = INT_MAX;
    far = false;
    i = 0;
  }
  template <int NW>
  __device__ __forceinline__ void find(const int* hi, int qb0, int wg_end, int i_lo, uint64_t* words, TileRun* r,
                                       int lane, int wave) {
    starts = hi;
    first_qb = qb0;
    groups = (wg_end + 3) / 4;
    far = __builtin_amdgcn_readfirstlane(hi[0]) < qb0;
    const int all = (groups + 63) / 64, nwords = min(all, REACH_MASK_WORDS), first = 64 * (all - nwords);
    for (int w = wave; w < nwords; w += NW) {
      const int m = first + 64 * w + lane, g = groups - 1 - m;
      const uint64_t bits = __ballot(g >= 0 && hi[max(g, 0)] >= qb0);
      if (lane == 0) words[w] = bits;
    }
    __syncthreads();
    if (wave == 0) write_reach_runs<false>(r, words, nwords, first, lane);
    __syncthreads();
    runs = r;
    i = 0;
    if (far) {
      run_to = i_lo - 1;
    } else {
      int from;
      next_run(from);   // (starts at tile 0)
    }
  }
  __device__ __forceinline__ void next_run(int& from) {
    const TileRun r = runs[i];
    const int hi = __builtin_amdgcn_readfirstlane(r.hi), lo = __builtin_amdgcn_readfirstlane(r.lo);
    if (__builtin_expect(hi == -2, 0)) {   // (and again at the next call: i stays)
      search(from);
      return;
    }
    ++i;
    from = 4 * (groups - 1 - hi);   // (past the workgroup's last tile at the end)
    run_to = hi < 0 ? INT_MAX : 4 * (groups - 1 - lo) + 3;
  }
  // The next run past tile run_to from hi: within 64 groups.
  __device__ __forceinline__ void search(int& from) {
    const int lane = threadIdx.x & 63;
    for (int g = (run_to + 1) / 4; g < groups; g += 64) {
      const uint64_t bits = __ballot(g + lane < groups && starts[min(g + lane, groups - 1)] >= first_qb);
      if (bits != 0) {
        const int at = __builtin_ctzll(bits);
        const uint64_t gaps = ~(bits >> at);   // (a shifted-in zero ends the run at the 64 groups' end)
        const int len = gaps != 0 ? __builtin_ctzll(gaps) : 64;
        from = 4 * (g + at);
        run_to = from + 4 * len - 1;
        return;
      }
    }
    from = 4 * groups;
    run_to = INT_MAX;
  }
  __device__ __forceinline__ int after(int kt) {
    int n = kt + 1;
    if (__builtin_expect(n > run_to, 0)) next_run(n);
    return n;
  }
};

// ---------------------------------------------------------------------------------------------
// Backward, query side. grid (ceil(T/128), nseq * H/G); wavefront w owns queries
// [x*128 + 32w, +32) of heads [gi*G, gi*G+G) (late query blocks launch first) and walks the key
// tiles up to its diagonal, with Q, dO and the dQ sums in registers. It recomputes P and dz as the
// key side does, and this group's share of head 0's g from the key side's checkpoint of U plus
// the suffix inside the tile. dQ = dz K takes dz through a per-wavefront LDS tile (as the A operand)
// and K^T from LDS (as the B operand).

template <class OP, int D, int G, bool CV>   // CV: see bwd_kv_kernel
__global__ __launch_bounds__(NTHREADS, (dq_min_blocks<OP, D>())) void bwd_dq_kernel(
    const typename OP::elem* __restrict__ q, const typename OP::elem* __restrict__ k,
    const typename OP::elem* __restrict__ v, const typename OP::elem* __restrict__ kt,
    const typename OP::elem* __restrict__ dout, Strides qs, Strides ks, Strides vs, Strides dos,
    const float* __restrict__ lse, const float* __restrict__ dbar, const float* __restrict__ carry,
    const float* __restrict__ ucheck, float* __restrict__ dq0h, float* __restrict__ dq0x, GradView dqv, int nseq,
    int H, int T, int64_t ldt, int exempt, float scale, BwdReach reach) {
  using elem = typename OP::elem;
  using frag = typename OP::frag;
  constexpr int NS = D / OP::KS;
  constexpr int DB = D / 32;
  constexpr int LDK = D + OP::KPAD;
  constexpr int LDKT = TILE + OP::KPAD;
  constexpr int LDZ = TILE + OP::KPAD;
  constexpr int AS = OP::acc_steps;
  constexpr int NH = G + 1;

  __shared__ __attribute__((aligned(16))) elem sK[NH][TILE * LDK];
  __shared__ __attribute__((aligned(16))) elem sKt[NH][D * LDKT];
  __shared__ __attribute__((aligned(16))) elem sV[G][TILE * LDK];
  __shared__ __attribute__((aligned(16))) elem sZ[NWAVES][TILE * LDZ];
  __shared__ uint64_t sMask[REACH_MASK_WORDS];   // the tiles to visit (QueryWalk)
  __shared__ TileRun sRuns[REACH_RUNS];

  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int n = lane & 31, h = lane >> 5;
  const int groups = H / G;
  const BlockXY bxy = work_order_block();
  const int b = bxy.y / groups, gi = bxy.y % groups;
  const int hd0 = gi * G;
  const bool has_h0 = (gi == 0);
  const int NB = (T + TILE - 1) / TILE;
  const int qsb = gridDim.x - 1 - bxy.x;
  const int qb = qsb * NWAVES + wave;
  const int qbase = qb * TILE;
  const int64_t seq_row = (int64_t)b * H;
  // view accessors (CV: the contiguous layout, strides as compile-time facts)
  auto view_head = [&](const elem* base, const Strides& vs_, int hh) -> const elem* {
    if constexpr (CV) return base + (seq_row + hh) * T * D;
    else return base + vs_.at(b, hh);
  };
  auto view_ld = [&](const Strides& vs_) -> int64_t {
    if constexpr (CV) return D;
    else return vs_.row;
  };
  const int my_end = (qb < NB) ? qb + 1 : 0;
  const int wg_end = min(qsb * NWAVES + NWAVES - 1, NB - 1) + 1;
  elem* zs = sZ[wave];
  // this wavefront's rows of the carry and U checkpoints (key offset added per tile)
  const int qb_c = qb < NB ? qb : NB - 1;
  const float* carry_row = carry + ((int64_t)b * NB + qb_c) * T;
  // (the row's keys end at (qb_c + 1) * TILE; the tiles past a wavefront's diagonal read, unused,
  // into the next row, and the last row spans every key tile: the reads stay inside the plane)
  const float* urow = ucheck + ((int64_t)gi * nseq + b) * utri_floats(NB) + utri_row(qb_c);

  // Query-side operands (A operands: lane = query row): the group's Q and dO rows and head 0's Q
  // rows in registers, as are the rows' statistics (element i: row crow(i, h)).
  frag q0a[NS];
  frag qa[G][NS], doa[G][NS];
#pragma unroll
  for (int g = 0; g < G; ++g) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      qa[g][s] = ld_std_bounded<OP>(view_head(q, qs, hd0 + g), view_ld(qs), qbase + n, T, h, s);
      doa[g][s] = ld_std_bounded<OP>(view_head(dout, dos, hd0 + g), view_ld(dos), qbase + n, T, h, s);
    }
  }
  auto q_frag = [&](int g, int s) -> frag { return qa[g][s]; };
  auto do_frag = [&](int g, int s) -> frag { return doa[g][s]; };
  f32x16 lse_r[G], ndb_r[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int64_t row = seq_row + hd0 + g;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = qbase + crow(i, h);
      const int rr = min(r, T - 1);
      const float lv = lse[row * ldt + rr], dv_ = dbar[row * ldt + rr];
      lse_r[g][i] = (r < T) ? lv : INFINITY;   // rows past the end: P = 0
      ndb_r[g][i] = (r < T) ? dv_ : 0.f;      // -dbar: dO.v accumulates onto it
    }
  }
  if (!has_h0) {
#pragma unroll
    for (int s = 0; s < NS; ++s) q0a[s] = ld_std_bounded<OP>(view_head(q, qs, 0), view_ld(qs), qbase + n, T, h, s);
  }

  f32x16 dqacc[G][DB], dq0acc[DB];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int db = 0; db < DB; ++db) dqacc[g][db] = zero16();
#pragma unroll
  for (int db = 0; db < DB; ++db) dq0acc[db] = zero16();

  const float sl2 = scale * LOG2E;
  const float neg_inv_scale = -1.f / scale;

  // Staging of one key tile: K, V, K^T of the group (+ head 0's K, K^T).
  RowTile<elem, D> nK[NH], nV[G];
  ColTile<elem, D> nKt[NH];
  // the key-side rows of this workgroup's heads (computed once, outside the tile loop)
  const elem* k_rows[NH];
  const elem* v_rows[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    k_rows[g] = view_head(k, ks, hd0 + g);
    v_rows[g] = view_head(v, vs, hd0 + g);
  }
  k_rows[G] = view_head(k, ks, 0);
  const int k_ld = (int)view_ld(ks), v_ld = (int)view_ld(vs);
  auto load_tile = [&](int ktile) {
    const int kbase = ktile * TILE;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int64_t row = seq_row + hd0 + g;
      nK[g].load(k_rows[g], k_ld, kbase, T, tid);
      nV[g].load(v_rows[g], v_ld, kbase, T, tid);
      nKt[g].load(kt + row * D * ldt, ldt, kbase, tid);
    }
    if (!has_h0) {
      nK[G].load(k_rows[G], k_ld, kbase, T, tid);
      nKt[G].load(kt + seq_row * D * ldt, ldt, kbase, tid);
    }
  };
  auto store_tile = [&]() {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      nK[g].template store<LDK>(sK[g], tid);
      nV[g].template store<LDK>(sV[g], tid);
      nKt[g].template store<LDKT>(sKt[g], tid);
    }
    if (!has_h0) {
      nK[G].template store<LDK>(sK[G], tid);
      nKt[G].template store<LDKT>(sKt[G], tid);
    }
  };

  // acc[db] (queries x D) += X K: X a C-layout (queries x keys) tile, sent through LDS to become
  // the A operand; K^T (rows d) staged in LDS is the B operand. With split, X's rounding residual
  // takes a second pass.
  auto acc_xk = [&](f32x16 (&acc)[DB], const f32x16& x, const elem* ktile, bool split) {
    frag zf[AS];
    if constexpr (sizeof(elem) == 2) {
      // bf16: X goes to the tile transposed (4 rows per write) and comes back through the
      // transposing read
      put_tr<false>(zs, x, n, h);
      lds_wave_sync();
#pragma unroll
      for (int s = 0; s < AS; ++s) zf[s] = get_tr(zs, lane, s);
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int s = 0; s < AS; ++s) acc[db] = OP::mma(zf[s], OP::ld_std(ktile, LDKT, db * 32 + n, h, s), acc[db]);
      if (split) {
        lds_wave_sync();
        put_tr<true>(zs, x, n, h);
        lds_wave_sync();
#pragma unroll
        for (int s = 0; s < AS; ++s) zf[s] = get_tr(zs, lane, s);
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int s = 0; s < AS; ++s) acc[db] = OP::mma(zf[s], OP::ld_std(ktile, LDKT, db * 32 + n, h, s), acc[db]);
      }
      lds_wave_sync();
      return;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) zs[crow(i, h) * LDZ + n] = OP::to_elem(x[i]);
    lds_wave_sync();
#pragma unroll
    for (int s = 0; s < AS; ++s) zf[s] = OP::ld_std(zs, LDZ, n, h, s);
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int s = 0; s < AS; ++s) acc[db] = OP::mma(zf[s], OP::ld_std(ktile, LDKT, db * 32 + n, h, s), acc[db]);
    if constexpr (OP::SPLIT) {
      if (split) {
        lds_wave_sync();
#pragma unroll
        for (int i = 0; i < 16; ++i) zs[crow(i, h) * LDZ + n] = OP::to_elem_lo(x[i]);
        lds_wave_sync();
#pragma unroll
        for (int s = 0; s < AS; ++s) zf[s] = OP::ld_std(zs, LDZ, n, h, s);
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int s = 0; s < AS; ++s) acc[db] = OP::mma(zf[s], OP::ld_std(ktile, LDKT, db * 32 + n, h, s), acc[db]);
      }
    }
    lds_wave_sync();
  };

  auto key_vals = [&](int ktile, float& hv, float& uv) {
    const int jj = ktile * TILE + n;
    hv = (jj < T) ? carry_row[jj] : 0.f;
    uv = (jj < T) ? urow[jj] : 0.f;
  };

  // tiles holding exempt keys [0, i_lo), then the interior ones (below every wavefront's diagonal,
  // which also keeps them clear of the sequence end), then the diagonals from i_hi on
  const int i_lo = min((exempt + TILE - 1) / TILE, wg_end);
  const int i_hi = max(i_lo, min(qsb * NWAVES, wg_end));
  QueryWalk walk;
  walk.none();
  if (reach.qstat)
    walk.template find<NWAVES>(reach.hi + ((int64_t)gi * nseq + b) * reach.nkg, qsb * NWAVES, wg_end, i_lo, sMask, sRuns,
                               lane, wave);

  // The tile loop in two instances, for the group holding head 0 and for the others (as on the
  // key side).
  auto sweep = [&](auto h0_tag) {
    constexpr bool H0 = decltype(h0_tag)::value;

    // one key tile; INTERIOR: no pair of the tile is masked or exempt for any wavefront, so the
    // body is straight-line code without the masks
    auto tile_step = [&](int ktile, auto interior_tag) {
      constexpr bool INTERIOR = decltype(interior_tag)::value;
      const int kbase = ktile * TILE;
      float hist, uin;
      load_tile(ktile);
      key_vals(ktile, hist, uin);
      if (!INTERIOR && walk.far && ktile < i_lo) uin = 0.f;   // (past the sweep's start: no row written)
      if (ktile > 0) __syncthreads();   // every wavefront is done with the previous tile
      store_tile();
      __syncthreads();
      if (ktile < my_end) {
        const int j = kbase + n;
        // tile body; edge: some pair of the tile is masked (diagonal, sequence end) or exempt
        const bool edge = !INTERIOR && ((kbase + TILE - 1 >= qbase) || (kbase + TILE > T) || kbase < exempt);
        const TileMasks mk(j, qbase, T, exempt, h);
        {
          const elem* k0s = H0 ? sK[0] : sK[G];
          f32x16 l0 = zero16();
  #pragma unroll
          for (int s = 0; s < NS; ++s)
            l0 = OP::mma(H0 ? q_frag(0, s) : q0a[s], OP::ld_std(k0s, LDK, n, h, s), l0);
          f32x16 fs;
          uint32_t gate;
          selection_tile<false>(l0, hist * neg_inv_scale, h, edge, mk, gate, fs);

          f32x16 zsum, dz0;
  #pragma unroll
          for (int g = 0; g < G; ++g) {
            f32x16 lg;   // q.k - F/s
            if (H0 && g == 0) {   // head 0 itself: its logits are l0, its dQ waits for g
  #pragma unroll
              for (int i = 0; i < 16; ++i) lg[i] = l0[i] + fs[i];
            } else {
              lg = fs;
  #pragma unroll
              for (int s = 0; s < NS; ++s)
                lg = OP::mma(q_frag(g, s), OP::ld_std(sK[g], LDK, n, h, s), lg);
            }
            f32x16 dp;   // dO.v - dbar
            dp = ndb_r[g];
  #pragma unroll
            for (int s = 0; s < NS; ++s)
              dp = OP::mma(do_frag(g, s), OP::ld_std(sV[g], LDK, n, h, s), dp);
            f32x16 pr, dz;
            p_dz_tile_r(lg, dp, lse_r[g], sl2, edge, mk, pr, dz);
            if (g == 0) {
              zsum = dz;
            } else {
  #pragma unroll
              for (int i = 0; i < 16; ++i) zsum[i] += dz[i];
            }
            if (H0 && g == 0) {
              dz0 = dz;
            } else {
              acc_xk(dqacc[g], dz, sKt[g], false);
            }
          }

          f32x16 gp;
          gpath_tile(zsum, uin, gate, h, gp);
          if constexpr (H0) {
            f32x16 dzh;
  #pragma unroll
            for (int i = 0; i < 16; ++i) dzh[i] = dz0[i] + gp[i];
            acc_xk(dqacc[0], dzh, sKt[0], big_tile(dzh));
          } else {
            acc_xk(dq0acc, gp, sKt[G], big_tile(gp));
          }
        }
      }
    };
    int ktile = 0;
    for (; ktile < i_lo; ktile = walk.after(ktile)) tile_step(ktile, std::false_type{});
    for (; ktile < i_hi; ktile = walk.after(ktile)) tile_step(ktile, std::true_type{});
    for (; ktile < wg_end; ktile = walk.after(ktile)) tile_step(ktile, std::false_type{});
  };
  if (has_h0) sweep(std::true_type{});
  else sweep(std::false_type{});

  if (qb >= NB) return;
  // heads other than 0: dQ (scaled) to the caller's view; head 0: unscaled fp32 sums, where the
  // other groups' shares join it
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int hh = hd0 + g;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = qbase + crow(i, h);
      if (r < T) {
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          if (hh == 0 && H > 1) dq0h[((int64_t)b * T + r) * D + db * 32 + n] = dqacc[g][db][i];
          else store_grad1(dqv, b, hh, r, db * 32 + n, dqacc[g][db][i] * scale);
        }
      }
    }
  }
  if (!has_h0) {   // this group's share of head 0's dQ (unscaled), in its own slot (group gi: slot gi - 1)
    float* dst = dq0x + ((int64_t)(gi - 1) * nseq * T + (int64_t)b * T) * D;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = qbase + crow(i, h);
      if (r < T) {
#pragma unroll
        for (int db = 0; db < DB; ++db) dst[(int64_t)r * D + db * 32 + n] = dq0acc[db][i];
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Backward, query side, bf16 storage at head dim 64 with one head per wavefront: bwd_dq_kernel's
// tile work with every key tile's operands -- the K, V and head 0's K rows (swzq; the K rows read
// as rows by the logit products and transposed by the dQ products, so no K^T is loaded), and each
// wavefront's carry and selection-suffix checkpoint values of the tile's keys -- loaded straight
// into LDS one tile ahead, two buffers as separate LDS variables (see bwd_kv64_kernel); one barrier
// per tile. Eight wavefronts (256 queries) per workgroup, one
// workgroup per CU: each key tile is staged once for twice the queries of a four-wavefront group
// (measured 3% faster; the operand staging, not its latency, is what the loads cost).

constexpr int DQ64_WAVES = 8;

struct DqTileBuf64 {
  __attribute__((aligned(16))) uint16_t k[2][TILE * 64];    // K rows, head 0's K rows (swzq)
  __attribute__((aligned(16))) uint16_t v[TILE * 64];       // V rows (swzq)
  __attribute__((aligned(16))) float hist[DQ64_WAVES][64];   // per wavefront: each lane's key's carry
  __attribute__((aligned(16))) float uin[DQ64_WAVES][64];    // ... and its U checkpoint
};

// CV: every view is the contiguous (nseq, H, T, D) layout of sa_backward. SOLO: one-head sequences
// only (head 0's loop alone is built, as in bwd_kv64_kernel). SNAKE: workgroups dealt in the order
// of work_order_block(order_slots) (an instance of its own, so the launches in the longest-first
// order run exactly the code they ran before it existed; order_slots is unused there).
template <bool CV, bool SOLO, bool SNAKE = false>
__global__ __launch_bounds__(DQ64_WAVES * 64, 1) void bwd_dq64_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    const uint16_t* __restrict__ dout, Strides qs, Strides ks, Strides vs, Strides dos,
    const float* __restrict__ lse, const float* __restrict__ dbar, const float* __restrict__ carry,
    const float* __restrict__ ucheck, float* __restrict__ dq0h, float* __restrict__ dq0x, GradView dqv, int nseq,
    int H, int T, int64_t ldt, int exempt, float scale, int order_slots, BwdReach reach) {
  using OP = OpBF16;
  using elem = uint16_t;
  using frag = OP::frag;
  constexpr int D = 64, NS = 4, DB = 2, AS = 2;
  // LDS lifetimes (t: the t-th key tile visited; key tile t where none is left out):
  //   sB0, sB1  tile t's K, head 0's K and V rows, each wavefront's carry and U-checkpoint values,
  //             buffer t mod 2. Filled: by direct loads (K rows by wavefronts 0-3, V rows by 4-7, a
  //             quarter each; every wavefront its own carry and checkpoint values), tile 0 before the
  //             first barrier, tile t in tile step t - 1. Drained: tile step t only (a wavefront
  //             whose diagonal lies before the tile reads nothing but still loads and synchronises).
  //             Separated: as in bwd_kv64_kernel, each tile step ends with wait_loads() and
  //             __syncthreads(), between the last reads of a buffer and its next fill, and between a
  //             fill and its reads. The last tile step loads nothing.
  //   sZ        per wavefront, the dz / g tile transposed for the dQ products: written and read by
  //             the same wavefront within a product (acc_xk); the LDS performs one wavefront's
  //             operations in issue order, so lds_wave_order (a compiler barrier) keeps each read
  //             after its write and the next write after the reads.
  //   sRow      per wavefront, its rows' lse and -dbar: written once before the first barrier, only
  //             read after it.
  __shared__ DqTileBuf64 sB0, sB1;
  __shared__ __attribute__((aligned(16))) elem sZ[DQ64_WAVES][TILE * TILE];   // per wavefront: dz, g transposed
  __shared__ __attribute__((aligned(16))) float sRow[DQ64_WAVES][2][TILE];   // per wavefront: its rows' lse, -dbar
  __shared__ uint64_t sMask[REACH_MASK_WORDS];   // the tiles to visit (QueryWalk): written before the first tile
  __shared__ TileRun sRuns[REACH_RUNS];

  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int n = lane & 31, h = lane >> 5;
  const BlockXY bxy = SNAKE ? work_order_block(order_slots) : work_order_block();
  const int b = bxy.y / H, hh = bxy.y % H;
  const bool has_h0 = (hh == 0);
  const int NB = (T + TILE - 1) / TILE;
  const int qsb = gridDim.x - 1 - bxy.x;
  const int qb = qsb * DQ64_WAVES + wave;
  const int qbase = qb * TILE;
  const int64_t seq_row = (int64_t)b * H;
  auto view_head = [&](const elem* base, const Strides& s_, int hd) -> const elem* {
    if constexpr (CV) return base + (seq_row + hd) * T * D;
    else return base + s_.at(b, hd);
  };
  auto view_ld = [&](const Strides& s_) -> int {
    if constexpr (CV) return D;
    else return (int)s_.row;
  };
  const int my_end = (qb < NB) ? qb + 1 : 0;
  const int wg_end = min(qsb * DQ64_WAVES + DQ64_WAVES - 1, NB - 1) + 1;
  elem* zs = sZ[wave];
  const int qb_c = qb < NB ? qb : NB - 1;

  // A operands (lane = query row): the Q, dO rows and head 0's Q rows in registers; the rows'
  // statistics in the wavefront's LDS rows (registers would spill)
  frag qa[NS], doa[NS], q0a[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    qa[s] = ld_std_bounded<OP>(view_head(q, qs, hh), view_ld(qs), qbase + n, T, h, s);
    doa[s] = ld_std_bounded<OP>(view_head(dout, dos, hh), view_ld(dos), qbase + n, T, h, s);
  }
  if (!has_h0) {
#pragma unroll
    for (int s = 0; s < NS; ++s) q0a[s] = ld_std_bounded<OP>(view_head(q, qs, 0), view_ld(qs), qbase + n, T, h, s);
  }
  if (lane < TILE) {
    const int64_t row = seq_row + hh;
    const int r = qbase + lane;
    const int rr = min(r, T - 1);
    const float lv = lse[row * ldt + rr], dv_ = dbar[row * ldt + rr];
    sRow[wave][0][lane] = (r < T) ? lv : INFINITY;   // rows past the end: P = 0
    sRow[wave][1][lane] = (r < T) ? dv_ : 0.f;       // -dbar: dO.v accumulates onto it
  }

  f32x16 dqacc[DB], dq0acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    dqacc[db] = zero16();
    dq0acc[db] = zero16();
  }
  const float sl2 = scale * LOG2E;
  const float neg_inv_scale = -1.f / scale;

  // key-side sources (buffer resources over one head's rows), this wavefront's rows of the carry
  // and of the U checkpoints (keys past them read zero)
  const int k_ld = view_ld(ks), v_ld = view_ld(vs);
  const __amdgpu_buffer_rsrc_t rs_k = rsrc(view_head(k, ks, hh), (int64_t)T * k_ld * 2);
  const __amdgpu_buffer_rsrc_t rs_k0 = rsrc(view_head(k, ks, 0), (int64_t)T * k_ld * 2);
  const __amdgpu_buffer_rsrc_t rs_v = rsrc(view_head(v, vs, hh), (int64_t)T * v_ld * 2);
  const __amdgpu_buffer_rsrc_t rs_c = rsrc(carry + ((int64_t)b * NB + qb_c) * T, (int64_t)T * 4);
  const __amdgpu_buffer_rsrc_t rs_u =
      rsrc(ucheck + ((int64_t)hh * nseq + b) * utri_floats(NB) + utri_row(qb_c), (int64_t)(qb_c + 1) * TILE * 4);
  const RowsLaneQ rl_k(k_ld, lane, wave & 3), rl_v(v_ld, lane, wave & 3);

  // everything key tile ktile needs, into buffer B, by direct loads only (see bwd_kv64_kernel):
  // wavefronts 0-3 load a quarter of the K rows (and of head 0's), 4-7 of the V rows
  auto load_tile = [&](int ktile, DqTileBuf64& B) {
    const int kbase = ktile * TILE;
    const int m = wave & 3;
    if (wave < 4) {
      g2l_rowsq(B.k[0], rs_k, rl_k, k_ld, kbase, m);
      if (!has_h0) g2l_rowsq(B.k[1], rs_k0, rl_k, k_ld, kbase, m);
    } else {
      g2l_rowsq(B.v, rs_v, rl_v, v_ld, kbase, m);
    }
    const int jo = (kbase + n) * 4;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_c, lds_ptr(B.hist[wave]), 4, jo, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_u, lds_ptr(B.uin[wave]), 4, jo, 0, 0, 0);
  };
  // fragment s of row n (lane = key) of a swzq tile
  auto rfrag = [&](const elem* tile, int s) -> frag {
    return *reinterpret_cast<const frag*>(tile + swzq(n, 2 * s + h));
  };
  // acc[db] (queries x D) += X K: X a C-layout (queries x keys) tile sent through the wavefront's
  // LDS tile to become the A operand (transposed write, transposing read), the K rows (swzq) read
  // transposed as the B operand; with split, X's rounding residual takes a second pass.
  // The tile zs is the wavefront's own: its writes and reads are ordered by lds_wave_order (the
  // previous tile's reads of zs precede this tile's writes in program order as well).
  auto acc_xk = [&](f32x16 (&acc)[DB], const f32x16& x, const elem* ktile, bool split) {
    frag zf[AS];
    put_tr<false>(zs, x, n, h);
    lds_wave_order();
#pragma unroll
    for (int s = 0; s < AS; ++s) zf[s] = get_tr(zs, lane, s);
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int s = 0; s < AS; ++s)
        acc[db] = OP::mma(zf[s], get_trq<false>(ktile, lane, db, s), acc[db]);
    if (split) {
      lds_wave_order();
      put_tr<true>(zs, x, n, h);
      lds_wave_order();
#pragma unroll
      for (int s = 0; s < AS; ++s) zf[s] = get_tr(zs, lane, s);
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int s = 0; s < AS; ++s)
          acc[db] = OP::mma(zf[s], get_trq<false>(ktile, lane, db, s), acc[db]);
    }
    lds_wave_order();
  };

  // the first key tile (position 0 is always exempt, so tile 0 is always visited)
  load_tile(0, sB0);
  // tiles holding exempt keys [0, i_lo), then the interior ones (below every wavefront's diagonal,
  // which also keeps them clear of the sequence end), then the diagonals from i_hi on
  const int i_lo = min((exempt + TILE - 1) / TILE, wg_end);
  const int i_hi = max(i_lo, min(qsb * DQ64_WAVES, wg_end));
  QueryWalk walk;
  walk.none();
  if (reach.qstat)
    walk.template find<DQ64_WAVES>(reach.hi + ((int64_t)hh * nseq + b) * reach.nkg, qsb * DQ64_WAVES, wg_end, i_lo, sMask,
                                   sRuns, lane, wave);
  int ktile = 0, next = walk.after(0);   // this tile and the one after it
  wait_loads();
  __syncthreads();

  // the tile loop in two instances, for head 0's workgroups and the others (see bwd_kv_kernel)
  auto sweep = [&](auto h0_tag) {
    constexpr bool H0 = decltype(h0_tag)::value;
    // key tile ktile, the t-th visited (buffer t mod 2, named by ODD); INTERIOR: no pair of the tile is
    // masked or exempt for any wavefront
    auto tile_step = [&](auto interior_tag, auto odd_tag) {
      constexpr bool INTERIOR = decltype(interior_tag)::value;
      constexpr bool ODD = decltype(odd_tag)::value;
      DqTileBuf64& B = ODD ? sB1 : sB0;
      const int kbase = ktile * TILE;
      if (next < wg_end) load_tile(next, ODD ? sB0 : sB1);   // free since the last barrier
      if (ktile < my_end) {
        const int j = kbase + n;
        const bool edge = !INTERIOR && ((kbase + TILE - 1 >= qbase) || (kbase + TILE > T) || kbase < exempt);
        const TileMasks mk(j, qbase, T, exempt, h);
        const float hist = B.hist[wave][lane];
        float uin = B.uin[wave][lane];
        if (!INTERIOR && walk.far && ktile < i_lo) uin = 0.f;   // (past the sweep's start: no row written)
        const elem* k0s = H0 ? B.k[0] : B.k[1];
        f32x16 l0 = zero16();
#pragma unroll
        for (int s = 0; s < NS; ++s) l0 = OP::mma(H0 ? qa[s] : q0a[s], rfrag(k0s, s), l0);
        f32x16 fs;
        uint32_t gate;
        selection_tile<false>(l0, hist * neg_inv_scale, h, edge, mk, gate, fs);
        f32x16 lg;   // q.k - F/s
        if constexpr (H0) {   // head 0 itself: its logits are l0
#pragma unroll
          for (int i = 0; i < 16; ++i) lg[i] = l0[i] + fs[i];
        } else {
          lg = fs;
#pragma unroll
          for (int s = 0; s < NS; ++s) lg = OP::mma(qa[s], rfrag(B.k[0], s), lg);
        }
        f32x16 dp = rows16(sRow[wave][1], h);   // dO.v - dbar
#pragma unroll
        for (int s = 0; s < NS; ++s) dp = OP::mma(doa[s], rfrag(B.v, s), dp);
        f32x16 pr, dz;
        p_dz_tile<false>(lg, dp, sRow[wave][0], sl2, h, edge, mk, pr, dz);
        f32x16 gp;
        gpath_tile(dz, uin, gate, h, gp);
        if constexpr (H0) {   // head 0's dQ takes g with its own dz
#pragma unroll
          for (int i = 0; i < 16; ++i) dz[i] += gp[i];
          acc_xk(dqacc, dz, B.k[0], big_tile(dz));
        } else {
          acc_xk(dqacc, dz, B.k[0], false);
          acc_xk(dq0acc, gp, B.k[1], big_tile(gp));
        }
      }
      wait_loads();
      __syncthreads();   // the next tile's operands are in; every wavefront is done with this one
    };
    bool odd = false;
    auto run = [&](int stop, auto interior_tag) {   // tiles from ktile up to `stop`, in pairs
      auto shift = [&]() {
        ktile = next;
        next = walk.after(next);
      };
      if (odd && ktile < stop) {
        tile_step(interior_tag, std::true_type{});
        shift();
        odd = false;
      }
      while (ktile < stop) {
        tile_step(interior_tag, std::false_type{});
        shift();
        if (ktile >= stop) {
          odd = true;
          break;
        }
        tile_step(interior_tag, std::true_type{});
        shift();
      }
    };
    run(i_lo, std::false_type{});
    run(i_hi, std::true_type{});
    run(wg_end, std::false_type{});
  };
  if (SOLO || has_h0) sweep(std::true_type{});
  else if constexpr (!SOLO) sweep(std::false_type{});

  if (qb >= NB) return;
  // heads other than 0: dQ (scaled) to the caller's view; head 0: unscaled fp32 sums, where the
  // other heads' shares join it (to its view too when it is the sequence's only head)
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = qbase + crow(i, h);
    if (r < T) {
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        if (has_h0 && H > 1) dq0h[((int64_t)b * T + r) * D + db * 32 + n] = dqacc[db][i];
        else store_grad1(dqv, b, hh, r, db * 32 + n, dqacc[db][i] * scale);
      }
    }
  }
  if (!has_h0) {   // this head's share of head 0's dQ (unscaled), in its own slot (head hh: slot hh - 1)
    float* dst = dq0x + ((int64_t)(hh - 1) * nseq * T + (int64_t)b * T) * D;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = qbase + crow(i, h);
      if (r < T) {
#pragma unroll
        for (int db = 0; db < DB; ++db) dst[(int64_t)r * D + db * 32 + n] = dq0acc[db][i];
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// fp32 storage, small grids: the four wavefronts of a workgroup share one 32-row tile (of queries, or of
// keys on the key side) and split the other axis between them, every fourth tile each.
//
// An fp32 tile is a chain of matrix products at the fp32 rate (64 cycles per 32x32x2 instruction, 96 of
// them per tile in the forward, 192 on the key side: 2.6 and 5.1 us at the least), and a launch lasts as long
// as its longest wavefront's sweep; with a wavefront per tile row a grid of this size leaves most of the
// chip's SIMDs idle meanwhile. Split four ways the longest sweep is a quarter and the grid four times as
// large, at four times the operand reads, which come from L2: nothing is shared through LDS, so nothing is
// staged there and the tile loops need no barrier but the key side's one per four tiles (below). The
// contraction runs over the head dim in the order that gives each lane contiguous elements (lane half h
// takes elements [h D/2, (h+1) D/2)), so a lane's rows load as 16-byte pieces; the products that contract
// over rows read the untransposed matrices a row per half-wavefront, whole 128-byte segments, so no
// transposed copies are made. Measured at B=1 H=4 T=512 D=64: forward 72 -> 26 us, key side 122 -> 53, query side
// 116 -> 45; at B=1 H=8 T=2048 every tile computed: key side 456 -> 382, query side 422 -> 331.
//
// Taken by split_f32_grid.

// A lane's half of its row (lane n: row row0 + n) of a row-major fp32 matrix, rows past the resource zero.
template <int D>
struct HalfRow {
  float f[D / 2];
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, int ld, int row, int h) {
#pragma unroll
    for (int c = 0; c < D / 8; ++c) {
      const auto x = __builtin_amdgcn_raw_buffer_load_b128(rs, (row * ld + h * (D / 2) + 4 * c) * 4, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) f[4 * c + e] = __uint_as_float(x[e]);
    }
  }
  __device__ __forceinline__ float sumsq() const {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < D / 2; ++i) s = fmaf(f[i], f[i], s);
    return s;
  }
};
// c += A B^T over the head dim, a and b the lanes' rows of A and B.
template <int D>
__device__ __forceinline__ f32x16 mma_rows(const HalfRow<D>& a, const HalfRow<D>& b, f32x16 c) {
#pragma unroll
  for (int s = 0; s < D / 2; ++s) c = OpF32::mma(a.f[s], b.f[s], c);
  return c;
}
// acc[db] (D x columns) += Y^T X: Y the 32 rows from row0 of a row-major matrix, X a C-layout tile (rows of Y
// x columns).
template <int D>
__device__ __forceinline__ void mma_cols(f32x16 (&acc)[D / 32], __amdgpu_buffer_rsrc_t rs, int ld, int row0, int n, int h,
                                         const f32x16& x) {
#pragma unroll
  for (int db = 0; db < D / 32; ++db) {
    float y[16];
#pragma unroll
    for (int s = 0; s < 16; ++s)
      y[s] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, ((row0 + crow(s, h)) * ld + db * 32 + n) * 4, 0, 0));
#pragma unroll
    for (int s = 0; s < 16; ++s) acc[db] = OpF32::mma(y[s], x[s], acc[db]);
  }
}
// Sums of four wavefronts' (D x 32 columns) C-layout tiles in wavefront order: thread t gets column t / 8,
// elements [(t mod 8) D/8, +D/8) of the sum. The barrier at the end frees the buffer.
template <int D>
__device__ __forceinline__ void sum_tiles(float (*buf)[32 * (D + 4)], const f32x16 (&acc)[D / 32], float scale, int n, int h,
                                          int wave, int tid, float (&out)[D / 8]) {
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int a = 0; a < 4; ++a)
      *reinterpret_cast<float4*>(&buf[wave][n * (D + 4) + db * 32 + 8 * a + 4 * h]) =
          make_float4(acc[db][4 * a] * scale, acc[db][4 * a + 1] * scale, acc[db][4 * a + 2] * scale,
                      acc[db][4 * a + 3] * scale);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < D / 32; ++c) {
    const int at = (tid >> 3) * (D + 4) + (tid & 7) * (D / 8) + 4 * c;
    float4 x = *reinterpret_cast<const float4*>(&buf[0][at]);
#pragma unroll
    for (int w = 1; w < NWAVES; ++w) {
      const float4 y = *reinterpret_cast<const float4*>(&buf[w][at]);
      x = make_float4(x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w);
    }
    out[4 * c] = x.x;
    out[4 * c + 1] = x.y;
    out[4 * c + 2] = x.z;
    out[4 * c + 3] = x.w;
  }
  __syncthreads();
}

// Forward (fwd_kernel's tile work, no damping). grid (ceil(Tq/32), nseq * H), the longest sweeps first; the
// wavefronts' partial softmax sums merge at the end.
template <int D>
__global__ __launch_bounds__(NTHREADS, 1) void fwd_split_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v, const float* __restrict__ carry,
    float* __restrict__ out, float* __restrict__ rmax, float* __restrict__ rden, float* __restrict__ y, Strides ys, int H,
    int Tq, int Tk, Strides qs, Strides ks, Strides vs, int q_off, int exempt, float scale) {
  constexpr int DB = D / 32, LDF = TILE + 4;
  __shared__ __attribute__((aligned(16))) float sF[NWAVES][TILE * LDF];
  __shared__ __attribute__((aligned(16))) float sSum[NWAVES][32 * (D + 4)];
  __shared__ float sM[NWAVES][TILE], sL[NWAVES][TILE];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int n = lane & 31, h = lane >> 5;
  const int b = blockIdx.y / H, hh = blockIdx.y % H;
  const bool whole = hh == 0;   // head 0's adjusted logits go through LDS whole (see fwd_kernel)
  const int NBq = (Tq + TILE - 1) / TILE, NKT = (Tk + TILE - 1) / TILE;
  const int rb = gridDim.x - 1 - blockIdx.x;
  const int q_rel = rb * TILE + n, q_abs = q_off + q_rel;
  const int end = min((q_off + rb * TILE + TILE - 1) / TILE + 1, NKT);
  auto head = [&](const float* p, const Strides& s, int x, int rows) {
    return rsrc(p + s.at(b, x), (int64_t)rows * s.row * 4);
  };
  const __amdgpu_buffer_rsrc_t rs_k = head(k, ks, hh, Tk), rs_k0 = head(k, ks, 0, Tk), rs_v = head(v, vs, hh, Tk);
  HalfRow<D> qf, q0f;
  qf.load(head(q, qs, hh, Tq), qs.row, q_rel, h);
  q0f.load(head(q, qs, 0, Tq), qs.row, q_rel, h);
  const float* crow_ = carry + ((int64_t)b * NBq + rb) * Tk;
  const float sl2 = scale * LOG2E, neg_inv_scale = -1.f / scale;
  float m = -INFINITY, l = 0.f;
  f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = zero16();

  for (int kt = end - 1 - wave; kt >= 0; kt -= NWAVES) {
    const int kbase = kt * TILE;
    const bool edge = (kbase + TILE - 1 >= q_off + rb * TILE) || (kbase + TILE > Tk) || kbase < exempt;
    HalfRow<D> kf, k0f;
    kf.load(rs_k, ks.row, kbase + n, h);
    if (!whole) k0f.load(rs_k0, ks.row, kbase + n, h);
    const int jk = kbase + n;
    float run = jk < Tk ? crow_[jk] * neg_inv_scale : 0.f;
    const f32x16 l0t = whole ? mma_rows<D>(q0f, kf, zero16()) : mma_rows<D>(q0f, k0f, zero16());
    f32x16 sel;
#pragma unroll
    for (int i = 0; i < 16; ++i) sel[i] = __builtin_amdgcn_fmed3f(-l0t[i], -3.0e38f, 0.f);
    if (edge) {
      const int thr = jk >= exempt ? jk - (q_off + rb * TILE) - 4 * h : 32;
#pragma unroll
      for (int i = 0; i < 16; ++i) sel[i] = crow(i, 0) > thr ? sel[i] : 0.f;
    }
    float* fw = sF[wave];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const Halves g = halves(((sel[4 * a] + sel[4 * a + 1]) + sel[4 * a + 2]) + sel[4 * a + 3]);
      float p = (h == 0) ? run : run + g.lo;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        fw[crow(4 * a + t, h) * LDF + n] = whole ? p + l0t[4 * a + t] : p;
        p += sel[4 * a + t];
      }
      run = (run + g.lo) + g.hi;
    }
    lds_wave_sync();
    f32x16 lg;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const float4 f4 = *reinterpret_cast<const float4*>(&fw[n * LDF + 8 * a + 4 * h]);
      lg[4 * a] = f4.x;
      lg[4 * a + 1] = f4.y;
      lg[4 * a + 2] = f4.z;
      lg[4 * a + 3] = f4.w;
    }
    lds_wave_sync();   // (the next tile's writes follow)
    if (!whole) lg = mma_rows<D>(kf, qf, lg);
    if (edge) {
      const int thr = min(q_abs, Tk - 1) - kbase - 4 * h;
#pragma unroll
      for (int i = 0; i < 16; ++i) lg[i] = crow(i, 0) <= thr ? lg[i] : -INFINITY;
    }
    float zmax = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) zmax = fmaxf(zmax, lg[i]);
    const Halves zh = halves(zmax);
    const float m_new = fmaxf(m, fmaxf(zh.lo, zh.hi) * sl2);
    if (__any(m_new > m)) {
      const float alpha = (m_new == -INFINITY) ? 1.f : fast_exp2(m - m_new);
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
    }
    const float mu = (m == -INFINITY) ? 0.f : m;
    float psum = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float p = fast_exp2(fmaf(lg[i], sl2, -mu));
      lg[i] = p;
      psum += p;
    }
    l += psum;
    mma_cols<D>(o, rs_v, vs.row, kbase, n, h, lg);
  }

  // merge: the row's maximum over the wavefronts, then their sums relative to it
  const Halves lh = halves(l);
  if (h == 0) {
    sM[wave][n] = m;
    sL[wave][n] = lh.lo + lh.hi;
  }
  __syncthreads();
  float M = sM[0][n];
#pragma unroll
  for (int w = 1; w < NWAVES; ++w) M = fmaxf(M, sM[w][n]);
  const float a = m == -INFINITY ? 0.f : fast_exp2(m - M);   // (a wavefront without a tile: no weight)
  // (a row whose every key weighs -inf or NaN: as the unsplit kernel, nothing to rescale by)
  float part[D / 8];
  sum_tiles<D>(sSum, o, m == M ? 1.f : a, n, h, wave, tid, part);
  const int qn = tid >> 3, row_rel = rb * TILE + qn;
  float Mq = sM[0][qn];
#pragma unroll
  for (int w = 1; w < NWAVES; ++w) Mq = fmaxf(Mq, sM[w][qn]);
  float ltot = 0.f;
#pragma unroll
  for (int w = 0; w < NWAVES; ++w) {
    const float mw = sM[w][qn];
    ltot += sL[w][qn] * (mw == Mq ? 1.f : mw == -INFINITY ? 0.f : fast_exp2(mw - Mq));
  }
  if (row_rel >= Tq) return;
  const float inv = 1.f / ltot;
  const int64_t row = (int64_t)blockIdx.y * Tq + row_rel;
  const int d0 = (tid & 7) * (D / 8);
#pragma unroll
  for (int c = 0; c < D / 32; ++c) {
    const float4 x = make_float4(part[4 * c] * inv, part[4 * c + 1] * inv, part[4 * c + 2] * inv, part[4 * c + 3] * inv);
    *reinterpret_cast<float4*>(out + row * D + d0 + 4 * c) = x;
    if (y) *reinterpret_cast<float4*>(y + ys.at(b, hh) + (int64_t)row_rel * ys.row + d0 + 4 * c) = x;
  }
  if ((tid & 7) == 0) {
    rmax[row] = Mq;
    rden[row] = ltot;
  }
}

// Key side (bwd_kv_kernel's tile work). grid (ceil(T/32), nseq * H); step t takes the four query tiles
// NB - 1 - 4t - w, one per wavefront w. The selection suffix entering a wavefront's tile is the one entering
// the step plus the sums of dz of the later wavefronts' tiles, exchanged through LDS with the step's barrier.
// With reach.qstat the steps without weight for these keys are left out (kv_last_block, the same search in
// every wavefront) and the query side finds the last block in hi, one per key tile; a tile stays with the
// wavefront that had it, so the sums keep their order.
template <int D>
__global__ __launch_bounds__(NTHREADS, 1) void bwd_kv_split_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v, const float* __restrict__ dout,
    Strides qs, Strides ks, Strides vs, Strides dos, const float* __restrict__ lse, const float* __restrict__ ndbar,
    const float* __restrict__ carry, float* __restrict__ ucheck, float* __restrict__ dk0h, float* __restrict__ dk0x,
    GradView dkv, GradView dvv, int nseq, int H, int T, int64_t ldt, int exempt, float scale, BwdReach reach) {
  constexpr int DB = D / 32;
  __shared__ __attribute__((aligned(16))) float sSum[NWAVES][32 * (D + 4)];
  __shared__ float sU[2][NWAVES][TILE];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int n = lane & 31, h = lane >> 5;
  const int b = blockIdx.y / H, hh = blockIdx.y % H;
  const bool has_h0 = hh == 0;
  const int NB = (T + TILE - 1) / TILE;
  const int kt = blockIdx.x, key0 = kt * TILE, j = key0 + n;
  auto head = [&](const float* p, const Strides& s, int x) { return rsrc(p + s.at(b, x), (int64_t)T * s.row * 4); };
  const __amdgpu_buffer_rsrc_t rs_q = head(q, qs, hh), rs_q0 = head(q, qs, 0), rs_do = head(dout, dos, hh);
  HalfRow<D> kf, k0f, vf;   // B operands: lane = key
  const float* carry_col = carry + (int64_t)b * NB * T + min(j, T - 1);
  const KvProbe probe = kv_probe(reach, blockIdx.y, carry + (int64_t)b * NB * T, T, NB, key0, lane);
  kf.load(head(k, ks, hh), ks.row, j, h);
  k0f.load(head(k, ks, 0), ks.row, j, h);
  vf.load(head(v, vs, hh), vs.row, j, h);
  f32x16 dkt[DB], dvt[DB], dk0t[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    dkt[db] = zero16();
    dvt[db] = zero16();
    dk0t[db] = zero16();
  }
  float* uplane = ucheck + ((int64_t)hh * nseq + b) * utri_floats(NB);
  const float* lse_row = lse + (int64_t)blockIdx.y * ldt;
  const float* ndb_row = ndbar + (int64_t)blockIdx.y * ldt;
  const float sl2 = scale * LOG2E, neg_inv_scale = -1.f / scale;
  const int ntiles = NB - kt;
  int t0 = 0;
  if (reach.qstat) {
    int top = NB - 1;
    if (kv_worth(probe, key0, T, reach.xk, lane)) {
      const float thr = kv_threshold(kf.sumsq(), vf.sumsq(), head_qstat(reach, blockIdx.y, lane, probe.q), scale);
      top = __builtin_amdgcn_readfirstlane(
          kv_last_block(probe, carry + (int64_t)b * NB * T, T, NB, key0, reach.xk, thr, lane));
    }
    if (tid == 0) reach.hi[((int64_t)hh * nseq + b) * reach.nkg + kt] = top;
    t0 = (NB - 1 - top) / 4;
  }
  float ucarry = 0.f;
  for (int t = t0; 4 * t < ntiles; ++t) {
    const int qb = NB - 1 - 4 * t - wave;
    const bool mine = qb >= kt;
    f32x16 dz = zero16();
    uint32_t gate = 0;
    const int qbase = qb * TILE;
    if (mine) {
      const bool edge = (qbase <= key0 + TILE - 1) || key0 < exempt;
      const TileMasks mk(j, qbase, T, exempt, h, reach.xk);
      HalfRow<D> rows;
      rows.load(rs_q0, qs.row, qbase + n, h);
      const float hist = j < T ? carry_col[(int64_t)qb * T] : 0.f;
      const f32x16 l0 = mma_rows<D>(rows, k0f, zero16());
      f32x16 lg;
      selection_tile<false>(l0, hist * neg_inv_scale, h, edge, mk, gate, lg);
      if (has_h0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) lg[i] = l0[i] + lg[i];
      } else {
        rows.load(rs_q, qs.row, qbase + n, h);
        lg = mma_rows<D>(rows, kf, lg);
      }
      rows.load(rs_do, dos.row, qbase + n, h);
      const f32x16 dp = mma_rows<D>(rows, vf, rows16(ndb_row + qbase, h));   // dO.v - dbar
      f32x16 pr;
      p_dz_tile_r(lg, dp, rows16(lse_row + qbase, h), sl2, edge, mk, pr, dz);
      mma_cols<D>(dvt, rs_do, dos.row, qbase, n, h, pr);
      if (!has_h0) mma_cols<D>(dkt, rs_q, qs.row, qbase, n, h, dz);
    }
    float tot = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) tot += dz[i];
    tot += xor32(tot);
    if (h == 0) sU[t & 1][wave][n] = tot;
    __syncthreads();   // (the buffer is written again two steps on, past the next step's barrier)
    float u_in = ucarry;
#pragma unroll
    for (int w = 0; w < NWAVES; ++w) {
      const float x = sU[t & 1][w][n];
      if (w < wave) u_in += x;
      ucarry += x;
    }
    if (mine) {
      if (h == 0 && j < T) uplane[utri_row(qb) + j] = u_in;
      f32x16 gp;
      gpath_tile(dz, u_in, gate, h, gp);
      if (has_h0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) dz[i] += gp[i];
        mma_cols<D>(dkt, rs_q, qs.row, qbase, n, h, dz);
      } else {
        mma_cols<D>(dk0t, rs_q0, qs.row, qbase, n, h, gp);
      }
    }
  }
  const int jn = key0 + (tid >> 3), d0 = (tid & 7) * (D / 8);
  const bool mine = jn < T && jn >= reach.xk;   // (the first xk keys' gradients: bwd_finish_kernel)
  float part[D / 8];
  auto quad = [&](int c) { return make_float4(part[4 * c], part[4 * c + 1], part[4 * c + 2], part[4 * c + 3]); };
  sum_tiles<D>(sSum, dvt, 1.f, n, h, wave, tid, part);
#pragma unroll
  for (int c = 0; c < DB; ++c)
    if (mine) store_grad4(dvv, b, hh, jn, d0 + 4 * c, quad(c));
  sum_tiles<D>(sSum, dkt, scale, n, h, wave, tid, part);
#pragma unroll
  for (int c = 0; c < DB; ++c) {
    if (!mine) continue;
    if (has_h0 && H > 1) *reinterpret_cast<float4*>(dk0h + ((int64_t)b * T + jn) * D + d0 + 4 * c) = quad(c);
    else store_grad4(dkv, b, hh, jn, d0 + 4 * c, quad(c));
  }
  if (has_h0) return;
  sum_tiles<D>(sSum, dk0t, scale, n, h, wave, tid, part);
#pragma unroll
  for (int c = 0; c < DB; ++c)
    if (mine)
      *reinterpret_cast<float4*>(dk0x + ((int64_t)(hh - 1) * nseq * T + (int64_t)b * T + jn) * D + d0 + 4 * c) = quad(c);
}

// Query side (bwd_dq_kernel's tile work). grid (ceil(T/32), nseq * H), the longest sweeps first. With
// reach.qstat it visits the key tiles whose sweep reached its block, and those of exempt keys, which keep
// weight but have no selection suffix: one bit per key tile, 64 tiles at a time.
template <int D>
__global__ __launch_bounds__(NTHREADS, 1) void bwd_dq_split_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v, const float* __restrict__ dout,
    Strides qs, Strides ks, Strides vs, Strides dos, const float* __restrict__ lse, const float* __restrict__ ndbar,
    const float* __restrict__ carry, const float* __restrict__ ucheck, float* __restrict__ dq0h, float* __restrict__ dq0x,
    GradView dqv, int nseq, int H, int T, int64_t ldt, int exempt, float scale, BwdReach reach) {
  constexpr int DB = D / 32, LDZ = TILE + 4;
  __shared__ __attribute__((aligned(16))) float sZ[NWAVES][TILE * LDZ];
  __shared__ __attribute__((aligned(16))) float sSum[NWAVES][32 * (D + 4)];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int n = lane & 31, h = lane >> 5;
  const int b = blockIdx.y / H, hh = blockIdx.y % H;
  const bool has_h0 = hh == 0;
  const int NB = (T + TILE - 1) / TILE;
  const int qb = gridDim.x - 1 - blockIdx.x, qbase = qb * TILE;
  auto head = [&](const float* p, const Strides& s, int x) { return rsrc(p + s.at(b, x), (int64_t)T * s.row * 4); };
  const __amdgpu_buffer_rsrc_t rs_k = head(k, ks, hh), rs_k0 = head(k, ks, 0), rs_v = head(v, vs, hh);
  HalfRow<D> qa, q0a, doa;   // A operands: lane = query row
  qa.load(head(q, qs, hh), qs.row, qbase + n, h);
  q0a.load(head(q, qs, 0), qs.row, qbase + n, h);
  doa.load(head(dout, dos, hh), dos.row, qbase + n, h);
  const f32x16 lse_r = rows16(lse + (int64_t)blockIdx.y * ldt + qbase, h);
  const f32x16 ndb_r = rows16(ndbar + (int64_t)blockIdx.y * ldt + qbase, h);
  const float* carry_row = carry + ((int64_t)b * NB + qb) * T;
  const float* urow = ucheck + ((int64_t)hh * nseq + b) * utri_floats(NB) + utri_row(qb);
  const float sl2 = scale * LOG2E, neg_inv_scale = -1.f / scale;
  f32x16 dq[DB], dq0[DB];   // (D x queries)
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    dq[db] = zero16();
    dq0[db] = zero16();
  }
  // acc (D x queries) += K^T X^T: X a (queries x keys) C-layout tile, transposed through the wavefront's LDS
  // rows into the (keys x queries) layout that mma_cols takes
  auto acc_xk = [&](f32x16 (&acc)[DB], const f32x16& x, __amdgpu_buffer_rsrc_t rs, int kbase) {
    float* z = sZ[wave];
#pragma unroll
    for (int i = 0; i < 16; ++i) z[crow(i, h) * LDZ + n] = x[i];
    lds_wave_sync();
    const f32x16 xt = rows16(z + n * LDZ, h);
    lds_wave_sync();
    mma_cols<D>(acc, rs, ks.row, kbase, n, h, xt);
  };
  uint64_t reached = ~0ull;
  for (int kt = wave; kt <= qb; kt += NWAVES) {
    if (reach.qstat && kt % 64 == wave) {
      const int x = kt - wave + lane;
      reached = __ballot(x < NB && reach.hi[((int64_t)hh * nseq + b) * reach.nkg + min(x, NB - 1)] >= qb);
    }
    const int kbase = kt * TILE, j = kbase + n;
    const bool suffix = (reached >> (kt % 64)) & 1;
    if (!suffix && kbase >= exempt) continue;
    const bool edge = (kbase + TILE - 1 >= qbase) || (kbase + TILE > T) || kbase < exempt;
    const TileMasks mk(j, qbase, T, exempt, h);
    HalfRow<D> rows;
    rows.load(rs_k0, ks.row, j, h);
    const float hist = j < T ? carry_row[j] : 0.f, uin = suffix && j < T ? urow[j] : 0.f;
    const f32x16 l0 = mma_rows<D>(q0a, rows, zero16());
    f32x16 lg;
    uint32_t gate;
    selection_tile<false>(l0, hist * neg_inv_scale, h, edge, mk, gate, lg);
    if (has_h0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) lg[i] = l0[i] + lg[i];
    } else {
      rows.load(rs_k, ks.row, j, h);
      lg = mma_rows<D>(qa, rows, lg);
    }
    rows.load(rs_v, vs.row, j, h);
    const f32x16 dp = mma_rows<D>(doa, rows, ndb_r);
    f32x16 pr, dz, gp;
    p_dz_tile_r(lg, dp, lse_r, sl2, edge, mk, pr, dz);
    gpath_tile(dz, uin, gate, h, gp);
    if (has_h0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) dz[i] += gp[i];
      acc_xk(dq, dz, rs_k, kbase);
    } else {
      acc_xk(dq, dz, rs_k, kbase);
      acc_xk(dq0, gp, rs_k0, kbase);
    }
  }
  const int rn = qbase + (tid >> 3), d0 = (tid & 7) * (D / 8);
  float part[D / 8];
  const bool sums = has_h0 && H > 1;   // head 0's unscaled sums, which the other heads' shares join
  sum_tiles<D>(sSum, dq, sums ? 1.f : scale, n, h, wave, tid, part);
#pragma unroll
  for (int c = 0; c < DB; ++c) {
    if (rn >= T) continue;
    const float4 x = make_float4(part[4 * c], part[4 * c + 1], part[4 * c + 2], part[4 * c + 3]);
    if (sums) *reinterpret_cast<float4*>(dq0h + ((int64_t)b * T + rn) * D + d0 + 4 * c) = x;
    else store_grad4(dqv, b, hh, rn, d0 + 4 * c, x);
  }
  if (has_h0) return;
  sum_tiles<D>(sSum, dq0, 1.f, n, h, wave, tid, part);
#pragma unroll
  for (int c = 0; c < DB; ++c)
    if (rn < T)
      *reinterpret_cast<float4*>(dq0x + ((int64_t)(hh - 1) * nseq * T + (int64_t)b * T + rn) * D + d0 + 4 * c) =
          make_float4(part[4 * c], part[4 * c + 1], part[4 * c + 2], part[4 * c + 3]);
}

// The gradient epilogue. Workgroups [0, main_blocks): head 0's gradients, its own fp32 sums plus the other
// groups' shares, summed slot after slot in group order (so every run adds the same values in the same
// order), (b, t, D) contiguous, four elements per thread, to the caller's views; nslots slots of total4
// float4s each. The workgroups past them: the first xk (exempt) keys' dK and dV of all R heads, the sums of
// bwd_rowprep_kernel's row segments: 32 float4s of a head per workgroup, eight threads along the segments,
// their sums added in order.
__global__ __launch_bounds__(NTHREADS) void bwd_finish_kernel(
    const float4* __restrict__ dq0h, const float4* __restrict__ dk0h, const float4* __restrict__ dq0x,
    const float4* __restrict__ dk0x, int nslots, GradView dqv, GradView dkv, GradView dvv, int D, int64_t TD,
    int64_t total4, float scale, int main_blocks, int R, int H, BwdReach reach) {
  if ((int)blockIdx.x >= main_blocks) {
    __shared__ float4 sSum[8][32];
    const int per = reach.xk * 2 * D / 4;   // float4s of one head: (key, dK | dV, D)
    const int64_t e = (int64_t)(blockIdx.x - main_blocks) * 32 + (threadIdx.x & 31);
    const bool ok = e < (int64_t)R * per;
    const int r = ok ? (int)(e / per) : 0, i = ok ? (int)(e % per) : 0, sl = threadIdx.x >> 5;
    const float4* p = reinterpret_cast<const float4*>(reach.xpart) + (int64_t)r * reach.nseg * per + i;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 8
    for (int s = sl; s < reach.nseg; s += 8) {
      const float4 x = p[(int64_t)s * per];
      a = make_float4(a.x + x.x, a.y + x.y, a.z + x.z, a.w + x.w);
    }
    sSum[sl][threadIdx.x & 31] = a;
    __syncthreads();
    if (sl != 0 || !ok) return;
#pragma unroll
    for (int w = 1; w < 8; ++w) {
      const float4 x = sSum[w][threadIdx.x];
      a = make_float4(a.x + x.x, a.y + x.y, a.z + x.z, a.w + x.w);
    }
    const int j = i / (2 * D / 4), c = i % (2 * D / 4), d = 4 * (c % (D / 4));
    if (c < D / 4) store_grad4(dkv, r / H, r % H, j, d, make_float4(a.x * scale, a.y * scale, a.z * scale, a.w * scale));
    else store_grad4(dvv, r / H, r % H, j, d, a);
    return;
  }
  for (int64_t e = (int64_t)blockIdx.x * NTHREADS + threadIdx.x; e < total4; e += (int64_t)main_blocks * NTHREADS) {
    const int64_t b = (4 * e) / TD, off = 4 * e - b * TD;
    const int t = (int)(off / D), d = (int)(off - (int64_t)t * D);
    float4 q = dq0h[e], k = dk0h[e];
    for (int sl = 0; sl < nslots; ++sl) {
      const float4 qx = dq0x[sl * total4 + e], kx = dk0x[sl * total4 + e];
      q = make_float4(q.x + qx.x, q.y + qx.y, q.z + qx.z, q.w + qx.w);
      k = make_float4(k.x + kx.x, k.y + kx.y, k.z + kx.z, k.w + kx.w);
    }
    store_grad4(dqv, b, 0, t, d, make_float4(q.x * scale, q.y * scale, q.z * scale, q.w * scale));
    if (t >= reach.xk) store_grad4(dkv, b, 0, t, d, k);
  }
}


// ---------------------------------------------------------------------------------------------
// Decode step: one new query per head (position t-1) over a key cache of t keys. HBM-bound: every
// cached K and V row is read once. grid (ceil(t / chunk), nseq * heads): a workgroup takes one
// head over `chunk` keys (a multiple of 256 the host picks so that the grid fills the chip),
// wavefront w the keys [w chunk/4, (w+1) chunk/4) of that range, DEC_STEP keys at a time.
//
// Lane layout: lane = (row slot kq, column slice dc), LPK = D / (elements per 16 bytes) lanes per
// cached row, so one 16-byte load instruction reads 64 / LPK whole rows, contiguous in HBM. A lane
// holds its slice of q and, per step, NR rows of K and the same NR rows of V (both issued before
// any arithmetic). The NR partial dot products reduce over the LPK lanes of a row by a
// reduce-scatter (log2 NR exchange rounds that halve the values a lane carries), after which lane
// (kq, dc) holds the full logit of row slot kq of load dc / (LPK / NR). The wavefront then takes
// the step's maximum, rescales its running output when the maximum rises, passes the
// probabilities through LDS to the lanes holding the V rows, and adds p_j v_j into each lane's
// column slice. The wavefronts' partials (max, sum, output) merge in LDS; one partial per
// workgroup goes to the workspace. The group's selector head writes the updated selection to the
// workspace's state rows; decode_finish_kernel merges the partials and copies the state rows over
// the caller's state after every head has read the old one (a kernel boundary later).

constexpr int DEC_NR = 8;   // cached rows of K (and of V) per lane per step, at most
template <typename E, int D>
struct DecLayout {
  static constexpr int EPC = 16 / (int)sizeof(E);   // elements per 16-byte load
  static constexpr int LPK = D / EPC;                // lanes per cached row
  static constexpr int KPI = 64 / LPK;               // rows per load instruction
  static constexpr int NR = LPK < DEC_NR ? LPK : DEC_NR;   // rows per lane per step (K, V each)
  static constexpr int DUP = LPK / NR;               // lanes holding one logit after the reduction
  static constexpr int STEP = KPI * NR;              // keys per wavefront step
};

__device__ __forceinline__ float wave_max(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x = fmaxf(x, __shfl_xor(x, o));
  return x;
}
__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
  return x;
}
template <typename E>
__device__ __forceinline__ float to_f32(E x) {
  if constexpr (sizeof(E) == 2) return __uint_as_float(((uint32_t)x) << 16);
  else return x;
}

template <typename E, int D>
__global__ __launch_bounds__(NTHREADS) void decode_partial_kernel(
    const E* __restrict__ q, const E* __restrict__ k, const E* __restrict__ v, const float* __restrict__ selected,
    int64_t state_ld, float* __restrict__ pm, float* __restrict__ pl, float* __restrict__ po,
    float* __restrict__ next_state, int heads, int groups, int t, int64_t kvs, int exempt, float scale, int chunk,
    int nchunk) {
  using L = DecLayout<E, D>;
  constexpr int EPC = L::EPC, LPK = L::LPK, KPI = L::KPI, NR = L::NR, DUP = L::DUP, STEP = L::STEP;
  union Row {
    uint4 u;
    E e[EPC];
  };
  __shared__ __align__(16) float sP[NWAVES][STEP];
  __shared__ float sPart[NWAVES][D + 2];

  const int cidx = blockIdx.x;
  const int64_t row = blockIdx.y;             // b * heads + head
  const int per = heads / groups;
  const int b = (int)(row / heads), hd = (int)(row % heads);
  const int64_t sg = (int64_t)b * groups + hd / per;
  const bool selector = (hd % per) == 0;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int kq = lane / LPK, dc = lane % LPK;
  const int ri = dc / DUP;                    // after the reduction: the logit of row kq of load ri
  const bool owner = dc % DUP == 0;           // one lane per logit writes it
  const int wkeys = chunk / NWAVES;
  const int kw0 = cidx * chunk + wave * wkeys;
  const int kw_end = min(kw0 + wkeys, t);
  const float* selrow = selected + sg * state_ld;
  float* nextrow = next_state + sg * t;

  float qf[EPC];
  {
    Row qq;
    qq.u = *reinterpret_cast<const uint4*>(q + row * D + EPC * dc);
#pragma unroll
    for (int e = 0; e < EPC; ++e) qf[e] = to_f32(qq.e[e]) * scale;
  }
  // buffer resources over the head's t cached rows: the loads take one lane offset (row slot and
  // column slice) plus a wavefront-uniform offset of the rows, and rows at or past t read as zero
  constexpr int RB = D * (int)sizeof(E);   // bytes per cached row
  const int nbytes = t * RB;               // < 2^31 (rows_fit, checked by the C ABI)
  const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc((void*)(k + row * kvs), 0, nbytes, RSRC_WORD3);
  const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc((void*)(v + row * kvs), 0, nbytes, RSRC_WORD3);
  const int loff = kq * RB + EPC * dc * (int)sizeof(E);
  float m = -INFINITY, l = 0.f, o[EPC];
#pragma unroll
  for (int e = 0; e < EPC; ++e) o[e] = 0.f;

  for (int kw = kw0; kw < kw_end; kw += STEP) {
    Row kr[NR], vr[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const auto x = __builtin_amdgcn_raw_buffer_load_b128(krs, loff, (kw + i * KPI) * RB, 0);
      kr[i].u = make_uint4(x[0], x[1], x[2], x[3]);
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const auto x = __builtin_amdgcn_raw_buffer_load_b128(vrs, loff, (kw + i * KPI) * RB, 0);
      vr[i].u = make_uint4(x[0], x[1], x[2], x[3]);
    }
    const int j = kw + ri * KPI + kq;         // this lane's logit after the reduction
    const bool jok = j < t;
    const float sel = jok ? selrow[j] : 0.f;
    float a[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      float s = 0.f;
#pragma unroll
      for (int e = 0; e < EPC; ++e) s = fmaf(qf[e], to_f32(kr[i].e[e]), s);
      a[i] = s;
    }
    // reduce-scatter over the row's lanes: the round with lane bit `s` keeps the upper half of the
    // values on lanes with the bit set, the lower half on the others, and adds the partner's copy
#pragma unroll
    for (int st = 1; st < NR; st <<= 1) {   // st = 1, 2, ..., NR/2: constant trip count, unrolled
      const int half = NR / (2 * st), s = LPK / (2 * st);
      // all-ones on lanes with the bit: a bitwise select (a ?: on the array elements becomes a
      // dynamically indexed read of the array)
      const uint32_t up = (lane & s) ? 0xffffffffu : 0u;
#pragma unroll
      for (int i = 0; i < half; ++i) {
        const uint32_t lo = __float_as_uint(a[i]), hi = __float_as_uint(a[i + half]);
        const float send = __uint_as_float((lo & up) | (hi & ~up));
        const float keep = __uint_as_float((hi & up) | (lo & ~up));
        a[i] = keep + __shfl_xor(send, s);
      }
    }
#pragma unroll
    for (int s = DUP / 2; s >= 1; s >>= 1) a[0] += __shfl_xor(a[0], s);
    const float raw = a[0];
    if (selector && owner && j >= exempt && j < t - 1) nextrow[j] = sel + fmaxf(raw, 0.f);
    const float z = jok ? (raw - sel) * LOG2E : -INFINITY;
    const float m_new = fmaxf(m, wave_max(z));   // finite: a step's first key is < t
    const float alpha = fast_exp2(m - m_new);    // 0 on the first step (m = -inf)
    const float p = jok ? fast_exp2(z - m_new) : 0.f;
    l = fmaf(l, alpha, owner ? p : 0.f);         // per lane; summed over the wavefront at the end
#pragma unroll
    for (int e = 0; e < EPC; ++e) o[e] *= alpha;
    m = m_new;
    if (owner) sP[wave][kq * NR + ri] = p;
    lds_wave_sync();
    float pr[NR];
#pragma unroll
    for (int i = 0; i < NR; i += 4) {
      const float4 p4 = *reinterpret_cast<const float4*>(&sP[wave][kq * NR + i]);
      pr[i] = p4.x;
      pr[i + 1] = p4.y;
      pr[i + 2] = p4.z;
      pr[i + 3] = p4.w;
    }
    lds_wave_sync();   // sP is rewritten next step
#pragma unroll
    for (int i = 0; i < NR; ++i)
#pragma unroll
      for (int e = 0; e < EPC; ++e) o[e] = fmaf(pr[i], to_f32(vr[i].e[e]), o[e]);
  }
  l = wave_sum(l);
#pragma unroll
  for (int sh = LPK; sh < 64; sh <<= 1)
#pragma unroll
    for (int e = 0; e < EPC; ++e) o[e] += __shfl_xor(o[e], sh);
  if (kq == 0) {
#pragma unroll
    for (int e = 0; e < EPC; ++e) sPart[wave][2 + EPC * dc + e] = o[e];
  }
  if (lane == 0) {
    sPart[wave][0] = m;   // -inf for a wavefront with no key (its l and o are 0)
    sPart[wave][1] = l;
  }
  __syncthreads();
  // merge the wavefronts' partials: wavefront 0, lanes over D + 2
  if (wave == 0) {
    float mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < NWAVES; ++w) mx = fmaxf(mx, sPart[w][0]);
    const int64_t slot = row * nchunk + cidx;
    for (int c = lane; c < D + 2; c += 64) {
      float acc = 0.f;
#pragma unroll
      for (int w = 0; w < NWAVES; ++w) {
        const float wt = sPart[w][0] == -INFINITY ? 0.f : fast_exp2(sPart[w][0] - mx);
        acc = fmaf(wt, sPart[w][c], acc);
      }
      if (c == 0) pm[slot] = mx;
      else if (c == 1) pl[slot] = acc;
      else po[slot * D + c - 2] = acc;
    }
  }
}

// Blocks [0, rows): out[row] = the row's partials merged, sum_p 2^(m_p - M) o_p / sum_p 2^(m_p - M)
// l_p. Thread i first takes the maxima and sums of partials i, i + 256, ... (the weights go to LDS),
// then thread (slot, column quad) the output quads of partials slot, slot + 1024/D, ..., a batch of
// DEC_FIN_UNROLL loads in flight at a time; slots reduce over lanes and then over wavefronts.
// Blocks from `rows` on: selected[g][j] = the selector heads' updates (rows of t in next_state),
// exempt <= j < t - 1, `sblocks` blocks of 1024 keys per state row.
constexpr int DEC_FIN_UNROLL = 8;
constexpr int DEC_FIN_MAXPARTS = 4096;   // LDS weights of one row: nparts <= this

template <int D>
__global__ __launch_bounds__(NTHREADS) void decode_finish_kernel(
    const float* __restrict__ pm, const float* __restrict__ pl, const float* __restrict__ po, float* __restrict__ out,
    int nparts, int rows, float* __restrict__ selected, const float* __restrict__ next_state, int64_t state_ld, int t,
    int exempt, int sblocks) {
  constexpr int QPP = D / 4;               // float4 quads per partial
  constexpr int SLOTS = NTHREADS / QPP;    // partials in flight per load instruction
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  if ((int)blockIdx.x >= rows) {
    const int s = (int)blockIdx.x - rows;
    const int64_t g = s / sblocks;
    const int j0 = (s % sblocks) * (4 * NTHREADS);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = j0 + u * NTHREADS + tid;
      if (j >= exempt && j < t - 1) selected[g * state_ld + j] = next_state[g * t + j];
    }
    return;
  }
  __shared__ float sW[DEC_FIN_MAXPARTS];
  __shared__ float sRed[NWAVES];
  __shared__ float4 sO[NWAVES][QPP];
  const int64_t row = blockIdx.x;
  const float* rm = pm + row * nparts;
  const float* rl = pl + row * nparts;
  const float4* ro = reinterpret_cast<const float4*>(po + row * nparts * (int64_t)D);

  float mx = -INFINITY;
  for (int i = tid; i < nparts; i += NTHREADS) {
    const float m = rm[i];
    sW[i] = m;
    mx = fmaxf(mx, m);
  }
  mx = wave_max(mx);
  if (lane == 0) sRed[wave] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(sRed[0], sRed[1]), fmaxf(sRed[2], sRed[3]));   // finite: every partial has a key
  __syncthreads();   // sRed is reused below
  float l = 0.f;
  for (int i = tid; i < nparts; i += NTHREADS) {
    const float w = fast_exp2(sW[i] - mx);
    sW[i] = w;
    l = fmaf(w, rl[i], l);
  }
  l = wave_sum(l);
  if (lane == 0) sRed[wave] = l;
  __syncthreads();
  l = sRed[0] + sRed[1] + sRed[2] + sRed[3];

  const int slot = tid / QPP, cq = tid % QPP;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int i0 = slot; i0 < nparts; i0 += SLOTS * DEC_FIN_UNROLL) {
    float4 x[DEC_FIN_UNROLL];
#pragma unroll
    for (int u = 0; u < DEC_FIN_UNROLL; ++u) {
      const int i = i0 + u * SLOTS;
      x[u] = i < nparts ? ro[(int64_t)i * QPP + cq] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < DEC_FIN_UNROLL; ++u) {
      const int i = i0 + u * SLOTS;
      const float w = i < nparts ? sW[i] : 0.f;
      acc.x = fmaf(w, x[u].x, acc.x);
      acc.y = fmaf(w, x[u].y, acc.y);
      acc.z = fmaf(w, x[u].z, acc.z);
      acc.w = fmaf(w, x[u].w, acc.w);
    }
  }
#pragma unroll
  for (int sh = QPP; sh < 64; sh <<= 1) {
    acc.x += __shfl_xor(acc.x, sh);
    acc.y += __shfl_xor(acc.y, sh);
    acc.z += __shfl_xor(acc.z, sh);
    acc.w += __shfl_xor(acc.w, sh);
  }
  if (lane < QPP) sO[wave][lane] = acc;
  __syncthreads();
  if (tid < QPP) {
    float4 o = sO[0][tid];
#pragma unroll
    for (int w = 1; w < NWAVES; ++w) {
      o.x += sO[w][tid].x;
      o.y += sO[w][tid].y;
      o.z += sO[w][tid].z;
      o.w += sO[w][tid].w;
    }
    const float inv = 1.f / l;
    reinterpret_cast<float4*>(out + row * D)[tid] = make_float4(o.x * inv, o.y * inv, o.z * inv, o.w * inv);
  }
}

// ---------------------------------------------------------------------------------------------
// Host side: launch sequences of one storage dtype and head dim.

template <class OP, int D>
int run_selection(const FwdCall& c, hipStream_t st) {
  using elem = typename OP::elem;
  const int NBq = (int)cdiv(c.Tq, TILE), NKT = (int)cdiv(c.Tk, TILE);
  const int64_t nkb = cdiv(c.Tk, NORM_KEYS);
  TimedLaunch timed(SA_KERNEL_SELECTION, st);
  auto norms_apart = [&]() {
    hipLaunchKernelGGL((key_norms_kernel<elem, D>), dim3((unsigned)nkb, (unsigned)(c.nseq * c.H)), dim3(NTHREADS), 0, st,
                       static_cast<const elem*>(c.k), static_cast<const elem*>(c.v), c.ks, c.vs, c.H, c.Tk, c.kn, c.kt);
  };
  if constexpr (sizeof(elem) == 2 && D == 64) {
    const int64_t wgs = cdiv(NKT, NWAVES * SEL_CARRY_KPW);
    // (its carry stores address one sequence's plane through a 32-bit buffer range)
    if (wgs * c.nseq >= SEL_CARRY_MIN_BLOCKS && (int64_t)NBq * c.Tk * 4 < ((int64_t)1 << 31)) {
      hipLaunchKernelGGL(sel_carry64_kernel, dim3((unsigned)wgs, (unsigned)c.nseq), dim3(NTHREADS), 0,
                         st, static_cast<const uint16_t*>(c.q), static_cast<const uint16_t*>(c.k), c.carry,
                         c.state_in, c.state_out, c.state_ld, c.Tq, c.Tk, c.qs, c.ks, c.q_off, c.exempt, c.scale, c.kt);
      if (c.kn) norms_apart();
      return launch_status();
    }
  }
  const int RB = SEL_RB;
  dim3 g1((unsigned)cdiv(NKT, NWAVES), (unsigned)cdiv(NBq, RB), (unsigned)c.nseq);
  // the key norms' workgroups, unless they would take z past a grid's limit (tens of thousands of sequences)
  const int64_t znorms = c.kn ? cdiv((int64_t)c.nseq * c.H * nkb, (int64_t)g1.x * g1.y) : 0;
  const bool norms_along = c.nseq + znorms <= 65535;
  if (norms_along) g1.z += (unsigned)znorms;
  hipLaunchKernelGGL((sel_colsum_kernel<OP, D>), g1, dim3(NTHREADS), 0, st, static_cast<const elem*>(c.q),
                     static_cast<const elem*>(c.k), c.carry, c.H, c.Tq, c.Tk, c.qs, c.ks, c.q_off, c.exempt, c.scale,
                     RB, static_cast<const elem*>(c.v), c.vs, c.nseq, c.kn, c.q_off > 0 ? c.state_in : nullptr, c.state_ld);
  dim3 g2((unsigned)cdiv(c.Tk, NTHREADS), (unsigned)c.nseq);
  hipLaunchKernelGGL(sel_scan_kernel, g2, dim3(NTHREADS), 0, st, c.carry, c.state_in, c.state_out, c.state_ld, NBq,
                     c.Tk, c.q_off, c.kt);
  if (!norms_along) norms_apart();
  return launch_status();
}

template <class OP, int D, int G>
void launch_fwd(const FwdCall& c, const typename OP::elem* vt, int64_t ldv) {   // vt: V^T (fwd_kernel only)
  using elem = typename OP::elem;
  const int NBq = (int)cdiv(c.Tq, TILE);
  dim3 grid((unsigned)cdiv(NBq, NWAVES), (unsigned)(c.nseq * (c.H / G)));
  // the layout of sa_forward: q contiguous, k rows D apart, k's sequences H heads apart
  const bool cv = c.qs.row == D && c.qs.head == (int64_t)c.Tq * D && c.qs.seq == (int64_t)c.H * c.qs.head &&
                  c.ks.row == D && c.ks.seq == (int64_t)c.H * c.ks.head;
  TimedLaunch timed(SA_KERNEL_FORWARD, c.st);
  if constexpr (sizeof(elem) == 2 && D == 64 && G <= 2) {   // the direct-load kernel
#define SA_LAUNCH_FWD64(CVV)                                                                                      \
  hipLaunchKernelGGL((fwd64_kernel<CVV, G>), grid, dim3(NTHREADS), 0, c.st, static_cast<const elem*>(c.q),       \
                     static_cast<const elem*>(c.k), static_cast<const elem*>(c.v), c.carry, c.out, c.rmax,        \
                     c.rden, static_cast<elem*>(c.y), c.ys, c.H, c.Tq, c.Tk, c.qs, c.ks, c.vs, c.q_off, c.exempt, \
                     c.scale, c.damp_mode, c.train_len, c.kn, c.kt)
    if (cv) SA_LAUNCH_FWD64(true);
    else SA_LAUNCH_FWD64(false);
#undef SA_LAUNCH_FWD64
  } else {
#define SA_LAUNCH_FWD(CVV)                                                                                        \
  hipLaunchKernelGGL((fwd_kernel<OP, D, G, CVV>), grid, dim3(NTHREADS), 0, c.st, static_cast<const elem*>(c.q),  \
                     static_cast<const elem*>(c.k), vt, c.carry, c.out, c.rmax, c.rden, static_cast<elem*>(c.y),  \
                     c.ys, c.H, c.Tq, c.Tk, c.qs, c.ks, c.q_off, ldv, c.exempt, c.scale, c.damp_mode, c.train_len, c.kn, \
                     c.kt)
    if (cv) SA_LAUNCH_FWD(true);
    else SA_LAUNCH_FWD(false);
#undef SA_LAUNCH_FWD
  }
}

template <class OP, int D>
int forward_impl(const FwdCall& c) {
  using elem = typename OP::elem;
  const int64_t ldv = sa_transposed_ld(c.Tk);
  elem* vt = static_cast<elem*>(c.ws);
  const int dtype = sizeof(elem) == 2 ? SA_DTYPE_BF16 : SA_DTYPE_F32;
  int G = auto_group(dtype, D, c.H, c.group, false);
  if constexpr (sizeof(elem) == 2 && D <= 64) {
    if (c.group <= 0 && G >= 2) G = fwd64_group(c.nseq, c.H, c.Tq, device_cus());
  }
  if constexpr (sizeof(elem) == 4 && D <= 64) {
    if (c.damp_mode == 0 && split_f32_grid(c.nseq, c.H, c.Tq, c.Tk, device_cus(), false)) {
      FwdCall sc = c;
      sc.kn = sc.kt = nullptr;   // (every tile is visited)
      const int rc = run_selection<OP, D>(sc, c.st);
      if (rc) return rc;
      TimedLaunch timed(SA_KERNEL_FORWARD, c.st);
      hipLaunchKernelGGL((fwd_split_kernel<D>), dim3((unsigned)cdiv(c.Tq, TILE), (unsigned)(c.nseq * c.H)), dim3(NTHREADS),
                         0, c.st, static_cast<const float*>(c.q), static_cast<const float*>(c.k),
                         static_cast<const float*>(c.v), c.carry, c.out, c.rmax, c.rden, static_cast<float*>(c.y), c.ys, c.H,
                         c.Tq, c.Tk, c.qs, c.ks, c.vs, c.q_off, c.exempt, c.scale);
      return launch_status();
    }
  }
  // V^T for fwd_kernel (fwd64_kernel, bf16 at head dim 64 with G <= 2, reads the V rows transposed
  // from LDS)
  if (!(sizeof(elem) == 2 && D == 64 && G <= 2))
    launch_transpose<elem, D>(static_cast<const elem*>(c.v), vt, c.Tk, ldv, c.vs, c.H, (int64_t)c.nseq * c.H, c.st);
  int rc = run_selection<OP, D>(c, c.st);
  if (rc) return rc;
  if (G == 4) {
    if constexpr (sizeof(elem) == 2 && D <= 64) launch_fwd<OP, D, 4>(c, vt, ldv);
  } else if (G == 2) {
    if constexpr (sizeof(elem) == 2 && D <= 64) launch_fwd<OP, D, 2>(c, vt, ldv);
  } else {
    launch_fwd<OP, D, 1>(c, vt, ldv);
  }
  return launch_status();
}

template <class OP, int D>
void launch_rowprep(const BwdCall& c, const PrepLaunch& p) {
  using elem = typename OP::elem;
#define SA_LAUNCH_PREP(ONE)                                                                                        \
  hipLaunchKernelGGL((bwd_rowprep_kernel<OP, D, ONE>), dim3((unsigned)cdiv(p.ldt, QSTAT_ROWS), (unsigned)(c.nseq * c.H)), \
                     dim3(NTHREADS), 0, c.st, static_cast<const elem*>(c.q), static_cast<const elem*>(c.k),              \
                     static_cast<const elem*>(c.v), static_cast<const elem*>(c.dout), c.qs, c.ks, c.vs, c.dos, c.H, c.T, \
                     c.out, c.rmax, c.rden, p.lse, p.ndbar, p.ldt, c.scale, p.reach)
  if (p.reach.xk == 1) SA_LAUNCH_PREP(true);
  else SA_LAUNCH_PREP(false);
#undef SA_LAUNCH_PREP
}

// Launch of the key-side kernel from its arguments (the grid as launch_bwd's).
template <class OP, int D, int G, bool CV>
void launch_kv_from(const KvLaunch& a) {
  using elem = typename OP::elem;
  dim3 grid((unsigned)cdiv(a.T, NWAVES * TILE), (unsigned)(a.nseq * (a.H / G)));
  hipLaunchKernelGGL((bwd_kv_kernel<OP, D, G, CV>), grid, dim3(NTHREADS), 0, a.st, static_cast<const elem*>(a.q),
                     static_cast<const elem*>(a.k), static_cast<const elem*>(a.v), static_cast<const elem*>(a.qt),
                     static_cast<const elem*>(a.dout), static_cast<const elem*>(a.dot), a.qs, a.ks, a.vs, a.dos, a.lse,
                     a.dbar, a.carry, a.ucheck, a.dk0h, a.dk0x, a.dkv, a.dvv, a.nseq, a.H, a.T, a.ldt, a.exempt,
                     a.scale, a.reach);
}

template <bool CV, bool SOLO>
void launch_kv64_from(const KvLaunch& a) {
  dim3 grid((unsigned)cdiv(a.T, NWAVES * TILE), (unsigned)(a.nseq * a.H));
  hipLaunchKernelGGL((bwd_kv64_kernel<CV, SOLO>), grid, dim3(NTHREADS), 0, a.st, static_cast<const uint16_t*>(a.q),
                     static_cast<const uint16_t*>(a.k), static_cast<const uint16_t*>(a.v),
                     static_cast<const uint16_t*>(a.dout), a.qs, a.ks, a.vs, a.dos, a.lse, a.dbar, a.carry, a.ucheck,
                     a.dk0h, a.dk0x, a.dkv, a.dvv, a.nseq, a.H, a.T, a.ldt, a.exempt, a.scale, a.reach);
}

// The two backward kernels; returns the launch status.
template <class OP, int D, int G>
int launch_bwd(const BwdCall& c, const typename OP::elem* qt, const typename OP::elem* kt,
                const typename OP::elem* dot, const float* lse, const float* dbar, float* ucheck, float* dq0h,
                float* dk0h, float* dq0x, float* dk0x, int64_t ldt, const BwdReach& reach) {
  using elem = typename OP::elem;
  const elem* q = static_cast<const elem*>(c.q);
  const elem* k = static_cast<const elem*>(c.k);
  const elem* v = static_cast<const elem*>(c.v);
  const elem* dout = static_cast<const elem*>(c.dout);
  dim3 grid((unsigned)cdiv(c.T, NWAVES * TILE), (unsigned)(c.nseq * (c.H / G)));
  // every view the contiguous (nseq, H, T, D) layout of sa_backward
  auto contiguous = [&](const Strides& s) {
    return s.row == D && s.head == (int64_t)c.T * D && s.seq == (int64_t)c.H * s.head;
  };
  const bool cv = contiguous(c.qs) && contiguous(c.ks) && contiguous(c.vs) && contiguous(c.dos);
  const int f32 = c.grad_dtype == SA_DTYPE_F32;
  const GradView dqv{c.dq, c.dqs, f32}, dkv{c.dk, c.dks, f32}, dvv{c.dv, c.dvs, f32};
  const KvLaunch kv{q,    k,       v,      qt,   dout, dot,    c.qs, c.ks, c.vs, c.dos,    lse,      dbar,
                    c.carry, ucheck, dk0h, dk0x, dkv,  dvv,    c.nseq, c.H,  c.T,  ldt,      c.exempt, c.scale,
                    reach, c.st};
  // bf16: the key-side kernel's instances live in a translation unit of their own (sa_bf16_kv.hip)
  auto launch_kv = [&](bool cvv) -> int {
    if constexpr (sizeof(elem) == 2) {
      return launch_bwd_kv_bf16(D, G, cvv, kv);
    } else {
      if (cvv) launch_kv_from<OP, D, G, true>(kv);
      else launch_kv_from<OP, D, G, false>(kv);
      return launch_status();
    }
  };
#define SA_LAUNCH_DQ(CVV)                                                                                         \
  hipLaunchKernelGGL((bwd_dq_kernel<OP, D, G, CVV>), grid, dim3(NTHREADS), 0, c.st, q, k, v, kt, dout, c.qs, c.ks, \
                     c.vs, c.dos, lse, dbar, c.carry, ucheck, dq0h, dq0x, dqv, c.nseq, c.H, c.T, ldt, c.exempt,   \
                     c.scale, reach)
  {
    TimedLaunch timed(SA_KERNEL_BACKWARD, c.st);
    const int rc = launch_kv(cv);
    if (rc) return rc;
  }
  {
    TimedLaunch timed(SA_KERNEL_BACKWARD_DQ, c.st);
    if constexpr (sizeof(elem) == 2 && D == 64 && G == 1) {   // one head per wavefront: the pipelined kernel
      const dim3 grid64((unsigned)cdiv(c.T, DQ64_WAVES * TILE), (unsigned)(c.nseq * c.H));
#define SA_LAUNCH_DQ64(CVV, SOLO, SNAKE)                                                                           \
  hipLaunchKernelGGL((bwd_dq64_kernel<CVV, SOLO, SNAKE>), grid64, dim3(DQ64_WAVES * 64), 0, c.st, q, k, v, dout, c.qs, \
                     c.ks, c.vs, c.dos, lse, dbar, c.carry, ucheck, dq0h, dq0x, dqv, c.nseq, c.H, c.T, ldt, c.exempt, \
                     c.scale, dq_slots, reach)
      const int dq_slots = bwd_snake_slots((int64_t)grid64.x * grid64.y, 1, device_cus());
      if (c.H == 1) {   // one-head sequences: head 0's loop only
        if (cv) SA_LAUNCH_DQ64(true, true, false);
        else SA_LAUNCH_DQ64(false, true, false);
      } else if (dq_slots > 0) {
        if (cv) SA_LAUNCH_DQ64(true, false, true);
        else SA_LAUNCH_DQ64(false, false, true);
      } else {
        if (cv) SA_LAUNCH_DQ64(true, false, false);
        else SA_LAUNCH_DQ64(false, false, false);
      }
#undef SA_LAUNCH_DQ64
    } else {
      if (cv) SA_LAUNCH_DQ(true);
      else SA_LAUNCH_DQ(false);
    }
  }
#undef SA_LAUNCH_DQ
  return launch_status();
}

template <class OP, int D>
int backward_impl(const BwdCall& c) {
  using elem = typename OP::elem;
  const int nseq = c.nseq, H = c.H, T = c.T;
  const hipStream_t st = c.st;
  const int dtype = sizeof(elem) == 2 ? SA_DTYPE_BF16 : SA_DTYPE_F32;
  const int G = bwd_group(dtype, D, H, c.group);
  const int64_t R = (int64_t)nseq * H, ldt = sa_transposed_ld(T);
  const BwdLayout L = bwd_layout(nseq, H, T, D, sizeof(elem), G);
  char* base = static_cast<char*>(c.ws);
  elem* qt = reinterpret_cast<elem*>(base + L.qt);
  elem* dot = reinterpret_cast<elem*>(base + L.dot);
  elem* kt = reinterpret_cast<elem*>(base + L.kt);
  float* lse = reinterpret_cast<float*>(base + L.lse);
  float* dbar = reinterpret_cast<float*>(base + L.dbar);
  float* dq0h = reinterpret_cast<float*>(base + L.dq);
  float* dk0h = reinterpret_cast<float*>(base + L.dk);
  float* dq0x = reinterpret_cast<float*>(base + L.dq0x);
  float* dk0x = reinterpret_cast<float*>(base + L.dk0x);
  float* ucheck = reinterpret_cast<float*>(base + L.ucheck);
  const elem* q = static_cast<const elem*>(c.q);
  const elem* k = static_cast<const elem*>(c.k);
  const elem* dout = static_cast<const elem*>(c.dout);

  // bf16 at head dim 64 the backward kernels read their Q, dO and K rows transposed from LDS
  // (bwd_kv64_kernel, bwd_dq64_kernel): no transposed copies
  bool split = false;
  if constexpr (sizeof(elem) == 4 && D <= 64) split = split_f32_grid(nseq, H, T, T, device_cus(), true);
  if (!(sizeof(elem) == 2 && D == 64) && !split) {
    launch_transpose<elem, D>(q, qt, T, ldt, c.qs, H, R, st);
    launch_transpose<elem, D>(dout, dot, T, ldt, c.dos, H, R, st);
    launch_transpose<elem, D>(k, kt, T, ldt, c.ks, H, R, st);
  }
  BwdReach reach{};
  reach.nseg = (int)cdiv(T, QSTAT_ROWS);
  reach.nkg = (int)cdiv(T, split ? TILE : NWAVES * TILE);
  if (c.reach) {
    reach.xk = exempt_apart(c.exempt);
    const BwdReachLayout RL = bwd_reach_layout(nseq, H, T, D, reach.xk);
    reach.qstat = reinterpret_cast<float2*>(c.reach + RL.qstat);
    reach.hi = reinterpret_cast<int*>(c.reach + RL.hi);
    reach.xpart = reinterpret_cast<float*>(c.reach + RL.xpart);
  }
  const PrepLaunch prep{lse, dbar, ldt, reach};
  if constexpr (sizeof(elem) == 2) launch_rowprep_bf16(c, prep);
  else launch_rowprep<OP, D>(c, prep);
  int rc = launch_status();   // the transposes and row statistics
  if (rc) return rc;
#define SA_LAUNCH_BWD(GG) launch_bwd<OP, D, GG>(c, qt, kt, dot, lse, dbar, ucheck, dq0h, dk0h, dq0x, dk0x, ldt, reach)
  if constexpr (sizeof(elem) == 2 && D <= 32) {
    rc = (G == 2) ? SA_LAUNCH_BWD(2) : SA_LAUNCH_BWD(1);
  } else if (split) {
    if constexpr (sizeof(elem) == 4 && D <= 64) {
      const dim3 grid((unsigned)cdiv(T, TILE), (unsigned)R);
      const int gf32 = c.grad_dtype == SA_DTYPE_F32;
      const float* v = static_cast<const float*>(c.v);
      {
        TimedLaunch timed(SA_KERNEL_BACKWARD, st);
        hipLaunchKernelGGL((bwd_kv_split_kernel<D>), grid, dim3(NTHREADS), 0, st, q, k, v, dout, c.qs, c.ks, c.vs, c.dos, lse,
                           dbar, c.carry, ucheck, dk0h, dk0x, GradView{c.dk, c.dks, gf32}, GradView{c.dv, c.dvs, gf32}, nseq,
                           H, T, ldt, c.exempt, c.scale, reach);
      }
      TimedLaunch timed(SA_KERNEL_BACKWARD_DQ, st);
      hipLaunchKernelGGL((bwd_dq_split_kernel<D>), grid, dim3(NTHREADS), 0, st, q, k, v, dout, c.qs, c.ks, c.vs, c.dos, lse,
                         dbar, c.carry, ucheck, dq0h, dq0x, GradView{c.dq, c.dqs, gf32}, nseq, H, T, ldt, c.exempt, c.scale,
                         reach);
      rc = launch_status();
    }
  } else {
    rc = SA_LAUNCH_BWD(1);
  }
#undef SA_LAUNCH_BWD
  if (rc) return rc;
  // (a one-head sequence's kernels wrote its gradients to the views, but for the exempt keys')
  if (H == 1 && reach.xk == 0) return SA_OK;
  // head 0's dQ, dK: its own sums plus the other groups' shares
  const int64_t total4 = H == 1 ? 0 : (int64_t)nseq * T * D / 4;
  const int f32 = c.grad_dtype == SA_DTYPE_F32;
  const unsigned main_blocks = (unsigned)std::min<int64_t>(cdiv(total4, NTHREADS), 8192);
  const unsigned exempt_blocks = (unsigned)cdiv(R * reach.xk * 2 * D / 4, 32);
  hipLaunchKernelGGL(bwd_finish_kernel, dim3(main_blocks + exempt_blocks),
                     dim3(NTHREADS), 0, st, reinterpret_cast<const float4*>(dq0h),
                     reinterpret_cast<const float4*>(dk0h), reinterpret_cast<const float4*>(dq0x),
                     reinterpret_cast<const float4*>(dk0x), H / G - 1, GradView{c.dq, c.dqs, f32},
                     GradView{c.dk, c.dks, f32}, GradView{c.dv, c.dvs, f32}, D,
                     (int64_t)T * D, total4, c.scale, (int)main_blocks, (int)R, H, reach);
  return launch_status();
}

// Keys per decode workgroup: the smallest power of two from 256 up that keeps the grid at or under
// 2048 workgroups (8 per CU) up to 4096 keys, and beyond that as far as a row's partials need to
// fit decode_finish_kernel's LDS.
inline int decode_chunk(int64_t rows, int64_t t) {
  int64_t chunk = 256;
  while ((chunk < 4096 && rows * cdiv(t, chunk) > 2048) || cdiv(t, chunk) > DEC_FIN_MAXPARTS) chunk *= 2;
  return (int)chunk;
}

template <class OP, int D>
int decode_impl(const DecCall& c) {
  using elem = typename OP::elem;
  const int64_t rows = (int64_t)c.nseq * c.heads;
  const int chunk = decode_chunk(rows, c.t);
  const int nchunk = (int)cdiv(c.t, chunk);
  if (nchunk > DEC_FIN_MAXPARTS) return SA_ERR_ARGUMENT;
  // workspace: maxima, sums (rows * nchunk each, padded to 4) and outputs (rows * nchunk * D) of the
  // partials, then the updated selection rows
  const int64_t np = align_up(rows * nchunk, 4);
  float* pm = static_cast<float*>(c.ws);
  float* pl = pm + np;
  float* po = pl + np;
  float* next_state = pm + decode_partials_floats(c.nseq, c.heads, c.t, D);
  dim3 g1((unsigned)nchunk, (unsigned)rows);
  {
    TimedLaunch timed(c.timed ? SA_KERNEL_DECODE : -1, c.st);
    hipLaunchKernelGGL((decode_partial_kernel<elem, D>), g1, dim3(NTHREADS), 0, c.st, static_cast<const elem*>(c.q),
                       static_cast<const elem*>(c.k), static_cast<const elem*>(c.v), c.selected, c.state_ld, pm, pl,
                       po, next_state, c.heads, c.groups, c.t, c.kvs, c.exempt, c.scale, chunk, nchunk);
  }
  const int sblocks = (int)cdiv(c.t, 4 * NTHREADS);
  const int64_t nblocks = rows + (int64_t)c.nseq * c.groups * sblocks;
  hipLaunchKernelGGL((decode_finish_kernel<D>), dim3((unsigned)nblocks), dim3(NTHREADS), 0, c.st, pm, pl, po, c.out,
                     nchunk, (int)rows, c.selected, next_state, c.state_ld, c.t, c.exempt, sblocks);
  return launch_status();
}

template <class OP>
int decode_entry(const DecCall& c) {
  if (c.head_dim == 32) return decode_impl<OP, 32>(c);
  if (c.head_dim == 64) return decode_impl<OP, 64>(c);
  return decode_impl<OP, 128>(c);
}

template <class OP>
int forward_entry(const FwdCall& c) {
  if (c.head_dim == 32) return forward_impl<OP, 32>(c);
  if (c.head_dim == 64) return forward_impl<OP, 64>(c);
  return forward_impl<OP, 128>(c);
}

template <class OP>
int backward_entry(const BwdCall& c) {
  if (c.head_dim == 32) return backward_impl<OP, 32>(c);
  if (c.head_dim == 64) return backward_impl<OP, 64>(c);
  return backward_impl<OP, 128>(c);
}

}  // namespace
