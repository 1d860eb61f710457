// Reductions and fused row ops (ops/reduce.cl semantics):
//   TOP_RED_PART / TOP_RED_COMB  two-phase flat reduce (reduce.cl:90-153, 529-549)
//   TOP_RED_SEG                  per-row reduce, GEMV dot mode (reduce.cl:165-281)
//   TOP_RED_STRIDED              reduce over an interior axis (reduce.cl:488-527)
//   TOP_SOFTMAX_SEG              row softmax (reduce.cl:304-392)
//   TOP_LAYERNORM_SEG            row layernorm (reduce.cl:399-479) + the affine /
//                                tanh-GELU / output-convert extension flags
//   TOP_ARGMAX_SEG               (value, first index) of the row maximum
// Float reductions accumulate in f32 through DPP wave reductions; integer ones are
// exact.  Kinds: 0 sum, 1 max, 2 min, 3 prod, 4 and, 5 or, 6 xor.
#pragma once
#include <type_traits>

#include "vm_math.h"

namespace vm {

// LDS-only block barrier: orders LDS traffic between the waves of the block
// without waiting for outstanding global loads (prefetches stay in flight).
VM_DEV void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

VM_DEV float* lds_f32() { return lds_ptr<float>(); }

template <class Op>
VM_DEV float block_reduce(float x, Op op, float* red) {
  const float w = wave_reduce(x, op);
  lds_barrier();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = w;
  lds_barrier();
  float r = red[0];
#pragma unroll
  for (int k = 1; k < kWaves; ++k) r = op(r, red[k]);
  return r;
}

VM_DEV float fred_ident(uint32_t kind) {
  return kind == 0 ? 0.0f : kind == 1 ? -INFINITY : kind == 2 ? INFINITY : 1.0f;
}
VM_DEV float fred(uint32_t kind, float a, float b) {
  return kind == 0 ? a + b : kind == 1 ? fmaxf(a, b) : kind == 2 ? fminf(a, b) : a * b;
}
VM_DEV float block_reduce_kind(float x, uint32_t kind, float* red) {
  switch (kind) {
    case 0: return block_reduce(x, OpSum(), red);
    case 1: return block_reduce(x, OpMax(), red);
    case 2: return block_reduce(x, OpMin(), red);
    default: return block_reduce(x, OpProd(), red);
  }
}

// ---- integer kinds (reduce.cl:16-40; u32 compares unsigned) -----------------------------
template <typename T>
VM_DEV T ired_ident(uint32_t kind, bool uns) {
  constexpr bool k64 = sizeof(T) == 8;
  switch (kind) {
    case 0: return 0;
    case 1: return uns ? T(0) : (k64 ? T(INT64_MIN) : T(INT32_MIN));
    case 2: return uns ? T(~T(0)) : (k64 ? T(INT64_MAX) : T(INT32_MAX));
    case 3: return 1;
    case 4: return T(~T(0));
    default: return 0;
  }
}
template <typename T, typename U>
VM_DEV T ired(uint32_t kind, bool uns, T a, T b) {
  switch (kind) {
    case 0: return T(U(a) + U(b));
    case 1: return uns ? (U(a) > U(b) ? a : b) : (a > b ? a : b);
    case 2: return uns ? (U(a) < U(b) ? a : b) : (a < b ? a : b);
    case 3: return T(U(a) * U(b));
    case 4: return a & b;
    case 5: return a | b;
    default: return a ^ b;
  }
}

// Block reduction of an integer value through an LDS tree (exact).
template <typename T, typename U>
VM_DEV T block_ireduce(T v, uint32_t kind, bool uns) {
  T* tree = lds_ptr<T>();
  lds_barrier();
  tree[threadIdx.x] = v;
  lds_barrier();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if (int(threadIdx.x) < s) tree[threadIdx.x] = ired<T, U>(kind, uns, tree[threadIdx.x], tree[threadIdx.x + s]);
    lds_barrier();
  }
  return tree[0];
}

VM_DEV int64_t load_i(const gbyte* p, uint32_t dt, uint64_t i) {
  switch (dt) {
    case DT_I64: return gcast<int64_t>(p)[i];
    case DT_U32: return int64_t(gcast<uint32_t>(p)[i]);
    case DT_BOOL: return p[i] != 0;
    default: return gcast<int32_t>(p)[i];
  }
}
VM_DEV void store_i(gbyte* p, uint32_t dt, uint64_t i, int64_t v) {
  switch (dt) {
    case DT_I64: gcast<int64_t>(p)[i] = v; break;
    case DT_BOOL: p[i] = uint8_t(v & 1); break;
    default: gcast<uint32_t>(p)[i] = uint32_t(uint64_t(v)); break;
  }
}
VM_DEV bool is_int_dt(uint32_t dt) { return dt == DT_I32 || dt == DT_U32 || dt == DT_I64 || dt == DT_BOOL; }

// Integer reduction of src[i0, i1) by the whole block.
VM_DEV int64_t block_int_range(const gbyte* src, uint32_t dt, uint32_t kind, uint64_t i0, uint64_t i1) {
  if (dt == DT_I64) {
    int64_t acc = ired_ident<int64_t>(kind, false);
    for (uint64_t i = i0 + threadIdx.x; i < i1; i += kBlock)
      acc = ired<int64_t, uint64_t>(kind, false, acc, load_i(src, dt, i));
    return block_ireduce<int64_t, uint64_t>(acc, kind, false);
  }
  const bool uns = dt == DT_U32;
  int32_t acc = ired_ident<int32_t>(kind, uns);
  if (dt == DT_BOOL && kind == 1) acc = 0;       // bool max identity is false
  if (dt == DT_BOOL && kind == 2) acc = 1;       // bool min identity is true
  for (uint64_t i = i0 + threadIdx.x; i < i1; i += kBlock)
    acc = ired<int32_t, uint32_t>(kind, uns, acc, int32_t(load_i(src, dt, i)));
  return int64_t(uint32_t(block_ireduce<int32_t, uint32_t>(acc, kind, uns)));
}

// ---- TOP_RED_PART / TOP_RED_COMB -----------------------------------------------------
// RED_PART: p0 n, p1 chunk, p2 kind; tile k reduces [k*chunk, (k+1)*chunk) into dst[k].
// RED_COMB: p0 n_parts, p1 kind; one tile reduces the partials into dst[0].
VM_TILE void red_flat_tiles(Args A, uint32_t ti, uint32_t lo, uint32_t hi, bool comb) {
  A = uargs(A);
  const VM_K Task& t = task_of(A, ti);
  const uint32_t n = t.p[0], chunk = comb ? t.p[0] : t.p[1], kind = comb ? t.p[1] : t.p[2];
  const uint32_t dt = (t.tile_op >> 8) & 0xFF;
  const gbyte* a = resolve(A, t.a);
  gbyte* d = resolve(A, t.dst);
  if (comb) hi = min(hi, 1u);
  for (uint32_t tile = lo; tile < hi; ++tile) {
    const uint64_t s0 = uint64_t(tile) * chunk, s1 = min(s0 + chunk, uint64_t(n));
    if (is_int_dt(dt)) {
      const int64_t r = block_int_range(a, dt, kind, s0, s1);
      if (threadIdx.x == 0) store_i(d, dt, tile, r);
    } else {
      float acc = fred_ident(kind);
      for (uint64_t i = s0 + threadIdx.x; i < s1; i += kBlock) acc = fred(kind, acc, load_f(a, dt, i));
      const float r = block_reduce_kind(acc, kind, lds_f32());
      if (threadIdx.x == 0) store_f(d, dt, tile, r);
    }
  }
}

// ---- TOP_RED_SEG -----------------------------------------------------------------------
// p0 n_out, p1 seg, p2 kind, p3 dot mode (row . vector at b, GEMV routing).
VM_TILE void red_seg_tiles(Args A, uint32_t ti, uint32_t lo, uint32_t hi) {
  A = uargs(A);
  const VM_K Task& t = task_of(A, ti);
  const uint32_t n_out = t.p[0], seg = t.p[1], kind = t.p[2], dot = t.p[3];
  const uint32_t dt = (t.tile_op >> 8) & 0xFF, adt = (t.tile_op >> 16) & 0xFF;
  const gbyte* a = resolve(A, t.a);
  const gbyte* bv = resolve(A, t.b);
  gbyte* d = resolve(A, t.dst);
  hi = min(hi, n_out);
  if (is_int_dt(dt) && !dot) {
    for (uint32_t o = lo; o < hi; ++o) {
      const int64_t r = block_int_range(a, dt, kind, uint64_t(o) * seg, uint64_t(o + 1) * seg);
      if (threadIdx.x == 0) store_i(d, dt, o, r);
    }
    return;
  }
  if (seg <= 32 && !dot) {             // short rows: one thread per row
    for (uint32_t o = lo + threadIdx.x; o < hi; o += kBlock) {
      float acc = fred_ident(kind);
      for (uint32_t j = 0; j < seg; ++j) acc = fred(kind, acc, load_f(a, adt, uint64_t(o) * seg + j));
      store_f(d, dt, o, acc);
    }
    return;
  }
  float* red = lds_f32();
  const bool vec = adt == DT_F32 && (seg & 3) == 0 && ((uintptr_t(a) | uintptr_t(bv)) & 15) == 0;
  for (uint32_t o = lo; o < hi; ++o) {
    const uint64_t base = uint64_t(o) * seg;
    float acc = dot ? 0.0f : fred_ident(kind);
    if (vec) {
      const VM_G v4f* r4 = (const VM_G v4f*)(gcast<float>(a) + base);
      const VM_G v4f* v4 = (const VM_G v4f*)gcast<float>(bv);
      for (uint32_t j = threadIdx.x; j < (seg >> 2); j += kBlock) {
        const v4f x = r4[j];
        if (dot) {
          const v4f y = v4[j];
          acc = fmaf(x.x, y.x, fmaf(x.y, y.y, fmaf(x.z, y.z, fmaf(x.w, y.w, acc))));
        } else {
          acc = fred(kind, acc, fred(kind, fred(kind, x.x, x.y), fred(kind, x.z, x.w)));
        }
      }
    } else {
      for (uint32_t j = threadIdx.x; j < seg; j += kBlock) {
        const float x = load_f(a, adt, base + j);
        acc = dot ? fmaf(x, load_f(bv, adt, j), acc) : fred(kind, acc, x);
      }
    }
    const float r = block_reduce_kind(acc, dot ? 0u : kind, red);
    if (threadIdx.x == 0) store_f(d, dt, o, r);
  }
}

// ---- TOP_RED_STRIDED ----------------------------------------------------------------------
// out[o*inner + i] = reduce_r in[(o*red + r)*inner + i]; p0 n_out, p1 red, p2 inner,
// p3 kind.  p4 = 0: tiles of ew_ts outputs.  p4 = S > 0 (extension, float types):
// tile t is split t % S of the 64 outputs at 64 (t / S), over its share of the
// rows; the split that arrives last at the block's counter in the task's scratch
// adds the S partials in split order ([block][S][64] floats, then a counter per
// block; agent-scope atomics, which go to memory past the XCD's L2).
//
// A block of 64 outputs is read by all 256 threads: 16 bytes (one element where
// inner or the base forbids it) of 16 (4) rows at a time, eight steps in flight, the
// row phases added through LDS in a fixed order.  One thread per output and one
// load at a time left a CU with 1 KiB in flight, and put a column sum of 8192 x 4096
// f32, a tile, on one CU: 41.4 ms; now 30.4 us (4.4 TB/s, what bounds it).  1024 x
// 2048 and 1024 x 256 f32 in the gradient step of an MLP: 3029 -> 440 us for the step.
constexpr uint32_t kRedCols = 64, kRedBatch = 8;

template <class Op, bool VEC>
VM_DEV float red_cols_block(Op op, float ident, const gbyte* a, uint32_t adt, uint32_t q0, uint32_t n_out, uint32_t red,
                            uint32_t inner, uint32_t r0, uint32_t r1) {
  constexpr uint32_t W = VEC ? 4 : 1, G = kRedCols / W, PH = kBlock / G;    // columns per thread, threads and rows per step
  float* lds = lds_f32();
  const uint32_t cg = threadIdx.x % G, ph = threadIdx.x / G;
  const uint32_t q = min(q0 + W * cg, n_out - W), o = q / inner;
  const uint64_t base = uint64_t(o) * red * inner + (q - o * inner);
  float acc[W];
#pragma unroll
  for (uint32_t w = 0; w < W; ++w) acc[w] = ident;
  for (uint32_t rb = r0; rb < r1; rb += PH * kRedBatch) {
    float x[kRedBatch][W];
#pragma unroll
    for (uint32_t u = 0; u < kRedBatch; ++u) {           // rows past r1 re-read the last one and are not added
      const uint64_t e = base + uint64_t(min(rb + ph + PH * u, r1 - 1)) * inner;
      if constexpr (VEC) {
        const v4f v = ld4(a, adt, e);
        x[u][0] = v.x; x[u][1] = v.y; x[u][2] = v.z; x[u][3] = v.w;
      } else {
        x[u][0] = load_f(a, adt, e);
      }
    }
#pragma unroll
    for (uint32_t u = 0; u < kRedBatch; ++u)
#pragma unroll
      for (uint32_t w = 0; w < W; ++w) acc[w] = rb + ph + PH * u < r1 ? op(acc[w], x[u][w]) : acc[w];
  }
  lds_barrier();
#pragma unroll
  for (uint32_t w = 0; w < W; ++w) lds[ph * (kRedCols + 4) + W * cg + w] = acc[w];
  lds_barrier();
  float r = ident;
  if (threadIdx.x < kRedCols)
#pragma unroll
    for (uint32_t p = 0; p < PH; ++p) r = op(r, lds[p * (kRedCols + 4) + threadIdx.x]);
  return r;                                              // threads 0..63: output q0 + threadIdx.x
}

// Outputs [q0, q1) over a short axis: one (VEC: four) per thread, eight loads in
// flight, no LDS.  A block of 64 outputs costs a round trip, an LDS pass and two
// barriers however few rows it has; here 1024 (256) outputs share a round trip per
// eight rows, single elements of up to four rows two for J = 4 groups of 256 outputs.
// Taken where a lane's blocks take no more round trips so (red_cols_tiles).  Whole
// launches on MI355X, us (blocks of 64 / one output per thread and one load at a time
// / this): 1M outputs f32 over 2 rows 75.6 / 14.9 / 7.2, 8 rows 77.3 / 48.3 / 10.6, 32
// rows 78.9 / 176 / 25.5, bf16 8 rows 111 / 43.5 / 10.7; 1000003 outputs over 2 rows 92 /
// 14.9 / 11.6, 8 rows 91 / 48.9 / 28; 512 x 8 x 4096 f32 over the 8 150 / 97 / 19.
// The stores are one 16-byte one or a rolled loop: unrolled, with a form more, the
// leaf was 129 KB, a short branch's reach (and 1M over 8 11.3, bf16 12.0).
template <uint32_t J, uint32_t W>
VM_DEV float pick(const float (&v)[J][W], uint32_t i) {      // v[i / W][i % W], from registers
  float r = v[0][0];
#pragma unroll
  for (uint32_t k = 1; k < J * W; ++k) r = i == k ? v[k / W][k % W] : r;
  return r;
}
template <class Op, bool VEC, uint32_t J>
VM_DEV void red_cols_short(Op op, float ident, const gbyte* a, uint32_t adt, gbyte* d, uint32_t dt, uint32_t q0,
                           uint32_t q1, uint32_t red, uint32_t inner) {
  constexpr uint32_t W = VEC ? 4 : 1, R = kRedBatch / J;
  for (uint32_t qb = q0 + W * threadIdx.x; qb < q1; qb += W * J * kBlock) {
    uint64_t base[J];
    float acc[J][W];
#pragma unroll
    for (uint32_t j = 0; j < J; ++j) {
      const uint32_t q = J == 1 ? qb : min(qb + W * j * kBlock, q1 - W), o = q / inner;    // past q1: read again, not stored
      base[j] = uint64_t(o) * red * inner + (q - o * inner);
#pragma unroll
      for (uint32_t w = 0; w < W; ++w) acc[j][w] = ident;
    }
    for (uint32_t rb = 0; rb < red; rb += R) {
      float x[R][J][W];
#pragma unroll
      for (uint32_t u = 0; u < R; ++u) {
        if (rb + u >= red) break;
#pragma unroll
        for (uint32_t j = 0; j < J; ++j) {
          const uint64_t e = base[j] + uint64_t(rb + u) * inner;
          if constexpr (VEC) {
            const v4f v = ld4(a, adt, e);
            x[u][j][0] = v.x; x[u][j][1] = v.y; x[u][j][2] = v.z; x[u][j][3] = v.w;
          } else {
            x[u][j][0] = load_f(a, adt, e);
          }
        }
      }
#pragma unroll
      for (uint32_t u = 0; u < R; ++u) {
        if (rb + u >= red) break;
#pragma unroll
        for (uint32_t j = 0; j < J; ++j)
#pragma unroll
          for (uint32_t w = 0; w < W; ++w) acc[j][w] = op(acc[j][w], x[u][j][w]);
      }
    }
    if constexpr (VEC) {
      if ((uintptr_t(d) & 15) == 0 && (dt == DT_F32 || dt == DT_BF16 || dt == DT_F16)) {
        st4(d, dt, qb, v4f_make(acc[0][0], acc[0][1], acc[0][2], acc[0][3]));
        continue;
      }
    }
#pragma unroll 1
    for (uint32_t j = 0; j < J * W; ++j) {
      const float v = pick(acc, j);
      const uint32_t q = VEC ? qb + j : qb + j * kBlock;
      if (q < q1) store_f(d, dt, q, v);
    }
  }
}

template <class Op>
VM_DEV void red_cols_tiles(Args A, uint32_t ti, uint32_t lo, uint32_t hi, Op op, float ident) {
  const VM_K Task& t = task_of(A, ti);
  const uint32_t n_out = t.p[0], red = t.p[1], inner = t.p[2], S = max(1u, t.p[4]);
  const uint32_t dt = (t.tile_op >> 8) & 0xFF, adt = (t.tile_op >> 16) & 0xFF;
  const gbyte* a = resolve(A, t.a);
  gbyte* d = resolve(A, t.dst);
  const uint32_t blocks = (n_out + kRedCols - 1) / kRedCols;
  if (!t.p[4]) {
    lo *= A->ew_ts / kRedCols;
    hi *= A->ew_ts / kRedCols;
  }
  hi = min(hi, blocks * S);
  const bool vec = (adt == DT_F32 || adt == DT_BF16 || adt == DT_F16) && inner % 4 == 0 && (uintptr_t(a) & 15) == 0;
  // 16 blocks (4: single elements) of a lane share red_cols_short's round trips, one
  // per eight rows; the same form for every lane of the task.  One block per lane is
  // one round trip either way (775 x 4 bf16 in single elements 5.5 us, 6.9 without LDS).
  const uint32_t per = min(vec ? 16u : 4u, blocks / A->n_lanes);
  if (S == 1 && blocks > A->n_lanes && red <= kRedBatch * per) {
    const uint32_t q0 = lo * kRedCols, q1 = min(hi * kRedCols, n_out);
    if (vec) red_cols_short<Op, true, 1>(op, ident, a, adt, d, dt, q0, q1, red, inner);
    else if (red <= 4) red_cols_short<Op, false, 4>(op, ident, a, adt, d, dt, q0, q1, red, inner);
    else red_cols_short<Op, false, 1>(op, ident, a, adt, d, dt, q0, q1, red, inner);
    return;
  }
  const uint32_t share = (red + S - 1) / S;
  for (uint32_t tile = lo; tile < hi; ++tile) {
    const uint32_t blk = tile / S, split = tile % S, q0 = blk * kRedCols;
    const uint32_t r0 = min(split * share, red), r1 = min(r0 + share, red);
    const float r = vec ? red_cols_block<Op, true>(op, ident, a, adt, q0, n_out, red, inner, r0, r1)
                        : red_cols_block<Op, false>(op, ident, a, adt, q0, n_out, red, inner, r0, r1);
    const bool out = threadIdx.x < kRedCols && q0 + threadIdx.x < n_out;
    if (S == 1) {
      if (out) store_f(d, dt, q0 + threadIdx.x, r);
      continue;
    }
    if (threadIdx.x >= kRedCols) continue;               // the rest is wave 0's
    uint32_t* sp = reinterpret_cast<uint32_t*>(A->scratch + A->task_scratch[ti]);
    uint32_t* arrivals = sp + uint64_t(blocks) * S * kRedCols;
    uint32_t* part = sp + uint64_t(blk) * S * kRedCols + threadIdx.x;
    __hip_atomic_store(part + split * kRedCols, __float_as_uint(r), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0x0F70);                  // vmcnt(0): the wave's partials are in memory
    uint32_t before = 0;
    if (threadIdx.x == 0)
      before = __hip_atomic_fetch_add(arrivals + blk, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    if (uni(before) != S - 1) continue;
    if (threadIdx.x == 0) __hip_atomic_store(arrivals + blk, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    float sum = ident;
    for (uint32_t s0 = 0; s0 < S; s0 += kRedBatch) {
      float x[kRedBatch];
#pragma unroll
      for (uint32_t u = 0; u < kRedBatch; ++u)
        x[u] = __uint_as_float(__hip_atomic_load(part + min(s0 + u, S - 1) * kRedCols, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT));
#pragma unroll
      for (uint32_t u = 0; u < kRedBatch; ++u) sum = s0 + u < S ? op(sum, x[u]) : sum;
    }
    if (out) store_f(d, dt, q0 + threadIdx.x, sum);
  }
}

VM_TILE void red_strided_tiles(Args A, uint32_t ti, uint32_t lo, uint32_t hi) {
  A = uargs(A);
  lo = uni(lo);
  hi = uni(hi);
  const VM_K Task& t = task_of(A, ti);
  const uint32_t n_out = t.p[0], red = t.p[1], inner = t.p[2], kind = t.p[3];
  const uint32_t dt = (t.tile_op >> 8) & 0xFF;
  if (!is_int_dt(dt) && n_out > 0 && red > 0) {
    switch (kind) {
      case 0: return red_cols_tiles(A, ti, lo, hi, OpSum(), 0.0f);
      case 1: return red_cols_tiles(A, ti, lo, hi, OpMax(), -INFINITY);
      case 2: return red_cols_tiles(A, ti, lo, hi, OpMin(), INFINITY);
      default: return red_cols_tiles(A, ti, lo, hi, OpProd(), 1.0f);
    }
  }
  const uint32_t adt = (t.tile_op >> 16) & 0xFF;
  const gbyte* a = resolve(A, t.a);
  gbyte* d = resolve(A, t.dst);
  const uint64_t e0 = uint64_t(lo) * A->ew_ts, e1 = min(uint64_t(hi) * A->ew_ts, uint64_t(n_out));
  for (uint64_t q = e0 + threadIdx.x; q < e1; q += kBlock) {
    const uint64_t o = q / inner, i = q % inner;
    const uint64_t base = o * uint64_t(red) * inner + i;
    if (is_int_dt(dt)) {
      if (dt == DT_I64) {
        int64_t acc = ired_ident<int64_t>(kind, false);
        for (uint32_t r = 0; r < red; ++r)
          acc = ired<int64_t, uint64_t>(kind, false, acc, load_i(a, dt, base + uint64_t(r) * inner));
        store_i(d, dt, q, acc);
      } else {
        const bool uns = dt == DT_U32;
        int32_t acc = ired_ident<int32_t>(kind, uns);
        if (dt == DT_BOOL && kind == 1) acc = 0;
        if (dt == DT_BOOL && kind == 2) acc = 1;
        for (uint32_t r = 0; r < red; ++r)
          acc = ired<int32_t, uint32_t>(kind, uns, acc, int32_t(load_i(a, dt, base + uint64_t(r) * inner)));
        store_i(d, dt, q, int64_t(uint32_t(acc)));
      }
    } else {
      float acc = fred_ident(kind);
      for (uint32_t r = 0; r < red; ++r) acc = fred(kind, acc, load_f(a, adt, base + uint64_t(r) * inner));
      store_f(d, dt, q, acc);
    }
  }
}

// ---- row-resident fused ops -------------------------------------------------------------
// A row of `seg` elements is held in registers, so it costs one HBM read and one
// write.  The next row's loads are issued before the current row's reductions.

// Wave-per-row layernorm, specialised on the input / output formats.  Each wave64
// owns every fourth row of the lane's range and holds a row as NV groups of 4
// elements per thread (thread t: groups t, t+64, ...; f32 rows as float4, bf16 rows
// packed two per register).  Rows stream through three rotating register buffers,
// so two rows are in flight while the third is reduced (DPP only, no block
// barriers) and written.  gamma / beta (1 / 0 when the op has no affine) are staged
// once into LDS.
template <bool BF16>
struct RowFmt {
  typedef v4f Raw;                       // f32: 4 elements in a float4
  static VM_DEV v4f unpack(Raw r) { return r; }
};
template <>
struct RowFmt<true> {
  typedef v2u Raw;                       // bf16: 4 elements in two registers
  static VM_DEV v4f unpack(Raw r) {
    return v4f_make(__uint_as_float(r.x << 16), __uint_as_float(r.x & 0xFFFF0000u), __uint_as_float(r.y << 16),
                    __uint_as_float(r.y & 0xFFFF0000u));
  }
};

struct LnRow {                 // per-row constants of one layernorm task
  const gbyte* a;
  gbyte* d;
  const v4f* lg;
  const v4f* lb;
  uint32_t seg, nv4, lane;
  uint32_t ichunk, istride;      // row interleave: row i -> (i % ichunk) * istride + i / ichunk
  float eps, inv_n;
  bool two_pass;
};

// Loads are never predicated: a load inside an exec-masked block makes the
// compiler drain every outstanding load (s_waitcnt vmcnt(0)) at the block
// boundary, which would serialise the row prefetch.  Groups past the row end
// re-read the row's last group and are masked out of the sums and stores.
// The rows are read once, so the loads are non-temporal (streaming): C2 with
// every step reading HBM (three rotating sets), alternating runs on one
// MI355X: 42.3 against 45.7-46.3 us; one set left in the memory-side cache
// then runs at about the same 41 us instead of 39.
template <int NV, bool IN_BF16, bool FULL>
VM_DEV void ln_load(typename RowFmt<IN_BF16>::Raw (&buf)[NV], const LnRow& L, uint32_t r) {
  typedef typename RowFmt<IN_BF16>::Raw Raw;
  r = (r % L.ichunk) * L.istride + r / L.ichunk;
  const VM_G Raw* rp = (const VM_G Raw*)(L.a + uint64_t(r) * L.seg * (IN_BF16 ? 2 : 4));
#pragma unroll
  for (int k = 0; k < NV; ++k)
    buf[k] = __builtin_nontemporal_load(&rp[FULL ? L.lane + 64 * k : min(L.lane + 64 * k, L.nv4 - 1)]);
}

template <int NV, bool IN_BF16, bool OUT_BF16, bool GELU, bool FULL>
VM_DEV void ln_process(const typename RowFmt<IN_BF16>::Raw (&buf)[NV], const LnRow& L, uint32_t r) {
  float s = 0.0f, s2 = 0.0f;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const bool valid = FULL || L.lane + 64 * k < L.nv4;
    const v4f x = RowFmt<IN_BF16>::unpack(buf[k]);
    const float ps = (x.x + x.y) + (x.z + x.w);
    s += valid ? ps : 0.0f;
    if (!L.two_pass) {
      const float p2 = fmaf(x.x, x.x, fmaf(x.y, x.y, fmaf(x.z, x.z, x.w * x.w)));
      s2 += valid ? p2 : 0.0f;
    }
  }
  const float mean = wave_sum(s) * L.inv_n;
  float var;
  if (L.two_pass) {
    float q2 = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const bool valid = FULL || L.lane + 64 * k < L.nv4;
      const v4f dv = RowFmt<IN_BF16>::unpack(buf[k]) - mean;
      const float p2 = fmaf(dv.x, dv.x, fmaf(dv.y, dv.y, fmaf(dv.z, dv.z, dv.w * dv.w)));
      q2 += valid ? p2 : 0.0f;
    }
    var = wave_sum(q2) * L.inv_n;
  } else {
    var = wave_sum(s2) * L.inv_n - mean * mean;
  }
  const float rstd = rsqrtf(var + L.eps);
  const float shift = -mean * rstd;
  r = (r % L.ichunk) * L.istride + r / L.ichunk;
  gbyte* rowd = L.d + uint64_t(r) * L.seg * (OUT_BF16 ? 2 : 4);
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    // one group at a time: keeps the GELU temporaries of 4 elements live, not 64
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t q = FULL ? L.lane + 64 * k : min(L.lane + 64 * k, L.nv4 - 1);
    {
      const v4f x = RowFmt<IN_BF16>::unpack(buf[k]);
      const v4f gg = L.lg[q], bb = L.lb[q];
      v4f z;
      z.x = fmaf(fmaf(x.x, rstd, shift), gg.x, bb.x);
      z.y = fmaf(fmaf(x.y, rstd, shift), gg.y, bb.y);
      z.z = fmaf(fmaf(x.z, rstd, shift), gg.z, bb.z);
      z.w = fmaf(fmaf(x.w, rstd, shift), gg.w, bb.w);
      if constexpr (GELU) {
        z.x = gelu(z.x);
        z.y = gelu(z.y);
        z.z = gelu(z.z);
        z.w = gelu(z.w);
      }
      if (FULL || L.lane + 64 * k < L.nv4) {
        // streaming stores: the rows are not read again by this launch (C2,
        // alternating runs: 38.2 against 38.7 us; streaming loads were slower)
        if constexpr (OUT_BF16)
          __builtin_nontemporal_store(v2u_make(pack_bf16x2(z.x, z.y), pack_bf16x2(z.z, z.w)), &((VM_G v2u*)rowd)[q]);
        else
          __builtin_nontemporal_store(z, &((VM_G v4f*)rowd)[q]);
      }
    }
  }
}

// Rows i = 0..mine-1 of this wave (row rbase + 4i) through rotating register
// buffers: while one row is reduced and written, the next one or two are in
// flight.  The prefetch is unconditional (past the last row it re-reads the last
// row) so no load sits behind a branch; `mine` is wave-uniform, so the loop exits
// are scalar branches.
template <int NV, bool IN_BF16, bool OUT_BF16, bool GELU, bool FULL>
VM_DEV void ln_stream(const LnRow& L, uint32_t rbase, uint32_t mine) {
  typedef typename RowFmt<IN_BF16>::Raw Raw;
  if (mine == 0) return;
  const uint32_t lastr = rbase + kWaves * (mine - 1);
  if constexpr (NV * sizeof(Raw) / 4 > 32) {
    // a row larger than 32 registers: two buffers (one row in flight)
    Raw b0[NV], b1[NV];
    ln_load<NV, IN_BF16, FULL>(b0, L, rbase);
    for (uint32_t i = 0; i < mine; i += 2) {
      const uint32_t r = rbase + kWaves * i;
      ln_load<NV, IN_BF16, FULL>(b1, L, min(r + kWaves, lastr));
      ln_process<NV, IN_BF16, OUT_BF16, GELU, FULL>(b0, L, r);
      if (i + 1 >= mine) break;
      ln_load<NV, IN_BF16, FULL>(b0, L, min(r + 2 * kWaves, lastr));
      ln_process<NV, IN_BF16, OUT_BF16, GELU, FULL>(b1, L, r + kWaves);
    }
    return;
  }
  Raw b0[NV], b1[NV], b2[NV];
  ln_load<NV, IN_BF16, FULL>(b0, L, rbase);
  ln_load<NV, IN_BF16, FULL>(b1, L, min(rbase + kWaves, lastr));
  for (uint32_t i = 0; i < mine; i += 3) {
    const uint32_t r = rbase + kWaves * i;
    ln_load<NV, IN_BF16, FULL>(b2, L, min(r + 2 * kWaves, lastr));
    ln_process<NV, IN_BF16, OUT_BF16, GELU, FULL>(b0, L, r);
    if (i + 1 >= mine) break;
    ln_load<NV, IN_BF16, FULL>(b0, L, min(r + 3 * kWaves, lastr));
    ln_process<NV, IN_BF16, OUT_BF16, GELU, FULL>(b1, L, r + kWaves);
    if (i + 2 >= mine) break;
    ln_load<NV, IN_BF16, FULL>(b1, L, min(r + 4 * kWaves, lastr));
    ln_process<NV, IN_BF16, OUT_BF16, GELU, FULL>(b2, L, r + 2 * kWaves);
  }
}

template <int NV, bool IN_BF16, bool OUT_BF16, bool FULL>
VM_DEV void ln_rows_fast(Args A, uint32_t ti, uint32_t r0, uint32_t r1) {
  A = uargs(A);
  const VM_K Task& t = task_of(A, ti);
  r0 = uni(r0);
  r1 = uni(r1);
  const uint32_t flags = t.p[3];
  const bool affine = flags & LN_AFFINE;
  LnRow L;
  L.seg = t.p[1];
  L.nv4 = L.seg >> 2;
  L.eps = __uint_as_float(t.p[2]);
  L.inv_n = 1.0f / float(L.seg);
  L.two_pass = flags & LN_TWO_PASS;
  L.a = resolve(A, t.a);
  L.d = resolve(A, t.dst);
  L.lane = threadIdx.x & 63;
  // p5: row interleave (0: none; the loader checks that it divides n_out)
  L.ichunk = t.p[5] ? t.p[5] : 0xFFFFFFFFu;
  L.istride = t.p[5] ? t.p[0] / t.p[5] : 1u;
  const uint32_t wave = uni(threadIdx.x >> 6);       // wave-uniform: scalar loop control
  v4f* lg = lds_ptr<v4f>();
  v4f* lb = lg + L.nv4;
  {
    const VM_G v4f* g4 = (const VM_G v4f*)gcast<float>(resolve(A, affine ? t.b : t.a));
    const VM_G v4f* b4 = (const VM_G v4f*)gcast<float>(resolve(A, affine ? t.p[4] : t.a));
    for (uint32_t q = threadIdx.x; q < L.nv4; q += kBlock) {
      lg[q] = affine ? g4[q] : v4f{1.0f, 1.0f, 1.0f, 1.0f};
      lb[q] = affine ? b4[q] : v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
  L.lg = lg;
  L.lb = lb;
  __syncthreads();
  const uint32_t mine = r1 > r0 + wave ? (r1 - r0 - wave + kWaves - 1) / kWaves : 0;
  if (flags & LN_GELU) ln_stream<NV, IN_BF16, OUT_BF16, true, FULL>(L, r0 + wave, mine);
  else ln_stream<NV, IN_BF16, OUT_BF16, false, FULL>(L, r0 + wave, mine);
}

// Rows in groups of 4 elements, read with 16- or 8-byte accesses that need only the
// element's own alignment, so odd row lengths stream like even ones; a row whose
// length is not a multiple of 4 ends in a group that overlaps the one before (its
// repeated elements count once in sums).
template <bool IN16>
struct RowRaw {
  typedef typename std::conditional<IN16, v2u, v4f>::type Raw;
  typedef float v4f_any __attribute__((ext_vector_type(4), aligned(4)));
  typedef uint32_t v2u_any __attribute__((ext_vector_type(2), aligned(2)));
  static VM_DEV Raw load(const gbyte* row, uint32_t e) {
    if constexpr (IN16) return *(const VM_G v2u_any*)(gcast<uint16_t>(row) + e);
    else return *(const VM_G v4f_any*)(gcast<float>(row) + e);
  }
  static VM_DEV v4f value(Raw r, bool bf) {
    if constexpr (IN16)
      return bf ? v4f_make(__uint_as_float(r.x << 16), __uint_as_float(r.x & 0xFFFF0000u), __uint_as_float(r.y << 16),
                           __uint_as_float(r.y & 0xFFFF0000u))
                : v4f_make(f16_to_f32(r.x & 0xFFFF), f16_to_f32(r.x >> 16), f16_to_f32(r.y & 0xFFFF), f16_to_f32(r.y >> 16));
    else return r;
  }
};
VM_DEV void row_store(gbyte* row, uint32_t dt, uint32_t e, v4f v) {
  typedef float v4f_any __attribute__((ext_vector_type(4), aligned(4)));
  typedef uint32_t v2u_any __attribute__((ext_vector_type(2), aligned(2)));
  if (dt == DT_F32) {
    *(VM_G v4f_any*)(gcast<float>(row) + e) = v;
  } else if (dt == DT_BF16) {
    *(VM_G v2u_any*)(gcast<uint16_t>(row) + e) = v2u_make(pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w));
  } else {
    *(VM_G v2u_any*)(gcast<uint16_t>(row) + e) = v2u_make(f32_to_f16(v.x) | (uint32_t(f32_to_f16(v.y)) << 16),
                                                          f32_to_f16(v.z) | (uint32_t(f32_to_f16(v.w)) << 16));
  }
}
// A row of seg >= 4 elements in groups of 4: group q starts at element at(q); its
// first dup(q) elements belong to the group before.
struct RowGroups {
  uint32_t seg, n;
  VM_DEV explicit RowGroups(uint32_t s) : seg(s), n((s + 3) >> 2) {}
  VM_DEV uint32_t at(uint32_t q) const { return min(4 * q, seg - 4); }
  VM_DEV uint32_t dup(uint32_t q) const { return 4 * q - at(q); }
};
VM_DEV float sum4(v4f v, uint32_t dup) {
  return (dup > 0 ? 0.0f : v.x) + (dup > 1 ? 0.0f : v.y) + ((dup > 2 ? 0.0f : v.z) + v.w);
}

// As row_store for a group read after other groups were stored: a destination that
// is the source may hold the results in its repeated elements already.
VM_DEV void row_store_own(gbyte* row, uint32_t dt, uint32_t e, v4f v, uint32_t dup) {
  if (!dup) return row_store(row, dt, e, v);
  if (dup < 2) store_f(row, dt, e + 1, v.y);
  if (dup < 3) store_f(row, dt, e + 2, v.z);
  store_f(row, dt, e + 3, v.w);
}

// Layernorm rows of any length and alignment, f16 rows, and rows past the streaming
// kernel's 4096: softmax_rows' forms (below), a row over the TH threads.
// gamma and beta stay in registers, for rows over 8192 elements they come from L2
// for every row.  Measured (MI355X, whole launches, us; before: f16 rows through
// scalar conversions and odd or long rows three times in single elements):
//   GELU, f32 -> bf16: 1000 x 777 17.5 -> 7.5, 3000 x 4097 186 -> 33, 2048 x 8192 44.8
//   -> 36.4, 100 x 30000 88 -> 29.6, 64 x 50257 164 -> 40; f16 4096 x 4096 186 -> 39.4,
//   4096 x 1024 54 -> 14.5.
// The groups a thread holds follow the row (1, 4, 8, 16 a wave, 6, 8, 32 a block):
// clamped ones are loaded and summed in vain.  With 4, 16, 8 and 32 only, f16 8656 x
// 192 took 15.6 (now 11.8, before the groups 12.0), 3439 x 192 10.2 (8.5, 8.3), 800 x
// 2048 12.0 (10.2, 10.1), bf16 1000 x 4608 19.0 (17.8, 17.5).  A row or two per lane
// still lose 3-6 % to the masks: f32 300 x 5000 10.4 -> 10.9 (11.3 with 8 groups), 256 x
// 6000 8.7 -> 9.3, f16 2000 x 768 9.1 -> 9.5.  (In leaves by register need, as softmax's,
// these take 10.2, 8.6 and 8.7, but the kernel's register saving then changes at every
// call: 0.7-1.2 us more a launch, 24.8 -> 25.5 for an MLP of two products.)
struct LnTask {
  const gbyte *a, *gp, *bp;
  gbyte* d;
  uint32_t dt, adt, ichunk, istride;
  float eps, inv_n;
  bool affine, do_gelu, two_pass;
  VM_DEV LnTask(Args A, const VM_K Task& t) {
    const uint32_t flags = t.p[3];
    a = resolve(A, t.a);
    d = resolve(A, t.dst);
    affine = flags & LN_AFFINE, do_gelu = flags & LN_GELU, two_pass = flags & LN_TWO_PASS;
    gp = resolve(A, affine ? t.b : t.a);
    bp = resolve(A, affine ? t.p[4] : t.a);
    dt = (t.tile_op >> 8) & 0xFF, adt = (t.tile_op >> 16) & 0xFF;
    eps = __uint_as_float(t.p[2]);
    inv_n = 1.0f / float(t.p[1]);
    ichunk = max(1u, t.p[5]);
    istride = t.p[0] / ichunk;
  }
  VM_DEV uint32_t row(uint32_t i) const { return (i % ichunk) * istride + i / ichunk; }     // p5, layernorm_tiles
  VM_DEV v4f out(v4f x, float rstd, float shift, v4f g, v4f b) const {
    v4f z = v4f_make(fmaf(x.x, rstd, shift), fmaf(x.y, rstd, shift), fmaf(x.z, rstd, shift), fmaf(x.w, rstd, shift));
    if (affine) z = v4f_make(fmaf(z.x, g.x, b.x), fmaf(z.y, g.y, b.y), fmaf(z.z, g.z, b.z), fmaf(z.w, g.w, b.w));
    if (do_gelu) z = v4f_make(gelu(z.x), gelu(z.y), gelu(z.z), gelu(z.w));
    return z;
  }
};
VM_DEV float sumsq4(v4f v, uint32_t dup) { return sum4(v4f_make(v.x * v.x, v.y * v.y, v.z * v.z, v.w * v.w), dup); }

template <int NV, bool IN16, int TH>
VM_DEV void ln_rows(Args A, uint32_t ti, uint32_t r0, uint32_t r1, uint32_t step) {
  typedef RowRaw<IN16> R;
  const VM_K Task& t = task_of(A, ti);
  const LnTask L(A, t);
  float* red = lds_f32();
  const RowGroups G(t.p[1]);
  const bool bf = L.adt == DT_BF16;
  const uint32_t me = TH == 64 ? threadIdx.x & 63 : threadIdx.x, dsz = L.dt == DT_F32 ? 4 : 2;
  if (r0 >= r1) return;
  typename R::Raw x[NV], xn[NV];
  auto load = [&](typename R::Raw (&buf)[NV], uint32_t i) {
    const gbyte* row = L.a + uint64_t(L.row(i)) * G.seg * (IN16 ? 2 : 4);
#pragma unroll
    for (int k = 0; k < NV; ++k) buf[k] = R::load(row, G.at(min(me + TH * k, G.n - 1)));
  };
  auto sum = [&](float v, float* p) {
    if constexpr (TH == 64) return wave_sum(v);
    else return block_reduce(v, OpSum(), p);
  };
  constexpr int U = NV <= 16 ? NV : 8;
  v4f g[U], b[U];
  auto load_gb = [&](int k0) {
    if (!L.affine) return;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t e = G.at(min(me + TH * (k0 + u), G.n - 1));
      g[u] = RowRaw<false>::load(L.gp, e);
      b[u] = RowRaw<false>::load(L.bp, e);
    }
  };
  load(x, r0);
  if (U == NV) load_gb(0);
  for (uint32_t r = r0; r < r1; r += step) {
    if (r + step < r1) load(xn, r + step);
    float s = 0.0f, s2 = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const v4f v = R::value(x[k], bf);
      const uint32_t q = me + TH * k;
      s += q < G.n ? sum4(v, G.dup(q)) : 0.0f;
      if (!L.two_pass) s2 += q < G.n ? sumsq4(v, G.dup(q)) : 0.0f;
    }
    const float mean = sum(s, red) * L.inv_n;
    if (L.two_pass) {
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        const uint32_t q = me + TH * k;
        s2 += q < G.n ? sumsq4(R::value(x[k], bf) - mean, G.dup(q)) : 0.0f;
      }
    }
    const float m2 = sum(s2, red + kWaves) * L.inv_n;
    const float rstd = rsqrtf((L.two_pass ? m2 : m2 - mean * mean) + L.eps), shift = -mean * rstd;
    gbyte* row = L.d + uint64_t(L.row(r)) * G.seg * dsz;
#pragma unroll
    for (int k0 = 0; k0 < NV; k0 += U) {
      if (U < NV) load_gb(k0);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t q = me + TH * (k0 + u);
        if (q < G.n) row_store(row, L.dt, G.at(q), L.out(R::value(x[k0 + u], bf), rstd, shift, g[u], b[u]));
      }
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) x[k] = xn[k];
  }
}

// Rows too long for the registers: the sums, (two-pass) the centred squares and the
// results each read the row, after the first time from L2 and the memory-side cache.
template <bool IN16>
VM_DEV void ln_rows_long(Args A, uint32_t ti, uint32_t r0, uint32_t r1) {
  typedef RowRaw<IN16> R;
  const VM_K Task& t = task_of(A, ti);
  const LnTask L(A, t);
  float* red = lds_f32();
  const RowGroups G(t.p[1]);
  const bool bf = L.adt == DT_BF16;
  constexpr int U = 8;
  for (uint32_t r = r0; r < r1; ++r) {
    const gbyte* src = L.a + uint64_t(L.row(r)) * G.seg * (IN16 ? 2 : 4);
    gbyte* row = L.d + uint64_t(L.row(r)) * G.seg * (L.dt == DT_F32 ? 4 : 2);
    auto each = [&](auto fn) {
      for (uint32_t q0 = threadIdx.x; q0 < G.n; q0 += U * kBlock) {
        typename R::Raw x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = R::load(src, G.at(min(q0 + u * kBlock, G.n - 1)));
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (q0 + u * kBlock < G.n) fn(q0 + u * kBlock, R::value(x[u], bf));
      }
    };
    float s = 0.0f, s2 = 0.0f;
    each([&](uint32_t q, v4f v) {
      s += sum4(v, G.dup(q));
      if (!L.two_pass) s2 += sumsq4(v, G.dup(q));
    });
    const float mean = block_reduce(s, OpSum(), red) * L.inv_n;
    if (L.two_pass) each([&](uint32_t q, v4f v) { s2 += sumsq4(v - mean, G.dup(q)); });
    const float m2 = block_reduce(s2, OpSum(), red + kWaves) * L.inv_n;
    const float rstd = rsqrtf((L.two_pass ? m2 : m2 - mean * mean) + L.eps), shift = -mean * rstd;
    each([&](uint32_t q, v4f v) {
      v4f g = v, b = v;
      if (L.affine) {
        g = RowRaw<false>::load(L.gp, G.at(q));
        b = RowRaw<false>::load(L.bp, G.at(q));
      }
      row_store_own(row, L.dt, G.at(q), L.out(v, rstd, shift, g, b), G.dup(q));
    });
  }
}

template <bool IN16>
VM_DEV void ln_dispatch(Args A, uint32_t ti, uint32_t lo, uint32_t hi) {
  const uint32_t n = (task_of(A, ti).p[1] + 3) >> 2, wave = uni(threadIdx.x >> 6);
  if (n <= 64) ln_rows<1, IN16, 64>(A, ti, lo + wave, hi, kWaves);
  else if (n <= 4 * 64) ln_rows<4, IN16, 64>(A, ti, lo + wave, hi, kWaves);
  else if (n <= 8 * 64) ln_rows<8, IN16, 64>(A, ti, lo + wave, hi, kWaves);
  else if (n <= 16 * 64) ln_rows<16, IN16, 64>(A, ti, lo + wave, hi, kWaves);
  else if (n <= 6 * kBlock) ln_rows<6, IN16, kBlock>(A, ti, lo, hi, 1);
  else if (n <= 8 * kBlock) ln_rows<8, IN16, kBlock>(A, ti, lo, hi, 1);
  else if (n <= 32 * kBlock) ln_rows<32, IN16, kBlock>(A, ti, lo, hi, 1);
  else ln_rows_long<IN16>(A, ti, lo, hi);
}

// Rows of less than four elements: single elements from global memory.
VM_DEV void ln_rows_generic(Args A, uint32_t ti, uint32_t r0, uint32_t r1) {
  A = uargs(A);
  const VM_K Task& t = task_of(A, ti);
  float* red = lds_f32();
  const uint32_t seg = t.p[1], flags = t.p[3];
  const float eps = __uint_as_float(t.p[2]);
  const uint32_t dt = (t.tile_op >> 8) & 0xFF, adt = (t.tile_op >> 16) & 0xFF;
  const gbyte* a = resolve(A, t.a);
  gbyte* d = resolve(A, t.dst);
  const bool affine = flags & LN_AFFINE, do_gelu = flags & LN_GELU, two_pass = flags & LN_TWO_PASS;
  const gbyte* gp = resolve(A, affine ? t.b : t.a);
  const gbyte* bp = resolve(A, affine ? t.p[4] : t.a);
  const float inv_n = 1.0f / float(seg);
  const uint32_t c = max(1u, t.p[5]), stride = t.p[0] / c;
  for (uint32_t i = r0; i < r1; ++i) {
    const uint64_t base = uint64_t((i % c) * stride + i / c) * seg;
    float s = 0.0f, s2 = 0.0f;
    for (uint32_t j = threadIdx.x; j < seg; j += kBlock) {
      const float v = load_f(a, adt, base + j);
      s += v;
      s2 = fmaf(v, v, s2);
    }
    const float mean = block_reduce(s, OpSum(), red) * inv_n;
    float var;
    if (two_pass) {
      float q = 0.0f;
      for (uint32_t j = threadIdx.x; j < seg; j += kBlock) {
        const float dv = load_f(a, adt, base + j) - mean;
        q = fmaf(dv, dv, q);
      }
      var = block_reduce(q, OpSum(), red + kWaves) * inv_n;
    } else {
      var = block_reduce(s2, OpSum(), red + kWaves) * inv_n - mean * mean;
    }
    const float rstd = rsqrtf(var + eps);
    const float shift = -mean * rstd;
    for (uint32_t j = threadIdx.x; j < seg; j += kBlock) {
      float z = fmaf(load_f(a, adt, base + j), rstd, shift);
      if (affine) z = fmaf(z, load_f(gp, DT_F32, j), load_f(bp, DT_F32, j));
      if (do_gelu) z = gelu(z);
      store_f(d, dt, base + j, z);
    }
  }
}

// Rows of the streaming kernel: whole aligned groups, up to 4096 elements.
VM_DEV bool row_vec_ok(uint32_t seg, const gbyte* a, const gbyte* d, uint32_t adt, uint32_t dt) {
  const bool fmt = (adt == DT_F32 || adt == DT_BF16) && (dt == DT_F32 || dt == DT_BF16);
  return fmt && (seg & 3) == 0 && seg <= 16 * 4 * 64 && ((uintptr_t(a) | uintptr_t(d)) & 15) == 0;
}

// LAYERNORM_SEG tiles [lo, hi).  Task p5 (scheduler, extension): the lanes'
// rows interleaved -- logical row i is row (i % p5) * (n_out / p5) + i / p5, so
// that at any moment the lanes stream neighbouring rows of the input (C2,
// alternating runs on one MI355X: 38.7 against 39.6 us).  Every row kernel
// applies it per row.
// A leaf with its row kernels inlined, for the reason ew_tile gives: as a
// function calling them it saved and reloaded 14 registers in scratch around
// every entry (C2, alternating runs: 41.6-41.8 against 42.2 us).
VM_LEAF void layernorm_tiles(Args A, uint32_t ti, uint32_t lo, uint32_t hi) {
  A = uargs(A);
  const VM_K Task& t = task_of(A, ti);
  const uint32_t n_out = t.p[0], nv4 = t.p[1] >> 2;
  const bool ib = ((t.tile_op >> 16) & 0xFF) == DT_BF16, ob = ((t.tile_op >> 8) & 0xFF) == DT_BF16;
  hi = min(hi, n_out);
  if (lo >= hi) return;
#define VM_LN_FAST(NVV, FULLV)                                                               \
  {                                                                                           \
    if (ib) return ob ? ln_rows_fast<NVV, true, true, FULLV>(A, ti, lo, hi)                    \
                      : ln_rows_fast<NVV, true, false, FULLV>(A, ti, lo, hi);                  \
    return ob ? ln_rows_fast<NVV, false, true, FULLV>(A, ti, lo, hi)                           \
              : ln_rows_fast<NVV, false, false, FULLV>(A, ti, lo, hi);                         \
  }
  if (nv4 == 4 * 64) VM_LN_FAST(4, true)
  if (nv4 < 4 * 64) VM_LN_FAST(4, false)
  if (nv4 == 16 * 64) VM_LN_FAST(16, true)
  VM_LN_FAST(16, false)
#undef VM_LN_FAST
}

// The other rows, in a leaf of their own: inlined into the streaming kernel's they
// cost it 2 % (8192 x 4096: 41.4 against 40.6 us).
VM_LEAF void layernorm_any(Args A, uint32_t ti, uint32_t lo, uint32_t hi) {
  A = uargs(A);
  const VM_K Task& t = task_of(A, ti);
  const uint32_t dt = (t.tile_op >> 8) & 0xFF, adt = (t.tile_op >> 16) & 0xFF;
  hi = min(hi, t.p[0]);
  if (lo >= hi) return;
  const bool in16 = adt == DT_BF16 || adt == DT_F16;
  const bool fmt = (in16 || adt == DT_F32) && (dt == DT_F32 || dt == DT_BF16 || dt == DT_F16);
  if (t.p[1] < 4 || !fmt) return ln_rows_generic(A, ti, lo, hi);
  if (in16) ln_dispatch<true>(A, ti, lo, hi);
  else ln_dispatch<false>(A, ti, lo, hi);
}

VM_DEV void layernorm_run(Args A, uint32_t ti, uint32_t lo, uint32_t hi) {
  const VM_K Task& t = task_of(A, ti);
  bool ok = row_vec_ok(t.p[1], resolve(A, t.a), resolve(A, t.dst), (t.tile_op >> 16) & 0xFF, (t.tile_op >> 8) & 0xFF);
  if (ok && (t.p[3] & LN_AFFINE)) ok = ((uintptr_t(resolve(A, t.b)) | uintptr_t(resolve(A, t.p[4]))) & 15) == 0;
  if (ok) layernorm_tiles(A, ti, lo, hi);
  else layernorm_any(A, ti, lo, hi);
}

// SOFTMAX_SEG rows: exp(x - max) / sum, f32 arithmetic.
//
// Forms, by how many registers a row takes and how many rows a lane has:
//   up to 4096 elements: a wave per row, four rows in flight per CU and the next
//     ones prefetched, DPP reductions and no block barrier;
//   up to 8192 and at most three rows a lane: softmax_rows_few;
//   up to 32768: a row over the block's registers, the next row prefetched;
//   longer: two passes over the row, the first keeping a running maximum and sum
//     per thread.
// Loads are not predicated (ln_load's reason), except in softmax_rows_few: groups
// past the row re-read its last.  Memory bounds them (MI355X, whole launches): 512 x
// 32000 f32 33.9 us (3.9 TB/s: two rows per CU, so the first row's load and the last
// one's store overlap nothing), 4096 x 4096 25.0 (5.4 TB/s), 4096 x 1001 8.9.
// Rows r0, r0 + step, ... < r1, a row over the TH threads (64: the wave; kBlock: the
// block), this thread's groups t, t + TH, ...
template <int NV, bool IN16, int TH>
VM_DEV void softmax_rows(Args A, uint32_t ti, uint32_t r0, uint32_t r1, uint32_t step) {
  typedef RowRaw<IN16> R;
  const VM_K Task& t = task_of(A, ti);
  float* red = lds_f32();
  const RowGroups G(t.p[1]);
  const uint32_t dt = (t.tile_op >> 8) & 0xFF, adt = (t.tile_op >> 16) & 0xFF;
  const bool bf = adt == DT_BF16;
  const gbyte* a = resolve(A, t.a);
  gbyte* d = resolve(A, t.dst);
  const uint32_t me = TH == 64 ? threadIdx.x & 63 : threadIdx.x;
  const uint32_t dsz = dt == DT_F32 ? 4 : 2;
  if (r0 >= r1) return;
  typename R::Raw x[NV], xn[NV];
  auto load = [&](typename R::Raw (&buf)[NV], uint32_t r) {
    const gbyte* row = a + uint64_t(r) * G.seg * (IN16 ? 2 : 4);
#pragma unroll
    for (int k = 0; k < NV; ++k) buf[k] = R::load(row, G.at(min(me + TH * k, G.n - 1)));
  };
  load(x, r0);
  for (uint32_t r = r0; r < r1; r += step) {
    load(xn, r + step < r1 ? r + step : r);
    float m = -INFINITY;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const v4f v = R::value(x[k], bf);
      m = fmaxf(m, fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w)));
    }
    if constexpr (TH == 64) m = wave_max(m);
    else m = block_reduce(m, OpMax(), red);
    v4f y[NV];
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const v4f v = R::value(x[k], bf);
      y[k] = v4f_make(__expf(v.x - m), __expf(v.y - m), __expf(v.z - m), __expf(v.w - m));
      const uint32_t q = me + TH * k;
      s += q < G.n ? sum4(y[k], G.dup(q)) : 0.0f;
    }
    if constexpr (TH == 64) s = wave_sum(s);
    else s = block_reduce(s, OpSum(), red + kWaves);
    const float inv = 1.0f / s;
    gbyte* row = d + uint64_t(r) * G.seg * dsz;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const uint32_t q = me + TH * k;
      if (q < G.n) row_store(row, dt, G.at(q), y[k] * inv);
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) x[k] = xn[k];
  }
}

// A lane's one to three rows, over the block's threads: one row's latency is what
// counts, so groups past the row are skipped (clamped ones cost four exponentials
// each), and a wave per row would leave waves idle.
template <int NV, bool IN16>
VM_DEV void softmax_rows_few(Args A, uint32_t ti, uint32_t r0, uint32_t r1) {
  typedef RowRaw<IN16> R;
  const VM_K Task& t = task_of(A, ti);
  float* red = lds_f32();
  const RowGroups G(t.p[1]);
  const uint32_t dt = (t.tile_op >> 8) & 0xFF, adt = (t.tile_op >> 16) & 0xFF;
  const bool bf = adt == DT_BF16;
  const gbyte* a = resolve(A, t.a);
  gbyte* d = resolve(A, t.dst);
  const uint32_t me = threadIdx.x, dsz = dt == DT_F32 ? 4 : 2;
  typename R::Raw x[NV], xn[NV];
  auto load = [&](typename R::Raw (&buf)[NV], uint32_t r) {
    const gbyte* row = a + uint64_t(r) * G.seg * (IN16 ? 2 : 4);
#pragma unroll
    for (int k = 0; k < NV; ++k)
      if (me + kBlock * k < G.n) buf[k] = R::load(row, G.at(me + kBlock * k));
  };
  load(x, r0);
  for (uint32_t r = r0; r < r1; ++r) {
    if (r + 1 < r1) load(xn, r + 1);
    v4f y[NV];
    float m = -INFINITY, s = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; ++k)
      if (me + kBlock * k < G.n) {
        y[k] = R::value(x[k], bf);
        m = fmaxf(m, fmaxf(fmaxf(y[k].x, y[k].y), fmaxf(y[k].z, y[k].w)));
      }
    m = block_reduce(m, OpMax(), red);
#pragma unroll
    for (int k = 0; k < NV; ++k)
      if (me + kBlock * k < G.n) {
        y[k] = v4f_make(__expf(y[k].x - m), __expf(y[k].y - m), __expf(y[k].z - m), __expf(y[k].w - m));
        s += sum4(y[k], G.dup(me + kBlock * k));
      }
    const float inv = 1.0f / block_reduce(s, OpSum(), red + kWaves);
    gbyte* row = d + uint64_t(r) * G.seg * dsz;
#pragma unroll
    for (int k = 0; k < NV; ++k)
      if (me + kBlock * k < G.n) row_store(row, dt, G.at(me + kBlock * k), y[k] * inv);
    if (r + 1 < r1)
#pragma unroll
      for (int k = 0; k < NV; ++k) x[k] = xn[k];
  }
}

// Rows too long for the registers: a running maximum and sum per thread, then a
// second read (from L2 and the memory-side cache) to store.
template <bool IN16>
VM_DEV void softmax_rows_long(Args A, uint32_t ti, uint32_t r0, uint32_t r1) {
  typedef RowRaw<IN16> R;
  const VM_K Task& t = task_of(A, ti);
  float* red = lds_f32();
  const RowGroups G(t.p[1]);
  const uint32_t dt = (t.tile_op >> 8) & 0xFF, adt = (t.tile_op >> 16) & 0xFF;
  const bool bf = adt == DT_BF16;
  constexpr int U = 8;
  for (uint32_t r = r0; r < r1; ++r) {
    const gbyte* src = resolve(A, t.a) + uint64_t(r) * G.seg * (IN16 ? 2 : 4);
    gbyte* row = resolve(A, t.dst) + uint64_t(r) * G.seg * (dt == DT_F32 ? 4 : 2);
    float m = -INFINITY, s = 0.0f;
    for (uint32_t q0 = threadIdx.x; q0 < G.n; q0 += U * kBlock) {
      typename R::Raw x[U];
#pragma unroll
      for (int u = 0; u < U; ++u) x[u] = R::load(src, G.at(min(q0 + u * kBlock, G.n - 1)));
      float nm = m;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const v4f v = R::value(x[u], bf);
        nm = fmaxf(nm, fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w)));
      }
      const float at = nm == -INFINITY ? 0.0f : nm;      // nothing but -inf so far: every term is 0
      s *= __expf(m - at);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const v4f v = R::value(x[u], bf);
        const uint32_t q = q0 + u * kBlock;
        s += q < G.n ? sum4(v4f_make(__expf(v.x - at), __expf(v.y - at), __expf(v.z - at), __expf(v.w - at)), G.dup(q)) : 0.0f;
      }
      m = nm;
    }
    const float M = block_reduce(m, OpMax(), red);
    s = block_reduce(m == -INFINITY ? 0.0f * s : s * __expf(m - M), OpSum(), red + kWaves);
    const float inv = 1.0f / s;
    for (uint32_t q0 = threadIdx.x; q0 < G.n; q0 += U * kBlock) {
      typename R::Raw x[U];
#pragma unroll
      for (int u = 0; u < U; ++u) x[u] = R::load(src, G.at(min(q0 + u * kBlock, G.n - 1)));
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const v4f v = R::value(x[u], bf);
        const uint32_t q = q0 + u * kBlock;
        if (q < G.n)
          row_store_own(row, dt, G.at(q),
                        v4f_make(__expf(v.x - M), __expf(v.y - M), __expf(v.z - M), __expf(v.w - M)) * inv, G.dup(q));
      }
    }
  }
}

// Rows of less than four elements or other types: single elements from memory.
VM_DEV void softmax_rows_generic(Args A, uint32_t ti, uint32_t lo, uint32_t hi) {
  const VM_K Task& t = task_of(A, ti);
  float* red = lds_f32();
  const uint32_t seg = t.p[1];
  const uint32_t dt = (t.tile_op >> 8) & 0xFF, adt = (t.tile_op >> 16) & 0xFF;
  const gbyte* a = resolve(A, t.a);
  gbyte* d = resolve(A, t.dst);
  for (uint32_t r = lo; r < hi; ++r) {
    const uint64_t base = uint64_t(r) * seg;
    float m = -INFINITY;
    for (uint32_t j = threadIdx.x; j < seg; j += kBlock) m = fmaxf(m, load_f(a, adt, base + j));
    m = block_reduce(m, OpMax(), red);
    float s = 0.0f;
    for (uint32_t j = threadIdx.x; j < seg; j += kBlock) s += __expf(load_f(a, adt, base + j) - m);
    s = block_reduce(s, OpSum(), red + kWaves);
    const float inv = 1.0f / s;
    for (uint32_t j = threadIdx.x; j < seg; j += kBlock) store_f(d, dt, base + j, __expf(load_f(a, adt, base + j) - m) * inv);
  }
}

// The forms in three leaves, by the registers they need: with all of them in one (135
// KB) the short ones paid for the long ones' registers and spills.  The whole-row and
// few-row rules with it, MI355X, whole launches, us (one leaf, a wave per row up to
// 4096 / a row per block / this): bf16 256 x 2304 9.2 / 5.6 / 5.2, 256 x 4096
// 9.8 / 5.9 / 5.3, 500 x 1500 9.1 / 6.2 / 5.7, 256 x 6000 8.0 / 6.8 / 6.7; f32 256 x 1500
// 7.5 / 5.2 / 5.3, 500 x 4096 8.9 / 7.7 / 7.5, 4096 x 48 7.5 / 14.8 / 5.5.  (Each form a
// leaf, ten calls in the kernel: the same, but 25.4 against 24.8 for an MLP of two
// products, whose code the calls push apart.  One function that calls them: 20-45 us
// an entry, saving what they clobber.)
enum SoftmaxForm : uint32_t {
  SM_WAVE1, SM_WAVE4, SM_FEW2, SM_FEW4,           // softmax_short
  SM_FEW8, SM_WAVE16, SM_BLOCK8,                  // softmax_mid
  SM_BLOCK32, SM_LONG, SM_ELEM                    // softmax_long
};
// By the task's rows per lane, not the entry's: one form for all rows of a task.
VM_DEV uint32_t softmax_form(Args A, const VM_K Task& t) {
  const uint32_t n = (t.p[1] + 3) >> 2, rows = (t.p[0] - 1) / A->n_lanes + 1;
  const uint32_t dt = (t.tile_op >> 8) & 0xFF, adt = (t.tile_op >> 16) & 0xFF;
  const bool fmt = (dt == DT_F32 || dt == DT_BF16 || dt == DT_F16) && (adt == DT_F32 || adt == DT_BF16 || adt == DT_F16);
  if (!fmt || t.p[1] < 4) return SM_ELEM;
  if (n <= 64) return SM_WAVE1;
  if (n <= 8 * kBlock && rows <= (n <= kBlock ? 2u : 3u)) return n <= 2 * kBlock ? SM_FEW2 : n <= 4 * kBlock ? SM_FEW4 : SM_FEW8;
  return n <= 4 * 64 ? SM_WAVE4 : n <= 16 * 64 ? SM_WAVE16 : n <= 8 * kBlock ? SM_BLOCK8 : n <= 32 * kBlock ? SM_BLOCK32 : SM_LONG;
}

template <bool IN16>
VM_DEV void softmax_short_rows(Args A, uint32_t ti, uint32_t lo, uint32_t hi, uint32_t form) {
  const uint32_t wave = uni(threadIdx.x >> 6);
  if (form == SM_WAVE1) softmax_rows<1, IN16, 64>(A, ti, lo + wave, hi, kWaves);
  else if (form == SM_WAVE4) softmax_rows<4, IN16, 64>(A, ti, lo + wave, hi, kWaves);
  else if (form == SM_FEW2) softmax_rows_few<2, IN16>(A, ti, lo, hi);
  else softmax_rows_few<4, IN16>(A, ti, lo, hi);
}
template <bool IN16>
VM_DEV void softmax_mid_rows(Args A, uint32_t ti, uint32_t lo, uint32_t hi, uint32_t form) {
  const uint32_t wave = uni(threadIdx.x >> 6);
  if (form == SM_FEW8) softmax_rows_few<8, IN16>(A, ti, lo, hi);
  else if (form == SM_WAVE16) softmax_rows<16, IN16, 64>(A, ti, lo + wave, hi, kWaves);
  else softmax_rows<8, IN16, kBlock>(A, ti, lo, hi, 1);
}
template <bool IN16>
VM_DEV void softmax_long_rows(Args A, uint32_t ti, uint32_t lo, uint32_t hi, uint32_t form) {
  if (form == SM_BLOCK32) softmax_rows<32, IN16, kBlock>(A, ti, lo, hi, 1);
  else softmax_rows_long<IN16>(A, ti, lo, hi);
}
VM_LEAF void softmax_short(Args A, uint32_t ti, uint32_t lo, uint32_t hi, uint32_t form) {
  A = uargs(A);
  const bool f32 = ((task_of(A, uni(ti)).tile_op >> 16) & 0xFF) == DT_F32;
  if (f32) softmax_short_rows<false>(A, uni(ti), uni(lo), uni(hi), uni(form));
  else softmax_short_rows<true>(A, uni(ti), uni(lo), uni(hi), uni(form));
}
VM_LEAF void softmax_mid(Args A, uint32_t ti, uint32_t lo, uint32_t hi, uint32_t form) {
  A = uargs(A);
  const bool f32 = ((task_of(A, uni(ti)).tile_op >> 16) & 0xFF) == DT_F32;
  if (f32) softmax_mid_rows<false>(A, uni(ti), uni(lo), uni(hi), uni(form));
  else softmax_mid_rows<true>(A, uni(ti), uni(lo), uni(hi), uni(form));
}
VM_LEAF void softmax_long(Args A, uint32_t ti, uint32_t lo, uint32_t hi, uint32_t form) {
  A = uargs(A);
  const bool f32 = ((task_of(A, uni(ti)).tile_op >> 16) & 0xFF) == DT_F32;
  if (uni(form) == SM_ELEM) softmax_rows_generic(A, uni(ti), uni(lo), uni(hi));
  else if (f32) softmax_long_rows<false>(A, uni(ti), uni(lo), uni(hi), uni(form));
  else softmax_long_rows<true>(A, uni(ti), uni(lo), uni(hi), uni(form));
}

VM_DEV void softmax_tiles(Args A, uint32_t ti, uint32_t lo, uint32_t hi) {
  const VM_K Task& t = task_of(A, ti);
  hi = min(hi, t.p[0]);
  if (lo >= hi) return;
  const uint32_t form = softmax_form(A, t);
  if (form <= SM_FEW4) softmax_short(A, ti, lo, hi, form);
  else if (form <= SM_BLOCK8) softmax_mid(A, ti, lo, hi, form);
  else softmax_long(A, ti, lo, hi, form);
}

// ARGMAX_SEG: dst = first index of the row maximum (a NaN wins: its first index),
// b = that value (a's dtype).  p0 n_out, p1 seg, p3 S: a row's elements split S
// ways (tile = row * S + split; S <= 1: one tile per row).  Each split finds its
// best (value, index); the split that arrives last at the row's counter in the
// task's scratch combines the S candidates (the order is total, so the result
// does not depend on which split is last) and resets the counter.  Candidates
// and counters are agent-scope atomics, which go to memory past the XCD's L2.
// Scratch (S > 1): [n_out * S] {value bits, index}, then n_out counters.
VM_DEV bool amax_better(float v, uint32_t i, float bv, uint32_t bi) {
  const bool vn = v != v, bn = bv != bv;
  if (vn != bn) return vn;
  if (vn) return i < bi;
  if (v != bv) return v > bv;
  return i < bi;
}

// Best (value, index) of elements [j0, j1) of a row over the block; the result
// is in sv[0] / si[0] (index 0xFFFFFFFF: no element).
VM_DEV void amax_block(const gbyte* a, uint32_t adt, uint64_t base, uint32_t j0, uint32_t j1, float* sv,
                       uint32_t* si) {
  float bv = -INFINITY;
  uint32_t bi = 0xFFFFFFFFu;
  auto take = [&](float v, uint32_t j) {
    if (bi == 0xFFFFFFFFu || amax_better(v, j, bv, bi)) {
      bv = v;
      bi = j;
    }
  };
  if (adt == DT_F32 && ((j0 | j1) & 3) == 0 && (((uintptr_t(a) + base * 4) & 15) == 0)) {
    // f32 rows (logits): 16-byte loads, 16 of them in flight per thread; each
    // thread still visits its elements in increasing index order
    const VM_G v4f* row = (const VM_G v4f*)(a + base * 4);
    const uint32_t q0b = j0 >> 2, n4 = j1 >> 2;
    constexpr int U = 16;
    for (uint32_t q0 = q0b + threadIdx.x; q0 < n4; q0 += U * kBlock) {
      v4f v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = row[min(q0 + u * kBlock, n4 - 1)];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t q = q0 + u * kBlock;
        if (q < n4) {
          take(v[u].x, 4 * q);
          take(v[u].y, 4 * q + 1);
          take(v[u].z, 4 * q + 2);
          take(v[u].w, 4 * q + 3);
        }
      }
    }
  } else {
    for (uint32_t j = j0 + threadIdx.x; j < j1; j += kBlock) take(load_f(a, adt, base + j), j);
  }
  lds_barrier();
  sv[threadIdx.x] = bv;
  si[threadIdx.x] = bi;
  lds_barrier();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if (int(threadIdx.x) < s) {
      const float v2 = sv[threadIdx.x + s];
      const uint32_t i2 = si[threadIdx.x + s];
      if (i2 != 0xFFFFFFFFu && (si[threadIdx.x] == 0xFFFFFFFFu || amax_better(v2, i2, sv[threadIdx.x], si[threadIdx.x]))) {
        sv[threadIdx.x] = v2;
        si[threadIdx.x] = i2;
      }
    }
    lds_barrier();
  }
}

VM_DEV void amax_store(gbyte* di, gbyte* dv, uint32_t dt, uint32_t adt, uint32_t o, float v, uint32_t i) {
  const uint32_t idx = i == 0xFFFFFFFFu ? 0u : i;
  if (dt == DT_I64) gcast<int64_t>(di)[o] = idx;
  else gcast<uint32_t>(di)[o] = idx;
  store_f(dv, adt, o, i == 0xFFFFFFFFu ? -INFINITY : v);
}

VM_TILE void argmax_tiles(Args A, uint32_t ti, uint32_t lo, uint32_t hi) {
  A = uargs(A);
  const VM_K Task& t = task_of(A, ti);
  const uint32_t n_out = t.p[0], seg = t.p[1], S = max(1u, t.p[3]);
  const uint32_t dt = (t.tile_op >> 8) & 0xFF, adt = (t.tile_op >> 16) & 0xFF;
  const gbyte* a = resolve(A, t.a);
  gbyte* di = resolve(A, t.dst);
  gbyte* dv = resolve(A, t.b);
  float* sv = lds_f32();
  uint32_t* si = reinterpret_cast<uint32_t*>(sv + kBlock);
  uint32_t* flag = si + kBlock;
  // split length: whole 16-byte runs
  const uint32_t per = ((seg + S - 1) / S + 3) & ~3u;
  hi = min(hi, n_out * S);
  for (uint32_t tile = lo; tile < hi; ++tile) {
    const uint32_t o = tile / S, split = tile % S;
    const uint32_t j0 = min(split * per, seg), j1 = min(seg, j0 + per);
    amax_block(a, adt, uint64_t(o) * seg, j0, j1, sv, si);
    if (S == 1) {
      if (threadIdx.x == 0) amax_store(di, dv, dt, adt, o, sv[0], si[0]);
      continue;
    }
    uint32_t* sp = reinterpret_cast<uint32_t*>(A->scratch + A->task_scratch[ti]);
    uint32_t* arrivals = sp + 2ull * n_out * S;
    if (threadIdx.x == 0) {
      uint32_t* mine = sp + 2ull * (uint64_t(o) * S + split);
      __hip_atomic_store(mine, __float_as_uint(sv[0]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(mine + 1, si[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __builtin_amdgcn_s_waitcnt(0x0F70);             // vmcnt(0): the candidate is in memory
      // acquire-release at agent scope: publishes this split's candidate, and the
      // last arriver sees every other split's before it combines
      const uint32_t before = __hip_atomic_fetch_add(arrivals + o, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
      const bool last = before == S - 1;
      if (last) __hip_atomic_store(arrivals + o, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *flag = last;
    }
    lds_barrier();
    if (*flag) {
      // candidate k by thread k, then the same tree as above
      float bv = -INFINITY;
      uint32_t bi = 0xFFFFFFFFu;
      for (uint32_t k = threadIdx.x; k < S; k += kBlock) {
        const uint32_t* c = sp + 2ull * (uint64_t(o) * S + k);
        const float v = __uint_as_float(__hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        const uint32_t i = __hip_atomic_load(c + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (i != 0xFFFFFFFFu && (bi == 0xFFFFFFFFu || amax_better(v, i, bv, bi))) {
          bv = v;
          bi = i;
        }
      }
      sv[threadIdx.x] = bv;
      si[threadIdx.x] = bi;
      lds_barrier();
      for (int s = kBlock / 2; s > 0; s >>= 1) {
        if (int(threadIdx.x) < s) {
          const float v2 = sv[threadIdx.x + s];
          const uint32_t i2 = si[threadIdx.x + s];
          if (i2 != 0xFFFFFFFFu &&
              (si[threadIdx.x] == 0xFFFFFFFFu || amax_better(v2, i2, sv[threadIdx.x], si[threadIdx.x]))) {
            sv[threadIdx.x] = v2;
            si[threadIdx.x] = i2;
          }
        }
        lds_barrier();
      }
      if (threadIdx.x == 0) amax_store(di, dv, dt, adt, o, sv[0], si[0]);
    }
    lds_barrier();                                    // flag / sv reused by the next tile
  }
}

}  // namespace vm
