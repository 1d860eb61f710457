// TOP_MMA output tiles of 64 x 64 and 128 x 128 through a four-stage LDS pipeline
// (f32, bf16, f16 operands, each either k-contiguous or row-contiguous).
//
// A matmul of a few hundred to a few thousand rows gives a CU one or two tiles
// whose K loop is a chain of global round trips of about 2 us each; the tile's
// matrix work is a fraction of that.  So three stages (32 KiB each) are in flight
// while the fourth is multiplied, and a stage is published by one block barrier.
// Operand memory order does not matter to the tile: what a dot_general contracts
// is k-contiguous in one operand and not in the other (x . W), in both
// (x . W^T: a tied embedding's logits, the gradient of an input) or in neither
// (x^T . g: the gradient of a weight), and each operand keeps its own layout in LDS:
//   k-contiguous (kc): T rows of 128 bytes (64 16-bit or 32 f32 k); the eight
//     16-byte chunks of row r at slots chunk ^ kc_swz(r); a fragment is one
//     ds_read_b128;
//   row-contiguous (rc): 64 (16-bit) or 32 (f32) k rows of T elements, slots
//     chunk ^ swz(k); a 16-bit fragment is two ds_read_b64_tr_b16, an f32 one a
//     ds_read_b32 per k step.
// Both swizzles keep the 64 banks distinct in each read's groups of lanes.
// Operands in whole aligned 16-byte chunks go global -> LDS directly
// (global_load_lds_dwordx4); others (odd row lengths) pass through registers
// with unaligned 16-byte loads, the part of a chunk past the operand shifted out.
//
// Measured on one MI355X (whole launches, us; before: register-staged tiles with
// one slab in flight, and per-element reads of any operand that was transposed or
// whose rows were not 16-byte aligned):
//   bf16 1024^3 23.4 -> 14.9, with W^T 180 -> 15.5, x^T 179 -> 15.8; 2048^3 51 -> 33;
//   f32 1024^3 53.5 -> 31.0, W^T 261 -> 31.4; 1001x777x1130 262 -> 48;
//   a decoder block over 512 tokens (d 768) 258 -> 145.
// What bounds a 64-wide tile of 1024 k in a launch of one round (8.9 us in 16
// bits): ~1.3 us of prologue, then LDS reads and one barrier per 128 k at one wave
// per SIMD; in f32 (25 us) the matrix cores, 14.6 us of it.
#pragma once

namespace vm {

// An operand as the pipelined tiles read it (vm_abi.h MmaOperand, its base resolved).
struct MmaOp {
  const gbyte* p;
  uint64_t gs;
  uint32_t ld, R;
  uint32_t kc, cls;
  uint32_t view;          // MOP_RUNS: the view (aux offset + 1) its chunks are read through
};
VM_DEV MmaOp mma_op(const VM_K MmaOperand& o, const gbyte* base, uint32_t R, uint32_t esz) {
  MmaOp x;
  x.p = base + uint64_t(o.off) * esz;
  x.gs = uint64_t(o.gs_lo) | uint64_t(o.gs_hi) << 32;
  x.ld = o.ld;
  x.R = R;
  x.kc = o.kc;
  x.cls = o.cls;
  x.view = o.view;
  return x;
}

enum { ELT_BF16 = 0, ELT_F16 = 1, ELT_F32 = 2 };

template <int T, int ELT>
struct Pipe {
  static constexpr uint32_t kEsz = ELT == ELT_F32 ? 4 : 2;
  static constexpr uint32_t kPer = 16 / kEsz;
  static constexpr uint32_t kSlabK = 128 / kEsz;            // k of one sub-slab
  static constexpr uint32_t kSub = T == 64 ? 2 : 1;         // sub-slabs of a stage
  static constexpr uint32_t kStageK = kSlabK * kSub;
  static constexpr uint32_t kOp = T * 128;                  // bytes of one operand's sub-slab
  static constexpr uint32_t kStage = 2 * kOp * kSub;        // 32 KiB
  static constexpr uint32_t kStages = 4;
  static constexpr int kB = T / 64;                         // 32-wide blocks of a wave along M and N
  static constexpr int kRounds = T / 32;                    // 16-byte transfers per thread, operand and sub-slab
  static constexpr uint32_t kRowB = T * kEsz;               // row bytes of an rc sub-slab
  static constexpr uint32_t kRowC = kRowB / 16;             // its chunks
};

// f32: MFMA step kk of a 16-deep slab takes k = kk in lanes 0-31 and k = 8 + kk in
// lanes 32-63, as every f32 tile here does, so the tiles' sums are the same bits
// (a sum near 0 decides a relu's gradient).  The two halves of a wave then read
// chunks c and c ^ 2 of their rows, and rows k and k + 8: eight consecutive rows of
// one parity take swizzles {0, 1, 4, 5} or {2, 3, 6, 7}.
template <int ELT>
VM_DEV uint32_t kc_swz(uint32_t r) {
  if constexpr (ELT == ELT_F32) return ((r >> 1) & 1) | (((r >> 3) & 1) << 1) | (((r >> 2) & 1) << 2);
  else return aswz(r);
}
template <int T, int ELT>
VM_DEV uint32_t rc_swz(uint32_t k) {
  if constexpr (ELT == ELT_F32) return 8 * ((k >> 3) & 1);
  else if constexpr (T == 128) return 4 * (k & 3);
  else return 4 * ((k >> 1) & 1);
}

// One operand's way into the stages: which chunk each thread moves in each round.
// Round j of wave w fills bytes [1024 (4 j + w), +1024) of the operand's sub-slab,
// 16 per lane.
template <int T, int ELT, bool KC>
struct PipeSrc {
  using P = Pipe<T, ELT>;
  const gbyte* base;        // kc: element (g, r0, 0); rc: element (g, 0, 0)
  uint32_t ld, k1;
  uint32_t off[P::kRounds]; // kc: row byte offset; rc: row byte offset of the round within a full sub-slab + column bytes
  uint32_t kq;              // kc: first k of this lane's chunk in a sub-slab; rc: its k row in round 0
  uint32_t cut[P::kRounds]; // rc, through registers: elements of the chunk past R
  bool edge;                // some lane's cut is not 0
  uint32_t colb[P::kRounds];   // rc: column byte offset (clamped into the operand)
  // MOP_RUNS
  ViewMap map;
  uint32_t lin[P::kRounds];

  template <bool RUNS>
  VM_DEV void init(const VM_K int32_t* aux, const MmaOp& o, uint32_t g, uint32_t r0, uint32_t K, uint32_t k1_) {
    const uint32_t l = threadIdx.x & 63, w = threadIdx.x >> 6;
    ld = o.ld;
    k1 = k1_;
    edge = false;
    if constexpr (KC) {
      base = o.p + (o.gs * g + uint64_t(r0) * ld) * P::kEsz;
      const uint32_t row0 = 8 * w + (l >> 3);
      kq = ((l & 7) ^ kc_swz<ELT>(row0)) * P::kPer;
#pragma unroll
      for (int j = 0; j < P::kRounds; ++j) {
        const uint32_t row = min(row0 + 32 * j + r0, o.R - 1);
        off[j] = (row - r0) * ld * P::kEsz;
        if constexpr (RUNS) lin[j] = (g * o.R + row) * K;
      }
      if constexpr (RUNS) {
        map = view_map(aux, o.view);
        base = o.p;
      }
    } else {
      base = o.p + o.gs * g * P::kEsz;
      kq = (1024 / P::kRowB) * w + l / P::kRowC;
#pragma unroll
      for (int j = 0; j < P::kRounds; ++j) {
        const uint32_t c = ((l % P::kRowC) ^ rc_swz<T, ELT>(krow(kq, j))) * P::kPer + r0;
        const uint32_t cc = min(c, o.R - P::kPer);
        cut[j] = c - cc;
        colb[j] = cc * P::kEsz;
        off[j] = krow(kq, j) * ld * P::kEsz + colb[j];
        edge |= __builtin_amdgcn_ballot_w64(c != cc) != 0;
      }
    }
  }
  // k row of round j (rc)
  static VM_DEV uint32_t krow(uint32_t kq, int j) { return kq + (4096 / P::kRowB) * j; }

  // Byte offset of round j's chunk from `at` (the returned scalar base) for the
  // sub-slab at k; every address is clamped into the operand.
  template <bool RUNS>
  VM_DEV uint32_t chunk(const VM_K int32_t* aux, uint32_t view, uint32_t k, int j) const {
    if constexpr (KC) {
      const uint32_t kk = min(k + kq, k1 - P::kPer);
      if constexpr (RUNS) return uint32_t(view_at(map, aux, view, lin[j] + kk)) * P::kEsz;
      return off[j] + kk * P::kEsz;
    } else {
      return (min(k + krow(kq, j), k1 - 1) - k) * ld * P::kEsz + colb[j];
    }
  }
  // sub-slab at k (below k1) into LDS at st
  template <bool RUNS>
  VM_DEV void dma(const VM_K int32_t* aux, uint32_t view, uint32_t k, uint32_t st) const {
    const uint32_t wo = uni(1024 * (threadIdx.x >> 6));
    const gbyte* b = KC ? base : base + uint64_t(k) * ld * P::kEsz;
    if (!KC && k + P::kSlabK <= k1) {
#pragma unroll
      for (int j = 0; j < P::kRounds; ++j) dma16(b, off[j], st + wo + 4096 * j);
    } else {
#pragma unroll
      for (int j = 0; j < P::kRounds; ++j) dma16(b, chunk<RUNS>(aux, view, k, j), st + wo + 4096 * j);
    }
  }
  // zero this lane's slots of the sub-slab at k that hold k >= k1 (after its
  // transfers have landed, before the block barrier that publishes the stage)
  VM_DEV void zero(uint32_t k, uint32_t st) const {
    typedef __attribute__((address_space(3))) v4u lds_v4u;
    const uint32_t at = st + 1024 * (threadIdx.x >> 6) + 16 * (threadIdx.x & 63);
#pragma unroll
    for (int j = 0; j < P::kRounds; ++j)
      if (k + (KC ? kq : krow(kq, j)) >= k1) *(lds_v4u*)uintptr_t(at + 4096 * j) = v4u_make(0, 0, 0, 0);
  }
  // The same chunks through registers: unaligned 16-byte loads of clamped
  // addresses; elements past the operand are shifted out (zeros come in).
  typedef uint32_t v4u_any __attribute__((ext_vector_type(4), aligned(2)));
  VM_DEV void load(v4u (&r)[P::kRounds], uint32_t k) const {
    const gbyte* b = KC ? base : base + uint64_t(min(k, k1 - 1)) * ld * P::kEsz;
#pragma unroll
    for (int j = 0; j < P::kRounds; ++j) {
      uint32_t o;
      if constexpr (KC) o = off[j] + min(k + kq, k1 - P::kPer) * P::kEsz;
      else o = (min(k + krow(kq, j), k1 - 1) - min(k, k1 - 1)) * ld * P::kEsz + colb[j];
      r[j] = *(const VM_G v4u_any*)(b + o);
    }
  }
  static VM_DEV v4u shift_out(v4u v, uint32_t elems) {
    const uint32_t s = elems * (8 * P::kEsz);
    const uint64_t lo = uint64_t(v.x) | uint64_t(v.y) << 32, hi = uint64_t(v.z) | uint64_t(v.w) << 32;
    const uint32_t sh = s & 63;
    const uint64_t l0 = sh ? (lo >> sh) | (hi << (64 - sh)) : lo, h0 = hi >> sh;
    const uint64_t l = s >= 128 ? 0 : s >= 64 ? h0 : l0, h = s >= 64 ? 0 : h0;
    return v4u_make(uint32_t(l), uint32_t(l >> 32), uint32_t(h), uint32_t(h >> 32));
  }
  VM_DEV void put(v4u (&r)[P::kRounds], uint32_t k, uint32_t st) const {
    typedef __attribute__((address_space(3))) v4u lds_v4u;
    const uint32_t at = st + 1024 * (threadIdx.x >> 6) + 16 * (threadIdx.x & 63);
    const bool tail = k + P::kSlabK > k1;                   // uniform; edge too
    if (!(tail || edge)) {
#pragma unroll
      for (int j = 0; j < P::kRounds; ++j) *(lds_v4u*)uintptr_t(at + 4096 * j) = r[j];
      return;
    }
#pragma unroll
    for (int j = 0; j < P::kRounds; ++j) {
      v4u v;
      if constexpr (KC) {
        v = shift_out(r[j], min(k + kq - min(k + kq, k1 - P::kPer), 16u));
      } else {
        v = shift_out(r[j], min(cut[j], 16u));
        if (k + krow(kq, j) >= k1) v = v4u_make(0, 0, 0, 0);
      }
      *(lds_v4u*)uintptr_t(at + 4096 * j) = v;
    }
  }
};

// Fragment addresses of one operand within a sub-slab, and the reads.
template <int T, int ELT, bool KC>
struct PipeFrag {
  using P = Pipe<T, ELT>;
  uint32_t a[4];
  // w2: the wave's half of the tile along this operand
  VM_DEV void init(uint32_t w2) {
    const uint32_t lane = threadIdx.x & 63;
    if constexpr (KC) {
      const uint32_t r = w2 * (T / 2) + (lane & 31);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t c = ELT == ELT_F32 ? 4 * (q >> 1) + (q & 1) + 2 * (lane >> 5) : 2 * q + (lane >> 5);
        a[q] = r * 128 + ((c ^ kc_swz<ELT>(r)) * 16);
      }
    } else if constexpr (ELT == ELT_F32) {
      const uint32_t c = w2 * (T / 2) + (lane & 31), row = 8 * (lane >> 5);
#pragma unroll
      for (int b = 0; b < P::kB; ++b)
        a[b] = row * P::kRowB + ((((c + 32 * b) >> 2) ^ rc_swz<T, ELT>(row)) * 16) + (c & 3) * 4;
    } else {
      const uint32_t gq = lane >> 4, e = (lane >> 2) & 3, q = lane & 3, row = 8 * (gq >> 1) + e;
#pragma unroll
      for (int b = 0; b < P::kB; ++b) {
        const uint32_t c = w2 * (T / 2) + 32 * b + 16 * (gq & 1) + 4 * q;
        a[b] = row * P::kRowB + (((c >> 3) ^ rc_swz<T, ELT>(row)) * 16) + (q & 1) * 8;
      }
    }
  }
  // 16-bit: the fragment of block b, k step kk (16 k)
  VM_DEV u16x8 frag16(const lds_u8* S, int kk, int b) const {
    if constexpr (KC) {
      return *(const lds_u16x8*)(S + a[kk] + 4096 * b);
    } else {
      const lds_u8* p = S + a[b] + 16 * kk * P::kRowB;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p);
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 4 * P::kRowB));
      return __builtin_bit_cast(u16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  }
  // f32: the four values of block b for k 16 (q / 2) + 4 (q % 2) + {0, 1, 2, 3} (+ 8 in lanes 32-63)
  VM_DEV v4f frag32(const lds_u8* S, int q, int b) const {
    typedef __attribute__((address_space(3))) v4f lds_v4f;
    typedef __attribute__((address_space(3))) float lds_f;
    if constexpr (KC) {
      return *(const lds_v4f*)(S + a[q] + 4096 * b);
    } else {
      const lds_u8* p = S + a[b] + (16 * (q >> 1) + 4 * (q & 1)) * P::kRowB;
      return v4f_make(*(const lds_f*)p, *(const lds_f*)(p + P::kRowB), *(const lds_f*)(p + 2 * P::kRowB),
                      *(const lds_f*)(p + 3 * P::kRowB));
    }
  }
};

template <int T, int ELT, bool KA, bool KB>
VM_DEV void pipe_stage(const lds_u8* S, const PipeFrag<T, ELT, KA>& fa, const PipeFrag<T, ELT, KB>& fb,
                       f32x16 (&acc)[Pipe<T, ELT>::kB][Pipe<T, ELT>::kB]) {
  using P = Pipe<T, ELT>;
#pragma unroll
  for (uint32_t u = 0; u < P::kSub; ++u) {
    const lds_u8* A = S + 2 * P::kOp * u;
    const lds_u8* B = A + P::kOp;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if constexpr (ELT == ELT_F32) {
        v4f x[P::kB], y[P::kB];
#pragma unroll
        for (int i = 0; i < P::kB; ++i) x[i] = fa.frag32(A, q, i);
#pragma unroll
        for (int j = 0; j < P::kB; ++j) y[j] = fb.frag32(B, q, j);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < P::kB; ++i)
#pragma unroll
            for (int j = 0; j < P::kB; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i][e], y[j][e], acc[i][j], 0, 0, 0);
      } else {
        u16x8 x[P::kB], y[P::kB];
#pragma unroll
        for (int i = 0; i < P::kB; ++i) x[i] = fa.frag16(A, q, i);
#pragma unroll
        for (int j = 0; j < P::kB; ++j) y[j] = fb.frag16(B, q, j);
#pragma unroll
        for (int i = 0; i < P::kB; ++i)
#pragma unroll
          for (int j = 0; j < P::kB; ++j) acc[i][j] = mfma16<ELT == ELT_BF16>(x[i], y[j], acc[i][j]);
      }
    }
  }
}

VM_DEV void wait_vm16() { __builtin_amdgcn_s_waitcnt(0x4F70); }   // s_waitcnt vmcnt(16)

// K loop, direct-to-LDS operands: three stages in flight.
template <int T, int ELT, bool KA, bool KB, bool RUNS>
VM_DEV void pipe_loop_dma(Args A, const MmaOp& oa, const MmaOp& ob, uint32_t g, uint32_t m0, uint32_t n0, uint32_t K,
                          uint32_t k0, uint32_t k1, uint32_t lds0,
                          f32x16 (&acc)[Pipe<T, ELT>::kB][Pipe<T, ELT>::kB]) {
  using P = Pipe<T, ELT>;
  static_assert(P::kRounds * 2 * P::kSub == 8, "transfers per stage and thread");
  const VM_K int32_t* aux = aux_of(A);
  PipeSrc<T, ELT, KA> sa;
  PipeSrc<T, ELT, KB> sb;
  sa.template init<RUNS>(aux, oa, g, m0, K, k1);
  sb.template init<false>(aux, ob, g, n0, K, k1);
  PipeFrag<T, ELT, KA> fa;
  PipeFrag<T, ELT, KB> fb;
  const uint32_t wave = threadIdx.x >> 6;
  fa.init(wave >> 1);
  fb.init(wave & 1);
  const uint32_t ns = (k1 - k0 + P::kStageK - 1) / P::kStageK;
  const lds_u8* L = (const lds_u8*)uintptr_t(lds0);
  // the sub-slabs of a last stage that start past k1 are transferred from clamped addresses, and zeroed
  auto issue = [&](uint32_t s) {
    const uint32_t st = lds0 + (s % P::kStages) * P::kStage;
#pragma unroll
    for (uint32_t u = 0; u < P::kSub; ++u) {
      const uint32_t k = min(k0 + s * P::kStageK + u * P::kSlabK, k1 - 1);
      sa.template dma<RUNS>(aux, oa.view, k, st + 2 * P::kOp * u);
      sb.template dma<false>(aux, 0, k, st + 2 * P::kOp * u + P::kOp);
    }
  };
  __syncthreads();                      // the previous user of the LDS is done
#pragma unroll
  for (uint32_t s = 0; s < P::kStages - 1; ++s)
    if (s < ns) issue(s);
  for (uint32_t s = 0; s < ns; ++s) {
    if (s + 2 < ns) wait_vm16();
    else if (s + 1 < ns) wait_vm8();
    else wait_vm0();
    const uint32_t so = (s % P::kStages) * P::kStage;
    if (s + 1 == ns && (k1 - k0) % P::kStageK) {
#pragma unroll
      for (uint32_t u = 0; u < P::kSub; ++u) {
        const uint32_t k = k0 + s * P::kStageK + u * P::kSlabK;
        sa.zero(k, lds0 + so + 2 * P::kOp * u);
        sb.zero(k, lds0 + so + 2 * P::kOp * u + P::kOp);
      }
    }
    __syncthreads();                    // stage s is published; every read of stage s - 1 is done
    if (s + P::kStages - 1 < ns) issue(s + P::kStages - 1);
    pipe_stage<T, ELT, KA, KB>(L + so, fa, fb, acc);
  }
}

// K loop, operands through registers: one stage in registers ahead, two in LDS.
template <int T, int ELT, bool KA, bool KB>
VM_DEV void pipe_loop_reg(Args A, const MmaOp& oa, const MmaOp& ob, uint32_t g, uint32_t m0, uint32_t n0, uint32_t K,
                          uint32_t k0, uint32_t k1, uint32_t lds0,
                          f32x16 (&acc)[Pipe<T, ELT>::kB][Pipe<T, ELT>::kB]) {
  using P = Pipe<T, ELT>;
  const VM_K int32_t* aux = aux_of(A);
  PipeSrc<T, ELT, KA> sa;
  PipeSrc<T, ELT, KB> sb;
  sa.template init<false>(aux, oa, g, m0, K, k1);
  sb.template init<false>(aux, ob, g, n0, K, k1);
  PipeFrag<T, ELT, KA> fa;
  PipeFrag<T, ELT, KB> fb;
  const uint32_t wave = threadIdx.x >> 6;
  fa.init(wave >> 1);
  fb.init(wave & 1);
  const uint32_t ns = (k1 - k0 + P::kStageK - 1) / P::kStageK;
  const lds_u8* L = (const lds_u8*)uintptr_t(lds0);
  struct Regs {
    v4u a[P::kSub][P::kRounds], b[P::kSub][P::kRounds];
  };
  Regs r[2];
  auto load = [&](Regs& x, uint32_t s) {
#pragma unroll
    for (uint32_t u = 0; u < P::kSub; ++u) {
      sa.load(x.a[u], k0 + s * P::kStageK + u * P::kSlabK);
      sb.load(x.b[u], k0 + s * P::kStageK + u * P::kSlabK);
    }
  };
  auto put = [&](Regs& x, uint32_t s) {
    const uint32_t st = lds0 + (s & 1) * P::kStage;
#pragma unroll
    for (uint32_t u = 0; u < P::kSub; ++u) {
      sa.put(x.a[u], k0 + s * P::kStageK + u * P::kSlabK, st + 2 * P::kOp * u);
      sb.put(x.b[u], k0 + s * P::kStageK + u * P::kSlabK, st + 2 * P::kOp * u + P::kOp);
    }
  };
  // loads past the last stage re-read its clamped addresses and are not used
  load(r[0], 0);
  load(r[1], 1);
  __syncthreads();                      // the previous user of the LDS is done
  auto step = [&](Regs& x, uint32_t s) {
    put(x, s);
    load(x, s + 2);
    __syncthreads();                    // stage s is published; reads of stage s - 2's buffer ended a barrier ago
    pipe_stage<T, ELT, KA, KB>(L + (s & 1) * P::kStage, fa, fb, acc);
  };
  for (uint32_t s = 0; s < ns; s += 2) {
    step(r[0], s);
    if (s + 1 >= ns) break;
    step(r[1], s + 1);
  }
}

// Store of a T x T tile: accumulators -> LDS (row stride T + 4 floats) -> rows of
// 16-byte (f32) or 8-byte (16-bit) stores with the epilogue on the way, four
// row groups at a time: their residual values are read together, and each
// micro-op is dispatched once for all sixteen values of a thread.
template <int T>
VM_DEV void store_pipe(Args A, const MmaDesc& D, const f32x16 (&acc)[T / 64][T / 64], uint32_t g, uint32_t m0,
                       uint32_t n0) {
  constexpr uint32_t LD = T + 4, CT = T / 4, RP = kBlock / CT, U = 4;   // threads per row, rows per step, steps per batch
  typedef float v4f_any __attribute__((ext_vector_type(4), aligned(4)));
  typedef uint32_t v2u_any __attribute__((ext_vector_type(2), aligned(2)));
  float* st = lds_ptr<float>();
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t wm = wave >> 1, wn = wave & 1;
  const VM_K int32_t* e = aux_of(A) + (D.epi ? D.epi - 1 : 0);
  const int nm = D.epi ? uni(e[0]) : 0;
  bool src1 = false, src2 = false;
  for (int k = 0; k < nm; ++k) {
    src1 |= e[2 + 4 * k] == 1;
    src2 |= e[2 + 4 * k] == 2;
  }
  const uint32_t c = (threadIdx.x % CT) * 4, col = n0 + c;
  const bool whole = col + 4 <= D.N;
  const VM_G float* res = (const VM_G float*)D.res;
  v4f ycol = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  if (src2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) ycol[i] = res[min(col + i, D.N - 1)];
  }
  __syncthreads();                      // the K loop's last LDS reads are done
#pragma unroll
  for (int i = 0; i < T / 64; ++i)
#pragma unroll
    for (int j = 0; j < T / 64; ++j) {
      float* p = st + (wm * (T / 2) + i * 32 + 4 * (lane >> 5)) * LD + wn * (T / 2) + j * 32 + (lane & 31);
#pragma unroll
      for (int v = 0; v < 16; ++v) p[(8 * (v >> 2) + (v & 3)) * LD] = acc[i][j][v];
    }
  __syncthreads();
  const uint64_t tile0 = (uint64_t(g) * D.M + m0) * D.N + n0;
  const uint32_t rows = min(uint32_t(T), D.M - m0);
  if (col >= D.N) return;
#pragma unroll 1
  for (uint32_t r0 = threadIdx.x / CT; r0 < rows; r0 += U * RP) {
    v4f x[U], y[U];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      const uint32_t r = min(r0 + u * RP, uint32_t(T - 1));
      x[u] = *reinterpret_cast<const v4f*>(st + r * LD + c);
    }
    if (src1) {
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) {
        const uint64_t at = tile0 + uint64_t(min(r0 + u * RP, rows - 1)) * D.N + c;
        if (whole) {
          y[u] = *(const VM_G v4f_any*)(res + at);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) y[u][i] = res[at + min(uint32_t(i), D.N - 1 - col)];
        }
      }
    }
    for (int k = 0; k < nm; ++k) {
      const uint32_t kind = uint32_t(e[1 + 4 * k]), src = uint32_t(e[2 + 4 * k]);
      const float s = __int_as_float(e[3 + 4 * k]), t = __int_as_float(e[4 + 4 * k]);
      v4f o[U];
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) o[u] = src == 1 ? y[u] : src == 2 ? ycol : src == 3 ? v4f_make(s, s, s, s) : x[u];
      epi_inline16(kind, x, o, s, t);
    }
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      const uint32_t r = r0 + u * RP;
      if (r >= rows) continue;
      const uint64_t at = tile0 + uint64_t(r) * D.N + c;
      if (whole) {
        if (D.dt == DT_F32) {
          *(VM_G v4f_any*)(D.d + at * 4) = x[u];
        } else {
          const bool bf = D.dt == DT_BF16;
          const uint32_t lo = bf ? pack_bf16x2(x[u].x, x[u].y) : f32_to_f16(x[u].x) | uint32_t(f32_to_f16(x[u].y)) << 16;
          const uint32_t hi = bf ? pack_bf16x2(x[u].z, x[u].w) : f32_to_f16(x[u].z) | uint32_t(f32_to_f16(x[u].w)) << 16;
          *(VM_G v2u_any*)(D.d + at * 2) = v2u_make(lo, hi);
        }
      } else {
#pragma unroll
        for (uint32_t i = 0; i < 3; ++i)
          if (col + i < D.N) store_f(D.d, D.dt, at + i, x[u][i]);
      }
    }
  }
}

// One T x T tile (or a K split's share of it).
template <int T, int ELT>
VM_DEV void mma_pipe_one(Args A, const MmaDesc& D, const MmaOp& oa, const MmaOp& ob, bool dma, const MmaPos& at) {
  using P = Pipe<T, ELT>;
  const uint32_t lds0 = uni(uint32_t(reinterpret_cast<uintptr_t>(lds_ptr<lds_u8>())));
  f32x16 acc[P::kB][P::kB];
#pragma unroll
  for (int i = 0; i < P::kB; ++i)
#pragma unroll
    for (int j = 0; j < P::kB; ++j) acc[i][j] = f32x16{};
  if (D.k1 > D.k0) {
#define VM_PIPE(KA, KB)                                                                                              \
  {                                                                                                                  \
    if (dma && oa.cls == MOP_RUNS) {                                                                                 \
      if constexpr (KA) pipe_loop_dma<T, ELT, KA, KB, true>(A, oa, ob, at.g, at.m0, at.n0, D.K, D.k0, D.k1, lds0, acc); \
    } else if (dma) {                                                                                                \
      pipe_loop_dma<T, ELT, KA, KB, false>(A, oa, ob, at.g, at.m0, at.n0, D.K, D.k0, D.k1, lds0, acc);               \
    } else {                                                                                                         \
      pipe_loop_reg<T, ELT, KA, KB>(A, oa, ob, at.g, at.m0, at.n0, D.K, D.k0, D.k1, lds0, acc);                      \
    }                                                                                                                \
  }
    if (oa.kc) {
      if (ob.kc) VM_PIPE(true, true) else VM_PIPE(true, false)
    } else {
      if (ob.kc) VM_PIPE(false, true) else VM_PIPE(false, false)
    }
#undef VM_PIPE
  }
  if (D.S > 1 && !mma_split_combine<T>(A, D, acc, at.id)) return;
  store_pipe<T>(A, D, acc, at.g, at.m0, at.n0);
}

// A task's tiles [lo, hi): one leaf with the loop and the tile inlined.  The
// classes and layouts of the operands are the task's, so every tile of it takes the
// same route.
template <int T, int ELT>
VM_LEAF void mma_pipe_tiles(Args A, uint32_t ti, uint32_t lo, uint32_t hi) {
  A = uargs(A);
  MmaDesc D = mma_desc(A, uni(ti));
  const VM_K MmaRec& r = rec_of(A, D.ti);
  const MmaOp oa = mma_op(r.a, D.a, r.M, Pipe<T, ELT>::kEsz), ob = mma_op(r.b, D.b, r.N, Pipe<T, ELT>::kEsz);
  const bool dma = oa.cls <= MOP_RUNS && ob.cls == MOP_DMA && ((uintptr_t(D.a) | uintptr_t(D.b)) & 15) == 0;
  for (uint32_t ts = uni(lo); ts < uni(hi); ++ts)
    for (uint32_t q = 0; q < r.subs; ++q) {
      MmaPos p;
      if (mma_pos(r, D, ts, q, &p)) mma_pipe_one<T, ELT>(A, D, oa, ob, dma, p);
    }
}

}  // namespace vm
