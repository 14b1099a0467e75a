// fp32 io kernels for gfx950 (MI355X): dense tensors, D in {16, 32, 64, 128}, any E.
//
// The tuned 16-bit kernels' algorithm in true fp32: v_mfma_f32_32x32x2_f32 with no rounding of h
// or dZ (the reference's io dtype is x's, flashmlp.py:87). A 32 x 32 x 2 product takes 64 clocks of
// a SIMD, during which its vector instructions wait too (counters of the forward at H=8 B=16384
// D=64 E=1024: matrix unit busy 73 % of the CU cycles, 2.5 vector instructions per product, no
// LDS conflicts, no time gained by interleaving the two), so the kernels are bound by the sum of
// the two: the fp32 matrix rate (157 TFLOP/s nominal, 154 reached by a library product) less the
// activation's and the address instructions' share.
//   * f32_fwd_kernel: a wave owns 32 rows, its X rows in registers; W1c [D][32] and W2c [32][D]
//     chunks go through a two-slot LDS ring (buffer loads with the LDS destination, one chunk
//     ahead; a chunk is 2-4 us of matrix work per SIMD). Z^T = W1c^T X^T leaves the MFMA with lane = row,
//     the A operand of O += h W2c.
//   * f32_bwd_kernel: dX programs (the same walk over E, with dO rows and dH^T = W2c dO^T, and
//     dX += dZ W1c^T) and dW programs (a wave owns 32 E-columns, whose weights stay in registers,
//     and walks 32-row subtiles of X and dO through the ring) in one launch, as in fmlp_bwd.hip.
// EP (run time): the workgroup's waves are RT = NW / EP row tiles times EP parts of E, each part
// with a ring of its own; the parts' partial tiles are added through LDS in part order. Likewise a
// dW program is CG column groups times RS = NW / CG sets of subtiles.
// Measured (SiLU, forward / backward us) against the generic kernels, whose operands come element by
// element from L1 / L2: H=12 B=1024 D=64 E=768 173 / 389 -> 34 / 93; H=8 B=16384 D=64 E=1024
// 1617 / 3497 -> 288 / 982 (119 / 122 TFLOP/s executed); H=8 B=4096 D=128 E=1024 788 / 2540 ->
// 153 / 527; H=32 B=4096 D=32 E=512 492 / 1016 -> 83 / 277. Rounding errors against 64 bits fall as
// well (2.7e-7 -> 2.1e-7 on the first), from the shorter chains of additions.
//
// K order: a product's two k-slots are g = lane / 32, so step (j, m) of a contraction over d takes
// d = 8 j + 4 g + m, m < 4: a lane's four consecutive values are one 16-byte piece. The C layout's
// rows 8 (i / 4) + 4 g + i % 4 have the same form, so a C tile is the next product's A operand
// with i = 4 j + m.
#include "fmlp_device.h"
#include "fmlp_launch.h"

#include <algorithm>
#include <mutex>

namespace fmlp {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// 8 waves (two per SIMD) up to D = 64; 4 at D = 128 (one per SIMD: a dX wave holds X, dO and dX
// rows and two tiles, ~230 registers; a dW wave its weights and both accumulators, ~290)
__host__ __device__ constexpr int f32_nw(int D) { return D <= 64 ? 8 : 4; }

__device__ __forceinline__ f32x16 mma2(float a, float b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 lds_f4(int off) { return *(const FMLP_LDS f32x4*)((FMLP_LDS char*)fmlp_lds + off); }
__device__ __forceinline__ float lds_f1(int off) { return *(const FMLP_LDS float*)((FMLP_LDS char*)fmlp_lds + off); }

// LDS tiles are rows of C fp32 values (C = 32 or D, at least eight 16-byte pieces); piece q of row r
// is stored at piece q ^ (r & 7) of its aligned group of eight, which keeps both read patterns
// (almost) conflict free:
//   row reads: lane = row l32, piece 2 j + g (four k steps): at row[j & 3] + (j / 4) 128
//   column reads: lane = columns V l32 .. + V - 1, row 8 j + 4 g + m: at col[m] + j 8 (4 C)
// V = D / 32 for the products whose columns are d: a lane owns V consecutive columns, so one read
// feeds its V tiles and the results are stored as vectors; V = 1 for W1c.
template <int C, int V>
struct Lanes {
  int row[4], col[4];
  __device__ __forceinline__ Lanes(int g, int l32) {
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int p = (V * l32) >> 2;
      row[m] = l32 * (C * 4) + (((2 * m + g) ^ (l32 & 7)) << 4);
      col[m] = (4 * g + m) * (C * 4) + ((p & ~7) << 4) + (((p ^ (4 * g + m)) & 7) << 4) + ((V * l32) & 3) * 4;
    }
  }
};
template <int V>
struct VecT {
  float v[V];
};
template <int V>
__device__ __forceinline__ VecT<V> lds_vec(int off) {
  VecT<V> r;
  if constexpr (V == 4) {
    const f32x4 x = lds_f4(off);
#pragma unroll
    for (int i = 0; i < 4; ++i) r.v[i] = x[i];
  } else if constexpr (V == 2) {
    const u32x2 x = lds_read8(off);
    r.v[0] = __uint_as_float(x[0]);
    r.v[1] = __uint_as_float(x[1]);
  } else {
    r.v[0] = lds_f1(off);
  }
  return r;
}

// E-chunks of one head's weights into an LDS slot: W1c [D][32], then W2c [32][D], by the nt threads
// of a part (t0 = 64 times the wave's index in the part). Columns at or past e_end, and rows and
// columns past DG, land as zeros. An fp32 product occupies the vector unit, so the loop's address
// work is kept off it: a lane's offsets are fixed (the swizzle of a 64-piece run differs from the
// first one's by bits that are XORed in) and the runs advance the scalar resource.
template <int D, int DG>
struct ChunkLoad {
  unsigned off1, off2;
  int q1;
  __device__ __forceinline__ ChunkLoad(int ldw, int lane) {
    const int r1 = lane >> 3, r2 = lane / (D / 4), s = lane % (D / 4), q2 = (s & ~7) | ((s ^ r2) & 7);
    q1 = (lane ^ r1) & 7;
    off1 = (unsigned)(r1 * ldw * 4 + q1 * 16);
    off2 = 4 * q2 < DG ? (unsigned)(r2 * DG * 4 + q2 * 16) : BUF_OOB;
  }
  __device__ __forceinline__ void operator()(const float* __restrict__ W1h, const float* __restrict__ W2h, int ldw,
                                             int e_end, int c, int slot, int t0, int nt) const {
    const int lim = e_end - c * 32;
    const unsigned o1 = 4 * q1 < lim ? off1 : BUF_OOB;
    for (int p0 = t0; p0 < 8 * D; p0 += nt) {
      const int r = p0 >> 3, rem = (DG - r) * ldw * 4 - 128 * c;
      buf_load16_lds(make_rsrc_words(W1h + (size_t)r * ldw + (size_t)c * 32, rem > 0 ? rem : 0), o1, slot + p0 * 16);
    }
    for (int p0 = t0; p0 < 8 * D; p0 += nt) {
      const int r = p0 / (D / 4);
      buf_load16_lds(make_rsrc_words(W2h + ((size_t)c * 32 + r) * DG, clamp0(lim - r, 32) * DG * 4),
                     D > 32 ? off2 ^ ((r & 7) << 4) : off2, slot + 128 * D + p0 * 16);
    }
  }
};

// this wave's loads have landed, then every wave's have (and every earlier LDS read is done)
__device__ __forceinline__ void ring_sync() {
  wait_vmcnt<0>();
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// adds parts 1 .. EP-1's tiles (NTN accumulators per wave) to part 0's through LDS, in part order
template <int NTN>
__device__ __forceinline__ void sum_parts(f32x16 (&acc)[NTN], int ep, int part, int rtile, int rt, int lane) {
  if (ep <= 1) return;
  auto slot = [&](int p) { return ((p - 1) * rt + rtile) * (NTN * 4096); };
  if (part > 0) {
#pragma unroll
    for (int nt = 0; nt < NTN; ++nt)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4)
        lds_write16(slot(part) + ((nt * 4 + i4) * 64 + lane) * 16,
                    u32x4{__float_as_uint(acc[nt][4 * i4]), __float_as_uint(acc[nt][4 * i4 + 1]),
                          __float_as_uint(acc[nt][4 * i4 + 2]), __float_as_uint(acc[nt][4 * i4 + 3])});
  }
  __syncthreads();
  if (part > 0) return;
  for (int p = 1; p < ep; ++p)
#pragma unroll
    for (int nt = 0; nt < NTN; ++nt)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const f32x4 v = lds_f4(slot(p) + ((nt * 4 + i4) * 64 + lane) * 16);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[nt][4 * i4 + j] += v[j];
      }
}

// 32 rows of a [rows][DG] tensor from tiles whose lane l32 holds columns NTN l32 + nt; rows at or
// past B fall outside the resource
template <int D, int DG>
__device__ __forceinline__ void store_cols(const f32x16 (&acc)[D / 32], float* __restrict__ out, int B, int b0, int g,
                                           int l32) {
  constexpr int NTN = D / 32;
  const Rsrc r = make_rsrc(out + (size_t)b0 * DG, clamp0(B - b0, 32) * DG * 4);
  const unsigned vo = NTN * l32 < DG ? (unsigned)((4 * g * DG + NTN * l32) * 4) : BUF_OOB;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int o = (int)vo + (8 * (i >> 2) + (i & 3)) * DG * 4;
    if constexpr (NTN == 4)
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{__float_as_uint(acc[0][i]), __float_as_uint(acc[1][i]),
                                                   __float_as_uint(acc[2][i]), __float_as_uint(acc[3][i])}, r, o, 0, 0);
    else if constexpr (NTN == 2)
      __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(acc[0][i]), __float_as_uint(acc[1][i])}, r, o, 0, 0);
    else
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[0][i]), r, o, 0, 0);
  }
}

// dW tiles (lane l32: columns d = NTN l32 + nt; rows e = e0 + 8 (i / 4) + 4 g + i % 4): dW2 [e][d] and
// dW1 [d][e], or with nS > 1 their partials, whose rows of E are padded to ldw
template <int D, int DG>
__device__ __forceinline__ void dw_store(const f32x16 (&a1)[D / 32], const f32x16 (&a2)[D / 32], float* __restrict__ dW1,
                                         float* __restrict__ dW2, float* __restrict__ ws, int H, int E, int ldw, int h,
                                         int s, int nS, int e0, int g, int l32) {
  constexpr int NTN = D / 32;
  if (NTN * l32 >= DG) return;
  const int pitch = nS > 1 ? ldw : E;
  float* p2 = (nS > 1 ? ws + ((size_t)s * H + h) * ldw * DG : dW2 + (size_t)h * E * DG) + NTN * l32;
  float* p1 = (nS > 1 ? ws + ((size_t)nS * H + (size_t)s * H + h) * ldw * DG : dW1 + (size_t)h * DG * E) +
              (size_t)(NTN * l32) * pitch;
#pragma unroll
  for (int i4 = 0; i4 < 4; ++i4) {
    const int eb = e0 + 8 * i4 + 4 * g;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      if (eb + m < E) {
        float* q = p2 + (size_t)(eb + m) * DG;
        if constexpr (NTN == 4) *(f32x4*)q = f32x4{a2[0][4 * i4 + m], a2[1][4 * i4 + m], a2[2][4 * i4 + m], a2[3][4 * i4 + m]};
        else if constexpr (NTN == 2) *(float2*)q = float2{a2[0][4 * i4 + m], a2[1][4 * i4 + m]};
        else *q = a2[0][4 * i4 + m];
      }
    }
#pragma unroll
    for (int nt = 0; nt < NTN; ++nt) {
      float* q = p1 + (size_t)nt * pitch + eb;
      if ((pitch & 3) == 0) {
        if (eb < E) *(f32x4*)q = f32x4{a1[nt][4 * i4], a1[nt][4 * i4 + 1], a1[nt][4 * i4 + 2], a1[nt][4 * i4 + 3]};
      } else {
#pragma unroll
        for (int m = 0; m < 4; ++m)
          if (eb + m < E) q[m] = a1[nt][4 * i4 + m];
      }
    }
  }
}

// The rows' walk over E, forward (BWD false: out = O) or dX (BWD true: out = dX): tile t of
// tiles_per_head, 32 rt rows per workgroup.
template <int D, int DG, int ACT, bool BWD>
__device__ __forceinline__ void rows_body(const float* __restrict__ X, const float* __restrict__ W1,
                                          const float* __restrict__ W2, const float* __restrict__ dO,
                                          float* __restrict__ out, int B, int E, int ldw, long long sx, long long sdo,
                                          int tiles_per_head, int ep,
                                          int t) {
  constexpr int NW = f32_nw(D), NTN = D / 32, KJ = DG / 8;
  constexpr int SLOT = 256 * D, W2OFF = 128 * D;
  const int lane = threadIdx.x & 63, g = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int rt = NW / ep, part = wave / rt, rtile = wave - part * rt;
  const int h = t / tiles_per_head, bt = t - h * tiles_per_head;
  const float* Xh = X + (size_t)h * sx;
  const float* W1h = W1 + (size_t)h * DG * ldw;
  const float* W2h = W2 + (size_t)h * E * DG;
  const int b_wave = (bt * rt + rtile) * 32;
  // the parts' shares of the chunks differ by at most one; every part runs the longest one's steps
  // (the barriers are the workgroup's) and computes its own
  const int nch = (E + 31) >> 5;
  const int c0 = part * nch / ep, mine = (part + 1) * nch / ep - c0, steps = (nch + ep - 1) / ep;
  const int ring = part * 2 * SLOT;
  const Lanes<32, 1> l1(g, l32);    // W1c
  const Lanes<D, NTN> l2(g, l32);   // W2c
  const ChunkLoad<D, DG> load_chunk(ldw, lane);

  load_chunk(W1h, W2h, ldw, E, c0, ring, rtile * 64, rt * 64);
  f32x4 xr[KJ], dr[BWD ? KJ : 1];
  const bool ok = b_wave + l32 < B;
#pragma unroll
  for (int j = 0; j < KJ; ++j) {
    const size_t o = (size_t)(b_wave + l32) * DG + 8 * j + 4 * g;
    xr[j] = ok ? *(const f32x4*)(Xh + o) : f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (BWD) dr[j] = ok ? *(const f32x4*)(dO + (size_t)h * sdo + o) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  f32x16 acc[NTN];
#pragma unroll
  for (int nt = 0; nt < NTN; ++nt) acc[nt] = zero16();
  ring_sync();
  for (int c = 0; c < steps; ++c) {
    const int base = ring + (c & 1) * SLOT;
    if (c + 1 < mine) load_chunk(W1h, W2h, ldw, E, c0 + c + 1, ring + ((c + 1) & 1) * SLOT, rtile * 64, rt * 64);
    if (c < mine) {
      // Z^T, then (dX) dH^T with act'(Z) between its products, then the chunk's products with the
      // remaining elements' activations between them, four elements ahead: the matrix core waits
      // only for Z's chain and the first elements
      f32x16 z, dh;
      float v[16];
#pragma unroll
      for (int j = 0; j < KJ; ++j)
#pragma unroll
        for (int m = 0; m < 4; ++m)
          z = mma2(lds_f1(base + l1.col[m] + j * 1024), xr[j][m], j + m == 0 ? zero16() : z);
      if constexpr (BWD) {
        constexpr int EPJ = 16 / KJ;  // elements per four products
#pragma unroll
        for (int j = 0; j < KJ; ++j) {
          const f32x4 w2 = lds_f4(base + W2OFF + l2.row[j & 3] + (j >> 2) * 128);
#pragma unroll
          for (int m = 0; m < 4; ++m) dh = mma2(w2[m], dr[j][m], j + m == 0 ? zero16() : dh);
#pragma unroll
          for (int i = j * EPJ; i < (j + 1) * EPJ; ++i) v[i] = act_d<ACT>(z[i]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      auto elems = [&](int i4) {
#pragma unroll
        for (int i = 4 * i4; i < 4 * i4 + 4; ++i) v[i] = BWD ? dh[i] * v[i] : act_f<ACT>(z[i]);
      };
      elems(0);
      // the chunk's products are summed on their own and then added: a chain of 16 steps and one of
      // E / 32 sums instead of one of E / 2 steps, which halves the rounding error of long sums
      f32x16 p[NTN];
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        if constexpr (BWD) {  // tile nt = columns 32 nt + l32
          f32x4 w1[NTN];
#pragma unroll
          for (int nt = 0; nt < NTN; ++nt) w1[nt] = lds_f4(base + l1.row[i4] + nt * 4096);
#pragma unroll
          for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int nt = 0; nt < NTN; ++nt) p[nt] = mma2(v[4 * i4 + m], w1[nt][m], i4 + m == 0 ? zero16() : p[nt]);
        } else {  // tile nt = columns NTN l32 + nt
#pragma unroll
          for (int m = 0; m < 4; ++m) {
            const VecT<NTN> w2 = lds_vec<NTN>(base + W2OFF + l2.col[m] + i4 * (32 * D));
#pragma unroll
            for (int nt = 0; nt < NTN; ++nt) p[nt] = mma2(v[4 * i4 + m], w2.v[nt], i4 + m == 0 ? zero16() : p[nt]);
          }
        }
        if (i4 < 3) elems(i4 + 1);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int nt = 0; nt < NTN; ++nt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[nt][i] += p[nt][i];
    }
    ring_sync();
  }
  sum_parts<NTN>(acc, ep, part, rtile, rt, lane);
  if (part > 0) return;
  if constexpr (BWD) store_rows<true, D, DG>(acc, out, (size_t)h * B * DG, B, b_wave, g, l32, 1);
  else store_cols<D, DG>(acc, out + (size_t)h * B * DG, B, b_wave, g, l32);
}

// dW program t = (head, B range s, E-tile of 32 cg columns): wave = column group wave % cg, set
// wave / cg of the subtiles (a set takes every rs-th).
template <int D, int DG, int ACT>
__device__ __forceinline__ void dw_body(const float* __restrict__ X, const float* __restrict__ W1,
                                        const float* __restrict__ W2, const float* __restrict__ dO,
                                        float* __restrict__ dW1, float* __restrict__ dW2, float* __restrict__ ws, int H,
                                        int B, int E, int ldw, long long sx, long long sdo,
                                        int cg, int nE, int nS, int rows_per_split, int t) {
  constexpr int NW = f32_nw(D), NTN = D / 32, KJ = DG / 8;
  constexpr int SUB = 128 * D;  // bytes of a [32][D] tile; a set's subtile is X, then dO
  const int lane = threadIdx.x & 63, g = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int rs = NW / cg, set = wave / cg, grp = wave - set * cg;
  const int et = t % nE, hs = t / nE, s = hs % nS, h = hs / nS;
  const int e0 = (et * cg + grp) * 32, e = e0 + l32;
  const int b_lo = s * rows_per_split, b_hi = min(B, b_lo + rows_per_split);
  const int nsub = b_hi > b_lo ? (b_hi - b_lo + 31) / 32 : 0, ngrp = (nsub + rs - 1) / rs;
  const float* Xh = X + (size_t)h * sx;
  const float* dOh = dO + (size_t)h * sdo;
  const int slot_bytes = rs * 2 * SUB;
  const Lanes<D, NTN> lt(g, l32);

  // 64 pieces are RW rows of a tile; the wave's runs in every tile start at the same row mod 8, so a
  // lane's offset inside a run is fixed
  constexpr int RW = 256 / D;
  const int run0 = (wave * 64) % (8 * D) / (D / 4);
  unsigned off;
  {
    const int r = lane / (D / 4), s4 = lane % (D / 4), q = (s4 & ~7) | ((s4 ^ (r + run0)) & 7);
    off = 4 * q < DG ? (unsigned)(r * DG * 4 + q * 16) : BUF_OOB;
  }
  auto issue = [&](int i) {  // subtiles rs i .. of the range into slot i % 2
    const int slot = (i & 1) * slot_bytes;
    for (int p0 = wave * 64; p0 < rs * 16 * D; p0 += NW * 64) {
      const int region = p0 / (8 * D);  // wave-uniform: 2 set + 0 (X) or 1 (dO)
      const int r0 = b_lo + (rs * i + (region >> 1)) * 32 + (p0 - region * 8 * D) / (D / 4);
      buf_load16_lds(make_rsrc_words(((region & 1) ? dOh : Xh) + (size_t)r0 * DG, clamp0(b_hi - r0, RW) * DG * 4), off,
                     slot + p0 * 16);
    }
  };
  if (ngrp > 0) issue(0);
  // the wave's weight operands (B of Z = X W1c and of dH = dO W2c^T: lane = column e)
  f32x4 w1r[KJ], w2r[KJ];
#pragma unroll
  for (int j = 0; j < KJ; ++j) {
    w1r[j] = w2r[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (e < E) {
#pragma unroll
      for (int m = 0; m < 4; ++m) w1r[j][m] = W1[((size_t)h * DG + 8 * j + 4 * g + m) * ldw + e];
      w2r[j] = *(const f32x4*)(W2 + ((size_t)h * E + e) * DG + 8 * j + 4 * g);
    }
  }
  f32x16 a1[NTN], a2[NTN];
#pragma unroll
  for (int nt = 0; nt < NTN; ++nt) {
    a1[nt] = zero16();
    a2[nt] = zero16();
  }
  ring_sync();
  for (int i = 0; i < ngrp; ++i) {
    if (i + 1 < ngrp) issue(i + 1);
    if (rs * i + set < nsub) {
      const int xb = (i & 1) * slot_bytes + set * 2 * SUB, db = xb + SUB;
      // Z, then dH with h and act'(Z) between its products, then the dW products, dZ first
      f32x16 z, dh;
      float hv[16], dz[16];
#pragma unroll
      for (int j = 0; j < KJ; ++j) {
        const f32x4 xa = lds_f4(xb + lt.row[j & 3] + (j >> 2) * 128);
#pragma unroll
        for (int m = 0; m < 4; ++m) z = mma2(xa[m], w1r[j][m], j + m == 0 ? zero16() : z);
      }
      constexpr int EPJ = 16 / KJ;
#pragma unroll
      for (int j = 0; j < KJ; ++j) {
        const f32x4 da = lds_f4(db + lt.row[j & 3] + (j >> 2) * 128);
#pragma unroll
        for (int m = 0; m < 4; ++m) dh = mma2(da[m], w2r[j][m], j + m == 0 ? zero16() : dh);
#pragma unroll
        for (int k = j * EPJ; k < (j + 1) * EPJ; ++k) act_hf<ACT>(z[k], hv[k], dz[k]);
        __builtin_amdgcn_sched_barrier(0);
      }
      // per subtile a sum of its own, as in rows_body; dZ between dW2's products
      f32x16 p[NTN];
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const VecT<NTN> d = lds_vec<NTN>(db + lt.col[k & 3] + (k >> 2) * (32 * D));
#pragma unroll
        for (int nt = 0; nt < NTN; ++nt) p[nt] = mma2(hv[k], d.v[nt], k == 0 ? zero16() : p[nt]);
        dz[k] *= dh[k];
      }
#pragma unroll
      for (int nt = 0; nt < NTN; ++nt)
#pragma unroll
        for (int k = 0; k < 16; ++k) a2[nt][k] += p[nt][k];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const VecT<NTN> x = lds_vec<NTN>(xb + lt.col[k & 3] + (k >> 2) * (32 * D));
#pragma unroll
        for (int nt = 0; nt < NTN; ++nt) p[nt] = mma2(dz[k], x.v[nt], k == 0 ? zero16() : p[nt]);
      }
#pragma unroll
      for (int nt = 0; nt < NTN; ++nt)
#pragma unroll
        for (int k = 0; k < 16; ++k) a1[nt][k] += p[nt][k];
    }
    ring_sync();
  }
  // the sets' sums: both accumulators of sets 1 .. go to set 0 one after the other
  sum_parts<NTN>(a2, rs, set, grp, cg, lane);
  if (rs > 1) __syncthreads();
  sum_parts<NTN>(a1, rs, set, grp, cg, lane);
  if (set == 0) dw_store<D, DG>(a1, a2, dW1, dW2, ws, H, E, ldw, h, s, nS, e0, g, l32);
}

template <int D, int DG, int ACT>
__global__ void __launch_bounds__(f32_nw(D) * 64) __attribute__((amdgpu_waves_per_eu(f32_nw(D) / 4, f32_nw(D) / 4)))
f32_fwd_kernel(const float* __restrict__ X, const float* __restrict__ W1, const float* __restrict__ W2,
               float* __restrict__ O, int B, int E, int ldw, long long sx, long long sdo, int tiles_per_head,
               int ep) {
  rows_body<D, DG, ACT, false>(X, W1, W2, nullptr, O, B, E, ldw, sx, sdo,
                               tiles_per_head, ep, xcd_remap(blockIdx.x, gridDim.x));
}

template <int D, int DG, int ACT>
__global__ void __launch_bounds__(f32_nw(D) * 64) __attribute__((amdgpu_waves_per_eu(f32_nw(D) / 4, f32_nw(D) / 4)))
f32_bwd_kernel(const float* __restrict__ X, const float* __restrict__ W1, const float* __restrict__ W2,
               const float* __restrict__ dO, float* __restrict__ dX, float* __restrict__ dW1, float* __restrict__ dW2,
               float* __restrict__ ws, int H, int B, int E, int ldw, long long sx, long long sdo, int tiles_per_head,
               int ep, int n_dx, int dx_first,
               int cg, int nE, int nS, int rows_per_split) {
  const int b = blockIdx.x, n_dw = (int)gridDim.x - n_dx;
  const int bx = dx_first ? b : b - n_dw;  // index among the dX programs
  if (bx >= 0 && bx < n_dx) {
    rows_body<D, DG, ACT, true>(X, W1, W2, dO, dX, B, E, ldw, sx, sdo, tiles_per_head, ep, xcd_remap(bx, n_dx));
  } else {
    dw_body<D, DG, ACT>(X, W1, W2, dO, dW1, dW2, ws, H, B, E, ldw, sx, sdo, cg, nE, nS, rows_per_split,
                        xcd_remap(dx_first ? b - n_dx : b, n_dw));
  }
}

// ------------------------------------------------------------------------------------
// plans and launches
// ------------------------------------------------------------------------------------
constexpr int kMaxLds = 160 * 1024;
// LDS of a rows program (ep rings of two chunks; at least the parts' sums) and of a dW program
int rows_lds(int D, int ep) { return std::max(ep * 512 * D, (f32_nw(D) - f32_nw(D) / ep) * (D / 32) * 4096); }
int dw_lds(int D, int cg) {
  const int nw = f32_nw(D), rs = nw / cg;
  return std::max(rs * 512 * D, (nw - cg) * (D / 32) * 4096);
}

// E parts of a rows program: the least (rounds of workgroups over the CUs) x (steps of a part, plus
// one for the program's start and end). The same for every call of a shape, so dX does not depend
// on the workspace.
int rows_parts(int64_t H, int64_t B, int D, int64_t E, int num_cus) {
  const long long nch = (E + 31) / 32, N = num_cus > 0 ? num_cus : 1;
  int best = 1;
  double cost = 1e300;
  for (int ep = 1; ep <= f32_nw(D) && ep <= nch; ep *= 2) {
    if (rows_lds(D, ep) > kMaxLds) break;
    const long long rows = 32LL * (f32_nw(D) / ep), wgs = H * ((B + rows - 1) / rows);
    const double c = (double)((wgs + N - 1) / N) * (double)((nch + ep - 1) / ep + 1);
    if (c < cost) {
      cost = c;
      best = ep;
    }
  }
  return best;
}

constexpr double kStepUs = 0.029;  // one 32x32x2 fp32 product on a SIMD, with what surrounds it
constexpr double kFixedUs = 3.0;   // a program's start and end
constexpr double kLaunchUs = 4.0, kHbmBytesPerUs = 5.0e6;

int tile_d(int64_t D) { return D < 32 ? 32 : (int)D; }

F32Plan make_plan(int64_t H, int64_t B, int64_t Dg, int64_t E, int num_cus, size_t max_ws) {
  const int D = tile_d(Dg), nw = f32_nw(D), wps = nw / 4;
  const long long N = num_cus > 0 ? num_cus : 1, nch = (E + 31) / 32;
  F32Plan p{};
  p.ep = rows_parts(H, B, D, E, num_cus);
  const long long rows = 32LL * (nw / p.ep);
  p.dx_tiles_per_head = (int)((B + rows - 1) / rows);
  p.n_dx = H * (long long)p.dx_tiles_per_head;
  const double tx = kFixedUs + (double)wps * ((nch + p.ep - 1) / p.ep) * 1.5 * (double)Dg * kStepUs;
  double best = 0.0;
  for (int cg = std::min(4, nw); cg >= 1; cg /= 2) {
    if (dw_lds(D, cg) > kMaxLds) break;
    const int rs = nw / cg;
    const long long nE = (E + 32 * cg - 1) / (32 * cg), max_ns = std::max<long long>(1, B / (64 * rs));
    for (long long ns = 1; ns <= max_ns && H * nE * ns <= std::max<long long>(4 * N, H * nE); ns += 1 + ns / 4) {
      long long rps = ((B + ns - 1) / ns + 31) / 32 * 32;
      if (rps < 32) rps = 32;
      const long long eff = std::max<long long>(1, (B + rps - 1) / rps);
      const size_t ws = eff > 1 ? (size_t)2 * eff * H * w1_pitch(E, 4) * Dg * sizeof(float) : 0;
      if (ws > max_ws) continue;
      const double tw = kFixedUs + (double)wps * ((rps + 32 * rs - 1) / (32 * rs)) * 2.0 * (double)Dg * kStepUs;
      const double red = eff > 1 ? kLaunchUs + 1.2 * (double)ws / kHbmBytesPerUs : 0.0;
      for (int o = 0; o < 2; ++o) {
        const double t = red + (o ? list_makespan(p.n_dx, tx, H * nE * eff, tw, N)
                                  : list_makespan(H * nE * eff, tw, p.n_dx, tx, N));
        if (best == 0.0 || t < best) {
          best = t;
          p.cg = cg;
          p.nE = (int)nE;
          p.nS = (int)eff;
          p.rows_per_split = (int)rps;
          p.dx_first = o == 1;
          p.n_dw = H * nE * eff;
          p.ws_bytes = ws;
        }
      }
    }
  }
  return p;
}

}  // namespace

// Plans are computed once per distinct call shape (a small cache of recent ones).
F32Plan plan_f32_bwd(int64_t H, int64_t B, int64_t D, int64_t E, int num_cus, size_t max_ws) {
  struct Entry {
    int64_t H, B, D, E;
    int cus;
    size_t max_ws;
    F32Plan plan;
  };
  static std::mutex mu;
  static Entry cache[16];
  static int used = 0, next = 0;
  {
    std::lock_guard<std::mutex> lock(mu);
    for (int i = 0; i < used; ++i) {
      const Entry& c = cache[i];
      if (c.H == H && c.B == B && c.D == D && c.E == E && c.cus == num_cus && c.max_ws == max_ws) return c.plan;
    }
  }
  const F32Plan p = make_plan(H, B, D, E, num_cus, max_ws);
  std::lock_guard<std::mutex> lock(mu);
  cache[next] = Entry{H, B, D, E, num_cus, max_ws, p};
  next = (next + 1) % 16;
  if (used < 16) ++used;
  return p;
}

namespace {

template <int D, int DG, int ACT>
hipError_t fwd_t(const FwdArgs& a, hipStream_t st) {
  const int ep = rows_parts(a.H, a.B, D, a.E, a.num_cus);
  const long long rows = 32LL * (f32_nw(D) / ep), tph = (a.B + rows - 1) / rows, grid = tph * a.H;
  if (grid <= 0) return hipSuccess;
  if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
  auto k = f32_fwd_kernel<D, DG, ACT>;
  static std::atomic<unsigned long long> lds_set{0};
  const hipError_t e = set_lds_once((const void*)k, kMaxLds, lds_set);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(f32_nw(D) * 64), rows_lds(D, ep), st, (const float*)a.x,
                     (const float*)a.w1, (const float*)a.w2, (float*)a.o, (int)a.B, (int)a.E, (int)a.ldw,
                     (long long)a.sx, 0LL, (int)tph, ep);
  return hipGetLastError();
}

template <int D, int DG, int ACT>
hipError_t bwd_t(const BwdArgs& a, const F32Plan& p, hipStream_t st) {
  const long long n_dx = a.want_dx ? p.n_dx : 0, n_dw = a.want_dw ? p.n_dw : 0, grid = n_dx + n_dw;
  if (grid <= 0) return hipSuccess;
  if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
  auto k = f32_bwd_kernel<D, DG, ACT>;
  static std::atomic<unsigned long long> lds_set{0};
  hipError_t e = set_lds_once((const void*)k, kMaxLds, lds_set);
  if (e != hipSuccess) return e;
  const int lds = std::max(n_dx > 0 ? rows_lds(D, p.ep) : 0, n_dw > 0 ? dw_lds(D, p.cg) : 0);
  hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(f32_nw(D) * 64), lds, st, (const float*)a.x, (const float*)a.w1,
                     (const float*)a.w2, (const float*)a.dout, (float*)a.dx, (float*)a.dw1, (float*)a.dw2, (float*)a.ws,
                     (int)a.H, (int)a.B, (int)a.E, (int)a.ldw, (long long)a.sx, (long long)a.sdo,
                     p.dx_tiles_per_head, p.ep, (int)n_dx, p.dx_first ? 1 : 0,
                     p.cg, p.nE, p.nS, p.rows_per_split);
  if ((e = hipGetLastError()) != hipSuccess || n_dw == 0) return e;
  return launch_dw_reduce_f32(a, p.nS, st);
}

template <int D, int DG>
hipError_t fwd_a(const FwdArgs& a, hipStream_t st) {
  switch (a.act) {
    case ACT_SILU: return fwd_t<D, DG, ACT_SILU>(a, st);
    case ACT_LEAKY: return fwd_t<D, DG, ACT_LEAKY>(a, st);
    case ACT_SIGMOID: return fwd_t<D, DG, ACT_SIGMOID>(a, st);
    default: return fwd_t<D, DG, ACT_NONE>(a, st);
  }
}
template <int D, int DG>
hipError_t bwd_a(const BwdArgs& a, const F32Plan& p, hipStream_t st) {
  switch (a.act) {
    case ACT_SILU: return bwd_t<D, DG, ACT_SILU>(a, p, st);
    case ACT_LEAKY: return bwd_t<D, DG, ACT_LEAKY>(a, p, st);
    case ACT_SIGMOID: return bwd_t<D, DG, ACT_SIGMOID>(a, p, st);
    default: return bwd_t<D, DG, ACT_NONE>(a, p, st);
  }
}

}  // namespace

hipError_t launch_f32_fwd(const FwdArgs& a, hipStream_t st) {
  switch (a.D) {
    case 16: return fwd_a<32, 16>(a, st);
    case 32: return fwd_a<32, 32>(a, st);
    case 64: return fwd_a<64, 64>(a, st);
    case 128: return fwd_a<128, 128>(a, st);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_f32_bwd(const BwdArgs& a, const F32Plan& p, hipStream_t st) {
  switch (a.D) {
    case 16: return bwd_a<32, 16>(a, p, st);
    case 32: return bwd_a<32, 32>(a, p, st);
    case 64: return bwd_a<64, 64>(a, p, st);
    case 128: return bwd_a<128, 128>(a, p, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace fmlp
