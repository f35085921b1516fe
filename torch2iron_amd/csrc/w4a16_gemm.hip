// Prompt-sized W4A16 GEMM for gfx950: y[M, N] = x[M, K] . W^T for some tens to thousands of
// rows, over the AutoGPTQ words.  (w4a16_linear.hip holds the 64 x 128 kernel that stays
// where it is the faster one; plan_prompt chooses.)
//
// A workgroup has WN waves along N and WK slices of K; a wave computes 16 MF rows x 16 NJ
// columns, a lane NJ consecutive columns (so pairs meet in a lane and results are stored
// from registers).  A step is one quantisation group (128 of K).
//   * Every operand of a step comes by loads into LDS, three tiles deep (a step's tile is
//     requested two steps ahead, its words three), counted by hand: a step ends when all but
//     its last requests, the words three steps ahead, have landed.
//   * A packed word becomes eight bf16 (144 + q - z): nibbles to bytes, 16 - z added to all
//     four bytes of a half, then each pair under the exponent byte 0x43: eleven VALU
//     instructions.  The bias is the same for every column, so the zero-point correction is
//     -144 x the row's sum over the group, which is where the accumulators start: one FMA
//     per output and group (total += scale * acc) instead of two.  A wave sums the rows of
//     one fragment of the next tile with MFMAs against bf16 -144 (or takes given sums), so
//     each row is summed once a workgroup and not once a wave.  It begins its steps with that
//     fragment, whose sums it still holds; the others' come through LDS behind the step's
//     barrier.  So every accumulator starts at its row sums: equal rows give equal bits
//     wherever they stand in the call.
//   * Step s + 1's words are unpacked beside step s's MFMAs, the previous fragment's sums
//     are folded beside the next one's, loads go out one every few MFMAs.  The order is the
//     program's (empty asm ties; the compiler otherwise sinks the folds and unpacking behind
//     the MFMAs and spills: 256 registers and scratch against 225 and none).
//   * The two waves of a SIMD step down in priority through a step, so the one that is
//     behind goes first; without it the older one runs ahead and waits at the step's barrier
//     while the other runs alone (497 -> 470 us at 8192 x 2048 x 12288 when it was added).
// What bounds it: instruction issue.  At 8192 x 2048 x 12288 (128 x 256 tiles) MFMAs take 47 % of
// the cycles of a SIMD that holds waves and VALU instructions 42 % beside them (unpacking,
// folding); the LDS index unit is busy for 35 % and waves wait to issue to it for 4 % of theirs.  A
// short K adds the prologue and the epilogue of its one workgroup a CU: MFMAs 32 % of the fused
// q|k|v projection at K = 1024.  Wider waves (64 columns) need more than 256 registers: one wave a SIMD then, measured slower
// (536 us).  Against the 64 x 128 kernel (us, M x K x N, graph-launched in turn): gate_up 8192 x
// 2048 x 12288 584 -> 438, down 4001 x 6144 x 2048 146 -> 103, 8192 x 2048 x 4096 190 -> 164, 8192
// x 1024 x 4096 107 -> 104; against the decode tiles, gate_up 331 x 2048 x 12288 52 -> 33.
#include <type_traits>

#include "t2i_common.h"
#include "w4a16_tile.h"
#include "prompt_plan.h"
#include "qk_prep.h"

namespace t2i {

constexpr float GM_BIAS = 144.0f;   // what an unpacked weight carries: 144 + (q - z)

constexpr int GM_RING = 3;          // k tiles in LDS

template <int MF, int NJ, int WN, int WK, int XSP>
struct GemmShape {
  static constexpr int BM = 16 * MF, BN = 16 * NJ * WN;
  static constexpr int WAVES = WN * WK, THREADS = 64 * WAVES;
  static constexpr int A_BYTES = BM * GS * 2;            // one slice's activation tile
  static constexpr int W_BYTES = GS / 8 * BN * 4;        // and its packed words
  // its scales, zero words and precomputed row sums, in pieces of 256 bytes
  static constexpr int P_SC = BN / 128, P_Z = 1, P_XS = BM > 64 ? BM / 64 : 1;
  static constexpr int PIECES = P_SC + P_Z + XSP * P_XS;
  static constexpr int S_BYTES = PIECES * 256;
  static constexpr int X_BYTES = 2 * BM * 4;             // -144 x the row sums, two steps
  static constexpr int STAGES = WK * (GM_RING * (A_BYTES + W_BYTES + S_BYTES) + X_BYTES);
  static constexpr int PART = WK > 1 ? WAVES * MF * NJ * 1024 : 0;      // the slices' partial sums
  static constexpr int TILE = BM * (BN + 8) * 2;                        // the bf16 tile of EPI_QKV_PREP
  static constexpr int LDS = STAGES > PART ? (STAGES > TILE ? STAGES : TILE) : (PART > TILE ? PART : TILE);
  // loads into LDS a wave issues each step
  static constexpr int OPS_A = KSG, OPS_W = W_BYTES / 1024 / WN, OPS_S = (PIECES + WN - 1) / WN;
  static constexpr int OPS = OPS_A + OPS_S + OPS_W;
  static_assert(MF == WN && (MF & (MF - 1)) == 0 && MF % WK == 0, "a row fragment a wave, whole pieces");
  static_assert(NJ == 2, "the epilogue stores a pair of columns a lane");
  static_assert(BN % 128 == 0 && ATT_D == 128, "whole heads and half groups of output sums a tile");
  static_assert(W_BYTES % (1024 * WN) == 0 && OPS_S <= 2, "the same number of loads in every wave");
};

// A word's eight weights as bf16(144 + q - z) in k order: nibbles spread to bytes
// (two permutes over w and w >> 4, one mask a half), 16 - z added to every byte, and
// each pair of bytes put under the exponent byte 0x43 by one permute.
__device__ __forceinline__ bf16x8 gemm_unpack(uint32_t w, uint32_t add, uint32_t exp4) {
  const uint32_t w4 = w >> 4;
  const uint32_t lo = (__builtin_amdgcn_perm(w4, w, 0x05010400u) & 0x0F0F0F0Fu) + add;   // k0 k1 k2 k3
  const uint32_t hi = (__builtin_amdgcn_perm(w4, w, 0x07030602u) & 0x0F0F0F0Fu) + add;   // k4 k5 k6 k7
  u32x4 d;
  d.x = __builtin_amdgcn_perm(exp4, lo, 0x04010400u);
  d.y = __builtin_amdgcn_perm(exp4, lo, 0x04030402u);
  d.z = __builtin_amdgcn_perm(exp4, hi, 0x04010400u);
  d.w = __builtin_amdgcn_perm(exp4, hi, 0x04030402u);
  return __builtin_bit_cast(bf16x8, d);
}

// The same in four parts, to be spread between MFMAs.
struct GemmUnpack {
  uint32_t w4, lo, hi;
  u32x4 d;
  __device__ __forceinline__ void part(int q, uint32_t w, uint32_t add, uint32_t exp4) {
    if (q == 0) {
      w4 = w >> 4;
      lo = (__builtin_amdgcn_perm(w4, w, 0x05010400u) & 0x0F0F0F0Fu) + add;
      asm volatile("" : "+v"(lo), "+v"(w4));
    } else if (q == 1) {
      d.x = __builtin_amdgcn_perm(exp4, lo, 0x04010400u);
      d.y = __builtin_amdgcn_perm(exp4, lo, 0x04030402u);
      hi = (__builtin_amdgcn_perm(w4, w, 0x07030602u) & 0x0F0F0F0Fu) + add;
      asm volatile("" : "+v"(d.x), "+v"(d.y), "+v"(hi));
    } else if (q == 2) {
      d.z = __builtin_amdgcn_perm(exp4, hi, 0x04010400u);
      asm volatile("" : "+v"(d.z));
    } else {
      d.w = __builtin_amdgcn_perm(exp4, hi, 0x04030402u);
      asm volatile("" : "+v"(d.w));
    }
  }
  __device__ __forceinline__ bf16x8 value() const { return __builtin_bit_cast(bf16x8, d); }
};

typedef __attribute__((ext_vector_type(4))) int i32x4;

// A buffer over everything from p on: loads at a byte offset a lane plus a uniform one
// (every offset used is inside the tensor: rows and groups are clamped).
__device__ __forceinline__ i32x4 tile_rsrc(const void* p) {
  const uint64_t a = (uint64_t)(uintptr_t)p;
  return i32x4{(int)__builtin_amdgcn_readfirstlane((uint32_t)a), (int)(__builtin_amdgcn_readfirstlane((uint32_t)(a >> 32)) & 0xFFFF), -1, 0x00027000};
}
// One 16-byte (dma4: 4-byte) piece a lane into LDS at lds + 16 (4) lane, written as asm so
// that the compiler's own waits (it waits for every load into LDS before any LDS read)
// leave it in flight; dma_wait covers it.  M0 takes the LDS address, with a wait state before
// the load.  The compiler does not look into asm for hazards: an SGPR that a VALU instruction
// wrote (a v_readfirstlane) is five wait states away from a VMEM instruction that reads it, and
// the two moves and the s_nop are five whatever stands before them (without the s_nop, whose
// place nothing the compiler emitted here needed, 0.2 to 0.5 % faster).  lanes: all (~0) or none
// (0: nothing is read or written, and nothing is assumed of when such a load counts or leaves the
// count: waits past one wait for everything); every call is made by whole waves, so all lanes
// are on again after it.
__device__ __forceinline__ void dma16(i32x4 rsrc, uint32_t off, uint32_t soff, uint32_t lds, uint64_t lanes) {
  asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %4\n\ts_nop 2\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds\n\ts_mov_b64 exec, -1"
               :: "s"(lds), "v"(off), "s"(rsrc), "s"(soff), "s"(lanes) : "memory", "m0");
}
__device__ __forceinline__ void dma4(i32x4 rsrc, uint32_t off, uint32_t soff, uint32_t lds, uint64_t lanes) {
  asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %4\n\ts_nop 2\n\tbuffer_load_dword %1, %2, %3 offen lds\n\ts_mov_b64 exec, -1"
               :: "s"(lds), "v"(off), "s"(rsrc), "s"(soff), "s"(lanes) : "memory", "m0");
}
// Until at most N of this wave's vector memory operations are in flight.
template <int N>
__device__ __forceinline__ void dma_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

template <int MF, int NJ, int WN, int WK, int XSP>
__global__ __launch_bounds__(64 * WN * WK, 2) void w4a16_prompt_kernel(const LinearParams p, const QkvPrepParams pp) {
  using S = GemmShape<MF, NJ, WN, WK, XSP>;
  constexpr int BM = S::BM, BN = S::BN;
  __shared__ __align__(16) unsigned char smem[S::LDS];
  unsigned char* const s_a = smem;                                    // [RING][WK] activation tiles
  unsigned char* const s_w = s_a + GM_RING * WK * S::A_BYTES;         // [RING][WK] packed words [16][BN]
  unsigned char* const s_s = s_w + GM_RING * WK * S::W_BYTES;         // [RING][WK] scales, zeros, row sums
  float* const s_x = reinterpret_cast<float*>(s_s + GM_RING * WK * S::S_BYTES);   // [2][WK][BM] -144 x row sums

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN, wk = wave / WN;
  const int c = lane & 15, r = lane >> 4;

  // tiles: each XCD takes one contiguous range; inside it, groups of 4 row tiles
  // column by column
  const int MT = (p.M + BM - 1) / BM, NT = p.N / BN, T = MT * NT;
  const int xcd = blockIdx.x & 7, base = T >> 3, rem = T & 7;
  const int t = xcd * base + min(xcd, rem) + (blockIdx.x >> 3);
  constexpr int GR = 4;
  const int grp = t / (GR * NT), in = t - grp * GR * NT;
  const int rows_in = min(GR, MT - grp * GR);
  const int m0 = (grp * GR + in % rows_in) * BM, n0 = (in / rows_in) * BN;
  const int lcol = wn * 16 * NJ + NJ * c;           // the lane's NJ columns of the tile
  const int ncol = n0 + lcol;

  const int groups = p.K / GS;
  const int steps = (groups + WK - 1) / WK;
  auto group_of = [&](int s) { return min(s * WK + wk, groups - 1); };

  // ---- loads into LDS (every offset stays inside the tensors: rows and groups are clamped) ----
  // Activations: the wave brings row fragment wn of its slice, one MFMA A operand
  // (lane (c, r): row c, k 32 ks + 8 r ..) a load.
  const int mlim = p.M - 1 - m0;
  const i32x4 xrsrc = tile_rsrc(p.x + (size_t)m0 * p.ldx);
  uint32_t xoff[KSG];
#pragma unroll
  for (int ks = 0; ks < KSG; ++ks)
    xoff[ks] = (uint32_t)min(16 * wn + c, mlim) * (uint32_t)(p.ldx * 2) + 16u * r + 64u * ks;
  // Packed words: 1 KB of the tile's [16][BN] a load.
  constexpr int WROWS = 256 / BN;   // word rows a load covers (BN = 128: 2)
  static_assert(BN == 128 || BN == 256, "whole word rows a load");
  const i32x4 wrsrc = tile_rsrc(p.qw + n0);
  const uint32_t woff = (uint32_t)(wn * S::OPS_W * WROWS + lane / (64 / WROWS)) * (uint32_t)(p.N * 4) + 16u * (lane % (64 / WROWS));
  // Pieces of scales, zeros and row sums: piece wn + WN i of the slice (past the last: the first again).
  i32x4 prsrc[S::OPS_S];
  uint32_t pstride[S::OPS_S], poff[S::OPS_S], plds[S::OPS_S];
  bool is_xs[S::OPS_S];
#pragma unroll
  for (int i = 0; i < S::OPS_S; ++i) {
    const int piece = wn + WN * i < S::PIECES ? wn + WN * i : 0;
    const unsigned char* src;
    is_xs[i] = XSP > 0 && piece > S::P_SC;
    if (piece < S::P_SC) {
      src = reinterpret_cast<const unsigned char*>(p.sc + n0 + 128 * piece);
      pstride[i] = (uint32_t)p.N * 2;
      poff[i] = 4u * lane;
    } else if (!is_xs[i]) {
      src = reinterpret_cast<const unsigned char*>(p.qz + (n0 >> 3));
      pstride[i] = (uint32_t)(p.N >> 3) * 4;
      poff[i] = 4u * min(lane, BN / 8 - 1);
    } else {
      const int u = (piece - S::P_SC - 1) / S::P_XS, h = (piece - S::P_SC - 1) % S::P_XS;
      src = reinterpret_cast<const unsigned char*>(p.xs + (size_t)u * p.ldxs + m0);
      pstride[i] = (uint32_t)XSP * p.ldxs * 4;
      poff[i] = 4u * min(min(64 * h + lane, BM - 1), mlim);
    }
    prsrc[i] = tile_rsrc(src);
    plds[i] = lds_address(s_s) + wk * S::S_BYTES + piece * 256;
  }
  const uint32_t lds_a = lds_address(s_a) + wk * S::A_BYTES + wn * S::OPS_A * 1024;
  const uint32_t lds_w = lds_address(s_w) + wk * S::W_BYTES + wn * S::OPS_W * 1024;
  const uint32_t wrow = (uint32_t)p.N * 4u;         // bytes of a word row
  // Steps past the last load nothing; an odd count's extra step loads the last group again (its
  // scales are zero, so it adds nothing as long as its products are finite whenever the last's are).
  const int loads = (steps + 1) & ~1;
  auto lanes_of = [&](int s) -> uint64_t {
    const uint32_t v = __builtin_amdgcn_readfirstlane(s < loads ? ~0u : 0u);
    return (uint64_t)v << 32 | v;
  };
  auto load_a = [&](int s, int slot, int q) {
    dma16(xrsrc, xoff[q], (uint32_t)group_of(s) * (GS * 2), lds_a + slot * WK * S::A_BYTES + q * 1024,
          lanes_of(s));
  };
  auto load_w = [&](int s, int slot, int q) {
    dma16(wrsrc, woff, (uint32_t)(16 * group_of(s) + q * WROWS) * wrow, lds_w + slot * WK * S::W_BYTES + q * 1024,
          lanes_of(s));
  };
  // step s's scales and zeros, or (row sums come with their tile, a step later) step s - 1's row sums
  auto load_s = [&](int s, int slot, int before, int i) {
    const int st = is_xs[i] ? s - 1 : s;
    dma4(prsrc[i], poff[i], __builtin_amdgcn_readfirstlane((uint32_t)group_of(st) * pstride[i]),
         __builtin_amdgcn_readfirstlane(plds[i] + (is_xs[i] ? before : slot) * WK * S::S_BYTES), lanes_of(st));
  };

  // ---- LDS reads ----
  // The wave takes the tile's row fragments from its own on: its fragment k is row fragment row_frag(k).
  auto row_frag = [&](int k) { return (wn + k) & (MF - 1); };
  const uint32_t aoff = wk * S::A_BYTES + 16 * lane;
  auto read_a = [&](int slot, int u) {   // unit u: k-step u % KSG of the wave's fragment u / KSG
    return *reinterpret_cast<const u32x4*>(s_a + slot * WK * S::A_BYTES + row_frag(u / KSG) * (KSG * 1024) + aoff +
                                           u % KSG * 1024);
  };
  auto read_w = [&](int slot, int ks, uint32_t (&w)[NJ]) {
    load_words<NJ>(reinterpret_cast<const uint32_t*>(s_w + (slot * WK + wk) * S::W_BYTES) + (4 * ks + r) * BN + lcol, w);
  };
  uint32_t exp4 = 0x43434343u;
  asm volatile("" : "+v"(exp4));
  // 16 - z of the lane's columns of step s in every byte, and their scales (zero for a step
  // past the slice's last group, which then adds nothing)
  auto read_sz = [&](int s, int slot, uint32_t (&add)[NJ], float (&sc)[NJ]) {
    const unsigned char* src = s_s + (slot * WK + wk) * S::S_BYTES;
    uint32_t sr[NJ / 2];
    load_scales<NJ>(reinterpret_cast<const uint16_t*>(src) + lcol, sr);
    const uint32_t zw = ~*reinterpret_cast<const uint32_t*>(src + S::P_SC * 256 + (lcol >> 3) * 4) >> ((lcol & 7) * 4);
    const bool live = s * WK + wk < groups;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      add[j] = ((zw >> (4 * j)) & 15u) * 0x01010101u;
      sc[j] = live ? f16_to_f32(half_of<NJ>(sr, j, false)) : 0.0f;
      asm volatile("" : "+v"(add[j]), "+v"(sc[j]));
    }
  };
  // -144 x the row sums, the accumulators' start: of the wave's fragment k (rows 4 r .. of it) ...
  auto xs_at = [&](int par, int k) {
    return reinterpret_cast<f32x4*>(s_x + (par * WK + wk) * BM + 16 * row_frag(k) + 4 * r);
  };
  // ... and, for its first fragment, from the precomputed sums (XSP > 0), or by MFMAs of the
  // fragment (units a) against bf16 -144.
  auto given_xs = [&](int slot) {
    const unsigned char* src = s_s + (slot * WK + wk) * S::S_BYTES + (S::P_SC + 1) * 256 + (16 * wn + 4 * r) * 4;
    f32x4 v = *reinterpret_cast<const f32x4*>(src);
    if constexpr (XSP == 2) {
      const f32x4 v2 = *reinterpret_cast<const f32x4*>(src + S::P_XS * 256);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] += v2[i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] *= -GM_BIAS;
    return v;
  };
  const u32x4 mbias = {0xC310C310u, 0xC310C310u, 0xC310C310u, 0xC310C310u};   // bf16 -144
  auto sum_unit = [&](u32x4 a, f32x4 xs) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, mbias), xs,
                                                   0, 0, 0);
  };

  f32x4 total[MF][NJ];
#pragma unroll
  for (int k = 0; k < MF; ++k)
#pragma unroll
    for (int j = 0; j < NJ; ++j) total[k][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 B0[KSG][NJ], B1[KSG][NJ];
  float sc0[NJ], sc1[NJ];

  // ---- prologue: step 0's tile and weights, then step 1's, then step 2's words; step 0's
  // row sums and unpacked weights while the later ones come ----
#pragma unroll
  for (int q = 0; q < S::OPS_W; ++q) load_w(0, 0, q);
#pragma unroll
  for (int i = 0; i < S::OPS_S; ++i) load_s(is_xs[i] ? 1 : 0, 0, 0, i);
#pragma unroll
  for (int q = 0; q < S::OPS_A; ++q) load_a(0, 0, q);
#pragma unroll
  for (int q = 0; q < S::OPS_W; ++q) load_w(1, 1, q);
#pragma unroll
  for (int i = 0; i < S::OPS_S; ++i) load_s(is_xs[i] ? 2 : 1, 1, 1, i);
#pragma unroll
  for (int q = 0; q < S::OPS_A; ++q) load_a(1, 1, q);
#pragma unroll
  for (int i = 0; i < S::OPS_S; ++i) load_s(2, 2, 1, i);
#pragma unroll
  for (int q = 0; q < S::OPS_W; ++q) load_w(2, 2, q);
  if (loads > 2) dma_wait<S::OPS + S::OPS_S + S::OPS_W>();
  else dma_wait<0>();          // (steps 2 and on are switched off)
  __syncthreads();
  f32x4 xown = {0.f, 0.f, 0.f, 0.f};   // the start of the wave's first fragment in the step to come
  if constexpr (XSP > 0) {
    xown = given_xs(0);
  } else {
#pragma unroll
    for (int ks = 0; ks < KSG; ++ks) xown = sum_unit(read_a(0, ks), xown);
  }
  if (c == 0) *xs_at(0, 0) = xown;
  {
    uint32_t add[NJ], w[KSG][NJ];
    read_sz(0, 0, add, sc0);
#pragma unroll
    for (int ks = 0; ks < KSG; ++ks) read_w(0, ks, w[ks]);
#pragma unroll
    for (int ks = 0; ks < KSG; ++ks)
#pragma unroll
      for (int j = 0; j < NJ; ++j) B0[ks][j] = gemm_unpack(w[ks][j], add[j], exp4);
#pragma unroll
    for (int ks = 0; ks < KSG; ++ks)
#pragma unroll
      for (int j = 0; j < NJ; ++j) asm volatile("" : "+v"(B0[ks][j]));
  }
  if (loads > 2) dma_wait<S::OPS_W>();   // behind it: step 2's words
  else dma_wait<0>();
  __syncthreads();             // (slot 0's words are consumed: step 0 loads step 3's there)

  // The first AHEAD k-steps' fragments are read before the step, its last fragment's sums are
  // carried into total during the next step (scp: their scales).
  constexpr int AHEAD = KSG + 2, RINGA = 2 * KSG;   // reads run this many k-steps ahead of their MFMAs
  constexpr int UNITS = KSG * MF;
  static_assert(UNITS % RINGA == 0 && MF > 1, "the ring of fragments starts every step at its first slot");
  u32x4 a[RINGA];
  f32x4 P[2][NJ];
  float scp[NJ];
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) a[u] = read_a(0, u);
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    P[0][j] = P[1][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    scp[j] = 0.0f;
  }
  auto step = [&](auto PAR, int s, int b0, int b1, int b2, bf16x8 (&B)[KSG][NJ], float (&sc)[NJ], bf16x8 (&Bn)[KSG][NJ],
                  float (&scn)[NJ]) {
    constexpr int par = decltype(PAR)::value;
    constexpr int NW = KSG * NJ, SLOTS = (MF - 1) * NW;   // words a lane, MFMAs after fragment 0
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    u32x4 an[KSG];
    f32x4 xv[4], xs = zero;
    uint32_t w[KSG][NJ], addn[NJ];
    GemmUnpack un[NW];
    // element e of fragment q: its sums v under the scales sv
    auto fma1 = [&](int q, int e, float v, const float (&sv)[NJ]) {
      const int j = e >> 2, i = e & 3;
      float y = fmaf(sv[j], v, total[q][j][i]);
      asm volatile("" : "+v"(y));                 // computed here, not where it is next used
      total[q][j][i] = y;
    };
#pragma unroll
    for (int k = 0; k < MF; ++k) {
      // the wave that is behind goes first (the older wave of a SIMD would else run through the
      // step and wait at its end while the other runs alone)
      if (k == 0) __builtin_amdgcn_s_setprio(3);
      else if (k * 4 == MF) __builtin_amdgcn_s_setprio(2);
      else if (k * 2 == MF) __builtin_amdgcn_s_setprio(1);
      else if (k * 4 == MF * 3) __builtin_amdgcn_s_setprio(0);
#pragma unroll
      for (int ks = 0; ks < KSG; ++ks) {
        const int u = k * KSG + ks;
        if (u % 2 == 0) asm volatile("" : "+v"(a[u % RINGA]), "+v"(a[(u + 1) % RINGA]));
        const bf16x8 av = __builtin_bit_cast(bf16x8, a[u % RINGA]);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const int e = ks * NJ + j;              // 0 .. 4 NJ - 1
          P[k & 1][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              av, B[ks][j], ks > 0 ? P[k & 1][j] : k == 0 ? xown : xv[k & 3], 0, 0, 0);
          if (j == 0) {
            const int n = u + AHEAD;
            if (k == 0 && ks == 0) xv[1] = *xs_at(par, 1);
            if (ks == 1 && k + 2 < MF) xv[(k + 2) & 3] = *xs_at(par, k + 2);
            if (k == 0) read_w(b1, ks, w[ks]);
            // the next tile's row sums: the wave's first fragment, read beside the first
            // fragment's products, summed beside the next one's and written after them
            if (XSP == 0 && k == 0) an[ks] = read_a(b1, ks);
            if (XSP == 0 && k == 1) xs = sum_unit(an[ks], ks == 0 ? zero : xs);
            a[n % RINGA] = n < UNITS ? read_a(b0, n) : read_a(b1, n - UNITS);
          } else if (j == 1) {
            // the loads, evenly over the fragments
            const int q = (u * S::OPS + UNITS - 1) / UNITS;
            if (q < S::OPS && q * UNITS / S::OPS == u) {
                if (q < S::OPS_A) load_a(s + 2, b2, q);
                else if (q < S::OPS_A + S::OPS_S) load_s(s + 3, b0, b2, q - S::OPS_A);
                else load_w(s + 3, b0, q - S::OPS_A - S::OPS_S);
              }
          }
          // the previous fragment's sums, from the third MFMA on (its own last ones are then done)
          if (e >= NJ) {
            const int q0 = ((e - NJ) * 4 + 2) / 3, q1 = ((e - NJ + 1) * 4 + 2) / 3;   // elements q with q * 3 / 4 = e - NJ
#pragma unroll
            for (int q = q0; q < q1; ++q) {
              const float v = P[(k + 1) & 1][q >> 2][q & 3];
              if (k == 0) fma1(MF - 1, q, v, scp);
              else fma1(k - 1, q, v, sc);
            }
          }
          if (k > 0) {
            const int slot = (k - 1) * NW + e;     // 4 parts a word, evenly over the slots
            const int t0 = (slot * 4 * NW + SLOTS - 1) / SLOTS, t1 = ((slot + 1) * 4 * NW + SLOTS - 1) / SLOTS;
#pragma unroll
            for (int t = t0; t < t1; ++t) {
              const int wks = t / 4 / NJ, wj = t / 4 % NJ;
              un[t / 4].part(t % 4, w[wks][wj], addn[wj], exp4);
              if (t % 4 == 3) Bn[wks][wj] = un[t / 4].value();
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (k == 0) read_sz(s + 1, b1, addn, scn);
      if (k == 1) {
        xown = XSP > 0 ? given_xs(b1) : xs;
        if (c == 0) *xs_at(1 - par, 0) = xown;
      }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) scp[j] = sc[j];
    // Tile s + 2 has landed; step s + 3's words may be on their way, unless they are switched
    // off: then the last loads that are on are waited for whatever the others count.
    if (s + 3 < loads) dma_wait<S::OPS_W>();
    else dma_wait<0>();
    __syncthreads();
  };
  {
    int b0 = 0, b1 = 1, b2 = 2;
    auto next = [&]() {
      const int b = b0;
      b0 = b1;
      b1 = b2;
      b2 = b;
    };
    for (int s = 0; s < steps; s += 2) {   // (an odd count ends with a step whose scales are zero)
      step(std::integral_constant<int, 0>{}, s, b0, b1, b2, B0, sc0, B1, sc1);
      next();
      step(std::integral_constant<int, 1>{}, s + 1, b0, b1, b2, B1, sc1, B0, sc0);
      next();
    }
#pragma unroll
    for (int e = 0; e < 4 * NJ; ++e)
      total[MF - 1][e >> 2][e & 3] = fmaf(scp[e >> 2], P[(MF - 1) & 1][e >> 2][e & 3], total[MF - 1][e >> 2][e & 3]);
    dma_wait<0>();      // tiles past the last are still on their way into the ring
    __syncthreads();
  }

  // ---- the slices' sums meet in LDS, in slice order; wave (wn, wk) keeps row
  // fragments wk MF / WK .. of its columns ----
  constexpr int MS = MF / WK;
  f32x4 out[MS][NJ];
  int fr[MS];   // the tile's row fragments of this wave's share
  if constexpr (WK == 1) {
#pragma unroll
    for (int mi = 0; mi < MF; ++mi) {
      fr[mi] = row_frag(mi);
#pragma unroll
      for (int j = 0; j < NJ; ++j) out[mi][j] = total[mi][j];
    }
  } else {
    f32x4* const part = reinterpret_cast<f32x4*>(smem);
#pragma unroll
    for (int mi = 0; mi < MF; ++mi)
#pragma unroll
      for (int j = 0; j < NJ; ++j) part[((wave * MF + mi) * NJ + j) * 64 + lane] = total[mi][j];
    __syncthreads();
#pragma unroll
    for (int mi = 0; mi < MS; ++mi) {
      const int own = wk * MS + mi;   // of the wave's fragments
      fr[mi] = row_frag(own);
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        f32x4 v = part[((wn * MF + own) * NJ + j) * 64 + lane];
#pragma unroll
        for (int k = 1; k < WK; ++k) v += part[(((k * WN + wn) * MF + own) * NJ + j) * 64 + lane];
        out[mi][j] = v;
      }
    }
    __syncthreads();
  }

  if (p.epi == EPI_QKV_PREP) {
    // The tile is BN / 128 heads of rows m0 ..: parked as bf16, then each 16-lane
    // row takes head vectors through prep_vector, as prefill_prep_kernel does.
    constexpr int LD = BN + 8;
    uint16_t* const tile = reinterpret_cast<uint16_t*>(smem);
#pragma unroll
    for (int mi = 0; mi < MS; ++mi)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        uint32_t* dst = reinterpret_cast<uint32_t*>(tile + (16 * fr[mi] + 4 * r + i) * LD + wn * 16 * NJ + NJ * c);
#pragma unroll
        for (int j = 0; j < NJ / 2; ++j) dst[j] = pack_bf16x2(out[mi][2 * j][i], out[mi][2 * j + 1][i]);
      }
    // The RoPE rows come first, all of them: one wait, behind the barrier, and not one a
    // vector.
    constexpr int HEADS = BN / ATT_D, VECS = BM * HEADS / (4 * S::WAVES);
    static_assert(VECS * 4 * S::WAVES == BM * HEADS, "whole rounds of head vectors");
    u32x4 rp[VECS];
    int tt[VECS], bb[VECS];
#pragma unroll
    for (int i = 0; i < VECS; ++i) {
      const int m = min(m0 + (4 * wave + r + 4 * S::WAVES * i) / HEADS, p.M - 1);
      bb[i] = m / pp.T;
      tt[i] = m - bb[i] * pp.T;
      rp[i] = *reinterpret_cast<const u32x4*>(pp.rope + (size_t)(pp.p0 + tt[i]) * ATT_D + 8 * c);
    }
    const u32x4 gq = prep_load(pp.qn, c, pp.style), gk = prep_load(pp.kn, c, pp.style);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < VECS; ++i) {
      const int v = 4 * wave + r + 4 * S::WAVES * i, row = v / HEADS, hh = v % HEADS;
      if (m0 + row >= p.M) continue;   // uniform over the 16-lane row
      const int head = n0 / ATT_D + hh;
      const bool isq = head < pp.Hq, normed = head < pp.Hq + pp.Hkv;
      const u32x4 raw = prep_load(tile + row * LD + hh * ATT_D, c, pp.style);
      const u32x4 y = prep_vector(raw, rp[i], isq ? gq : gk, normed, pp.style, pp.eps);
      uint16_t* dst;
      if (isq) dst = pp.q + (((size_t)bb[i] * pp.Hq + head) * pp.T + tt[i]) * ATT_D;
      else if (normed) dst = pp.kc + (((size_t)bb[i] * pp.Hkv + (head - pp.Hq)) * pp.cap + pp.p0 + tt[i]) * ATT_D;
      else dst = pp.vc + (((size_t)bb[i] * pp.Hkv + (head - pp.Hq - pp.Hkv)) * pp.cap + pp.p0 + tt[i]) * ATT_D;
      prep_store(dst, c, pp.style, y);
    }
    return;
  }
  const bool paired = p.epi == EPI_SWIGLU || p.epi == EPI_PAIRED;
  float* const s_ys = reinterpret_cast<float*>(smem);   // [BM][WN]
#pragma unroll
  for (int mi = 0; mi < MS; ++mi) {
    const int row0 = m0 + 16 * fr[mi] + 4 * r;
    if (!paired) {
      uint32_t res[4][NJ / 2];
      if (p.epi == EPI_RESIDUAL) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t* src = reinterpret_cast<const uint32_t*>(p.residual + (size_t)min(row0 + i, p.M - 1) * p.ldy + ncol);
#pragma unroll
          for (int j = 0; j < NJ / 2; ++j) res[i][j] = src[j];
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        uint32_t v[NJ / 2];
#pragma unroll
        for (int j = 0; j < NJ / 2; ++j) {
          v[j] = pack_bf16x2(out[mi][2 * j][i], out[mi][2 * j + 1][i]);
          if (p.epi == EPI_RESIDUAL)
            v[j] = pack_bf16x2(bf16_lo(v[j]) + bf16_lo(res[i][j]), bf16_hi(v[j]) + bf16_hi(res[i][j]));
        }
        if (row0 + i < p.M) {
          uint32_t* dst = reinterpret_cast<uint32_t*>(p.y0 + (size_t)(row0 + i) * p.ldy + ncol);
          dst[0] = v[0];
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float o0[NJ / 2], o1[NJ / 2];
        float hs = 0.0f;
#pragma unroll
        for (int j = 0; j < NJ / 2; ++j) {
          const float g = round_bf16(out[mi][2 * j][i]), u = round_bf16(out[mi][2 * j + 1][i]);
          o0[j] = p.epi == EPI_SWIGLU ? round_bf16(round_bf16(silu_fast(g)) * u) : g;
          o1[j] = u;
          hs += o0[j];
        }
        const size_t off = (size_t)(row0 + i) * p.ldy + (ncol >> 1);
        if (row0 + i < p.M) {
          p.y0[off] = (uint16_t)f32_to_bf16(o0[0]);
          if (p.epi == EPI_PAIRED) p.y1[off] = (uint16_t)f32_to_bf16(o1[0]);
        }
        if (p.ys) {   // the wave's 8 NJ output columns of the row
          hs = row_sum16(hs);
          if (c == 0) s_ys[(16 * fr[mi] + 4 * r + i) * WN + wn] = hs;
        }
      }
    }
  }
  if (p.ys) {
    // 64 output columns (128 of the tile's) are one half group of the next product's k
    constexpr int WH = 128 / (16 * NJ);   // waves a half group
    __syncthreads();
    for (int q = tid; q < BM * (BN / 128); q += S::THREADS) {
      const int row = q % BM, h = q / BM;
      float v = s_ys[row * WN + h * WH];
#pragma unroll
      for (int w = 1; w < WH; ++w) v += s_ys[row * WN + h * WH + w];
      if (m0 + row < p.M) p.ys[(size_t)((n0 >> 7) + h) * p.ldys + m0 + row] = v;
    }
  }
}

}  // namespace t2i

namespace {
using namespace t2i;

template <int MF, int NJ, int WN, int WK, bool GIVEN>
hipError_t launch_one(const LinearParams& p, const QkvPrepParams& pp, hipStream_t s) {
  using S = GemmShape<MF, NJ, WN, WK, 0>;
  const unsigned tiles = (unsigned)((p.M + S::BM - 1) / S::BM) * (unsigned)(p.N / S::BN);
  if (!p.xs) {
    hipLaunchKernelGGL((w4a16_prompt_kernel<MF, NJ, WN, WK, 0>), dim3(tiles), dim3(S::THREADS), 0, s, p, pp);
  } else if constexpr (GIVEN) {
    if (p.xs_parts == 1) hipLaunchKernelGGL((w4a16_prompt_kernel<MF, NJ, WN, WK, 1>), dim3(tiles), dim3(S::THREADS), 0, s, p, pp);
    else hipLaunchKernelGGL((w4a16_prompt_kernel<MF, NJ, WN, WK, 2>), dim3(tiles), dim3(S::THREADS), 0, s, p, pp);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

// Tile forms (PROMPT_FORMS of prompt_plan.h): row fragments a wave, columns a lane, waves along
// N, k slices, and whether it is built for given row sums.
#define T2I_PROMPT_CONFIGS(X) \
  X(8, 2, 8, 1, true)         \
  X(4, 2, 4, 1, false)        \
  X(4, 2, 4, 2, true)

namespace t2i_host {

hipError_t launch_prompt_ring(const PromptPlan& pl, const LinearParams& p, const QkvPrepParams& pp, hipStream_t s) {
  if (!prompt_form_serves(pl, p.N, p.xs != nullptr)) return hipErrorInvalidValue;
#define T2I_PROMPT_LAUNCH(a, b, c, d, given) \
  if (pl.cfg[0] == a && pl.cfg[1] == b && pl.cfg[2] == c && pl.cfg[3] == d) return launch_one<a, b, c, d, given>(p, pp, s);
  T2I_PROMPT_CONFIGS(T2I_PROMPT_LAUNCH)
#undef T2I_PROMPT_LAUNCH
  return hipErrorInvalidValue;
}

}  // namespace t2i_host
