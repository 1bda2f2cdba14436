// bf16 MFMA GEMM core for gfx950: C[M, N] = A[M, K] * B[N, K]^T, fp32 accumulation.
//
// Both operands are row-major with K contiguous (the layout of hidden [N, H]
// and of the LM head [V, H]), 16-byte aligned, row strides and K multiples of
// 8 elements.
//
// Workgroup tile 256 x 256, k-block 64, 512 threads in a 4 x 2 grid of waves, each owning a
// 64 x 128 block of C as 4 x 8 tiles of v_mfma_f32_16x16x32_bf16 (128 fp32 accumulators per
// lane), two waves per SIMD, so one wave's MFMAs can run while the other waits at the barrier
// or for LDS data.
//
// Why the 16x16x32 shape: these kernels run at the card's power limit, and per FLOP it moves
// half the accumulator traffic of 32x32x16 through the register file for twice the (16-bit)
// operand traffic. In the same loop it ran 3% faster. Why a k-block of 64: a K-major row is
// then 128 bytes in memory, one L2 request, where a k-block of 32 made two.
//
// Operands go from HBM straight into LDS with buffer_load_dwordx4 ... lds
// (no staging registers): a wave's load instruction fills 1 KiB of LDS, lane i
// at the wave's base + 16 * i. LDS is a ring of five 32 KiB operand tiles (all 160 KiB of a
// CU): the A and B tiles of the k-block in use, both of the next, and A of the one after, so
// A is loaded two k-blocks ahead and B one; with four tiles (two stages of A and B) the same
// loop was 1-2% slower. One barrier per k-block; the MFMA operand fragments are read half a
// k-step ahead, with the LDS reads and global loads placed between MFMAs (see mainloop).
// Buffer resources make out-of-range rows (and the k tail) read as zeros, so partial tiles
// need no branches.
//
// LDS rows of a K-major tile are 128 B (64 bf16) with the eight 16-byte chunks XOR-swizzled by
// (row >> 1) & 7 (see swz), which makes the MFMA operand ds_read_b128s free of bank conflicts.
//
// MFMA 16x16x32 bf16 lane layout: the first operand's lane l holds row l % 16,
// k = (l / 16) * 8 + e for e < 8; the second's lane l column l % 16 with the same k;
// accumulator element e is D[4 * (l / 16) + e][l % 16]. B is passed first, so D is C
// transposed and a lane holds, of each 16 x 16 tile of C, row l % 16 and the four consecutive
// columns 4 * (l / 16) + e: an epilogue reads and writes C in 16-byte accesses straight from
// the accumulators.
//
// Either operand may instead be stored MN-major (element (r, k) at k * ld + r,
// e.g. dlogits [N, V] read as the [V, N] operand of the weight gradient, or
// the LM head [V, H] read as the [H, V] operand of the hidden gradient). Such
// a tile sits in LDS as 64 k-rows of 256 bf16 (512 B, XOR-swizzled in 32-byte units, see
// swz_t) and the MFMA fragments come out of it transposed by
// ds_read_b64_tr_b16: within each 16-lane group, lane i receives element j of
// the 4 that lane 4j + i/4 addressed, element i % 4 of them (checked on the
// device). So lane s of group g addressing (k = kb + s / 4, r = rb + 4 (s % 4))
// makes lane i of the group receive X[rb + i][kb + j], j < 4: two such reads
// (kb and kb + 4) give the 8 k of an MFMA fragment without a transpose pass.
//
// Measured on MI355X at [8192, 4096] x [128256, 4096] (two waves per SIMD, one run): logits
// with row statistics 7.20 -> 6.56 ms, the whole loss and gradients 22.5 -> 20.9 ms, against
// a k-block of 32 with 32x32x16 MFMAs and four stages.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

#include "common.hpp"
#include "plan.hpp"

namespace ts_gemm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) bf16x4* lds_bf16x4_t;

// Storage of a GEMM operand: K-major (element (r, k) at r * ld + k) or
// MN-major (element (r, k) at k * ld + r).
enum Major : int { kKMajor = 0, kMNMajor = 1 };

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) uint32_t* lds_ptr_t;

constexpr int BM = 256;
constexpr int BN = 256;
constexpr int BK = ts_plan::kGemmBlockK;
constexpr int kRowBytes = BK * 2;                       // 128
constexpr int kTileBytes = BM * kRowBytes;              // 32 KiB per operand per k-block
constexpr int kSlots = 5;                               // operand tiles of the LDS ring
constexpr size_t kLdsBytes = (size_t)kSlots * kTileBytes;
static_assert(BK == 64 && BM == ts_plan::kGemmTile, "the plan's tile");
constexpr uint32_t kOob = 0x80000000u;  // voffset beyond every resource's range -> reads 0

// Wave layout: kW waves, wave wid owns rows [wm * RW, +RW) and columns
// [wn * 128, +128) of the tile, wm = wid >> 1, wn = wid & 1.
template <int kW>
struct Cfg {
  static_assert(kW == 8, "wave layout");
  static constexpr int kThreads = 64 * kW;
  static constexpr int kLoads = 32 / kW;  // 1 KiB loads per wave per operand per k-block
  static constexpr int kTI = 32 / kW;     // 16-row tiles per wave (and 8 of 16 columns)
  static constexpr int RW = 16 * kTI;     // rows per wave
};

template <int kTI>
struct Acc {
  f32x4 t[kTI][8];
};

__device__ void buffer_load_lds(i32x4 rsrc, lds_ptr_t lds, int size, int voffset, int soffset,
                                int offset, int aux) __asm("llvm.amdgcn.raw.buffer.load.lds");

// Raw buffer resource over [base, base + bytes) (gfx9 word 3).
__device__ inline i32x4 make_rsrc(const void* base, uint64_t bytes) {
  const uint64_t a = (uint64_t)base;
  i32x4 r;
  r[0] = (int32_t)(uint32_t)a;
  r[1] = (int32_t)((uint32_t)(a >> 32) & 0xffffu);
  r[2] = (int32_t)(bytes > 0xffffffffull ? 0xffffffffu : (uint32_t)bytes);
  r[3] = 0x00020000;
  return r;
}

// s_waitcnt vmcnt(n) with the other counters left alone (gfx9 encoding).
template <int N>
__device__ inline void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// Waits for this wave's LDS reads and until at most N of its loads are outstanding.
template <int N>
__device__ inline void wait_lgkm0_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4));
}

// LDS position of logical 16-byte chunk c (0..7) of LDS row `row` (128-byte rows). A
// fragment read has 16 rows at one c: two rows share a 256-byte bank line, and XOR with bits
// 1-3 of the row puts the eight lines' chunks in distinct positions. Measured on MI355X with
// SQ_LDS_BANK_CONFLICT: 0 conflict cycles.
__device__ inline int swz(int row, int c) { return c ^ ((row >> 1) & 7); }

// K-major tile loads: rows [row0, row0 + 256) of a [nrows, ld] matrix,
// out-of-range rows read zeros. Wave load u fills LDS rows
// [(u * kW + wid) * 8, +8) (1 KiB); off[u] is this lane's byte offset
// (relative to the tile's first row) of the logical chunk its LDS position
// holds, at k0 = 0.
template <int kW>
struct TileLoader {
  i32x4 rsrc;
  uint32_t off[Cfg<kW>::kLoads];
};

template <int kW>
__device__ inline TileLoader<kW> make_loader(const __bf16* g, int64_t ld, int64_t nrows,
                                             int64_t row0) {
  TileLoader<kW> t;
  const int wid = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  int64_t valid = nrows - row0;
  if (valid > BM) valid = BM;
  if (valid < 0) valid = 0;
  t.rsrc = make_rsrc(g + row0 * ld, (uint64_t)valid * (uint64_t)ld * 2);
#pragma unroll
  for (int u = 0; u < Cfg<kW>::kLoads; ++u) {
    const int row = (u * kW + wid) * 8 + (lane >> 3);
    const int chunk = swz(row, lane & 7);  // the logical chunk LDS position lane&7 holds
    t.off[u] = (uint32_t)(row * ld * 2 + chunk * 16);
  }
  return t;
}

// Issues this wave's loads of k-block [k0, k0 + BK) into the LDS tile. kFull: the whole
// block lies below K, so the block's offset rides in the scalar offset operand (which the
// hardware adds after the range check: rows past the matrix still read zeros) and a load
// costs no vector instruction.
template <bool kFull, int kW>
__device__ inline void issue_loads(const TileLoader<kW>& t, int64_t k0, int64_t K,
                                   uint8_t* lds_tile) {
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int u = 0; u < Cfg<kW>::kLoads; ++u) {
    uint8_t* dst = lds_tile + (u * kW + wid) * 1024;
    if constexpr (kFull) {
      buffer_load_lds(t.rsrc, (lds_ptr_t)dst, 16, (int)t.off[u], (int)(k0 * 2), 0, 0);
    } else {
      // logical chunk of this lane for the load's row (same swizzle as make_loader)
      const int row = (u * kW + wid) * 8 + (lane >> 3);
      const int chunk = swz(row, lane & 7);
      const bool in_k = k0 + chunk * 8 < K;
      const uint32_t voff = in_k ? t.off[u] + (uint32_t)(k0 * 2) : kOob;
      buffer_load_lds(t.rsrc, (lds_ptr_t)dst, 16, (int)voff, 0, 0, 0);
    }
  }
}

// MN-major tile loads: rows [r0, r0 + 256) of the operand, k-block [k0,
// k0 + BK). LDS byte (kr, p) of the tile (kr < BK, p < 512) holds logical byte
// p ^ swz_t(kr) of k-row kr: the 16-byte chunk at p is 8 consecutive r.
// A half-wave of ds_read_b64_tr_b16 (see read_op_t) reads 32 bytes from each of the 8 k-rows
// k, k + 1, k + 2, k + 3 and k + 8 .. k + 11; the swizzle puts them in the 8 distinct 32-byte
// slots of a 256-byte bank window (0 conflict cycles measured).
// Wave load u covers LDS chunks [(u * kW + wid) * 64, +64): k-rows
// 2 (u * kW + wid) and 2 (u * kW + wid) + 1.
template <int kW>
struct TileLoaderT {
  const __bf16* base;              // element (k = 0, r = r0)
  int64_t ld;                      // elements between consecutive k
  uint32_t off[Cfg<kW>::kLoads];   // byte offset within a k-block window, kOob past the rows
  int kr[Cfg<kW>::kLoads];         // k-row (0 .. BK - 1) of this lane's chunk
};

__device__ inline int swz_t(int kr) { return ((kr & 3) << 6) | (((kr >> 3) & 1) << 5); }

template <int kW>
__device__ inline TileLoaderT<kW> make_loader_t(const __bf16* g, int64_t ld, int64_t nrows,
                                                int64_t r0) {
  TileLoaderT<kW> t;
  const int wid = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  t.base = g + r0;
  t.ld = ld;
#pragma unroll
  for (int u = 0; u < Cfg<kW>::kLoads; ++u) {
    const int c = (u * kW + wid) * 64 + lane;  // 16-byte LDS chunk of the tile
    const int kr = c >> 5;
    const int lbyte = ((c & 31) << 4) ^ swz_t(kr);  // logical byte within the k-row
    const int64_t r = r0 + (lbyte >> 1);
    t.kr[u] = kr;
    t.off[u] = r < nrows ? (uint32_t)(kr * ld * 2 + lbyte) : kOob;
  }
  return t;
}

// Issues this wave's loads of k-block [k0, k0 + BK) into the LDS tile (kFull: all below K).
// The buffer resource spans the k-block's BK k-rows, so offsets stay 32-bit
// whatever the operand's size.
template <bool kFull, int kW>
__device__ inline void issue_loads_t(const TileLoaderT<kW>& t, int64_t k0, int64_t K,
                                     uint8_t* lds_tile) {
  const i32x4 rsrc = make_rsrc(t.base + k0 * t.ld, (uint64_t)BK * (uint64_t)t.ld * 2);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int u = 0; u < Cfg<kW>::kLoads; ++u) {
    const uint32_t voff = kFull || k0 + t.kr[u] < K ? t.off[u] : kOob;
    uint8_t* dst = lds_tile + (u * kW + wid) * 1024;
    buffer_load_lds(rsrc, (lds_ptr_t)dst, 16, (int)voff, 0, 0, 0);
  }
}

// Fragments (k-step ks, 32 deep) of kN 16-row blocks starting at row r_base of a
// K-major tile: one ds_read_b128 each.
template <int kN>
__device__ inline void read_op_k(const uint8_t* Xs, int r_base, int lane, int ks, bf16x8* f) {
  const int r = lane & 15;
  const int c = ks * 4 + (lane >> 4);
#pragma unroll
  for (int i = 0; i < kN; ++i) {
    const int row = r_base + i * 16 + r;
    f[i] = *reinterpret_cast<const bf16x8*>(Xs + row * kRowBytes + (swz(row, c) << 4));
  }
}

// The same fragments from an MN-major tile: two ds_read_b64_tr_b16 each.
template <int kN>
__device__ inline void read_op_t(const uint8_t* Xs, int r_base, int lane, int ks, bf16x8* f) {
  const int g = lane >> 4;
  const int sl = lane & 15;
#pragma unroll
  for (int i = 0; i < kN; ++i) {
    const int r = r_base + i * 16 + 4 * (sl & 3);
    bf16x4 h[2];
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int k = ks * 32 + 8 * g + 4 * hh + (sl >> 2);
      const int byte = k * 512 + ((2 * r) ^ swz_t(k));
      h[hh] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4_t)(Xs + byte));
    }
    f[i] = __builtin_shufflevector(h[0], h[1], 0, 1, 2, 3, 4, 5, 6, 7);
  }
}

// Loader of one operand of the given storage.
template <int kMajor, int kW> struct OpLoader;
template <int kW> struct OpLoader<kKMajor, kW> {
  TileLoader<kW> t;
  __device__ inline OpLoader(const __bf16* g, int64_t ld, int64_t nrows, int64_t r0)
      : t(make_loader<kW>(g, ld, nrows, r0)) {}
  template <bool kFull>
  __device__ inline void issue(int64_t k0, int64_t K, uint8_t* tile) const {
    issue_loads<kFull, kW>(t, k0, K, tile);
  }
};
template <int kW> struct OpLoader<kMNMajor, kW> {
  TileLoaderT<kW> t;
  __device__ inline OpLoader(const __bf16* g, int64_t ld, int64_t nrows, int64_t r0)
      : t(make_loader_t<kW>(g, ld, nrows, r0)) {}
  template <bool kFull>
  __device__ inline void issue(int64_t k0, int64_t K, uint8_t* tile) const {
    issue_loads_t<kFull, kW>(t, k0, K, tile);
  }
};

template <int kMajor, int kN>
__device__ inline void read_op(const uint8_t* Xs, int r_base, int lane, int ks, bf16x8* f) {
  if constexpr (kMajor == kKMajor) read_op_k<kN>(Xs, r_base, lane, ks, f);
  else read_op_t<kN>(Xs, r_base, lane, ks, f);
}

// LDS read instructions of kN fragments.
template <int kMajor>
constexpr int frag_reads(int n) { return (kMajor == kMNMajor ? 2 : 1) * n; }

// The MFMAs of a half step: every row tile against the four column tiles of `half`. B is the
// first operand (see the layout of C above).
template <int kTI>
__device__ inline void mma_half(const bf16x8 (&a)[kTI], const bf16x8 (&b)[4], Acc<kTI>& acc,
                                int half) {
#pragma unroll
  for (int q = 0; q < kTI * 4; ++q)
    acc.t[q / 4][half * 4 + q % 4] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
        b[q % 4], a[q / 4], acc.t[q / 4][half * 4 + q % 4], 0, 0, 0);
}

// Instruction interleaving. A wave issues MFMAs one at a time and waits for
// the matrix core to accept each; other instructions placed between two MFMAs
// issue in the shadow of the first for free. These scheduling groups ask the
// compiler for such an order (the grouped instructions are independent of
// the MFMAs they sit between).
template <int kMask, int kCount>
__device__ inline void sched_group() {
  if constexpr (kCount > 0) __builtin_amdgcn_sched_group_barrier(kMask, kCount, 0);
}

// kM MFMAs with kR LDS reads spread over the slots after the first kSR of them and kV
// global->LDS loads over the slots after the others.
template <int kR, int kV, int kM, int kSR, int... I>
__device__ inline void sched_mix_impl(std::integer_sequence<int, I...>) {
  constexpr int kSV = kM - kSR;
  ((sched_group<0x008, 1>(),                                                       // MFMA
    sched_group<0x100, I < kSR ? kR * (I + 1) / kSR - kR * I / kSR : 0>(),         // LDS read
    sched_group<0x020, I < kSR ? 0 : kV * (I - kSR + 1) / kSV - kV * (I - kSR) / kSV>()),
   ...);
}
template <int kR, int kV, int kM, int kSR>
__device__ inline void sched_mix() {
  static_assert(kSR > 0 && kSR < kM, "slots");
  sched_mix_impl<kR, kV, kM, kSR>(std::make_integer_sequence<int, kM>());
}

// Main loop for the tile at (m0, n0). `smem` holds kLdsBytes (16-byte aligned).
//
// Steady state, per k-block kt: four half steps of 16 MFMAs (k-step 0 or 1 against the low or
// high 64 columns of the wave's block), each with the LDS reads of what the next one needs:
//   (0, low)   reads the high columns' B fragments of k-step 0
//   (0, high)  reads A and the low B fragments of k-step 1
//   (1, low)   reads the high B fragments of k-step 1; this wave is then done with the tiles
//              of kt, waits for its loads of kt+1 and meets the barrier
//   (1, high)  reads A and the low B fragments of (kt+1, 0) and issues the loads of B(kt+2)
//              and A(kt+3) into the tiles every wave has finished reading
// A's fragments are double-buffered by k-step, B's halves overwrite each other: 64 VGPRs of
// fragments beside the 128 accumulators. The barrier comes before the last half step rather
// than inside it (2 or 4 MFMAs ahead of it were 2-4% slower). The last k-blocks run a plain
// drain loop, so the steady-state body has no branches (a branch there splits the interleaved
// block and makes the register allocator shuffle the accumulators) and its loads, all of
// whole k-blocks, need no bounds arithmetic.
template <int kMA, int kMB, int kW>
__device__ inline void mainloop(const __bf16* __restrict__ A, int64_t lda, int64_t M,
                                const __bf16* __restrict__ B, int64_t ldb, int64_t N, int64_t K,
                                int64_t m0, int64_t n0, uint8_t* smem, Acc<Cfg<kW>::kTI>& acc) {
  using C = Cfg<kW>;
  constexpr int kRA = frag_reads<kMA>(C::kTI), kRB = frag_reads<kMB>(4);
  constexpr int kH = C::kTI * 4;  // MFMAs of a half step
  const int wid = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int wm = wid >> 1;
  const int wn = wid & 1;
#pragma unroll
  for (int i = 0; i < C::kTI; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc.t[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const OpLoader<kMA, kW> la(A, lda, M, m0);
  const OpLoader<kMB, kW> lb(B, ldb, N, n0);
  const int64_t KT = (K + BK - 1) / BK;
  // ring of operand tiles A(0) B(0) A(1) B(1) A(2) ..., tile n in slot n % kSlots
  constexpr std::true_type kWhole{};
  constexpr std::false_type kPart{};
  auto tile = [&](int slot) { return smem + slot * kTileBytes; };
  auto issue_a = [&](auto full, int64_t t, int slot) {
    la.template issue<decltype(full)::value>(t * BK, K, tile(slot));
  };
  auto issue_b = [&](auto full, int64_t t, int slot) {
    lb.template issue<decltype(full)::value>(t * BK, K, tile(slot));
  };
  auto next = [](int s) { return s >= kSlots - 2 ? s - (kSlots - 2) : s + 2; };
  if (0 < KT) {
    issue_a(kPart, 0, 0);
    issue_b(kPart, 0, 1);
  }
  if (1 < KT) {
    issue_a(kPart, 1, 2);
    issue_b(kPart, 1, 3);
  }
  if (2 < KT) issue_a(kPart, 2, 4);
  // k-block 0 landed (vmcnt counts loads in issue order, kLoads a tile)
  if (KT > 2) wait_vmcnt<3 * C::kLoads>();
  else if (KT > 1) wait_vmcnt<2 * C::kLoads>();
  else wait_vmcnt<0>();
  __builtin_amdgcn_s_barrier();
  bf16x8 a0[C::kTI], a1[C::kTI], bl[4], bh[4];
  const int ra = wm * C::RW, rb = wn * 128;
  int sa = 0, sb = 1;  // slots of the current k-block's tiles
  read_op<kMA, C::kTI>(tile(sa), ra, lane, 0, a0);
  read_op<kMB, 4>(tile(sb), rb, lane, 0, bl);
  int64_t kt = 0;
  for (const int64_t whole = K / BK; kt + 3 < whole; ++kt) {
    const uint8_t* As = tile(sa);
    const uint8_t* Bs = tile(sb);
    read_op<kMB, 4>(Bs, rb + 64, lane, 0, bh);
    mma_half(a0, bl, acc, 0);
    sched_mix<kRB, 0, kH, kH / 2>();
    __builtin_amdgcn_sched_barrier(0);
    read_op<kMA, C::kTI>(As, ra, lane, 1, a1);
    read_op<kMB, 4>(Bs, rb, lane, 1, bl);
    mma_half(a0, bh, acc, 1);
    sched_mix<kRA + kRB, 0, kH, kH * 3 / 4>();
    __builtin_amdgcn_sched_barrier(0);
    read_op<kMB, 4>(Bs, rb + 64, lane, 1, bh);
    mma_half(a1, bl, acc, 0);
    sched_mix<kRB, 0, kH, kH / 2>();
    __builtin_amdgcn_sched_barrier(0);
    // A(kt+1) and B(kt+1) landed; A(kt+2), issued after them, may be in flight
    wait_lgkm0_vmcnt<C::kLoads>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    const int na = next(sa), nb = next(sb);
    read_op<kMA, C::kTI>(tile(na), ra, lane, 0, a0);
    read_op<kMB, 4>(tile(nb), rb, lane, 0, bl);
    issue_b(kWhole, kt + 2, sa);
    issue_a(kWhole, kt + 3, sb);
    mma_half(a1, bh, acc, 1);
    sched_mix<kRA + kRB, 2 * C::kLoads, kH, kH / 2>();
    __builtin_amdgcn_sched_barrier(0);
    sa = na;
    sb = nb;
  }
  // drain: the last k-blocks, whose loads may be partial or past the end
  for (; kt < KT; ++kt) {
    const uint8_t* As = tile(sa);
    const uint8_t* Bs = tile(sb);
    read_op<kMB, 4>(Bs, rb + 64, lane, 0, bh);
    __builtin_amdgcn_sched_barrier(0);
    mma_half(a0, bl, acc, 0);
    __builtin_amdgcn_sched_barrier(0);
    read_op<kMA, C::kTI>(As, ra, lane, 1, a1);
    read_op<kMB, 4>(Bs, rb, lane, 1, bl);
    __builtin_amdgcn_sched_barrier(0);
    mma_half(a0, bh, acc, 1);
    __builtin_amdgcn_sched_barrier(0);
    read_op<kMB, 4>(Bs, rb + 64, lane, 1, bh);
    __builtin_amdgcn_sched_barrier(0);
    mma_half(a1, bl, acc, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (kt + 1 < KT) {
      if (kt + 2 < KT) wait_lgkm0_vmcnt<C::kLoads>();
      else wait_lgkm0_vmcnt<0>();
      __builtin_amdgcn_s_barrier();
      if (kt + 2 < KT) issue_b(kPart, kt + 2, sa);
      if (kt + 3 < KT) issue_a(kPart, kt + 3, sb);
      sa = next(sa);
      sb = next(sb);
      read_op<kMA, C::kTI>(tile(sa), ra, lane, 0, a0);
      read_op<kMB, 4>(tile(sb), rb, lane, 0, bl);
    }
    __builtin_amdgcn_sched_barrier(0);
    mma_half(a1, bh, acc, 1);
    __builtin_amdgcn_sched_barrier(0);
  }
}

}  // namespace ts_gemm
