// fp32 GEMM for gfx950 (CDNA4):  C[M,N] = act( opA(A) . opB(B) ).
//
// Replaces the reference's dense products and their activation passes:
//   ns_matmul + ns_act2          /root/reference/src/codegen/codegen.cpp:1257-1265, 1244-1255
//   ns_matmul_grad_a  (transB)   codegen.cpp:1318-1326
//   ns_matmul_grad_w  (transA)   codegen.cpp:1329-1337
// (CUDA counterparts ns_gemm_kernel / ns_grad_a_kernel / ns_grad_w_kernel,
// /root/reference/src/codegen/cuda_backend.cpp:58-79, 446-467.)
//
// Design (wave64).  Three kernels, one set of operand modes and epilogues:
//  * gemm_bf3_kernel (16-byte aligned operands): fp32 products as six bf16
//    MFMAs over three-piece operands (split3.h).  Operands are read as fp32,
//    split in registers on their way to LDS, and each K slab of 16 is held
//    there as [piece][k / 8][row] of 16-byte chunks, which is the MFMA operand
//    order for either memory order of the operand (8 consecutive k of one row
//    per lane), read back as conflict-free float4s.
//  * gemm_f32_kernel (any alignment): fp32 MFMA 32x32x2, 128x128 tiles.
//  * gemm_small_kernel: products of a few tiles, whose K is dealt out to the
//    waves of a workgroup.
//  * The first two: K advances in 16-wide slabs staged in LDS, double buffered, one
//    barrier per slab, global loads in flight under the MFMAs; workgroup ids
//    are remapped so each XCD (ids are dealt round-robin over the 8 XCDs)
//    owns a contiguous run of tiles, grouped 8 tile-rows at a time for L2
//    reuse of the B panel; the epilogue works on the accumulators before the
//    single store.
//
// The fp32 kernel keeps each operand's global memory order in LDS (no
// transposing stores): k-contiguous operands are read back as float4 along k,
// row-contiguous operands as four scalars.  Within a 16-slab, lane half h of
// MFMA step q of group g consumes k = 8g + 4h + q for BOTH operands, a fixed
// bijection, so the contraction is unchanged.
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "split3.h"

namespace nship {

constexpr int BM = 128, BN = 128, BK = 16;  // the fp32 kernel's tile (2x2 waves of 64x64)
constexpr int KPAD = 4;    // pitch of k-contiguous rows: 20 floats
constexpr int RPAD = 4;    // pitch of row-contiguous k rows: ROWS + 4 floats
constexpr int NT = 256;

// LDS layout of one ROWS x 16 operand tile.
template <bool KC, int ROWS>
struct TileLayout;
template <int ROWS>
struct TileLayout<true, ROWS> {  // [rows][k], k contiguous
  static constexpr int kSize = ROWS * (BK + KPAD);
  __device__ static int at(int row, int k) { return row * (BK + KPAD) + k; }
};
template <int ROWS>
struct TileLayout<false, ROWS> {  // [k][rows], rows contiguous
  static constexpr int kSize = BK * (ROWS + RPAD);
  __device__ static int at(int row, int k) { return k * (ROWS + RPAD) + row; }
};

// Global -> register staging of one ROWS x 16 operand tile by NTH threads.
//  KC: element (row, k) at base[row*ld + k]   (k contiguous)
//  MC: element (row, k) at base[k*ld + row]   (row contiguous)
// `rows` = extent of the row dimension (M or N), `K` = contraction extent.
// init() resolves what stays fixed over the K loop: with VEC, each thread's
// load addresses at k = 0 (row maps looked up once), so a slab's load is one
// add per float4; load<CHK = false> is for tiles whose rows and K slabs are
// all in range (no per-element checks).
template <bool KC, bool VEC, int ROWS, int NTH>
struct Stage {
  static constexpr int kVec = ROWS * BK / 4 / NTH;  // float4 per thread (VEC)
  static constexpr int kSca = ROWS * BK / NTH;      // floats per thread
  static constexpr int kPtr = VEC ? kVec : 1;
  float v[kSca];
  const float* p[kPtr];
  unsigned rin;  // VEC: bit i set = the rows of load i are in range
  // the arguments (the scalar path resolves them per element)
  const float* base_;
  const int* rmap_;
  int row0_, rows_;

  __device__ __forceinline__ static void vec_pos(int idx, int& r, int& k) {
    if (KC) { r = idx / (BK / 4); k = (idx % (BK / 4)) * 4; } else { k = idx / (ROWS / 4); r = (idx % (ROWS / 4)) * 4; }
  }
  // rmap (optional): row r of the operand is row rmap[r] of `base`.
  __device__ __forceinline__ void init(const float* __restrict__ base, int64_t ld, int row0, int rows, int t,
                       const int* __restrict__ rmap = nullptr) {
    base_ = base, rmap_ = rmap, row0_ = row0, rows_ = rows;
    if (VEC) {
      rin = 0;
#pragma unroll
      for (int i = 0; i < kPtr; i++) {
        int r, k;
        vec_pos(t + NTH * i, r, k);
        const int gr = row0 + r;
        const bool in = gr < rows;
        rin |= in ? 1u << i : 0u;  // whole float4 in or out: the contiguous extent is a multiple of 4
        const int64_t rr = !in ? 0 : rmap ? (int64_t)rmap[gr] : (int64_t)gr;
        p[i] = KC ? base + rr * ld + k : base + (int64_t)k * ld + (in ? gr : 0);
      }
    }
  }
  // K-blocked operand (kblk_ > 0, VEC only): slab k0 lies in block k0 / kblk_
  int kblk_ = 0;
  int64_t sk_ = 0;
  template <bool CHK = true>
  __device__ __forceinline__ void load(int64_t ld, int k0, int K, int t) {
    if (VEC) {
      int64_t kb = 0;
      int kl = k0;
      if (kblk_) {
        kb = (int64_t)(k0 / kblk_) * sk_;
        kl = k0 % kblk_;
      }
      const int64_t off = kb + (KC ? (int64_t)kl : (int64_t)kl * ld);
#pragma unroll
      for (int i = 0; i < kVec; i++) {
        float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
        bool ok = true;
        if (CHK) {
          int r, k;
          vec_pos(t + NTH * i, r, k);
          ok = ((rin >> i) & 1) && k0 + k < K;
        }
        if (ok) x = *reinterpret_cast<const float4*>(p[i] + off);
        v[4 * i + 0] = x.x; v[4 * i + 1] = x.y; v[4 * i + 2] = x.z; v[4 * i + 3] = x.w;
      }
    } else {
#pragma unroll
      for (int i = 0; i < kSca; i++) {
        const int idx = t + NTH * i;
        int r, k;
        if (KC) { r = idx / BK; k = idx % BK; } else { k = idx / ROWS; r = idx % ROWS; }
        const int gr = row0_ + r, gk = k0 + k;
        float x = 0.f;
        if (!CHK || (gr < rows_ && gk < K)) {
          const int64_t rr = rmap_ ? (int64_t)rmap_[gr] : (int64_t)gr;
          x = KC ? base_[rr * ld + gk] : base_[(int64_t)gk * ld + gr];
        }
        v[i] = x;
      }
    }
  }
  __device__ __forceinline__ void store(float* __restrict__ lds, int t) const {
    if (VEC) {
#pragma unroll
      for (int i = 0; i < kVec; i++) {
        const int idx = t + NTH * i;
        int r, k;
        if (KC) { r = idx / (BK / 4); k = (idx % (BK / 4)) * 4; } else { k = idx / (ROWS / 4); r = (idx % (ROWS / 4)) * 4; }
        float* p = lds + TileLayout<KC, ROWS>::at(r, k);
        *reinterpret_cast<float4*>(p) = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < kSca; i++) {
        const int idx = t + NTH * i;
        int r, k;
        if (KC) { r = idx / BK; k = idx % BK; } else { k = idx / ROWS; r = idx % ROWS; }
        lds[TileLayout<KC, ROWS>::at(r, k)] = v[i];
      }
    }
  }
};

// Four operand values of one lane for MFMA steps q = 0..3 of group g.
template <bool KC, int ROWS>
__device__ __forceinline__ void read_frag(const float* __restrict__ lds, int row, int kb, float f[4]) {
  if (KC) {
    const float4 x = *reinterpret_cast<const float4*>(lds + TileLayout<true, ROWS>::at(row, kb));
    f[0] = x.x; f[1] = x.y; f[2] = x.z; f[3] = x.w;
  } else {
#pragma unroll
    for (int q = 0; q < 4; q++) f[q] = lds[TileLayout<false, ROWS>::at(row, kb + q)];
  }
}

// Workgroup b of T -> a linear index such that each XCD (ids are dealt
// round-robin over the 8 XCDs) owns one contiguous run; a bijection on [0, T).
__device__ __forceinline__ int xcd_linear(int b, int T) {
  const int per = T >> 3, rem = T & 7;
  const int x = b & 7, i = b >> 3;
  return x * per + (x < rem ? x : rem) + i;
}

// Logical tile of workgroup b: XCD-contiguous runs, then 8-row groups.
__device__ __forceinline__ void tile_of(int b, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int L = xcd_linear(b, tiles_m * tiles_n);
  const int group = 8 * tiles_n;
  const int first_m = (L / group) * 8;
  const int gsize = min(tiles_m - first_m, 8);
  const int in = L % group;
  tm = first_m + in % gsize;
  tn = in / gsize;
}

// Plain epilogue C = acc * act'(aux) for one wave's TM x TN blocks of 32x32
// from (mw, nw) (aux with C's row and column indices, pitch ldaux): the aux
// values are loaded one block ahead of that block's stores (the loads of
// block b + 1 are in flight while block b is stored).  Its own loop nest, so
// that the main epilogue's loops stay fully unrolled and the accumulators in
// registers.
template <int CODE, int TM, int TN>
__device__ __forceinline__ void store_act_grad(const floatx16 (&acc)[TM][TN], const GemmArgs& g, float* __restrict__ C,
                                               int mw, int nw, int l32, int kh, int m_end) {
  if (g.mask_in) {
    // relu' from the sign bits: one 16-bit load per lane and 32x32 block,
    // bit v for the lane's accumulator v (the layout the forward wrote)
    unsigned bits[TM * TN];
#pragma unroll
    for (int blk = 0; blk < TM * TN; blk++) {
      const int col = nw + (blk % TN) * 32 + l32;
      const int rb = mw + (blk / TN) * 32;
      bits[blk] = col < g.N && rb < m_end ? g.mask_in[(int64_t)(2 * (rb / 32) + kh) * g.ldmask + col] : 0u;
    }
#pragma unroll
    for (int blk = 0; blk < TM * TN; blk++) {
      const int r = blk / TN, c = blk % TN;
      const int col = nw + c * 32 + l32;
      const int row0 = mw + r * 32 + 4 * kh;
      const bool cin = col < g.N;
      float* cp = C + (int64_t)row0 * g.ldc + col;
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int dr = 8 * (v >> 2) + (v & 3);
        if (cin && row0 + dr < m_end) cp[(int64_t)dr * g.ldc] = acc[r][c][v] * ((bits[blk] >> v) & 1u ? 1.f : 0.f);
      }
    }
    return;
  }
  float au[2][16];
  auto load = [&](int blk, float(&dst)[16]) {
    const int col = nw + (blk % TN) * 32 + l32;
    const int row0 = mw + (blk / TN) * 32 + 4 * kh;
    const bool cin = col < g.N;
    const float* ap = g.aux + (int64_t)row0 * g.ldaux + col;
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int dr = 8 * (v >> 2) + (v & 3);
      dst[v] = cin && row0 + dr < m_end ? ap[(int64_t)dr * g.ldaux] : 0.f;
    }
  };
  load(0, au[0]);
#pragma unroll
  for (int blk = 0; blk < TM * TN; blk++) {
    if (blk + 1 < TM * TN) load(blk + 1, au[(blk + 1) & 1]);
    const int r = blk / TN, c = blk % TN;
    const int col = nw + c * 32 + l32;
    const int row0 = mw + r * 32 + 4 * kh;
    const bool cin = col < g.N;
    float* cp = C + (int64_t)row0 * g.ldc + col;
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int dr = 8 * (v >> 2) + (v & 3);
      if (cin && row0 + dr < m_end) cp[(int64_t)dr * g.ldc] = acc[r][c][v] * act_deriv(au[blk & 1][v], CODE);
    }
  }
}

// Sign bits of the pre-activation for a relu gradient later (the layout of
// GemmArgs::mask_out): each lane's 16 rows of a 32x32 block in one 16-bit
// value.  Its own loop nest, as store_act_grad.
template <int TM, int TN>
__device__ __forceinline__ void store_relu_bits(const floatx16 (&acc)[TM][TN], const GemmArgs& g, int mw, int nw,
                                                int l32, int kh, int m_end) {
#pragma unroll
  for (int r = 0; r < TM; r++)
#pragma unroll
    for (int c = 0; c < TN; c++) {
      const int col = nw + c * 32 + l32;
      const int rb = mw + r * 32;
      unsigned bits = 0u;
#pragma unroll
      for (int v = 0; v < 16; v++) bits |= (acc[r][c][v] > 0.f ? 1u : 0u) << v;
      if (col < g.N && rb < m_end) g.mask_out[(int64_t)(2 * (rb / 32) + kh) * g.ldmask + col] = (uint16_t)bits;
    }
}

// What one workgroup computes: C[m0.., n0..] over k in [kbeg, kend).
struct Job {
  const float* A;
  const float* B;
  float* C;
  int kbeg, kend, m0, n0, m_end;
};

// The job of this workgroup under g's mode (batch, K-grouped, K-chunked,
// split K, grouped) for BMT x BNT tiles; false: nothing to do (uniform).
template <int BMT, int BNT>
__device__ __forceinline__ bool tile_job(const GemmArgs& g, Job& j) {
  j.A = g.A + (int64_t)blockIdx.y * g.sA;
  j.B = g.B + (int64_t)blockIdx.y * g.sB;
  j.C = g.C + (int64_t)blockIdx.y * g.sC;
  j.m_end = g.M;
  // K-grouped: group blockIdx.y contracts over k in [kseg[y], kseg[y+1]).
  j.kbeg = 0;
  j.kend = g.K;
  if (g.kseg) {
    j.kbeg = g.kseg[blockIdx.y];
    j.kend = g.kseg[blockIdx.y + 1];
  }
  if (g.kitems) {
    if ((int)blockIdx.y >= *g.nkitems) return false;
    const int* it = g.kitems + 4 * blockIdx.y;
    j.kbeg = it[1];
    j.kend = it[2];
    j.A = g.A;
    j.B = g.B;
    j.C = it[3] < 0 ? g.C + (int64_t)it[0] * g.sC : g.kpart + (int64_t)it[3] * g.sC;
  }
  if (g.kchunk) {
    j.kbeg = (int)blockIdx.z * g.kchunk;
    j.kend = min(g.K, j.kbeg + g.kchunk);
    j.C += (int64_t)blockIdx.z * g.sCk;
  }
  if (g.groups) {
    // Grouped: tile entry -> (group, m tile); rows [seg[e], seg[e+1]) of the
    // group, B advanced by e * sBg.  Entries run XCD-contiguously with all
    // their n tiles, so a gathered A tile is fetched into one XCD's L2 only.
    // The grid is an upper bound: the workgroups past the device-side tile
    // count exit (uniformly), and the rest are spread over the 8 XCDs by
    // that count, not by the grid size, so each XCD gets an equal share.
    const int T = *g.ntiles * g.tiles_n;
    if ((int)blockIdx.x >= T) return false;
    const int L = xcd_linear(blockIdx.x, T);
    const int entry = L / g.tiles_n;
    const int e = g.tiles[2 * entry], mt = g.tiles[2 * entry + 1];
    j.m0 = g.seg[e] + mt * BMT;
    j.m_end = g.seg[e + 1];
    j.n0 = (L % g.tiles_n) * BNT;
    j.B += (int64_t)e * g.sBg;
  } else {
    int tm, tn;
    tile_of(blockIdx.x, g.tiles_m, g.tiles_n, tm, tn);
    j.m0 = tm * BMT;
    j.n0 = tn * BNT;
  }
  return true;
}

template <int TM, int TN>
__device__ __forceinline__ void zero_acc(floatx16 (&acc)[TM][TN]) {
#pragma unroll
  for (int r = 0; r < TM; r++)
#pragma unroll
    for (int c = 0; c < TN; c++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[r][c][v] = 0.f;
}

// Floats of LDS the fp32 loop needs for a BMT x BNT tile.
template <bool TA, bool TB, int BMT, int BNT>
constexpr int f32_lds_floats() {
  return 2 * (TileLayout<!TA, BMT>::kSize + TileLayout<TB, BNT>::kSize);
}

// fp32-MFMA K loop of one tile, WM x WN waves of TM x TN 32x32 blocks.
template <bool TA, bool TB, bool VEC, int WM, int WN, int TM, int TN>
__device__ __forceinline__ void mainloop_f32(const GemmArgs& g, const Job& j, float* __restrict__ smem,
                                             floatx16 (&acc)[TM][TN]) {
  constexpr int BMT = 32 * WM * TM, BNT = 32 * WN * TN, NTT = 64 * WM * WN;
  constexpr bool AKC = !TA, BKC = TB;
  constexpr int ASZ = TileLayout<AKC, BMT>::kSize, BSZ = TileLayout<BKC, BNT>::kSize;
  // buffer b: A tile at smem + b*(ASZ+BSZ), B tile right after it
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave / WN, wn = wave % WN, l32 = lane & 31, kh = lane >> 5;
  const int64_t lda = g.lda, ldb = g.ldb;
  const int kbeg = j.kbeg, kend = j.kend;
  zero_acc(acc);
  Stage<AKC, VEC, BMT, NTT> sa;
  Stage<BKC, VEC, BNT, NTT> sb;
  const int nk = (kend - kbeg + BK - 1) / BK;
  sa.init(j.A, lda, j.m0, j.m_end, t, g.a_rows);
  sb.init(j.B, ldb, j.n0, g.N, t);
  sa.kblk_ = g.kblk;
  sa.sk_ = g.sAk;
  sb.kblk_ = g.kblk;
  sb.sk_ = g.sBk;
  sa.load(lda, kbeg, kend, t);
  sb.load(ldb, kbeg, kend, t);
  sa.store(smem, t);
  sb.store(smem + ASZ, t);
  __syncthreads();
  // every row and K slab of the tile in range: loads without checks
  const bool full = j.m0 + BMT <= j.m_end && j.n0 + BNT <= g.N && (kend - kbeg) % BK == 0;

  for (int kt = 0; kt < nk; kt++) {
    const int cur = kt & 1;
    const bool more = kt + 1 < nk;
    if (more) {
      if (full) {
        sa.template load<false>(lda, kbeg + (kt + 1) * BK, kend, t);
        sb.template load<false>(ldb, kbeg + (kt + 1) * BK, kend, t);
      } else {
        sa.load(lda, kbeg + (kt + 1) * BK, kend, t);
        sb.load(ldb, kbeg + (kt + 1) * BK, kend, t);
      }
    }
    const float* as = smem + cur * (ASZ + BSZ);
    const float* bs = as + ASZ;
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int g2 = 0; g2 < 2; g2++) {
      const int kb = 8 * g2 + 4 * kh;
      float fa[TM][4], fb[TN][4];
#pragma unroll
      for (int r = 0; r < TM; r++) read_frag<AKC, BMT>(as, (wm * TM + r) * 32 + l32, kb, fa[r]);
#pragma unroll
      for (int c = 0; c < TN; c++) read_frag<BKC, BNT>(bs, (wn * TN + c) * 32 + l32, kb, fb[c]);
#pragma unroll
      for (int q = 0; q < 4; q++)
#pragma unroll
        for (int r = 0; r < TM; r++)
#pragma unroll
          for (int c = 0; c < TN; c++)
            acc[r][c] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[r][q], fb[c][q], acc[r][c], 0, 0, 0);
    }
    __builtin_amdgcn_s_setprio(0);
    if (more) {
      float* nxt = smem + (cur ^ 1) * (ASZ + BSZ);
      sa.store(nxt, t);
      sb.store(nxt + ASZ, t);
    }
    __syncthreads();
  }
}

// Epilogue of one wave's TM x TN 32x32 blocks, the first at (mw, nw).
// PLAIN: no row scatter, no row scale; epilogue kEpiAct (with the
// pre-activation / activation pair when C2 is set), kEpiActGrad or kEpiAccum.
// ACTS: bit c set = activation c may be asked for (each costs a copy of the
// stores of every accumulator).
constexpr unsigned kAllActs = 0xff;
template <bool PLAIN, unsigned ACTS, int TM, int TN>
__device__ __forceinline__ void store_tile(const floatx16 (&acc)[TM][TN], const GemmArgs& g, float* __restrict__ C,
                                           int mw, int nw, int l32, int kh, int m_end) {
  const int N = g.N;
  const int64_t ldc = g.ldc;
  // Accumulator v of lane (l32, kh) in a 32x32 block sits at
  // row 8*(v/4) + 4*kh + v%4, column l32.
  if constexpr (PLAIN) {
    if (g.mode == kEpiActGrad) {
      // C = acc * relu'(aux): the only activation gradient the plain path
      // takes (plain_act_grad)
      store_act_grad<kActRelu>(acc, g, C, mw, nw, l32, kh, m_end);
      return;
    }
    if (g.mask_out) store_relu_bits(acc, g, mw, nw, l32, kh, m_end);
    // plain stores, the activation resolved once per 32x32 block
#pragma unroll
    for (int r = 0; r < TM; r++)
#pragma unroll
      for (int c = 0; c < TN; c++) {
        const int col = nw + c * 32 + l32;
        const int row0 = mw + r * 32 + 4 * kh;
        float* cp = C + (int64_t)row0 * ldc + col;
        const bool cin = col < N;
#define NSH_STORE16(CODE)                                                          \
  _Pragma("unroll") for (int v = 0; v < 16; v++) {                                 \
    const int dr = 8 * (v >> 2) + (v & 3);                                         \
    if (cin && row0 + dr < m_end) cp[(int64_t)dr * ldc] = act_apply(acc[r][c][v], CODE); \
  }
        if (g.mode == kEpiAccum) {
#pragma unroll
          for (int v = 0; v < 16; v++) {
            const int dr = 8 * (v >> 2) + (v & 3);
            if (cin && row0 + dr < m_end) cp[(int64_t)dr * ldc] += acc[r][c][v];
          }
          continue;
        }
        if (g.C2) {
          // pre-activation to C, then the activation to C2 below
#pragma unroll
          for (int v = 0; v < 16; v++) {
            const int dr = 8 * (v >> 2) + (v & 3);
            if (cin && row0 + dr < m_end) cp[(int64_t)dr * ldc] = acc[r][c][v];
          }
          cp = g.C2 + (int64_t)blockIdx.y * g.sC + (int64_t)row0 * ldc + col;
        }
        switch (g.act) {
          case kActRelu: if constexpr ((ACTS >> kActRelu) & 1) { NSH_STORE16(kActRelu); } break;
          case kActLeaky: if constexpr ((ACTS >> kActLeaky) & 1) { NSH_STORE16(kActLeaky); } break;
          case kActSigmoid: if constexpr ((ACTS >> kActSigmoid) & 1) { NSH_STORE16(kActSigmoid); } break;
          case kActTanh: if constexpr ((ACTS >> kActTanh) & 1) { NSH_STORE16(kActTanh); } break;
          case kActSilu: if constexpr ((ACTS >> kActSilu) & 1) { NSH_STORE16(kActSilu); } break;
          case kActGelu: if constexpr ((ACTS >> kActGelu) & 1) { NSH_STORE16(kActGelu); } break;
          case kActGeluMoe: if constexpr ((ACTS >> kActGeluMoe) & 1) { NSH_STORE16(kActGeluMoe); } break;
          default: NSH_STORE16(kActId); break;
        }
#undef NSH_STORE16
      }
    return;
  }
  // General epilogue (row scatter, row scale, activation gradient or
  // accumulate).  The rows a lane holds in a 32-row block share their output
  // row and scale between the two column blocks: they are looked up once,
  // eight rows at a time with all eight loads in flight together.
#pragma unroll
  for (int r = 0; r < TM; r++)
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int rbase = mw + r * 32 + 16 * h + 4 * kh;
      int crow[8];
      float rs[8];
      // rows past m_end read row m_end - 1's entries (the tile has rows) and are
      // then marked -1: the loads carry no branch and issue together
#pragma unroll
      for (int u = 0; u < 8; u++) crow[u] = min(rbase + 8 * (u >> 2) + (u & 3), m_end - 1);
      if (g.c_rows) {
#pragma unroll
        for (int u = 0; u < 8; u++) crow[u] = g.c_rows[crow[u]];
      }
#pragma unroll
      for (int u = 0; u < 8; u++) rs[u] = g.row_scale ? g.row_scale[crow[u]] : 1.f;
#pragma unroll
      for (int u = 0; u < 8; u++)
        if (rbase + 8 * (u >> 2) + (u & 3) >= m_end) crow[u] = -1;
#pragma unroll
      for (int c = 0; c < TN; c++) {
        const int col = nw + c * 32 + l32;
        if (col >= N) continue;
#pragma unroll
        for (int u = 0; u < 8; u++) {
          if (crow[u] < 0) continue;
          const int row = rbase + 8 * (u >> 2) + (u & 3);
          float* dst = C + (int64_t)crow[u] * ldc + col;
          const float x = acc[r][c][8 * h + u];
          const float a = g.row_scale ? x * rs[u] : x;
          if (g.mode == kEpiAccum) {
            *dst = *dst + a;
          } else if constexpr (ACTS == 1u) {
            *dst = a;
          } else {
            if (g.mode == kEpiAct) *dst = act_apply(a, g.act);
            else *dst = a * act_deriv(g.aux[(int64_t)row * g.ldaux + col], g.act);
          }
        }
      }
    }
}

// opA(A)[m,k]: TA ? A[k*lda+m] : A[m*lda+k]   (KC for A <=> !TA)
// opB(B)[k,n]: TB ? B[n*ldb+k] : B[k*ldb+n]   (KC for B <=>  TB)
// The fp32 kernel: 256 threads = 2x2 waves of 64x64.  It takes what the split
// kernel does not (bf3_takes): operands that cannot be read as float4, and
// products too small to be worth the split.
template <bool TA, bool TB, bool VEC, bool PLAIN>
__global__ __launch_bounds__(NT, VEC ? 4 : 1) void gemm_f32_kernel(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) float smem[f32_lds_floats<TA, TB, BM, BN>()];
  Job j;
  if (!tile_job<BM, BN>(g, j)) return;
  floatx16 acc[2][2];
  mainloop_f32<TA, TB, VEC, 2, 2, 2, 2>(g, j, smem, acc);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  store_tile<PLAIN, kAllActs>(acc, g, j.C, j.m0 + (wave >> 1) * 64, j.n0 + (wave & 1) * 64, lane & 31, lane >> 5, j.m_end);
}

// ---- three-piece bf16 kernel ---------------------------------------------------

// LDS layout of one operand's 16-wide K slab: [piece][k / 8][row] chunks of 8
// bf16.  The two k-halves are 64 bytes further apart than ROWS chunks, so the
// staging stores of a k-contiguous operand (8 lanes = 4 rows x 2 halves)
// cover all banks.
template <int ROWS>
struct Bf3Layout {
  static constexpr int kHalf = ROWS * 16 + 64;
  static constexpr int kPiece = 2 * kHalf;
  static constexpr int kBytes = 3 * kPiece;
};

// Global -> register -> LDS staging of one ROWS x 16 slab by NTH threads, W
// consecutive k of one row at a time: two float4 of a k-contiguous operand,
// or W loads a row pitch apart of a row-contiguous one, whose consecutive
// rows lie in consecutive lanes.  The slabs are taken in order.  No load and
// no step between slabs branches, so the K loop's body is one block in which
// the split of one slab is scheduled among the MFMAs of another: CHK = true
// (rows or a K slab past the end) reads from an address in range instead and
// puts zeros in at the store.
template <bool KC, int ROWS, int NTH>
struct Bf3Stage {
  static constexpr int W = ROWS * 2 >= NTH ? 8 : 4;
  static constexpr int NC = BK / W;             // W-chunks of a slab
  static constexpr int kN = ROWS * NC / NTH;    // chunks per thread
  static_assert(kN >= 1 && kN * NTH == ROWS * NC, "the chunks divide evenly");
  float v[2][kN][W];   // two slabs in flight (even, odd)
  const float* p[kN];  // chunk i of slab 0: its row (in range), or (KC false) the tile's first row
  uint32_t ro[kN];     // KC false: byte offset of chunk i's row (in range) from there
  unsigned rin;        // bit i set: the row of chunk i is in range
  int64_t off, wrap;   // of the next slab; what the end of a K block adds
  int k, inblk, kblk;  // next slab, its place in its K block, the block's length
  int lim[2];          // k of the held slabs below lim exist

  __device__ __forceinline__ static void pos(int idx, int& r, int& kc) {
    // (KC false: ROWS is a multiple of the wave, so kc is uniform and the
    // loads' addresses are scalar but for the row offset)
    if (KC) { r = idx / NC; kc = idx % NC; } else { kc = __builtin_amdgcn_readfirstlane(idx / ROWS); r = idx % ROWS; }
  }
  // rmap (optional, KC): row r of the operand is row rmap[r] of `base`.  kb > 0:
  // K blocks of kb steps, sk floats apart.
  __device__ __forceinline__ void init(const float* __restrict__ base, int64_t ld, int row0, int rows, int kbeg, int t,
                                       const int* __restrict__ rmap, int kb, int64_t sk) {
    rin = 0;
#pragma unroll
    for (int i = 0; i < kN; i++) {
      int r, kc;
      pos(t + NTH * i, r, kc);
      const int gr = row0 + r;
      const bool in = gr < rows;
      rin |= in ? 1u << i : 0u;
      if (KC) {
        p[i] = base + (!in ? 0 : rmap ? (int64_t)rmap[gr] : (int64_t)gr) * ld;
      } else {
        p[i] = base + row0 + (int64_t)(kc * W) * ld;
        ro[i] = (uint32_t)min(r, rows - 1 - row0) * 4u;
      }
    }
    kblk = kb > 0 ? kb : INT32_MAX;
    k = kbeg;
    inblk = kb > 0 ? kbeg % kb : kbeg;
    const int64_t unit = KC ? 1 : ld;
    wrap = kb > 0 ? sk - kb * unit : 0;
    off = (kb > 0 ? kbeg / kb * wrap : 0) + kbeg * unit;
  }
  // The next slab into set Z, then on by one; past the last one (k >= kend -
  // BK) it stays (nothing reads the slab then loaded again).
  template <bool CHK, int Z>
  __device__ __forceinline__ void load(int64_t ld, int kend, int t) {
    lim[Z] = kend - k;
#pragma unroll
    for (int i = 0; i < kN; i++) {
      int r, kc;
      pos(t + NTH * i, r, kc);
      if (KC) {
#pragma unroll
        for (int u = 0; u < W; u += 4) {
          // (whole float4: kend and k are multiples of 4)
          const int ku = CHK ? min(kc * W + u, lim[Z] - 4) : kc * W + u;
          const float4 x = *reinterpret_cast<const float4*>(p[i] + off + ku);
          v[Z][i][u] = x.x; v[Z][i][u + 1] = x.y; v[Z][i][u + 2] = x.z; v[Z][i][u + 3] = x.w;
        }
      } else {
        const float* q = p[i] + off;
#pragma unroll
        for (int u = 0; u < W; u++) {
          if (CHK) q = p[i] + off + (int64_t)min(u, lim[Z] - 1 - kc * W) * ld;
          v[Z][i][u] = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(q) + ro[i]);
          if (!CHK) q += ld;
        }
      }
    }
    const bool more = k + BK < kend;
    k += more ? BK : 0;
    off += more ? (KC ? (int64_t)BK : BK * ld) : 0;
    inblk += more ? BK : 0;
    const bool next = inblk >= kblk;
    off += next ? wrap : 0;
    inblk = next ? 0 : inblk;
  }
  template <bool CHK, int Z>
  __device__ __forceinline__ void store(char* __restrict__ lds, int t, bool& bad) {
    using L = Bf3Layout<ROWS>;
#pragma unroll
    for (int i = 0; i < kN; i++) {
      int r, kc;
      pos(t + NTH * i, r, kc);
      uint32_t w0[W / 2], w1[W / 2], w2[W / 2];
#pragma unroll
      for (int u = 0; u < W; u++) {
        if (CHK) v[Z][i][u] = ((rin >> i) & 1) && kc * W + u < lim[Z] ? v[Z][i][u] : 0.f;
        v[Z][i][u] *= kSplitUp;
      }
      split_run<W>(v[Z][i], w0, w1, w2, bad);
      if constexpr (W == 8) {
        char* d = lds + kc * L::kHalf + r * 16;
        *reinterpret_cast<uintx4*>(d) = uintx4{w0[0], w0[1], w0[2], w0[3]};
        *reinterpret_cast<uintx4*>(d + L::kPiece) = uintx4{w1[0], w1[1], w1[2], w1[3]};
        *reinterpret_cast<uintx4*>(d + 2 * L::kPiece) = uintx4{w2[0], w2[1], w2[2], w2[3]};
      } else {
        char* d = lds + (kc >> 1) * L::kHalf + r * 16 + (kc & 1) * 8;
        *reinterpret_cast<uintx2*>(d) = uintx2{w0[0], w0[1]};
        *reinterpret_cast<uintx2*>(d + L::kPiece) = uintx2{w1[0], w1[1]};
        *reinterpret_cast<uintx2*>(d + 2 * L::kPiece) = uintx2{w2[0], w2[1]};
      }
    }
  }
};

// The activations that the split kernel's epilogues hold, by use: a dense
// layer's (NN) all; transposed products (gradients) and the general epilogue
// none; an expert layer's GELU.  bf3_takes sends the rest elsewhere.
constexpr unsigned kActsNone = 1u << kActId;
constexpr unsigned kActsMoe = 1u << kActId | 1u << kActGeluMoe;

// WM x WN waves, each 2 x 2 blocks of 32x32.
//
// Two accumulators a block: `acc` takes the products of the leading pieces,
// `lo` the other five, and they are added once at the end.  An MFMA aligns its
// products to its accumulator and truncates below two guard bits, which
// shrinks sums of mixed sign by about 2^-27 sqrt(K); in `lo`, 2^-8 the size,
// both that and the roundings vanish, and `acc` is rounded once per 16 of K.
// Error against float64, one accumulator -> two (fp32 MFMA): K = 4096 1.0e-6
// -> 4.0e-7 (1.1e-6), K = 512 3.4e-7 -> 1.3e-7 (4.1e-7).
//
// Bound by the matrix cores and the power they draw: a register-only loop of
// the same MFMAs runs at 1.8 PFLOP/s, 300 TFLOP/s of fp32 products; 8192 x
// 4096 x 4096 runs at 216 (fp32 MFMA 127), 16384 x 512 x 8192 at 203 (126).
// 64x64 per wave is what two accumulators leave room for at two waves per
// SIMD; 128x64 per wave with one accumulator ran at 234, with the error above.
// Two slabs of loads are in flight: a load has two slabs of MFMAs to arrive
// (one: 1500 us on that product against 1390, 197 against 184 on 16384 x 512 x
// 2048, same box).  Measured and not kept: the two waves of a SIMD taking turns
// at the matrix core, one barrier per turn (1475 us).
template <bool TA, bool TB, bool PLAIN, unsigned ACTS, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_bf3_kernel(GemmArgs g) {
  constexpr int TM = 2, TN = 2;
  constexpr int BMT = 32 * WM * TM, BNT = 32 * WN * TN, NTT = 64 * WM * WN;
  using LA = Bf3Layout<BMT>;
  using LB = Bf3Layout<BNT>;
  constexpr int kBuf = LA::kBytes + LB::kBytes;
  constexpr int kF32 = 4 * f32_lds_floats<TA, TB, BMT, BNT>();
  __shared__ __attribute__((aligned(16))) char smem[2 * kBuf > kF32 ? 2 * kBuf : kF32];
  Job j;
  if (!tile_job<BMT, BNT>(g, j)) return;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave / WN, wn = wave % WN, l32 = lane & 31, kh = lane >> 5;
  const int kbeg = j.kbeg, kend = j.kend, nk = (kend - kbeg + BK - 1) / BK;
  const int64_t lda = g.lda, ldb = g.ldb;
  floatx16 acc[TM][TN];
  zero_acc(acc);
  bool bad = false;
  {
    floatx16 lo[TM][TN];
    zero_acc(lo);
    auto kloop = [&](auto chk) {
      constexpr bool CHK = decltype(chk)::value;
      Bf3Stage<!TA, BMT, NTT> sa;
      Bf3Stage<TB, BNT, NTT> sb;
      sa.init(j.A, lda, j.m0, j.m_end, kbeg, t, g.a_rows, g.kblk, g.sAk);
      sb.init(j.B, ldb, j.n0, g.N, kbeg, t, nullptr, g.kblk, g.sBk);
      auto load = [&](auto z) {
        constexpr int Z = decltype(z)::value;
        sa.template load<CHK, Z>(lda, kend, t);
        sb.template load<CHK, Z>(ldb, kend, t);
      };
      auto store = [&](auto z, char* __restrict__ to) {
        constexpr int Z = decltype(z)::value;
        sa.template store<CHK, Z>(to, t, bad);
        sb.template store<CHK, Z>(to + LA::kBytes, t, bad);
      };
      using Even = std::integral_constant<int, 0>;
      using Odd = std::integral_constant<int, 1>;
      load(Even{});
      load(Odd{});
      store(Even{}, smem);
      load(Even{});
      __syncthreads();
      // slab kt; slab kt + 1 (set z) to LDS, slab kt + 3 into its registers
      auto slab = [&](int kt, auto z) {
        const char* as = smem + (kt & 1) * kBuf + kh * LA::kHalf + (wm * TM * 32 + l32) * 16;
        const char* bs = smem + (kt & 1) * kBuf + LA::kBytes + kh * LB::kHalf + (wn * TN * 32 + l32) * 16;
        char* nx = smem + ((kt + 1) & 1) * kBuf;
        bf16x8 fa[TM][3], fb[TN][3];
#pragma unroll
        for (int c = 0; c < TN; c++)
#pragma unroll
          for (int p = 0; p < 3; p++) fb[c][p] = *reinterpret_cast<const bf16x8*>(bs + c * 512 + p * LB::kPiece);
#pragma unroll
        for (int r = 0; r < TM; r++)
#pragma unroll
          for (int p = 0; p < 3; p++) fa[r][p] = *reinterpret_cast<const bf16x8*>(as + r * 512 + p * LA::kPiece);
#pragma unroll
        for (int r = 0; r < TM; r++) {
#pragma unroll
          for (int q = 0; q < 5; q++)
#pragma unroll
            for (int c = 0; c < TN; c++)
              lo[r][c] =
                  __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[r][kPieceA[q]], fb[c][kPieceB[q]], lo[r][c], 0, 0, 0);
#pragma unroll
          for (int c = 0; c < TN; c++)
            acc[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[r][0], fb[c][0], acc[r][c], 0, 0, 0);
        }
        store(z, nx);
        load(z);
        __syncthreads();
      };
      for (int kt = 0; kt < nk; kt += 2) {
        slab(kt, Odd{});
        if (kt + 1 < nk) slab(kt + 1, Even{});
      }
    };
    // every row and K slab of the tile in range: no checks
    if (nk > 0) {
      if (j.m0 + BMT <= j.m_end && j.n0 + BNT <= g.N && (kend - kbeg) % BK == 0) kloop(std::false_type{});
      else kloop(std::true_type{});
    }
#pragma unroll
    for (int r = 0; r < TM; r++)
#pragma unroll
      for (int c = 0; c < TN; c++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
          acc[r][c][v] = (acc[r][c][v] + lo[r][c][v]) * kSplitDown;
          bad |= !(fabsf(acc[r][c][v]) <= 3.402823466e38f);
        }
  }
  // a tile with values the split cannot hold, or whose sums left the range
  if (__syncthreads_or(bad))
    mainloop_f32<TA, TB, true, WM, WN, TM, TN>(g, j, reinterpret_cast<float*>(smem), acc);
  store_tile<PLAIN, ACTS>(acc, g, j.C, j.m0 + wm * TM * 32, j.n0 + wn * TN * 32, l32, kh, j.m_end);
}

// ---- products too small for the tiled kernels ------------------------------------

// Few output tiles leave most CUs idle and every K slab of the tiled kernels
// waits for its loads (about 1 us a slab with one workgroup on a CU).  Here a
// workgroup takes 32 TM x 32 outputs, its 8 waves deal out the 16-steps of K,
// each loading its operands straight into registers, kSmallU steps at a time
// and without barriers, and the eight partial sums meet in LDS.  Bound by the
// memory traffic (each workgroup reads its 32 columns of B once, and A through
// L2) and, below a few microseconds, by its one or two round trips.
constexpr int kSmallW = 8;  // waves, each every 8th step of K
constexpr int kSmallU = 4;  // steps of loads in flight per wave

// One 32 x 16 operand step in registers: this lane's row, 8 consecutive k.
template <bool KC>
struct SmallStep {
  float v[8];
  // row: this lane's (in range), k: first of its 8; kend: the contraction's end
  __device__ __forceinline__ void load(const float* __restrict__ base, int64_t ld, int64_t row, int64_t kb, int k,
                                       int kloc, int kend) {
    if (KC) {
      const float* p = base + row * ld + kb;
#pragma unroll
      for (int u = 0; u < 8; u += 4) {
        // (whole float4: kend is a multiple of 4)
        const bool in = k + u < kend;
        const float4 x = *reinterpret_cast<const float4*>(p + (in ? kloc + u : 0));
        v[u] = in ? x.x : 0.f; v[u + 1] = in ? x.y : 0.f; v[u + 2] = in ? x.z : 0.f; v[u + 3] = in ? x.w : 0.f;
      }
    } else {
      const float* p = base + row + kb;
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const bool in = k + u < kend;
        const float x = p[(int64_t)(in ? kloc + u : 0) * ld];
        v[u] = in ? x : 0.f;
      }
    }
  }
};

// PIECES: three-piece bf16 with two accumulators, as gemm_bf3_kernel; else, and
// for what the pieces cannot hold, fp32 MFMA (step j of a 16-step pairs k = j
// and 8 + j).  Epilogue: kEpiAct (with the pre-activation / activation pair),
// kEpiActGrad from aux, kEpiAccum.
template <bool TA, bool TB, bool PIECES, int TM>
__global__ __launch_bounds__(64 * kSmallW, 2) void gemm_small_kernel(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) float part[kSmallW][TM * 32 * 32];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, l32 = lane & 31, kh = lane >> 5;
  const int M = g.M, N = g.N, K = g.K;
  const int m0 = (int)(blockIdx.x / g.tiles_n) * 32 * TM, n0 = (int)(blockIdx.x % g.tiles_n) * 32;
  const float* __restrict__ A = g.A + (int64_t)blockIdx.y * g.sA;
  const float* __restrict__ B = g.B + (int64_t)blockIdx.y * g.sB;
  int64_t ra[TM];
#pragma unroll
  for (int r = 0; r < TM; r++) ra[r] = min(m0 + r * 32 + l32, M - 1);
  const int64_t rb = min(n0 + l32, N - 1);
  const int steps = (K + 15) / 16;
  floatx16 acc[TM];
  bool bad = false;
  auto run = [&](auto pieces) {
    constexpr bool P3 = decltype(pieces)::value;
    floatx16 lo[TM];
#pragma unroll
    for (int r = 0; r < TM; r++)
#pragma unroll
      for (int v = 0; v < 16; v++) { acc[r][v] = 0.f; lo[r][v] = 0.f; }
    for (int s0 = w; s0 < steps; s0 += kSmallW * kSmallU) {
      SmallStep<!TA> a[kSmallU][TM];
      SmallStep<TB> b[kSmallU];
#pragma unroll
      for (int u = 0; u < kSmallU; u++) {
        if (s0 + u * kSmallW >= steps) break;  // (uniform)
        const int k = (s0 + u * kSmallW) * 16 + 8 * kh;
        const int blk = g.kblk ? k / g.kblk : 0, kloc = g.kblk ? k % g.kblk : k;
        const bool in = k < K;  // (not for the upper half of a last step of 8)
#pragma unroll
        for (int r = 0; r < TM; r++) a[u][r].load(A, g.lda, ra[r], in ? blk * g.sAk : 0, k, kloc, K);
        b[u].load(B, g.ldb, rb, in ? blk * g.sBk : 0, k, kloc, K);
      }
#pragma unroll
      for (int u = 0; u < kSmallU; u++) {
        if (s0 + u * kSmallW >= steps) break;
        if constexpr (P3) {
          bf16x8 fb[3], fa[TM][3];
          auto pieces_of = [&](float(&x)[8], bf16x8(&f)[3]) {
            uint32_t q[3][4];
#pragma unroll
            for (int j = 0; j < 8; j++) x[j] *= kSplitUp;
            split_run<8>(x, q[0], q[1], q[2], bad);
#pragma unroll
            for (int p = 0; p < 3; p++)
              f[p] = __builtin_bit_cast(bf16x8, uintx4{q[p][0], q[p][1], q[p][2], q[p][3]});
          };
          pieces_of(b[u].v, fb);
#pragma unroll
          for (int r = 0; r < TM; r++) {
            pieces_of(a[u][r].v, fa[r]);
#pragma unroll
            for (int q = 0; q < 5; q++)
              lo[r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[r][kPieceA[q]], fb[kPieceB[q]], lo[r], 0, 0, 0);
            acc[r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[r][0], fb[0], acc[r], 0, 0, 0);
          }
        } else {
#pragma unroll
          for (int j = 0; j < 8; j++)
#pragma unroll
            for (int r = 0; r < TM; r++)
              acc[r] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u][r].v[j], b[u].v[j], acc[r], 0, 0, 0);
        }
      }
    }
    if constexpr (P3) {
#pragma unroll
      for (int r = 0; r < TM; r++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
          acc[r][v] = (acc[r][v] + lo[r][v]) * kSplitDown;
          bad |= !(fabsf(acc[r][v]) <= 3.402823466e38f);
        }
    }
  };
  run(std::integral_constant<bool, PIECES>{});
  if constexpr (PIECES) {
    if (__syncthreads_or(bad)) run(std::false_type{});
  }
#pragma unroll
  for (int r = 0; r < TM; r++)
#pragma unroll
    for (int v = 0; v < 16; v++)
      part[w][(r * 32 + 8 * (v >> 2) + 4 * kh + (v & 3)) * 32 + l32] = acc[r][v];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TM * 2; i++) {
    const int e = t + 64 * kSmallW * i, row = m0 + e / 32, col = n0 + e % 32;
    float x = 0.f;
#pragma unroll
    for (int q = 0; q < kSmallW; q++) x += part[q][e];
    if (row < M && col < N) {
      const int64_t at = (int64_t)blockIdx.y * g.sC + (int64_t)row * g.ldc + col;
      if (g.mode == kEpiAccum) {
        g.C[at] += x;
      } else if (g.mode == kEpiActGrad) {
        g.C[at] = x * act_deriv(g.aux[(int64_t)row * g.ldaux + col], g.act);
      } else if (g.C2) {
        g.C[at] = x;
        g.C2[at] = act_apply(x, g.act);
      } else {
        g.C[at] = act_apply(x, g.act);
      }
    }
  }
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Whether both operands can be read as float4: each one's contiguous extent,
// leading dimension, batch stride and base 4-float aligned.  (K-grouped
// segments start anywhere, so a k-contiguous operand needs the scalar path
// there.)
static bool reads_float4(const GemmArgs& g, bool tA, bool tB) {
  const bool seg = g.kseg || g.kitems;
  const bool va = aligned16(g.A) && g.lda % 4 == 0 && g.sA % 4 == 0 && ((tA ? g.M : g.K) % 4 == 0) && (tA || !seg);
  const bool vb = aligned16(g.B) && g.ldb % 4 == 0 && g.sB % 4 == 0 && ((tB ? g.K : g.N) % 4 == 0) && (!tB || !seg);
  return va && vb && (!g.kblk || (g.sAk % 4 == 0 && g.sBk % 4 == 0));
}

// Whether gemm_small_kernel can read the operands: a row-contiguous one at any
// alignment, a k-contiguous one as float4; not both transposed.
static bool small_reads(const GemmArgs& g, bool tA, bool tB) {
  const bool ka = tA || (aligned16(g.A) && g.lda % 4 == 0 && g.sA % 4 == 0 && g.K % 4 == 0 && g.sAk % 4 == 0);
  const bool kb = !tB || (aligned16(g.B) && g.ldb % 4 == 0 && g.sB % 4 == 0 && g.K % 4 == 0 && g.sBk % 4 == 0);
  return ka && kb && !(tA && tB);
}

// Activation gradients the plain epilogue applies itself: ReLU's (the
// training MLPs'); the others take the general epilogue.
static bool plain_act_grad(const GemmArgs& g) { return g.mode == kEpiActGrad && g.aux && g.act == kActRelu; }

// Compute units of the current device (cached per device).
static int device_cus() {
  static int cus[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!cus[dev]) {
    int n = 0;
    cus[dev] = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0 ? n : 256;
  }
  return cus[dev];
}

// The split kernel takes every product of at least kBf3MinK steps that it can
// read as float4 and whose epilogue it holds.  Transposed both ways (no caller
// but the entry point), a transposed product with an activation and the
// general epilogue's activations stay on the fp32 kernel, and so do products
// that ask for it (GemmArgs::f32).
// Short K: one MFMA aligns its 16 products to the largest and drops what lies
// below fp32's last place there, and the split drops up to 2^-24 of a product
// (split3.h).  Over a long sum both are far below the roundings of the sum
// itself; a short one with a dominant term has up to 1.8 x 2^-24 instead of
// 1.0, and its product is bound by its memory traffic either way.
// Long sums against float64, 2-norm in units of 2^-24, fp32 MFMA -> this, 2048 x
// 2048 outputs: N(0, 1), K = 128 3.4 -> 1.1, 512 6.8 -> 2.1, 4096 9.6 -> 4.6; e^(2
// N(0, 1)), 512 12.5 -> 2.7, 4096 32 -> 4.3; softmax(N(0, 1)) less one-hot, 4096 9.7
// -> 5.0; the gradients of an output layer of 8192 classes 5.9..9.6 -> 3.3..5.3.
// Few large terms among thousands that vanish beside them are the exception:
// softmax(8 N(0, 1)) less one-hot, 512 2.9 -> 2.2, but 2048 2.3 -> 2.6 and 4096 2.7
// -> 3.2 (a slab's leading products summed apart and added by VALU: 2.3 and 2.8,
// every product 7 to 10% slower).
constexpr int kBf3MinK = 128;
static bool bf3_takes(const GemmArgs& g, bool vec, bool plain, bool tA, bool tB) {
  if (!vec || (tA && tB) || g.f32 || g.K < kBf3MinK) return false;
  if (g.mode == kEpiAccum || (plain && g.mode == kEpiActGrad)) return true;
  const unsigned acts = !plain || tA || tB ? kActsNone : g.groups ? kActsMoe : kAllActs;
  return g.mode == kEpiAct && ((acts >> g.act) & 1);
}

// ---- which kernel, which tile, how many K chunks --------------------------------

// The split kernel's tiles, by use: 256x128 (8 waves, one workgroup on a CU),
// 128x128 (4 waves, two on a CU), and for grouped products 128x256; and the
// fp32 kernel's one, 128x128.
enum Tile : int { kT256x128 = 0, kT128, kBf3Tiles, kTF32 = kBf3Tiles };

// Estimated time (us) of M x N x K (x batch) on one tile shape with the K
// range cut into `splits`: whole rounds of the CUs, each tile with a prologue
// and epilogue worth ~64 steps of K.  Measured rates (N(0,1) operands): 256x128
// tiles 210 TFLOP/s, 128x128 190 with two workgroups on a CU and ~130 with
// one; the fp32 kernel two thirds of that.  The splits' partial sums are
// written and read once more at ~4 TB/s.
static double tile_time(int tile, int64_t M, int64_t N, int64_t K, int64_t batch, int64_t splits, int cus) {
  const int64_t bm = tile == kT256x128 ? 256 : 128, bn = 128;
  const int64_t tiles = ceil_div(M, bm) * ceil_div(N, bn) * batch * splits;
  const int64_t n = ceil_div(tiles, cus);  // tiles of the busiest CU
  const double bf3 = tile == kT256x128 ? 210. : n >= 2 ? 190. : 130.;
  const double rate = (tile == kTF32 ? bf3 * 2 / 3 : bf3) * 1e6 / cus;  // FLOP per us and CU
  const double t = (double)n * 2. * bm * bn * ((double)ceil_div(K, splits) + 64.) / rate;
  return splits > 1 ? t + 6. + (double)M * N * batch * splits * 8. / 4e6 : t;
}

struct TilePick {
  int tile;
  int64_t splits;
  double us;
};
// The least estimated time of g's shape over the split kernel's tiles (bf3) or
// the fp32 kernel's, and lo .. hi K chunks.
static TilePick pick_tile(const GemmArgs& g, bool bf3, int64_t batch, int64_t lo, int64_t hi, int cus) {
  TilePick best{kT128, lo, 1e30};
  for (int tile = bf3 ? 0 : kTF32; tile < (bf3 ? kBf3Tiles : kTF32 + 1); tile++)
    for (int64_t sp = lo; sp <= std::max(lo, hi); sp++) {
      const double t = tile_time(tile, g.M, g.N, g.K, batch, sp, cus);
      if (t < best.us) best = {tile, sp, t};
    }
  return best;
}

// K chunks that a product may be cut into: of at least 256, at most 32 of them.
static int64_t most_splits(const GemmArgs& g) { return std::max<int64_t>(1, std::min<int64_t>(32, g.K / 256)); }

// Estimated time (us) of gemm_small_kernel: whole rounds of the CUs, each a
// launch's latency and the wave's share of K (measured: one round of 64 x 32
// tiles 9 us at K = 512, 15 at 1024, 47 at 4096; of 32 x 32 tiles 30 at 4096).
static double small_time(const GemmArgs& g, int batch, int cus) {
  const int tm = g.M > 32 ? 2 : 1;
  const int64_t wgs = ceil_div(g.M, 32 * tm) * ceil_div(g.N, 32) * batch;
  return 1. + (double)ceil_div(wgs, cus) * (3. + (tm == 2 ? 0.0105 : 0.0065) * g.K);
}

// Whether a product runs on gemm_small_kernel: where its estimate is below
// four fifths of the tiled kernels' best with K split as it may be (their
// estimate is that much too high where one workgroup sits on a CU).  E.g.
// 33 x 4096 x 1024: 27 us against 40 with the call; 33 x 4096 x 4096: 57
// against 52, not taken; 1024 x 512 x 512: 24 against 37; 1024 x 2048 x 512: 52
// against 43, not taken.
static bool small_takes(const GemmArgs& g, int batch, int cus) {
  if (g.groups || g.kseg || g.kitems || g.kchunk || g.a_rows || g.c_rows || g.row_scale || g.mask_out || g.K <= 0)
    return false;
  return small_time(g, batch, cus) < 0.8 * pick_tile(g, true, batch, 1, g.C2 ? 1 : most_splits(g), cus).us;
}

int launch_gemm_ex(const GemmArgs& in, bool tA, bool tB, int batch, hipStream_t s) {
  if (in.M <= 0 || in.N <= 0 || batch <= 0) return 0;
  GemmArgs g = in;
  if (g.kitems && (g.kseg || g.groups || g.kchunk || g.a_rows || g.c_rows || !g.nkitems)) {
    set_error("gemm: K-chunked groups exclude the other grouping modes and row maps");
    return -1;
  }
  if (g.kblk && (g.kblk % BK != 0 || g.kseg || g.kitems || g.groups)) {
    set_error("gemm: K blocks must be a multiple of 16 and exclude K-grouped and grouped modes");
    return -1;
  }
  const bool vec = reads_float4(g, tA, tB);
  if (g.kblk && !vec) {
    set_error("gemm: K-blocked operands need 16-byte aligned, 4-float strided operands");
    return -1;
  }
  // plain epilogue: no row maps or scaling; activation, activation gradient,
  // accumulate or the pre-activation / activation pair (kchunk partials are
  // always kEpiAct)
  const bool plain = !g.c_rows && !g.row_scale &&
                     (g.mode == kEpiAct || g.mode == kEpiAccum || plain_act_grad(g));
  if (g.C2 && !(plain && g.mode == kEpiAct)) {
    set_error("gemm: the pre-activation / activation pair needs the plain activation epilogue");
    return -1;
  }
  if ((g.mask_out && !(g.C2 && g.act == kActRelu && batch == 1)) || (g.mask_in && !plain_act_grad(g)) ||
      ((g.mask_out || g.mask_in) && g.ldmask < g.N)) {
    set_error("gemm: sign bits need a relu pre-activation / activation pair or a relu gradient, ldmask >= N");
    return -1;
  }
  const int zs = g.kchunk ? (int)ceil_div(g.K, g.kchunk) : 1;
  const int cus = device_cus();
  if (small_reads(g, tA, tB) && small_takes(g, batch, cus)) {
    const int tm = g.M > 32 ? 2 : 1;
    g.tiles_m = (int)ceil_div(g.M, 32 * tm);
    g.tiles_n = (int)ceil_div(g.N, 32);
    const dim3 sgrid(g.tiles_m * g.tiles_n, batch), sblock(64 * kSmallW);
    const bool pieces = !g.f32 && g.K >= kBf3MinK;
#define NSH_SMALL(TA_, TB_)                                                                              \
  do {                                                                                                   \
    if (pieces && tm == 2) hipLaunchKernelGGL((gemm_small_kernel<TA_, TB_, true, 2>), sgrid, sblock, 0, s, g);  \
    else if (pieces) hipLaunchKernelGGL((gemm_small_kernel<TA_, TB_, true, 1>), sgrid, sblock, 0, s, g);        \
    else if (tm == 2) hipLaunchKernelGGL((gemm_small_kernel<TA_, TB_, false, 2>), sgrid, sblock, 0, s, g);      \
    else hipLaunchKernelGGL((gemm_small_kernel<TA_, TB_, false, 1>), sgrid, sblock, 0, s, g);                   \
  } while (0)
    if (!tA && !tB) NSH_SMALL(false, false);
    else if (!tA) NSH_SMALL(false, true);
    else NSH_SMALL(true, false);
#undef NSH_SMALL
    NSH_LAUNCHED();
    return 0;
  }
  const bool bf3 = bf3_takes(g, vec, plain, tA, tB);
  int bm = BM, bn = BN, tile = kT128;
  if (bf3 && g.groups) {
    bn = 256;  // 128-row tiles (the caller's tile list), 256 columns
  } else if (bf3 && plain && !g.kitems && !g.kseg) {
    tile = pick_tile(g, true, batch, zs, zs, cus).tile;
    bm = tile == kT128 ? 128 : 256;
  }
  g.tiles_m = (int)ceil_div(g.M, bm);
  g.tiles_n = (int)ceil_div(g.N, bn);
  // grouped: an upper bound on tile entries, sum_e ceil(n_e / BM) <= M/BM + E
  const int entries = g.groups ? g.tiles_m + g.groups : g.tiles_m;
  const dim3 grid(entries * g.tiles_n, batch, zs);
#define NSH_F32(TA_, TB_, V_)                                                                     \
  do {                                                                                            \
    if (plain) hipLaunchKernelGGL((gemm_f32_kernel<TA_, TB_, V_, true>), grid, dim3(NT), 0, s, g);  \
    else hipLaunchKernelGGL((gemm_f32_kernel<TA_, TB_, V_, false>), grid, dim3(NT), 0, s, g);       \
  } while (0)
#define NSH_BF3(TA_, TB_, ACTS_)                                                                              \
  do {                                                                                                        \
    if (!plain)                                                                                               \
      hipLaunchKernelGGL((gemm_bf3_kernel<TA_, TB_, false, kActsNone, 2, 2>), grid, dim3(256), 0, s, g);        \
    else if (tile == kT256x128)                                                                               \
      hipLaunchKernelGGL((gemm_bf3_kernel<TA_, TB_, true, ACTS_, 4, 2>), grid, dim3(512), 0, s, g);             \
    else hipLaunchKernelGGL((gemm_bf3_kernel<TA_, TB_, true, ACTS_, 2, 2>), grid, dim3(256), 0, s, g);          \
  } while (0)
  if (bf3 && g.groups) {
    if (!tB && plain) hipLaunchKernelGGL((gemm_bf3_kernel<false, false, true, kActsMoe, 2, 4>), grid, dim3(512), 0, s, g);
    else if (!tB) hipLaunchKernelGGL((gemm_bf3_kernel<false, false, false, kActsNone, 2, 4>), grid, dim3(512), 0, s, g);
    else if (plain) hipLaunchKernelGGL((gemm_bf3_kernel<false, true, true, kActsNone, 2, 4>), grid, dim3(512), 0, s, g);
    else hipLaunchKernelGGL((gemm_bf3_kernel<false, true, false, kActsNone, 2, 4>), grid, dim3(512), 0, s, g);
  } else if (bf3) {
    if (!tA && !tB) NSH_BF3(false, false, kAllActs);
    else if (!tA) NSH_BF3(false, true, kActsNone);
    else NSH_BF3(true, false, kActsNone);
  } else if (!tA && !tB) { if (vec) NSH_F32(false, false, true); else NSH_F32(false, false, false); }
  else if (!tA && tB) { if (vec) NSH_F32(false, true, true); else NSH_F32(false, true, false); }
  else if (tA && !tB) { if (vec) NSH_F32(true, false, true); else NSH_F32(true, false, false); }
  else { if (vec) NSH_F32(true, true, true); else NSH_F32(true, true, false); }
#undef NSH_F32
#undef NSH_BF3
  NSH_LAUNCHED();
  return 0;
}

// Sum of the K-chunk partials in chunk order, then the GEMM's epilogue.
// ws holds [splits][batch][M][N]; thread per output element.
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ ws, int splits, int64_t zstride,
                                                            GemmArgs g) {
  const int64_t n_out = (int64_t)g.M * g.N;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n_out) return;
  const int y = blockIdx.y;
  const int64_t off = (int64_t)y * n_out + i;
  float a = 0.f;
  for (int z = 0; z < splits; z++) a += ws[(int64_t)z * zstride + off];
  const int row = (int)(i / g.N), col = (int)(i % g.N);
  float* dst = g.C + (int64_t)y * g.sC + (int64_t)row * g.ldc + col;
  if (g.mode == kEpiAct) *dst = act_apply(a, g.act);
  else if (g.mode == kEpiActGrad) *dst = a * act_deriv(g.aux[(int64_t)row * g.ldaux + col], g.act);
  else *dst = *dst + a;
}

static bool splittable(const GemmArgs& g) {
  return !g.groups && !g.kseg && !g.kitems && !g.a_rows && !g.c_rows && !g.row_scale && !g.C2 && g.kchunk == 0;
}

// Chunk length for `splits` chunks: a multiple of BK (and so of 4, keeping
// float4 staging aligned).
static int split_chunk(int K, int splits) { return (int)(ceil_div(ceil_div(K, splits), BK) * BK); }

// Chunks of at most `sp` that cover K.
static int chunks_of(const GemmArgs& g, int64_t sp) {
  return sp < 2 ? 1 : (int)ceil_div(g.K, split_chunk(g.K, (int)sp));
}

// The product of one K chunk: plain, into the workspace.
static GemmArgs chunk_args(const GemmArgs& in) {
  GemmArgs p = in;
  p.mode = kEpiAct;
  p.act = 0;
  p.aux = nullptr;
  p.mask_in = nullptr;  // the reduction applies relu' from aux
  return p;
}

// The estimate prices the partial sums against the CUs that a few tiles leave
// idle, on the kernel that will run the chunks: a count of 1 where
// gemm_small_kernel takes the product, which needs its operands' alignment (33
// x 64 x 1201, which it cannot read, on the fp32 kernel: 1 chunk 145 us, 4 54).
// Over 27 shapes that only the fp32 kernel reads (K 512 to 8192, 1 to 289 tiles)
// the count's time is within 6% of the best of all counts with chunks of 256.
int gemm_split_count(const GemmArgs& g, bool tA, bool tB, int batch) {
  if (!splittable(g) || g.M <= 0 || g.N <= 0 || batch <= 0) return 1;
  const int cus = device_cus();
  if (small_reads(g, tA, tB) && small_takes(g, batch, cus)) return 1;
  const bool bf3 = bf3_takes(chunk_args(g), reads_float4(g, tA, tB), true, tA, tB);
  return chunks_of(g, pick_tile(g, bf3, batch, 1, most_splits(g), cus).splits);
}

int gemm_split_most(const GemmArgs& g, int batch) {
  if (!splittable(g) || g.M <= 0 || g.N <= 0 || batch <= 0) return 1;
  const int cus = device_cus();
  int n = 1;
  for (const bool bf3 : {false, true})
    n = std::max(n, chunks_of(g, pick_tile(g, bf3, batch, 1, most_splits(g), cus).splits));
  return n;
}

size_t gemm_split_workspace(const GemmArgs& g, int batch, int splits) {
  return splits <= 1 ? 0 : (size_t)splits * batch * g.M * g.N;
}

int launch_gemm_split(const GemmArgs& in, bool tA, bool tB, int batch, int splits, float* ws, hipStream_t s) {
  if (splits <= 1 || !ws || !splittable(in) || in.K < 2 * BK) return launch_gemm_ex(in, tA, tB, batch, s);
  if (in.M <= 0 || in.N <= 0 || batch <= 0) return 0;
  const int chunk = split_chunk(in.K, splits);
  const int zs = (int)ceil_div(in.K, chunk);
  const int64_t n_out = (int64_t)in.M * in.N;
  GemmArgs p = chunk_args(in);
  p.C = ws;
  p.ldc = in.N;
  p.sC = n_out;
  p.kchunk = chunk;
  p.sCk = n_out * batch;
  if (launch_gemm_ex(p, tA, tB, batch, s) != 0) return -1;
  const dim3 grid((unsigned)ceil_div(n_out, 256), batch);
  hipLaunchKernelGGL(splitk_reduce_kernel, grid, dim3(256), 0, s, ws, zs, n_out * batch, in);
  NSH_LAUNCHED();
  return 0;
}

int launch_gemm(const float* A, const float* B, float* C, int64_t M, int64_t N, int64_t K,
                int64_t lda, int64_t ldb, int64_t ldc, bool tA, bool tB, int act, hipStream_t s) {
  if (M > INT32_MAX || N > INT32_MAX || K > INT32_MAX) {
    set_error("gemm: dimension exceeds int32");
    return -1;
  }
  GemmArgs g;
  g.A = A; g.B = B; g.C = C;
  g.M = (int)M; g.N = (int)N; g.K = (int)K;
  g.lda = lda; g.ldb = ldb; g.ldc = ldc;
  g.act = act;
  return launch_gemm_ex(g, tA, tB, 1, s);
}

}  // namespace nship
