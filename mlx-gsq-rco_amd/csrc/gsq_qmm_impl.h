// Tiled quantized matrix-matrix product (QMM) for prefill: y[M,N] = x[M,K] * W[N,K]^T.
//
// Counterpart of the reference's tiled decode-once kernel
// (mlx_gsq/runtime/kernels/qmm.py:252-325, dispatched by quantized_matmul qmm.py:559-594):
// every weight is decoded once per activation tile into fp16 (the reference's decoded tile is
// half, qmm.py:181), activations are staged as fp16 (qmm.py:150-165) and products accumulate
// in fp32.
//
// gfx950 kernel (fp16 activations), one workgroup of 8 waves (4 on 64-row tiles) per CU:
//  * output tile = BM activation rows x 256 weight rows; wave w owns 32 (64) weight rows of the
//    tile and all BM rows, so its weights are private to it: the wave decodes them
//    straight into v_mfma_f32_16x16x32_f16 first operands (lane l: row l%16 of a 16-row block,
//    weights 8(l/16)..+7 of the 32-weight group) and they never pass through LDS as fp16.
//  * the wave's superblocks of the current 256-wide K column sit in a private
//    two-column LDS ring, filled by global_load_lds DMA one column ahead; each row has a
//    16-byte aligned slot holding the granules that cover its (2-byte aligned) superblock.
//  * activations: a ring of `lx` K32 stages of BM x 32 fp16 shared by the waves, filled
//    by DMA lx-1 stages ahead into a layout whose 16-byte octets are XOR-swizzled per row
//    (octet o of row m at position o ^ ((m >> 2) & 3)) so that the ds_read_b128 A-operand
//    reads of a wave are free of bank conflicts.
//  * all DMA waits are exact s_waitcnt vmcnt counts derived from the fixed issue order; one
//    s_barrier per K32 stage (per pair of stages on rings of four or more stages) guards the
//    shared activation ring.
//  * work split: as many workgroups as there are CUs; each takes whole tiles while there are
//    enough for all, and the (tile, K column) units of the tiles left over are divided evenly
//    (stream-K), so shapes whose tile count is not a multiple of the CU count (17408 = 17 * 1024
//    rows) still fill the chip. Tiles split between workgroups go to a workspace as fp32 partials,
//    which a second launch sums in a fixed order (deterministic).
//  * tiles are numbered weight tile fastest and workgroups renumbered so that work done at the
//    same time (one activation tile, neighbouring weight tiles and K ranges) lands on one XCD and
//    shares its L2.
// Other activations (fp32, bf16, not 16-byte aligned) are laid out as fp16 in the workspace before
// this kernel; the generic kernel below serves calls without that area.
#pragma once
#include <cstdlib>
#include <type_traits>
#include <utility>

#include "gsq_decode.h"
#include "gsq_qmm_decode.h"

namespace gsq {

enum { QDT_F32 = 0, QDT_F16 = 1, QDT_BF16 = 2 };

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

// Final outputs are not read again by the kernel, so fp32 ones are written as streaming
// (nontemporal) stores; the split-K partials, which the reduction reads back, keep plain stores.
__device__ __forceinline__ void qmm_store_y(void* y, int dt, int64_t i, float v) {
  if (dt == QDT_F16) reinterpret_cast<_Float16*>(y)[i] = (_Float16)v;
  else if (dt == QDT_BF16) reinterpret_cast<uint16_t*>(y)[i] = (uint16_t)f32_to_bf16_bits(v);
  else __builtin_nontemporal_store(v, reinterpret_cast<float*>(y) + i);
}

// ---- MFMA kernel ----------------------------------------------------------------------
constexpr int kQBN = 256;                   // weight rows per tile
constexpr int kQLds = 160 * 1024;

// WV waves per workgroup (4: one per SIMD, or 8: two per SIMD), each owning kQBN / WV weight
// rows of the tile.
template <int T, int WV>
struct QmmGeo {
  static constexpr int kBB = BlockBytes<T>::v;
  static constexpr int kRows = kQBN / WV;  // weight rows per wave
  static constexpr int kNB = kRows / 16;   // 16-row B blocks per wave
  // granules per row slot: enough for a superblock at any 2-byte offset (up to 14) within its
  // first granule, rounded up to an odd count so that the sixteen rows a wave reads at once
  // fall into distinct LDS bank groups (except Q6_K with 8 waves, whose rings would otherwise
  // leave no room for two activation stages of 256 rows)
  static constexpr int kNeed = (kBB + 14 + 15) / 16;
  static constexpr int kGran = (T == Q6_K && WV == 8) ? kNeed : (kNeed | 1);
  static constexpr int kSlot = kGran * 16;
  static constexpr int kGW = (kRows * kGran + 63) / 64;  // DMA instructions per column per wave
  static constexpr int kCol = kGW * 1024;                // one column of the wave's ring
  static constexpr int kRing = 2 * kCol;                 // per wave: two columns
};

// Byte size of a type's LDS table image (fp16 codebook followed by the 16 nibble sign masks,
// and for IQ2_XXS / IQ2_XS the 128 ksigns masks of four words that their decoders read; for
// IQ1_S / IQ1_M the codebook with each delta added; built by build_qmm_table in gsq_qmv.hip);
// checked against the host-built image at launch.
template <int T>
constexpr int qmm_tbl_bytes() {
  return T == IQ1_S || T == IQ1_M ? 2 * 2048 * 8 * 2
       : T == IQ2_XXS            ? 256 * 8 * 2 + 16 * 8 + 128 * 16
       : T == IQ2_XS             ? 512 * 8 * 2 + 16 * 8 + 128 * 16
       : T == IQ2_S              ? 1024 * 8 * 2 + 16 * 8
       : T == IQ3_XXS            ? 256 * 4 * 2 + 16 * 8
       : T == IQ3_S              ? 512 * 4 * 2 + 16 * 8
                                 : 0;
}

// LDS plan of (type, activation tile height MF x 16 rows, waves): table image, activation ring
// of kLx K32 stages (as deep as the LDS left over allows, up to 8) and the waves' weight rings.
template <int T, int MF, int WV>
struct QmmPlan {
  static constexpr int kTbl = qmm_tbl_bytes<T>();
  static constexpr int kW = WV * QmmGeo<T, WV>::kRing;
  static constexpr int kLx0 = (kQLds - kTbl - kW) / (16 * MF * 64);
  // a third stage alone is no gain over two (no barrier saved; IQ1_S at 2048 rows 431 against 414 us)
  static constexpr int kLx = kLx0 > 8 ? 8 : (kLx0 == 3 ? 2 : kLx0);
  static constexpr int kXOff = kTbl;
  static constexpr int kWOff = kXOff + kLx * 16 * MF * 64;
  static constexpr int kLds = kWOff + kW;
  static constexpr bool kValid = kLx >= 2 && MF >= WV;  // every wave issues activation DMA
};

// The DMA schedule of one wave (per K32 stage q of Q): the table copy, then column 0 and
// activation stages 0 .. P-1; each stage issues the next activation stage (NX instructions,
// while it exists) and, at a column start, the next column (GW instructions). With one barrier
// per stage (BP false), P = LX - 1 and stage q issues activation stage q + LX - 1; it needs the
// column of stage q + 1 and activation stage q. With one barrier per pair of stages (BP: rings of four
// or more stages), P = LX - 2 and the pair (q, q + 1), q even, issues activation stages
// q + LX - 2 and q + LX - 1 after its barrier, into the slots of stages q - 2 and q - 1, which
// every wave has finished; it needs activation stages q and q + 1 and the columns of stages
// q + 1 and q + 2. qmm_wait_n is the number of this wave's instructions that may still be in
// flight at a wait (vmcnt is in order).
constexpr int qmm_pro_x(int Q, int LX, bool BP) {
  const int p = BP ? LX - 2 : LX - 1;
  return p < Q ? p : Q;
}
constexpr int qmm_issued_before(int q, int Q, int LX, int NX, int GW, bool BP) {
  const int P = qmm_pro_x(Q, LX, BP);
  int x = 0;
  if (BP) x = (q + LX - 2 < Q ? q + LX - 2 : Q) - P;
  else x = q < Q - LX + 1 ? q : Q - LX + 1;
  const int cols = (q + 7) / 8 < Q / 8 - 1 ? (q + 7) / 8 : Q / 8 - 1;
  return GW + NX * P + NX * (x > 0 ? x : 0) + GW * cols;
}
constexpr int qmm_end_x(int k, int Q, int LX, int NX, int GW, bool BP) {
  const int P = qmm_pro_x(Q, LX, BP);
  if (k < P) return GW + NX * (k + 1);
  if (!BP) return qmm_issued_before(k - LX + 1, Q, LX, NX, GW, false) + NX;
  const int qp = 2 * ((k - LX + 2) >> 1);  // the pair that issues stage k
  return qmm_issued_before(qp, Q, LX, NX, GW, true) + NX * (k - (qp + LX - 2) + 1);
}
constexpr int qmm_end_w(int c, int Q, int LX, int NX, int GW, bool BP) {
  if (c == 0) return GW;
  const int qp = 8 * (c - 1);  // the stage (pair) that issues column c, after its activations
  const int nx = BP ? (qp + LX - 2 < Q ? 1 : 0) + (qp + LX - 1 < Q ? 1 : 0) : (qp + LX - 1 < Q ? 1 : 0);
  return qmm_issued_before(qp, Q, LX, NX, GW, BP) + NX * nx + GW;
}
constexpr int qmm_wait_n(int q, int Q, int LX, int NX, int GW, bool BP) {
  int need = 0, wc = -1;
  if (BP) {
    need = qmm_end_x(q + 1, Q, LX, NX, GW, true);
    wc = (q + 2 < Q ? q + 2 : q + 1) >> 3;
  } else {
    need = qmm_end_x(q, Q, LX, NX, GW, false);
    wc = q + 1 < Q ? (q + 1) >> 3 : -1;
  }
  if (wc >= 0) {
    const int ew = qmm_end_w(wc, Q, LX, NX, GW, BP);
    need = need > ew ? need : ew;
  }
  return qmm_issued_before(q, Q, LX, NX, GW, BP) - need;
}
// Every count the schedule produces (column counts 1..40 cover the start, steady state and
// end of any range), distinct, in descending order.
struct QmmWaitSet {
  int v[64];
  int n;
};
template <int LX, int NX, int GW, bool BP>
constexpr QmmWaitSet qmm_wait_set() {
  QmmWaitSet w{};
  w.n = 0;
  for (int cols = 1; cols <= 40; ++cols)
    for (int q = 0; q < 8 * cols; q += BP ? 2 : 1) {
      int c = qmm_wait_n(q, 8 * cols, LX, NX, GW, BP);
      if (c > 63) c = 63;
      bool seen = false;
      for (int i = 0; i < w.n; ++i) seen = seen || w.v[i] == c;
      if (!seen && w.n < 64) w.v[w.n++] = c;
    }
  for (int i = 0; i < w.n; ++i)
    for (int j = i + 1; j < w.n; ++j)
      if (w.v[j] > w.v[i]) {
        const int t = w.v[i];
        w.v[i] = w.v[j];
        w.v[j] = t;
      }
  return w;
}
template <int N>
__device__ __forceinline__ void wait_vm_imm() {
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}
// s_waitcnt vmcnt(c) for the largest schedule count c <= n: a short chain of compile-time
// immediates, largest (steady-state) counts first
template <int LX, int NX, int GW, bool BP, int K = 0>
__device__ __forceinline__ void qmm_wait(int n) {
  constexpr QmmWaitSet W = qmm_wait_set<LX, NX, GW, BP>();
  if constexpr (K >= W.n) {
    wait_vm_imm<0>();
  } else {
    constexpr int c = W.v[K];
    if (n >= c) wait_vm_imm<c>();
    else qmm_wait<LX, NX, GW, BP, K + 1>(n);
  }
}

struct QmmMfmaArgs {
  const uint8_t* packed;
  const _Float16* x;
  void* y;
  int M, N, K;
  int y_dtype;
  int nblk;              // superblocks per row (K / 256)
  long long row_bytes;
  int mt;                // activation tiles
  int nt;                // weight tiles (kQBN rows)
  int nfast;             // tile t = (activation tile t / nt, weight tile t % nt), else (t % mt, t / mt)
  int G;                 // workgroups
  int rounds;            // whole tiles of every workgroup: tile r * G + w in round r
  int units;             // (tile, K column) units of the tiles after those,
  int GS;                // split evenly over the first GS workgroups
  int xcd_remap;         // G is a multiple of 8
  const uint8_t* tbl;    // the type's table image (codebook + sign masks), or null
  int tbl_bytes;         // multiple of 16
  float* part;           // 2 * G partial slots of slot_floats
  int slot_floats;       // floats per partial slot: MC * NB * 64 * WV * 4 (a tile)
};

// A partial tile goes to the workspace as whole 16-byte stores in accumulator order (block (i, j)
// of the thread at ((i NB + j) 64 WV + thread) * 16 bytes of the slot) and is read back the same
// way by the reduction kernel, so both sides move whole cache lines. Slot 2w: the tile workgroup w
// starts in; slot 2w + 1: the tile it ends in.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t qmm_slot_rsrc(float* part, int slot, int slot_floats) {
  return __builtin_amdgcn_make_buffer_rsrc(part + (size_t)slot * (size_t)slot_floats, 0, slot_floats * 4, 0x00020000);
}
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

// The weight row (0 .. 16 NB - 1 of a wave's rows) decoded as operand row r of its block j: a
// lane's accumulators of the NB blocks then hold 4 NB consecutive outputs of one activation row.
template <int NB>
__device__ __forceinline__ int qmm_row(int j, int r) {
  return 4 * NB * (r >> 2) + 4 * j + (r & 3);
}

// Ranges are [floor(w * units / G), floor((w + 1) * units / G)). The plain 64-bit form: w * q + w * r / G
// in 32 bits, with an estimated owner corrected by two loops, was 1-4% slower in the small-batch kernel
// at up to 16 rows (7959 x 2048 9.06 against 8.65 us, 1024 x 5120 7.82 against 7.63, IQ2_S / IQ2_XS from
// a graph) and within 1% in the tiled kernel.
__device__ __forceinline__ int qmm_first_col(int w, int units, int G) {
  return (int)((long long)w * units / G);
}
// workgroup whose range holds column u
__device__ __forceinline__ int qmm_owner(int u, int units, int G) {
  return (int)(((long long)(u + 1) * G + units - 1) / units) - 1;
}

// A loop over 0 .. N - 1 unrolled at compile time (each index a constant): code over the
// accumulator arrays whose unrolled size exceeds the loop unroller's limits (MF x NB = 64 float4
// with 4 waves) would otherwise index them at run time, which moves the whole array to scratch
// memory (a scratch load and store around every MFMA).
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// The outputs of one 16-row activation block held by a lane (row m + lane % 16; v[j][e]: column
// n0 + 4 NB (lane / 16) + 4 j + e): 4 NB consecutive ones, in 16-byte pieces. Rows of odd N leave
// the pieces unaligned, which gfx950 stores as well: value by value they cost 31% of a 1227 x 7959
// x 512 product.
template <int NB>
__device__ __forceinline__ void qmm_store_block(void* y, int ydt, int M, int N, const float4_t (&v)[NB], int m, int n0,
                                                int lane) {
  typedef float4_t float4u_t __attribute__((aligned(4)));
  typedef u32x4_t u32x4u_t __attribute__((aligned(2)));
  const int mm = m + (lane & 15), n = n0 + 4 * NB * (lane >> 4);
  if (mm >= M) return;
  const int64_t at = (int64_t)mm * N + n;
  if (n + 4 * NB <= N) {
    if (ydt == QDT_F32) {
#pragma unroll
      for (int j = 0; j < NB; ++j)
        __builtin_nontemporal_store(v[j], reinterpret_cast<float4u_t*>(static_cast<float*>(y) + at + 4 * j));
    } else {
      u32x4_t o[NB / 2];
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          uint32_t lo, hi;
          if (ydt == QDT_F16) {
            lo = __builtin_bit_cast(uint16_t, (_Float16)v[j][e]);
            hi = __builtin_bit_cast(uint16_t, (_Float16)v[j][e + 1]);
          } else {
            lo = f32_to_bf16_bits(v[j][e]) & 0xFFFFu;
            hi = f32_to_bf16_bits(v[j][e + 1]) & 0xFFFFu;
          }
          o[j / 2][2 * (j & 1) + e / 2] = lo | (hi << 16);
        }
#pragma unroll
      for (int j = 0; j < NB / 2; ++j) *reinterpret_cast<u32x4u_t*>(static_cast<uint16_t*>(y) + at + 8 * j) = o[j];
    }
  } else {
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + 4 * j + e < N) qmm_store_y(y, ydt, at + 4 * j + e, v[j][e]);
  }
}

// Issues the activation stages of one workgroup in order: stage q (ring slot b) of tile t,
// column c; row[i] = this lane's source row (clamped to the matrix) and octet for DMA
// instruction i, laid out for the XOR-swizzled ring (octet o of row m at o ^ ((m >> 2) & 3)).
template <int NX, int BM, int TM, int LX>
struct QmmXIter {
  const _Float16* x;
  int M, K, mt, nt, nfast, nblk, G, c0, left, n, ts, cs;  // left: whole tiles to go, n: columns to go in this one
  int q, t, c, b;
  const _Float16* row[NX];
  __device__ __forceinline__ void rows(int wave, int lane) {
    const int m0 = (nfast ? t / nt : t % mt) * TM;
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int s = (wave * NX + i) * 64 + lane;
      const int m = s >> 2;
      const int o = (s & 3) ^ ((m >> 2) & 3);
      row[i] = x + (long long)min(m0 + min(m, TM - 1), M - 1) * K + 8 * o;
    }
  }
  // `rounds` whole tiles w, w + G, ..., each from column c0 on, then the units from us on
  __device__ __forceinline__ void init(const _Float16* x_, int M_, int K_, int mt_, int nt_, int nfast_, int nblk_, int G_,
                                       int rounds, int w, int c0_, int us, int wave, int lane) {
    x = x_;
    M = M_;
    K = K_;
    mt = mt_;
    nt = nt_;
    nfast = nfast_;
    nblk = nblk_;
    G = G_;
    left = rounds;
    n = nblk;
    c0 = c0_;
    ts = us / nblk;
    cs = us - ts * nblk;
    q = 0;
    b = 0;
    t = rounds ? w : ts;
    c = rounds ? c0 : cs;
    rows(wave, lane);
  }
  __device__ __forceinline__ void issue(uint8_t* xring, int wave, int lane) {
    const int kk = c * 256 + (q & 7) * 32;
    uint8_t* buf = xring + b * (BM * 64) + wave * NX * 1024;
#pragma unroll
    for (int i = 0; i < NX; ++i)
      __builtin_amdgcn_global_load_lds(static_cast<const void*>(row[i] + kk), (lds_ptr_t)(buf + i * 1024), 16, 0, 0);
    ++q;
    if (++b == LX) b = 0;
    if ((q & 7) == 0) {
      if (++c == nblk) {
        c = 0;
        if (left == 0) {
          ++t;
          rows(wave, lane);
        }
      }
      if (left > 0 && --n == 0) {
        --left;
        n = nblk;
        t = left ? t + G : ts;
        c = left ? c0 : cs;
        rows(wave, lane);
      }
    }
  }
};

// The type's table image in static LDS (LDS address 0).
template <int B>
struct QmmTblLds {
  __device__ __forceinline__ static uint8_t* get() {
    __shared__ __attribute__((aligned(16))) uint8_t t[B];
    return t;
  }
};
template <>
struct QmmTblLds<0> {
  __device__ __forceinline__ static uint8_t* get() { return nullptr; }
};

// Whether a wave's MFMAs are spread over the phases of its decode (see the stage below) or follow
// it. Spread against whole, mean of five shapes, 97 to 2048 rows: the IQ1, IQ2 and IQ3 types 2-11%
// faster (IQ2_S 17408 x 5120 at 2048 rows 433 against 446 us), Q2_K, Q4_K and IQ4_XS 1% slower to
// 2.5% faster, Q6_K 1.4% slower at 97 rows to 1.6% faster at 2048 (537 against 538 us there): Q6_K,
// whose decode holds the most registers, stays whole.
template <int T>
constexpr bool qmm_spread() { return T != Q6_K; }

template <int T, int MF, int MC, bool A4, int WV>
__global__ void __launch_bounds__(64 * WV, 1) qmm_mfma_kernel(QmmMfmaArgs args) {
  // the arguments as plain values (no reference to the argument block escapes, so it is never
  // copied to scratch memory, whose loads would wait on the DMA counter)
  const uint8_t* const packed = args.packed;
  const _Float16* const xg = args.x;
  void* const yg = args.y;
  const int M = args.M, N = args.N, K = args.K, ydt = args.y_dtype, nblk = args.nblk, mt = args.mt;
  const int nt = args.nt, nfast = args.nfast;
  auto tile_m = [&](int t) { return nfast ? t / nt : t % mt; };
  auto tile_n = [&](int t) { return nfast ? t % nt : t / mt; };
  const int G = args.G, xcd = args.xcd_remap, tbl_bytes = args.tbl_bytes;
  const long long row_bytes = args.row_bytes;
  const uint8_t* const tblg = args.tbl;
  float* const part = args.part;
  const int slot_floats = args.slot_floats;
  using Geo = QmmGeo<T, WV>;
  constexpr int BB = Geo::kBB, GW = Geo::kGW, GR = Geo::kGran, S = Geo::kSlot;
  constexpr int RW = Geo::kRows, NB = Geo::kNB, TH = 64 * WV;
  constexpr int BM = 16 * MF, NX = MF / WV;  // NX: activation DMA instructions per wave per stage
  constexpr int TM = 16 * MC;                // activation rows of a tile (the stage's rows past them repeat the last)
  using Plan = QmmPlan<T, MF, WV>;
  constexpr int LX = Plan::kLx;
  static_assert(Plan::kValid, "activation ring needs two stages");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform
  const int bid = blockIdx.x;
  const int w = xcd ? (bid & 7) * (G >> 3) + (bid >> 3) : bid;
  // local columns: those of `rounds` whole tiles, then a range of the split units
  const int rounds = args.rounds, wc = rounds * nblk, split0 = rounds * G * nblk;
  const int ub = split0 + (w < args.GS ? qmm_first_col(w, args.units, args.GS) : 0);
  const int ncols = wc + (w < args.GS ? split0 + qmm_first_col(w + 1, args.units, args.GS) - ub : 0);  // >= 1
  const int Q = 8 * ncols;    // K32 stages of this workgroup
  // whole tiles start at a column of the workgroup's own and wrap around: the 32 workgroups of an
  // XCD read one activation tile, so each loads a share of it early for the others; all starting
  // at column 0, every one waited for each column's first read from HBM (2048 rows of 17408 x 5120
  // IQ3_S with new activations every call 487 -> 459 us)
  const int c0 = (w & 31) * nblk >> 5;
  auto unit = [&](int cl) {   // (tile, column) unit of local column cl
    if (cl >= wc) return ub + cl - wc;
    const int r = cl / nblk, c = cl - r * nblk + c0;
    return (r * G + w) * nblk + (c < nblk ? c : c - nblk);
  };
  constexpr int lx = LX;
  // the table image is static LDS at address 0 (its reads fold the base into their address
  // arithmetic); the plan's other offsets count from the table's start, where dynamic LDS
  // begins after the table
  uint8_t* dyn = lds - Plan::kTbl;
  uint8_t* xring = dyn + Plan::kXOff;
  uint8_t* wring = dyn + Plan::kWOff + wave * Geo::kRing;
  uint8_t* tbl = QmmTblLds<Plan::kTbl>::get();

  // the type's table image first in this wave's DMA order: the first wait covers it
  if (tbl_bytes) dma_copy(tblg, tbl_bytes, tbl, wave, WV, lane);

  // activation stages are issued in order by an iterator
  QmmXIter<NX, BM, TM, LX> xi;
  xi.init(xg, M, K, mt, nt, nfast, nblk, G, rounds, w, c0, ub, wave, lane);
  // weight column cl (local index): the wave's RW superblocks, granule e of the column at
  // byte 16e (row e / GR, granule e % GR of that row); granules past a row's last one reload
  // its last granule, and lanes past the last row (whole instructions) reload the last row's,
  // so every lane stays active and the count stays fixed
  auto issue_w = [&](int cl) {
    const int u = unit(cl);
    const int tile = u / nblk, c = u - tile * nblk;
    const int n0 = tile_n(tile) * kQBN + wave * RW;
    uint8_t* buf = wring + (cl & 1) * Geo::kCol;
#pragma unroll
    for (int i = 0; i < GW; ++i) {
      const int e = i * 64 + lane;
      const int r = min(e / GR, RW - 1), qg = e - (e / GR) * GR;
      const int n = min(n0 + qmm_row<NB>(r >> 4, r & 15), N - 1);
      const uintptr_t p = reinterpret_cast<uintptr_t>(packed) + (uintptr_t)((long long)n * row_bytes) +
                          (uintptr_t)c * BB;
      const uintptr_t a0 = p & ~(uintptr_t)15;
      const int ng = (int)((p + BB + 15 - a0) >> 4);
      const uintptr_t src = a0 + (uintptr_t)(qg < ng ? qg : ng - 1) * 16;
      __builtin_amdgcn_global_load_lds(reinterpret_cast<const void*>(src), (lds_ptr_t)(buf + i * 1024), 16, 0, 0);
    }
  };

  // one barrier per pair of stages when the ring has four or more stages (the DMA schedule
  // above; the waves drift apart by up to a stage between barriers)
  constexpr bool BP = LX >= 4;
  const int P = qmm_pro_x(Q, lx, BP);

  // B operands of stage q: the 16-row blocks of the wave's weight rows, group q % 8 of column
  // q / 8; dl = the low address bits of the lane's superblocks in that column. work(c) (c = 0 ..
  // 3 NB - 1, compile-time) runs between the phases of the decode.
  auto decode = [&](int q, const uint32_t (&dl)[NB], half8_t (&bf)[NB], auto work) __attribute__((always_inline)) {
    const uint8_t* wb = wring + ((q >> 3) & 1) * Geo::kCol;
    static_for<NB>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      uint32_t o[4];
      QmmDec<T, A4>::run(wb + (16 * j + (lane & 15)) * S, dl[j], tbl, q & 7, lane >> 4, o,
                         [&] { work(std::integral_constant<int, 3 * j>{}); },
                         [&] { work(std::integral_constant<int, 3 * j + 1>{}); });
      bf[j] = __builtin_bit_cast(half8_t, o);
      work(std::integral_constant<int, 3 * j + 2>{});
    });
  };
  auto col_delta = [&](int q, uint32_t (&dl)[NB]) {
    const int u = unit(q >> 3);
    const int tl = u / nblk, c = u - tl * nblk;
    const int n0 = tile_n(tl) * kQBN + wave * RW;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int n = min(n0 + qmm_row<NB>(j, lane & 15), N - 1);
      dl[j] = (uint32_t)((reinterpret_cast<uintptr_t>(packed) + (uintptr_t)((long long)n * row_bytes) +
                          (uintptr_t)c * BB) & 15u);
    }
  };
  // A operands of a stage: MF 16-row blocks (row l % 16, octet l / 16, swizzled)
  const int xoff = (lane & 15) * 64 + (((lane >> 4) ^ ((lane >> 2) & 3)) << 4);
  auto load_a = [&](int slot, int i) {
    const uint32_t* p = reinterpret_cast<const uint32_t*>(xring + slot * (BM * 64) + xoff) + i * 256;
    const uint32_t aw[4] = {p[0], p[1], p[2], p[3]};
    return __builtin_bit_cast(half8_t, aw);
  };
  // prologue: table, column 0 and the first activation stages in flight; stage 0's weights
  issue_w(0);
  for (int q = 0; q < P; ++q) xi.issue(xring, wave, lane);
  qmm_wait<LX, NX, GW, BP>(NX * (P - 1));  // table, column 0 and stage 0 (this wave's share)
  __syncthreads();
  uint32_t dl[NB];
  col_delta(0, dl);
  half8_t bcur[NB];
  decode(0, dl, bcur, [](auto) {});
  half8_t bnext[NB];
  int rb = 0;  // ring slot of the next activations read

  // one segment = this workgroup's columns of one tile; stage q multiplies its activations
  // with weights decoded during stage q - 1 and decodes the weights of stage q + 1
  for (int q0 = 0; q0 < Q;) {
    const int u0 = unit(q0 >> 3);
    const int tile = u0 / nblk;
    const bool round = q0 < 8 * wc;
    const int q1 = q0 + 8 * (round ? nblk : min(ncols - (q0 >> 3), (tile + 1) * nblk - u0));
    const int m0 = tile_m(tile) * TM, n0 = tile_n(tile) * kQBN + wave * RW;
    float4_t acc[MC][NB];
#pragma unroll
    for (int i = 0; i < MC; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = (float4_t){0.f, 0.f, 0.f, 0.f};

    // stage q: its weights ub_ were decoded during stage q - 1; this stage decodes those of stage
    // q + 1 into nb (after the last stage from stale, in-bounds LDS: not used). The MFMAs are
    // spread over the decode: between its phases (LDS field reads, codebook reads, arithmetic) the
    // wave issues the MFMAs of a few 16-row activation blocks, whose operands were read AD blocks
    // ahead, so that no LDS latency is waited for without work to cover it.
    constexpr int AD = MC < 4 ? MC : 4, NW = 3 * NB;
    auto stage = [&](int q, const half8_t (&ub_)[NB], half8_t (&nb)[NB]) __attribute__((always_inline)) {
      const int cl = q >> 3;
      if (!BP || (q & 1) == 0) {
        // the activations read until the next wait and the columns decoded until then have
        // landed (this wave's DMAs)
        qmm_wait<LX, NX, GW, BP>(qmm_wait_n(q, Q, lx, NX, GW, BP));
        // every wave's DMAs of those stages are in; every wave is done with the slots of the
        // stages before them
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if constexpr (BP) {
          if (q + lx - 2 < Q) xi.issue(xring, wave, lane);
          if (q + lx - 1 < Q) xi.issue(xring, wave, lane);
        } else {
          if (q + lx - 1 < Q) xi.issue(xring, wave, lane);
        }
        if ((q & 7) == 0 && cl + 1 < ncols) issue_w(cl + 1);
      }
      if (((q + 1) & 7) == 0) col_delta(q + 1, dl);
      half8_t a[MC];
      auto mma = [&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ub_[j], a[i], acc[i][j], 0, 0, 0);
      };
      if constexpr (qmm_spread<T>()) {
        static_for<AD>([&](auto ic) { a[decltype(ic)::value] = load_a(rb, decltype(ic)::value); });
        decode(q + 1, dl, nb, [&](auto cc) __attribute__((always_inline)) {
          constexpr int c = decltype(cc)::value, i0 = c * MC / NW, i1 = (c + 1) * MC / NW;
          __builtin_amdgcn_sched_barrier(0);
          static_for<i1 - i0>([&](auto ic) {
            constexpr int i = i0 + decltype(ic)::value;
            mma(std::integral_constant<int, i>{});
            if constexpr (i + AD < MC) a[i + AD] = load_a(rb, i + AD);
          });
          __builtin_amdgcn_sched_barrier(0);
        });
      } else {
        decode(q + 1, dl, nb, [](auto) {});
        // LDS reads stay in this order: the decode's table reads are waited for without waiting
        // for the activation reads issued after them (LDS completes in order)
        __builtin_amdgcn_sched_barrier(0x1 | 0x2 | 0x4 | 0x8);
        // a wave issuing its MFMAs takes issue priority over the SIMD's other wave, which is
        // still decoding: the matrix pipe gets its next instruction as soon as it can take one
        // (2-4% faster at M = 512 and 2048)
        __builtin_amdgcn_s_setprio(1);
        static_for<MC>([&](auto ic) { a[decltype(ic)::value] = load_a(rb, decltype(ic)::value); });
        static_for<MC>(mma);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(0);
      }
      if (++rb == lx) rb = 0;
    };
    // a segment is whole columns: its stage count is a multiple of 8
    for (int q = q0; q < q1; q += 2) {
      stage(q, bcur, bnext);
      stage(q + 1, bnext, bcur);
    }

    // end of this workgroup's part of `tile`: the whole tile goes to y, a part of it to the
    // workspace, summed by the reduction kernel; 16-row blocks wholly past M go nowhere
    const bool whole = round || (u0 == tile * nblk && q1 - q0 == 8 * nblk);
    if (whole) {
      static_for<MC>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if (m0 + 16 * i < M) qmm_store_block<NB>(yg, ydt, M, N, acc[i], m0 + 16 * i, n0, lane);
      });
    } else {
      const __amdgpu_buffer_rsrc_t ps = qmm_slot_rsrc(part, 2 * w + (u0 == ub ? 0 : 1), slot_floats);
      static_for<MC>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if (m0 + 16 * i < M) {
#pragma unroll
          for (int j = 0; j < NB; ++j)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, acc[i][j]), ps, ((i * NB + j) * TH + tid) * 16, 0,
                                                   16 /* sc1: written through */);
        }
      });
    }
    q0 = q1;
  }
}

// Sums the partials of the split tiles in workgroup order (deterministic) and writes y: one
// workgroup per (boundary between two workgroups' ranges, 16-row activation block, half of the
// tile's waves), working only at the first boundary inside each split tile, with up to eight
// partials' loads in flight. Its own launch, so that every CU reads partials at
// once: summed inside the main kernel by a tile's last workgroup to arrive, one CU read all of a
// tile's partials (2 to 13 of 128-256 KB) with the others idle, 25-38 us at the end of a launch.
template <int T, int MC, int NB, int WV>  // T: one kernel symbol per translation unit
__global__ void __launch_bounds__(256) qmm_reduce_kernel(QmmMfmaArgs a) {
  constexpr int TH = 64 * WV, UN = 8;
  // four of the main kernel's waves per workgroup
  const int tid = blockIdx.z * 256 + threadIdx.x, lane = tid & 63, wave = tid >> 6, i = blockIdx.y;
  const int w = (int)blockIdx.x + 1, ub = qmm_first_col(w, a.units, a.GS), st = ub / a.nblk;  // st: split tile
  if (ub == st * a.nblk || qmm_first_col(w - 1, a.units, a.GS) > st * a.nblk) return;
  const int tile = a.rounds * a.G + st;
  const int m0 = (a.nfast ? tile / a.nt : tile % a.mt) * 16 * MC + 16 * i;
  if (m0 >= a.M) return;
  const int n0 = (a.nfast ? tile % a.nt : tile / a.mt) * kQBN + wave * (16 * NB);
  const int wf = w - 1, wl = qmm_owner(st * a.nblk + a.nblk - 1, a.units, a.GS);
  // only the first piece can follow another one in its workgroup's range
  const int s0 = 2 * wf + (qmm_first_col(wf, a.units, a.GS) / a.nblk == st ? 0 : 1);
  auto slot = [&](int v) {
    return a.part + (size_t)(v == wf ? s0 : 2 * v) * (size_t)a.slot_floats + ((size_t)(i * NB) * TH + tid) * 4;
  };
  float4_t sum[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) sum[j] = (float4_t){0.f, 0.f, 0.f, 0.f};
  for (int v = wf; v <= wl; v += UN) {
    float4_t ld[UN][NB];
#pragma unroll
    for (int u = 0; u < UN; ++u)
      if (v + u <= wl) {
        const float* p = slot(v + u);
#pragma unroll
        for (int j = 0; j < NB; ++j) ld[u][j] = *reinterpret_cast<const float4_t*>(p + (size_t)j * TH * 4);
      }
#pragma unroll
    for (int u = 0; u < UN; ++u)
      if (v + u <= wl) {
#pragma unroll
        for (int j = 0; j < NB; ++j) sum[j] += ld[u][j];
      }
  }
  qmm_store_block<NB>(a.y, a.y_dtype, a.M, a.N, sum, m0, n0, lane);
}

// ---- generic kernel (fp32 / bf16 activations) ------------------------------------------
// 64 x 64 output tile per 256 threads over K steps of 64: half of the threads decode 64 rows x
// two groups of weights (exact fp32 -> fp16), the other half stage the activations as fp16
// (qmm.py:160-165 converts fp32 activations to half the same way); each wave multiplies a
// 32 x 32 sub-tile with v_mfma_f32_16x16x32_f16.
constexpr int kGBM = 64, kGBN = 64, kGKS = 64, kGStride = kGKS + 8;

struct QmmArgs {
  const uint8_t* packed;
  const void* x;
  void* y;
  int64_t M, N;
  int K, x_dtype, y_dtype;
  DevTables tb;
};

__device__ __forceinline__ float qmm_load_x(const void* x, int dt, int64_t i) {
  if (dt == QDT_F16) return (float)reinterpret_cast<const _Float16*>(x)[i];
  if (dt == QDT_BF16) return __builtin_bit_cast(float, (uint32_t)reinterpret_cast<const uint16_t*>(x)[i] << 16);
  return reinterpret_cast<const float*>(x)[i];
}

template <int T>
__global__ void __launch_bounds__(256) qmm_generic_kernel(QmmArgs a) {
  constexpr int BB = BlockBytes<T>::v;
  __shared__ __attribute__((aligned(16))) _Float16 wt[kGBN * kGStride];
  __shared__ __attribute__((aligned(16))) _Float16 xt[kGBM * kGStride];
  const int tid = threadIdx.x;
  const int64_t n0 = (int64_t)blockIdx.x * kGBN;
  const int64_t m0 = (int64_t)blockIdx.y * kGBM;
  const int nb = a.K / 256;
  const int wave = tid >> 6, lane = tid & 63;
  const int wm = wave >> 1, wn = wave & 1;

  float4_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = (float4_t){0.f, 0.f, 0.f, 0.f};

  for (int k0 = 0; k0 < a.K; k0 += kGKS) {
    if (tid < 128) {
      const int r = tid >> 1, kg = tid & 1;
      const int64_t n = n0 + r;
      _Float16* dst = wt + r * kGStride + 32 * kg;
      if (n < a.N) {
        const int gidx = (k0 >> 5) + kg;
        const uint8_t* blk = a.packed + (n * nb + (gidx >> 3)) * BB;
        float v[32];
        dq_group<T>(blk, gidx & 7, a.tb, v);
#pragma unroll
        for (int i = 0; i < 32; ++i) dst[i] = (_Float16)v[i];
      } else {
#pragma unroll
        for (int i = 0; i < 32; ++i) dst[i] = (_Float16)0.f;
      }
    } else {
      const int t = tid - 128, r = t >> 1, half = t & 1;
      const int64_t m = m0 + r;
      _Float16* dst = xt + r * kGStride + 32 * half;
      if (m < a.M) {
        const int64_t base = m * a.K + k0 + 32 * half;
#pragma unroll
        for (int i = 0; i < 32; ++i) dst[i] = (_Float16)qmm_load_x(a.x, a.x_dtype, base + i);
      } else {
#pragma unroll
        for (int i = 0; i < 32; ++i) dst[i] = (_Float16)0.f;
      }
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < kGKS; kk += 32) {
      half8_t af[2], bf[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        af[i] = *reinterpret_cast<const half8_t*>(xt + (wm * 32 + i * 16 + (lane & 15)) * kGStride + kk + 8 * (lane >> 4));
#pragma unroll
      for (int j = 0; j < 2; ++j)
        bf[j] = *reinterpret_cast<const half8_t*>(wt + (wn * 32 + j * 16 + (lane & 15)) * kGStride + kk + 8 * (lane >> 4));
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i], bf[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  // C layout: lane holds rows 4*(lane/16)+e (e=0..3) of column lane%16 of each 16x16 tile
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t n = n0 + wn * 32 + j * 16 + (lane & 15);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t m = m0 + wm * 32 + i * 16 + 4 * (lane >> 4) + e;
        if (m < a.M && n < a.N) qmm_store_y(a.y, a.y_dtype, m * a.N + n, acc[i][j][e]);
      }
    }
}

}  // namespace gsq

#include "gsq_qmm_small.h"

namespace gsq {

// Tiles of 192 or 256 rows: a column of a tile costs about 4 + its 16-row blocks (the decode and the
// per-stage work count as four: IQ2_S 17408 x 5120 8.1 us against 10.2), so 192 where that covers M
// for less (182 rows: 98 -> 76 us with everything else of this plan; 800 rows: 242 us with 192, 228
// with 256).
static int qmm_tall_blocks(long long M) {
  return (M + 191) / 192 * (4 + 12) < (M + 255) / 256 * (4 + 16) ? 12 : 16;
}

// ---- host side --------------------------------------------------------------------------
extern QmmTuning g_qmm_tuning;

int qmm_table_bytes(int qt);  // the QMM kernels' LDS table image of a type (gsq_qmv.hip)
static bool qmm_grid_type(int qt) {
  return qt == IQ1_S || qt == IQ1_M || qt == IQ2_XXS || qt == IQ2_XS || qt == IQ2_S || qt == IQ3_XXS || qt == IQ3_S;
}

// Launch plans of the tiled kernel: ring height MF and tile height MC (16-row blocks) and waves.
// MF 16 holds tiles of 16 or 12 blocks (192 rows), so that 129-192 rows (and the like of larger
// batches) do not multiply padding.
template <int T, int MF, int MC, bool A4, int WV>
static hipError_t launch_mfma_k(const QmmMfmaArgs& a, hipStream_t s) {
  using Plan = QmmPlan<T, MF, WV>;
  static_assert(Plan::kValid);
  auto k = qmm_mfma_kernel<T, MF, MC, A4, WV>;
  static LdsLimit limit;
  if (hipError_t e = limit.raise((const void*)k, kQLds - Plan::kTbl); e != hipSuccess) return e;
  hipLaunchKernelGGL(k, dim3(a.G), dim3(64 * WV), Plan::kLds - Plan::kTbl, s, a);
  return hipGetLastError();
}

template <int T, int MF, int MC, int WV>
static hipError_t launch_mfma_t(const QmmMfmaArgs& a, bool a4, hipStream_t s) {
  constexpr int NB = QmmGeo<T, WV>::kNB;
  hipError_t e;
  if constexpr (BlockBytes<T>::v % 4 == 0) {
    e = a4 ? launch_mfma_k<T, MF, MC, true, WV>(a, s) : launch_mfma_k<T, MF, MC, false, WV>(a, s);
  } else {
    e = launch_mfma_k<T, MF, MC, false, WV>(a, s);
  }
  // unless every range starts at a tile's first column
  if (e == hipSuccess && a.GS > 1 && (a.units % a.GS != 0 || (a.units / a.GS) % a.nblk != 0)) {
    hipLaunchKernelGGL((qmm_reduce_kernel<T, MC, NB, WV>), dim3(a.GS - 1, MC, WV / 4), dim3(256), 0, s, a);
    e = hipGetLastError();
  }
  return e;
}

// Plan and launch the MFMA kernel for type T: tile height from M (64 rows up to 64, 128 up to 128,
// 192 or 256 beyond), then the stream-K grid: one workgroup per CU, at most one per two (tile, K
// column) units.
template <int T>
static hipError_t launch_mfma(QmmMfmaArgs& a, int num_cus, const QmmWorkspace& ws, hipStream_t s) {
  if (a.tbl_bytes != qmm_tbl_bytes<T>()) return hipErrorInvalidValue;
  int mc = g_qmm_tuning.mf;
  if (mc == 0) mc = a.M <= 64 ? 4 : (a.M <= 128 ? 8 : qmm_tall_blocks(a.M));
  if (mc != 4 && mc != 8 && mc != 12 && mc != 16) return hipErrorInvalidValue;
  const bool a4 = (reinterpret_cast<uintptr_t>(a.packed) & 3) == 0;
  // at least min_cols columns per workgroup: fewer workgroups share each tile when the
  // problem is small, which bounds the partial-tile traffic
  const int min_cols = g_qmm_tuning.min_cols > 0 ? g_qmm_tuning.min_cols : 2;
  for (;;) {
    const int bm = 16 * mc;
    a.mt = (a.M + bm - 1) / bm;
    a.nt = (int)((a.N + kQBN - 1) / kQBN);
    // weight tile fastest: the workgroups of one XCD (consecutive units) share an activation
    // tile in its L2 (3-6% faster at M = 2048 than activation tile fastest)
    a.nfast = g_qmm_tuning.order == 2 ? 0 : 1;
    const long long tiles = (long long)a.mt * a.nt;
    if (tiles * a.nblk >= (1ll << 31)) return hipErrorInvalidValue;
    const int cap = num_cus < ws.max_groups ? num_cus : ws.max_groups;
    const int gmax = (int)((tiles * a.nblk + min_cols - 1) / min_cols);
    a.G = cap < gmax ? cap : gmax;
    // whole tiles first: 2048 rows of 17408 x 5120 (544 tiles on 256 CUs) go through 287 partial
    // tiles instead of 480
    a.rounds = (int)(tiles / a.G);
    a.units = (int)(tiles - (long long)a.rounds * a.G) * a.nblk;
    const int smax = (a.units + min_cols - 1) / min_cols;
    a.GS = a.G < smax ? a.G : smax;
    // a workspace too small for this tile height's partials at this grid: lower tiles
    a.slot_floats = mc * 16 * kQBN;
    if (2ll * a.GS * a.slot_floats * 4 <= ws.part_bytes) break;
    if (mc == 4) return hipErrorInvalidValue;
    mc = mc > 8 ? 8 : 4;
  }
  a.xcd_remap = (a.G % 8 == 0) ? 1 : 0;
  a.part = ws.part;
  switch (mc) {
    case 4: return launch_mfma_t<T, 4, 4, 4>(a, a4, s);
    case 8: return launch_mfma_t<T, 8, 8, 8>(a, a4, s);
    case 12: return launch_mfma_t<T, 16, 12, 8>(a, a4, s);
    default: return launch_mfma_t<T, 16, 16, 8>(a, a4, s);
  }
}

// Lane layout of the small-batch kernel's decode: whole groups per lane (HX) for every type but
// Q6_K and Q2_K, whose fragment decoders share few field reads between a group's octets (at
// M = 4 and 16 on 17408 / 8192 / 4096-row products: the codebook types 1-17% faster, IQ4_XS
// 2-8%, Q4_K 1-7%, Q2_K -1 to +3%, Q6_K 8-16% slower). GSQ_QMS_HX=0 / 1 sets it for every type
// at up to 16 activation rows (read once, for measurements).
template <int T>
constexpr bool qms_group_layout() { return T != Q6_K && T != Q2_K; }

template <int T, int WV, int NB, int MB>
static hipError_t launch_qms_a4(const QmsArgs& a, bool a4, hipStream_t s) {
  constexpr bool HX = qms_group_layout<T>();
  if constexpr (MB == 1) {
    static const int env_hx = [] {
      const char* v = std::getenv("GSQ_QMS_HX");
      return v ? std::atoi(v) : -1;
    }();
    if (env_hx >= 0 && (env_hx > 0) != HX) {
      if constexpr (BlockBytes<T>::v % 4 == 0)
        if (a4) return launch_qms_t<T, true, WV, NB, !HX, MB>(a, s);
      return launch_qms_t<T, false, WV, NB, !HX, MB>(a, s);
    }
  }
  if constexpr (BlockBytes<T>::v % 4 == 0)
    if (a4) return launch_qms_t<T, true, WV, NB, HX, MB>(a, s);
  return launch_qms_t<T, false, WV, NB, HX, MB>(a, s);
}

// Activation blocks of 16 rows the small-batch kernel takes M rows in, or 0: M > 96 (two launches of
// 64 rows take as long as one 128-row tile of the tiled kernel: 66 against 58 us on 17408 x 5120
// Q4_K), or a type whose ring of two columns does not fit beside that many (Q6_K past 64 rows and the
// IQ1 types past 48, whose superblocks or tables are the largest). Wherever it has a plan it is the
// faster one: 1024-17408 rows or columns, 17-64 rows 1.7-2.6x, 96 rows 1.2-1.6x.
template <int T>
static int qms_blocks(int64_t M) {
  const int mb = M <= 16 ? 1 : M <= 32 ? 2 : M <= 48 ? 3 : M <= 64 ? 4 : M <= 96 ? 6 : 0;
  const bool ok = mb == 6   ? QmsPlan<T, 8, 1, 6>::kValid
                  : mb == 4 ? QmsPlan<T, 8, 1, 4>::kValid
                  : mb == 3 ? QmsPlan<T, 8, 1, 3>::kValid
                            : mb > 0 && QmsPlan<T, 8, 1, 2>::kValid;
  return ok ? mb : 0;
}

// Plan and launch the small-batch kernel for type T (qms_blocks(M) > 0): row groups of WV * 16 * NB
// weight rows (8 waves of 16 rows unless the tuning asks otherwise), units divided over at most one
// workgroup per CU, at least min_cols columns each.
template <int T>
static hipError_t launch_qms(QmsArgs& a, int num_cus, const QmmWorkspace& ws, hipStream_t s) {
  if (a.tbl_bytes != qmm_tbl_bytes<T>()) return hipErrorInvalidValue;
  const int mb = qms_blocks<T>(a.M);
  // 16 waves of 16 rows on products of at least 2^26 weights and up to 16 activation rows (the
  // 17408-row and 17408-wide 27B projections: 4-10% faster than 8 waves, whose two waves per SIMD
  // leave the decode's LDS and MFMA latency exposed; the smaller products, with fewer row groups per
  // CU, are faster with 8). With more activation rows the MFMAs cover that latency: 8 waves are
  // within 4% at 32 rows and even at 64.
  const bool big = mb == 1 && (long long)a.N * a.K >= (1ll << 26) && QmsPlan<T, 16, 1, 1>::kValid;
  const int wv = mb > 1 ? 8
               : g_qmm_tuning.small_waves == 4 ? 4
               : g_qmm_tuning.small_waves == 16 ? 16
               : g_qmm_tuning.small_waves == 8 ? 8 : (big ? 16 : 8);
  const int nb = mb > 1 ? 1 : g_qmm_tuning.small_nb == 2 ? 2 : (g_qmm_tuning.small_nb == 4 ? 4 : 1);
  const int rg = wv * 16 * nb;
  const long long units = (((long long)a.N + rg - 1) / rg) * a.nblk;
  if (units >= (1ll << 31)) return hipErrorInvalidValue;
  a.units = (int)units;
  const int min_cols = g_qmm_tuning.small_min_cols > 0 ? g_qmm_tuning.small_min_cols : 1;
  const int gmax = (a.units + min_cols - 1) / min_cols;
  a.G = num_cus < gmax ? num_cus : gmax;
  if (a.G > ws.max_groups) a.G = ws.max_groups;
  // the partials of G workgroups must fit the workspace (slot: MB * NB * 64 * WV float4)
  while (a.G > 1 && 2ll * a.G * (mb * nb * 64 * wv * 16) > ws.part_bytes) --a.G;
  a.xcd_remap = (a.G % 8 == 0) ? 1 : 0;
  a.part = ws.part;
  a.part_bytes = ws.part_bytes;
  a.cnt = ws.cnt;
  const bool a4 = (reinterpret_cast<uintptr_t>(a.packed) & 3) == 0;
  switch (mb) {
    case 1: break;
    case 2: return launch_qms_a4<T, 8, 1, 2>(a, a4, s);
    case 3: return launch_qms_a4<T, 8, 1, 3>(a, a4, s);
    case 4: return launch_qms_a4<T, 8, 1, 4>(a, a4, s);
    case 6: return launch_qms_a4<T, 8, 1, 6>(a, a4, s);
    default: return hipErrorInvalidValue;
  }
  if (wv == 16) return launch_qms_a4<T, 16, 1, 1>(a, a4, s);
  if (wv == 8)
    return nb == 4 ? launch_qms_a4<T, 8, 4, 1>(a, a4, s) : nb == 2 ? launch_qms_a4<T, 8, 2, 1>(a, a4, s)
                                                                   : launch_qms_a4<T, 8, 1, 1>(a, a4, s);
  return nb == 4 ? launch_qms_a4<T, 4, 4, 1>(a, a4, s) : nb == 2 ? launch_qms_a4<T, 4, 2, 1>(a, a4, s)
                                                                 : launch_qms_a4<T, 4, 1, 1>(a, a4, s);
}

template <int T>
static hipError_t launch_generic_t(const QmmArgs& a, hipStream_t s) {
  dim3 grid((unsigned)((a.N + kGBN - 1) / kGBN), (unsigned)((a.M + kGBM - 1) / kGBM));
  hipLaunchKernelGGL(qmm_generic_kernel<T>, grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

template <int T>
static hipError_t launch_qmm_type(const uint8_t* packed, const void* x, int xdt, void* y, int ydt, int64_t M,
                                  int64_t N, int K, const DevTables& tb, int num_cus, const QmmWorkspace& ws,
                                  hipStream_t s) {
  const bool small = M >= 1 && (g_qmm_tuning.small_max_m == 0 || M <= g_qmm_tuning.small_max_m) && qms_blocks<T>(M) > 0;
  const bool x16 = (reinterpret_cast<uintptr_t>(x) & 15) == 0;  // the MFMA kernels read 16-byte pieces
  if (xdt == QDT_F16 && x16 && ws.part && small && N < (1ll << 31)) {
    QmsArgs a{};
    a.packed = packed;
    a.x = static_cast<const _Float16*>(x);
    a.y = y;
    a.M = (int)M;
    a.N = (int)N;
    a.K = K;
    a.y_dtype = ydt;
    a.nblk = K / 256;
    a.row_bytes = (long long)a.nblk * BlockBytes<T>::v;
    if (qmm_grid_type(T)) {
      if (!tb.qmm_tbl) return hipErrorInvalidValue;
      a.tbl = tb.qmm_tbl;
      a.tbl_bytes = qmm_table_bytes(T);
    }
    return launch_qms<T>(a, num_cus, ws, s);
  }
  if (xdt == QDT_F16 && x16 && ws.part && M < (1ll << 31) && N < (1ll << 31)) {
    QmmMfmaArgs a{};
    a.packed = packed;
    a.x = static_cast<const _Float16*>(x);
    a.y = y;
    a.M = (int)M;
    a.N = (int)N;
    a.K = K;
    a.y_dtype = ydt;
    a.nblk = K / 256;
    a.row_bytes = (long long)a.nblk * BlockBytes<T>::v;
    if (qmm_grid_type(T)) {
      if (!tb.qmm_tbl) return hipErrorInvalidValue;
      a.tbl = tb.qmm_tbl;
      a.tbl_bytes = qmm_table_bytes(T);
    }
    return launch_mfma<T>(a, num_cus, ws, s);
  }
  QmmArgs a;
  a.packed = packed; a.x = x; a.y = y; a.M = M; a.N = N; a.K = K; a.x_dtype = xdt; a.y_dtype = ydt; a.tb = tb;
  return launch_generic_t<T>(a, s);
}

}  // namespace gsq
