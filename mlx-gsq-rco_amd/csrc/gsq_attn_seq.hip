// Gated grouped-query attention of a prompt (several new tokens at once) for the Qwen3.5-hybrid
// decoder: what models/qwen35.py's torch formulation of FullAttention computes between the q / k /
// v projections and the output projection (the reference runs mlx-lm's attention there,
// mlx_gsq/models/qwen35.py:114-152), in two launches:
//
//  * attn_prep_seq_kernel: q and k RMS-normalized per head and rotated, k and v into the caches;
//  * attn_seq_kernel: online-softmax attention over the caches and the sigmoid gate; for a few tokens
//    over a long context in chunks of positions, whose sums attn_merge_seq_kernel puts together.
//
// Before, the torch formulation took tens of launches, float32 copies of the caches, two float32
// GEMMs over all max_len positions and several passes over a (heads, tokens, max_len) float32
// score matrix: ~1790 us of a layer over 1024 tokens with a 4096-position cache (24 heads of 256);
// these two kernels 22 + 51 us.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "gsq_common.h"

namespace gsq {

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// 16-bit activation types. Terms: how many 16-bit values hold a softmax probability (fp32) to fp32
// accuracy: 11 + 11 bits in fp16 (scaled by 2^14, so that the low part of every probability that
// matters is a normal number), 8 + 8 + 8 in bf16.
template <bool BF>
struct A16;
template <>
struct A16<false> {
  static constexpr int kTerms = 2;
  static constexpr float kScale = 14.f;  // log2
  // two values rounded to nearest, and as a pair of floats again
  __device__ static uint32_t pack(f32x2 v) { return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2)); }
  __device__ static f32x2 unpack(uint32_t w) { return __builtin_convertvector(__builtin_bit_cast(f16x2, w), f32x2); }
  __device__ static float ld(uint16_t b) { return (float)__builtin_bit_cast(_Float16, b); }
  __device__ static uint16_t mk(float v) { return __builtin_bit_cast(uint16_t, (_Float16)v); }
  __device__ static f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
template <>
struct A16<true> {
  static constexpr int kTerms = 3;
  static constexpr float kScale = 0.f;
  __device__ static uint32_t pack(f32x2 v) { return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2)); }
  __device__ static f32x2 unpack(uint32_t w) { return (f32x2){ld((uint16_t)w), ld((uint16_t)(w >> 16))}; }
  __device__ static float ld(uint16_t b) { return __builtin_bit_cast(float, (uint32_t)b << 16); }
  __device__ static uint16_t mk(float v) { return (uint16_t)f32_to_bf16_bits(v); }
  __device__ static f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};

// True (uniformly) if the new tokens do not all lie inside the cache: every output row is then NaN
// and the caches are left alone, as the single-token kernels do for such a position.
__device__ __forceinline__ bool seq_pos_invalid(const AttnSeqArgs& a) {
  return a.pos[0] < 0 || a.pos[0] > (int64_t)a.L - a.S;
}

template <int N>
__device__ __forceinline__ void wait_vm() {
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// v_exp_f32: 2^x to one ulp (results below the normal range are 0)
__device__ __forceinline__ float exp2_raw(float x) { return __builtin_amdgcn_exp2f(x); }

// Transposing LDS read: 16 lanes read 4 rows of 16 values (lane j: values 4 (j % 4) .. + 3 of row
// j / 4, 8 bytes); lane j gets column j of the four rows.
__device__ __forceinline__ s16x4 tr_read(const uint8_t* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
}

}  // namespace

// One workgroup per token: a wave per head over the query and key heads, kPrepHeads at a time, all
// their loads issued before the rotary factors of the position are formed (angles in double, as
// the single-token kernels form them) and before any is used: RMS norm and rounding, rotate-half
// on the first rd dims and rounding; k and v go into the caches, q to scratch as (B, H, S, hd).
// Bound by memory latency (q, k, v read once and written once): 1024 tokens of 28 heads of 256 took
// 28 us with each head's loads waited for in turn, 22 so.
constexpr int kPrepHeads = 8;

template <bool BF, int HD>
__global__ void __launch_bounds__(256) attn_prep_seq_kernel(AttnSeqArgs a) {
  using E = A16<BF>;
  constexpr int V = HD / 64;  // consecutive values per lane
  typedef uint16_t vec_t __attribute__((ext_vector_type(V)));
  __shared__ float row[4][HD], cs[HD / 2], sn[HD / 2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, d0 = V * lane;
  const int t = blockIdx.x, bb = blockIdx.y, rd = a.rd, hr = rd / 2, nh = a.H + a.Hkv;
  if (seq_pos_invalid(a)) return;
  const int64_t p = a.pos[0] + t, r = (int64_t)bb * a.S + t;
  const uint16_t* qg = static_cast<const uint16_t*>(a.qg) + r * a.qg_stride + d0;
  const uint16_t* kn = static_cast<const uint16_t*>(a.k) + r * a.k_stride + d0;
  const uint16_t* vn = static_cast<const uint16_t*>(a.v) + r * a.v_stride + d0;
  float wq[V], wk[V];
#pragma unroll
  for (int j = 0; j < V; ++j) {
    wq[j] = E::ld(static_cast<const uint16_t*>(a.q_norm_w)[d0 + j]);
    wk[j] = E::ld(static_cast<const uint16_t*>(a.k_norm_w)[d0 + j]);
  }
  for (int h0 = wave; h0 < nh; h0 += 4 * kPrepHeads) {
    uint16_t x[kPrepHeads][V];
#pragma unroll
    for (int u = 0; u < kPrepHeads; ++u) {
      const int h = min(h0 + 4 * u, nh - 1);
      const uint16_t* src = h < a.H ? qg + (int64_t)h * 2 * HD : kn + (int64_t)(h - a.H) * HD;
#pragma unroll
      for (int j = 0; j < V; ++j) x[u][j] = src[j];
    }
    if (h0 == wave) {
      if (tid < hr) {
        const double ang = (double)p * a.inv_freq[tid];
        cs[tid] = (float)cos(ang);
        sn[tid] = (float)sin(ang);
      }
      __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < kPrepHeads; ++u) {
      const int h = h0 + 4 * u, kh = h - a.H;
      if (h >= nh) break;
      const bool isq = h < a.H;
      const int64_t cache = (((int64_t)bb * a.Hkv + kh) * a.L + p) * HD + d0;
      uint16_t* dst = isq ? static_cast<uint16_t*>(a.q) + (((int64_t)bb * a.H + h) * a.S + t) * HD + d0
                          : static_cast<uint16_t*>(a.kc) + cache;
      float f[V], ss = 0.f;
#pragma unroll
      for (int j = 0; j < V; ++j) {
        f[j] = E::ld(x[u][j]);
        ss += f[j] * f[j];
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
      const float rn = 1.f / sqrtf(ss / (float)HD + a.eps);
      // the wave's own row area: its LDS operations complete in order
#pragma unroll
      for (int j = 0; j < V; ++j) row[wave][d0 + j] = f[j] = E::ld(E::mk(f[j] * rn * (isq ? wq[j] : wk[j])));
      __builtin_amdgcn_wave_barrier();
      vec_t o;
#pragma unroll
      for (int j = 0; j < V; ++j) {
        const int d = d0 + j;
        float v = f[j];
        if (d < rd) {
          const int i = d < hr ? d : d - hr;
          const float other = d < hr ? -row[wave][d + hr] : row[wave][i];
          v = v * cs[i] + other * sn[i];
        }
        o[j] = E::mk(v);
      }
      *reinterpret_cast<vec_t*>(dst) = o;
      if (!isq) {
        vec_t vv;
#pragma unroll
        for (int j = 0; j < V; ++j) vv[j] = vn[(int64_t)kh * HD + j];
        *reinterpret_cast<vec_t*>(static_cast<uint16_t*>(a.vc) + cache) = vv;
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// 64 query tokens of one head per workgroup, 16 per wave, over tiles of 64 cached positions: two
// groups of four waves take the even and the odd tiles, and their maxima, sums and outputs are
// merged at the end (a prompt's last query tile is a chain of all its key tiles, and
// that chain is the kernel's time: 1024 tokens of 24 heads of 256, 72 us with one group and two
// workgroups per CU, 51 with two and the powers of two below).
//
//  * Both products are formed transposed: S^T = K Q^T puts a query on each lane column (lane % 16)
//    and keys 4 (lane / 16) + e of every 16-key block on its registers, which is what the B operand
//    of O^T = V^T P^T needs (its k-slots 8 g .. 8 g + 7 of lane group g hold keys 4 g .. + 3 of
//    two blocks): probabilities never leave their lane, the softmax state is per lane, and the
//    rescaling of O is one multiply per register.
//  * P stays at fp32 accuracy: 2 fp16 or 3 bf16 terms (A16), each its own MFMA; K, V and Q are the
//    16-bit values the caches hold, so the products with them are exact.
//  * K and V tiles come by DMA into one LDS buffer each, V's while the scores are formed and the
//    next K's while P V is: 64 KB a group at hd = 256. 16-byte octets are
//    XOR-swizzled by key so that the reads are free of bank conflicts; V^T operands are
//    transposing reads (four keys x 16 dims per 16 lanes).
//
// Bound by LDS reads (every wave reads the whole K and V tile: ~2000 cycles a tile of 64 x 64
// against ~1500 of MFMA); late tiles of the triangle are started first.
//
// SPLIT: workgroup z of a query tile takes positions z * chunk .. + chunk - 1 and leaves its maximum,
// sum and unnormalized outputs to attn_merge_seq_kernel. A tile's chain of key tiles costs 29 ns a
// position, and 2 tokens of 24 heads are 24 workgroups: unsplit 956 us over 32768 positions and 4070
// over 131072 (the torch formulation 722 and 1748), in 8 and 10 chunks 189 and 550.
template <bool BF, int HD, bool SPLIT>
__global__ void __launch_bounds__(512, 2) attn_seq_kernel(AttnSeqArgs a) {
  using E = A16<BF>;
  constexpr int NO = HD / 8, KS = HD / 32, NI = NO / 4, DB = HD / 16, RB = HD * 2;  // RB: bytes of a row
  constexpr int SH = HD == 64 ? 1 : 0;  // 128-byte rows: two rows to the 64 banks
  // dynamic LDS: reads of a static array would wait for every DMA in flight, the other buffer's too
  extern __shared__ __attribute__((aligned(16))) uint8_t attn_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave8 = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave = wave8 & 3, grp = wave8 >> 2;
  uint8_t* const kt = attn_lds + grp * 128 * RB;
  uint8_t* const vt = kt + 64 * RB;
  const int g = lane >> 4, c = lane & 15;
  const int ntile = (a.S + 63) / 64, h = blockIdx.x % a.H, tile = ntile - 1 - blockIdx.x / a.H, bb = blockIdx.y;
  const int t0 = tile * 64, tw = t0 + 16 * wave, t = min(tw + c, a.S - 1);  // rows past S repeat the last
  const bool on = tw + c < a.S;
  uint16_t* const out = static_cast<uint16_t*>(a.out) + ((int64_t)bb * a.S + t) * a.out_stride + (int64_t)h * HD;
  if (seq_pos_invalid(a)) {
    if (!SPLIT && on && grp == 0)
      for (int i = 0; i < DB; ++i)
        for (int e = 0; e < 4; ++e) out[16 * i + 4 * g + e] = E::mk(__builtin_nanf(""));
    return;
  }
  const int pos = (int)a.pos[0], len = pos + a.S;
  // key tiles kt_begin .. kt_end - 1, an even number of them unless they end the tile's keys
  const int nk = (pos + min(t0 + 63, a.S - 1)) / 64 + 1;
  const int kt_begin = SPLIT ? (int)blockIdx.z * (a.chunk / 64) : 0;
  const int kt_end = SPLIT ? min(nk, kt_begin + a.chunk / 64) : nk;
  if (SPLIT && kt_begin >= nk) return;  // every position of the chunk is past the tile's last token
  const int64_t base = ((int64_t)bb * a.Hkv + h / (a.H / a.Hkv)) * a.L * HD;
  const uint16_t* const Kg = static_cast<const uint16_t*>(a.kc) + base;
  const uint16_t* const Vg = static_cast<const uint16_t*>(a.vc) + base;
  auto ksw = [](int key) { return (key >> SH) & (NO < 16 ? NO - 1 : 15); };
  auto vsw = [](int key) { return ((key >> SH) & (NO < 16 ? NO / 2 - 1 : 7)) << 1; };
  auto issue = [&](const uint16_t* src, uint8_t* dst, int k0, auto sw) {  // keys past the last repeat it
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int e = (wave * NI + i) * 64 + lane, key = e / NO, o = (e % NO) ^ sw(key);
      __builtin_amdgcn_global_load_lds(src + (int64_t)min(k0 + key, len - 1) * HD + 8 * o,
                                       (lds_ptr_t)(dst + (wave * NI + i) * 1024), 16, 0, 0);
    }
  };
  issue(Kg, kt, 64 * (kt_begin + grp), ksw);
  issue(Vg, vt, 64 * (kt_begin + grp), vsw);
  u32x4 qf[KS];
  {
    const uint16_t* q = static_cast<const uint16_t*>(a.q) + (((int64_t)bb * a.H + h) * a.S + t) * HD + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = *reinterpret_cast<const u32x4*>(q + 32 * s);
  }
  f32x4 acc[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i) acc[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;  // l: this lane's share of the row sum
  // probabilities as powers of two of one fused multiply-add: the products are not rounded before the
  // maximum is taken off, and the rounding of (maximum x c) is common to a row
  const float c_ = 1.44269504088896340736f / sqrtf((float)HD);
  const int qpos = pos + t, wmin = pos + min(tw, a.S - 1), wmax = pos + min(tw + 15, a.S - 1);
  // lane bases of the K and V reads (their swizzles depend on the lane only)
  const uint8_t* const kb = kt + c * RB;
  const int kx = ksw(c), vkey = 4 * g + (c >> 2), vx = vsw(vkey);
  const uint8_t* const vb = vt + vkey * RB + (((c & 3) >> 1) << 4) + ((c & 1) << 3);
  // the query fragments (loaded after the tiles' DMA) are in registers before the loop counts loads
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  for (int kt0 = kt_begin; kt0 < kt_end; kt0 += 2) {
    const int k0 = (kt0 + grp) * 64;
    const bool live = k0 <= wmax, more = kt0 + 2 < kt_end;  // a tile past the wave's last position: barriers only
    wait_vm<NI>();  // K has landed (V's DMA may be in flight)
    asm volatile("s_barrier" ::: "memory");
    f32x4 s[4];
    if (live) {
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        s[b] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          s[b] = E::mma(*reinterpret_cast<const u32x4*>(kb + 16 * b * RB + (((4 * ks + g) ^ kx) << 4)), qf[ks], s[b]);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // every wave is done with K
    if (more) issue(Kg, kt, k0 + 128, ksw);
    u32x4 pf[E::kTerms][2];
    if (live) {
      float mx = -INFINITY;
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (k0 + 63 > wmin && k0 + 16 * b + 4 * g + e > qpos) s[b][e] = -INFINITY;
          mx = fmaxf(mx, s[b][e]);
        }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float mn = fmaxf(m, mx), ms = mn == -INFINITY ? 0.f : mn;
      const float alpha = exp2_raw((m - ms) * c_), off = E::kScale - ms * c_;
      m = mn;
      float sum = 0.f;
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[b][e] = exp2_raw(__builtin_fmaf(s[b][e], c_, off));
          sum += s[b][e];
        }
      l = l * alpha + sum;
      if (__any(alpha != 1.f)) {
#pragma unroll
        for (int i = 0; i < DB; ++i) acc[i] *= alpha;
      }
#pragma unroll
      for (int n = 0; n < E::kTerms; ++n)
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
          for (int j = 0; j < 4; ++j) {  // a pair of k-slots
            f32x4& v = s[2 * hf + (j >> 1)];
            const f32x2 p2 = j & 1 ? v.zw : v.xy;
            const uint32_t w = E::pack(p2);
            pf[n][hf][j] = w;
            if (n + 1 < E::kTerms) {  // what the term leaves, for the next one
              const f32x2 left = p2 - E::unpack(w);
              if (j & 1) v.zw = left;
              else v.xy = left;
            }
          }
    }
    if (more) wait_vm<NI>();  // V has landed (the next K's DMA may be in flight)
    else wait_vm<0>();
    asm volatile("s_barrier" ::: "memory");
    if (live) {
#pragma unroll
      for (int i = 0; i < DB; ++i) {
        const uint8_t* va = vb + (((2 * i) ^ vx) << 4);
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
          struct { s16x4 a, b; } v;
          v.a = tr_read(va + (32 * hf) * RB);
          v.b = tr_read(va + (32 * hf + 16) * RB);
          const u32x4 vf = __builtin_bit_cast(u32x4, v);
#pragma unroll
          for (int n = 0; n < E::kTerms; ++n) acc[i] = E::mma(vf, pf[n][hf], acc[i]);
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // every wave is done with V
    if (more) issue(Vg, vt, k0 + 128, vsw);
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  // merge (every wave is past its last tile read): each group gives its twin lane the other half of
  // the dims through LDS and finishes its own
  constexpr int HB = DB / 2;
  f32x4* const mo = reinterpret_cast<f32x4*>(attn_lds) + wave * HB * 64 + lane;
  float2* const ml = reinterpret_cast<float2*>(attn_lds + 8 * HB * 1024) + wave * 64 + lane;
  static_assert(8 * HB * 1024 + 8 * 512 <= 256 * RB);
#pragma unroll
  for (int i = 0; i < HB; ++i) mo[grp * 4 * HB * 64 + i * 64] = grp ? acc[i] : acc[HB + i];
  ml[grp * 256] = make_float2(m, l);
  __syncthreads();
  if (!on) return;
  const float2 o1 = ml[(grp ^ 1) * 256];
  const float mm = fmaxf(m, o1.x), ms = mm == -INFINITY ? 0.f : mm;
  const float s0 = exp2_raw((m - ms) * c_), s1 = exp2_raw((o1.x - ms) * c_);  // a group without keys: 0 of nothing
  if constexpr (SPLIT) {
    const int64_t rows = (int64_t)a.B * a.H * a.S * a.nsplit;
    const int64_t r = (((int64_t)bb * a.H + h) * a.S + t) * a.nsplit + blockIdx.z;
    float* const po = a.part + r * HD + 16 * grp * HB + 4 * g;
#pragma unroll
    for (int i = 0; i < HB; ++i)
      *reinterpret_cast<f32x4*>(po + 16 * i) =
          (grp ? acc[HB + i] : acc[i]) * s0 + mo[(grp ^ 1) * 4 * HB * 64 + i * 64] * s1;
    if (grp == 0 && g == 0)
      *reinterpret_cast<float2*>(a.part + rows * HD + 2 * r) = make_float2(mm, l * s0 + o1.y * s1);
    return;
  }
  const float inv = 1.f / (l * s0 + o1.y * s1);
  const uint16_t* gate = static_cast<const uint16_t*>(a.qg) + ((int64_t)bb * a.S + t) * a.qg_stride + (int64_t)h * 2 * HD + HD;
#pragma unroll
  for (int i = 0; i < HB; ++i) {
    const int d = 16 * (grp * HB + i) + 4 * g;
    const f32x4 v = (grp ? acc[HB + i] : acc[i]) * s0 + mo[(grp ^ 1) * 4 * HB * 64 + i * 64] * s1;
    const uint2 gw = *reinterpret_cast<const uint2*>(gate + d);
    const uint16_t gv[4] = {(uint16_t)gw.x, (uint16_t)(gw.x >> 16), (uint16_t)gw.y, (uint16_t)(gw.y >> 16)};
    uint16_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = E::mk(v[e] * inv * (1.f / (1.f + expf(-E::ld(gv[e])))));
    *reinterpret_cast<uint2*>(out + d) =
        make_uint2((uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16));
  }
}

// Outputs of a split prompt: a wave per (row, head, token) weighs the chunks that hold positions of the
// token by their maxima, as the wave groups are merged above, normalizes and gates. Bound by reading
// the partial outputs once (24 heads, 16 tokens, 10 chunks of 256 dims: 3.9 MB).
template <bool BF, int HD>
__global__ void __launch_bounds__(256) attn_merge_seq_kernel(AttnSeqArgs a) {
  using E = A16<BF>;
  constexpr int V = HD / 64;
  const int64_t rows = (int64_t)a.B * a.H * a.S, i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (i >= rows) return;
  const int d = V * (threadIdx.x & 63), t = (int)(i % a.S), h = (int)(i / a.S % a.H);
  const int64_t tok = i / a.S / a.H * a.S + t;
  uint16_t* const out = static_cast<uint16_t*>(a.out) + tok * a.out_stride + (int64_t)h * HD + d;
  const uint16_t* const gate = static_cast<const uint16_t*>(a.qg) + tok * a.qg_stride + (int64_t)h * 2 * HD + HD + d;
  const bool invalid = seq_pos_invalid(a);
  const int nz = invalid ? 0 : (int)((a.pos[0] + t) / a.chunk) + 1;
  const float* const po = a.part + i * a.nsplit * HD + d;
  const float2* const ml = reinterpret_cast<const float2*>(a.part + rows * a.nsplit * HD) + i * a.nsplit;
  const float c_ = 1.44269504088896340736f / sqrtf((float)HD);
  float m = -INFINITY, l = 0.f, o[V];
#pragma unroll
  for (int j = 0; j < V; ++j) o[j] = 0.f;
  for (int z = 0; z < nz; ++z) m = fmaxf(m, ml[z].x);
  const float ms = m == -INFINITY ? 0.f : m;
  for (int z = 0; z < nz; ++z) {
    const float w = exp2_raw((ml[z].x - ms) * c_);
    l += ml[z].y * w;
#pragma unroll
    for (int j = 0; j < V; ++j) o[j] += po[(int64_t)z * HD + j] * w;
  }
  const float inv = 1.f / l;
#pragma unroll
  for (int j = 0; j < V; ++j)
    out[j] = E::mk(invalid ? __builtin_nanf("") : o[j] * inv * (1.f / (1.f + expf(-E::ld(gate[j])))));
}

template <bool BF>
static hipError_t launch_attn_seq_t(const AttnSeqArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)((a.S + 63) / 64 * a.H), (unsigned)a.B, (unsigned)a.nsplit);
  const dim3 pgrid((unsigned)a.S, (unsigned)a.B);
  auto launch = [&](auto hd) -> hipError_t {
    constexpr int HD = decltype(hd)::value;
    constexpr int lds = 2 * 2 * 64 * HD * 2;  // two groups' K and V tiles: 64 rows of 2 hd bytes each
    const bool split = a.nsplit > 1;
    const int64_t rows = (int64_t)a.B * a.H * a.S;
    if (split && (rows + 3) / 4 >= (1ll << 31)) return hipErrorInvalidValue;
    static LdsLimit limit, split_limit;
    const hipError_t e = split ? split_limit.raise((const void*)attn_seq_kernel<BF, HD, true>, lds)
                               : limit.raise((const void*)attn_seq_kernel<BF, HD, false>, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((attn_prep_seq_kernel<BF, HD>), pgrid, dim3(256), 0, s, a);
    if (split) {
      hipLaunchKernelGGL((attn_seq_kernel<BF, HD, true>), grid, dim3(512), lds, s, a);
      hipLaunchKernelGGL((attn_merge_seq_kernel<BF, HD>), dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s, a);
    } else {
      hipLaunchKernelGGL((attn_seq_kernel<BF, HD, false>), grid, dim3(512), lds, s, a);
    }
    return hipGetLastError();
  };
  if (a.hd == 256) return launch(std::integral_constant<int, 256>{});
  if (a.hd == 128) return launch(std::integral_constant<int, 128>{});
  if (a.hd == 64) return launch(std::integral_constant<int, 64>{});
  return hipErrorInvalidValue;
}

hipError_t launch_attn_seq(bool bf16, const AttnSeqArgs& a, hipStream_t s) {
  return bf16 ? launch_attn_seq_t<true>(a, s) : launch_attn_seq_t<false>(a, s);
}

}  // namespace gsq
