// Gated grouped-query attention of a prompt (several new tokens at once) for the Qwen3.5-hybrid
// decoder: what models/qwen35.py's torch formulation of FullAttention computes between the q / k /
// v projections and the output projection (the reference runs mlx-lm's attention there,
// mlx_gsq/models/qwen35.py:114-152), in two launches:
//
//  * attn_prep_seq_kernel: q and k RMS-normalized per head and rotated, k and v into the caches;
//  * attn_seq_kernel: online-softmax attention over the caches and the sigmoid gate.
//
// Before, the torch formulation took tens of launches, float32 copies of the caches, two float32
// GEMMs over all max_len positions and several passes over a (heads, tokens, max_len) float32
// score matrix: ~1790 us of a layer over 1024 tokens with a 4096-position cache (24 heads of 256);
// these two kernels 26 + 72 us.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "gsq_common.h"

namespace gsq {

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
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
  static constexpr float kScale = 16384.f;
  __device__ static float ld(uint16_t b) { return (float)__builtin_bit_cast(_Float16, b); }
  __device__ static uint16_t mk(float v) { return __builtin_bit_cast(uint16_t, (_Float16)v); }
  __device__ static f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
template <>
struct A16<true> {
  static constexpr int kTerms = 3;
  static constexpr float kScale = 1.f;
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

// Transposing LDS read: 16 lanes read 4 rows of 16 values (lane j: values 4 (j % 4) .. + 3 of row
// j / 4, 8 bytes); lane j gets column j of the four rows.
__device__ __forceinline__ s16x4 tr_read(const uint8_t* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
}

}  // namespace

// One workgroup per token: the rotary factors of its position once (angles in double, as the
// single-token kernels form them), then a wave per head over the query and key heads: RMS norm and
// rounding, rotate-half on the first rd dims and rounding; k and v go into the caches, q to scratch
// as (B, H, S, hd). Bound by memory (q, k, v read once and written once).
template <bool BF>
__global__ void __launch_bounds__(256) attn_prep_seq_kernel(AttnSeqArgs a) {
  using E = A16<BF>;
  __shared__ float row[4][256], cs[128], sn[128];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int t = blockIdx.x, bb = blockIdx.y, hd = a.hd, rd = a.rd, hr = rd / 2;
  if (seq_pos_invalid(a)) return;
  const int64_t p = a.pos[0] + t, r = (int64_t)bb * a.S + t;
  if (tid < hr) {
    const double ang = (double)p * a.inv_freq[tid];
    cs[tid] = (float)cos(ang);
    sn[tid] = (float)sin(ang);
  }
  __syncthreads();
  const uint16_t* qg = static_cast<const uint16_t*>(a.qg) + r * a.qg_stride;
  const uint16_t* kn = static_cast<const uint16_t*>(a.k) + r * a.k_stride;
  const uint16_t* vn = static_cast<const uint16_t*>(a.v) + r * a.v_stride;
  for (int h = wave; h < a.H + a.Hkv; h += 4) {
    const bool isq = h < a.H;
    const int kh = h - a.H;
    const uint16_t* src = isq ? qg + (int64_t)h * 2 * hd : kn + (int64_t)kh * hd;
    const uint16_t* w = static_cast<const uint16_t*>(isq ? a.q_norm_w : a.k_norm_w);
    const int64_t cache = (((int64_t)bb * a.Hkv + kh) * a.L + p) * hd;
    uint16_t* dst = isq ? static_cast<uint16_t*>(a.q) + (((int64_t)bb * a.H + h) * a.S + t) * hd
                        : static_cast<uint16_t*>(a.kc) + cache;
    float x[4], wv[4], ss = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int d = lane + 64 * j;
      x[j] = d < hd ? E::ld(src[d]) : 0.f;
      wv[j] = d < hd ? E::ld(w[d]) : 0.f;
      ss += x[j] * x[j];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
    const float rn = 1.f / sqrtf(ss / (float)hd + a.eps);
    // the wave's own row area: its LDS operations complete in order
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (lane + 64 * j < hd) row[wave][lane + 64 * j] = x[j] = E::ld(E::mk(x[j] * rn * wv[j]));
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int d = lane + 64 * j;
      if (d >= hd) continue;
      float v = x[j];
      if (d < rd) {
        const int i = d < hr ? d : d - hr;
        const float other = d < hr ? -row[wave][d + hr] : row[wave][i];
        v = v * cs[i] + other * sn[i];
      }
      dst[d] = E::mk(v);
      if (!isq) static_cast<uint16_t*>(a.vc)[cache + d] = vn[(int64_t)kh * hd + d];
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// 64 query tokens of one head per workgroup, 16 per wave, over tiles of 64 cached positions.
//
//  * Both products are formed transposed: S^T = K Q^T puts a query on each lane column (lane % 16)
//    and keys 4 (lane / 16) + e of every 16-key block on its registers, which is what the B operand
//    of O^T = V^T P^T needs (its k-slots 8 g .. 8 g + 7 of lane group g hold keys 4 g .. + 3 of
//    two blocks): probabilities never leave their lane, the softmax state is per lane, and the
//    rescaling of O is one multiply per register.
//  * P stays at fp32 accuracy: 2 fp16 or 3 bf16 terms (A16), each its own MFMA; K, V and Q are the
//    16-bit values the caches hold, so the products with them are exact.
//  * K and V tiles come by DMA into one LDS buffer each, V's while the scores are formed and the
//    next K's while P V is: 64 KB at hd = 256, two workgroups per CU. 16-byte octets are
//    XOR-swizzled by key so that the reads are free of bank conflicts; V^T operands are
//    transposing reads (four keys x 16 dims per 16 lanes).
//
// Bound by LDS reads (every wave reads the whole K and V tile: ~2000 cycles a tile of 64 x 64
// against ~1500 of MFMA); late tiles of the triangle are started first.
template <bool BF, int HD>
__global__ void __launch_bounds__(256, 2) attn_seq_kernel(AttnSeqArgs a) {
  using E = A16<BF>;
  constexpr int NO = HD / 8, KS = HD / 32, NI = NO / 4, DB = HD / 16, RB = HD * 2;  // RB: bytes of a row
  constexpr int SH = HD == 64 ? 1 : 0;  // 128-byte rows: two rows to the 64 banks
  // dynamic LDS: reads of a static array would wait for every DMA in flight, the other buffer's too
  extern __shared__ __attribute__((aligned(16))) uint8_t attn_lds[];
  uint8_t* const kt = attn_lds;
  uint8_t* const vt = attn_lds + 64 * RB;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c = lane & 15;
  const int ntile = (a.S + 63) / 64, h = blockIdx.x % a.H, tile = ntile - 1 - blockIdx.x / a.H, bb = blockIdx.y;
  const int t0 = tile * 64, tw = t0 + 16 * wave, t = min(tw + c, a.S - 1);  // rows past S repeat the last
  const bool on = tw + c < a.S;
  uint16_t* const out = static_cast<uint16_t*>(a.out) + ((int64_t)bb * a.S + t) * a.out_stride + (int64_t)h * HD;
  if (seq_pos_invalid(a)) {
    if (on)
      for (int i = 0; i < DB; ++i)
        for (int e = 0; e < 4; ++e) out[16 * i + 4 * g + e] = E::mk(__builtin_nanf(""));
    return;
  }
  const int pos = (int)a.pos[0], len = pos + a.S;
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
  issue(Kg, kt, 0, ksw);
  issue(Vg, vt, 0, vsw);
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
  const float scale = 1.f / sqrtf((float)HD);
  const int qpos = pos + t, wmin = pos + min(tw, a.S - 1), wmax = pos + min(tw + 15, a.S - 1);
  const int nk = (pos + min(t0 + 63, a.S - 1)) / 64 + 1;
  // lane bases of the K and V reads (their swizzles depend on the lane only)
  const uint8_t* const kb = kt + c * RB;
  const int kx = ksw(c), vkey = 4 * g + (c >> 2), vx = vsw(vkey);
  const uint8_t* const vb = vt + vkey * RB + (((c & 3) >> 1) << 4) + ((c & 1) << 3);
  // the query fragments (loaded after the tiles' DMA) are in registers before the loop counts loads
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  for (int kt0 = 0; kt0 < nk; ++kt0) {
    const int k0 = kt0 * 64;
    const bool live = k0 <= wmax, more = kt0 + 1 < nk;  // a tile past the wave's last position: barriers only
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
    if (more) issue(Kg, kt, k0 + 64, ksw);
    u32x4 pf[E::kTerms][2];
    if (live) {
      float mx = -INFINITY;
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[b][e] *= scale;
          if (k0 + 63 > wmin && k0 + 16 * b + 4 * g + e > qpos) s[b][e] = -INFINITY;
          mx = fmaxf(mx, s[b][e]);
        }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float mn = fmaxf(m, mx), ms = mn == -INFINITY ? 0.f : mn;
      const float alpha = expf(m - ms);
      m = mn;
      float sum = 0.f;
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[b][e] = expf(s[b][e] - ms) * E::kScale;
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
            float* v = &(reinterpret_cast<float*>(&s[2 * hf + (j >> 1)])[2 * (j & 1)]);
            const uint16_t lo = E::mk(v[0]), hi = E::mk(v[1]);
            pf[n][hf][j] = (uint32_t)lo | ((uint32_t)hi << 16);
            v[0] -= E::ld(lo);
            v[1] -= E::ld(hi);
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
    if (more) issue(Vg, vt, k0 + 64, vsw);
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  const float inv = 1.f / l;
  if (!on) return;
  const uint16_t* gate = static_cast<const uint16_t*>(a.qg) + ((int64_t)bb * a.S + t) * a.qg_stride + (int64_t)h * 2 * HD + HD;
#pragma unroll
  for (int i = 0; i < DB; ++i) {
    const uint2 gw = *reinterpret_cast<const uint2*>(gate + 16 * i + 4 * g);
    const uint16_t gv[4] = {(uint16_t)gw.x, (uint16_t)(gw.x >> 16), (uint16_t)gw.y, (uint16_t)(gw.y >> 16)};
    uint16_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = E::mk(acc[i][e] * inv * (1.f / (1.f + expf(-E::ld(gv[e])))));
    *reinterpret_cast<uint2*>(out + 16 * i + 4 * g) =
        make_uint2((uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16));
  }
}

template <bool BF>
static hipError_t launch_attn_seq_t(const AttnSeqArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)((a.S + 63) / 64 * a.H), (unsigned)a.B);
  const size_t lds = (size_t)a.hd * 256;  // a K and a V tile: 64 rows of 2 hd bytes each
  hipLaunchKernelGGL(attn_prep_seq_kernel<BF>, dim3((unsigned)a.S, (unsigned)a.B), dim3(256), 0, s, a);
  if (a.hd == 256) hipLaunchKernelGGL((attn_seq_kernel<BF, 256>), grid, dim3(256), lds, s, a);
  else if (a.hd == 128) hipLaunchKernelGGL((attn_seq_kernel<BF, 128>), grid, dim3(256), lds, s, a);
  else if (a.hd == 64) hipLaunchKernelGGL((attn_seq_kernel<BF, 64>), grid, dim3(256), lds, s, a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_attn_seq(bool bf16, const AttnSeqArgs& a, hipStream_t s) {
  return bf16 ? launch_attn_seq_t<true>(a, s) : launch_attn_seq_t<false>(a, s);
}

}  // namespace gsq
