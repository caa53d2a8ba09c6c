// Fused GroupNorm (+FiLM) + SiLU, forward and backward, NHWC bf16 with fp32 statistics.
//
// Reference sites (diffusion/unet.py): F.silu(self.norm1(x)) at :151 and
// self.dropout(F.silu((w + 1) * self.norm2(x) + b)) at :157-159, with nn.GroupNorm(32, C)
// (:132-133, eps 1e-5, affine). Under autocast GroupNorm runs in fp32; the FP8 conv then
// rounds its input to bf16 (diffusion/fp8_kernels.py:835), which is what `out` stores.
//
// Layout: one workgroup per (image n, 64-channel slab): PLN pixel lanes (32, 64 or 128 by
// image size) x 8 granules of 8 channels (16 B of bf16). Every group of the slab lies inside
// the slab (64 % (C/G) == 0), so the statistics reduce inside the workgroup: 4-channel
// half-granule partials -> wave shuffles over the 8 pixel lanes of a wave -> LDS over the
// waves. Each lane keeps four 16-B loads in flight. The kernels make several passes over
// their inputs (after the first mostly from L2).
//
// Images of up to 1024 pixels, and of up to 4096 in launches that fill the GPU, use a resident
// form instead, whose workgroups hold their slab in registers. Others of 256+ pixels use a
// chunked form, which spreads each (image, slab) over workgroups of 128 pixels (against one
// workgroup per slab, whose passes were latency-bound): every workgroup holds its chunk in
// registers, and the per-group statistics cross workgroups through a workspace between two
// launches.
//   forward:  stats (chunk mean and sum of squared deviations per group) ->
//             apply (merge the chunks in order, Chan et al.'s pairwise update; normalise)
//   backward: sums (per-channel chunk sums of the four backward terms) ->
//             apply (chunk sums in order -> group means -> dx; chunk 0 also writes the
//             per-image dgamma/dbeta partials and the FiLM gradients)
#include "dpa_common.hpp"

#include <type_traits>

namespace dpa {

constexpr int kSlab = 64;  // channels per workgroup
constexpr int kGnUnrollFwd = 4;  // pixels per lane per loop iteration (loads in flight)
constexpr int kGnUnrollBwd = 2;  // (two sources per pixel)

struct GnArgs {
  const void* x;  // [N][HW][C] bf16, or fp32 for the chunked and small-image forms
  const uint16_t* dout;
  const float* gamma;
  const float* beta;
  const float* fs;  // film scale [N][C] or null
  const float* fb;  // film shift [N][C]
  void* out;  // forward: bf16 output; backward: dx in x's type
  float* mean;
  float* rstd;
  float* part;  // bwd: [2][N][C] per-image channel sums of dgamma / dbeta
  float* dfs;   // bwd: FiLM gradients [N][C] or null
  float* dfb;
  const uint16_t* wb;  // or FiLM from the bf16 time projection [N][2C]: scale bf16(w + 1), shift b
  uint16_t* dwb;       // bwd: its gradient [N][2C] bf16, or null
  const uint64_t* drop_seed;  // dropout after the SiLU: seed in device memory, or null
  uint32_t drop_keep;         // keep an element when its 16-bit hash is >= this (p * 2^16)
  float drop_scale;           // RN32(1 / (1 - p))
  const void* dx_add;  // bwd: a gradient added to dx (chunked and small forms), or null
  int dx_add_bf16;     // bwd: dx_add is bf16 while x and dx are fp32
  uint16_t* x_bf16;    // fwd: fp32 x also written as bf16 here (chunked and small forms), or null
  uint32_t* xb_part;   // fwd: with x_bf16, one amax partial of its bf16 values per workgroup,
  uint32_t xb_room;    //   and zeros in the rest of the room
  // Two-source x (a decoder stage's first GroupNorm with the upsample-and-concatenate before
  // it, diffusion/unet.py:379-382): channels [0, cat_ca) are the 2x nearest upsampling of
  // cat_a ([N][H/2][W/2][cat_ca], bf16), the others cat_h ([N][H][W][C - cat_ca], bf16 or
  // fp32); the concatenation they replace is fp32 and holds exactly these values. Images of
  // cat_w columns.
  const uint16_t* cat_a;
  const uint16_t* cat_h;
  int cat_ca, cat_w;
  int cat_hf;        // cat_h (and its gradient) fp32 instead of bf16 (forms with an fp32 x)
  uint16_t* cat_ga;  // bwd: gradient of cat_a (each 2x2 window of dx summed), bf16
  void* cat_gh;      // bwd: gradient of cat_h, in cat_h's type
  // Producer-fused cast for a delayed-scaling consumer (chunked and small forms): instead of
  // the bf16 output (fwd) or bf16 dx (bwd), e4m3(bf16 value / *q_scale) goes to q, and each
  // workgroup leaves the amax of its bf16 values in q_part[workgroup] (count in *q_count)
  uint8_t* q;
  const float* q_scale;
  uint32_t* q_part;
  uint32_t* q_count;
  int N, HW, C, G, cpg;
  float eps;
};

// Dropout of the GroupNorm+SiLU output (diffusion/unet.py:160, nn.Dropout before conv_2): the
// keep decision of element idx (NHWC index) is a counter hash of (seed, idx), so the backward
// recomputes the mask instead of storing it; kept values are scaled by 1 / (1 - p) in fp32
// before the bf16 rounding, as the reference drops its fp32 SiLU output before the conv's
// bf16 cast. The hash: splitmix64 of seed + (idx / 4) * golden ratio, one output per four
// elements: element idx is kept when bits [16 (idx % 4), 16 (idx % 4) + 16) of its hash, as
// a 16-bit number, are >= floor(p * 2^16). Four elements per 64-bit hash halve the hash's vector
// instructions against one per pair (its multiplies are done in 32-bit halves); 16 bits
// still give a drop rate within 2^-16 of p.
// The decisions come as masks of bf16 pairs (0xffff: kept), to be and'ed into packed values:
// four packed 16-bit instructions per pair instead of an extract, a compare and a select per
// element. r >= k is sat(k - r) == 0 in 16 bits, and min(., 1) - 1 turns that into the mask.
constexpr uint64_t kDropGolden = 0x9E3779B97F4A7C15ull;

// hash input of element idx (a multiple of 4)
__device__ __forceinline__ uint64_t drop_z(uint64_t seed, int64_t idx) {
  return seed + (uint64_t)(idx >> 2) * kDropGolden;
}

__device__ __forceinline__ uint32_t drop_mask2(uint32_t r, uint32_t keep2) {
  uint32_t m;
  // (as instructions of its own: the compiler turns the form into compares and selects)
  asm("v_pk_sub_u16 %0, %1, %2 clamp\n\tv_pk_min_u16 %0, %0, %3\n\tv_pk_sub_i16 %0, %0, %3"
      : "=&v"(m)
      : "v"(keep2), "v"(r), "v"(0x00010001u));
  return m;
}

// Masks of the 8 elements whose hash input starts at z0; keep2: the threshold in both halves.
__device__ __forceinline__ uint4 drop_mask8(uint64_t z0, uint32_t keep2) {
  uint32_t m[4];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    uint64_t z = z0 + (uint64_t)i * kDropGolden;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    m[2 * i] = drop_mask2((uint32_t)z, keep2);
    m[2 * i + 1] = drop_mask2((uint32_t)(z >> 32), keep2);
  }
  return uint4{m[0], m[1], m[2], m[3]};
}

__device__ __forceinline__ uint32_t drop_keep2(const GnArgs& p) {
  return p.drop_keep | (p.drop_keep << 16);
}

__device__ __forceinline__ uint4 and4(uint4 a, uint4 b) {
  return uint4{a.x & b.x, a.y & b.y, a.z & b.z, a.w & b.w};
}

// sigmoid(v) = 1 / (1 + e^-v) from the hardware exp2 and reciprocal (v_exp_f32, v_rcp_f32,
// about 1 ulp each), e^-v = 2^(-v log2 e). The SiLU and its derivative are rounded to bf16
// (2^16 fp32 ulps), so this changes an output bit only at rounding ties; the IEEE-exact
// exponential and division cost about a third of the forward kernels' time. Saturates as the
// exact form does: e^-v overflows to inf below v = -88.7 and the result is 0.
__device__ __forceinline__ float sigmoid_hw(float v) {
  const float e = __builtin_amdgcn_exp2f(v * -1.44269504f);
  return __builtin_amdgcn_rcpf(1.0f + e);
}

__device__ __forceinline__ void unpack8(uint4 v, float (&f)[8]) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __uint_as_float(w[i] << 16);
    f[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
  }
}

// Sum v over the PLN pixel lanes that share this thread's granule (64 / NG per wave by shuffles,
// then the waves in order through LDS); result valid in every lane. red holds
// (NG PLN / 64) waves x NG granules x NV floats.
template <int NV, int PLN, int NG = 8>
__device__ __forceinline__ void slab_reduce(float (&v)[NV], float* red) {
  constexpr int kWaves = NG * PLN / 64;
  const int gq = threadIdx.x & (NG - 1);
  const int wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    float s = v[k];
#pragma unroll
    for (int x = NG; x < 64; x *= 2) s += __shfl_xor(s, x, 64);
    v[k] = s;
  }
  if ((threadIdx.x & 63) < NG) {
#pragma unroll
    for (int k = 0; k < NV; ++k) red[(wave * NG + gq) * NV + k] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = red[gq * NV + k];
  // (with few values the reads of all waves are in flight at once)
#pragma unroll(NV <= 2 ? kWaves : 1)
  for (int w = 1; w < kWaves; ++w) {
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] += red[(w * NG + gq) * NV + k];
  }
  __syncthreads();
}

// Per-group value from half-granule (4-channel) sums hs[16] of the slab: group of this
// thread's channel half h (0/1) = consecutive cpg/4 half-granules.
__device__ __forceinline__ float group_sum(const float* hs, int half_idx, int cpg) {
  const int hpg = cpg / 4;  // half-granules per group (1, 2, 4, ... 16)
  const int g0 = (half_idx / hpg) * hpg;
  float s = 0.f;
  for (int i = 0; i < hpg; ++i) s += hs[g0 + i];
  return s;
}

// 8 consecutive floats (two 16-B loads when the address allows, as it does for torch's tensors)
__device__ __forceinline__ void load8f(const float* src, float (&v)[8]) {
  if ((reinterpret_cast<uintptr_t>(src) & 15) == 0) {
    const float4 a = reinterpret_cast<const float4*>(src)[0];
    const float4 b = reinterpret_cast<const float4*>(src)[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = src[e];
  }
}

// The same 8 floats as they are in memory, to be looked at later
__device__ __forceinline__ void load8raw(const float* src, uint4 (&v)[2]) {
  if ((reinterpret_cast<uintptr_t>(src) & 15) == 0) {
    v[0] = reinterpret_cast<const uint4*>(src)[0];
    v[1] = reinterpret_cast<const uint4*>(src)[1];
  } else {
    const uint32_t* s = reinterpret_cast<const uint32_t*>(src);
    v[0] = uint4{s[0], s[1], s[2], s[3]};
    v[1] = uint4{s[4], s[5], s[6], s[7]};
  }
}

__device__ __forceinline__ void floats8(const uint4 (&v)[2], float (&f)[8]) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    f[4 * h] = __uint_as_float(v[h].x);
    f[4 * h + 1] = __uint_as_float(v[h].y);
    f[4 * h + 2] = __uint_as_float(v[h].z);
    f[4 * h + 3] = __uint_as_float(v[h].w);
  }
}

// FiLM scale/shift of channels ch..ch+7 of image n: fp32 [N][C] pairs, or the bf16 time
// projection [N][2C] with scale bf16(w + 1) (the reference adds 1 in bf16) and shift b; no FiLM
// gives 1 and 0. Loading and use are apart: a kernel issues these loads before its pixels'
// (vector loads return in order: behind them, the first use would wait for every pixel) and
// looks at them after.
struct GnFilm {
  uint4 s[2], b[2];
  __device__ __forceinline__ void load(const GnArgs& p, int n, int ch) {
    if (p.fs) {
      load8raw(p.fs + (int64_t)n * p.C + ch, s);
      load8raw(p.fb + (int64_t)n * p.C + ch, b);
    } else if (p.wb) {
      const uint16_t* w = p.wb + (int64_t)n * 2 * p.C + ch;
      if ((reinterpret_cast<uintptr_t>(w) & 15) == 0) {  // (uniform: base alignment)
        s[0] = *reinterpret_cast<const uint4*>(w);
        b[0] = *reinterpret_cast<const uint4*>(w + p.C);
      } else {
        uint32_t t[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          t[e] = w[2 * e] | ((uint32_t)w[2 * e + 1] << 16);
          t[4 + e] = w[p.C + 2 * e] | ((uint32_t)w[p.C + 2 * e + 1] << 16);
        }
        s[0] = uint4{t[0], t[1], t[2], t[3]};
        b[0] = uint4{t[4], t[5], t[6], t[7]};
      }
    }
  }
  __device__ __forceinline__ bool get(const GnArgs& p, float (&fsc)[8], float (&fsh)[8]) const {
    if (p.fs) {
      floats8(s, fsc);
      floats8(b, fsh);
      return true;
    }
    if (p.wb) {
      float wf[8];
      unpack8(s[0], wf);
      unpack8(b[0], fsh);
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const uint32_t pk = pack_bf16x2(wf[e] + 1.0f, wf[e + 1] + 1.0f);
        fsc[e] = __uint_as_float(pk << 16);
        fsc[e + 1] = __uint_as_float(pk & 0xffff0000u);
      }
      return true;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      fsc[e] = 1.0f;
      fsh[e] = 0.0f;
    }
    return false;
  }
};

__device__ __forceinline__ bool load_film(const GnArgs& p, int n, int ch, float (&fsc)[8],
                                          float (&fsh)[8]) {
  GnFilm f;
  f.load(p, n, ch);
  return f.get(p, fsc, fsh);
}

// Pixel loop of a pass: lane pl visits pixels pl, pl + PLN, ... in groups of U whose 16-B
// loads (from each of the NL sources) are all issued before any is used; pixels past HW load
// pixel HW - 1 (a valid address) and reach body(px, ok, v0, v1) with ok false.
template <int PLN, int NL, int U, typename F>
__device__ __forceinline__ void gn_pixels(const uint16_t* const (&src)[NL], int C, int pl, int HW,
                                          F body) {
  for (int px0 = pl; px0 < HW; px0 += U * PLN) {
    int pxs[U];
    bool oks[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int px = px0 + u * PLN;
      oks[u] = px < HW;
      pxs[u] = oks[u] ? px : HW - 1;
    }
    uint4 v[NL][U];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int l = 0; l < NL; ++l)
        v[l][u] = *reinterpret_cast<const uint4*>(src[l] + (int64_t)pxs[u] * C);
#pragma unroll
    for (int u = 0; u < U; ++u) body(pxs[u], oks[u], v[0][u], v[NL - 1][u]);
  }
}

// Layout: one workgroup per (image n, 64-channel slab): 8 x PLN threads = PLN pixel lanes x
// 8 granules of 8 channels (16 B of bf16).
template <int PLN>
__global__ __launch_bounds__(8 * PLN) void gn_silu_fwd_kernel(const GnArgs p) {
  __shared__ float red[(PLN / 8) * 8 * 2];
  __shared__ float hs[16];
  const int n = blockIdx.y;
  const int c0 = blockIdx.x * kSlab;
  const int gq = threadIdx.x & 7;
  const int pl = threadIdx.x >> 3;
  const int ch = c0 + gq * 8;
  const int HW = p.HW;
  const uint16_t* xb = static_cast<const uint16_t*>(p.x) + (int64_t)n * HW * p.C + ch;

  // pass 1: mean
  float s[2] = {0.f, 0.f};
  const uint16_t* const xsrc[1] = {xb};
  gn_pixels<PLN, 1, kGnUnrollFwd>(xsrc, p.C, pl, HW, [&](int, bool ok, uint4 xv, uint4) {
    float f[8];
    unpack8(xv, f);
    if (ok) {
      s[0] += (f[0] + f[1]) + (f[2] + f[3]);
      s[1] += (f[4] + f[5]) + (f[6] + f[7]);
    }
  });
  slab_reduce<2, PLN>(s, red);
  if ((threadIdx.x >> 3) == 0) {
    hs[2 * gq] = s[0];
    hs[2 * gq + 1] = s[1];
  }
  __syncthreads();
  const float inv_cnt = 1.0f / (float)((int64_t)HW * p.cpg);
  const float mu[2] = {group_sum(hs, 2 * gq, p.cpg) * inv_cnt,
                       group_sum(hs, 2 * gq + 1, p.cpg) * inv_cnt};
  __syncthreads();

  // pass 2: biased variance around the mean
  float q[2] = {0.f, 0.f};
  gn_pixels<PLN, 1, kGnUnrollFwd>(xsrc, p.C, pl, HW, [&](int, bool ok, uint4 xv, uint4) {
    float f[8];
    unpack8(xv, f);
    if (ok) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = f[e] - mu[e >> 2];
        q[e >> 2] += d * d;
      }
    }
  });
  slab_reduce<2, PLN>(q, red);
  if ((threadIdx.x >> 3) == 0) {
    hs[2 * gq] = q[0];
    hs[2 * gq + 1] = q[1];
  }
  __syncthreads();
  float rs[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const float var = group_sum(hs, 2 * gq + h, p.cpg) * inv_cnt;
    rs[h] = 1.0f / sqrtf(var + p.eps);
  }
  // statistics out: one writer per group
  if (pl == 0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int cc = ch + 4 * h;
      if (cc % p.cpg == 0) {
        const int g = cc / p.cpg;
        p.mean[n * p.G + g] = mu[h];
        p.rstd[n * p.G + g] = rs[h];
      }
    }
  }

  // pass 3: normalise, affine, FiLM, SiLU, bf16
  float a[8], b[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    a[e] = p.gamma[ch + e];
    b[e] = p.beta[ch + e];
  }
  float fsc[8], fsh[8];
  const bool film = load_film(p, n, ch, fsc, fsh);
  uint16_t* ob = static_cast<uint16_t*>(p.out) + (int64_t)n * HW * p.C + ch;
  gn_pixels<PLN, 1, kGnUnrollFwd>(xsrc, p.C, pl, HW, [&](int px, bool ok, uint4 xv, uint4) {
    float f[8];
    unpack8(xv, f);
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      float z[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int ee = e + k;
        float v = (f[ee] - mu[ee >> 2]) * rs[ee >> 2] * a[ee] + b[ee];
        if (film) v = fsc[ee] * v + fsh[ee];
        z[k] = v * sigmoid_hw(v);
      }
      o[e >> 1] = f32_to_bf16_bits(z[0]) | (f32_to_bf16_bits(z[1]) << 16);
    }
    if (ok) st_nt16(ob + (int64_t)px * p.C, uint4{o[0], o[1], o[2], o[3]});
  });
}

// Backward. With zp = film? fs*z + fb : z (z = GN output), u = silu(zp):
//   g   = dout * sig(zp) * (1 + zp * (1 - sig(zp)))        (d u / d zp)
//   dfs = sum_hw g * z,  dfb = sum_hw g;   gz = film? g * fs : g
//   dgamma += sum gz * xhat, dbeta += sum gz;   gxh = gz * gamma
//   dx = rstd * (gxh - mean_grp(gxh) - xhat * mean_grp(gxh * xhat))
template <int PLN>
__global__ __launch_bounds__(8 * PLN) void gn_silu_bwd_kernel(const GnArgs p) {
  __shared__ float red[(PLN / 8) * 8 * 32];
  __shared__ float hs[2][16];
  const int n = blockIdx.y;
  const int c0 = blockIdx.x * kSlab;
  const int gq = threadIdx.x & 7;
  const int pl = threadIdx.x >> 3;
  const int ch = c0 + gq * 8;
  const int HW = p.HW;
  const int64_t base = (int64_t)n * HW * p.C + ch;

  float mu[2], rs[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int g = (ch + 4 * h) / p.cpg;
    mu[h] = p.mean[n * p.G + g];
    rs[h] = p.rstd[n * p.G + g];
  }
  float gm[8], bt[8], fsc[8], fsh[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    gm[e] = p.gamma[ch + e];
    bt[e] = p.beta[ch + e];
  }
  load_film(p, n, ch, fsc, fsh);

  // pass 1: per-channel sums of gz, gz*xhat, g*z, g
  float acc[4][8];
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[k][e] = 0.f;
  const uint16_t* const srcs[2] = {static_cast<const uint16_t*>(p.x) + base, p.dout + base};
  gn_pixels<PLN, 2, kGnUnrollBwd>(srcs, p.C, pl, HW, [&](int, bool ok, uint4 xv, uint4 dv) {
    float f[8], d[8];
    unpack8(xv, f);
    unpack8(dv, d);
    if (ok) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float xh = (f[e] - mu[e >> 2]) * rs[e >> 2];
        const float z = xh * gm[e] + bt[e];
        const float zp = fsc[e] * z + fsh[e];
        const float sg = sigmoid_hw(zp);
        const float g = d[e] * (sg * (1.0f + zp * (1.0f - sg)));
        const float gz = g * fsc[e];
        acc[0][e] += gz;
        acc[1][e] += gz * xh;
        acc[2][e] += g * z;
        acc[3][e] += g;
      }
    }
  });
  // reduce the 32 per-channel sums over pixel lanes
  {
    float* v = &acc[0][0];
    float tmp[32];
#pragma unroll
    for (int k = 0; k < 32; ++k) tmp[k] = v[k];
    slab_reduce<32, PLN>(tmp, red);
#pragma unroll
    for (int k = 0; k < 32; ++k) v[k] = tmp[k];
  }
  // per-image channel partials for dgamma/dbeta and the FiLM gradients
  if (pl == 0) {
    const int64_t nc = (int64_t)p.N * p.C;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int64_t o = (int64_t)n * p.C + ch + e;
      p.part[0 * nc + o] = acc[1][e];  // dgamma partial
      p.part[1 * nc + o] = acc[0][e];  // dbeta partial
      if (p.dfs) {                      // FiLM gradients are per image: final here
        p.dfs[o] = acc[2][e];
        p.dfb[o] = acc[3][e];
      } else if (p.dwb) {
        const int64_t ob = (int64_t)n * 2 * p.C + ch + e;
        p.dwb[ob] = (uint16_t)f32_to_bf16_bits(acc[2][e]);
        p.dwb[ob + p.C] = (uint16_t)f32_to_bf16_bits(acc[3][e]);
      }
    }
    // group sums of gxh = gz*gamma and gxh*xhat, per 4-channel half
    float h1[2] = {0.f, 0.f}, h2[2] = {0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      h1[e >> 2] += acc[0][e] * gm[e];
      h2[e >> 2] += acc[1][e] * gm[e];
    }
    hs[0][2 * gq] = h1[0];
    hs[0][2 * gq + 1] = h1[1];
    hs[1][2 * gq] = h2[0];
    hs[1][2 * gq + 1] = h2[1];
  }
  __syncthreads();
  const float inv_cnt = 1.0f / (float)((int64_t)HW * p.cpg);
  float m1[2], m2[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    m1[h] = group_sum(hs[0], 2 * gq + h, p.cpg) * inv_cnt;
    m2[h] = group_sum(hs[1], 2 * gq + h, p.cpg) * inv_cnt;
  }

  // pass 2: dx
  gn_pixels<PLN, 2, kGnUnrollBwd>(srcs, p.C, pl, HW, [&](int px, bool ok, uint4 xv, uint4 dv) {
    float f[8], d[8];
    unpack8(xv, f);
    unpack8(dv, d);
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      float r2[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int ee = e + k;
        const int h = ee >> 2;
        const float xh = (f[ee] - mu[h]) * rs[h];
        const float z = xh * gm[ee] + bt[ee];
        const float zp = fsc[ee] * z + fsh[ee];
        const float sg = sigmoid_hw(zp);
        const float g = d[ee] * (sg * (1.0f + zp * (1.0f - sg)));
        const float gxh = g * fsc[ee] * gm[ee];
        r2[k] = rs[h] * (gxh - m1[h] - xh * m2[h]);
      }
      o[e >> 1] = f32_to_bf16_bits(r2[0]) | (f32_to_bf16_bits(r2[1]) << 16);
    }
    if (ok) st_nt16(static_cast<uint16_t*>(p.out) + base + (int64_t)px * p.C, uint4{o[0], o[1], o[2], o[3]});
  });
}

// dgamma[c] = sum_n part[0][n][c], dbeta[c] = sum_n part[1][n][c]: 16 interleaved image
// slices (slice s sums images s, s + 16, ... in order, all its loads in flight at once), then
// a fixed pairwise tree over the slices (deterministic). One workgroup per 64 channels:
// 64 channel lanes x 16 image slices.
constexpr int kPrSlices = 16;
__global__ __launch_bounds__(64 * kPrSlices) void gn_param_reduce_kernel(
    const float* __restrict__ part, float* __restrict__ dgamma, float* __restrict__ dbeta, int N,
    int C) {
  __shared__ float red[2][kPrSlices][64];
  const int lane = threadIdx.x & 63;
  const int slice = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  const int64_t nc = (int64_t)N * C;
  float sg = 0.f, sb = 0.f;
  if (c < C) {
#pragma unroll 8
    for (int n = slice; n < N; n += kPrSlices) {
      sg += part[(int64_t)n * C + c];
      sb += part[nc + (int64_t)n * C + c];
    }
  }
  red[0][slice][lane] = sg;
  red[1][slice][lane] = sb;
  __syncthreads();
  if (slice < 2 && c < C) {
    float v[kPrSlices];
#pragma unroll
    for (int i = 0; i < kPrSlices; ++i) v[i] = red[slice][i][lane];
#pragma unroll
    for (int w = kPrSlices / 2; w >= 1; w /= 2)
#pragma unroll
      for (int i = 0; i < w; ++i) v[i] = v[i] + v[i + w];
    (slice == 0 ? dgamma : dbeta)[c] = v[0];
  }
}

// ---- chunked form (HW >= kChunkMinHW) ----
constexpr int kChPLN = 32;                 // pixel lanes per workgroup (256 threads)
constexpr int kChU = 4;                    // pixels per lane, all loads in flight
constexpr int kChunkPx = kChPLN * kChU;    // 128 pixels per workgroup
constexpr int kChunkMinHW = 256;
constexpr int kMaxChunks = 64;             // larger images run the one-launch form
static_assert(8 * kChPLN == 4 * kSlab, "backward apply: four chunk slices of 64 channels");

// Lane pl's pixels of the chunk starting at px0: px0 + pl + 32 u; pixels past HW load pixel
// HW - 1 (a valid address) with ok false.
template <int NL>
__device__ __forceinline__ void chunk_load(const uint8_t* const (&src)[NL],
                                           const int (&stride)[NL], int px0, int pl, int HW,
                                           uint4 (&v)[NL][kChU], bool (&ok)[kChU],
                                           int (&pxs)[kChU]) {
#pragma unroll
  for (int u = 0; u < kChU; ++u) {
    const int px = px0 + pl + u * kChPLN;
    ok[u] = px < HW;
    pxs[u] = ok[u] ? px : HW - 1;
  }
#pragma unroll
  for (int u = 0; u < kChU; ++u)
#pragma unroll
    for (int l = 0; l < NL; ++l)
      v[l][u] = *reinterpret_cast<const uint4*>(src[l] + (int64_t)pxs[u] * stride[l]);
}

// Sources of the chunk loop: the 8 channels of x at element offset off (one 16-B part in
// bf16, two in fp32), then, with kDout, the bf16 gradient of the output.
template <bool kF32, bool kDout>
struct GnSrc {
  static constexpr int kX = kF32 ? 2 : 1;
  static constexpr int kN = kX + (kDout ? 1 : 0);
  const uint8_t* src[kN];
  int stride[kN];  // bytes per pixel
  __device__ __forceinline__ GnSrc(const GnArgs& p, int64_t off) {
    constexpr int eb = kF32 ? 4 : 2;
    const uint8_t* xp = static_cast<const uint8_t*>(p.x) + off * eb;
#pragma unroll
    for (int k = 0; k < kX; ++k) {
      src[k] = xp + 16 * k;
      stride[k] = p.C * eb;
    }
    if (kDout) {
      src[kN - 1] = reinterpret_cast<const uint8_t*>(p.dout + off);
      stride[kN - 1] = p.C * 2;
    }
  }
};

// x of pixel u from the loaded parts
template <bool kF32, int NL, int U>
__device__ __forceinline__ void unpack_x(const uint4 (&v)[NL][U], int u, float (&f)[8]) {
  if constexpr (kF32) {
    const uint4 a = v[0][u], b = v[1][u];
    f[0] = __uint_as_float(a.x);
    f[1] = __uint_as_float(a.y);
    f[2] = __uint_as_float(a.z);
    f[3] = __uint_as_float(a.w);
    f[4] = __uint_as_float(b.x);
    f[5] = __uint_as_float(b.y);
    f[6] = __uint_as_float(b.z);
    f[7] = __uint_as_float(b.w);
  } else {
    unpack8(v[0][u], f);
  }
}

// This workgroup's number and the launch's workgroups
struct GnBlk {
  uint32_t blk = (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
  uint32_t count = gridDim.x * gridDim.y * gridDim.z;
};

// The producer-fused cast in one thread (GnArgs::q): the window scale, its reciprocal for the
// fast quotient, and the running amax of the bf16 values cast.
struct GnQ {
  float s = 1.0f, r = 0.0f;
  us2 acc = {0, 0};
  // (made before a kernel's pixels are loaded, set up after: see GnFilm)
  __device__ __forceinline__ explicit GnQ(const GnArgs& p) {
    if (p.q) s = *p.q_scale;
  }
  __device__ __forceinline__ void setup(const GnArgs& p) {
    if (p.q) r = quant_recip(s);
  }
  // the 8 bf16 values v of element offset off
  __device__ __forceinline__ void put(const GnArgs& p, int64_t off, uint4 v) {
    st_nt8(p.q + off, quant8_delayed(v, s, r));
    acc = absmax8(acc, v);
  }
  // the workgroup's amax partial (every thread; red: one u32 per wave)
  __device__ __forceinline__ void finish(const GnArgs& p, uint32_t* red, GnBlk b = GnBlk()) const {
    store_amax_partial(acc, red, p.q_part, p.q_count, b.blk, b.count);
  }
};

// A 16-B store of a slab of NG granules: nontemporal where the slab covers whole cache lines;
// the pieces of a line that thinner slabs write meet in the L2 (32-B pieces, forward and
// backward of 32 images of 64x64 x 128: nontemporal 42.0 / 53.6 us, plain 19.5 / 29.1; 64-B
// pieces of 64 images of 2048 pixels: 15.7 / 28.4 and 18.2 / 27.3, so the forward of those
// stores as whole lines do).
template <int NG>
__device__ __forceinline__ void gn_st16(void* dst, uint4 v) {
  if constexpr (NG == 8)
    st_nt16(dst, v);
  else
    *static_cast<uint4*>(dst) = v;
}

// dx of 8 channels at element offset off, in x's type; dx(e) gives channel e's value
template <bool kF32, int NG = 8, typename F>
__device__ __forceinline__ void store_dx(const GnArgs& p, int64_t off, F dx, GnQ& qo) {
  // with dx_add: dx + add as torch's gradient accumulation forms it (one fp32 add; in bf16 the
  // sum of the two bf16 gradients, rounded once more)
  const bool add = p.dx_add != nullptr;
  if constexpr (kF32) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = dx(e);
    if (add && p.dx_add_bf16) {
      float a[8];
      unpack8(*reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p.dx_add) + off), a);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += a[e];
    } else if (add) {
      const float* a = static_cast<const float*>(p.dx_add) + off;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint4 w = *reinterpret_cast<const uint4*>(a + 4 * h);
        v[4 * h] += __uint_as_float(w.x);
        v[4 * h + 1] += __uint_as_float(w.y);
        v[4 * h + 2] += __uint_as_float(w.z);
        v[4 * h + 3] += __uint_as_float(w.w);
      }
    }
    float* d = static_cast<float*>(p.out) + off;
#pragma unroll
    for (int h = 0; h < 2; ++h)
      gn_st16<NG>(d + 4 * h, uint4{__float_as_uint(v[4 * h]), __float_as_uint(v[4 * h + 1]),
                                   __float_as_uint(v[4 * h + 2]), __float_as_uint(v[4 * h + 3])});
  } else {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = dx(e);
    if (add) {
      float a[8];
      unpack8(*reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p.dx_add) + off), a);
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const uint32_t w = pack_bf16x2(v[e], v[e + 1]);
        v[e] = __uint_as_float(w << 16) + a[e];
        v[e + 1] = __uint_as_float(w & 0xffff0000u) + a[e + 1];
      }
    }
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 8; e += 2) o[e >> 1] = pack_bf16x2(v[e], v[e + 1]);
    if (p.q)
      qo.put(p, off, uint4{o[0], o[1], o[2], o[3]});
    else
      gn_st16<NG>(static_cast<uint16_t*>(p.out) + off, uint4{o[0], o[1], o[2], o[3]});
  }
}

// fp32 x also stored rounded to bf16 (RNE), for a consumer that rounds it anyway (the residual
// block's 1x1 skip conv), so no separate cast pass reads x again
template <int NG = 8>
__device__ __forceinline__ uint4 store_x_bf16(const GnArgs& p, int64_t off, const float (&f)[8]) {
  uint32_t o[4];
#pragma unroll
  for (int e = 0; e < 8; e += 2) o[e >> 1] = pack_bf16x2(f[e], f[e + 1]);
  const uint4 w = uint4{o[0], o[1], o[2], o[3]};
  gn_st16<NG>(p.x_bf16 + off, w);
  return w;
}

// The workgroup's amax partial of the bf16 copy of x (every thread; red: one u32 per wave), for
// the current-scaling FP8 conv that quantizes that copy next
__device__ __forceinline__ void finish_xb_amax(const GnArgs& p, us2 acc, uint32_t* red,
                                               GnBlk b = GnBlk()) {
  store_amax_partial(acc, red, p.xb_part, nullptr, b.blk, b.count);
  // (its reader takes the whole room, of which the thin slabs use a part)
  if (threadIdx.x == 0)
    for (uint32_t i = b.blk + b.count; i < p.xb_room; i += b.count) p.xb_part[i] = 0;
}

// The channel constants of this thread's 8 channels (gamma, beta, FiLM) and, for the backward,
// their groups' mean and rstd: loaded before a kernel's pixels, looked at after (see GnFilm).
template <bool kFilm, bool kStats>
struct GnChan {
  uint4 g[2], b[2];
  GnFilm film;
  float mu[2], rs[2];
  __device__ __forceinline__ GnChan(const GnArgs& p, int n, int ch) {
    load8raw(p.gamma + ch, g);
    load8raw(p.beta + ch, b);
    if (kFilm) film.load(p, n, ch);
    if (kStats) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int gi = n * p.G + (ch + 4 * h) / p.cpg;
        mu[h] = p.mean[gi];
        rs[h] = p.rstd[gi];
      }
    }
  }
};

// The forward's per-channel affine of this thread's 8 channels: out = silu(x A + B) with
// A = rstd gamma and B = beta - mean A, both times the FiLM scale (plus its shift in B) --
// normalise, affine and FiLM in one fma per element.
template <bool kFilm>
__device__ __forceinline__ void fwd_affine(const GnArgs& p, const GnChan<kFilm, false>& k,
                                           const float (&mu)[2], const float (&rs)[2],
                                           float (&A)[8], float (&B)[8]) {
  float gm[8], bt[8], fsc[8], fsh[8];
  floats8(k.g, gm);
  floats8(k.b, bt);
  if (kFilm) k.film.get(p, fsc, fsh);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float a = rs[e >> 2] * gm[e];
    const float b = __builtin_fmaf(-mu[e >> 2], a, bt[e]);
    A[e] = kFilm ? fsc[e] * a : a;
    B[e] = kFilm ? __builtin_fmaf(fsc[e], b, fsh[e]) : b;
  }
}

// The same constants through LDS, for the bf16 forward at 16 pixels per lane without dropout: its
// 128 registers do not hold them through two reductions. Every thread loads those of one channel
// before its pixels (threads of equal channels the same values), put() stores them, and the affine
// reads 8 channels' back after the reductions' barriers.
template <bool kFilm, int NG>
struct GnChanLds {
  static constexpr int kFloats = 8 * NG * (kFilm ? 4 : 2);
  float g, b, s = 1.0f, h = 0.0f;
  int c;
  __device__ __forceinline__ GnChanLds(const GnArgs& p, int n, int c0) {
    c = threadIdx.x & (8 * NG - 1);
    const int ch = c0 + c;
    g = p.gamma[ch];
    b = p.beta[ch];
    if (kFilm) {
      if (p.fs) {
        s = p.fs[(int64_t)n * p.C + ch];
        h = p.fb[(int64_t)n * p.C + ch];
      } else {
        s = __uint_as_float((uint32_t)p.wb[(int64_t)n * 2 * p.C + ch] << 16);
        h = __uint_as_float((uint32_t)p.wb[(int64_t)n * 2 * p.C + p.C + ch] << 16);
      }
    }
  }
  __device__ __forceinline__ void put(const GnArgs& p, float* lds) const {
    lds[c] = g;
    lds[8 * NG + c] = b;
    if (kFilm) {
      // (the time projection's scale is bf16(w + 1))
      lds[16 * NG + c] = p.fs ? s : __uint_as_float(pack_bf16x2(s + 1.0f, 0.0f) << 16);
      lds[24 * NG + c] = h;
    }
  }
  static __device__ __forceinline__ void affine(const float* lds, const float (&mu)[2],
                                                const float (&rs)[2], float (&A)[8],
                                                float (&B)[8]) {
    const float* l = lds + 8 * (threadIdx.x & (NG - 1));
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float a = rs[e >> 2] * l[e];
      const float b = __builtin_fmaf(-mu[e >> 2], a, l[8 * NG + e]);
      A[e] = kFilm ? a * l[16 * NG + e] : a;
      B[e] = kFilm ? __builtin_fmaf(b, l[16 * NG + e], l[24 * NG + e]) : b;
    }
  }
};

// 8 outputs silu(f A + B) (dropout: kept ones times drop_scale, the rest 0), packed bf16
template <bool kDrop>
__device__ __forceinline__ uint4 fwd_out8(const float (&f)[8], const float (&A)[8],
                                          const float (&B)[8], uint4 mask, float drop_scale) {
  float z[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float t = __builtin_fmaf(f[e], A[e], B[e]);
    float o = t * sigmoid_hw(t);
    if (kDrop) o = o * drop_scale;
    z[e] = o;
  }
  const uint4 o = uint4{pack_bf16x2(z[0], z[1]), pack_bf16x2(z[2], z[3]), pack_bf16x2(z[4], z[5]),
                        pack_bf16x2(z[6], z[7])};
  return kDrop ? and4(o, mask) : o;
}

__device__ __forceinline__ int chunk_pixels(int HW, int chunk) {
  const int r = HW - chunk * kChunkPx;
  return r < kChunkPx ? r : kChunkPx;
}

// Forward, launch 1: grid (C / 64, N, chunks). cs[n][chunk][g] = (chunk mean, chunk sum of
// squared deviations from it) of group g.
template <bool kF32>
__global__ __launch_bounds__(8 * kChPLN) void gn_chunk_stats_kernel(const GnArgs p,
                                                                   float2* __restrict__ cs,
                                                                   int nchunk) {
  __shared__ float red[(kChPLN / 8) * 8 * 2];
  __shared__ float hs[16];
  const int n = blockIdx.y, chunk = blockIdx.z;
  const int c0 = blockIdx.x * kSlab;
  const int gq = threadIdx.x & 7;
  const int pl = threadIdx.x >> 3;
  const int ch = c0 + gq * 8;
  const GnSrc<kF32, false> in(p, (int64_t)n * p.HW * p.C + ch);
  uint4 v[in.kN][kChU];
  bool ok[kChU];
  int pxs[kChU];
  chunk_load(in.src, in.stride, chunk * kChunkPx, pl, p.HW, v, ok, pxs);
  float f[kChU][8];
#pragma unroll
  for (int u = 0; u < kChU; ++u) unpack_x<kF32>(v, u, f[u]);

  float sm[2] = {0.f, 0.f};
#pragma unroll
  for (int u = 0; u < kChU; ++u)
    if (ok[u]) {
      sm[0] += (f[u][0] + f[u][1]) + (f[u][2] + f[u][3]);
      sm[1] += (f[u][4] + f[u][5]) + (f[u][6] + f[u][7]);
    }
  slab_reduce<2, kChPLN>(sm, red);
  if (pl == 0) {
    hs[2 * gq] = sm[0];
    hs[2 * gq + 1] = sm[1];
  }
  __syncthreads();
  const float inv_cnt = 1.0f / (float)(chunk_pixels(p.HW, chunk) * p.cpg);
  const float mu[2] = {group_sum(hs, 2 * gq, p.cpg) * inv_cnt,
                       group_sum(hs, 2 * gq + 1, p.cpg) * inv_cnt};
  __syncthreads();
  float q[2] = {0.f, 0.f};
#pragma unroll
  for (int u = 0; u < kChU; ++u)
    if (ok[u]) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = f[u][e] - mu[e >> 2];
        q[e >> 2] += d * d;
      }
    }
  slab_reduce<2, kChPLN>(q, red);
  if (pl == 0) {
    hs[2 * gq] = q[0];
    hs[2 * gq + 1] = q[1];
  }
  __syncthreads();
  if (pl == 0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int cc = ch + 4 * h;
      if (cc % p.cpg == 0)
        cs[((int64_t)n * nchunk + chunk) * p.G + cc / p.cpg] =
            float2{mu[h], group_sum(hs, 2 * gq + h, p.cpg)};
    }
  }
}

// Forward, launch 2: merge the chunk statistics of the slab's groups in chunk order, then
// normalise, affine, FiLM, SiLU, bf16 for this workgroup's chunk. Chunk 0 writes mean/rstd.
template <bool kF32, bool kFilm, bool kDrop>
__global__ __launch_bounds__(8 * kChPLN) void gn_chunk_apply_kernel(const GnArgs p,
                                                                   const float2* __restrict__ cs,
                                                                   int nchunk) {
  __shared__ uint32_t qred[8 * kChPLN / 64];
  __shared__ float2 gstat[kSlab / 4];
  __shared__ float2 lcs[kMaxChunks * (kSlab / 4)];
  const int n = blockIdx.y, chunk = blockIdx.z;
  const int c0 = blockIdx.x * kSlab;
  const int gq = threadIdx.x & 7;
  const int pl = threadIdx.x >> 3;
  const int ch = c0 + gq * 8;
  const GnSrc<kF32, false> in(p, (int64_t)n * p.HW * p.C + ch);
  uint4 v[in.kN][kChU];
  bool ok[kChU];
  int pxs[kChU];
  chunk_load(in.src, in.stride, chunk * kChunkPx, pl, p.HW, v, ok, pxs);

  // the slab's chunk statistics, all loads in flight at once, then merged from LDS
  const int ngs = kSlab / p.cpg;
  const int g0 = c0 / p.cpg;
  for (int i = threadIdx.x; i < ngs * nchunk; i += 8 * kChPLN) {
    const int k = i / ngs;
    lcs[i] = cs[((int64_t)n * nchunk + k) * p.G + g0 + (i - k * ngs)];
  }
  __syncthreads();
  if ((int)threadIdx.x < ngs) {
    const int g = g0 + threadIdx.x;
    float na = 0.f, mean = 0.f, m2 = 0.f;
    for (int k = 0; k < nchunk; ++k) {
      const float2 b = lcs[k * ngs + threadIdx.x];
      const float nb = (float)(chunk_pixels(p.HW, k) * p.cpg);
      const float nt = na + nb;
      const float d = b.x - mean;
      const float wgt = nb / nt;
      mean += d * wgt;
      m2 += b.y + d * d * (na * wgt);
      na = nt;
    }
    const float rs = 1.0f / sqrtf(m2 / na + p.eps);
    gstat[threadIdx.x] = float2{mean, rs};
    if (chunk == 0) {
      p.mean[n * p.G + g] = mean;
      p.rstd[n * p.G + g] = rs;
    }
  }
  __syncthreads();
  float mu[2], rs[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const float2 st = gstat[(ch + 4 * h - c0) / p.cpg];
    mu[h] = st.x;
    rs[h] = st.y;
  }
  // The channel constants and the cast scale only here: held from before the pixels they cost 16 to
  // 24 registers and with FiLM a wave per SIMD (24 images of 64x64 x 128 with FiLM 17.8 us, so
  // 15.3).
  float A[8], B[8];
  fwd_affine<kFilm>(p, GnChan<kFilm, false>(p, n, ch), mu, rs, A, B);
  uint16_t* ob = static_cast<uint16_t*>(p.out) + (int64_t)n * p.HW * p.C + ch;
  const uint64_t seed = kDrop ? *p.drop_seed : 0;
  GnQ qo(p);
  qo.setup(p);
  us2 xacc = {0, 0};
#pragma unroll
  for (int u = 0; u < kChU; ++u) {
    float f[8];
    unpack_x<kF32>(v, u, f);
    const int64_t off = ((int64_t)n * p.HW + pxs[u]) * p.C + ch;
    if constexpr (kF32) {
      if (p.x_bf16 && ok[u]) xacc = absmax8(xacc, store_x_bf16(p, off, f));
    }
    const uint4 mk = kDrop ? drop_mask8(drop_z(seed, off), drop_keep2(p)) : uint4{};
    const uint4 o = fwd_out8<kDrop>(f, A, B, mk, p.drop_scale);
    if (ok[u]) {
      if (p.q)
        qo.put(p, off, o);
      else
        st_nt16(ob + (int64_t)pxs[u] * p.C, o);
    }
  }
  if (p.q) qo.finish(p, qred);
  if constexpr (kF32) {
    if (p.x_bf16 && p.xb_part) {
      __syncthreads();  // qred is reused
      finish_xb_amax(p, xacc, qred);
    }
  }
}

struct GnBwdSetup {
  float mu[2], rs[2], nmr[2], gm[8], bt[8], fsc[8], fsh[8], gC[8];  // nmr = -mu rs, gC = fs gm
};

// The backward terms of one pixel's 8 channels (see gn_silu_bwd_kernel): xhat, and g = dout
// times d silu(zp) / d zp at zp = fs (xhat gamma + beta) + fb (no FiLM: fs = 1, fb = 0).
template <bool kFilm>
__device__ __forceinline__ void bwd_terms(const float (&f)[8], const float (&d)[8],
                                          const GnBwdSetup& st, float (&xh)[8], float (&g)[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    xh[e] = __builtin_fmaf(f[e], st.rs[e >> 2], st.nmr[e >> 2]);
    const float z = __builtin_fmaf(xh[e], st.gm[e], st.bt[e]);
    const float zp = kFilm ? __builtin_fmaf(st.fsc[e], z, st.fsh[e]) : z;
    const float sg = sigmoid_hw(zp);
    g[e] = d[e] * (sg * __builtin_fmaf(zp, 1.0f - sg, 1.0f));
  }
}

// dout of 8 channels, masked and scaled by the forward's dropout; z: its hash input
template <bool kDrop>
__device__ __forceinline__ void bwd_dout(uint4 v, uint64_t z, const GnArgs& p, float (&d)[8]) {
  if (kDrop) v = and4(v, drop_mask8(z, drop_keep2(p)));
  unpack8(v, d);
  if (kDrop) {
#pragma unroll
    for (int e = 0; e < 8; ++e) d[e] = d[e] * p.drop_scale;
  }
}

template <bool kFilm>
__device__ __forceinline__ void gn_bwd_setup(const GnArgs& p, const GnChan<kFilm, true>& k,
                                             GnBwdSetup& st) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    st.mu[h] = k.mu[h];
    st.rs[h] = k.rs[h];
    st.nmr[h] = -st.mu[h] * st.rs[h];
  }
  floats8(k.g, st.gm);
  floats8(k.b, st.bt);
  if (kFilm) {
    k.film.get(p, st.fsc, st.fsh);
  } else {  // compile-time identity: the FiLM terms fold away
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      st.fsc[e] = 1.0f;
      st.fsh[e] = 0.0f;
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) st.gC[e] = kFilm ? st.fsc[e] * st.gm[e] : st.gm[e];
}

// Backward, launch 1: grid (C / 64, N, chunks). cp[chunk][n][c] = chunk sums of
// (gz, gz * xhat, g * z, g) of channel c. FiLM scale/shift, gamma and beta are constant per
// (image, channel), so all four follow from S1 = sum g and S2 = sum g * xhat:
// (fs S1, fs S2, gamma S2 + beta S1, S1); only those two sums are accumulated.
template <bool kFilm, bool kF32, bool kDrop>
__global__ __launch_bounds__(8 * kChPLN) void gn_chunk_bwd_sums_kernel(const GnArgs p,
                                                                      float4* __restrict__ cp) {
  constexpr int NS = 16;
  __shared__ float red[(kChPLN / 8) * 8 * NS];
  const int n = blockIdx.y, chunk = blockIdx.z;
  const int c0 = blockIdx.x * kSlab;
  const int gq = threadIdx.x & 7;
  const int pl = threadIdx.x >> 3;
  const int ch = c0 + gq * 8;
  const int64_t base = (int64_t)n * p.HW * p.C + ch;
  const uint64_t seed = kDrop ? *p.drop_seed : 0;
  const GnChan<kFilm, true> kc0(p, n, ch);  // (before the pixels only where the FiLM is formed)
  const GnSrc<kF32, true> in(p, base);
  uint4 v[in.kN][kChU];
  bool ok[kChU];
  int pxs[kChU];
  chunk_load(in.src, in.stride, chunk * kChunkPx, pl, p.HW, v, ok, pxs);
  const GnChan<kFilm, true> kc = kFilm ? kc0 : GnChan<kFilm, true>(p, n, ch);
  GnBwdSetup st;
  gn_bwd_setup<kFilm>(p, kc, st);
  float acc[NS];
#pragma unroll
  for (int k = 0; k < NS; ++k) acc[k] = 0.f;
#pragma unroll
  for (int u = 0; u < kChU; ++u) {
    float f[8], d[8], xh[8], g[8];
    unpack_x<kF32>(v, u, f);
    bwd_dout<kDrop>(v[in.kN - 1][u], kDrop ? drop_z(seed, base + (int64_t)pxs[u] * p.C) : 0, p, d);
    bwd_terms<kFilm>(f, d, st, xh, g);
    if (ok[u]) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        acc[e] += g[e];
        acc[8 + e] += g[e] * xh[e];
      }
    }
  }
  slab_reduce<NS, kChPLN>(acc, red);
  if (pl == 0) {
    float4* o = cp + ((int64_t)chunk * p.N + n) * p.C + ch;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float s1 = acc[e], s2 = acc[8 + e];
      o[e] = kFilm ? float4{st.fsc[e] * s1, st.fsc[e] * s2, st.gm[e] * s2 + st.bt[e] * s1, s1}
                   : float4{s1, s2, 0.f, 0.f};
    }
  }
}

// Backward, launch 2: per-channel totals over the chunks in order, group means of
// gxh = gz * gamma and gxh * xhat, then dx for this chunk. Chunk 0 writes the per-image
// channel partials of dgamma/dbeta and the FiLM gradients.
template <bool kFilm, bool kF32, bool kDrop>
__global__ __launch_bounds__(8 * kChPLN) void gn_chunk_bwd_apply_kernel(const GnArgs p,
                                                                       const float4* __restrict__ cp,
                                                                       int nchunk) {
  __shared__ uint32_t qred[8 * kChPLN / 64];
  __shared__ float4 tot[kSlab];
  __shared__ float4 slice[4][kSlab];
  __shared__ float hs[2][16];
  const int n = blockIdx.y, chunk = blockIdx.z;
  const int c0 = blockIdx.x * kSlab;
  const int gq = threadIdx.x & 7;
  const int pl = threadIdx.x >> 3;
  const int ch = c0 + gq * 8;
  const int64_t base = (int64_t)n * p.HW * p.C + ch;
  const uint64_t seed = kDrop ? *p.drop_seed : 0;
  const GnChan<kFilm, true> kc0(p, n, ch);  // (before the pixels only where the FiLM is formed)
  GnQ qo(p);
  const GnSrc<kF32, true> in(p, base);
  uint4 v[in.kN][kChU];
  bool ok[kChU];
  int pxs[kChU];
  chunk_load(in.src, in.stride, chunk * kChunkPx, pl, p.HW, v, ok, pxs);
  const GnChan<kFilm, true> kc = kFilm ? kc0 : GnChan<kFilm, true>(p, n, ch);
  GnBwdSetup st;
  gn_bwd_setup<kFilm>(p, kc, st);
  qo.setup(p);

  // channel totals over the chunks: four interleaved slices of chunks per channel (loads
  // in flight together), then the slices in order (deterministic)
  {
    const int cl = threadIdx.x & (kSlab - 1), sl = threadIdx.x >> 6;
    const float4* q = cp + (int64_t)n * p.C + c0 + cl;
    const int64_t stride = (int64_t)p.N * p.C;
    float4 t = float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int k = sl; k < nchunk; k += 4) {
      const float4 b = q[k * stride];
      t.x += b.x;
      t.y += b.y;
      t.z += b.z;
      t.w += b.w;
    }
    slice[sl][cl] = t;
  }
  __syncthreads();
  if (threadIdx.x < kSlab) {
    const int c = c0 + threadIdx.x;
    float4 t = slice[0][threadIdx.x];
#pragma unroll
    for (int sl = 1; sl < 4; ++sl) {
      const float4 b = slice[sl][threadIdx.x];
      t.x += b.x;
      t.y += b.y;
      t.z += b.z;
      t.w += b.w;
    }
    tot[threadIdx.x] = t;
    if (chunk == 0) {
      const int64_t nc = (int64_t)p.N * p.C;
      const int64_t o = (int64_t)n * p.C + c;
      p.part[o] = t.y;       // dgamma partial
      p.part[nc + o] = t.x;  // dbeta partial
      if (p.dfs) {
        p.dfs[o] = t.z;
        p.dfb[o] = t.w;
      } else if (p.dwb) {
        const int64_t ob = (int64_t)n * 2 * p.C + c;
        p.dwb[ob] = (uint16_t)f32_to_bf16_bits(t.z);
        p.dwb[ob + p.C] = (uint16_t)f32_to_bf16_bits(t.w);
      }
    }
  }
  __syncthreads();
  if (pl == 0) {
    float h1[2] = {0.f, 0.f}, h2[2] = {0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float4 t = tot[gq * 8 + e];
      h1[e >> 2] += t.x * st.gm[e];
      h2[e >> 2] += t.y * st.gm[e];
    }
    hs[0][2 * gq] = h1[0];
    hs[0][2 * gq + 1] = h1[1];
    hs[1][2 * gq] = h2[0];
    hs[1][2 * gq + 1] = h2[1];
  }
  __syncthreads();
  const float inv_cnt = 1.0f / (float)((int64_t)p.HW * p.cpg);
  float m1[2], m2[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    m1[h] = group_sum(hs[0], 2 * gq + h, p.cpg) * inv_cnt;
    m2[h] = group_sum(hs[1], 2 * gq + h, p.cpg) * inv_cnt;
  }
#pragma unroll
  for (int u = 0; u < kChU; ++u) {
    float f[8], d[8], xh[8], g[8];
    unpack_x<kF32>(v, u, f);
    bwd_dout<kDrop>(v[in.kN - 1][u], kDrop ? drop_z(seed, base + (int64_t)pxs[u] * p.C) : 0, p, d);
    bwd_terms<kFilm>(f, d, st, xh, g);
    auto dx = [&](int e) __attribute__((always_inline)) {
      const int h = e >> 2;
      return st.rs[h] * __builtin_fmaf(-xh[e], m2[h], g[e] * st.gC[e] - m1[h]);
    };
    if (ok[u]) store_dx<kF32>(p, base + (int64_t)pxs[u] * p.C, dx, qo);
  }
  if (p.q) qo.finish(p, qred);
}

// ---- resident form (HW <= kResMaxHW: the 32x32, 16x16, 8x8 and 4x4 levels; up to four times
// that on slabs of NG = 4 or 2 granules in the launches that gn_res_shape names): one workgroup
// per (image, slab) of PLN pixel lanes x NG granules holds all of the slab's pixels in registers
// (U per lane, packed as loaded), so the forward and the backward each read their inputs once and
// write their outputs once; every pass unpacks from those registers ----
constexpr int kResMaxHW = 1024;

// A workgroup's image and slab of 8 NG channels. 64-channel slabs: grid (C / 64, N). Thinner ones
// take part of every cache line of an image, so the workgroups of one image go to one XCD (its
// L2 then reads and writes each line once): grid 8 ceil(slabs / 8), block b on XCD b mod 8,
// which has a contiguous range of the slabs in image order.
template <int NG>
struct GnSlab {
  int n, c0;
  uint32_t idx, total;
  __device__ __forceinline__ explicit GnSlab(const GnArgs& p) {
    if constexpr (NG == 8) {
      n = blockIdx.y;
      c0 = blockIdx.x * kSlab;
      idx = total = 0;
    } else {
      const uint32_t per_image = p.C / (8 * NG);
      total = per_image * p.N;
      idx = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
      n = (int)(idx / per_image);
      c0 = (int)(idx - n * per_image) * 8 * NG;
    }
  }
  __device__ __forceinline__ bool live() const { return NG == 8 || idx < total; }
  __device__ __forceinline__ GnBlk blk() const {
    GnBlk b;
    if (NG != 8) {
      b.blk = idx;
      b.count = total;
    }
    return b;
  }
};

// Whether a lane's u-th pixel lies past the image in every lane (workgroup-uniform): its turn in
// a pass is left out (in the backward's first pass of 16 pixels per lane four at a time: a branch at
// each costs a full image 2 % of the backward). All of them are loaded (the ones past the end load
// the last pixel again, from the L1), so that every load is in flight before the first is waited for.
template <int PLN>
__device__ __forceinline__ bool res_past(const GnArgs& p, int u) {
  return u > 0 && u * PLN >= p.HW;
}

// v unchanged, but opaque to the optimiser (no value numbering across this point)
__device__ __forceinline__ void opaque_u4(uint4& v) {
  asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w));
}

// Lane pl's pixels pl + PLN u; pixels past HW load pixel HW - 1 (a valid address) with ok false.
// kLate: the last source's last kLate pixels are left to the caller.
template <int NL, int PLN, int U, int kLate = 0>
__device__ __forceinline__ void res_load(const uint8_t* const (&src)[NL], const int (&stride)[NL],
                                         int pl, int HW, uint4 (&v)[NL][U], bool (&ok)[U],
                                         int (&pxs)[U]) {
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int px = pl + u * PLN;
    ok[u] = px < HW;
    pxs[u] = ok[u] ? px : HW - 1;
  }
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int l = 0; l < NL; ++l)
      if (l < NL - 1 || u < U - kLate)
        v[l][u] = *reinterpret_cast<const uint4*>(src[l] + (int64_t)pxs[u] * stride[l]);
}

// Two-source x (GnArgs::cat_a / cat_h) of channels ch .. ch + 7 (all of them from one source:
// cat_ca is a multiple of the slab), lane pl's pixels pl + PLN u as res_load's. kF32: x as
// fp32 bits in v[0] (channels 0-3) and v[1] (4-7), bf16 sources widened; else bf16 in v[0]
// (cat_h bf16). kDout: dout of the pixel in v[NL - 1].
template <int NL, int PLN, int U, bool kF32, bool kDout>
__device__ __forceinline__ void cat_load(const GnArgs& p, int n, int ch, int pl, uint4 (&v)[NL][U],
                                         bool (&ok)[U], int (&pxs)[U]) {
  static_assert(NL == (kF32 ? 2 : 1) + (kDout ? 1 : 0), "x parts and dout");
  const int W = p.cat_w, wl = W >> 1, ca = p.cat_ca;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int px = pl + PLN * u;
    ok[u] = px < p.HW;
    pxs[u] = ok[u] ? px : p.HW - 1;
  }
  auto widen = [&](int u) __attribute__((always_inline)) {
    if constexpr (kF32) {
      const uint4 b = v[0][u];
      v[0][u] = uint4{b.x << 16, b.x & 0xffff0000u, b.y << 16, b.y & 0xffff0000u};
      v[1][u] = uint4{b.z << 16, b.z & 0xffff0000u, b.w << 16, b.w & 0xffff0000u};
    }
  };
  if (ch < ca) {
    const uint16_t* a = p.cat_a + (int64_t)n * (p.HW >> 2) * ca + ch;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int y = pxs[u] / W, x = pxs[u] - y * W;
      v[0][u] = *reinterpret_cast<const uint4*>(a + ((y >> 1) * wl + (x >> 1)) * ca);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) widen(u);
  } else {
    const int chh = p.C - ca;
    const int64_t off = (int64_t)n * p.HW * chh + (ch - ca);
    bool f32 = false;
    if constexpr (kF32) f32 = p.cat_hf != 0;
    if (f32) {
      const float* h = static_cast<const float*>(static_cast<const void*>(p.cat_h)) + off;
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int k = 0; k < (kF32 ? 2 : 1); ++k)
          v[k][u] = *reinterpret_cast<const uint4*>(h + (int64_t)pxs[u] * chh + 4 * k);
    } else {
      const uint16_t* h = p.cat_h + off;
#pragma unroll
      for (int u = 0; u < U; ++u) v[0][u] = *reinterpret_cast<const uint4*>(h + (int64_t)pxs[u] * chh);
#pragma unroll
      for (int u = 0; u < U; ++u) widen(u);
    }
  }
  if constexpr (kDout) {
    const uint16_t* d = p.dout + (int64_t)n * p.HW * p.C + ch;
#pragma unroll
    for (int u = 0; u < U; ++u)
      v[NL - 1][u] = *reinterpret_cast<const uint4*>(d + (int64_t)pxs[u] * p.C);
  }
}

// Each pass unpacks x from the packed registers again and the pixel numbers are formed again at
// the end, so that at 16 pixels per lane of bf16 x two workgroups fit a CU (128 registers) and
// one's loads run under the other's arithmetic: the two-source form at 32x32 x 512 (2048
// workgroups) 111 -> 94 us. With dropout the masks hashed under the loads take that room instead
// (256 workgroups 18.4 us; with two per CU and the hash at the end a tenth more).
template <int PLN, int U, bool kFilm, bool kF32, bool kDrop, bool kCat = false, int NG = 8>
__global__ __launch_bounds__(NG * PLN, U >= 16 && !kF32 && !kDrop ? 4 : 1) void gn_res_fwd_kernel(const GnArgs p) {
  static_assert(!kCat || NG == 8, "64-channel slabs");
  static_assert(!kCat || PLN * U == 1024 || (kF32 && PLN * U == 256), "32x32 or 16x16 images");
  __shared__ uint32_t qred[NG * PLN / 64];
  __shared__ float red[(NG * PLN / 64) * NG * 2];
  __shared__ float hs[16];
  GnSlab<NG> sl(p);
  if (!sl.live()) return;  // (workgroup-uniform)
  const int n = sl.n;
  const int gq = threadIdx.x & (NG - 1);
  const int pl = threadIdx.x / NG;
  const int ch = sl.c0 + gq * 8;
  constexpr bool kChanLds = U >= 16 && !kF32 && !kDrop;  // (the instances held to 128 registers)
  using ChanLds = GnChanLds<kFilm, NG>;
  __shared__ __attribute__((aligned(16))) float chan[kChanLds ? ChanLds::kFloats : 4];
  using Chan = std::conditional_t<kChanLds, ChanLds, GnChan<kFilm, false>>;
  // The channel constants are loaded before the pixels where there is something to do with the
  // time (the FiLM's forming, the dropout hash), else behind them: 128 images of 16x16 x 512 fp32
  // 17.7 us before, 17.2 behind; bf16 with FiLM and dropout 16.3 and 17.4.
  constexpr bool kChanFirst = kFilm || kDrop;
  const Chan kc0(p, n, kChanLds ? sl.c0 : ch);
  GnQ qo(p);
  const uint64_t seed = kDrop ? *p.drop_seed : 0;
  const GnSrc<kF32, false> in(p, (int64_t)n * p.HW * p.C + ch);
  uint4 v[in.kN][U];
  bool ok[U];
  int pxs[U];
  if constexpr (kCat)
    cat_load<in.kN, PLN, U, kF32, false>(p, n, ch, pl, v, ok, pxs);
  else
    res_load<in.kN, PLN, U>(in.src, in.stride, pl, p.HW, v, ok, pxs);
  const Chan kc = kChanFirst ? kc0 : Chan(p, n, kChanLds ? sl.c0 : ch);
  if constexpr (kCat && !kF32) {
    // the bf16 copy of the concatenation is the loaded values themselves
    if (p.x_bf16) {
      us2 xacc = {0, 0};
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (ok[u]) {
          st_nt16(p.x_bf16 + ((int64_t)n * p.HW + pxs[u]) * p.C + ch, v[0][u]);
          xacc = absmax8(xacc, v[0][u]);
        }
      if (p.xb_part) finish_xb_amax(p, xacc, qred, sl.blk());
    }
  } else if constexpr (kF32) {
    if (p.x_bf16) {
      us2 xacc = {0, 0};
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (ok[u]) {
          float f[8];
          unpack_x<kF32>(v, u, f);
          xacc = absmax8(xacc, store_x_bf16<NG>(p, ((int64_t)n * p.HW + pxs[u]) * p.C + ch, f));
        }
      if (p.xb_part) finish_xb_amax(p, xacc, qred, sl.blk());
    }
  }
  // the dropout masks, hashed while the loads are in flight (beside 128 registers of fp32 x, and
  // at four pixels per lane, where they cost a wave per SIMD: at their use)
  constexpr bool kEarly = kDrop && U >= 8 && !(kF32 && U >= 16);
  const uint64_t z0 = kDrop ? drop_z(seed, ((int64_t)n * p.HW + pl) * p.C + ch) : 0;
  const uint64_t zs = (uint64_t)(PLN * p.C / 4) * kDropGolden;  // per pixel of the lane
  auto mask_of = [&](int u) __attribute__((always_inline)) {
    return kDrop ? drop_mask8(z0 + (uint64_t)u * zs, drop_keep2(p)) : uint4{};
  };
  uint4 mask[kEarly ? U : 1];
  if constexpr (kEarly) {
    // (straight through where most pixels are there: in pieces the hash takes 128 images of 32x32 x
    // 128 from 18.3 us to 18.9; left out past the image it takes 16 of 20x20 x 256 from 11.2 to 9.5)
    if (U < 16 || p.HW > 12 * PLN) {
#pragma unroll
      for (int u = 0; u < U; ++u) mask[u] = mask_of(u);
    } else {
#pragma unroll
      for (int u0 = 0; u0 < 12; u0 += 4) {
        if (res_past<PLN>(p, u0)) continue;
#pragma unroll
        for (int u = u0; u < u0 + 4; ++u) mask[kEarly && U >= 16 ? u : 0] = mask_of(u);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (kChanLds) kc.put(p, chan);
  float sm[2] = {0.f, 0.f};
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (ok[u]) {
      float f[8];
      unpack_x<kF32>(v, u, f);
      sm[0] += (f[0] + f[1]) + (f[2] + f[3]);
      sm[1] += (f[4] + f[5]) + (f[6] + f[7]);
    }
  slab_reduce<2, PLN, NG>(sm, red);
  if (pl == 0) {
    hs[2 * gq] = sm[0];
    hs[2 * gq + 1] = sm[1];
  }
  __syncthreads();
  const float inv_cnt = 1.0f / (float)(p.HW * p.cpg);
  const float mu[2] = {group_sum(hs, 2 * gq, p.cpg) * inv_cnt,
                       group_sum(hs, 2 * gq + 1, p.cpg) * inv_cnt};
  __syncthreads();
  // with the masks held too, the unpacked values do not fit beside the packed ones: each pass
  // unpacks again (hidden from the compiler)
  auto reopen = [&](int u) __attribute__((always_inline)) {
    if constexpr (U >= 16 && !kF32) {
#pragma unroll
      for (int l = 0; l < in.kN; ++l) opaque_u4(v[l][u]);
    }
  };
  float q[2] = {0.f, 0.f};
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (ok[u]) {
      reopen(u);
      float f[8];
      unpack_x<kF32>(v, u, f);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = f[e] - mu[e >> 2];
        q[e >> 2] += d * d;
      }
    }
  slab_reduce<2, PLN, NG>(q, red);
  if (pl == 0) {
    hs[2 * gq] = q[0];
    hs[2 * gq + 1] = q[1];
  }
  __syncthreads();
  float rs[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) rs[h] = 1.0f / sqrtf(group_sum(hs, 2 * gq + h, p.cpg) * inv_cnt + p.eps);
  if (pl == 0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int cc = ch + 4 * h;
      if (cc % p.cpg == 0) {
        p.mean[n * p.G + cc / p.cpg] = mu[h];
        p.rstd[n * p.G + cc / p.cpg] = rs[h];
      }
    }
  }
  float A[8], B[8];
  if constexpr (kChanLds)
    ChanLds::affine(chan, mu, rs, A, B);
  else
    fwd_affine<kFilm>(p, kc, mu, rs, A, B);
  uint16_t* ob = static_cast<uint16_t*>(p.out) + (int64_t)n * p.HW * p.C + ch;
  qo.setup(p);
  // (the pixel numbers formed again, not kept across the reductions)
  int pl2 = pl;
  asm volatile("" : "+v"(pl2));
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (U >= 16 && !kCat && res_past<PLN>(p, u)) continue;
    reopen(u);
    const int px = pl2 + u * PLN;
    if (px < p.HW) {
      float f[8];
      unpack_x<kF32>(v, u, f);
      const uint4 o = fwd_out8<kDrop>(f, A, B, kEarly ? mask[kEarly ? u : 0] : mask_of(u),
                                      p.drop_scale);
      if (p.q)
        qo.put(p, ((int64_t)n * p.HW + px) * p.C + ch, o);
      else
        gn_st16<kF32 || NG != 4 ? NG : 8>(ob + (int64_t)px * p.C, o);
    }
    if constexpr (U >= 16) __builtin_amdgcn_sched_barrier(0);
  }
  if (p.q) qo.finish(p, qred, sl.blk());
}

// The backward keeps x in registers (packed) and the fp32 g of every pixel, formed in the first
// pass as the loads arrive: the sigmoid's exp2 and reciprocal, which issue at a quarter rate,
// and the dropout hash are its largest costs and run once. At 16 pixels per lane, whose x and
// g take 192 registers (fp32 x: 256), the first few pixels' g lie in LDS. 128 images of 32x32 x
// 128 bf16 with FiLM and dropout: 41.2 us with g formed in both passes and dout in LDS, 30.1 so.
// At four pixels per lane many workgroups share a CU, so the bf16 form is held to four waves per
// SIMD: 128 images of 4x4 x 512 with FiLM 15.2 us at three, 11.4 at four (with g formed twice 11.4).
template <int U, bool kFilm, bool kF32, bool kCat>
constexpr int kGnResLdsG = U < 16 ? 0 : (kF32 ? 9 : (kCat ? 8 : (kFilm ? 6 : 3)));

//
// kAgain (below 16 pixels per lane): g formed again in the second pass, for fp32 x of 8 pixels per
// lane without FiLM and dropout where a CU holds several workgroups: what they load and store is
// then the longer part, and a second pass with arithmetic between its stores the shorter whole
// (images of 16x16, us, g kept / again: 128 x 256 channels 22.4 / 18.9, 64 x 512 22.6 / 21.1, 128 x
// 512 36.8 / 35.0; 16 x 256, one workgroup per CU, 9.9 / 11.6).
template <int PLN, int U, bool kFilm, bool kF32, bool kDrop, bool kCat = false, int NG = 8,
          bool kAgain = false>
__global__ __launch_bounds__(NG * PLN, U == 4 && !kF32 ? 4 : 1) void gn_res_bwd_kernel(const GnArgs p) {
  static_assert(!kAgain || (U < 16 && !kCat), "g is kept");
  static_assert(!kCat || (!kF32 && PLN == 64 && U == 16) || (kF32 && PLN == 32 && U == 8),
                "32x32 images (bf16 sources) or 16x16 (cat_h bf16 or fp32)");
  constexpr int kGL = kGnResLdsG<U, kFilm, kF32, kCat>;
  __shared__ __attribute__((aligned(16))) uint8_t gls[kGL ? kGL * 2 * NG * PLN * 16 : 16];
  __shared__ uint32_t qred[NG * PLN / 64];
  __shared__ float red[(NG * PLN / 64) * NG * 16];
  __shared__ float hs[2][16];
  // kCat: the pixel rows of one 2x2 window exchange
  constexpr int kXR = U >= 16 ? 2 : 4;
  __shared__ __attribute__((aligned(16))) float xch[kCat ? kXR * (PLN / 4) * 8 * 16 : 4];
  GnSlab<NG> sl(p);
  if (!sl.live()) return;  // (workgroup-uniform)
  const int n = sl.n;
  const int gq = threadIdx.x & (NG - 1);
  const int pl = threadIdx.x / NG;
  const int ch = sl.c0 + gq * 8;
  const int64_t base = (int64_t)n * p.HW * p.C + ch;
  const uint64_t seed = kDrop ? *p.drop_seed : 0;
  const GnChan<kFilm, true> kc(p, n, ch);
  GnQ qo(p);
  const GnSrc<kF32, true> in(p, base);
  constexpr int kStep = U >= 16 ? 4 : 1;  // pixels per look at res_past
  // fp32 x and dout of 16 pixels are 192 registers: the last four pixels' dout is loaded as the
  // first pixels' dies, or the first pass spills
  constexpr int kLate = kF32 && U >= 16 ? 4 : 0;
  uint4 v[in.kN][U];
  bool ok[U];
  int pxs[U];
  if constexpr (kCat) {
    cat_load<in.kN, PLN, U, kF32, true>(p, n, ch, pl, v, ok, pxs);
  } else {
    res_load<in.kN, PLN, U, kLate>(in.src, in.stride, pl, p.HW, v, ok, pxs);
  }
  GnBwdSetup st;
  gn_bwd_setup<kFilm>(p, kc, st);
  // per-channel S1 = sum g, S2 = sum g * xhat over the image (every lane gets the totals)
  float acc[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) acc[k] = 0.f;
  // hash input of the lane's first pixel, and its step from one pixel of the lane to the next
  const uint64_t z0 = kDrop ? drop_z(seed, base + (int64_t)pl * p.C) : 0;
  const uint64_t zs = (uint64_t)(PLN * p.C / 4) * kDropGolden;
  float gk[U][8];
  v4f* gl = reinterpret_cast<v4f*>(gls) + threadIdx.x;  // pixel u < kGL: entries 2u, 2u + 1
#pragma unroll
  for (int u0 = 0; u0 < U; u0 += kStep) {
    if (!kCat && res_past<PLN>(p, u0)) continue;
#pragma unroll
    for (int u = u0; u < u0 + kStep; ++u) {
      if (u > 0 && u <= kLate) {
        const int w = U - kLate + u - 1;
        v[in.kN - 1][w] = *reinterpret_cast<const uint4*>(in.src[in.kN - 1] +
                                                          (int64_t)pxs[w] * in.stride[in.kN - 1]);
      }
      float f[8], d[8], xh[8], g[8];
      unpack_x<kF32>(v, u, f);
      bwd_dout<kDrop>(v[in.kN - 1][u], z0 + (uint64_t)u * zs, p, d);
      bwd_terms<kFilm>(f, d, st, xh, g);
      if (ok[u]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          acc[e] += g[e];
          acc[8 + e] += g[e] * xh[e];
        }
      }
      if (kAgain) {
      } else if (u < kGL) {
        gl[(2 * u) * NG * PLN] = v4f{g[0], g[1], g[2], g[3]};
        gl[(2 * u + 1) * NG * PLN] = v4f{g[4], g[5], g[6], g[7]};
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) gk[u][e] = g[e];
      }
      // one pixel at a time: the packed inputs stay resident, each pixel's unpacked terms die
      // before the next pixel's are formed (else the interleaved pixels exceed the registers)
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if constexpr (U >= 16) {
    const GnChan<kFilm, true> kc2(p, n, ch);  // (again, not kept across the pixels)
    slab_reduce<16, PLN, NG>(acc, red);
    gn_bwd_setup<kFilm>(p, kc2, st);
  } else {
    slab_reduce<16, PLN, NG>(acc, red);
  }
  if (pl == 0) {
    const int64_t nc = (int64_t)p.N * p.C;
    float h1[2] = {0.f, 0.f}, h2[2] = {0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float s1 = acc[e], s2 = acc[8 + e];
      const float gz = st.fsc[e] * s1, gzx = st.fsc[e] * s2;  // sums of gz and gz * xhat
      const int64_t o = (int64_t)n * p.C + ch + e;
      p.part[o] = gzx;       // dgamma partial
      p.part[nc + o] = gz;   // dbeta partial
      if (kFilm) {
        const float gzs = st.gm[e] * s2 + st.bt[e] * s1;  // sum g * z
        if (p.dfs) {
          p.dfs[o] = gzs;
          p.dfb[o] = s1;
        } else if (p.dwb) {
          const int64_t ob = (int64_t)n * 2 * p.C + ch + e;
          p.dwb[ob] = (uint16_t)f32_to_bf16_bits(gzs);
          p.dwb[ob + p.C] = (uint16_t)f32_to_bf16_bits(s1);
        }
      }
      h1[e >> 2] += gz * st.gm[e];
      h2[e >> 2] += gzx * st.gm[e];
    }
    hs[0][2 * gq] = h1[0];
    hs[0][2 * gq + 1] = h1[1];
    hs[1][2 * gq] = h2[0];
    hs[1][2 * gq + 1] = h2[1];
  }
  __syncthreads();
  const float inv_cnt = 1.0f / (float)(p.HW * p.cpg);
  float m1[2], m2[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    m1[h] = group_sum(hs[0], 2 * gq + h, p.cpg) * inv_cnt;
    m2[h] = group_sum(hs[1], 2 * gq + h, p.cpg) * inv_cnt;
  }
  qo.setup(p);
  // pixel u's dx. The second pass unpacks x again from the packed registers: hidden from the
  // compiler, which would otherwise keep the first pass's unpacked values of every pixel alive
  // across the reduction (8 registers per pixel more)
  auto pixel_dx = [&](int u, float (&t)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int l = 0; l < (kAgain ? in.kN : in.kX); ++l) opaque_u4(v[l][u]);
    float f[8], ga[8];
    unpack_x<kF32>(v, u, f);
    if constexpr (kAgain) {
      float d[8], xh[8];
      bwd_dout<kDrop>(v[in.kN - 1][u], z0 + (uint64_t)u * zs, p, d);
      bwd_terms<kFilm>(f, d, st, xh, ga);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int h = e >> 2;
      const float xh = __builtin_fmaf(f[e], st.rs[h], st.nmr[h]);
      const float g = kAgain ? ga[e] : u < kGL ? gl[(2 * u + h) * NG * PLN][e & 3] : gk[u][e];
      t[e] = st.rs[h] * __builtin_fmaf(-xh, m2[h], g * st.gC[e] - m1[h]);
    }
  };
  if constexpr (kCat) {
    // The concatenation's fp32 gradient (plus the bf16 skip-path gradient, as autograd adds
    // it), split as the upsample-and-concatenate's backward does: cat_h's channels in
    // cat_h's type (bf16: rounded); cat_a's summed over each 2x2 window from zero in
    // row-major order, then rounded to bf16 (torch's upsample_nearest2d_backward). The
    // images are PLN / 2 wide, so pixel pl + PLN u is row 2u + pl / kW, column pl mod kW:
    // window (u, j) holds lanes 2j, 2j + 1 (row 2u) and 2j + kW, 2j + kW + 1 (row 2u + 1). The
    // odd lane's value comes by a shuffle (8 threads on), the lower row's two through LDS
    // (an exchange buffer), kXR pixels per exchange.
    constexpr int kW = PLN / 2;
    constexpr int kEnt = (kW / 2) * 8 * 16;  // floats per pixel row pair: (window, granule) x 16
    const bool in_a = ch < p.cat_ca;  // workgroup-uniform
    const bool even = (pl & 1) == 0;
    bool hf = false;
    if constexpr (kF32) hf = p.cat_hf != 0;
    // (the pixel numbers formed again, not kept across the reduction)
    int pl2 = pl;
    asm volatile("" : "+v"(pl2));
#pragma unroll
    for (int u0 = 0; u0 < U; u0 += kXR) {
      float t[kXR][8];
#pragma unroll
      for (int k = 0; k < kXR; ++k) {
        const int u = u0 + k;
        pixel_dx(u, t[k]);
        if (p.dx_add) {
          float a[8];
          unpack8(*reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p.dx_add) +
                                                  base + (int64_t)(pl2 + PLN * u) * p.C), a);
#pragma unroll
          for (int e = 0; e < 8; ++e) t[k][e] += a[e];
        }
        if (!in_a) {
          const int64_t o = ((int64_t)n * p.HW + pl2 + PLN * u) * (p.C - p.cat_ca) + (ch - p.cat_ca);
          if (hf) {
            float* gh = static_cast<float*>(p.cat_gh) + o;
#pragma unroll
            for (int q4 = 0; q4 < 2; ++q4)
              st_nt16(gh + 4 * q4, uint4{__float_as_uint(t[k][4 * q4]), __float_as_uint(t[k][4 * q4 + 1]),
                                         __float_as_uint(t[k][4 * q4 + 2]), __float_as_uint(t[k][4 * q4 + 3])});
          } else {
            uint32_t w[4];
#pragma unroll
            for (int e = 0; e < 8; e += 2) w[e >> 1] = pack_bf16x2(t[k][e], t[k][e + 1]);
            st_nt16(static_cast<uint16_t*>(p.cat_gh) + o, uint4{w[0], w[1], w[2], w[3]});
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (in_a) {
        __syncthreads();  // every thread has read the buffer
        float r[kXR][8];  // the odd neighbour's values (lane + 8: pixel lane pl + 1)
#pragma unroll
        for (int k = 0; k < kXR; ++k)
#pragma unroll
          for (int e = 0; e < 8; ++e) r[k][e] = __shfl_down(t[k][e], 8, 64);
        // row u0 + k, entry (window column j, granule gq): row 2u + 1's pair, 16 floats
        const int ent = (((pl % kW) >> 1) * 8 + gq) * 16;
        if (pl >= kW && even) {
#pragma unroll
          for (int k = 0; k < kXR; ++k) {
            float* e0 = xch + k * kEnt + ent;
#pragma unroll
            for (int q4 = 0; q4 < 2; ++q4) {
              *reinterpret_cast<v4f*>(e0 + 4 * q4) =
                  v4f{t[k][4 * q4], t[k][4 * q4 + 1], t[k][4 * q4 + 2], t[k][4 * q4 + 3]};
              *reinterpret_cast<v4f*>(e0 + 8 + 4 * q4) =
                  v4f{r[k][4 * q4], r[k][4 * q4 + 1], r[k][4 * q4 + 2], r[k][4 * q4 + 3]};
            }
          }
        }
        __syncthreads();
        if (pl < kW && even) {
#pragma unroll
          for (int k = 0; k < kXR; ++k) {
            const float* e0 = xch + k * kEnt + ent;
            float acc[8];
#pragma unroll
            for (int q4 = 0; q4 < 2; ++q4) {
              const v4f lo = *reinterpret_cast<const v4f*>(e0 + 4 * q4);
              const v4f hi = *reinterpret_cast<const v4f*>(e0 + 8 + 4 * q4);
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const int c = 4 * q4 + e;
                acc[c] = 0.0f;
                acc[c] += t[k][c];  // (2u, 2j)
                acc[c] += r[k][c];  // (2u, 2j + 1)
                acc[c] += lo[e];    // (2u + 1, 2j)
                acc[c] += hi[e];    // (2u + 1, 2j + 1)
              }
            }
            uint32_t w[4];
#pragma unroll
            for (int e = 0; e < 8; e += 2) w[e >> 1] = pack_bf16x2(acc[e], acc[e + 1]);
            const int wi = (u0 + k) * (kW / 2) + (pl >> 1);  // window row u0 + k, column pl / 2
            st_nt16(p.cat_ga + ((int64_t)n * (p.HW >> 2) + wi) * p.cat_ca + ch,
                    uint4{w[0], w[1], w[2], w[3]});
          }
        }
        // (the buffer's next writes come after the next pixels' first barrier)
      }
    }
  } else {
    // (the pixel numbers formed again, not kept across the reduction)
    int pl2 = pl;
    asm volatile("" : "+v"(pl2));
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (res_past<PLN>(p, u)) continue;
      float t[8];
      pixel_dx(u, t);
      auto dx = [&](int e) __attribute__((always_inline)) { return t[e]; };
      const int px = pl2 + u * PLN;
      if (px < p.HW) store_dx<kF32, NG>(p, base + (int64_t)px * p.C, dx, qo);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (p.q) qo.finish(p, qred, sl.blk());
}

// Resident-form geometry of a launch: pixels per lane and granules of a slab, or zeros where the
// resident form is not taken. Above kResMaxHW pixels a slab has 32 channels (up to 2048 pixels) or
// 16 (up to 4096), which have to be whole groups, and the chunked form is there too, whose time
// grows with the bytes alone. A thin slab's workgroup takes about the same time however few there
// are, so what decides is how full its rounds are: one workgroup per CU (two in the bf16 forward
// without dropout, whose loads then run under the other's arithmetic, but not before both are
// there). gn_thin_pays has the lines, each drawn so that no launch of 1025 to 4096 pixels at 128,
// 256 or 512 channels takes more than a few hundredths above the chunked form's time, on one set of
// buffers or on three in turn. us on three in turn, chunked -> resident, images of 128 channels:
//   2048 pixels, FiLM and dropout, forward / backward: 128 slabs 14.9 / 24.1 -> 16.8 / 28.5, 192
//     18.3 / 34.0 -> 17.6 / 30.2, 256 23.1 / 41.8 -> 19.9 / 35.5, 288 26.9 / 46.2 -> 33.1 / 59.2, 512
//     42.4 / 76.0 -> 35.9 / 73.8
//   4096 pixels: 256 slabs 21.3 / 41.1 -> 18.5 / 31.4 (with FiLM 23.2 / 37.7 -> 19.0 / 36.5, fp32 33.3 /
//     54.6 -> 30.0 / 45.9), 288 25.5 / 44.8 -> 24.4 / 53.7, 512 40.4 / 74.9 -> 39.8 / 65.2 (with FiLM
//     42.3 / 69.4 -> 40.4 / 74.2)
struct GnRes {
  int u, ng;
};
struct GnForm {
  bool bwd, f32, film, drop;
};
static bool gn_thin_pays(int64_t slabs, int64_t per_image, int HW, const GnForm& f) {
  const bool wide = HW <= 2 * kResMaxHW;
  const int64_t cus = num_cus(), k = ceil_div(slabs, cus);
  // share of the CUs that the last round of one workgroup per CU uses, in sixteenths
  const int64_t last = 16 * (slabs - (k - 1) * cus) / cus;
  if (f.bwd) {
    if (f.f32) return last >= 12 && (wide || k == 1);
    // (an image's lines in more than 16 pieces: 8 images of 64x64 x 512 40.9 -> 44.1 us)
    if (f.film) return wide ? k <= 2 && last >= 12 : k == 1 && last >= 14 && per_image <= 16;
    return k <= 2 && last >= 12;
  }
  // the fp32 forward's chunked form reads 8 B per element twice: its pixels count too
  if (f.f32 && k == 1)
    return last >= 12 && 16 * slabs * HW >= 9 * cus * (wide ? 2 : 4) * kResMaxHW;
  if (f.f32) return k == 2 && wide && !f.drop && last >= 12;
  if (!wide) return k == 1 && last >= 15 && HW >= 7 * kResMaxHW / 2;
  if (f.drop) return k == 1 && last >= 12;
  return k == 1 ? last >= 12 : (k > 2 || last >= 8);
}
static GnRes gn_res_shape(int N, int HW, int C, int G, const GnForm& f) {
  // The backward with an fp32 x holds 2 x 16 B of x per pixel in registers: that fits at 16
  // pixels per lane without FiLM and dropout (their per-channel terms and masks are the
  // registers that do not fit); with them, images above 256 pixels take the chunked form.
  if (HW > 256 && f.bwd && f.f32 && (f.film || f.drop)) return {0, 0};
  if (HW <= 128) return {4, 8};
  if (HW <= 256) return {8, 8};
  if (HW <= kResMaxHW) return {16, 8};
  const int ng = HW <= 2 * kResMaxHW ? 4 : 2;
  if (HW > 4 * kResMaxHW || (8 * ng) % (C / G) != 0) return {0, 0};
  const int64_t per_image = C / (8 * ng);
  return gn_thin_pays(per_image * N, per_image, HW, f) ? GnRes{16, ng} : GnRes{0, 0};
}

static int gn_chunks(int HW) {
  const int k = (int)ceil_div(HW, kChunkPx);
  return HW >= kChunkMinHW && k <= kMaxChunks ? k : 0;
}

// Pixel lanes per workgroup: enough that every lane has a few pixels to stream.
static int gn_pixel_lanes(int HW) { return HW >= 1024 ? 128 : (HW >= 256 ? 64 : 32); }

static bool gn_shape_ok(int N, int HW, int C, int G) {
  if (N <= 0 || HW <= 0 || C <= 0 || G <= 0) return false;
  if (C % G != 0 || C % kSlab != 0) return false;
  const int cpg = C / G;
  return cpg >= 4 && kSlab % cpg == 0;
}

}  // namespace dpa

using namespace dpa;


// Calls f(bool_constant<a>, bool_constant<b>, bool_constant<c>): one launch site for the
// eight compile-time variants of a kernel.
template <typename F>
static void dispatch3(bool a, bool b, bool c, F f) {
  auto lc = [&](auto A, auto B) {
    if (c)
      f(A, B, std::true_type{});
    else
      f(A, B, std::false_type{});
  };
  auto lb = [&](auto A) {
    if (b)
      lc(A, std::true_type{});
    else
      lc(A, std::false_type{});
  };
  if (a)
    lb(std::true_type{});
  else
    lb(std::false_type{});
}

// The producer-fused e4m3 output of the fp8 entry points (GnArgs::q).
struct GnQOut {
  void* q;
  const float* scale;
  uint32_t* part;
  int cap;
  uint32_t* count;
};

// Room for the amax partials of the launch that writes the output, 0 for the form without the
// fused cast (HW > 8192 pixels): one per workgroup of the resident form up to kResMaxHW pixels and
// of the chunked form above, which has more of them than the thin slabs (HW / 128 chunks of 64
// channels against two slabs of 32, or four of 16 above 2048 pixels).
static int64_t gn_q_blocks(int N, int HW, int C) {
  const int nchunk = gn_chunks(HW);
  const int64_t slabs = (int64_t)(C / kSlab) * N;
  return HW <= kResMaxHW ? slabs : slabs * nchunk;
}

// Launch grid of a resident kernel (GnSlab)
static dim3 gn_res_grid(const GnRes& rs, int N, int C) {
  if (rs.ng == 8) return dim3((unsigned)(C / kSlab), (unsigned)N);
  return dim3((unsigned)(8 * ceil_div((int64_t)(C / (8 * rs.ng)) * N, 8)));
}

static int gn_set_q(GnArgs& a, const GnQOut* qo, int64_t nblk) {
  if (!qo) return DPA_OK;
  if (!qo->q || !qo->scale || !qo->part || !qo->count) return DPA_ERR_NULL;
  if (nblk <= 0) return DPA_ERR_SHAPE;
  if (qo->cap < nblk) return DPA_ERR_WORKSPACE;
  if (!aligned(qo->q, 8) || !aligned(qo->scale, 4) || !aligned(qo->part, 4) ||
      !aligned(qo->count, 4))
    return DPA_ERR_ALIGN;
  a.q = (uint8_t*)qo->q;
  a.q_scale = qo->scale;
  a.q_part = qo->part;
  a.q_count = qo->count;
  return DPA_OK;
}

static int64_t gn_fwd_workspace(int N, int HW, int G) {
  return (int64_t)N * gn_chunks(HW) * G * (int64_t)sizeof(float2);
}

// Dropout arguments: keep when the 16-bit hash is >= floor(p * 2^16) (p < 1: at most 65535);
// scale 1 / (1 - p) rounded as torch's dropout forms it (1 - p in double, rounded to fp32, its
// reciprocal rounded to fp32).
static int gn_set_dropout(GnArgs& a, const void* seed, float p) {
  if (!seed) return DPA_OK;
  if (!(p >= 0.0f && p < 1.0f)) return DPA_ERR_SIZE;
  if (!aligned(seed, 8)) return DPA_ERR_ALIGN;
  a.drop_seed = (const uint64_t*)seed;
  a.drop_keep = (uint32_t)((double)p * 65536.0);
  const float pa = (float)(1.0 - (double)p);
  a.drop_scale = (float)(1.0 / (double)pa);
  return DPA_OK;
}

static int gn_fwd(const void* x, const float* gamma, const float* beta, const float* film_scale,
                  const float* film_shift, const void* film_wb, void* out, float* mean,
                  float* rstd, int N, int HW, int C, int G, float eps, void* stream,
                  void* workspace = nullptr, int64_t workspace_bytes = 0, bool x_f32 = false,
                  const void* drop_seed = nullptr, float drop_p = 0.0f, void* x_bf16 = nullptr,
                  const GnQOut* qo = nullptr, uint32_t* xb_part = nullptr,
                  int xb_part_cap = 0) {
  if (!x || !gamma || !beta || (!out && !qo) || !mean || !rstd) return DPA_ERR_NULL;
  if (qo && out) return DPA_ERR_SHAPE;  // one output: bf16 or e4m3
  if ((film_scale == nullptr) != (film_shift == nullptr)) return DPA_ERR_NULL;
  if (!gn_shape_ok(N, HW, C, G)) return DPA_ERR_SHAPE;
  if (!aligned(x, 16) || !aligned(out, 16) || !aligned(film_wb, 2)) return DPA_ERR_ALIGN;
  GnArgs a{};
  a.x = x;
  a.gamma = gamma;
  a.beta = beta;
  a.fs = film_scale;
  a.fb = film_shift;
  a.wb = (const uint16_t*)film_wb;
  a.out = out;
  a.mean = mean;
  a.rstd = rstd;
  a.N = N; a.HW = HW; a.C = C; a.G = G; a.cpg = C / G; a.eps = eps;
  const int nchunk = gn_chunks(HW);
  const GnRes rs = gn_res_shape(
      N, HW, C, G, {false, x_f32, film_scale || film_wb, drop_seed != nullptr});
  const bool ws_ok = nchunk > 0 && workspace && workspace_bytes >= gn_fwd_workspace(N, HW, G) &&
                     aligned(workspace, 8);
  // (above kResMaxHW a call without the chunked form's workspace keeps its one-launch form)
  const bool resident = rs.ng > 0 && (HW <= kResMaxHW || ws_ok);
  const bool chunked = !resident && ws_ok;
  // fp32 x and dropout: the resident form or the chunked form (workspace)
  if ((x_f32 || drop_seed) && !chunked && !resident)
    return nchunk > 0 ? DPA_ERR_WORKSPACE : DPA_ERR_SHAPE;
  if (x_bf16 && !x_f32) return DPA_ERR_SHAPE;  // the bf16 copy is of an fp32 x
  if (!aligned(x_bf16, 16)) return DPA_ERR_ALIGN;
  a.x_bf16 = (uint16_t*)x_bf16;
  if (xb_part) {
    // one partial per workgroup of the launch that writes the copy (the resident form, or
    // the chunked form's apply launch)
    if (!x_bf16) return DPA_ERR_NULL;
    if (!chunked && !resident) return nchunk > 0 ? DPA_ERR_WORKSPACE : DPA_ERR_SHAPE;
    if (xb_part_cap < gn_q_blocks(N, HW, C)) return DPA_ERR_WORKSPACE;
    if (!aligned(xb_part, 4)) return DPA_ERR_ALIGN;
    a.xb_part = xb_part;
    a.xb_room = (uint32_t)gn_q_blocks(N, HW, C);
  }
  const int dst = gn_set_dropout(a, drop_seed, drop_p);
  if (dst != DPA_OK) return dst;
  if (qo) {
    if (!chunked && !resident) return nchunk > 0 ? DPA_ERR_WORKSPACE : DPA_ERR_SHAPE;
    const int qst = gn_set_q(a, qo, gn_q_blocks(N, HW, C));
    if (qst != DPA_OK) return qst;
    a.out = qo->q;  // not written: the kernels store through a.q
  }
  hipStream_t s = (hipStream_t)stream;
  if (chunked) {
    dim3 cgrid((unsigned)(C / kSlab), (unsigned)N, (unsigned)nchunk);
    float2* cs = (float2*)workspace;
    if (x_f32)
      gn_chunk_stats_kernel<true><<<cgrid, 8 * kChPLN, 0, s>>>(a, cs, nchunk);
    else
      gn_chunk_stats_kernel<false><<<cgrid, 8 * kChPLN, 0, s>>>(a, cs, nchunk);
    int st = launch_status();
    if (st != DPA_OK) return st;
    dispatch3(x_f32, a.fs || a.wb, a.drop_seed != nullptr, [&](auto F32, auto FILM, auto DROP) {
      gn_chunk_apply_kernel<decltype(F32)::value, decltype(FILM)::value, decltype(DROP)::value>
          <<<cgrid, 8 * kChPLN, 0, s>>>(a, cs, nchunk);
    });
    return launch_status();
  }
  if (resident) {
    const dim3 rgrid = gn_res_grid(rs, N, C);
    dispatch3(a.fs || a.wb, x_f32, a.drop_seed != nullptr, [&](auto FILM, auto F32, auto DROP) {
      constexpr bool kF = decltype(FILM)::value, k3 = decltype(F32)::value,
                     kD = decltype(DROP)::value;
      if (rs.u == 4)
        gn_res_fwd_kernel<32, 4, kF, k3, kD><<<rgrid, 8 * 32, 0, s>>>(a);
      else if (rs.u == 8)
        gn_res_fwd_kernel<32, 8, kF, k3, kD><<<rgrid, 8 * 32, 0, s>>>(a);
      else if (rs.ng == 8)
        gn_res_fwd_kernel<64, 16, kF, k3, kD><<<rgrid, 8 * 64, 0, s>>>(a);
      else if (rs.ng == 4)
        gn_res_fwd_kernel<128, 16, kF, k3, kD, false, 4><<<rgrid, 4 * 128, 0, s>>>(a);
      else
        gn_res_fwd_kernel<256, 16, kF, k3, kD, false, 2><<<rgrid, 2 * 256, 0, s>>>(a);
    });
    return launch_status();
  }
  dim3 grid((unsigned)(C / kSlab), (unsigned)N);
  const int pln = gn_pixel_lanes(HW);
  if (pln == 128)
    gn_silu_fwd_kernel<128><<<grid, 8 * 128, 0, (hipStream_t)stream>>>(a);
  else if (pln == 64)
    gn_silu_fwd_kernel<64><<<grid, 8 * 64, 0, (hipStream_t)stream>>>(a);
  else
    gn_silu_fwd_kernel<32><<<grid, 8 * 32, 0, (hipStream_t)stream>>>(a);
  return launch_status();
}

extern "C" int dpa_gn_silu_fwd_bf16(const void* x, const float* gamma, const float* beta,
                                    const float* film_scale, const float* film_shift, void* out,
                                    float* mean, float* rstd, int N, int HW, int C, int G,
                                    float eps, void* stream) {
  return gn_fwd(x, gamma, beta, film_scale, film_shift, nullptr, out, mean, rstd, N, HW, C, G,
                eps, stream);
}

extern "C" int dpa_gn_silu_film_fwd_bf16(const void* x, const float* gamma, const float* beta,
                                         const void* film_wb, void* out, float* mean, float* rstd,
                                         int N, int HW, int C, int G, float eps, void* stream) {
  if (!film_wb) return DPA_ERR_NULL;
  return gn_fwd(x, gamma, beta, nullptr, nullptr, film_wb, out, mean, rstd, N, HW, C, G, eps,
                stream);
}

extern "C" int64_t dpa_gn_silu_fwd_workspace_bytes(int N, int HW, int C, int G) {
  if (!gn_shape_ok(N, HW, C, G)) return 0;
  return gn_fwd_workspace(N, HW, G);
}

extern "C" int dpa_gn_silu_fwd_ws_bf16(const void* x, const float* gamma, const float* beta,
                                       const float* film_scale, const float* film_shift,
                                       const void* film_wb, void* out, float* mean, float* rstd,
                                       void* workspace, int64_t workspace_bytes, int N, int HW,
                                       int C, int G, float eps, void* stream) {
  if (film_wb && film_scale) return DPA_ERR_SHAPE;  // one FiLM form at a time
  if (gn_shape_ok(N, HW, C, G) && workspace_bytes < gn_fwd_workspace(N, HW, G))
    return DPA_ERR_WORKSPACE;
  if (workspace_bytes > 0 && !workspace) return DPA_ERR_WORKSPACE;
  if (!aligned(workspace, 8)) return DPA_ERR_ALIGN;
  return gn_fwd(x, gamma, beta, film_scale, film_shift, film_wb, out, mean, rstd, N, HW, C, G,
                eps, stream, workspace, workspace_bytes);
}

extern "C" int dpa_gn_silu_fwd_ex(const void* x, int x_dtype, const float* gamma,
                                  const float* beta, const float* film_scale,
                                  const float* film_shift, const void* film_wb, void* out,
                                  float* mean, float* rstd, void* workspace,
                                  int64_t workspace_bytes, int N, int HW, int C, int G, float eps,
                                  const void* drop_seed, float drop_p, void* x_bf16,
                                  void* stream) {
  if (x_dtype != DPA_DTYPE_BF16 && x_dtype != DPA_DTYPE_F32) return DPA_ERR_SHAPE;
  if (film_wb && film_scale) return DPA_ERR_SHAPE;
  if (gn_shape_ok(N, HW, C, G) && workspace_bytes < gn_fwd_workspace(N, HW, G))
    return DPA_ERR_WORKSPACE;
  if (workspace_bytes > 0 && !workspace) return DPA_ERR_WORKSPACE;
  if (!aligned(workspace, 8)) return DPA_ERR_ALIGN;
  return gn_fwd(x, gamma, beta, film_scale, film_shift, film_wb, out, mean, rstd, N, HW, C, G,
                eps, stream, workspace, workspace_bytes, x_dtype == DPA_DTYPE_F32, drop_seed,
                drop_p, x_bf16);
}

extern "C" int dpa_gn_silu_fwd_ex_amax(const void* x, int x_dtype, const float* gamma,
                                       const float* beta, const float* film_scale,
                                       const float* film_shift, const void* film_wb, void* out,
                                       float* mean, float* rstd, void* workspace,
                                       int64_t workspace_bytes, int N, int HW, int C, int G,
                                       float eps, const void* drop_seed, float drop_p,
                                       void* x_bf16, uint32_t* xb_partials, int xb_partials_cap,
                                       void* stream) {
  if (x_dtype != DPA_DTYPE_BF16 && x_dtype != DPA_DTYPE_F32) return DPA_ERR_SHAPE;
  if (film_wb && film_scale) return DPA_ERR_SHAPE;
  if (!xb_partials) return DPA_ERR_NULL;
  if (gn_shape_ok(N, HW, C, G) && workspace_bytes < gn_fwd_workspace(N, HW, G))
    return DPA_ERR_WORKSPACE;
  if (workspace_bytes > 0 && !workspace) return DPA_ERR_WORKSPACE;
  if (!aligned(workspace, 8)) return DPA_ERR_ALIGN;
  return gn_fwd(x, gamma, beta, film_scale, film_shift, film_wb, out, mean, rstd, N, HW, C, G,
                eps, stream, workspace, workspace_bytes, x_dtype == DPA_DTYPE_F32, drop_seed,
                drop_p, x_bf16, nullptr, xb_partials, xb_partials_cap);
}

// per-image channel partials of dgamma/dbeta, then (chunked form) the chunk sums
static int64_t gn_bwd_workspace(int N, int HW, int C) {
  return (int64_t)2 * N * C * 4 + (int64_t)gn_chunks(HW) * N * C * (int64_t)sizeof(float4);
}

extern "C" int64_t dpa_gn_silu_bwd_workspace_bytes(int N, int HW, int C, int G) {
  (void)G;
  if (N <= 0 || HW <= 0 || C <= 0) return 0;
  return gn_bwd_workspace(N, HW, C);
}

static int gn_bwd(const void* x, const void* dout, const float* gamma, const float* beta,
                  const float* film_scale, const float* film_shift, const void* film_wb,
                  const float* mean, const float* rstd, void* dx, float* dgamma, float* dbeta,
                  float* dfilm_scale, float* dfilm_shift, void* dfilm_wb, void* workspace,
                  int64_t workspace_bytes, int N, int HW, int C, int G, void* stream,
                  bool x_f32 = false, const void* drop_seed = nullptr, float drop_p = 0.0f,
                  const void* dx_add = nullptr, bool dx_add_bf16 = false,
                  const GnQOut* qo = nullptr) {
  if (qo) dx = qo->q;  // the e4m3 dx replaces the bf16 one
  if (!x || !dout || !gamma || !beta || !mean || !rstd || !dx || !dgamma || !dbeta)
    return DPA_ERR_NULL;
  if ((film_scale == nullptr) != (film_shift == nullptr)) return DPA_ERR_NULL;
  if (film_scale && (!dfilm_scale || !dfilm_shift)) return DPA_ERR_NULL;
  if (film_wb && !dfilm_wb) return DPA_ERR_NULL;
  if (!gn_shape_ok(N, HW, C, G)) return DPA_ERR_SHAPE;
  if (!workspace || workspace_bytes < (int64_t)2 * N * C * 4) return DPA_ERR_WORKSPACE;
  if (!aligned(x, 16) || !aligned(dout, 16) || !aligned(dx, 16) || !aligned(workspace, 4) ||
      !aligned(film_wb, 2) || !aligned(dfilm_wb, 2))
    return DPA_ERR_ALIGN;
  GnArgs a{};
  a.x = x;
  a.dout = (const uint16_t*)dout;
  a.gamma = gamma;
  a.beta = beta;
  a.fs = film_scale;
  a.fb = film_shift;
  a.wb = (const uint16_t*)film_wb;
  a.out = dx;
  a.mean = const_cast<float*>(mean);
  a.rstd = const_cast<float*>(rstd);
  a.part = (float*)workspace;
  a.dfs = film_scale ? dfilm_scale : nullptr;
  a.dfb = film_scale ? dfilm_shift : nullptr;
  a.dwb = film_wb ? (uint16_t*)dfilm_wb : nullptr;
  a.N = N; a.HW = HW; a.C = C; a.G = G; a.cpg = C / G; a.eps = 0.f;
  hipStream_t s = (hipStream_t)stream;
  const int nchunk = gn_chunks(HW);
  const GnRes rs = gn_res_shape(
      N, HW, C, G, {true, x_f32, film_scale || film_wb, drop_seed != nullptr});
  const bool ws_ok = nchunk > 0 && workspace_bytes >= gn_bwd_workspace(N, HW, C) &&
                     aligned(workspace, 16);
  const bool resident = rs.ng > 0 && (HW <= kResMaxHW || ws_ok);
  const bool chunked = !resident && ws_ok;
  if ((x_f32 || drop_seed || dx_add) && !chunked && !resident)
    return nchunk > 0 ? DPA_ERR_WORKSPACE : DPA_ERR_SHAPE;
  if (!aligned(dx_add, 16)) return DPA_ERR_ALIGN;
  a.dx_add = dx_add;
  a.dx_add_bf16 = x_f32 && dx_add_bf16;
  const int dst = gn_set_dropout(a, drop_seed, drop_p);
  if (dst != DPA_OK) return dst;
  if (qo) {
    if (x_f32 || dx_add) return DPA_ERR_SHAPE;  // e4m3 of a bf16 dx, nothing added
    if (!chunked && !resident) return nchunk > 0 ? DPA_ERR_WORKSPACE : DPA_ERR_SHAPE;
    const int qst = gn_set_q(a, qo, gn_q_blocks(N, HW, C));
    if (qst != DPA_OK) return qst;
  }
  const bool film = a.fs || a.wb;
  int st = DPA_OK;
  if (chunked) {
    // chunk sums after the 2*N*C per-image partials (16-B aligned: 8*N*C bytes, C % 64 == 0)
    float4* cp = (float4*)((float*)workspace + (int64_t)2 * N * C);
    dim3 cgrid((unsigned)(C / kSlab), (unsigned)N, (unsigned)nchunk);
    const bool drop = a.drop_seed != nullptr;
    dispatch3(film, x_f32, drop, [&](auto FILM, auto F32, auto DROP) {
      gn_chunk_bwd_sums_kernel<decltype(FILM)::value, decltype(F32)::value, decltype(DROP)::value>
          <<<cgrid, 8 * kChPLN, 0, s>>>(a, cp);
    });
    st = launch_status();
    if (st != DPA_OK) return st;
    dispatch3(film, x_f32, drop, [&](auto FILM, auto F32, auto DROP) {
      gn_chunk_bwd_apply_kernel<decltype(FILM)::value, decltype(F32)::value, decltype(DROP)::value>
          <<<cgrid, 8 * kChPLN, 0, s>>>(a, cp, nchunk);
    });
  } else if (resident) {
    const dim3 rgrid = gn_res_grid(rs, N, C);
    dispatch3(film, x_f32, a.drop_seed != nullptr, [&](auto FILM, auto F32, auto DROP) {
      constexpr bool kF = decltype(FILM)::value, k3 = decltype(F32)::value,
                     kD = decltype(DROP)::value;
      if (rs.u == 4) {
        gn_res_bwd_kernel<32, 4, kF, k3, kD><<<rgrid, 8 * 32, 0, s>>>(a);
      } else if (rs.u == 8) {
        if constexpr (k3 && !kF && !kD) {
          if ((int64_t)(C / kSlab) * N >= 2 * num_cus()) {
            gn_res_bwd_kernel<32, 8, false, true, false, false, 8, true><<<rgrid, 8 * 32, 0, s>>>(a);
            return;
          }
        }
        gn_res_bwd_kernel<32, 8, kF, k3, kD><<<rgrid, 8 * 32, 0, s>>>(a);
      } else if constexpr (!k3 || (!kF && !kD)) {  // (gn_res_shape)
        if (rs.ng == 8)
          gn_res_bwd_kernel<64, 16, kF, k3, kD><<<rgrid, 8 * 64, 0, s>>>(a);
        else if (rs.ng == 4)
          gn_res_bwd_kernel<128, 16, kF, k3, kD, false, 4><<<rgrid, 4 * 128, 0, s>>>(a);
        else
          gn_res_bwd_kernel<256, 16, kF, k3, kD, false, 2><<<rgrid, 2 * 256, 0, s>>>(a);
      }
    });
  } else {
    dim3 grid((unsigned)(C / kSlab), (unsigned)N);
    const int pln = gn_pixel_lanes(HW);
    if (pln == 128)
      gn_silu_bwd_kernel<128><<<grid, 8 * 128, 0, s>>>(a);
    else if (pln == 64)
      gn_silu_bwd_kernel<64><<<grid, 8 * 64, 0, s>>>(a);
    else
      gn_silu_bwd_kernel<32><<<grid, 8 * 32, 0, s>>>(a);
  }
  st = launch_status();
  if (st != DPA_OK) return st;
  gn_param_reduce_kernel<<<(unsigned)ceil_div(C, 64), 64 * kPrSlices, 0, s>>>(
      (const float*)workspace, dgamma, dbeta, N, C);
  return launch_status();
}

extern "C" int dpa_gn_silu_bwd_bf16(const void* x, const void* dout, const float* gamma,
                                    const float* beta, const float* film_scale,
                                    const float* film_shift, const float* mean,
                                    const float* rstd, void* dx, float* dgamma, float* dbeta,
                                    float* dfilm_scale, float* dfilm_shift, void* workspace,
                                    int64_t workspace_bytes, int N, int HW, int C, int G,
                                    void* stream) {
  return gn_bwd(x, dout, gamma, beta, film_scale, film_shift, nullptr, mean, rstd, dx, dgamma,
                dbeta, dfilm_scale, dfilm_shift, nullptr, workspace, workspace_bytes, N, HW, C, G,
                stream);
}

extern "C" int dpa_gn_silu_film_bwd_bf16(const void* x, const void* dout, const float* gamma,
                                         const float* beta, const void* film_wb,
                                         const float* mean, const float* rstd, void* dx,
                                         float* dgamma, float* dbeta, void* dfilm_wb,
                                         void* workspace, int64_t workspace_bytes, int N, int HW,
                                         int C, int G, void* stream) {
  if (!film_wb || !dfilm_wb) return DPA_ERR_NULL;
  return gn_bwd(x, dout, gamma, beta, nullptr, nullptr, film_wb, mean, rstd, dx, dgamma, dbeta,
                nullptr, nullptr, dfilm_wb, workspace, workspace_bytes, N, HW, C, G, stream);
}

extern "C" int dpa_gn_silu_bwd_ex(const void* x, int x_dtype, const void* dout, const float* gamma,
                                  const float* beta, const float* film_scale,
                                  const float* film_shift, const void* film_wb, const float* mean,
                                  const float* rstd, void* dx, const void* dx_add,
                                  int dx_add_dtype, float* dgamma,
                                  float* dbeta, float* dfilm_scale, float* dfilm_shift,
                                  void* dfilm_wb, void* workspace, int64_t workspace_bytes, int N,
                                  int HW, int C, int G, const void* drop_seed, float drop_p,
                                  void* stream) {
  if (x_dtype != DPA_DTYPE_BF16 && x_dtype != DPA_DTYPE_F32) return DPA_ERR_SHAPE;
  if (film_wb && film_scale) return DPA_ERR_SHAPE;
  // the added gradient is x's dtype, or bf16 beside an fp32 x; nothing else is read
  if (dx_add && dx_add_dtype != DPA_DTYPE_BF16 && dx_add_dtype != DPA_DTYPE_F32)
    return DPA_ERR_SHAPE;
  if (dx_add && x_dtype == DPA_DTYPE_BF16 && dx_add_dtype != DPA_DTYPE_BF16)
    return DPA_ERR_SHAPE;
  return gn_bwd(x, dout, gamma, beta, film_scale, film_shift, film_wb, mean, rstd, dx, dgamma,
                dbeta, dfilm_scale, dfilm_shift, dfilm_wb, workspace, workspace_bytes, N, HW, C, G,
                stream, x_dtype == DPA_DTYPE_F32, drop_seed, drop_p, dx_add,
                dx_add_dtype == DPA_DTYPE_BF16);
}

extern "C" int dpa_gn_silu_fp8_partials(int N, int HW, int C, int G) {
  if (!gn_shape_ok(N, HW, C, G)) return 0;
  const int64_t nb = gn_q_blocks(N, HW, C);
  return nb <= INT32_MAX ? (int)nb : 0;
}

extern "C" int dpa_gn_silu_fwd_fp8(const void* x, int x_dtype, const float* gamma,
                                   const float* beta, const float* film_scale,
                                   const float* film_shift, const void* film_wb, void* q,
                                   const float* q_scale, uint32_t* q_partials,
                                   int q_partials_cap, uint32_t* q_count, float* mean,
                                   float* rstd, void* workspace, int64_t workspace_bytes, int N,
                                   int HW, int C, int G, float eps, const void* drop_seed,
                                   float drop_p, void* x_bf16, void* stream) {
  if (x_dtype != DPA_DTYPE_BF16 && x_dtype != DPA_DTYPE_F32) return DPA_ERR_SHAPE;
  if (film_wb && film_scale) return DPA_ERR_SHAPE;
  if (!q) return DPA_ERR_NULL;
  if (gn_shape_ok(N, HW, C, G) && workspace_bytes < gn_fwd_workspace(N, HW, G))
    return DPA_ERR_WORKSPACE;
  if (workspace_bytes > 0 && !workspace) return DPA_ERR_WORKSPACE;
  if (!aligned(workspace, 8)) return DPA_ERR_ALIGN;
  const GnQOut qo{q, q_scale, q_partials, q_partials_cap, q_count};
  return gn_fwd(x, gamma, beta, film_scale, film_shift, film_wb, nullptr, mean, rstd, N, HW, C,
                G, eps, stream, workspace, workspace_bytes, x_dtype == DPA_DTYPE_F32, drop_seed,
                drop_p, x_bf16, &qo);
}

extern "C" int dpa_gn_silu_fwd_fp8_amax(const void* x, int x_dtype, const float* gamma,
                                        const float* beta, const float* film_scale,
                                        const float* film_shift, const void* film_wb, void* q,
                                        const float* q_scale, uint32_t* q_partials,
                                        int q_partials_cap, uint32_t* q_count, float* mean,
                                        float* rstd, void* workspace, int64_t workspace_bytes,
                                        int N, int HW, int C, int G, float eps,
                                        const void* drop_seed, float drop_p, void* x_bf16,
                                        uint32_t* xb_partials, int xb_partials_cap,
                                        void* stream) {
  if (x_dtype != DPA_DTYPE_BF16 && x_dtype != DPA_DTYPE_F32) return DPA_ERR_SHAPE;
  if (film_wb && film_scale) return DPA_ERR_SHAPE;
  if (!q || !xb_partials) return DPA_ERR_NULL;
  if (gn_shape_ok(N, HW, C, G) && workspace_bytes < gn_fwd_workspace(N, HW, G))
    return DPA_ERR_WORKSPACE;
  if (workspace_bytes > 0 && !workspace) return DPA_ERR_WORKSPACE;
  if (!aligned(workspace, 8)) return DPA_ERR_ALIGN;
  const GnQOut qo{q, q_scale, q_partials, q_partials_cap, q_count};
  return gn_fwd(x, gamma, beta, film_scale, film_shift, film_wb, nullptr, mean, rstd, N, HW, C,
                G, eps, stream, workspace, workspace_bytes, x_dtype == DPA_DTYPE_F32, drop_seed,
                drop_p, x_bf16, &qo, xb_partials, xb_partials_cap);
}

extern "C" int dpa_gn_silu_bwd_fp8(const void* x, const void* dout, const float* gamma,
                                   const float* beta, const float* film_scale,
                                   const float* film_shift, const void* film_wb,
                                   const float* mean, const float* rstd, void* dxq,
                                   const float* dx_scale, uint32_t* dx_partials,
                                   int dx_partials_cap, uint32_t* dx_count, float* dgamma,
                                   float* dbeta, float* dfilm_scale, float* dfilm_shift,
                                   void* dfilm_wb, void* workspace, int64_t workspace_bytes,
                                   int N, int HW, int C, int G, const void* drop_seed,
                                   float drop_p, void* stream) {
  if (film_wb && film_scale) return DPA_ERR_SHAPE;
  if (!dxq) return DPA_ERR_NULL;
  const GnQOut qo{dxq, dx_scale, dx_partials, dx_partials_cap, dx_count};
  return gn_bwd(x, dout, gamma, beta, film_scale, film_shift, film_wb, mean, rstd, dxq, dgamma,
                dbeta, dfilm_scale, dfilm_shift, dfilm_wb, workspace, workspace_bytes, N, HW, C, G,
                stream, false, drop_seed, drop_p, nullptr, false, &qo);
}

// ---- a decoder stage's first GroupNorm+SiLU fused with the upsample-and-concatenate before
// it (diffusion/unet.py:379-382 and :151): x = cat([up2(a), h], channels), read from a (bf16)
// and h (bf16, or fp32 at 16x16), NHWC, instead of the fp32 concatenation; the backward
// writes the gradients of a and h instead of the concatenation's. The resident forms of
// 32x32 images (64 pixel lanes x 16 pixels, h bf16) and 16x16 images (32 x 8). ----

static int upcat_gn_check(const void* a, const void* h, int h_dtype, int N, int H, int W,
                          int Ca, int Ch, int G) {
  if (!a || !h) return DPA_ERR_NULL;
  if (N <= 0 || H <= 0 || W <= 0 || Ca <= 0 || Ch <= 0) return DPA_ERR_SIZE;
  if (h_dtype != DPA_DTYPE_BF16 && h_dtype != DPA_DTYPE_F32) return DPA_ERR_SHAPE;
  const bool s32 = H == 32 && W == 32 && h_dtype == DPA_DTYPE_BF16;
  const bool s16 = H == 16 && W == 16;
  if (!(s32 || s16) || Ca % kSlab != 0 || Ch % kSlab != 0 ||
      !gn_shape_ok(N, H * W, Ca + Ch, G))
    return DPA_ERR_SHAPE;
  if ((int64_t)N * H * W * (Ca + Ch) > 0x7fffffffLL) return DPA_ERR_SIZE;
  if (!aligned(a, 16) || !aligned(h, 16)) return DPA_ERR_ALIGN;
  return DPA_OK;
}

extern "C" int dpa_upcat_gn_silu_fwd(const void* a, const void* h, int h_dtype, int N, int H,
                                     int W, int Ca, int Ch, const float* gamma,
                                     const float* beta, void* out, void* q,
                                     const float* q_scale, uint32_t* q_partials,
                                     int q_partials_cap, uint32_t* q_count, float* mean,
                                     float* rstd, void* x_bf16, uint32_t* xb_partials,
                                     int xb_partials_cap, int G, float eps, void* stream) {
  const int st0 = upcat_gn_check(a, h, h_dtype, N, H, W, Ca, Ch, G);
  if (st0 != DPA_OK) return st0;
  if (!gamma || !beta || !mean || !rstd || (!out && !q)) return DPA_ERR_NULL;
  if (out && q) return DPA_ERR_SHAPE;  // one output: bf16 or e4m3
  if (xb_partials && !x_bf16) return DPA_ERR_NULL;
  if (!aligned(out, 16) || !aligned(x_bf16, 16) || !aligned(xb_partials, 4)) return DPA_ERR_ALIGN;
  const int C = Ca + Ch, HW = H * W;
  GnArgs g{};
  g.x = h;  // (not read: the kernel reads cat_a and cat_h)
  g.cat_a = (const uint16_t*)a;
  g.cat_h = (const uint16_t*)h;
  g.cat_ca = Ca;
  g.cat_w = W;
  g.cat_hf = h_dtype == DPA_DTYPE_F32;
  g.gamma = gamma;
  g.beta = beta;
  g.out = out;
  g.mean = mean;
  g.rstd = rstd;
  g.x_bf16 = (uint16_t*)x_bf16;
  g.N = N; g.HW = HW; g.C = C; g.G = G; g.cpg = C / G; g.eps = eps;
  const int64_t nblk = gn_q_blocks(N, HW, C);
  if (xb_partials) {
    if (xb_partials_cap < nblk) return DPA_ERR_WORKSPACE;
    g.xb_part = xb_partials;
  }
  if (q) {
    const GnQOut qo{q, q_scale, q_partials, q_partials_cap, q_count};
    const int qst = gn_set_q(g, &qo, nblk);
    if (qst != DPA_OK) return qst;
    g.out = q;  // not written: the kernel stores through g.q
  }
  dim3 grid((unsigned)(C / kSlab), (unsigned)N);
  hipStream_t s = (hipStream_t)stream;
  if (H == 32)
    gn_res_fwd_kernel<64, 16, false, false, false, true><<<grid, 8 * 64, 0, s>>>(g);
  else
    gn_res_fwd_kernel<32, 8, false, true, false, true><<<grid, 8 * 32, 0, s>>>(g);
  return launch_status();
}

extern "C" int dpa_upcat_gn_silu_bwd(const void* a, const void* h, int h_dtype, int N, int H,
                                     int W, int Ca, int Ch, const void* dout, const float* gamma,
                                     const float* beta, const float* mean, const float* rstd,
                                     const void* dx_add, void* ga, void* gh, float* dgamma,
                                     float* dbeta, void* workspace, int64_t workspace_bytes,
                                     int G, void* stream) {
  const int st0 = upcat_gn_check(a, h, h_dtype, N, H, W, Ca, Ch, G);
  if (st0 != DPA_OK) return st0;
  if (!dout || !gamma || !beta || !mean || !rstd || !ga || !gh || !dgamma || !dbeta)
    return DPA_ERR_NULL;
  const int C = Ca + Ch, HW = H * W;
  if (!workspace || workspace_bytes < (int64_t)2 * N * C * 4) return DPA_ERR_WORKSPACE;
  if (!aligned(dout, 16) || !aligned(dx_add, 16) || !aligned(ga, 16) || !aligned(gh, 16) ||
      !aligned(workspace, 4))
    return DPA_ERR_ALIGN;
  GnArgs g{};
  g.x = h;  // (not read: the kernel reads cat_a and cat_h)
  g.cat_a = (const uint16_t*)a;
  g.cat_h = (const uint16_t*)h;
  g.cat_ca = Ca;
  g.cat_w = W;
  g.cat_hf = h_dtype == DPA_DTYPE_F32;
  g.cat_ga = (uint16_t*)ga;
  g.cat_gh = gh;
  g.dout = (const uint16_t*)dout;
  g.gamma = gamma;
  g.beta = beta;
  g.mean = const_cast<float*>(mean);
  g.rstd = const_cast<float*>(rstd);
  g.part = (float*)workspace;
  g.dx_add = dx_add;
  g.dx_add_bf16 = 1;
  g.N = N; g.HW = HW; g.C = C; g.G = G; g.cpg = C / G; g.eps = 0.f;
  hipStream_t s = (hipStream_t)stream;
  dim3 grid((unsigned)(C / kSlab), (unsigned)N);
  if (H == 32)
    gn_res_bwd_kernel<64, 16, false, false, false, true><<<grid, 8 * 64, 0, s>>>(g);
  else
    gn_res_bwd_kernel<32, 8, false, true, false, true><<<grid, 8 * 32, 0, s>>>(g);
  int st = launch_status();
  if (st != DPA_OK) return st;
  gn_param_reduce_kernel<<<(unsigned)ceil_div(C, 64), 64 * kPrSlices, 0, s>>>(
      (const float*)workspace, dgamma, dbeta, N, C);
  return launch_status();
}
