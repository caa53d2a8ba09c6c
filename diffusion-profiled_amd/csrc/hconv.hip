// FP8 3x3 / stride-1 / pad-1 convolution (forward and data gradient) with a halo-patch pixel
// operand, for images that its tiles divide (the OHWI-weight form: 16 or 32 pixels wide).
//
// Reference: diffusion/fp8_kernels.py conv2d_fwd_fp8_kernel :142-247 and conv2d_dx_fp8_kernel
// :250-318 (the same arithmetic as igemm.hip, which serves every other shape).
//
// The nine taps of a 3x3 conv read the same input pixels shifted by (dy, dx). An output tile
// of 256 pixels is TR x TC = 8 x 32 or 16 x 16 pixels of one image, so its input is one
// (TR + 2) x (TC + 2) pixel patch. Per 128-channel chunk the patch goes into LDS once and the nine
// K-steps (one per tap) read their pixel fragments from it at offset dy * (TC + 2) + dx.
//
// Schedule: persistent, one workgroup of 8 waves per CU, XCD-aware contiguous tile ranges;
// K-steps are (chunk, tap) with taps inner. Workgroup tile 256 pixels x 128 channels; each
// wave owns 128 pixels x 32 channels and keeps its own weight fragments in registers: a
// three-deep ring of per-tap fragments loaded from L2 two taps ahead. No wave reads data
// another wave loads except the patch, so the waves synchronise once per chunk (the patch's
// double buffer), not once per K-step: two waves share each SIMD and while one stalls the
// other issues MFMAs. The next chunk's patch is staged through registers (global loads at
// the chunk start, LDS stores late in the chunk), so every wait is the compiler's own
// precise count. Each fragment's reads are issued two fragments ahead of their MFMAs, and
// scheduling barriers keep the compiler from sinking them (or the weight loads) next to
// their consumers.
//
// Weights: in the fragment-native layout (WFRAG, written by weight_frag_kernel from the
// OHWI e4m3 weight) each per-lane fragment load is one contiguous 1 KB per wave; from the
// OHWI weight itself each load touches 16 half-used cache lines (measured 6 us slower per
// cfg2 launch), which the op-level entry without a weight preparation still accepts.
// Epilogue: the wave's accumulators go through its 8 KB LDS slot and leave as 16-B
// nontemporal stores of 64-B channel runs (8-B stores straight from the accumulators,
// nontemporal or not, were 9-17 us slower per launch; plain 16-B stores 2 us slower). The data
// gradient is the same kernel on dy with the transposed weight and the taps mirrored (baked into
// its fragment layout).
#include "dpa_common.hpp"

#include <type_traits>

namespace dpa {

constexpr int kHcThreads = 512;
constexpr int kHcWaves = kHcThreads / 64;
constexpr int kHcBM = 256;  // output pixels per tile (a patch of TR rows x TC columns)
constexpr int kHcBN = 128;  // output channels per tile
constexpr int kHcBK = 128;  // K bytes per step (MFMA depth)
constexpr int kHcWM = 128;  // pixels per wave
constexpr int kHcWN = 32;   // channels per wave
constexpr int kHcPF = kHcWM / 16;                          // pixel fragments per wave (8)
constexpr int kHcPitch = 144;                              // patch pixel pitch in LDS
constexpr int kHcPatchSlots = 3072;                        // 16-B slots per patch buffer
constexpr int kHcPatchBytes = kHcPatchSlots * 16;          // 48 KB >= 340 pixels x 144 B
constexpr int kHcPatchLoads = kHcPatchSlots / kHcThreads;  // 6 slots per thread per patch
constexpr int kHcSlotBytes = kHcWM * kHcWN * 2;            // epilogue: 128 px x 32 ch bf16
static_assert(kHcWaves == (kHcBM / kHcWM) * (kHcBN / kHcWN), "wave grid");
static_assert(kHcPatchLoads == 6, "six staging registers");

struct HconvArgs {
  const uint8_t* act;  // [N][H][W][C]
  const uint8_t* wgt;  // OHWI [Cout][3][3][C], or the fragment layout (weight_frag_kernel)
  uint16_t* out;       // bf16 [N][H][W][Cout]
  const float* sa;
  const float* sb;
  const float* bias;  // [Cout] or null
  int N, H, W, C, Cout;
  int TR, TC, PC;     // output rows and columns per tile, patch row pitch (TC + 2) in pixels
  int tcshift;        // log2(TC)
  int tiles_x;        // tiles per image row (W / TC)
  int rslots;         // small tiles: 16-B LDS slots per patch row
  int thshift;        // small tiles: log2 of the tile's rows in one image (TR, or H for whole images)
  int KC, nk;         // 128-channel chunks, K-steps per tile (9 * KC)
  int tiles_n, tiles, tiles_per_xcd, wg_per_xcd;
  int flip;           // OHWI weight only: 1 = data gradient (weight tap 8 - t)
  FastDiv divTN, divTX, divKC, divH;
};

__device__ __attribute__((aligned(64))) uint8_t hc_zero16[64];

// Two patch buffers (the current chunk's and the next one's) and the per-wave epilogue slots:
// 96 + 64 = 160 KB, all of the CU's LDS.
__shared__ __attribute__((aligned(1024))) uint8_t hc_patch[2][kHcPatchBytes];
__shared__ __attribute__((aligned(1024))) uint8_t hc_slot[kHcWaves][kHcSlotBytes];

// Patch pixels sit at a 144-B pitch (128 B of channels + 16 B gap), so consecutive pixels are
// 9 16-B bank slots apart (64 banks = 16 slots), and every tap's address is the pixel's base
// plus a wave-uniform offset. gfx950 serves a ds_read_b128 in four 16-lane cycles: per
// half-wave, the lanes whose bits 2..4 have even parity (0-3, 12-15, 20-27) and the odd ones
// (4-11, 16-19, 28-31). A fragment's lane l reads column l & 15 at K byte 32 (l >> 4), so a
// cycle mixes columns 0-3, 12-15 at one K offset with columns 4-11 at the next (2 slots on);
// with column c on pixel c of the run two columns share a slot in every cycle. Columns 4-11
// take the run's even pixels and the others its odd pixels (hc_col_px): the slots 9 p of even
// and odd pixels p are even and odd, the 2-slot shift keeps parity, and no cycle conflicts.
__device__ __forceinline__ int hc_col_px(int c) {
  return (c >= 4 && c < 12) ? 2 * (c - 4) : 2 * ((c & 3) | ((c >> 1) & 4)) + 1;
}
__device__ __forceinline__ v8i hc_frag2(const uint8_t* base, uint32_t a0) {
  const uint4 lo = *reinterpret_cast<const uint4*>(base + a0);
  const uint4 hi = *reinterpret_cast<const uint4*>(base + a0 + 16);
  return v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
}

__device__ __forceinline__ v8i hc_gload2(const uint8_t* lo_src, const uint8_t* hi_src) {
  const uint4 lo = *reinterpret_cast<const uint4*>(lo_src);
  const uint4 hi = *reinterpret_cast<const uint4*>(hi_src);
  return v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
}

// kRows: the tile is whole image rows (W = TC), so a tile's pixels are consecutive and a patch
// slot's column is in the image or not for every tile (128 images of 32x32, us, checked per tile /
// so: 128 -> 128 20.1 / 19.8, 256 -> 256 61.3 / 59.8, 512 -> 256 113.1 / 109.7).
template <bool WFRAG, bool kRows>
__global__ __launch_bounds__(kHcThreads, 1) void hconv_fp8_kernel(const HconvArgs p) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1;   // pixel half (128 output pixels)
  const int wn = wave >> 1;  // channel quarter (32 output channels)
  const int frow = lane & 15, fq = lane >> 4;

  const int xcd = blockIdx.x & 7;
  const int wi = blockIdx.x >> 3;
  const int t_begin = xcd * p.tiles_per_xcd + wi;
  int t_end = (xcd + 1) * p.tiles_per_xcd;
  if (t_end > p.tiles) t_end = p.tiles;
  if (t_begin >= t_end) return;
  const int nt = (t_end - t_begin + p.wg_per_xcd - 1) / p.wg_per_xcd;
  const int nchunks = nt * p.KC;
  const float scale = p.sa[0] * p.sb[0];

  // ---- patch slots of this thread: slot e = d * 512 + tid covers LDS bytes [16e, +16):
  // pixel e / 9 of the patch, granule e % 9 (granule 8 is the pitch gap). Per slot: patch
  // row | column << 8 | (1 << 16 if the slot is a patch pixel's data), and the source offset
  // from the tile's first pixel (pixel (n, y0 - 1, x0 - 1) is row 0, column 0).
  const int patch_px = (p.TR + 2) * p.PC;
  int prw[kHcPatchLoads], pxo[kHcPatchLoads];
#pragma unroll
  for (int d = 0; d < kHcPatchLoads; ++d) {
    const int e = d * kHcThreads + tid;
    const int px = e / 9, g = e - px * 9;
    const int pr = px / p.PC;  // once per kernel: plain divisions are fine
    const int pc = px - pr * p.PC;
    const int ok = (g < 8) & (px < patch_px) & (!kRows | ((pc >= 1) & (pc <= p.W)));
    prw[d] = pr | (pc << 8) | (ok << 16);
    pxo[d] = ((pr - 1) * p.W + (pc - 1)) * p.C + g * 16;
  }

  // per-chunk scalars: chunk g -> tile (m0, n0), channel chunk kc; patch origin and first
  // image row; weight base
  struct Chunk {
    int live, m0, n0, y0, x0, pbase, wbase;
  };
  const int cb16 = p.Cout >> 4;  // 16-row weight blocks per tap (fragment layout)
  auto chunk_info = [&](int g) __attribute__((always_inline)) {
    Chunk c;
    c.live = g < nchunks;
    const int gg = c.live ? g : 0;
    const int j = (int)fdiv((uint32_t)gg, p.divKC);
    const int kc = gg - j * p.KC;
    const int tile = t_begin + j * p.wg_per_xcd;
    const int tm = (int)fdiv((uint32_t)tile, p.divTN);
    const int ty = kRows ? tm : (int)fdiv((uint32_t)tm, p.divTX);
    c.x0 = kRows ? 0 : (tm - ty * p.tiles_x) * p.TC;
    c.n0 = (tile - tm * p.tiles_n) * kHcBN;
    const int row0 = ty * p.TR;  // global output row n * H + y0
    c.y0 = row0 - (int)fdiv((uint32_t)row0, p.divH) * p.H;
    c.m0 = kRows ? tm * kHcBM : row0 * p.W + c.x0;
    c.pbase = c.m0 * p.C + kc * kHcBK;
    if (WFRAG)  // 2 KB block of (kc, tap 0, this wave's first 16 rows)
      c.wbase = ((kc * 9) * cb16 + (c.n0 >> 4) + wn * (kHcWN / 16)) * 2048 + lane * 16;
    else
      c.wbase = c.n0 * 9 * p.C + kc * kHcBK;
    return c;
  };

  // The patch of chunk c into registers (out-of-image slots and dead chunks read zeros), and
  // from there into LDS buffer buf. Six named registers with the slot index spelled out: an
  // array here is indexed before the loops unroll and would be promoted to LDS.
  uint4 st0, st1, st2, st3, st4, st5;
#define HC_LD(d, dst, c)                                                                   \
  {                                                                                        \
    const int y_ = (c).y0 + (prw[d] & 0xff) - 1;                                           \
    const int x_ = (c).x0 + ((prw[d] >> 8) & 0xff) - 1;                                    \
    const bool ok_ = (c).live & ((prw[d] >> 16) != 0) & ((unsigned)y_ < (unsigned)p.H) &   \
                     (kRows || (unsigned)x_ < (unsigned)p.W);                              \
    const uint8_t* src_ = ok_ ? p.act + (uint32_t)((c).pbase + pxo[d]) : hc_zero16;        \
    dst = *reinterpret_cast<const uint4*>(src_);                                           \
  }
#define HC_LOAD_PATCH(c) \
  HC_LD(0, st0, c) HC_LD(1, st1, c) HC_LD(2, st2, c) HC_LD(3, st3, c) HC_LD(4, st4, c) HC_LD(5, st5, c)
#define HC_ST(d, src, buf) \
  *reinterpret_cast<uint4*>(&hc_patch[(buf)][((d) * kHcThreads + tid) * 16]) = src;
#define HC_STORE_PATCH(buf)                                                                \
  HC_ST(0, st0, buf) HC_ST(1, st1, buf) HC_ST(2, st2, buf) HC_ST(3, st3, buf)              \
  HC_ST(4, st4, buf) HC_ST(5, st5, buf)

  // weight fragments of (chunk c, tap t) for the wave's two 16-channel blocks: lane
  // (frow, fq) holds row 16 cb + frow, K bytes [32 fq, +32) of the chunk (L2-resident; the
  // two pixel halves of a channel quarter read the same lines)
  int wrow[2];
#pragma unroll
  for (int cb = 0; cb < 2; ++cb) wrow[cb] = (wn * kHcWN + cb * 16 + frow) * 9 * p.C + fq * 32;
  auto load_w = [&](const Chunk& c, int t, v8i (&w)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      if (WFRAG) {
        const uint8_t* src = p.wgt + (uint32_t)(c.wbase + (t * cb16 + cb) * 2048);
        w[cb] = hc_gload2(src, src + 1024);
      } else {
        const int tap = p.flip ? 8 - t : t;
        const uint8_t* src = p.wgt + (uint32_t)(c.wbase + wrow[cb] + tap * p.C);
        w[cb] = hc_gload2(src, src + 16);
      }
    }
  };

  // pixel fragment pf: lane (frow, fq) reads pixel hc_col_px(frow) of the fragment's 16-pixel
  // run (patch centre + tap offset), granules 2 fq and 2 fq + 1; base address per pf, plus
  // (dy * PC + dx) * 144 per tap
  uint32_t abase[kHcPF];
#pragma unroll
  for (int pf = 0; pf < kHcPF; ++pf) {
    const int m = wm * kHcWM + pf * 16 + hc_col_px(frow);
    const int orow = m >> p.tcshift, ocol = m & (p.TC - 1);
    abase[pf] = (uint32_t)(((orow + 1) * p.PC + ocol + 1) * kHcPitch + 32 * fq);
  }
  auto tap_off = [&](int t) __attribute__((always_inline)) {
    const int ty = t / 3, tx = t - 3 * ty;
    return (uint32_t)(((ty - 1) * p.PC + tx - 1) * kHcPitch);
  };

  v4f acc[2][kHcPF];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < kHcPF; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  // Epilogue per finished tile: bf16(RN32(acc * RN32(sa * sb)) [+ bias]). Lane (frow, fq)
  // of block (cb, pf) holds channels 16 cb + 4 fq .. + 3 of pixel 16 pf + hc_col_px(frow):
  // all of them go into the wave's slot [128 px][64 B] first (granule g of row r at
  // g ^ ((r >> 2) & 3): conflict-free both ways), then lane l reads pixel 16 pf + l / 4,
  // granule l % 4 and stores 16 B nontemporally; a store instruction covers 16 pixels x 64 B.
  // All writes before any read, so the LDS latency is paid once per tile, not once per
  // fragment.
  uint8_t* slot = hc_slot[wave];
  auto epilogue = [&](int m0, int n0) __attribute__((always_inline)) {
#pragma unroll
    for (int pf = 0; pf < kHcPF; ++pf) {
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[cb][pf][e] * scale;
        if (p.bias) {
          const int c = n0 + wn * kHcWN + cb * 16 + 4 * fq;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = v[e] + p.bias[c + e];
        }
        const int r = pf * 16 + hc_col_px(frow), g = cb * 2 + (fq >> 1);
        *reinterpret_cast<uint2*>(slot + r * 64 + ((g ^ ((r >> 2) & 3)) * 16) + (fq & 1) * 8) =
            uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        acc[cb][pf] = v4f{0.f, 0.f, 0.f, 0.f};
      }
    }
    const int g_rd = lane & 3;
#pragma unroll
    for (int pf = 0; pf < kHcPF; ++pf) {
      const int r = pf * 16 + (lane >> 2);
      const uint4 o = *reinterpret_cast<const uint4*>(slot + r * 64 + ((g_rd ^ ((r >> 2) & 3)) * 16));
      const int m = wm * kHcWM + r;
      const int pix = kRows ? m0 + m : m0 + (m >> p.tcshift) * p.W + (m & (p.TC - 1));
      st_nt16(p.out + (uint32_t)(pix * p.Cout + n0 + wn * kHcWN + g_rd * 8), o);
    }
  };

  // ---- prologue: patch of chunk 0 and the weights of its first two taps ----
  Chunk cc = chunk_info(0);   // current chunk
  Chunk cn = chunk_info(1);   // next chunk
  v8i w0[2], w1[2], w2[2];    // weight ring: taps with t % 3 == 0, 1, 2
  HC_LOAD_PATCH(cc)
  load_w(cc, 0, w0);
  load_w(cc, 1, w1);
  HC_STORE_PATCH(0)

  for (int gc = 0; gc < nchunks; ++gc) {
    // this chunk's patch is complete (own stores done, then every wave's); every wave is
    // past the previous chunk, so the other buffer is free for the next patch
    wait_lgkmcnt0();
    lds_barrier();
    HC_LOAD_PATCH(cn)
    const uint8_t* pa = hc_patch[gc & 1];
    v8i fa[3];
    fa[0] = hc_frag2(pa, abase[0] + tap_off(0));
    fa[1] = hc_frag2(pa, abase[1] + tap_off(0));
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      v8i(&wc)[2] = t % 3 == 0 ? w0 : (t % 3 == 1 ? w1 : w2);
      v8i(&wp)[2] = t % 3 == 0 ? w2 : (t % 3 == 1 ? w0 : w1);
      // the weights of the step two ahead (this chunk's tap t + 2, or the next chunk's);
      // each stage below is closed by a scheduling barrier, so the loads stay two taps and
      // the fragment reads two stages ahead of their use
      if (t < 7)
        load_w(cc, t + 2, wp);
      else
        load_w(cn, t - 7, wp);
#pragma unroll
      for (int pf = 0; pf < kHcPF; ++pf) {
        const int f = t * kHcPF + pf;
        const int f2 = f + 2;
        if (f2 < 9 * kHcPF)
          fa[f2 % 3] = hc_frag2(pa, abase[f2 % kHcPF] + tap_off(f2 / kHcPF));
        acc[0][pf] = mfma16x16x128_e4m3(wc[0], fa[f % 3], acc[0][pf]);
        acc[1][pf] = mfma16x16x128_e4m3(wc[1], fa[f % 3], acc[1][pf]);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (t == 6) {
        HC_STORE_PATCH((gc + 1) & 1)
      }
    }
    const int j = (int)fdiv((uint32_t)gc, p.divKC);
    if (gc - j * p.KC == p.KC - 1) epilogue(cc.m0, cc.n0);
    cc = cn;
    cn = chunk_info(gc + 2);
  }
#undef HC_LD
#undef HC_LOAD_PATCH
#undef HC_ST
#undef HC_STORE_PATCH
}

// The same convolution on tiles of 128 (PF = 8) or 64 (PF = 4) output pixels x 128 channels, for
// launches whose 256-pixel tiles would leave CUs idle and for images they do not divide
// (weights in the fragment layout only). A tile this small has fewer pixels per weight
// fragment, so what bounds it is the weights' way from L2 through the L1 to the registers
// (16 KB per tap, 64 B a cycle): two waves that share a channel quarter would fetch every
// fragment twice. Instead each of the four channel quarters has two waves that own all of the
// tile's pixels and half of the K-steps: wave group kg takes taps 0-4 of the chunks whose
// running number has its parity and taps 5-8 of the others. At the tile's end the two exchange
// halves of their sums through LDS (kg 0 finishes the tile's first half of the pixels, kg 1
// the second; kg 0's sum + kg 1's in both) and store them.
template <int PF>
struct HsCfg {
  static constexpr int kBM = PF * 16;                 // output pixels per tile
  static constexpr bool kImages = PF == 4;            // a tile may hold several whole images
  static constexpr int kPatchLoads = PF == 8 ? 4 : 3;  // 16-B slots per thread per patch
  static constexpr int kPatchBytes = kPatchLoads * kHcThreads * 16;
  static constexpr int kHalf = PF / 2;                // fragments a wave finishes
  static constexpr int kXchBytes = kHalf * 2 * 64 * 16;  // a wave's sums for its partner
};
// patches of (8 + 2) x (16 + 2) pixels, and of (4 + 2) x (16 + 2), (8 + 2) x (8 + 2) or
// 4 x (4 + 2) x (4 + 2)
static_assert(HsCfg<8>::kPatchBytes >= 10 * 162 * 16 && HsCfg<4>::kPatchBytes >= 6 * 162 * 16 &&
                  HsCfg<4>::kPatchBytes >= 10 * 104 * 16 && HsCfg<4>::kPatchBytes >= 24 * 60 * 16,
              "patch buffers");
static_assert(HsCfg<8>::kHalf * 16 * kHcWN * 2 <= HsCfg<8>::kXchBytes &&
                  HsCfg<4>::kHalf * 16 * kHcWN * 2 <= HsCfg<4>::kXchBytes,
              "the bf16 slot fits the exchange block it takes over");

template <int PF>
__global__ __launch_bounds__(kHcThreads, 1) void hconv_small_kernel(const HconvArgs p) {
  using Cfg = HsCfg<PF>;
  __shared__ __attribute__((aligned(1024))) uint8_t patch[2][Cfg::kPatchBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t xch[kHcWaves][Cfg::kXchBytes];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 3;   // channel quarter (32 output channels)
  const int kg = wave >> 2;  // K-step group
  const int frow = lane & 15, fq = lane >> 4;

  const int xcd = blockIdx.x & 7;
  const int wi = blockIdx.x >> 3;
  const int t_begin = xcd * p.tiles_per_xcd + wi;
  int t_end = (xcd + 1) * p.tiles_per_xcd;
  if (t_end > p.tiles) t_end = p.tiles;
  if (t_begin >= t_end) return;
  const int nt = (t_end - t_begin + p.wg_per_xcd - 1) / p.wg_per_xcd;
  const int nchunks = nt * p.KC;
  const float scale = p.sa[0] * p.sb[0];

  // patch slots, as in hconv_fp8_kernel but with p.rslots slots per patch row: row e / rslots,
  // then 9 per pixel. A tile of several whole images has the patch rows of one after those
  // of the other; prw holds the row within the image's patch, and the image << 24.
  const int th = 1 << p.thshift;  // output rows of the tile in one image
  int prw[Cfg::kPatchLoads], pxo[Cfg::kPatchLoads];
#pragma unroll
  for (int d = 0; d < Cfg::kPatchLoads; ++d) {
    const int e = d * kHcThreads + tid;
    const int pr = e / p.rslots;  // once per kernel: plain divisions are fine
    const int rem = e - pr * p.rslots;
    const int pc = rem / 9, g = rem - pc * 9;
    const int im = Cfg::kImages ? pr / (th + 2) : 0, ir = pr - im * (th + 2);
    const int ok = (g < 8) & (im < (p.TR >> p.thshift)) & (ir < th + 2) & (pc < p.PC);
    prw[d] = ir | (pc << 8) | (ok << 16) | (im << 24);
    pxo[d] = ((im * p.H + ir - 1) * p.W + (pc - 1)) * p.C + g * 16;
  }

  struct Chunk {
    int live, m0, n0, y0, x0, n_left, pbase, wbase;
  };
  const int cb16 = p.Cout >> 4;  // 16-row weight blocks per tap
  auto chunk_info = [&](int g) __attribute__((always_inline)) {
    Chunk c;
    c.live = g < nchunks;
    const int gg = c.live ? g : 0;
    const int j = (int)fdiv((uint32_t)gg, p.divKC);
    const int kc = gg - j * p.KC;
    const int tile = t_begin + j * p.wg_per_xcd;
    const int tm = (int)fdiv((uint32_t)tile, p.divTN);
    const int ty = (int)fdiv((uint32_t)tm, p.divTX);
    c.x0 = (tm - ty * p.tiles_x) * p.TC;
    c.n0 = (tile - tm * p.tiles_n) * kHcBN;
    const int row0 = ty * p.TR;  // global output row n * H + y0
    const int n = (int)fdiv((uint32_t)row0, p.divH);
    c.y0 = row0 - n * p.H;
    c.n_left = p.N - n;  // images from the tile's first one on
    c.m0 = row0 * p.W + c.x0;
    c.pbase = c.m0 * p.C + kc * kHcBK;
    c.wbase = ((kc * 9) * cb16 + (c.n0 >> 4) + wn * (kHcWN / 16)) * 2048 + lane * 16;
    return c;
  };

  uint4 st0, st1, st2, st3;
#define HS_LD(d, dst, c)                                                                   \
  if constexpr ((d) < Cfg::kPatchLoads) {                                                  \
    const int y_ = (c).y0 + (prw[(d)] & 0xff) - 1;                                         \
    const int x_ = (c).x0 + ((prw[(d)] >> 8) & 0xff) - 1;                                  \
    const bool ok_ = (c).live & ((prw[(d)] >> 16 & 1) != 0) & ((unsigned)y_ < (unsigned)p.H) & \
                     ((unsigned)x_ < (unsigned)p.W) &                                      \
                     (!Cfg::kImages || (prw[(d)] >> 24) < (c).n_left);                     \
    const uint8_t* src_ = ok_ ? p.act + (uint32_t)((c).pbase + pxo[(d)]) : hc_zero16;      \
    dst = *reinterpret_cast<const uint4*>(src_);                                           \
  }
#define HS_LOAD_PATCH(c) HS_LD(0, st0, c) HS_LD(1, st1, c) HS_LD(2, st2, c) HS_LD(3, st3, c)
#define HS_ST(d, src, buf)                                                                 \
  if constexpr ((d) < Cfg::kPatchLoads)                                                    \
    *reinterpret_cast<uint4*>(&patch[(buf)][((d) * kHcThreads + tid) * 16]) = src;
#define HS_STORE_PATCH(buf) \
  HS_ST(0, st0, buf) HS_ST(1, st1, buf) HS_ST(2, st2, buf) HS_ST(3, st3, buf)

  auto load_w = [&](const Chunk& c, int t, v8i (&w)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      const uint8_t* src = p.wgt + (uint32_t)(c.wbase + (t * cb16 + cb) * 2048);
      w[cb] = hc_gload2(src, src + 1024);
    }
  };

  uint32_t abase[PF];
#pragma unroll
  for (int pf = 0; pf < PF; ++pf) {
    const int m = pf * 16 + hc_col_px(frow);
    const int orow = m >> p.tcshift, ocol = m & (p.TC - 1);
    const int prow = orow + 1 + (Cfg::kImages ? 2 * (orow >> p.thshift) : 0);
    abase[pf] = (uint32_t)(prow * p.rslots * 16 + (ocol + 1) * kHcPitch + 32 * fq);
  }
  auto tap_off = [&](int t) __attribute__((always_inline)) {
    const int ty = (t * 11) >> 5, tx = t - 3 * ty;  // t / 3 for t < 16
    return (uint32_t)((ty - 1) * p.rslots * 16 + (tx - 1) * kHcPitch);
  };

  v4f acc[2][PF];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < PF; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  v8i w0[2], w1[2], w2[2];  // weight ring: the group's taps in order, loaded two taps ahead
  // one tap on fragment buffers fa[.], which hold its first two fragments; nfa: the offset of
  // the tap whose first two fragments are read at its end (the tap's own again at a chunk's
  // last: read and not used, so the code has no branch)
  v8i fa[3];
  auto run_tap = [&](auto phase, const uint8_t* pa, uint32_t off, uint32_t noff, v8i (&wc)[2])
                     __attribute__((always_inline)) {
    constexpr int F0 = decltype(phase)::value;  // buffer of the tap's first fragment
#pragma unroll
    for (int pf = 0; pf < PF; ++pf) {
      fa[(F0 + pf + 2) % 3] =
          hc_frag2(pa, abase[(pf + 2) % PF] + (pf + 2 < PF ? off : noff));
      acc[0][pf] = mfma16x16x128_e4m3(wc[0], fa[(F0 + pf) % 3], acc[0][pf]);
      acc[1][pf] = mfma16x16x128_e4m3(wc[1], fa[(F0 + pf) % 3], acc[1][pf]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto rotate = [&]() __attribute__((always_inline)) {  // one tap on in the ring
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      w0[cb] = w1[cb];
      w1[cb] = w2[cb];
    }
  };

  // A finished tile: the halves of the sums exchanged, then bf16(RN32(sum * RN32(sa * sb))
  // [+ bias]) through the block just read (only this wave reads it, and its writer does not
  // write it again before the next tile's end, past a barrier) as hconv_fp8_kernel's epilogue.
  auto epilogue = [&](auto kgc, int m0, int n0) __attribute__((always_inline)) {
    constexpr int KG = decltype(kgc)::value, H = Cfg::kHalf;
    constexpr int keep = KG * H, send = H - keep;  // first fragment of the kept and sent half
    v4f* mine = reinterpret_cast<v4f*>(xch[wave]) + lane;
#pragma unroll
    for (int pf = 0; pf < H; ++pf)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) mine[(pf * 2 + cb) * 64] = acc[cb][send + pf];
    wait_lgkmcnt0();
    lds_barrier();
    uint8_t* slot = xch[wave ^ 4];
    const v4f* theirs = reinterpret_cast<const v4f*>(slot) + lane;
#pragma unroll
    for (int pf = 0; pf < H; ++pf)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) acc[cb][keep + pf] = acc[cb][keep + pf] + theirs[(pf * 2 + cb) * 64];
    wait_lgkmcnt0();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int pf = 0; pf < H; ++pf) {
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[cb][keep + pf][e] * scale;
        if (p.bias) {
          const int c = n0 + wn * kHcWN + cb * 16 + 4 * fq;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = v[e] + p.bias[c + e];
        }
        const int r = pf * 16 + hc_col_px(frow), g = cb * 2 + (fq >> 1);
        *reinterpret_cast<uint2*>(slot + r * 64 + ((g ^ ((r >> 2) & 3)) * 16) + (fq & 1) * 8) =
            uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      }
    }
    const int g_rd = lane & 3;
#pragma unroll
    for (int pf = 0; pf < H; ++pf) {
      const int r = pf * 16 + (lane >> 2);
      const uint4 o = *reinterpret_cast<const uint4*>(slot + r * 64 + ((g_rd ^ ((r >> 2) & 3)) * 16));
      const int m = keep * 16 + r;
      const int pix = m0 + (m >> p.tcshift) * p.W + (m & (p.TC - 1));
      if (!Cfg::kImages || pix < p.N * p.H * p.W)  // (whole images: a ragged last tile)
        st_nt16(p.out + (uint32_t)(pix * p.Cout + n0 + wn * kHcWN + g_rd * 8), o);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < PF; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
  };

  Chunk cc = chunk_info(0);
  Chunk cn = chunk_info(1);
  HS_LOAD_PATCH(cc)
  load_w(cc, 5 * kg, w0);
  load_w(cc, 5 * kg + 1, w1);
  HS_STORE_PATCH(0)
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  for (int gc = 0; gc < nchunks; ++gc) {
    // this chunk's patch is complete and every wave is past the previous one
    wait_lgkmcnt0();
    lds_barrier();
    HS_LOAD_PATCH(cn)
    const uint8_t* pa = patch[gc & 1];
    // this chunk's taps: four from t0, and tap 4 for the group that began at tap 0; the next
    // chunk's begin at n0
    const bool five = (gc & 1) == kg;
    const int t0 = five ? 0 : 5, n0 = 5 - t0;
    const uint32_t o0 = tap_off(t0), o1 = tap_off(t0 + 1), o2 = tap_off(t0 + 2),
                   o3 = tap_off(t0 + 3), o4 = tap_off(4);
    fa[0] = hc_frag2(pa, abase[0] + o0);
    fa[1] = hc_frag2(pa, abase[1] + o0);
    load_w(cc, t0 + 2, w2);
    run_tap(std::integral_constant<int, 0>{}, pa, o0, o1, w0);
    load_w(cc, t0 + 3, w0);
    run_tap(std::integral_constant<int, PF % 3>{}, pa, o1, o2, w1);
    load_w(five ? cc : cn, five ? 4 : n0, w1);
    run_tap(std::integral_constant<int, 2 * PF % 3>{}, pa, o2, o3, w2);
    HS_STORE_PATCH((gc + 1) & 1)
    load_w(cn, five ? n0 : n0 + 1, w2);
    run_tap(std::integral_constant<int, 3 * PF % 3>{}, pa, o3, five ? o4 : o3, w0);
    rotate();
    if (five) {
      load_w(cn, n0 + 1, w2);
      run_tap(std::integral_constant<int, 4 * PF % 3>{}, pa, o4, o4, w0);
      rotate();
    }
    const int j = (int)fdiv((uint32_t)gc, p.divKC);
    if (gc - j * p.KC == p.KC - 1) {
      if (kg == 0)
        epilogue(I0{}, cc.m0, cc.n0);
      else
        epilogue(I1{}, cc.m0, cc.n0);
    }
    cc = cn;
    cn = chunk_info(gc + 2);
  }
#undef HS_LD
#undef HS_LOAD_PATCH
#undef HS_ST
#undef HS_STORE_PATCH
}

// Fragment-native weight layout for hconv_fp8_kernel<true, .>: 2 KB blocks, block
// (kc * T + t) * (rows / 16) + rb holds, at byte half * 1024 + lane * 16 + b, row
// 16 rb + (lane & 15), K byte 128 kc + 32 (lane >> 4) + 16 half + b of tap t. The forward
// weight is read as [rows = Cout][T][K = Cin] (OHWI); the data gradient's as the transpose
// with the taps mirrored: row ci, K co, tap t <- w[co][T - 1 - t][ci]. One thread per 16 B.
__global__ __launch_bounds__(256) void weight_frag_kernel(const uint8_t* __restrict__ w,
                                                          uint8_t* __restrict__ out, int rows,
                                                          int K, int T, int transpose) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // 16-B unit
  const int64_t units = (int64_t)rows * K * T / 16;
  if (i >= units) return;
  const int lane = (int)(i & 63), half = (int)((i >> 6) & 1);
  const int64_t blk = i >> 7;
  const int nrb = rows >> 4;
  const int rb = (int)(blk % nrb);
  const int64_t kt = blk / nrb;
  const int t = (int)(kt % T), kc = (int)(kt / T);
  const int row = rb * 16 + (lane & 15);
  const int k0 = kc * 128 + (lane >> 4) * 32 + half * 16;
  uint4 v;
  if (!transpose) {
    v = *reinterpret_cast<const uint4*>(w + ((int64_t)row * T + t) * K + k0);
  } else {
    const int ts = T - 1 - t;
    uint32_t b[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) b[j] = w[((int64_t)(k0 + j) * T + ts) * rows + row];
    v.x = b[0] | (b[1] << 8) | (b[2] << 16) | (b[3] << 24);
    v.y = b[4] | (b[5] << 8) | (b[6] << 16) | (b[7] << 24);
    v.z = b[8] | (b[9] << 8) | (b[10] << 16) | (b[11] << 24);
    v.w = b[12] | (b[13] << 8) | (b[14] << 16) | (b[15] << 24);
  }
  *reinterpret_cast<uint4*>(out + i * 16) = v;
}

// The tile of an image: 8 rows x 32 columns where W allows, else 16 x 16 (340 and 324 patch
// pixels; 0: neither divides the image).
static int hconv_tile_cols(int H, int W) {
  if (W % 32 == 0 && H % 8 == 0) return 32;
  if (W % 16 == 0 && H % 16 == 0) return 16;
  return 0;
}

static bool hconv_sizes_ok(int N, int H, int W, int C, int Cout) {
  if (N <= 0 || H <= 0 || W <= 0 || C <= 0 || Cout <= 0) return false;
  if (C % kHcBK != 0 || Cout % kHcBN != 0) return false;
  // 32-bit offsets
  return (int64_t)N * H * W * C <= 0x7fffffff && (int64_t)N * H * W * Cout <= 0x7fffffff &&
         (int64_t)Cout * 9 * C <= 0x7fffffff;
}

static int hconv_grid(HconvArgs& a, int tile_px, int num_cus) {
  a.tiles_x = a.W / a.TC;
  a.tiles_n = a.Cout / kHcBN;
  a.tiles = (int)ceil_div((int64_t)a.N * a.H * a.W, tile_px) * a.tiles_n;
  a.tiles_per_xcd = (int)ceil_div(a.tiles, 8);
  int grid = (num_cus / 8) * 8;
  if (grid < 8) grid = 8;
  if (grid > a.tiles_per_xcd * 8) grid = a.tiles_per_xcd * 8;
  a.wg_per_xcd = grid / 8;
  a.KC = a.C / kHcBK;
  a.nk = 9 * a.KC;
  a.divTN = make_fastdiv((uint32_t)a.tiles_n);
  a.divTX = make_fastdiv((uint32_t)a.tiles_x);
  a.divKC = make_fastdiv((uint32_t)a.KC);
  a.divH = make_fastdiv((uint32_t)a.H);
  return grid;
}

static HconvArgs hconv_args(const void* act, const void* wgt, const float* sa, const float* sb,
                            const float* bias, void* out, int N, int H, int W, int C, int Cout) {
  HconvArgs a{};
  a.act = (const uint8_t*)act;
  a.wgt = (const uint8_t*)wgt;
  a.out = (uint16_t*)out;
  a.sa = sa;
  a.sb = sb;
  a.bias = bias;
  a.N = N; a.H = H; a.W = W; a.C = C; a.Cout = Cout;
  return a;
}

static int hconv_launch(HconvArgs& a, int flip, int wfrag, int num_cus, hipStream_t s) {
  a.TC = hconv_tile_cols(a.H, a.W);
  a.TR = kHcBM / a.TC;
  a.PC = a.TC + 2;
  a.tcshift = a.TC == 32 ? 5 : 4;
  a.flip = flip;
  const int grid = hconv_grid(a, kHcBM, num_cus);
  if (!wfrag)  // (OHWI weights: whole rows, hconv_supported)
    hconv_fp8_kernel<false, true><<<(unsigned)grid, kHcThreads, 0, s>>>(a);
  else if (a.TC == a.W)
    hconv_fp8_kernel<true, true><<<(unsigned)grid, kHcThreads, 0, s>>>(a);
  else
    hconv_fp8_kernel<true, false><<<(unsigned)grid, kHcThreads, 0, s>>>(a);
  return launch_status();
}

// ---- the small tiles (hconv_small_kernel): tile of the image, 0 columns: none ----
template <int PF>
static int hconv_small_cols(int H, int W) {
  constexpr int BM = HsCfg<PF>::kBM;
  if (W % 16 == 0 && H % (BM / 16) == 0) return 16;
  if (PF == 4 && W % 8 == 0 && H % 8 == 0) return 8;
  if (PF == 4 && W == 4 && H == 4) return 4;  // four whole images
  return 0;
}

template <int PF>
static int hconv_small_launch(HconvArgs& a, int num_cus, hipStream_t s) {
  a.TC = hconv_small_cols<PF>(a.H, a.W);
  a.TR = HsCfg<PF>::kBM / a.TC;
  a.PC = a.TC + 2;
  a.tcshift = a.TC == 16 ? 4 : (a.TC == 8 ? 3 : 2);
  const int th = a.TC == 4 ? 4 : a.TR;
  a.thshift = th == 16 ? 4 : (th == 8 ? 3 : 2);
  // 16-B slots per patch row: 9 per pixel, and for the 8- and 4-column tiles, whose 16-pixel
  // fragments span rows, 14 and 6 more: with them the fragment reads are free of bank conflicts
  // (of the paddings that fit, found by listing the slots that each 16-lane cycle reads)
  a.rslots = a.TC == 16 ? 162 : (a.TC == 8 ? 104 : 60);
  const int grid = hconv_grid(a, HsCfg<PF>::kBM, num_cus);
  hconv_small_kernel<PF><<<(unsigned)grid, kHcThreads, 0, s>>>(a);
  return launch_status();
}

// Output pixels per tile for a launch with the weight in its fragment layout, or 0 where no
// tile divides the image: the smallest tile that still gives every workgroup one tile, else the
// largest. One round of 64-pixel tiles costs 0.55 of one of 256-pixel tiles and 0.7 of one of
// 128-pixel tiles (us at 128 / 256 / 512 input channels: 5.9 / 8.4 / 12.5, 8.5 / 12.1 / 18.5,
// 10.4 / 15.5 / 25.5), while two rounds cost more than one round of tiles twice the size (256
// channels, 100 images of 16x16: 21.2 us in 64-pixel tiles, 19.0 in 128, 16.7 in 256; 50 of
// them 12.5, 11.7, 15.5; 16 of them 7.8, 10.8, 14.9).
static int hconv_pick_tile(int N, int H, int W, int Cout, int num_cus) {
  const bool t256 = hconv_tile_cols(H, W) != 0, t128 = hconv_small_cols<8>(H, W) != 0,
             t64 = hconv_small_cols<4>(H, W) != 0;
  const int64_t px = (int64_t)N * H * W, tn = Cout / kHcBN;
  if (t64 && ceil_div(px, 64) * tn <= num_cus) return 64;
  if (t128 && px / 128 * tn <= num_cus) return 128;
  return t256 ? 256 : (t128 ? 128 : (t64 ? 64 : 0));
}

}  // namespace dpa

// Entry points used by igemm.hip's dispatch (same library, C++ linkage).
namespace dpa {
// The shapes of the OHWI entries and of dpa_conv2d_*_fp8_wf: 256-pixel tiles of whole rows.
bool hconv_supported(int N, int H, int W, int C, int Cout) {
  return (W == 16 || W == 32) && hconv_tile_cols(H, W) == W && hconv_sizes_ok(N, H, W, C, Cout);
}
// The shapes of the dpa_conv2d_*_fp8_frag entries.
bool hconv_frag_supported(int N, int H, int W, int C, int Cout, int num_cus) {
  return hconv_sizes_ok(N, H, W, C, Cout) && hconv_pick_tile(N, H, W, Cout, num_cus) != 0;
}
// wgt: the OHWI weight (flip = 1: the data gradient's transposed weight, taps mirrored), or
// with wfrag = 1 the fragment layout of weight_frag_run (taps already in consumption order).
int hconv_run(const void* act, const void* wgt, const float* sa, const float* sb,
              const float* bias, void* out, int N, int H, int W, int C, int Cout, int flip,
              int wfrag, int num_cus, hipStream_t s) {
  HconvArgs a = hconv_args(act, wgt, sa, sb, bias, out, N, H, W, C, Cout);
  return hconv_launch(a, flip, wfrag, num_cus, s);
}
// The fragment-layout conv with the tile that hconv_pick_tile chooses (hconv_frag_supported
// must hold).
int hconv_frag_run(const void* act, const void* wf, const float* sa, const float* sb,
                   const float* bias, void* out, int N, int H, int W, int C, int Cout,
                   int num_cus, hipStream_t s) {
  HconvArgs a = hconv_args(act, wf, sa, sb, bias, out, N, H, W, C, Cout);
  switch (hconv_pick_tile(N, H, W, Cout, num_cus)) {
    case 256: return hconv_launch(a, 0, 1, num_cus, s);
    case 128: return hconv_small_launch<8>(a, num_cus, s);
    case 64: return hconv_small_launch<4>(a, num_cus, s);
  }
  return DPA_ERR_SHAPE;
}
// Fragment layout of an e4m3 weight w: [rows][T][K] (transpose = 0) or, for the data
// gradient, [K][T][rows] read transposed with the taps mirrored (transpose = 1).
// rows % 16 == 0, K % 128 == 0.
int weight_frag_run(const void* w, void* out, int rows, int K, int T, int transpose,
                    hipStream_t s) {
  if (rows % 16 != 0 || K % 128 != 0 || T <= 0) return DPA_ERR_SHAPE;
  const int64_t units = (int64_t)rows * K * T / 16;
  weight_frag_kernel<<<(unsigned)ceil_div(units, 256), 256, 0, s>>>(
      (const uint8_t*)w, (uint8_t*)out, rows, K, T, transpose);
  return launch_status();
}
}  // namespace dpa
