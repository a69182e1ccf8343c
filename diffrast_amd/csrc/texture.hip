// Texture sampling for gfx950: 2D textures and cube maps, nearest / bilinear / mipmapped
// lookups with wrap, clamp or zero boundaries, their gradients, and the mip chain.
//
// The arithmetic follows the reference backend: texel coordinates and boundaries
// (src/diffrast/backends/reference.py:555-672), level of detail and level blending
// (reference.py:491-501, 522-552), cube-map projection and the integer edge fold
// (src/diffrast/backends/_cube.py:44-143). One thread per pixel computes the tap addresses
// of its one or two levels once; it takes up to four channels itself, and more are taken by
// consecutive lanes. All levels live in one packed buffer [tex_batch, texels, channels], so a
// mipmapped lookup is two bilinear lookups wherever the pixel's levels are.
//
// The backward pass writes the coordinate, derivative and bias gradients per pixel; texel
// gradients are summed per workgroup in an LDS table (fixed point, after runs of neighbouring
// pixels on one texel have summed) and reach global memory with one fp32 atomic per row and
// channel. The mip chain uses exact area weights (reference.py:449-488): where sizes halve
// exactly, a workgroup takes a tile of up to 32 x 32 texels through up to five levels in LDS;
// other sizes go level by level, and the last, small levels are one workgroup's. Its adjoint is a
// gather, so it needs no atomics.
#include <type_traits>

#include "common.h"
#include "texture_math.h"

namespace dr {
namespace {

using namespace tex;

// Channels [c0, c0 + N) of a texel or pixel at p, 0 past C.
template <int N>
__device__ __forceinline__ void load_channels(const float* __restrict__ p, int C, int c0,
                                              float (&v)[N]) {
  if (c0 + N <= C) {  // uniform; known when compiling for 1-4 channels
    load_floats(p + c0, v);
    return;
  }
#pragma unroll
  for (int c = 0; c < N; ++c) v[c] = c0 + c < C ? p[c0 + c] : 0.0f;
}

// Channels [c0, c0 + N) of the four taps (0 past C or for an invalid tap), all loads issued
// together.
template <int N>
__device__ __forceinline__ void fetch_taps(const float* __restrict__ texels, const Bilinear<float>& L,
                                           int C, int c0, float (&t)[4][N]) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (L.valid[k]) {
      load_channels<N>(texels + (size_t)L.index[k] * C, C, c0, t[k]);
    } else {
#pragma unroll
      for (int c = 0; c < N; ++c) t[k][c] = 0.0f;
    }
  }
}

template <int N>
__device__ __forceinline__ void tap_column(const float (&t)[4][N], int c, float (&out)[4]) {
#pragma unroll
  for (int k = 0; k < 4; ++k) out[k] = t[k][c];
}

// One to four channels. Every tap is loaded before the stores. FILTER and BOUNDARY: a.filter and
// a.boundary, fixed when compiling (DR_BOUNDARY_CUBE for cube maps).
template <int C, bool CUBE, int FILTER, int BOUNDARY>
__global__ __launch_bounds__(256) void tex_fwd_kernel(DrTextureArgs a, float* __restrict__ out) {
  const int64_t pixel = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (pixel >= (int64_t)a.batch * a.height * a.width) return;
  float* o = out + pixel * C;
  Lookup<float> K;
  lookup_setup<float, CUBE, FILTER>(a, pixel, K);
  if (K.dir_invalid) {
    for (int c = 0; c < C; ++c) o[c] = 0.0f;
    return;
  }
  // The image's texture (the division only for per-image textures: it is some 40 VALU
  // instructions in 64 bits).
  const int64_t image = a.tex_batch > 1 ? pixel / ((int64_t)a.height * a.width) : 0;
  const float* __restrict__ texels = a.texels + image * a.num_texels * C;
  const float nan = __int_as_float(0x7fc00000);
  if (K.levels == 0) {
    uint32_t index;
    bool valid;
    const bool bad = nearest_setup<BOUNDARY>(a, K, index, valid);
    for (int c = 0; c < C; ++c) o[c] = bad ? nan : (valid ? texels[(size_t)index * C + c] : 0.0f);
    return;
  }
  const LevelDims D = lookup_levels(a, K);
  const Bilinear<float> L0 = level_setup<CUBE, BOUNDARY>(a, K, D, 0);
  const bool two = K.levels == 2;
  const Bilinear<float> L1 = two ? level_setup<CUBE, BOUNDARY>(a, K, D, 1) : L0;
  const bool bad = K.bad || L0.bad || (two && L1.bad);
  const float frac = K.level_weight[1];
  float t[4][C], u[4][C], res[C];
  fetch_taps<C>(texels, L0, C, 0, t);
  if (two) fetch_taps<C>(texels, L1, C, 0, u);
#pragma unroll
  for (int c = 0; c < C; ++c) {
    float tc[4], uc[4];
    tap_column(t, c, tc);
    if (two) {
      tap_column(u, c, uc);
      res[c] = bilinear_value(L0, tc) * (1.0f - frac) + bilinear_value(L1, uc) * frac;
    } else {
      res[c] = bilinear_value(L0, tc);
    }
    if (bad) res[c] = nan;
  }
  store_floats(o, res);
}

// A pixel's lookup as the wide kernel keeps it in LDS: per level its taps (kNoTexel: reads zero)
// and fractions, the weight of the missing tap at a cube corner, the share of the second level,
// the image, and how many levels (0: nearest, one tap; kBadLookup: NaN).
constexpr uint32_t kNoTexel = 0xffffffffu;
constexpr int kBadLookup = -1;
template <bool CUBE>
struct WideLevel {
  uint32_t index[4];
  float fx, fy;
  float missing;  // the same taps' mean counts this much (a third of their sum: at_corner)
  bool at_corner;
};
template <>
struct WideLevel<false> {
  uint32_t index[4];
  float fx, fy;
};
template <bool CUBE>
struct WideLookup {
  WideLevel<CUBE> level[2];
  float frac;
  int levels;
  uint32_t image;
};

template <bool CUBE>
__device__ __forceinline__ void keep_level(const Bilinear<float>& L, WideLevel<CUBE>& W) {
#pragma unroll
  for (int k = 0; k < 4; ++k) W.index[k] = L.valid[k] ? L.index[k] : kNoTexel;
  W.fx = L.fx;
  W.fy = L.fy;
  if constexpr (CUBE) {
    W.missing = (1.0f - L.fy) * ((1.0f - L.fx) * L.corner[0] + L.fx * L.corner[1]) +
                L.fy * ((1.0f - L.fx) * L.corner[2] + L.fx * L.corner[3]);
    W.at_corner = L.at_corner;
  }
}

// N channels of a level's lookup, from texels + element offset (bilinear_value's arithmetic).
template <int N, bool CUBE>
__device__ __forceinline__ void wide_value(const WideLevel<CUBE>& W, const float (&t)[4][N],
                                           float (&v)[N]) {
  const float fx = W.fx, fy = W.fy;
#pragma unroll
  for (int c = 0; c < N; ++c) {
    v[c] = (1.0f - fy) * ((1.0f - fx) * t[0][c] + fx * t[1][c]) +
           fy * ((1.0f - fx) * t[2][c] + fx * t[3][c]);
    if constexpr (CUBE) {
      float share = W.missing * (t[0][c] + t[1][c] + t[2][c] + t[3][c]);
      if (W.at_corner) share = share / 3.0f;
      v[c] = v[c] + share;
    }
  }
}

// More than four channels, four to a lane: each thread works out one pixel's taps, then consecutive
// lanes take a pixel's channels in turn, so that texels and output go in whole lines and the taps
// are worked out once. (A pixel per thread and four channels at a time, two 720 x 1280 images with
// 16 channels: 180 us; this one 60.) A last group past the end moves back over the one before, and
// the channels that both have are written twice, the same. (Lanes of one or two channels for counts
// that four does not divide, trilinear, two 720 x 1280 images: 5 channels 48 us, 30 this way; 7 64 and 31; 10 52 and 39.)
template <bool CUBE, int FILTER, int BOUNDARY>
__global__ __launch_bounds__(256) void tex_fwd_wide_kernel(DrTextureArgs a,
                                                           float* __restrict__ out) {
  __shared__ WideLookup<CUBE> s_lookup[256];
  const int64_t pixels = (int64_t)a.batch * a.height * a.width;
  const int64_t pixel0 = (int64_t)blockIdx.x * 256, pixel = pixel0 + threadIdx.x;
  if (pixel < pixels) {
    WideLookup<CUBE>& W = s_lookup[threadIdx.x];
    Lookup<float> K;
    lookup_setup<float, CUBE, FILTER>(a, pixel, K);
    W.image = a.tex_batch > 1 ? (uint32_t)(pixel / ((int64_t)a.height * a.width)) : 0u;
    W.frac = 0.0f;
    W.levels = K.levels;
    if (K.dir_invalid) {  // reads zero
      W.levels = 0;
      W.level[0].index[0] = kNoTexel;
    } else if (K.levels == 0) {
      uint32_t index;
      bool valid;
      if (nearest_setup<BOUNDARY>(a, K, index, valid)) W.levels = kBadLookup;
      W.level[0].index[0] = valid ? index : kNoTexel;
    } else {
      const LevelDims D = lookup_levels(a, K);
      const Bilinear<float> L0 = level_setup<CUBE, BOUNDARY>(a, K, D, 0);
      bool bad = K.bad || L0.bad;
      keep_level(L0, W.level[0]);
      if (K.levels == 2) {
        const Bilinear<float> L1 = level_setup<CUBE, BOUNDARY>(a, K, D, 1);
        bad = bad || L1.bad;
        keep_level(L1, W.level[1]);
        W.frac = K.level_weight[1];
      }
      if (bad) W.levels = kBadLookup;
    }
  }
  __syncthreads();
  constexpr int N = 4;
  const int C = a.channels, per = (C + N - 1) / N;  // elements per pixel
  const int count = (int)min((int64_t)256, pixels - pixel0);
  // A step of 256 elements moves (pixel, element) by (dj, de).
  const int dj = 256 / per, de = 256 % per;
  int j = (int)threadIdx.x / per, e = (int)threadIdx.x % per;
  for (; j < count;) {
    const WideLookup<CUBE>& W = s_lookup[j];
    const int at = min(e * N, C - N);
    const float* texels = a.texels + (int64_t)W.image * a.num_texels * C + at;
    auto fetch = [&](uint32_t index, float(&v)[N]) {
      if (index != kNoTexel) {
        load_floats(texels + (size_t)index * C, v);
      } else {
#pragma unroll
        for (int c = 0; c < N; ++c) v[c] = 0.0f;
      }
    };
    float res[N];
    if (W.levels <= 0) {
      if (W.levels == 0) {
        fetch(W.level[0].index[0], res);
      } else {
#pragma unroll
        for (int c = 0; c < N; ++c) res[c] = __int_as_float(0x7fc00000);
      }
    } else {
      float t[4][N], u[4][N];
#pragma unroll
      for (int k = 0; k < 4; ++k) fetch(W.level[0].index[k], t[k]);
      if (W.levels == 2)
#pragma unroll
        for (int k = 0; k < 4; ++k) fetch(W.level[1].index[k], u[k]);
      wide_value(W.level[0], t, res);
      if (W.levels == 2) {
        const float frac = W.frac;
        float above[N];
        wide_value(W.level[1], u, above);
#pragma unroll
        for (int c = 0; c < N; ++c) res[c] = res[c] * (1.0f - frac) + above[c] * frac;
      }
    }
    store_floats(out + (pixel0 + j) * C + at, res);
    j += dj;
    e += de;
    if (e >= per) {
      e -= per;
      ++j;
    }
  }
}

// Coordinate-gradient contributions of one level: d/dfx, d/dfy summed over channels with the
// level weight, and the level's value per channel for the blend-factor gradient.
template <int N>
__device__ __forceinline__ void level_coordinate_grads(const Bilinear<float>& L,
                                                       const float* __restrict__ texels,
                                                       const float* __restrict__ g, int C,
                                                       float level_weight, float& g_fx,
                                                       float& g_fy, bool want_value,
                                                       float& g_value) {
  for (int c0 = 0; c0 < C; c0 += N) {
    float t[4][N], gc[N];
    fetch_taps<N>(texels, L, C, c0, t);
    load_channels<N>(g, C, c0, gc);
#pragma unroll
    for (int c = 0; c < N; ++c) {
      if (c0 + c >= C) continue;
      float tc[4], dfx, dfy;
      tap_column(t, c, tc);
      const float value = bilinear_grad_value(L, tc, dfx, dfy);
      const float gl = gc[c] * level_weight;
      g_fx += gl * dfx;
      g_fy += gl * dfy;
      if (want_value) g_value += gc[c] * value;
    }
  }
}

// Table keys (texel rows of the packed buffer, 0xffffffff for none) and weights of a level's
// taps. A tap of weight 0 (the second level when the blend factor is 0, or an axis with fraction
// 0) adds nothing and gets no key.
__device__ __forceinline__ void level_taps(const Bilinear<float>& L, float level_weight,
                                           int64_t tex_off, uint32_t* key, float* weight) {
  float t0[4] = {0.f, 0.f, 0.f, 0.f}, wgt[4], dfx, dfy;
  bilinear_grad(L, t0, wgt, dfx, dfy);  // the weights do not depend on texel values
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    weight[k] = level_weight * wgt[k];
    key[k] = L.valid[k] && weight[k] != 0.0f ? (uint32_t)(tex_off + L.index[k]) : 0xffffffffu;
  }
}

// What a pixel's 2D lookup depends on, as bits: coordinates, derivatives and bias.
template <bool MIP>
struct RawLookup {
  uint32_t v[MIP ? 7 : 2];
};

template <bool MIP>
__device__ __forceinline__ RawLookup<MIP> raw_lookup(const DrTextureArgs& a, int64_t pixel) {
  RawLookup<MIP> r;
  __builtin_memcpy(r.v, a.uv + 2 * pixel, 8);
  if constexpr (MIP) {
#pragma unroll
    for (int i = 2; i < 7; ++i) r.v[i] = 0u;
    if (a.uv_da) __builtin_memcpy(r.v + 2, a.uv_da + 4 * pixel, 16);
    if (a.bias) __builtin_memcpy(r.v + 6, a.bias + pixel, 4);
  }
  return r;
}

// Texel gradients of strips (a wave's 16 x 4 pixels of a tile) whose pixels all share one lookup:
// in practice the background, whose coordinates are zero. Its taps are the same texels
// everywhere, and one texel takes atomic additions from all those tiles one after another (~9 ns
// each), so of up to kStripTiles tiles side by side the first whose strip shares the lookup
// takes the upstream gradients of the others' strips too. A wave finds out for itself:
//   - the wave's taps differ: nothing changes (a register comparison is all it cost);
//   - they are shared, by a strip further left too: the wave has nothing to add, its keys go;
//   - they are shared, first here: lane k keeps tap k alone, and the result is the mask of the
//     tiles, from this one on, whose gradients the wave sums (strip_sum).
// Texture forward and backward with four tiles side by side, against none: a 1080 x 1920 image,
// 79 % background, 3 channels 164 -> 131 us; two 720 x 1280 with 16 channels 564 -> 474; eight
// 1024^2, 38 % background, 4 channels 495 -> 493, 79 % of one texel lookup each 477 -> 292. Eight
// tiles are 1-8 % slower (a wave of the background looks at all of them), two up to 12 %.
// What it costs where no strip shares a lookup: the trilinear kernels of one to three channels
// hold 63-72 VGPRs, seven waves, instead of 58-64 and eight (four 1024^2 images, backward alone:
// 3 channels 564 -> 589 us, 1 channel 317 -> 330, texels a quarter of a pixel apart 296 -> 327).
// Bit d of the result: the strip of the d-th tile to the right; 0: an ordinary wave.
constexpr int kStripTiles = 4;

template <bool MIP>
__device__ __forceinline__ uint32_t shared_strips(const DrTextureArgs& a, const TilePixel& tp,
                                                  uint32_t (&key)[8], float (&weight)[8]) {
  // The first lane's pixel is inside the image unless the whole strip lies below it.
  bool same = true;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    same = same && key[k] == (uint32_t)__builtin_amdgcn_readfirstlane((int)key[k]);
    same = same && __float_as_int(weight[k]) ==
                       __builtin_amdgcn_readfirstlane(__float_as_int(weight[k]));
  }
  if (__ballot(tp.inside && !same) != 0) return 0u;
  if (__builtin_amdgcn_readfirstlane(tp.inside ? 1 : 0) == 0) return 0u;
  const RawLookup<MIP> own = raw_lookup<MIP>(a, tp.inside ? tp.pixel : 0);
  RawLookup<MIP> shared;
#pragma unroll
  for (int i = 0; i < (MIP ? 7 : 2); ++i)
    shared.v[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)own.v[i]);
  auto differs = [&](const RawLookup<MIP>& r) {
    bool d = false;
#pragma unroll
    for (int i = 0; i < (MIP ? 7 : 2); ++i) d = d || r.v[i] != shared.v[i];
    return d;
  };
  if (__ballot(tp.inside && differs(own)) != 0) return 0u;
  const int at = __builtin_amdgcn_readfirstlane(tp.x / 16) % kStripTiles;
  uint32_t found = 1u << at;
#pragma unroll 2
  for (int d = 0; d < kStripTiles; ++d) {
    if (d == at) continue;  // uniform
    const int x = tp.x + 16 * (d - at);
    const int x0 = __builtin_amdgcn_readfirstlane(x);
    if (x0 >= a.width) continue;  // past the last tile
    const bool inside = x < a.width && tp.y < a.height;
    const RawLookup<MIP> r = raw_lookup<MIP>(a, inside ? tp.pixel + 16 * (d - at) : 0);
    if (__ballot(inside && differs(r)) == 0) found |= 1u << d;
  }
  const bool first = (found & ((1u << at) - 1u)) == 0u;
  const int lane = lane_id();
  uint32_t k0 = 0xffffffffu;
  float w0 = 0.0f;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    // From the first lane: a lane outside the image has no taps of its own.
    const uint32_t kk = (uint32_t)__builtin_amdgcn_readfirstlane((int)key[k]);
    const float wk = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(weight[k])));
    k0 = lane == k && first ? kk : k0;
    w0 = lane == k && first ? wk : w0;
    key[k] = 0xffffffffu;
    weight[k] = 0.0f;
  }
  key[0] = k0;
  weight[0] = w0;
  return first ? found >> at : 0u;
}

// `weight` times channels [c0, c0 + N) of the upstream gradient summed over the strips of
// `strips`. Up to 256 values meet here that the row table would otherwise add in 64 bits, so the
// sum is in float64: it is rounded once, after the tap's weight has scaled it.
template <int N>
__device__ __forceinline__ void strip_sum(const DrTextureArgs& a, const TilePixel& tp,
                                          uint32_t strips, const float* grad_out, int C, int c0,
                                          float weight, float (&scaled)[N]) {
  double sum[N];
#pragma unroll
  for (int c = 0; c < N; ++c) sum[c] = 0.0;
#pragma unroll 1
  for (int d = 0; d < kStripTiles; ++d) {
    if (((strips >> d) & 1u) == 0u) continue;  // uniform over the wave
    if (tp.x + 16 * d < a.width && tp.y < a.height) {
      float g[N];
      load_channels<N>(grad_out + (tp.pixel + 16 * d) * C, C, c0, g);
#pragma unroll
      for (int c = 0; c < N; ++c) sum[c] += (double)g[c];
    }
  }
#pragma unroll
  for (int c = 0; c < N; ++c) scaled[c] = (float)(wave_sum_f64(sum[c]) * (double)weight);
}

// Channels per pass of the backward kernel for CHANNELS channels: 1-4 of them, or 0 for more, in
// fours.
template <int CHANNELS>
constexpr int kPassChannels = CHANNELS == 0 ? 4 : CHANNELS;

// Waves per SIMD that the 2D kernels are held to. Trilinear lookups and more than four channels:
// seven, 72 VGPRs, as many as the table's LDS allows (trilinear ones of 2-4 and of more than four
// channels then spill two or three registers under wrapping; at eight, 64 VGPRs, texture forward
// and backward at 8 x 1024^2 with a 1024^2 texture of 4 channels went from 493 to 510 us). The
// others: eight, as nearly all take by themselves (4 channels, clamped, nearest level, two
// 720 x 1280 images: 55 us at 66 VGPRs, 53 at 56). The cube-map kernels spill at either (239 -> 320 us
// at seven) and keep their own.
template <int CHANNELS, int FILTER>
constexpr int bwd_waves() {
  return CHANNELS == 0 || FILTER == DR_FILTER_MIP_LINEAR ? 7 : 8;
}

template <int CHANNELS, bool CUBE, int FILTER, int BOUNDARY>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(CUBE ? 1 : bwd_waves<CHANNELS, FILTER>()))) void
tex_bwd_kernel(DrTextureArgs a, const float* grad_out, float* grad_texels, float* grad_uv,
               float* grad_uv_da, float* grad_bias) {
  constexpr int NC = kPassChannels<CHANNELS>;
  using Table = RowTable<512, 4>;
  __shared__ Table table;
  table.init();
  const TilePixel tp = tile_pixel(a.batch, a.height, a.width);
  const int64_t pixel = tp.pixel;
  const int C = CHANNELS > 0 ? CHANNELS : a.channels;
  constexpr bool cube = CUBE;
  const float* g = grad_out + (tp.inside ? pixel * C : 0);
  const int64_t tex_off = a.tex_batch > 1 ? (int64_t)tp.b * a.num_texels : 0;
  const float* texels = a.texels + tex_off * C;

  Lookup<float> K;
  // Texel gradient targets: taps 0-3 of the first level, 4-7 of the second.
  uint32_t tap_key[8];
  float tap_weight[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    tap_key[k] = Table::kEmpty;
    tap_weight[k] = 0.0f;
  }
  float g_s = 0.0f, g_t = 0.0f, g_lod = 0.0f;
  bool live = false;
  if (tp.inside) {
    lookup_setup<float, CUBE, FILTER>(a, pixel, K);
    live = !K.dir_invalid;
  }
  if (live && K.levels == 0) {
    uint32_t index;
    bool valid;
    const bool bad = nearest_setup<BOUNDARY>(a, K, index, valid);
    if (!bad && valid) {
      tap_key[0] = (uint32_t)(tex_off + index);
      tap_weight[0] = 1.0f;
    }
    live = false;  // no coordinate gradient
  } else if (live) {
    const LevelDims D = lookup_levels(a, K);
    const Bilinear<float> L0 = level_setup<CUBE, BOUNDARY>(a, K, D, 0);
    Bilinear<float> L1 = L0;
    const bool two = K.levels == 2;
    if (two) L1 = level_setup<CUBE, BOUNDARY>(a, K, D, 1);
    if (K.bad || L0.bad || (two && L1.bad)) {
      live = false;
    } else {
      float fx0 = 0.f, fy0 = 0.f, fx1 = 0.f, fy1 = 0.f, v0 = 0.f, v1 = 0.f;
      level_coordinate_grads<NC>(L0, texels, g, C, K.level_weight[0], fx0, fy0, two, v0);
      level_taps(L0, K.level_weight[0], tex_off, tap_key, tap_weight);
      if (L0.pass_x) g_s += fx0 * L0.size_x;
      if (L0.pass_y) g_t += fy0 * L0.size_y;
      if (two) {
        level_coordinate_grads<NC>(L1, texels, g, C, K.level_weight[1], fx1, fy1, true, v1);
        level_taps(L1, K.level_weight[1], tex_off, tap_key + 4, tap_weight + 4);
        if (L1.pass_x) g_s += fx1 * L1.size_x;
        if (L1.pass_y) g_t += fy1 * L1.size_y;
        g_lod = K.lod_grad ? v1 - v0 : 0.0f;
      }
    }
  }

  if (tp.inside) {
    float g_da[4] = {0.f, 0.f, 0.f, 0.f};
    const bool has_da = K.mip && a.uv_da != nullptr;
    if (live && has_da && g_lod != 0.0f) {
      const Deriv4<float> da = cube ? Deriv4<float>{K.P.st_da[0], K.P.st_da[1], K.P.st_da[2],
                                                    K.P.st_da[3]}
                                    : load_deriv4(a.uv_da + 4 * pixel);
      footprint_lod_grad(da, a.level_height[0], a.level_width[0], g_lod, g_da);
    }
    if (grad_bias) grad_bias[pixel] = live ? g_lod : 0.0f;
    if (cube) {
      float gdir[3] = {0.f, 0.f, 0.f}, gdir_da[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (live) cube_project_backward(K.P, g_s, g_t, has_da, g_da, gdir, gdir_da);
      if (grad_uv)
        for (int k = 0; k < 3; ++k) grad_uv[3 * pixel + k] = gdir[k];
      if (grad_uv_da)
        for (int k = 0; k < 6; ++k) grad_uv_da[6 * pixel + k] = gdir_da[k];
    } else {
      if (grad_uv) {
        grad_uv[2 * pixel] = live ? g_s : 0.0f;
        grad_uv[2 * pixel + 1] = live ? g_t : 0.0f;
      }
      if (grad_uv_da)
        for (int k = 0; k < 4; ++k) grad_uv_da[4 * pixel + k] = live ? g_da[k] : 0.0f;
    }
  }
  if (grad_texels == nullptr) return;  // uniform over the workgroup

  uint32_t strips = 0u;
  constexpr bool kMip = FILTER == DR_FILTER_MIP_NEAREST || FILTER == DR_FILTER_MIP_LINEAR;
  if constexpr (!CUBE) strips = shared_strips<kMip>(a, tp, tap_key, tap_weight);

  // Texel gradients, four channels per pass through the workgroup's table: tap k adds
  // g[c] * weight[k] to its texel row.
  const float strip_weight = tap_weight[0];
  if (strips != 0u) tap_weight[0] = 1.0f;  // strip_sum applies it
  float w_max = 0.0f;
#pragma unroll
  for (int k = 0; k < 8; ++k)
    if (tap_key[k] != Table::kEmpty) w_max = fmaxf(w_max, fabsf(tap_weight[k]));
  for (int c0 = 0; c0 < C; c0 += 4) {
    const int n = min(4, C - c0);
    float gc[4];
    if (strips != 0u)  // uniform over the wave
      strip_sum<4>(a, tp, strips, grad_out, C, c0, strip_weight, gc);
    else
      load_channels<4>(g, C, c0, gc);
    // The largest |g[c] * weight[k]| of this lane (rounding is monotone, so the product of the
    // two largest factors is the largest product).
    float g_max = 0.0f;
    bool finite = true;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      finite = finite && isfinite(gc[c]);
      g_max = fmaxf(g_max, fabsf(gc[c]));
    }
    if (!finite) g_max = __int_as_float(0x7f800000);
    const float lane_max = w_max > 0.0f ? g_max * w_max : 0.0f;
    const FixedPass f = table.begin(lane_max);
    // One tap at a time (the tap index is uniform): unrolled, the taps' table updates would
    // interleave and hold many more registers. In 2D, neighbouring pixels of a tile row whose
    // tap on the finer level falls on the same texel sum first, and the last of them adds the
    // sum; the coarser level's taps (4-7) and cube faces go to the table directly, where the
    // summing costs more than the table updates it saves (measured: texture backward at
    // 8 x 1024^2 with a 1024^2 texture 491 -> 481 us without the coarser level's sums).
#pragma unroll 1
    for (int k = 0; k < 8; ++k) {
      const uint32_t key = tap_key[k];
      float v[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) v[c] = gc[c] * tap_weight[k];
      if constexpr (CUBE) {
        table.add_wave(key, v, n, grad_texels + c0, C, f);
      } else {
        if (__ballot(key != Table::kEmpty) == 0) continue;  // uniform
        const bool last = k >= 4 || row_run_sums(key, v);
        if (last && key != Table::kEmpty) table.add_or_global(key, v, n, grad_texels + c0, C, f);
      }
    }
    __syncthreads();
    table.flush(grad_texels + c0, C, n, f);
    if (c0 + 4 < C) {
      __syncthreads();
      table.reset();
    }
  }
}

// ---- mip chain --------------------------------------------------------------------------

// Weight of source texel i in destination texel r along an axis of n source texels: the
// overlap of their extents when n texels are split into ceil(n / 2) equal bins, over the bin
// width (reference.py:449-488). Exact integers scaled by 1 / n.
__device__ __forceinline__ float axis_weight(int r, int i, int n) {
  if (n == 1) return (r == 0 && i == 0) ? 1.0f : 0.0f;
  if ((n & 1) == 0) return (i >> 1) == r ? 0.5f : 0.0f;
  const int m = (n + 1) / 2;
  const int overlap = min((r + 1) * n, (i + 1) * m) - max(r * n, i * m);
  return overlap > 0 ? (float)overlap / (float)n : 0.0f;
}

// First source texel and tap count of destination texel r along an axis.
__device__ __forceinline__ void axis_taps(int r, int n, int& first, int& count) {
  if (n == 1) { first = 0; count = 1; return; }
  if ((n & 1) == 0) { first = 2 * r; count = 2; return; }
  const int m = (n + 1) / 2;
  first = (int)((int64_t)r * n / m);
  count = min(3, n - first);
}

struct MipLevels {
  int h[DR_MAX_LEVELS], w[DR_MAX_LEVELS];
  int64_t off[DR_MAX_LEVELS];
};

// Value i of level k + 1 ((row, col, channel) order) from level k of one image and face.
__device__ __forceinline__ void down_value(const float* src, float* dst, int C, int h, int w,
                                           int w2, uint32_t i) {
  const uint32_t texel = i / (uint32_t)C;
  const int c = (int)(i - texel * (uint32_t)C);
  const int row = (int)(texel / (uint32_t)w2), col = (int)(texel - (uint32_t)row * w2);
  int r0, nr, c0, nc;
  axis_taps(row, h, r0, nr);
  axis_taps(col, w, c0, nc);
  float sum = 0.0f;
  for (int ri = 0; ri < nr; ++ri) {
    const float wr = axis_weight(row, r0 + ri, h);
    for (int ci = 0; ci < nc; ++ci) {
      const float wc = axis_weight(col, c0 + ci, w);
      sum += (wr * wc) * src[((int64_t)(r0 + ri) * w + (c0 + ci)) * C + c];
    }
  }
  dst[(int64_t)i] = sum;
}

// Adjoint of down_value: value idx of level k gathers the gradient of the texels of level k + 1
// whose bins overlap it.
__device__ __forceinline__ void up_value(float* src, const float* dst, int C, int h, int w,
                                         int h2, int w2, uint32_t idx) {
  const uint32_t texel = idx / (uint32_t)C;
  const int c = (int)(idx - texel * (uint32_t)C);
  const int i = (int)(texel / (uint32_t)w), j = (int)(texel - (uint32_t)i * w);
  // Destination rows (cols) that can overlap source row i (col j).
  const int r_mid = (h & 1) ? (int)((int64_t)i * h2 / h) : i / 2;
  const int c_mid = (w & 1) ? (int)((int64_t)j * w2 / w) : j / 2;
  float sum = 0.0f;
  for (int r = max(r_mid - 1, 0); r <= min(r_mid + 1, h2 - 1); ++r) {
    const float wr = axis_weight(r, i, h);
    if (wr == 0.0f) continue;
    for (int cc = max(c_mid - 1, 0); cc <= min(c_mid + 1, w2 - 1); ++cc) {
      const float wc = axis_weight(cc, j, w);
      if (wc == 0.0f) continue;
      sum += (wr * wc) * dst[((int64_t)r * w2 + cc) * C + c];
    }
  }
  src[(int64_t)idx] += sum;
}

// Level lvl of (image, face) number `face_of`, image by image.
__device__ __forceinline__ float* level_of(float* texels, int64_t num_texels, int C,
                                           const MipLevels& L, int lvl, int64_t image, int face) {
  return texels + image * num_texels * C +
         (L.off[lvl] + (int64_t)face * L.h[lvl] * L.w[lvl]) * C;
}

// Level k + 1 from level k, one thread per destination texel and channel of all images and faces:
// `values` of them each, `count` (below 2^32, as any launch's threads) in all.
__global__ __launch_bounds__(256) void mip_down(float* texels, int C, int64_t num_texels,
                                                int faces, MipLevels L, int k, uint32_t values,
                                                uint32_t count) {
  const uint32_t thread = blockIdx.x * blockDim.x + threadIdx.x;
  if (thread >= count) return;
  const uint32_t which = thread / values, i = thread - which * values;
  const int64_t image = which / (uint32_t)faces;
  const int face = (int)(which % (uint32_t)faces);
  down_value(level_of(texels, num_texels, C, L, k, image, face),
             level_of(texels, num_texels, C, L, k + 1, image, face), C, L.h[k], L.w[k],
             L.w[k + 1], i);
}

// Adjoint of mip_down: one thread per source texel and channel.
__global__ __launch_bounds__(256) void mip_up(float* grad, int C, int64_t num_texels, int faces,
                                              MipLevels L, int k, uint32_t values,
                                              uint32_t count) {
  const uint32_t thread = blockIdx.x * blockDim.x + threadIdx.x;
  if (thread >= count) return;
  const uint32_t which = thread / values, i = thread - which * values;
  const int64_t image = which / (uint32_t)faces;
  const int face = (int)(which % (uint32_t)faces);
  up_value(level_of(grad, num_texels, C, L, k, image, face),
           level_of(grad, num_texels, C, L, k + 1, image, face), C, L.h[k], L.w[k], L.h[k + 1],
           L.w[k + 1], i);
}

// Levels k + 1 .. last from level k, one workgroup per (image, face): for levels so small that
// a launch each would be nearly all launch (kMipTailValues values). Odd sizes included.
constexpr int kMipTailThreads = 1024;

__global__ __launch_bounds__(kMipTailThreads) void mip_down_tail(float* texels, int C,
                                                                 int64_t num_texels, int faces,
                                                                 MipLevels L, int k, int last) {
  const int64_t image = blockIdx.x / (uint32_t)faces;
  const int face = (int)(blockIdx.x % (uint32_t)faces);
  for (int lvl = k; lvl < last; ++lvl) {
    const float* src = level_of(texels, num_texels, C, L, lvl, image, face);
    float* dst = level_of(texels, num_texels, C, L, lvl + 1, image, face);
    const uint32_t count = (uint32_t)(L.h[lvl + 1] * L.w[lvl + 1] * C);
    for (uint32_t i = threadIdx.x; i < count; i += blockDim.x)
      down_value(src, dst, C, L.h[lvl], L.w[lvl], L.w[lvl + 1], i);
    __syncthreads();  // the next level reads what the workgroup wrote
  }
}

// Adjoint of mip_down_tail.
__global__ __launch_bounds__(kMipTailThreads) void mip_up_tail(float* grad, int C,
                                                               int64_t num_texels, int faces,
                                                               MipLevels L, int k, int last) {
  const int64_t image = blockIdx.x / (uint32_t)faces;
  const int face = (int)(blockIdx.x % (uint32_t)faces);
  for (int lvl = last - 1; lvl >= k; --lvl) {
    float* src = level_of(grad, num_texels, C, L, lvl, image, face);
    const float* dst = level_of(grad, num_texels, C, L, lvl + 1, image, face);
    const uint32_t count = (uint32_t)(L.h[lvl] * L.w[lvl] * C);
    for (uint32_t i = threadIdx.x; i < count; i += blockDim.x)
      up_value(src, dst, C, L.h[lvl], L.w[lvl], L.h[lvl + 1], L.w[lvl + 1], i);
    __syncthreads();  // the next level reads what the workgroup wrote
  }
}

// ---- mip chain in tile stages ------------------------------------------------------------
//
// Where a level's sizes are divisible by 2^G (G >= 2), the next G levels halve exactly and each
// texel has exactly one parent: a workgroup then takes a tile of 2^G x 2^G texels of the bottom
// level through all G levels, keeping the levels in between in LDS, instead of one launch (and
// one pass over memory) per level. The arithmetic is mip_down's and mip_up's for even sizes:
// a texel is ((a / 4 + b / 4) + c / 4) + d / 4 of its children in row-major order, and in the
// adjoint a child adds a quarter of its parent's total.

// At most 32 x 32 bottom texels per tile (16 x 16 above it in LDS): a 1024^2 level gives 1024
// workgroups, and the chain above 32^2 is one more single-workgroup stage. (Tiles of 64 x 64
// gave a quarter as many workgroups and 32 KB of LDS each: mip chain 1024^2 x 4, built and
// folded back, 63 -> 53 us; tiles of 16 x 16 need a third stage, 66 us.)
constexpr int kMipStageLevels = 5;

// The stages work on elements of a texel: float4 when the channels come in fours on a 16-byte
// aligned buffer, Rgb for three channels, else single channels. Consecutive lanes take a texel's elements in turn, so
// that a wave's loads cover whole lines whatever the channel count (one lane per texel and
// group of four, a pass per group, at 1024^2 x 16: 199 us to build the chain and 178 to fold
// it; now 37 and 44).
__device__ __forceinline__ float quad_mean(float a, float b, float c, float d) {
  return ((0.25f * a + 0.25f * b) + 0.25f * c) + 0.25f * d;
}
__device__ __forceinline__ float4 quad_mean(float4 a, float4 b, float4 c, float4 d) {
  return make_float4(quad_mean(a.x, b.x, c.x, d.x), quad_mean(a.y, b.y, c.y, d.y),
                     quad_mean(a.z, b.z, c.z, d.z), quad_mean(a.w, b.w, c.w, d.w));
}
__device__ __forceinline__ float add_quarter(float own, float parent) {
  return own + 0.25f * parent;
}
__device__ __forceinline__ float4 add_quarter(float4 own, float4 parent) {
  return make_float4(add_quarter(own.x, parent.x), add_quarter(own.y, parent.y),
                     add_quarter(own.z, parent.z), add_quarter(own.w, parent.w));
}

// Three channels in one access, with no alignment but a float's (as three elements, the adjoint at
// 1024^2 took 26 us; this way 21).
struct Rgb {
  float x, y, z;
};
__device__ __forceinline__ Rgb quad_mean(Rgb a, Rgb b, Rgb c, Rgb d) {
  return {quad_mean(a.x, b.x, c.x, d.x), quad_mean(a.y, b.y, c.y, d.y),
          quad_mean(a.z, b.z, c.z, d.z)};
}
__device__ __forceinline__ Rgb add_quarter(Rgb own, Rgb parent) {
  return {add_quarter(own.x, parent.x), add_quarter(own.y, parent.y),
          add_quarter(own.z, parent.z)};
}

// Elements of a texel that a stage takes at a time (LDS: 20 KB), and the LDS of the levels of a
// tile 2^j texels across: even j in one buffer (at most 16 x 16), odd j in the other (8 x 8).
template <class V>
constexpr int kStageElements = std::is_same_v<V, Rgb> ? 1 : 64 / (int)sizeof(V);
template <class V>
struct MipStage {
  V even[256 * kStageElements<V>], odd[64 * kStageElements<V>];
  __device__ __forceinline__ V* side(int j) { return (j & 1) ? odd : even; }
};

// (texel, element) of a stage's element i, for NE elements per texel (0: ne, at run time).
template <int NE>
__device__ __forceinline__ void stage_element(int i, int ne, int& texel, int& e) {
  const uint32_t n = NE > 0 ? (uint32_t)NE : (uint32_t)ne;
  texel = (int)((uint32_t)i / n);
  e = i - texel * (int)n;
}

// The tile of this workgroup: (image, face) and tile coordinates in units of 2^G bottom texels.
struct MipTile {
  int64_t image;
  int face, tx, ty;
};

__device__ __forceinline__ MipTile mip_tile(const MipLevels& L, int k, int G, int faces) {
  const int tiles_x = L.w[k] >> G, tiles_y = L.h[k] >> G;
  int64_t b = blockIdx.x;
  MipTile T;
  T.tx = (int)(b % tiles_x);
  b /= tiles_x;
  T.ty = (int)(b % tiles_y);
  b /= tiles_y;
  T.face = (int)(b % faces);
  T.image = b / faces;
  return T;
}

// Levels k + 1 .. k + G from level k, one tile per workgroup. With `base` (k == 0 only), level
// 0 is read from there -- [images, faces * h * w, C], the layout of level 0 on its own -- and
// copied into the packed buffer on the way (each of its texels is read once). E: elements per
// texel, C in elements of type V.
template <class V, int NE>
__global__ __launch_bounds__(256) void mip_down_stage(V* texels, const V* base, int E,
                                                      int64_t num_texels, int faces,
                                                      MipLevels L, int k, int G) {
  __shared__ MipStage<V> stage;
  const MipTile T = mip_tile(L, k, G, faces);
  auto level_at = [&](int lvl) {
    return texels + (T.image * num_texels + L.off[lvl] + (int64_t)T.face * L.h[lvl] * L.w[lvl]) * E;
  };
  for (int e0 = 0; e0 < E; e0 += kStageElements<V>) {
    const int ne = min(kStageElements<V>, E - e0);
    {
      const int j = G - 1, side = 1 << j;  // the tile's side at level k + 1
      V* level = level_at(k) + e0;
      const V* src =
          base ? base + (T.image * faces + T.face) * (int64_t)L.h[0] * L.w[0] * E + e0 : level;
      V* dst = level_at(k + 1) + e0;
      const int64_t w = (int64_t)L.w[k] * E, w1 = (int64_t)L.w[k + 1] * E;
      V* out = stage.side(j);
#pragma unroll 2
      for (int i = threadIdx.x; i < side * side * ne; i += blockDim.x) {
        int texel, e;
        stage_element<NE>(i, ne, texel, e);
        const int r = T.ty * side + (texel >> j), c = T.tx * side + (texel & (side - 1));
        const int64_t at = 2 * r * w + (int64_t)(2 * c) * E + e;
        const V* p = src + at;
        const V v00 = p[0], v01 = p[E], v10 = p[w], v11 = p[w + E];
        if (base) {
          V* q = level + at;
          q[0] = v00;
          q[E] = v01;
          q[w] = v10;
          q[w + E] = v11;
        }
        const V o = quad_mean(v00, v01, v10, v11);
        dst[r * w1 + (int64_t)c * E + e] = o;
        out[i] = o;
      }
    }
    for (int lvl = k + 2; lvl <= k + G; ++lvl) {
      __syncthreads();
      const int j = k + G - lvl, side = 1 << j;
      const V* s = stage.side(j + 1);
      V* out = stage.side(j);
      V* dst = level_at(lvl) + e0;
      const int64_t wl = (int64_t)L.w[lvl] * E;
      for (int i = threadIdx.x; i < side * side * ne; i += blockDim.x) {
        int texel, e;
        stage_element<NE>(i, ne, texel, e);
        const int r = texel >> j, c = texel & (side - 1);
        const V* q = s + ((2 * r * 2 * side) + 2 * c) * ne + e;
        const V o = quad_mean(q[0], q[ne], q[2 * side * ne], q[(2 * side + 1) * ne]);
        dst[(T.ty * side + r) * wl + (int64_t)(T.tx * side + c) * E + e] = o;
        out[i] = o;
      }
    }
    __syncthreads();  // the next elements reuse the LDS
  }
}

// Adjoint of mip_down_stage: the totals of level k + G (final: the stages above ran first) fold
// down through levels k + G - 1 .. k of the tile, each texel adding a quarter of its parent's
// total to its own gradient, which becomes its total.
template <class V, int NE>
__global__ __launch_bounds__(256) void mip_up_stage(V* grad, int E, int64_t num_texels, int faces,
                                                    MipLevels L, int k, int G) {
  __shared__ MipStage<V> stage;
  const MipTile T = mip_tile(L, k, G, faces);
  auto level_at = [&](int lvl) {
    return grad + (T.image * num_texels + L.off[lvl] + (int64_t)T.face * L.h[lvl] * L.w[lvl]) * E;
  };
  for (int e0 = 0; e0 < E; e0 += kStageElements<V>) {
    const int ne = min(kStageElements<V>, E - e0);
    if ((int)threadIdx.x < ne)
      stage.side(0)[threadIdx.x] =
          level_at(k + G)[((int64_t)T.ty * L.w[k + G] + T.tx) * E + e0 + threadIdx.x];
    for (int lvl = k + G - 1; lvl >= k; --lvl) {
      __syncthreads();
      const int j = k + G - lvl, side = 1 << j;
      const V* s = stage.side(j - 1);
      V* out = stage.side(j);
      V* g = level_at(lvl) + e0;
      const int64_t wl = (int64_t)L.w[lvl] * E;
      // Four elements per thread and step, all loaded before the first is stored (the stores
      // go to the buffer the loads read: nothing else would keep the loads together).
      constexpr int kStep = 4;
      const int count = side * side * ne;
      for (int i0 = threadIdx.x; i0 < count; i0 += kStep * 256) {
        V own[kStep];
        V* at[kStep];
#pragma unroll
        for (int u = 0; u < kStep; ++u) {
          const int i = min(i0 + 256 * u, count - 1);
          int texel, e;
          stage_element<NE>(i, ne, texel, e);
          const int r = texel >> j, c = texel & (side - 1);
          at[u] = g + (T.ty * side + r) * wl + (int64_t)(T.tx * side + c) * E + e;
          own[u] = *at[u];
        }
#pragma unroll
        for (int u = 0; u < kStep; ++u) {
          const int i = i0 + 256 * u;
          if (i >= count) break;
          int texel, e;
          stage_element<NE>(i, ne, texel, e);
          const int r = texel >> j, c = texel & (side - 1);
          const V o = add_quarter(own[u], s[((r >> 1) * (side >> 1) + (c >> 1)) * ne + e]);
          *at[u] = o;
          if (lvl > k) out[i] = o;
        }
      }
    }
    __syncthreads();  // the next elements reuse the LDS
  }
}

// Calls f(element type tag, elements per texel as a constant (0: at run time)) for C channels at
// the given buffers.
template <typename F>
void stage_elements(int C, const void* texels, const void* base, F f) {
  using std::integral_constant;
  const bool wide = C % 4 == 0 &&
                    ((reinterpret_cast<uintptr_t>(texels) | reinterpret_cast<uintptr_t>(base)) &
                     15u) == 0;
  if (wide) {
    switch (C) {
      case 4: return f(float4(), integral_constant<int, 1>());
      case 8: return f(float4(), integral_constant<int, 2>());
      default:  // a whole number of full passes, or the count at run time
        return C % 16 == 0 ? f(float4(), integral_constant<int, 4>())
                           : f(float4(), integral_constant<int, 0>());
    }
  }
  switch (C) {
    case 1: return f(float(), integral_constant<int, 1>());
    case 2: return f(float(), integral_constant<int, 2>());
    case 3: return f(Rgb(), integral_constant<int, 1>());
    default: return f(float(), integral_constant<int, 0>());
  }
}

// Up to this many values of a level (per image and face), the rest of the chain is one
// workgroup's: it takes 4 values per thread at a time, in about a launch's time each (limits of
// 2048 to 16384 within 3 % of a step of 1500 x 1500 x 16: 722, 720 and 740 us).
constexpr int64_t kMipTailValues = 4096;

// Whether level k's values (per image and face) end the chain in one workgroup's levels. Not
// where there are many tiny ones: 100 k images of 3 x 3, built and folded back, 67 us level by
// level, 210 in workgroups of one wave; of 7 x 7 x 3 756 and 551, 16384 of 3 x 2 x 16 70 and 76.
bool tail_level(int64_t values, int64_t images) {
  return values <= kMipTailValues && (images <= 4096 || values > 128);
}

// Threads of a tail's workgroups: all of them while the workgroups are few enough to run at once
// (two to a CU); more workgroups finish sooner with fewer threads each (4096 images of
// 24 x 24 x 3: 341 us with 1024 threads, 225 with a thread per 16 values; 1024 images: 122 either).
int tail_threads(const MipLevels& L, int k, int channels, int64_t images) {
  if (images <= 512) return kMipTailThreads;
  const int64_t values = (int64_t)L.h[k] * L.w[k] * channels;
  return (int)(values / 16 / 64 + 1) * 64;  // at most 320
}

// Parts of a chain: part (k, G) builds levels k + 1 .. k + G, in one tile-stage launch when
// G >= 2, else (G == 1) with mip_down; the part at index `tail`, if any, is the last, with
// mip_down_tail.
struct MipPlan {
  int count;
  int tail;
  int k[DR_MAX_LEVELS], G[DR_MAX_LEVELS];
};

MipPlan mip_plan(const MipLevels& L, int num_levels, int channels, int64_t images) {
  MipPlan P{};
  P.tail = -1;
  for (int k = 0; k + 1 < num_levels;) {
    int G = 0;
    while (G < kMipStageLevels && k + G + 1 < num_levels && L.h[k] % (2 << G) == 0 &&
           L.w[k] % (2 << G) == 0)
      ++G;
    if (G < 2) G = 1;
    if (k + G + 1 < num_levels && tail_level((int64_t)L.h[k] * L.w[k] * channels, images)) {
      P.tail = P.count;  // more than one launch otherwise
      G = num_levels - 1 - k;
    }
    P.k[P.count] = k;
    P.G[P.count] = G;
    ++P.count;
    k += G;
  }
  return P;
}

int64_t stage_tiles(const MipLevels& L, int k, int G, int64_t images) {
  return images * (int64_t)(L.h[k] >> G) * (L.w[k] >> G);
}

// Whether every launch that builds the plan's levels (up: folds them back), and the copy of
// level 0 where one is needed, has fewer than 2^32 threads: the runtime does not refuse every
// larger one, but runs a part of its workgroups.
bool launchable(const MipPlan& P, const MipLevels& L, int channels, int64_t images, bool up,
                bool copied) {
  constexpr int64_t kLimit = (int64_t)1 << 32;
  auto values = [&](int k) { return images * L.h[k] * L.w[k] * channels + 255; };
  if (copied && values(0) >= kLimit) return false;
  for (int s = 0; s < P.count; ++s) {
    const int k = P.k[s], G = P.G[s];
    const int64_t threads = s == P.tail ? images * tail_threads(L, k, channels, images)
                            : G >= 2    ? stage_tiles(L, k, G, images) * 256
                                        : values(up ? k : k + 1);
    if (threads >= kLimit) return false;
  }
  return true;
}

bool valid_levels(int num_levels, const int32_t* h, const int32_t* w, const int64_t* off) {
  if (num_levels < 1 || num_levels > DR_MAX_LEVELS || !h || !w || !off) return false;
  for (int k = 0; k < num_levels; ++k)
    if (h[k] <= 0 || w[k] <= 0 || off[k] < 0) return false;
  for (int k = 0; k + 1 < num_levels; ++k)
    if (h[k + 1] != (h[k] + 1) / 2 || w[k + 1] != (w[k] + 1) / 2) return false;
  return true;
}

MipLevels copy_levels(int n, const int32_t* h, const int32_t* w, const int64_t* off) {
  MipLevels L{};
  for (int k = 0; k < n; ++k) {
    L.h[k] = h[k];
    L.w[k] = w[k];
    L.off[k] = off[k];
  }
  return L;
}

// Calls f(channels (0: more than 4), cube, filter, boundary) with each as a compile-time constant
// (std::integral_constant), from a's channel count and modes (checked by valid_args): the
// kernels are compiled for every combination, each without the other modes' code.
template <typename F>
int texture_modes(const DrTextureArgs& a, F f) {
  auto with_boundary = [&](auto nc, auto filter) {
    using std::integral_constant;
    switch (a.boundary) {
      case DR_BOUNDARY_CUBE:
        return f(nc, std::true_type(), filter, integral_constant<int, DR_BOUNDARY_CUBE>());
      case DR_BOUNDARY_WRAP:
        return f(nc, std::false_type(), filter, integral_constant<int, DR_BOUNDARY_WRAP>());
      case DR_BOUNDARY_CLAMP:
        return f(nc, std::false_type(), filter, integral_constant<int, DR_BOUNDARY_CLAMP>());
      default:
        return f(nc, std::false_type(), filter, integral_constant<int, DR_BOUNDARY_ZERO>());
    }
  };
  auto with_filter = [&](auto nc) {
    using std::integral_constant;
    switch (a.filter) {
      case DR_FILTER_NEAREST:
        return with_boundary(nc, integral_constant<int, DR_FILTER_NEAREST>());
      case DR_FILTER_LINEAR:
        return with_boundary(nc, integral_constant<int, DR_FILTER_LINEAR>());
      case DR_FILTER_MIP_NEAREST:
        return with_boundary(nc, integral_constant<int, DR_FILTER_MIP_NEAREST>());
      default:
        return with_boundary(nc, integral_constant<int, DR_FILTER_MIP_LINEAR>());
    }
  };
  return exact_channels(a.channels, with_filter);
}

bool valid_args(const DrTextureArgs* a) {
  if (!a || !a->texels || !a->uv || a->batch < 0 || a->height <= 0 || a->width <= 0) return false;
  // Texel indices within an image's packed buffer are 32-bit.
  if (a->num_texels < 1 || a->num_texels >= 0xffffffffLL) return false;
  if (a->channels <= 0 || a->tex_batch < 1 || a->num_levels < 1 || a->num_levels > DR_MAX_LEVELS)
    return false;
  if (a->filter < 0 || a->filter > 3 || a->boundary < 0 || a->boundary > 3) return false;
  if ((a->boundary == DR_BOUNDARY_CUBE) != (a->faces == 6)) return false;
  if (a->faces != 1 && a->faces != 6) return false;
  for (int k = 0; k < a->num_levels; ++k)
    if (a->level_height[k] <= 0 || a->level_width[k] <= 0) return false;
  return true;
}

}  // namespace
}  // namespace dr

using namespace dr;

extern "C" int dr_texture_forward(const DrTextureArgs* a, float* out, void* stream) {
  if (!valid_args(a) || !out) return DR_ERR_ARGUMENT;
  const int64_t pixels = (int64_t)a->batch * a->height * a->width;
  if (pixels == 0) return DR_OK;
  const DrTextureArgs args = *a;
  return texture_modes(args, [&](auto nc, auto cube, auto filter, auto boundary) {
    constexpr int NC = decltype(nc)::value, FILTER = decltype(filter)::value;
    constexpr int BOUNDARY = decltype(boundary)::value;
    constexpr bool CUBE = decltype(cube)::value;
    const int blocks = blocks_for(pixels, 256);
    const hipStream_t st = (hipStream_t)stream;
    if constexpr (NC > 0)
      tex_fwd_kernel<NC, CUBE, FILTER, BOUNDARY><<<blocks, 256, 0, st>>>(args, out);
    else
      tex_fwd_wide_kernel<CUBE, FILTER, BOUNDARY><<<blocks, 256, 0, st>>>(args, out);
    return launch_status();
  });
}

extern "C" int dr_texture_backward(const DrTextureArgs* a, const float* grad_out,
                                   float* grad_texels, float* grad_uv, float* grad_uv_da,
                                   float* grad_bias, void* stream) {
  if (!valid_args(a) || !grad_out) return DR_ERR_ARGUMENT;
  const int64_t pixels = (int64_t)a->batch * a->height * a->width;
  if (pixels == 0) return DR_OK;
  if ((int64_t)a->tex_batch * a->num_texels >= 0xffffffffLL) return DR_ERR_ARGUMENT;
  const DrTextureArgs args = *a;
  const int64_t blocks = tile_blocks(args.batch, args.height, args.width);
  float* g_da = args.uv_da ? grad_uv_da : nullptr;
  float* g_bias = args.bias ? grad_bias : nullptr;
  return texture_modes(args, [&](auto nc, auto cube, auto filter, auto boundary) {
    // Cube maps read the filter at run time, one kernel per channel count for all four. Fixed when
    // compiling, three channels on four 1024^2 images (backward alone, us): trilinear 237 / 237
    // (six channels 424 / 453), bilinear 420 / 418, nearest 101 / 98, bilinear in the nearest
    // level 172 / 149.
    constexpr bool kCube = decltype(cube)::value;
    constexpr int kFilter = kCube ? kAnyMode : decltype(filter)::value;
    tex_bwd_kernel<decltype(nc)::value, kCube, kFilter, decltype(boundary)::value>
        <<<blocks, 256, 0, (hipStream_t)stream>>>(args, grad_out, grad_texels, grad_uv, g_da,
                                                  g_bias);
    return launch_status();
  });
}

// Copies level 0 from its own array into the packed buffer (when no tile stage does it):
// `count` values, base_values per batch entry of `base`, packed_values per entry of `texels`.
__global__ __launch_bounds__(256) void mip_copy_base(float* texels, const float* base,
                                                     int64_t packed_values, int64_t base_values,
                                                     int64_t count) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const int64_t image = i / base_values, v = i - image * base_values;
  texels[image * packed_values + v] = base[i];
}

extern "C" int dr_mip_build(float* texels, const float* base, int32_t tex_batch,
                            int32_t channels, int64_t num_texels, int32_t faces,
                            int32_t num_levels, const int32_t* level_height,
                            const int32_t* level_width, const int64_t* level_offset,
                            void* stream) {
  if (!texels || tex_batch < 1 || channels < 1 || (faces != 1 && faces != 6) ||
      !valid_levels(num_levels, level_height, level_width, level_offset))
    return DR_ERR_ARGUMENT;
  const MipLevels L = copy_levels(num_levels, level_height, level_width, level_offset);
  const int64_t images = (int64_t)tex_batch * faces;
  const MipPlan P = mip_plan(L, num_levels, channels, images);
  const int64_t base_texels = (int64_t)faces * L.h[0] * L.w[0];
  if (base != nullptr && base_texels > num_texels) return DR_ERR_ARGUMENT;
  // Level 0 from `base`: the first tile stage copies it as it reads it; otherwise a copy first.
  const bool staged_copy = base != nullptr && P.count > 0 && P.G[0] >= 2 && P.tail != 0;
  if (!launchable(P, L, channels, images, false, base != nullptr && !staged_copy))
    return DR_ERR_ARGUMENT;
  if (base != nullptr && !staged_copy) {
    const int64_t count = (int64_t)tex_batch * base_texels * channels;
    mip_copy_base<<<blocks_for(count, 256), 256, 0, (hipStream_t)stream>>>(
        texels, base, num_texels * channels, base_texels * channels, count);
  }
  for (int s = 0; s < P.count; ++s) {
    const int k = P.k[s], G = P.G[s];
    if (s == P.tail) {
      mip_down_tail<<<(unsigned)images, tail_threads(L, k, channels, images), 0,
                      (hipStream_t)stream>>>(
          texels, channels, num_texels, faces, L, k, k + G);
      continue;
    }
    if (G >= 2) {
      const float* from = s == 0 && staged_copy ? base : nullptr;
      stage_elements(channels, texels, from, [&](auto v, auto ne) {
        using V = decltype(v);
        mip_down_stage<V, decltype(ne)::value>
            <<<(unsigned)stage_tiles(L, k, G, images), 256, 0, (hipStream_t)stream>>>(
                (V*)texels, (const V*)from, channels / (int)(sizeof(V) / 4), num_texels, faces, L,
                k, G);
      });
      continue;
    }
    const int64_t values = (int64_t)L.h[k + 1] * L.w[k + 1] * channels;
    mip_down<<<blocks_for(images * values, 256), 256, 0, (hipStream_t)stream>>>(
        texels, channels, num_texels, faces, L, k, (uint32_t)values, (uint32_t)(images * values));
  }
  return launch_status();
}

extern "C" int dr_mip_build_backward(float* grad_texels, int32_t tex_batch, int32_t channels,
                                     int64_t num_texels, int32_t faces, int32_t num_levels,
                                     const int32_t* level_height, const int32_t* level_width,
                                     const int64_t* level_offset, void* stream) {
  if (!grad_texels || tex_batch < 1 || channels < 1 || (faces != 1 && faces != 6) ||
      !valid_levels(num_levels, level_height, level_width, level_offset))
    return DR_ERR_ARGUMENT;
  const MipLevels L = copy_levels(num_levels, level_height, level_width, level_offset);
  const int64_t images = (int64_t)tex_batch * faces;
  const MipPlan P = mip_plan(L, num_levels, channels, images);
  if (!launchable(P, L, channels, images, true, false)) return DR_ERR_ARGUMENT;
  for (int s = P.count - 1; s >= 0; --s) {
    const int k = P.k[s], G = P.G[s];
    if (s == P.tail) {
      mip_up_tail<<<(unsigned)images, tail_threads(L, k, channels, images), 0,
                    (hipStream_t)stream>>>(
          grad_texels, channels, num_texels, faces, L, k, k + G);
      continue;
    }
    if (G >= 2) {
      stage_elements(channels, grad_texels, nullptr, [&](auto v, auto ne) {
        using V = decltype(v);
        mip_up_stage<V, decltype(ne)::value>
            <<<(unsigned)stage_tiles(L, k, G, images), 256, 0, (hipStream_t)stream>>>(
                (V*)grad_texels, channels / (int)(sizeof(V) / 4), num_texels, faces, L, k, G);
      });
      continue;
    }
    const int64_t values = (int64_t)L.h[k] * L.w[k] * channels;
    mip_up<<<blocks_for(images * values, 256), 256, 0, (hipStream_t)stream>>>(
        grad_texels, channels, num_texels, faces, L, k, (uint32_t)values,
        (uint32_t)(images * values));
  }
  return launch_status();
}
