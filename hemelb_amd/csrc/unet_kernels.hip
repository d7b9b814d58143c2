// HIP kernels of the warm-start 3D U-Net (gfx950): 3x3x3 convolutions as
// implicit GEMMs on bfloat16 MFMA with binary32 accumulation (forward,
// backward-data through the same kernel with flipped, transposed weights,
// backward-weight with fixed-order partial sums), and the elementwise
// pieces of training: ReLU, 2x2x2 mean pooling, 2x nearest upsampling,
// channel concatenation, masked MSE, bias and head reductions, Adam.
//
// Tensors are channels-last: element (p, c) of a [P][C] tensor, where p
// enumerates (n, d, h, w) with w fastest.  bfloat16 values are stored as
// uint16 bit patterns.  Convolution weights are [27][Cout][Cin], tap
// t = 9*kd + 3*kh + kw for offsets (kd-1, kh-1, kw-1).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "unet_internal.h"
#include "unet_plan.h"

namespace hlbn {
namespace {

typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(uint16_t b) {
  return __uint_as_float((uint32_t)b << 16);
}
// Round to nearest even (finite inputs).
__device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

struct Grid3 {
  int N, D, H, W;
  __host__ __device__ __forceinline__ int64_t P() const { return (int64_t)N * D * H * W; }
};

// Coordinates (w, h, d) of position p inside its sample (P < 2^31).
struct Coord3 {
  int w, h, d;
};
__device__ __forceinline__ Coord3 coord_of(const Grid3& g, int p) {
  const int r1 = p / g.W, r2 = r1 / g.H;
  return Coord3{p - r1 * g.W, r1 - r2 * g.H, r2 % g.D};
}
// The coordinates of position p + step from those of p (no division).
__device__ __forceinline__ void advance(const Grid3& g, Coord3& c, int step) {
  c.w += step;
  while (c.w >= g.W) {
    c.w -= g.W;
    if (++c.h == g.H) {
      c.h = 0;
      if (++c.d == g.D) c.d = 0;
    }
  }
}

// --------------------------------------------------------------------------
// Forward 3x3x3 convolution (also backward-data): an implicit GEMM on
// gfx950's v_mfma_f32_16x16x32_bf16 with M = positions, N = output channels
// and K = 27 taps x input channels.  One wave computes MT tiles of 16
// consecutive positions x NT tiles of 16 output channels.  K advances in
// steps of 32: two half-steps of 16 (tap, 16-channel group) pairs, tap-major,
// the 28th tap of an odd count padded with zeros.  Lane l supplies row l%16
// of A (its position) and column l%16 of B (its output channel) with the 8
// K-values 8*(l/16)..+7, each one 16-byte load of 8 consecutive channels
// (channels-last activations, [27][Cout][Cin] weights); it receives rows
// 4*(l/16)..+3 of column l%16.  An A fragment serves NT MFMAs, a B fragment
// MT.  Coarse levels, with few positions and long K, split K over
// gridDim.y slices of `hpw` half-steps: each slice writes its raw sums to
// ws[slice][position][co] and k_conv_reduce adds them in slice order.
// --------------------------------------------------------------------------
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x8_t load8(const uint16_t* p) {
  return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(p));
}

template <int MT, int NT>
__global__ __launch_bounds__(256) void k_conv_fwd(Grid3 g, const uint16_t* __restrict__ x,
                                                  int ci, const uint16_t* __restrict__ w,
                                                  const float* __restrict__ bias, int co,
                                                  float* __restrict__ y32,
                                                  uint16_t* __restrict__ y16, int yc,
                                                  int yoff, int relu, int hpw,
                                                  float* __restrict__ ws) {
  const int lane = threadIdx.x & 63;
  const int64_t wave = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int ngroups = (co / 16 + NT - 1) / NT;
  const int64_t pgroup = wave / ngroups;
  const int tile0 = (int)(wave % ngroups) * NT;
  const int64_t P = g.P();
  const int64_t p0 = pgroup * 16 * MT;
  if (p0 >= P) return;
  const int row = lane & 15, q = lane >> 4;
  const int half = q >> 1, sub = q & 1;
  int64_t pp[MT];
  bool pv[MT];
  Coord3 pc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    pp[m] = p0 + 16 * m + row;
    pv[m] = pp[m] < P;
    pc[m] = pv[m] ? coord_of(g, (int)pp[m]) : Coord3{0, 0, 0};
  }
  f32x4_t acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[m][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int cpt = ci / 16;       // 16-channel groups per tap
  const int split = blockIdx.y;
  const int hbeg = split * hpw;
  const int nhalf = min(27 * cpt, hbeg + hpw);  // half-steps of 16 K-values
  const bf16x8_t zero = __builtin_bit_cast(bf16x8_t, u32x4_t{0u, 0u, 0u, 0u});
  for (int h0 = hbeg; h0 < nhalf; h0 += 2) {
    const int h = h0 + half;
    const bool hv = h < nhalf;
    const int t = hv ? h / cpt : 0;
    const int c = (h - t * cpt) * 16 + 8 * sub;
    const int dz = t / 9 - 1, dyy = (t / 3) % 3 - 1, dx = t % 3 - 1;
    const int64_t off = ((int64_t)dz * g.H + dyy) * g.W + dx;
    bf16x8_t a[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const bool inside = hv && pv[m] && (unsigned)(pc[m].d + dz) < (unsigned)g.D &&
                          (unsigned)(pc[m].h + dyy) < (unsigned)g.H &&
                          (unsigned)(pc[m].w + dx) < (unsigned)g.W;
      a[m] = inside ? load8(x + (pp[m] + off) * ci + c) : zero;
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int oc = (tile0 + j) * 16 + row;
      const bf16x8_t b = (hv && oc < co) ? load8(w + ((int64_t)t * co + oc) * ci + c) : zero;
#pragma unroll
      for (int m = 0; m < MT; ++m)
        acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], b, acc[m][j], 0, 0, 0);
    }
  }
  if (ws) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int oc = (tile0 + j) * 16 + row;
      if (oc >= co) continue;
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int64_t pos = p0 + 16 * m + 4 * q + r;
          if (pos < P) ws[((int64_t)split * P + pos) * co + oc] = acc[m][j][r];
        }
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int oc = (tile0 + j) * 16 + row;
    if (oc >= co) continue;
    const float bv = bias ? bias[oc] : 0.f;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t pos = p0 + 16 * m + 4 * q + r;
        if (pos >= P) continue;
        float v = acc[m][j][r] + bv;
        if (relu) v = v > 0.f ? v : 0.f;
        const int64_t o = pos * yc + yoff + oc;
        if (y32) y32[o] = v;
        if (y16) y16[o] = f2bf(v);
      }
  }
}

// --------------------------------------------------------------------------
// The same convolution from LDS.  k_conv_fwd loads every A fragment from
// global memory, 27 times per activation, each with its own address and
// bounds arithmetic: 67-144 us a layer at 64^3 x 4, 10x what the bytes or the
// matrix cores need.  Here a workgroup of four waves stages a BD x BH x BW box
// of positions and its one-voxel halo, all input channels, once, as planes of
// 8 channels ([plane][position][8]: the 16 positions that one quarter of the
// wave reads are 256 contiguous bytes, one pass over the banks), and reads
// every tap's fragment from there at a constant offset.  Positions outside the volume are
// staged as zeros, so the K loop has no tests.  The weights stream from the
// caches, one K step (even group counts: one tap) ahead.
//
// Waves: WM along positions x 4 / WM along output channels, each MT tiles of
// 16 positions x NT tiles of 16 channels.  The product is formed transposed
// (A = weights, B = positions), so that a lane ends with 4 consecutive
// channels of one position and stores them at once.
//
// The input may come in two parts: the first `cu` channels from `xu`, a
// tensor of half the resolution (read at (d/2, h/2, w/2): nearest
// upsampling), the others from x.
//
// K runs as in k_conv_fwd, in the same steps and slices: the partial sum of
// `kps` steps is added to the total after each slice, so the results are the
// same bits whichever kernel runs.
//
// Measured at 64^3 x 4 (k_conv_fwd before): 16 -> 16 channels 67 -> 25 us
// (575 TF/s; its 67 MB take 13), 48 -> 16 147 -> 75, 16 -> 48 in binary32 144
// -> 66 (its bytes take 45), 96 -> 32 at 32^3 106 -> 59; all convolutions and
// data gradients of a training iteration 1.65 -> 0.63 ms.  No unit is near its
// limit now: by the counters the LDS is active for 9 to 26 % of the cycles and
// the matrix cores for 5 to 32 %, and waves wait 36 to 61 % of their time, for
// the box, staged before its products, and for the weights, with one or two
// workgroups a CU to cover it.
// --------------------------------------------------------------------------
template <int I, int N, typename F>
__device__ __forceinline__ void sfor(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    sfor<I + 1, N>(f);
  }
}

// 16 zero bytes, the source of LDS pieces outside the volume.
__device__ const uint16_t zero_piece[8] __attribute__((aligned(16))) = {0};

// 16 bytes from the lane's global address to lds + 16 * lane (lds the same in
// all lanes), without passing through registers; complete after
// wait_for_loads() and a barrier.
__device__ __forceinline__ void load_to_lds(const uint16_t* p, void* lds) {
  __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) const void*)p,
                                   (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}
__device__ __forceinline__ void wait_for_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// x / D for 0 <= x < LIMIT by a 24-bit product and a shift (full-rate vector
// instructions; the compiler's exact division multiplies in 32 x 32 bits at a
// quarter of that rate).
template <int D, int LIMIT>
__device__ __forceinline__ int small_div(int x) {
  constexpr unsigned kMul = (1u << 20) / D + 1;
  static_assert([] {
    for (unsigned v = 0; v < (unsigned)LIMIT; ++v)
      if (((v * kMul) >> 20) != v / D || v * kMul >= (1ull << 32)) return false;
    return kMul < (1u << 24) && LIMIT <= (1 << 12);
  }(), "inexact");
  return (int)(__umul24((unsigned)x, kMul) >> 20);
}

// Where a lane's piece of a halo box lies: its coordinates in the box, and
// whether and where the position is in the volume, for a box whose first halo
// position is (d, h, w) of sample n (possibly -1).
struct HaloPos {
  int d, h, w;
};
template <int HH, int HW, int LIMIT>
__device__ __forceinline__ HaloPos halo_pos(int pos) {
  const int r = small_div<HW, LIMIT>(pos), d = small_div<HH, LIMIT>(r);
  return HaloPos{d, r - d * HH, pos - r * HW};
}
__device__ __forceinline__ bool halo_inside(const Grid3& g, const HaloPos& o, int d, int h, int w) {
  return (unsigned)(d + o.d) < (unsigned)g.D && (unsigned)(h + o.h) < (unsigned)g.H &&
         (unsigned)(w + o.w) < (unsigned)g.W;
}
// Offset of the position from the box's first one, in positions.
__device__ __forceinline__ int halo_offset(const Grid3& g, const HaloPos& o) {
  return __mul24(__mul24(o.d, g.H) + o.h, g.W) + o.w;
}
// Index of its parent in the tensor of half the resolution.
__device__ __forceinline__ int halo_parent(const Grid3& g, const HaloPos& o, int n, int d, int h,
                                           int w) {
  return ((n * (g.D / 2) + (d + o.d) / 2) * (g.H / 2) + (h + o.h) / 2) * (g.W / 2) + (w + o.w) / 2;
}

struct ConvSrc {
  const uint16_t* x;    // [P][ci - cu]
  const uint16_t* xu;   // [P/8][cu], or null
  int cu;
};

template <int NG, int NT, int MT, int WM, int BD, int BH, int BW>
struct ConvBox {
  static constexpr int WN = 4 / WM;
  static constexpr int HH = BH + 2, HW = BW + 2, NPOS = (BD + 2) * HH * HW;
  static constexpr int PB = (NPOS + 63) / 64;       // 64-position chunks of a plane
  static constexpr int PLANE = PB * 1024;           // bytes of one 8-channel plane
  static constexpr int RPT = 16 / BW;               // rows of w per 16-position tile
  static constexpr int LDS = 2 * NG * PLANE;
  static_assert(BD * BH * BW == 16 * MT * WM, "box and waves disagree");
  static_assert(BW == 16 || (BW == 8 && BH % 2 == 0), "tiles are rows of w");
  static constexpr int TPD = BH / RPT;              // tiles per d plane
  static_assert(MT % TPD == 0 || TPD % MT == 0, "a wave's tiles at constant offsets");
  // halo position of the first site of tile m, relative to the wave's first
  static constexpr int tile_off(int m) { return (m / TPD) * HH * HW + (m % TPD) * RPT * HW; }
  static constexpr int tap_off(int t) { return ((t / 9) * HH + (t / 3) % 3) * HW + t % 3; }
  // workgroups (waves per SIMD) a CU's 160 KB of LDS has room for, at most 2
  static constexpr int WAVES = 163840 / LDS < 2 ? 163840 / LDS : 2;
  // byte offset of half-step h (tap, 16-channel group)
  static constexpr int half_off(int h) { return (h % NG) * 2 * PLANE + tap_off(h / NG) * 16; }
};

template <int NG, int NT, int MT, int WM, int BD, int BH, int BW, bool SLICES>
__global__ __launch_bounds__(256, (ConvBox<NG, NT, MT, WM, BD, BH, BW>::WAVES)) void k_conv_box(Grid3 g, ConvSrc src,
                                                  const uint16_t* __restrict__ w,
                                                  const float* __restrict__ bias, int co,
                                                  float* __restrict__ y32,
                                                  uint16_t* __restrict__ y16, int yc, int yoff,
                                                  int relu, int kps) {
  using B = ConvBox<NG, NT, MT, WM, BD, BH, BW>;
  constexpr int ci = 16 * NG;
  __shared__ __attribute__((aligned(16))) unsigned char lds[B::LDS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = lane & 15, q = lane >> 4, half = q >> 1, sub = q & 1;
  const int nbw = (g.W + BW - 1) / BW, nbh = (g.H + BH - 1) / BH, nbd = (g.D + BD - 1) / BD;
  int b = blockIdx.x;
  const int w0 = (b % nbw) * BW;
  b /= nbw;
  const int h0 = (b % nbh) * BH;
  b /= nbh;
  const int d0 = (b % nbd) * BD, n = b / nbd;
  const int wm = wv % WM, wn = wv / WM;
  const int ntiles = co / 16;
  const int tile0 = (blockIdx.y * B::WN + wn) * NT;
  // the wave's first position, the lane's row inside a tile
  constexpr int TPD = B::TPD;
  const int t0 = wm * MT, bd = t0 / TPD, bh = (t0 % TPD) * B::RPT;
  const int rh = row / BW, rw = row % BW;
  const int abase = ((bd * B::HH + bh + rh) * B::HW + rw) * 16 + sub * B::PLANE;
  const uint16_t* wp[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
    wp[j] = w + (int64_t)((min(tile0 + j, ntiles - 1)) * 16 + row) * ci + sub * 8;
  const bf16x8_t zero = __builtin_bit_cast(bf16x8_t, u32x4_t{0u, 0u, 0u, 0u});
  auto lds8 = [&](int off) {
    return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(lds + off));
  };
  // Weights are loaded a chunk of K steps ahead of their use (their latency is
  // hundreds of cycles, a step MT * NT * 16); the first chunk before staging.
  // Even NG: a K step is two groups of one tap and a chunk the three taps of
  // one (kd, kh).  Odd NG: a step may straddle two taps.
  constexpr bool kEven = NG % 2 == 0;
  constexpr int NH = 27 * NG, KS = (NH + 1) / 2;
  constexpr int KC = kEven ? 3 * NG / 2 : NG == 1 && NT == 1 ? KS : NT == 1 ? 7 : 10 / NT;
  constexpr int kChunks = (KS + KC - 1) / KC;
  const int64_t tap = (int64_t)co * ci;
  bf16x8_t bn[KC][NT];
  auto load_chunk = [&](auto first) {   // odd NG: constant first step
    sfor<0, KC>([&](auto ki) {
      constexpr int k = decltype(first)::value + decltype(ki)::value;
      constexpr int ha = 2 * k, hb = ha + 1 < NH ? ha + 1 : ha;
      if constexpr (ha < NH) {
        const int64_t off = half ? (hb / NG) * tap + (hb % NG) * 16 : (ha / NG) * tap + (ha % NG) * 16;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          bn[decltype(ki)::value][j] = load8(wp[j] + off);
          if (ha + 1 >= NH && half) bn[decltype(ki)::value][j] = zero;
        }
      }
    });
  };
  auto load_row = [&](int r) {          // even NG: the taps 3r .. 3r+2
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int k = 0; k < NG / 2; ++k)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          bn[x * (NG / 2) + k][j] = load8(wp[j] + (3 * r + x) * tap + k * 32 + half * 16);
  };
  if constexpr (kEven) load_row(0);
  else load_chunk(std::integral_constant<int, 0>{});
  // Stage the halo box: 16 bytes per lane straight into LDS, every load in
  // flight at once (through registers, in two or three batches, staging cost
  // as much as the products).  A wave takes the 8-channel pieces of 64
  // positions, its neighbours the same positions' other pieces; positions
  // outside the volume load zeros.
  {
    const int cx = ci - src.cu;
    const int dz = d0 - 1, hz = h0 - 1, wz = w0 - 1;
    const int64_t first = (((int64_t)n * g.D + dz) * g.H + hz) * g.W + wz;
#pragma unroll
    for (int r = 0; r < (2 * NG * B::PB + 3) / 4; ++r) {
      const int chunk = r * 4 + wv;
      if (chunk < 2 * NG * B::PB) {
        const int block = chunk / (2 * NG), piece = chunk % (2 * NG), c = piece * 8;
        const HaloPos o = halo_pos<B::HH, B::HW, B::PB * 64>(block * 64 + lane);
        const uint16_t* p;
        if (c < src.cu)   // the same for the whole wave
          p = src.xu + halo_parent(g, o, n, dz, hz, wz) * src.cu + c;
        else
          p = src.x + first * cx + c - src.cu + __mul24(halo_offset(g, o), cx);
        load_to_lds(halo_inside(g, o, dz, hz, wz) ? p : zero_piece,
                    lds + piece * B::PLANE + block * 1024);
      }
    }
  }
  wait_for_loads();
  __syncthreads();
  if (tile0 >= ntiles) return;
  f32x4_t acc[MT][NT], total[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[m][j] = total[m][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // SLICES: a scalar branch after every K step.  It ends the block of code that
  // the compiler schedules, so the next step's fragments are read before it;
  // without slices the steps are one block (16 -> 16 channels at 64^3 x 4: 28.0
  // us with the branches, 25.3 without).
  int left = kps;  // K steps left in the slice
  auto products = [&](const bf16x8_t (&a)[MT], const bf16x8_t (&b)[NT]) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[m], acc[m][j], 0, 0, 0);
    if constexpr (SLICES) {
      if (--left == 0) {
        left = kps;
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            total[m][j] += acc[m][j];
            acc[m][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
          }
      }
    }
  };
  bf16x8_t an[MT];  // SLICES: the next step's fragments
  if constexpr (kEven) {
    const int a0 = abase + half * 2 * B::PLANE;
    auto fragments = [&](int at, int k, bf16x8_t (&a)[MT]) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
        a[m] = lds8(at + (k / (NG / 2)) * 16 + 4 * (k % (NG / 2)) * B::PLANE + B::tile_off(m) * 16);
    };
    if constexpr (SLICES) fragments(a0, 0, an);
#pragma unroll 1
    for (int r = 0; r < 9; ++r) {
      bf16x8_t bw[KC][NT];
#pragma unroll
      for (int k = 0; k < KC; ++k)
#pragma unroll
        for (int j = 0; j < NT; ++j) bw[k][j] = bn[k][j];
      const int rn = min(r + 1, 8);
      load_row(rn);
      const int at = a0 + (r / 3 * B::HH + r % 3) * B::HW * 16;
      const int next = a0 + (rn / 3 * B::HH + rn % 3) * B::HW * 16;
#pragma unroll
      for (int k = 0; k < KC; ++k) {
        bf16x8_t a[MT];
        if constexpr (SLICES) {
#pragma unroll
          for (int m = 0; m < MT; ++m) a[m] = an[m];
          if (k + 1 < KC) fragments(at, k + 1, an);
          else fragments(next, 0, an);
        } else {
          fragments(at, k, a);
        }
        products(a, bw[k]);
      }
    }
  } else {
    // every offset is a constant, plus the lane's half times one of a few
    // differences
    auto fragments = [&](auto ki, bf16x8_t (&a)[MT]) {
      constexpr int ha = 2 * decltype(ki)::value, hb = ha + 1 < NH ? ha + 1 : ha;
      constexpr int oa = B::half_off(ha), diff = B::half_off(hb) - oa;
      const int at = abase + half * diff;
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        a[m] = lds8(at + oa + B::tile_off(m) * 16);
        if (ha + 1 >= NH && half) a[m] = zero;  // the last step's second half
      }
    };
    if constexpr (SLICES) fragments(std::integral_constant<int, 0>{}, an);
    sfor<0, kChunks>([&](auto ch) {
      constexpr int first = decltype(ch)::value * KC;
      bf16x8_t bw[KC][NT];
#pragma unroll
      for (int k = 0; k < KC; ++k)
#pragma unroll
        for (int j = 0; j < NT; ++j) bw[k][j] = bn[k][j];
      if constexpr (first + KC < KS) load_chunk(std::integral_constant<int, first + KC>{});
      sfor<0, KC>([&](auto ki) {
        constexpr int step = first + decltype(ki)::value;
        if constexpr (step < KS) {
          bf16x8_t a[MT];
          if constexpr (SLICES) {
#pragma unroll
            for (int m = 0; m < MT; ++m) a[m] = an[m];
            if constexpr (step + 1 < KS) fragments(std::integral_constant<int, step + 1>{}, an);
          } else {
            fragments(std::integral_constant<int, step>{}, a);
          }
          products(a, bw[decltype(ki)::value]);
        }
      });
    });
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int tile = t0 + m;
    const int d = d0 + tile / TPD, h = h0 + (tile % TPD) * B::RPT + rh, x = w0 + rw;
    if (d >= g.D || h >= g.H || x >= g.W) continue;
    const int64_t o = (int64_t)(((n * g.D + d) * g.H + h) * g.W + x) * yc + yoff + 4 * q;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      if (tile0 + j >= ntiles) continue;
      const int c = (tile0 + j) * 16;
      f32x4_t v = total[m][j] + acc[m][j];
      if (bias) v += *reinterpret_cast<const f32x4_t*>(bias + c + 4 * q);
      if (relu)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = v[r] > 0.f ? v[r] : 0.f;
      if (y32) *reinterpret_cast<f32x4_t*>(y32 + o + c) = v;
      if (y16) {
        ushort4 p;
        p.x = f2bf(v[0]);
        p.y = f2bf(v[1]);
        p.z = f2bf(v[2]);
        p.w = f2bf(v[3]);
        *reinterpret_cast<ushort4*>(y16 + o + c) = p;
      }
    }
  }
}

// y = (relu)(sum over the K slices of ws, in slice order, + bias).
__global__ void k_conv_reduce(int64_t P, int co, int nsplit, const float* __restrict__ ws,
                              const float* __restrict__ bias, int relu,
                              float* __restrict__ y32, uint16_t* __restrict__ y16, int yc,
                              int yoff) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P * co) return;
  const int oc = (int)(i % co);
  const int64_t pos = i / co;
  float v = 0.f;
  for (int k = 0; k < nsplit; ++k) v += ws[(int64_t)k * P * co + i];
  v += bias ? bias[oc] : 0.f;
  if (relu) v = v > 0.f ? v : 0.f;
  const int64_t o = pos * yc + yoff + oc;
  if (y32) y32[o] = v;
  if (y16) y16[o] = f2bf(v);
}

// --------------------------------------------------------------------------
// Backward-weight: dW[t][co][ci] = sum_p dy[p][co] * x[p + off_t][ci].  Per
// wave: one chunk of positions, TG taps (one kd plane: kh, kw in 0..2), one
// 16 x 16 (co x ci) tile; MFMA with A = dy^T (co x 16 positions), loaded once
// per K step for all TG taps, and B = the shifted input (16 positions x ci).
// Partial sums of chunk k go to part[k][27][co][ci]; a second kernel adds the
// chunks in order.
// --------------------------------------------------------------------------
template <int TG>
__global__ __launch_bounds__(256) void k_conv_wgrad(Grid3 g, const uint16_t* __restrict__ x,
                                                    int ci, const uint16_t* __restrict__ dy,
                                                    int co, int64_t chunk64,
                                                    float* __restrict__ part) {
  // 32-bit positions and element offsets (the host keeps P * channels < 2^31)
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int mt = co / 16, nt = ci / 16, ngr = 27 / TG;
  const int per_chunk = ngr * mt * nt;
  const int k = wave / per_chunk;
  const int P = (int)g.P();
  const int chunk = (int)chunk64;
  const int nchunks = (P + chunk - 1) / chunk;
  if (k >= nchunks) return;
  int rem = wave % per_chunk;
  const int tg = rem / (mt * nt);
  rem %= (mt * nt);
  const int m0 = rem / nt, n0 = rem % nt;
  const int row = lane & 15, kq = lane >> 4;
  const int oc = m0 * 16 + row, ic = n0 * 16 + row;
  float4_t acc[TG];
#pragma unroll
  for (int i = 0; i < TG; ++i) acc[i] = float4_t{0.f, 0.f, 0.f, 0.f};
  const int pbeg = k * chunk, pend = min(P, pbeg + chunk);
  const int kd = tg * TG / 9 - 1;  // TG = 9: one kd plane per tap group
  // Coordinates of the lane's four positions, advanced by 16 per step
  // instead of divided out again.
  Coord3 pc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) pc[j] = coord_of(g, min(pbeg + 4 * kq + j, P - 1));
  for (int pk = pbeg; pk < pend; pk += 16) {
    short4_t a = short4_t{0, 0, 0, 0};
    int pos[4];
    unsigned okd = 0;  // bit j: position j valid and its kd-plane neighbour inside
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      pos[j] = pk + 4 * kq + j;
      if (pos[j] < pend) {
        a[j] = (short)dy[pos[j] * co + oc];
        if ((unsigned)(pc[j].d + kd) < (unsigned)g.D) okd |= 1u << j;
      }
    }
#pragma unroll
    for (int tt = 0; tt < TG; ++tt) {
      const int dyy = tt / 3 - 1, dx = tt % 3 - 1;
      const int off = (kd * g.H + dyy) * g.W + dx;
      short4_t b = short4_t{0, 0, 0, 0};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if ((okd >> j) & 1u) {
          if ((unsigned)(pc[j].h + dyy) < (unsigned)g.H && (unsigned)(pc[j].w + dx) < (unsigned)g.W)
            b[j] = (short)x[(pos[j] + off) * ci + ic];
        }
      }
      acc[tt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[tt], 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) advance(g, pc[j], 16);
  }
#pragma unroll
  for (int tt = 0; tt < TG; ++tt) {
    const int t = tg * TG + tt;
    float* out = part + ((int64_t)(k * 27 + t) * co) * ci;
#pragma unroll
    for (int r = 0; r < 4; ++r) out[(m0 * 16 + 4 * kq + r) * ci + ic] = acc[tt][r];
  }
}

// --------------------------------------------------------------------------
// Backward-weight on v_mfma_f32_16x16x32_bf16 with the operands staged in
// LDS: dW[t][co][ci] = sum_p dy[p][co] x[p + off_t][ci] is, per tap, a GEMM
// with M = 16 output channels, N = 16 input channels and K = positions, which
// channels-last storage does not make contiguous.  A workgroup takes NCO
// output-channel tiles, one input-channel tile and a run of `bpw` boxes of
// BD x BH x BW = 256 positions (BW = 16 or 8).  Per box it stages dy and x
// with its one-voxel halo as they lie in memory, [position][16 channels],
// straight into LDS, the next box while it computes this one.  The transposed
// LDS read (ds_read_b64_tr_b16: 16 lanes read 4 rows of 16 channels and lane
// i gets the 4 values of channel i) then gives a lane its 8 positions of any
// tap in two reads.  Wave w accumulates taps w, w+4, ... over the box's 8 K
// steps of 32 positions (octets of 8 consecutive w).  Each run of boxes
// writes one partial sum.
//
// Transposing on the way into LDS (dword loads, packing, three copies
// shifted by dx) took most of the time before.  Measured at 64^3 x 4, a layer
// of 16 -> 16 channels 75 -> 28 us (510 TF/s), all 14 layers of a training
// iteration 0.62 -> 0.30 ms.  By the counters, the LDS active 22 to 34 % of the
// cycles, the matrix cores 23 to 34 %, waves waiting 30 to 48 % of their time at
// the larger levels: the staging of 2.5 positions per position is not covered.
// --------------------------------------------------------------------------
template <int BW>
struct WBox {
  static constexpr int BD = 4, BH = 256 / (4 * BW);
  static constexpr int HH = BH + 2, HW = BW + 2, NPOS = (BD + 2) * HH * HW;
  static constexpr int XC = (NPOS * 2 + 63) / 64;   // 1 KB pieces of the x halo
  static constexpr int DY = 256 * 32;               // bytes of one dy tile
};

// In LDS the two quads of every odd octet of positions are swapped (of dy, and
// of the 16-wide x rows), so that the octets two quarters of the wave read,
// 256 bytes apart, fall on different banks.
__host__ __device__ constexpr int quad_swap(int pos) { return pos ^ ((pos >> 3 & 1) << 2); }

// Two transposed reads: 4 + 4 positions (32-byte rows) of the lane's channel;
// lo and hi are the lane's pieces of the two quads.
__device__ __forceinline__ bf16x8_t read_transposed(const unsigned char* lo_at,
                                                    const unsigned char* hi_at) {
  typedef __attribute__((address_space(3))) short4_t lds_short4;
  const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)lo_at);
  const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)hi_at);
  return __builtin_bit_cast(bf16x8_t,
                            __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int BW, int NCO>
__global__ __launch_bounds__(256, 2) void k_conv_wgrad_box(Grid3 g, ConvSrc src, int ci,
                                                           const uint16_t* __restrict__ dy,
                                                           int co, int bpw,
                                                           float* __restrict__ part) {
  using B = WBox<BW>;
  __shared__ __attribute__((aligned(16))) unsigned char s_dy[2][NCO * B::DY];
  __shared__ __attribute__((aligned(16))) unsigned char s_x[2][B::XC * 1024];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = lane & 15, q = lane >> 4;
  const int nct = co / (16 * NCO), nit = ci / 16;
  const int tile = blockIdx.x % (nct * nit), chunk = blockIdx.x / (nct * nit);
  const int co0 = (tile / nit) * 16 * NCO, ci0 = (tile % nit) * 16;
  const int nbd = g.D / B::BD, nbh = g.H / B::BH, nbw = g.W / BW;
  const int nboxes = g.N * nbd * nbh * nbw;
  const bool upper = ci0 < src.cu;   // the tile's channels come from the coarse tensor
  const int cx = ci - src.cu;
  // The lane's pieces, the same in every box: dy positions as offsets in
  // elements, halo positions as coordinates and offsets.
  int dy_off[2 * NCO], x_off[(B::XC + 3) / 4];
  HaloPos x_pos[(B::XC + 3) / 4];
  const int c8 = (lane & 1) * 8;
#pragma unroll
  for (int r = 0; r < 2 * NCO; ++r) {
    const int piece = r * 4 + wv, pos = quad_swap((piece % 8) * 32 + (lane >> 1));
    dy_off[r] = ((pos / (BW * B::BH) * g.H + pos / BW % B::BH) * g.W + pos % BW) * co + co0 +
                (piece / 8) * 16 + c8;
  }
#pragma unroll
  for (int r = 0; r < (B::XC + 3) / 4; ++r) {
    x_pos[r] = halo_pos<B::HH, B::HW, (B::XC + 3) / 4 * 128>((r * 4 + wv) * 32 + (lane >> 1));
    if (BW == 16) x_pos[r].w = quad_swap(x_pos[r].w);
    x_off[r] = halo_offset(g, x_pos[r]) * cx + ci0 - src.cu + c8;
  }
  auto stage = [&](int b, int buf) {
    const int bw0 = (b % nbw) * BW, bh0 = ((b / nbw) % nbh) * B::BH;
    const int bd0 = ((b / (nbw * nbh)) % nbd) * B::BD, n = b / (nbw * nbh * nbd);
    const int dz = bd0 - 1, hz = bh0 - 1, wz = bw0 - 1;
    const uint16_t* dy0 = dy + ((((int64_t)n * g.D + bd0) * g.H + bh0) * g.W + bw0) * co;
#pragma unroll
    for (int r = 0; r < 2 * NCO; ++r) load_to_lds(dy0 + dy_off[r], &s_dy[buf][(r * 4 + wv) * 1024]);
    const uint16_t* x0 = src.x + ((((int64_t)n * g.D + dz) * g.H + hz) * g.W + wz) * cx;
#pragma unroll
    for (int r = 0; r < (B::XC + 3) / 4; ++r) {
      const int piece = r * 4 + wv;
      if (piece < B::XC) {
        const HaloPos& o = x_pos[r];
        const uint16_t* p = x0 + x_off[r];
        if (upper) p = src.xu + halo_parent(g, o, n, dz, hz, wz) * src.cu + ci0 + c8;
        load_to_lds(halo_inside(g, o, dz, hz, wz) ? p : zero_piece, &s_x[buf][piece * 1024]);
      }
    }
  };
  f32x4_t acc[7][NCO];
#pragma unroll
  for (int k = 0; k < 7; ++k)
#pragma unroll
    for (int j = 0; j < NCO; ++j) acc[k][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // byte offsets of the lane's octet of K step 0 (a step is two rows of 16 or
  // four of 8 positions: the others are at constant distances)
  const int oh = BW == 16 ? q >> 1 : q, ow = BW == 16 ? (q & 1) * 8 : 0;
  const int r4 = row >> 2, piece = (row & 3) * 8;
  const int dy_pos = oh * BW + ow + r4;
  const int dy_lo = quad_swap(dy_pos) * 32 + piece, dy_hi = quad_swap(dy_pos + 4) * 32 + piece;
  int x_lo[7], x_hi[7];
#pragma unroll
  for (int k = 0; k < 7; ++k) {
    // (there is no tap 27: wave 3 computes tap 26 again and drops it, cheaper
    // than a branch that splits every K step for the scheduler)
    const int t = min(wv + 4 * k, 26), x = t % 3 + ow + r4;
    const int at = (t / 9 * B::HH + t / 3 % 3 + oh) * B::HW;
    x_lo[k] = (at + (BW == 16 ? quad_swap(x) : x)) * 32 + piece;
    x_hi[k] = (at + (BW == 16 ? quad_swap(x + 4) : x + 4)) * 32 + piece;
  }
  const int b_begin = chunk * bpw, b_end = min(nboxes, b_begin + bpw);
  stage(b_begin, 0);
  for (int b = b_begin; b < b_end; ++b) {
    const int buf = (b - b_begin) & 1;
    wait_for_loads();
    __syncthreads();  // this box is there, the other buffer's reads are done
    if (b + 1 < b_end) stage(b + 1, buf ^ 1);
    const unsigned char* pdy = s_dy[buf];
    const unsigned char* px = s_x[buf];
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      constexpr int kRows = 32 / BW;   // rows of w per K step
      const int xo = ((ks / 2) * B::HH + (ks % 2) * kRows) * B::HW * 32;
      bf16x8_t a[NCO];
#pragma unroll
      for (int j = 0; j < NCO; ++j) {
        const unsigned char* at = pdy + j * B::DY + ks * 1024;
        a[j] = read_transposed(at + dy_lo, at + dy_hi);
      }
#pragma unroll
      for (int k = 0; k < 7; ++k) {
        const bf16x8_t bb = read_transposed(px + x_lo[k] + xo, px + x_hi[k] + xo);
#pragma unroll
        for (int j = 0; j < NCO; ++j)
          acc[k][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j], bb, acc[k][j], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 7; ++k) {
    const int t = wv + 4 * k;
    if (t >= 27) continue;
    float* out = part + ((int64_t)chunk * 27 + t) * co * ci;
#pragma unroll
    for (int j = 0; j < NCO; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        out[(int64_t)(co0 + j * 16 + 4 * q + r) * ci + ci0 + row] = acc[k][j][r];
  }
}

// out[i] = sum over k of part[k][i] in a fixed order (deterministic): a
// 256-thread block covers kOut consecutive outputs; each of its 256 / kOut
// phases adds the chunks k = phase, phase + phases, ... in order, and the
// phase sums are then added in phase order.
template <int kOut>
__global__ __launch_bounds__(256) void k_sum_chunks(const float* __restrict__ part,
                                                    int64_t nchunks, int64_t n,
                                                    float* __restrict__ out) {
  constexpr int kPhases = 256 / kOut;
  __shared__ float sh[256];
  const int j = (int)threadIdx.x % kOut, q = (int)threadIdx.x / kOut;
  const int64_t i = (int64_t)blockIdx.x * kOut + j;
  float s = 0.f;
  if (i < n)
#pragma unroll 8
    for (int64_t k = q; k < nchunks; k += kPhases) s += part[k * n + i];
  sh[threadIdx.x] = s;
  __syncthreads();
  if (q == 0 && i < n) {
    float t = sh[j];
    for (int r = 1; r < kPhases; ++r) t += sh[r * kOut + j];
    out[i] = t;
  }
}

// part[k][c] = sum of a[p][c] over the positions p of chunk k, for C
// dividing 256: one block per chunk reads the chunk's [positions][C] slab
// with consecutive threads on consecutive elements (thread t always on
// channel t % C), then adds the threads of each channel in a fixed tree.
__global__ __launch_bounds__(256) void k_channel_sum_block(const float* __restrict__ a,
                                                           int64_t P, int C, int64_t chunk,
                                                           float* __restrict__ part) {
  __shared__ float sh[256];
  const int64_t k = blockIdx.x;
  const int64_t e0 = k * chunk * C, e1 = min(P, (k + 1) * chunk) * C;
  float s = 0.f;
  for (int64_t e = e0 + threadIdx.x; e < e1; e += 256) s += a[e];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int stride = 128; stride >= C; stride >>= 1) {
    if ((int)threadIdx.x < stride) sh[threadIdx.x] += sh[threadIdx.x + stride];
    __syncthreads();
  }
  if ((int)threadIdx.x < C) part[k * C + threadIdx.x] = sh[threadIdx.x];
}

// dpre = dpost where post > 0, else 0 (ReLU backward), as bf16, and the
// per-channel sums of its binary32 values (the bias gradient) in one pass;
// dpost is formed on the way from where the layer's output went:
//   kDprePlain  the data gradient of the next convolution
//   kDpreHead   sum_o dout[p][o] W[o][c] of the 1x1x1 head
//   kDpreUp     the sum of the 8 children in channels [0, C) of the concatenated
//           gradient one level up (nearest upsampling)
//   kDpreSkip   channels [off, off + C) of the concatenated gradient plus the
//           parent's share of the pooled gradient
// Bound by the bytes: one read of each operand, one bf16 write.  Before, the
// gradient was written out in binary32 by each of these operations, masked by
// a second kernel into a bf16 and a binary32 copy, and read again for the
// sums.  A block per chunk adds elements in k_channel_sum_block's order, so
// the sums are the same bits.  Positions fit 32 bits; elements of a wide
// concatenated gradient need not.
// (NO: the head's outputs, or 16 for any number of them.)
template <int SRC, int NO>
__global__ __launch_bounds__(256) void k_dpre(Grid3 g, int C, DpreSrc s,
                                              const uint16_t* __restrict__ post, int chunk,
                                              uint16_t* __restrict__ dpre16,
                                              float* __restrict__ part) {
  __shared__ float sh[256];
  const int t = threadIdx.x, c = t % C, step = 256 / C;
  const int P = (int)g.P(), p0 = blockIdx.x * chunk, pend = min(P, p0 + chunk);
  float wh[NO];
  if constexpr (SRC == kDpreHead)
#pragma unroll
    for (int o = 0; o < NO; ++o) wh[o] = o < s.n ? s.b[o * C + c] : 0.f;
  float sum = 0.f;
#pragma unroll 4
  for (int p = p0 + t / C; p < pend; p += step) {
    const int64_t e = (int64_t)p * C + c;
    float v;
    if constexpr (SRC == kDprePlain) {
      v = s.a[e];
    } else if constexpr (SRC == kDpreHead) {
      v = 0.f;
#pragma unroll
      for (int o = 0; o < NO; ++o)
        if (NO == 4 || o < s.n) v += s.a[(int64_t)p * s.n + o] * wh[o];
    } else if constexpr (SRC == kDpreUp) {
      // row of (n, d, h) and its first child; the fine tensor is 2H x 2W
      const int r1 = p / g.W, w = p - r1 * g.W, r2 = r1 / g.H, h = r1 - r2 * g.H;
      const int child = ((2 * r2) * (2 * g.H) + 2 * h) * (2 * g.W) + 2 * w;
      v = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k)
        v += s.a[(int64_t)(child + ((k >> 2) * (2 * g.H) + (k >> 1 & 1)) * (2 * g.W) + (k & 1)) *
                     s.n + c];
    } else {
      const int r1 = p / g.W, w = p - r1 * g.W, r2 = r1 / g.H, h = r1 - r2 * g.H;
      const int parent = ((r2 >> 1) * (g.H / 2) + (h >> 1)) * (g.W / 2) + (w >> 1);
      v = s.a[(int64_t)p * s.n + s.off + c];
      v += s.b[(int64_t)parent * C + c] * 0.125f;
    }
    if (!(bf2f(post[e]) > 0.f)) v = 0.f;
    dpre16[e] = f2bf(v);
    sum += v;
  }
  sh[t] = sum;
  __syncthreads();
  for (int stride = 128; stride >= C; stride >>= 1) {
    if (t < stride) sh[t] += sh[t + stride];
    __syncthreads();
  }
  if (t < C) part[blockIdx.x * C + t] = sh[t];
}

// The same in three steps for channel counts that do not divide 256: dpost in
// binary32 (kDpreHead, kDpreUp and kDpreSkip), the mask, and the sums.
// Per-channel sums for any C: one thread per (chunk, channel).
__global__ void k_channel_sum_part(const float* __restrict__ a, int64_t P, int C,
                                   int64_t chunk, float* __restrict__ part) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nchunks = (P + chunk - 1) / chunk;
  if (i >= nchunks * C) return;
  const int64_t k = i / C;
  const int c = (int)(i % C);
  const int64_t end = min(P, (k + 1) * chunk);
  float s = 0.f;
  for (int64_t p = k * chunk; p < end; ++p) s += a[p * C + c];
  part[k * C + c] = s;
}

// bf16 copies of the weights for the forward pass, w16[t][co][ci], and for
// backward-data, wt16[26 - t][ci][co], of every layer in one launch instead of
// one per layer, most of which lasted no longer than a launch.  A workgroup
// takes one tap of a 16 x 16 tile through LDS, so that both copies are written
// in whole 32-byte rows: bound by the bytes once a network is large.  (A weight
// per thread with the transposed copy in strided 2-byte stores takes 13.4 us
// on the default network, this 7.3; with Adam on the 75 M weights of channels
// 128 to 1024 1000 us and 785.)  64-bit offsets, as a layer may have 2^31
// weights.
__global__ __launch_bounds__(256) void k_refresh_weights(WeightLayers layers, uint32_t first,
                                                         const float* __restrict__ params) {
  __shared__ uint16_t tile[16][17];
  const uint32_t b = first + blockIdx.x;
  int k = 0;
  while (k + 1 < WeightLayers::kCount && b >= layers.first_tile[k + 1]) ++k;
  const WeightLayers::Layer& l = layers.layer[k];
  const uint32_t nc = l.ci / 16, per_tap = l.co / 16 * nc, in_layer = b - layers.first_tile[k];
  const uint32_t t = in_layer / per_tap, at = in_layer - t * per_tap;
  const uint32_t to = at / nc, tc = at - to * nc;
  const int i = threadIdx.x / 16, j = threadIdx.x % 16;
  const int64_t in = ((int64_t)t * l.co + to * 16 + i) * l.ci + tc * 16 + j;
  const uint16_t v = f2bf(params[l.woff + in]);
  l.w16[in] = v;
  tile[i][j] = v;
  __syncthreads();
  l.wt16[((int64_t)(26 - t) * l.ci + tc * 16 + i) * l.co + to * 16 + j] = tile[j][i];
}

// dpre_bf16[i] = dpost[i] if post[i] > 0 else 0  (ReLU backward)
__global__ void k_relu_bwd(const float* __restrict__ dpost, const uint16_t* __restrict__ post,
                           int64_t n, uint16_t* __restrict__ dpre16,
                           float* __restrict__ dpre32) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float v = bf2f(post[i]) > 0.f ? dpost[i] : 0.f;
  dpre16[i] = f2bf(v);
  if (dpre32) dpre32[i] = v;
}

// 2x2x2 mean pooling of bf16 [N,D,H,W,C] -> bf16 [N,D/2,H/2,W/2,C].
__global__ void k_pool(Grid3 g, int C, const uint16_t* __restrict__ x,
                       uint16_t* __restrict__ y) {
  const Grid3 h{g.N, g.D / 2, g.H / 2, g.W / 2};
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= h.P() * C) return;
  const int c = (int)(i % C);
  const int64_t q = i / C;
  const int w = (int)(q % h.W), hh = (int)((q / h.W) % h.H), d = (int)((q / h.W / h.H) % h.D);
  const int64_t n = q / ((int64_t)h.W * h.H * h.D);
  float s = 0.f;
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b)
      for (int e = 0; e < 2; ++e) {
        const int64_t p = ((n * g.D + 2 * d + a) * g.H + 2 * hh + b) * g.W + 2 * w + e;
        s += bf2f(x[p * C + c]);
      }
  y[i] = f2bf(s * 0.125f);
}

// dx[p] += dy[parent(p)] / 8 (float), x at full resolution.
__global__ void k_pool_bwd_add(Grid3 g, int C, const float* __restrict__ dy,
                               float* __restrict__ dx) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g.P() * C) return;
  const int c = (int)(i % C);
  const int64_t p = i / C;
  const int w = (int)(p % g.W), h = (int)((p / g.W) % g.H), d = (int)((p / g.W / g.H) % g.D);
  const int64_t n = p / ((int64_t)g.W * g.H * g.D);
  const int64_t q = ((n * (g.D / 2) + d / 2) * (g.H / 2) + h / 2) * (g.W / 2) + w / 2;
  dx[i] += dy[q * C + c] * 0.125f;
}

// Nearest 2x upsampling of bf16 [N,D,H,W,C] into channels [off, off+C) of
// the bf16 tensor y [N,2D,2H,2W,yc].
__global__ void k_up(Grid3 g, int C, const uint16_t* __restrict__ x, uint16_t* __restrict__ y,
                     int yc, int yoff) {
  const Grid3 f{g.N, 2 * g.D, 2 * g.H, 2 * g.W};
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= f.P() * C) return;
  const int c = (int)(i % C);
  const int64_t p = i / C;
  const int w = (int)(p % f.W), h = (int)((p / f.W) % f.H), d = (int)((p / f.W / f.H) % f.D);
  const int64_t n = p / ((int64_t)f.W * f.H * f.D);
  const int64_t q = ((n * g.D + d / 2) * g.H + h / 2) * g.W + w / 2;
  y[p * yc + yoff + c] = x[q * C + c];
}

// dx[q][c] = sum of the 8 children of q in channels [off, off+C) of dy.
__global__ void k_up_bwd(Grid3 g, int C, const float* __restrict__ dy, int dyc, int dyoff,
                         float* __restrict__ dx) {
  const Grid3 f{g.N, 2 * g.D, 2 * g.H, 2 * g.W};
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g.P() * C) return;
  const int c = (int)(i % C);
  const int64_t q = i / C;
  const int w = (int)(q % g.W), h = (int)((q / g.W) % g.H), d = (int)((q / g.W / g.H) % g.D);
  const int64_t n = q / ((int64_t)g.W * g.H * g.D);
  float s = 0.f;
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b)
      for (int e = 0; e < 2; ++e) {
        const int64_t p = ((n * f.D + 2 * d + a) * f.H + 2 * h + b) * f.W + 2 * w + e;
        s += dy[p * dyc + dyoff + c];
      }
  dx[i] = s;
}

// Copies bf16 channels: y[p][yoff + c] = x[p][c], c < C.
__global__ void k_copy_channels(int64_t P, int C, const uint16_t* __restrict__ x,
                                uint16_t* __restrict__ y, int yc, int yoff) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P * C) return;
  y[(i / C) * yc + yoff + (i % C)] = x[i];
}

// dx[p][c] (+)= dy[p][dyoff + c], c < C.
__global__ void k_take_channels(int64_t P, int C, const float* __restrict__ dy, int dyc,
                                int dyoff, float* __restrict__ dx, int add) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P * C) return;
  const float v = dy[(i / C) * dyc + dyoff + (i % C)];
  dx[i] = add ? dx[i] + v : v;
}

// Input packing: float [P][cin] -> bf16 [P][16] with zero padding, a position
// per thread (an element per thread with its division took 40 us at
// 64^3 x 4, this 12).
__global__ void k_pack_input(int64_t P, int cin, const float* __restrict__ in,
                             uint16_t* __restrict__ x) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  uint32_t v[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const uint32_t lo = 2 * k < cin ? f2bf(in[p * cin + 2 * k]) : 0u;
    const uint32_t hi = 2 * k + 1 < cin ? f2bf(in[p * cin + 2 * k + 1]) : 0u;
    v[k] = lo | (hi << 16);
  }
  u32x4_t* out = reinterpret_cast<u32x4_t*>(x + p * 16);
  out[0] = u32x4_t{v[0], v[1], v[2], v[3]};
  out[1] = u32x4_t{v[4], v[5], v[6], v[7]};
}

// 1x1x1 head: out[p][o] = sum_k h[p][k] W[o][k] + b[o]   (binary32), a
// position per thread: h is read once, 16 bytes at a time, instead of once
// per output in 2-byte loads.  NO: O, or 16 for any O.
template <int NO>
__global__ __launch_bounds__(256) void k_head_fwd(int64_t P, int K, int O,
                                                  const uint16_t* __restrict__ h,
                                                  const float* __restrict__ W,
                                                  const float* __restrict__ b,
                                                  float* __restrict__ out) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  float s[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o) s[o] = NO == 4 || o < O ? b[o] : 0.f;
  for (int k0 = 0; k0 < K; k0 += 8) {
    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(h + p * K + k0);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float x = __uint_as_float(k & 1 ? v[k >> 1] & 0xFFFF0000u : v[k >> 1] << 16);
#pragma unroll
      for (int o = 0; o < NO; ++o)
        if (NO == 4 || o < O) s[o] += x * W[o * K + k0 + k];
    }
  }
  if constexpr (NO == 4) {
    *reinterpret_cast<f32x4_t*>(out + p * 4) = f32x4_t{s[0], s[1], s[2], s[3]};
  } else {
#pragma unroll
    for (int o = 0; o < NO; ++o)
      if (o < O) out[p * O + o] = s[o];
  }
}

// dh[p][k] = sum_o dout[p][o] W[o][k]
__global__ void k_head_bwd_data(int64_t P, int K, int O, const float* __restrict__ dout,
                                const float* __restrict__ W, float* __restrict__ dh) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P * K) return;
  const int k = (int)(i % K);
  const int64_t p = i / K;
  float s = 0.f;
  for (int o = 0; o < O; ++o) s += dout[p * O + o] * W[o * K + k];
  dh[i] = s;
}

// part[chunk][o*K + k] = sum over the chunk of dout[p][o] h[p][k]
__global__ void k_head_wgrad_part(int64_t P, int K, int O, const float* __restrict__ dout,
                                  const uint16_t* __restrict__ h, int64_t chunk,
                                  float* __restrict__ part) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nchunks = (P + chunk - 1) / chunk;
  if (i >= nchunks * O * K) return;
  const int64_t c = i / ((int64_t)O * K);
  const int ok = (int)(i % ((int64_t)O * K));
  const int o = ok / K, k = ok % K;
  const int64_t end = min(P, (c + 1) * chunk);
  float s = 0.f;
#pragma unroll 8
  for (int64_t p = c * chunk; p < end; ++p) s += dout[p * O + o] * bf2f(h[p * K + k]);
  part[i] = s;
}

// Masked weighted MSE: per-position loss terms and the gradient
// dout = 2 w_c (out - t) m / (count * O).
__global__ void k_mse(int64_t P, int O, const float* __restrict__ out,
                      const float* __restrict__ target, const uint8_t* __restrict__ mask,
                      ChannelWeights wc, float inv_count,
                      float* __restrict__ dout, float* __restrict__ lterm) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P * O) return;
  const int o = (int)(i % O);
  const float m = mask[i / O] ? 1.f : 0.f;
  const float d = (out[i] - target[i]) * m;
  dout[i] = 2.f * wc.w[o] * d * inv_count;
  lterm[i] = wc.w[o] * d * d * inv_count;
}

// Adam (decoupled weight decay) on binary32 master parameters.
__global__ void k_adam(int64_t n, float* __restrict__ p, const float* __restrict__ g,
                       float* __restrict__ m, float* __restrict__ v, float lr, float b1,
                       float b2, float eps, float wd, float c1, float c2) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float mh = mi / c1, vh = vi / c2;
  p[i] -= lr * (mh / (sqrtf(vh) + eps) + wd * p[i]);
}

inline dim3 blocks_for(int64_t n, int t = 256) { return dim3((unsigned)((n + t - 1) / t)); }

// out[i] = sum over k of part[k * n + i] (fixed order): 16 outputs per
// block in 16 chunk phases, or, for few outputs (the biases, the head),
// 4 outputs in 64 phases or one output in 256 phases, so that the grid
// still has thousands of threads.
void sum_chunks(const float* part, int64_t nchunks, int64_t n, float* out, hipStream_t s) {
  if (n >= 2048)
    hipLaunchKernelGGL(k_sum_chunks<16>, blocks_for(n, 16), dim3(256), 0, s, part, nchunks, n,
                       out);
  else if (n >= 256)
    hipLaunchKernelGGL(k_sum_chunks<4>, blocks_for(n, 4), dim3(256), 0, s, part, nchunks, n,
                       out);
  else
    hipLaunchKernelGGL(k_sum_chunks<1>, blocks_for(n, 1), dim3(256), 0, s, part, nchunks, n,
                       out);
}

}  // namespace

namespace {
struct BoxCall {
  Grid3 g;
  ConvSrc src;
  const uint16_t* w;
  const float* bias;
  int co;
  float* y32;
  uint16_t* y16;
  int yc, yoff, relu;
  int kps;  // K steps per slice; 0: one slice
  hipStream_t stream;
};
template <int NG, int NT, int MT, int WM, int BD, int BH, int BW>
void box_launch(const BoxCall& c) {
  using B = ConvBox<NG, NT, MT, WM, BD, BH, BW>;
  const int64_t boxes = (int64_t)c.g.N * ((c.g.D + BD - 1) / BD) * ((c.g.H + BH - 1) / BH) *
                        ((c.g.W + BW - 1) / BW);
  const int per = 16 * NT * B::WN;
  const dim3 grid((unsigned)boxes, (unsigned)((c.co + per - 1) / per)), block(256);
  if (c.kps)
    hipLaunchKernelGGL((k_conv_box<NG, NT, MT, WM, BD, BH, BW, true>), grid, block, 0, c.stream,
                       c.g, c.src, c.w, c.bias, c.co, c.y32, c.y16, c.yc, c.yoff, c.relu, c.kps);
  else
    hipLaunchKernelGGL((k_conv_box<NG, NT, MT, WM, BD, BH, BW, false>), grid, block, 0, c.stream,
                       c.g, c.src, c.w, c.bias, c.co, c.y32, c.y16, c.yc, c.yoff, c.relu, 0);
}
// False where no such form exists.
bool box_launch_form(const BoxCall& c, const BoxForm& f) {
#define HLBN_BOX(NG, NT, MT, WM, BD, BH, BW)       \
  if (f == BoxForm{NG, NT, MT, WM, BD, BH, BW}) {  \
    box_launch<NG, NT, MT, WM, BD, BH, BW>(c);     \
    return true;                                   \
  }
  HLBN_BOX_FORMS(HLBN_BOX)
#undef HLBN_BOX
  return false;
}
}  // namespace

int64_t conv_fwd_ws(const ConvGeom& cg, int ci, int co) {
  if (box_form(cg, ci, co).ng) return 0;
  const FwdPlan f = fwd_plan(cg, ci, co);
  return f.nsplit > 1 ? (int64_t)f.nsplit * cg.N * cg.D * cg.H * cg.W * co : 0;
}

namespace {
// Boxes per workgroup: at least about 1024 workgroups over the tile pairs.
int64_t wgrad_boxes_per_group(const ConvGeom& cg, int ci, int co) {
  const int64_t nboxes = (int64_t)cg.N * cg.D * cg.H * cg.W / 256;
  const int64_t tiles = (int64_t)(co / 16) * (ci / 16);
  return std::max<int64_t>(1, nboxes * tiles / 1024);
}
}  // namespace

bool conv_takes_parts(const ConvGeom& cg, int ci) {
  return box_form(cg, ci, 16).ng != 0 && wgrad_box_width(cg) != 0;
}

int conv_fwd(const ConvGeom& cg, const uint16_t* x, const uint16_t* xu, int cu, int ci,
             const uint16_t* w,
             const float* bias, int co, float* y32, uint16_t* y16, int yc, int yoff, int relu,
             float* ws, void* stream) {
  const Grid3 g{cg.N, cg.D, cg.H, cg.W};
  const int64_t P = (int64_t)cg.N * cg.D * cg.H * cg.W;
  const FwdPlan f = fwd_plan(cg, ci, co);
  const BoxForm form = box_form(cg, ci, co);
  if (form.ng) {
    const BoxCall c{g, ConvSrc{x, xu, xu ? cu : 0}, w, bias, co, y32, y16, yc, yoff, relu,
                    f.nsplit > 1 ? f.hpw / 2 : 0, (hipStream_t)stream};
    if (!box_launch_form(c, form)) return (int)hipErrorInvalidValue;
    return (int)hipGetLastError();
  }
  if (xu) return (int)hipErrorInvalidValue;
  if (f.nsplit > 1 && !ws) return (int)hipErrorInvalidValue;
  float* slices = f.nsplit > 1 ? ws : nullptr;
  const dim3 grid((unsigned)((f.waves + 3) / 4), (unsigned)f.nsplit), block(256);
  hipStream_t s = (hipStream_t)stream;
  bool launched = false;
#define HLBN_FWD(M_, N_)                                                                   \
  if (!launched && f.mt == M_ && f.nt == N_) {                                             \
    hipLaunchKernelGGL((k_conv_fwd<M_, N_>), grid, block, 0, s, g, x, ci, w, bias, co, y32,  \
                       y16, yc, yoff, relu, f.hpw, slices);                                \
    launched = true;                                                                       \
  }
  HLBN_FWD(4, 1) HLBN_FWD(2, 1) HLBN_FWD(1, 1)
  HLBN_FWD(4, 2) HLBN_FWD(2, 2) HLBN_FWD(1, 2)
  HLBN_FWD(4, 4) HLBN_FWD(2, 4) HLBN_FWD(1, 4)
  HLBN_FWD(2, 8) HLBN_FWD(1, 8)
#undef HLBN_FWD
  if (!launched) return (int)hipErrorInvalidValue;
  if (slices)
    hipLaunchKernelGGL(k_conv_reduce, blocks_for(P * co), dim3(256), 0, s, P, co, f.nsplit,
                       slices, bias, relu, y32, y16, yc, yoff);
  return (int)hipGetLastError();
}

int64_t wgrad_chunk(const ConvGeom& cg) {
  // up to 2048 chunks: with one wave per (chunk, tap plane, 16x16 tile) the
  // finest level still has thousands of waves
  const int64_t P = (int64_t)cg.N * cg.D * cg.H * cg.W;
  int64_t chunk = (P + 2047) / 2048;
  chunk = (chunk + 15) / 16 * 16;
  return chunk < 256 ? 256 : chunk;
}

int64_t wgrad_parts(const ConvGeom& cg, int ci, int co) {
  const int64_t P = (int64_t)cg.N * cg.D * cg.H * cg.W;
  int64_t nchunks;
  if (wgrad_box_width(cg)) {
    const int64_t bpw = wgrad_boxes_per_group(cg, ci, co);
    nchunks = (P / 256 + bpw - 1) / bpw;
  } else {
    const int64_t chunk = wgrad_chunk(cg);
    nchunks = (P + chunk - 1) / chunk;
  }
  return nchunks * 27 * co * ci;
}

int conv_wgrad(const ConvGeom& cg, const uint16_t* x, const uint16_t* xu, int cu, int ci,
               const uint16_t* dy, int co,
               float* part, float* dw, void* stream) {
  const Grid3 g{cg.N, cg.D, cg.H, cg.W};
  const int64_t P = g.P();
  hipStream_t s = (hipStream_t)stream;
  const int64_t n = (int64_t)27 * co * ci;
  const int bw = wgrad_box_width(cg);
  if (bw) {
    const int64_t bpw = wgrad_boxes_per_group(cg, ci, co);
    const int64_t nchunks = (P / 256 + bpw - 1) / bpw;
    // two output-channel tiles per workgroup where they come in pairs: each
    // read of x then serves two products
    const ConvSrc src{x, xu, xu ? cu : 0};
    auto go = [&](auto width, auto tiles) {
      constexpr int BW = decltype(width)::value, NCO = decltype(tiles)::value;
      hipLaunchKernelGGL((k_conv_wgrad_box<BW, NCO>),
                         dim3((unsigned)(nchunks * (co / (16 * NCO)) * (ci / 16))), dim3(256), 0, s,
                         g, src, ci, dy, co, (int)bpw, part);
    };
    using std::integral_constant;
    if (bw == 16 && co % 32 == 0) go(integral_constant<int, 16>{}, integral_constant<int, 2>{});
    else if (bw == 16) go(integral_constant<int, 16>{}, integral_constant<int, 1>{});
    else if (co % 32 == 0) go(integral_constant<int, 8>{}, integral_constant<int, 2>{});
    else go(integral_constant<int, 8>{}, integral_constant<int, 1>{});
    sum_chunks(part, nchunks, n, dw, s);
    return (int)hipGetLastError();
  }
  if (xu) return (int)hipErrorInvalidValue;
  const int64_t chunk = wgrad_chunk(cg);
  const int64_t nchunks = (P + chunk - 1) / chunk;
  constexpr int TG = 9;
  const int64_t waves = nchunks * (27 / TG) * (co / 16) * (ci / 16);
  hipLaunchKernelGGL((k_conv_wgrad<TG>), dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, g,
                     x, ci, dy, co, chunk, part);
  sum_chunks(part, nchunks, n, dw, s);
  return (int)hipGetLastError();
}

int channel_sum(const float* a, int64_t P, int C, float* part, int64_t chunk, float* out,
                void* stream) {
  const int64_t nchunks = (P + chunk - 1) / chunk;
  hipStream_t s = (hipStream_t)stream;
  if (C > 0 && 256 % C == 0)
    hipLaunchKernelGGL(k_channel_sum_block, dim3((unsigned)nchunks), dim3(256), 0, s, a, P, C,
                       chunk, part);
  else
    hipLaunchKernelGGL(k_channel_sum_part, blocks_for(nchunks * C), dim3(256), 0, s, a, P, C,
                       chunk, part);
  sum_chunks(part, nchunks, (int64_t)C, out, s);
  return (int)hipGetLastError();
}

int refresh_weights(WeightLayers layers, const float* params, void* stream) {
  uint32_t tiles = 0;
  for (int k = 0; k < WeightLayers::kCount; ++k) {
    layers.first_tile[k] = tiles;
    tiles += 27u * (layers.layer[k].co / 16) * (layers.layer[k].ci / 16);
  }
  // (a grid has fewer than 2^32 threads)
  constexpr uint32_t kLaunch = 1u << 23;
  for (uint32_t first = 0; first < tiles; first += kLaunch)
    hipLaunchKernelGGL(k_refresh_weights, dim3(std::min(tiles - first, kLaunch)), dim3(256), 0,
                       (hipStream_t)stream, layers, first, params);
  return (int)hipGetLastError();
}

bool dpre_fused(int C) { return C <= 256 && 256 % C == 0; }

namespace {
template <int SRC, int NO = 1>
void dpre_launch(const ConvGeom& cg, int C, const DpreSrc& src, const uint16_t* post,
                 int64_t chunk, uint16_t* dpre16, float* part, hipStream_t s) {
  const Grid3 g{cg.N, cg.D, cg.H, cg.W};
  hipLaunchKernelGGL((k_dpre<SRC, NO>), dim3((unsigned)((g.P() + chunk - 1) / chunk)), dim3(256), 0, s,
                     g, C, src, post, (int)chunk, dpre16, part);
}
}  // namespace

int dpre(const ConvGeom& cg, int C, int kind, const DpreSrc& src, const uint16_t* post,
         uint16_t* dpre16, float* part, float* db, void* stream) {
  hipStream_t s = (hipStream_t)stream;
  const int64_t chunk = wgrad_chunk(cg), P = (int64_t)cg.N * cg.D * cg.H * cg.W;
  if (!dpre_fused(C)) return (int)hipErrorInvalidValue;
  if (kind == kDprePlain) dpre_launch<kDprePlain>(cg, C, src, post, chunk, dpre16, part, s);
  else if (kind == kDpreHead && src.n == 4)
    dpre_launch<kDpreHead, 4>(cg, C, src, post, chunk, dpre16, part, s);
  else if (kind == kDpreHead)
    dpre_launch<kDpreHead, 16>(cg, C, src, post, chunk, dpre16, part, s);
  else if (kind == kDpreUp) dpre_launch<kDpreUp>(cg, C, src, post, chunk, dpre16, part, s);
  else dpre_launch<kDpreSkip>(cg, C, src, post, chunk, dpre16, part, s);
  sum_chunks(part, (P + chunk - 1) / chunk, (int64_t)C, db, s);
  return (int)hipGetLastError();
}

int relu_bwd(const float* dpost, const uint16_t* post, int64_t n, uint16_t* dpre16,
             float* dpre32, void* stream) {
  hipLaunchKernelGGL(k_relu_bwd, blocks_for(n), dim3(256), 0, (hipStream_t)stream, dpost, post,
                     n, dpre16, dpre32);
  return (int)hipGetLastError();
}

int pool(const ConvGeom& cg, int C, const uint16_t* x, uint16_t* y, void* stream) {
  const Grid3 g{cg.N, cg.D, cg.H, cg.W};
  hipLaunchKernelGGL(k_pool, blocks_for(g.P() / 8 * C), dim3(256), 0, (hipStream_t)stream, g, C,
                     x, y);
  return (int)hipGetLastError();
}

int pool_bwd_add(const ConvGeom& cg, int C, const float* dy, float* dx, void* stream) {
  const Grid3 g{cg.N, cg.D, cg.H, cg.W};
  hipLaunchKernelGGL(k_pool_bwd_add, blocks_for(g.P() * C), dim3(256), 0, (hipStream_t)stream,
                     g, C, dy, dx);
  return (int)hipGetLastError();
}

int up(const ConvGeom& coarse, int C, const uint16_t* x, uint16_t* y, int yc, int yoff,
       void* stream) {
  const Grid3 g{coarse.N, coarse.D, coarse.H, coarse.W};
  hipLaunchKernelGGL(k_up, blocks_for(g.P() * 8 * C), dim3(256), 0, (hipStream_t)stream, g, C, x,
                     y, yc, yoff);
  return (int)hipGetLastError();
}

int up_bwd(const ConvGeom& coarse, int C, const float* dy, int dyc, int dyoff, float* dx,
           void* stream) {
  const Grid3 g{coarse.N, coarse.D, coarse.H, coarse.W};
  hipLaunchKernelGGL(k_up_bwd, blocks_for(g.P() * C), dim3(256), 0, (hipStream_t)stream, g, C,
                     dy, dyc, dyoff, dx);
  return (int)hipGetLastError();
}

int copy_channels(int64_t P, int C, const uint16_t* x, uint16_t* y, int yc, int yoff,
                  void* stream) {
  hipLaunchKernelGGL(k_copy_channels, blocks_for(P * C), dim3(256), 0, (hipStream_t)stream, P, C,
                     x, y, yc, yoff);
  return (int)hipGetLastError();
}

int take_channels(int64_t P, int C, const float* dy, int dyc, int dyoff, float* dx, int add,
                  void* stream) {
  hipLaunchKernelGGL(k_take_channels, blocks_for(P * C), dim3(256), 0, (hipStream_t)stream, P, C,
                     dy, dyc, dyoff, dx, add);
  return (int)hipGetLastError();
}

int pack_input(int64_t P, int cin, const float* in, uint16_t* x, void* stream) {
  hipLaunchKernelGGL(k_pack_input, blocks_for(P), dim3(256), 0, (hipStream_t)stream, P, cin, in,
                     x);
  return (int)hipGetLastError();
}

int head_fwd(int64_t P, int K, int O, const uint16_t* h, const float* W, const float* b,
             float* out, void* stream) {
  if (O == 4)
    hipLaunchKernelGGL(k_head_fwd<4>, blocks_for(P), dim3(256), 0, (hipStream_t)stream, P, K, O,
                       h, W, b, out);
  else
    hipLaunchKernelGGL(k_head_fwd<16>, blocks_for(P), dim3(256), 0, (hipStream_t)stream, P, K, O,
                       h, W, b, out);
  return (int)hipGetLastError();
}

int head_bwd_data(int64_t P, int K, int O, const float* dout, const float* W, float* dh,
                  void* stream) {
  hipLaunchKernelGGL(k_head_bwd_data, blocks_for(P * K), dim3(256), 0, (hipStream_t)stream, P, K,
                     O, dout, W, dh);
  return (int)hipGetLastError();
}

int head_wgrad(int64_t P, int K, int O, const float* dout, const uint16_t* h, float* part,
               int64_t chunk, float* dW, float* db, void* stream) {
  hipStream_t s = (hipStream_t)stream;
  const int64_t nchunks = (P + chunk - 1) / chunk;
  hipLaunchKernelGGL(k_head_wgrad_part, blocks_for(nchunks * O * K), dim3(256), 0, s, P, K, O,
                     dout, h, chunk, part);
  sum_chunks(part, nchunks, (int64_t)O * K, dW, s);
  return channel_sum(dout, P, O, part, chunk, db, stream);
}

int mse(int64_t P, int O, const float* out, const float* target, const uint8_t* mask,
        const ChannelWeights& wc, float inv_count, float* dout, float* lterm, void* stream) {
  hipLaunchKernelGGL(k_mse, blocks_for(P * O), dim3(256), 0, (hipStream_t)stream, P, O, out,
                     target, mask, wc, inv_count, dout, lterm);
  return (int)hipGetLastError();
}

int adam(int64_t n, float* p, const float* g, float* m, float* v, float lr, float b1, float b2,
         float eps, float wd, float c1, float c2, void* stream) {
  hipLaunchKernelGGL(k_adam, blocks_for(n), dim3(256), 0, (hipStream_t)stream, n, p, g, m, v, lr,
                     b1, b2, eps, wd, c1, c2);
  return (int)hipGetLastError();
}

}  // namespace hlbn
