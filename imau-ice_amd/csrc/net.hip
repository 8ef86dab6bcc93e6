// net.hip -- kernels of the warm-start network: 3x3 convolutions on the
// matrix cores (v_mfma_f32_16x16x32_bf16 for 32 input channels and for the
// weight gradients, v_mfma_f32_16x16x16_bf16 for 16: BF16 operands, FP32
// accumulation), 2x2 pooling, upsampling with skip addition, the
// backward passes of those, a weighted squared-error loss and Adam.
//
// Convolution as a matrix product per tile: D[cout][pixel] = W[cout][9 cin] X[9 cin][pixel],
// one wavefront per tile of IMAU_NET_TR x IMAU_NET_TC pixels (IMAU_NET_TR
// column blocks of 16 pixels), the layer's weights held in registers as the A
// operands, the input pixels (channels contiguous) staged in LDS as
// the B operands.  Operand layout of the 16x16x16 instruction, lane l:
// A[i][k] with i = l % 16, k = 4 (l / 16) + e;  B[k][j] with j = l % 16,
// k = 4 (l / 16) + e;  D[i][j] with j = l % 16, i = 4 (l / 16) + e  (e = 0..3).
#include <algorithm>

#include "net.h"

namespace {

using imau::net::LevelView;
using imau::net::NImg;
using imau::net::NTile;

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int TR = IMAU_NET_TR, TC = IMAU_NET_TC;

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
// round to nearest, ties to even (NaN kept quiet)
__device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ s4 ld4(const uint16_t *p) { return *reinterpret_cast<const s4 *>(p); }
__device__ __forceinline__ void st4(uint16_t *p, s4 v) { *reinterpret_cast<s4 *>(p) = v; }

// ---------------------------------------------------------------------------
// convolution
// ---------------------------------------------------------------------------
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f8 __attribute__((ext_vector_type(8)));
// 16-byte accesses to global memory need no more than a dword's alignment
typedef b8 b8u __attribute__((aligned(4)));
typedef f2 f2u __attribute__((aligned(4)));
__device__ __forceinline__ b8 ld8(const uint16_t *p) { return *reinterpret_cast<const b8u *>(p); }

// LDS written and read by the same wavefront: its LDS operations complete in
// order, so only the compiler has to keep them so
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Bound by its bytes: CIN + COUT channels per pixel.  Each wavefront stages its
// tile plus a one-pixel halo ((TR+2) x (TC+2) pixels) in LDS with 16-byte loads
// that are all in flight together (the tile's descriptor came a tile earlier;
// outside the image they read pixel (0, 0)
// and are replaced by zeros); the next tile's loads are issued before this
// one's products.  A staged row serves the three tile rows that it touches, in
// the order of the taps.  32 channels: one v_mfma_f32_16x16x32_bf16 per tap and
// 16 outputs (lane l holds k = 8 (l / 16) + e of its row / column), pixels
// padded to 40 channels against bank conflicts; 16 channels:
// v_mfma_f32_16x16x16_bf16.  With 32 outputs the weight rows are dealt so that
// a lane ends with 8 neighbouring channels, one 16-byte store per pixel.  The
// tiles are dealt to the 8 XCDs in contiguous runs, so halos are found in
// their L2.  Over 1.37 million pixels (floors at the rate of a
// copy: 36 us for 32 -> 32, 27 for 16 -> 32, 20 for 32 -> 2): 32 -> 32 73 -> 38
// us, 16 -> 32 95 -> 32 (it staged nothing), 32 -> 2 FP32 33 -> 24.
template <int CIN, int COUT, bool OUTF>
__global__ void __launch_bounds__(256) k_conv(const NTile *__restrict__ tiles, int ntiles,
                                              const uint16_t *__restrict__ x,
                                              const uint16_t *__restrict__ w, const float *__restrict__ bias,
                                              int relu, void *__restrict__ yv) {
  constexpr int NCT = COUT / 16, KL = CIN / 4;  // KL: channels per lane and instruction
  constexpr int XR = TR + 2, XC = TC + 2, CP = CIN == 32 ? 40 : 16, WSZ = XR * XC * CP;
  constexpr int CH = CIN / 8, NQ = XR * XC * CH, NL = (NQ + 63) / 64;  // 16-byte pieces of a pixel, of a tile, per lane
  typedef short sk __attribute__((ext_vector_type(KL)));
  __shared__ __align__(16) uint16_t sx[4 * WSZ];
  const int lane = threadIdx.x & 63, lc = lane & 15, lk = lane >> 4, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint16_t *my = sx + wv * WSZ;
  // blocks b, b + 8, .. run on one XCD
  const int ng = (ntiles + 3) / 4, gx = (ng + 7) / 8, gs = (int)gridDim.x / 8;
  const int g0 = ((int)blockIdx.x & 7) * gx, g1 = min(ng, g0 + gx);
  int tix = 4 * (g0 + ((int)blockIdx.x >> 3)) + wv;
  const int tend = min(ntiles, 4 * g1);
  if (tix >= tend) return;  // uniform per wavefront; there is no barrier below

  // output channel of row i of weight block ct
  auto co_of = [](int ct, int i) { return NCT == 2 ? 8 * (i >> 2) + 4 * ct + (i & 3) : i; };
  b8 pre[NL];
  auto load = [&](const NTile &t) {
    const uint16_t *xi = x + t.off * CIN;
#pragma unroll
    for (int l = 0; l < NL; ++l) {
      const int q = lane + 64 * l, px = q / CH, ch = q % CH;
      const int hr = px / XC, hc = px - hr * XC;
      const int rr = t.r0 + hr - 1, cc = t.c0 + hc - 1;
      const bool ok = rr >= 0 && rr < t.rows && cc >= 0 && cc < t.cols;
      const b8 v = ld8(xi + (ok ? ((long long)rr * t.cols + cc) * CIN : 0) + 8 * ch);
      pre[l] = ok ? v : b8{};
    }
  };
  const int dt = 4 * gs;
  NTile tc = tiles[tix], tn = tiles[min(tix + dt, ntiles - 1)];
  load(tc);
  sk wa[9][NCT];
#pragma unroll
  for (int tap = 0; tap < 9; ++tap)
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct)
      wa[tap][ct] = *reinterpret_cast<const sk *>(w + (size_t)(tap * COUT + co_of(ct, lc)) * CIN + KL * lk);
  float bs[NCT][4];
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
    for (int e = 0; e < 4; ++e) bs[ct][e] = bias ? bias[co_of(ct, 4 * lk + e)] : 0.0f;

  for (;;) {
#pragma unroll
    for (int l = 0; l < NL; ++l) {
      const int q = lane + 64 * l;
      if (64 * l + 63 < NQ || q < NQ) *reinterpret_cast<b8 *>(my + (q / CH) * CP + 8 * (q % CH)) = pre[l];
    }
    wave_lds_sync();
    tix += dt;
    const bool more = tix < tend;
    const NTile tl = tn;
    if (more) {
      load(tl);
      tn = tiles[min(tix + dt, ntiles - 1)];
    }
    f4 acc[TR][NCT];
#pragma unroll
    for (int r = 0; r < TR; ++r)
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) acc[r][ct] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int hr = 0; hr < XR; ++hr)
#pragma unroll
      for (int dc = 0; dc < 3; ++dc) {
        const sk b = *reinterpret_cast<const sk *>(my + (hr * XC + lc + dc) * CP + KL * lk);
#pragma unroll
        for (int dr = 0; dr < 3; ++dr) {
          const int r = hr - dr;
          if (r < 0 || r >= TR) continue;
#pragma unroll
          for (int ct = 0; ct < NCT; ++ct) {
            if constexpr (CIN == 32)
              acc[r][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  __builtin_bit_cast(b8, wa[3 * dr + dc][ct]), __builtin_bit_cast(b8, b), acc[r][ct], 0, 0, 0);
            else
              acc[r][ct] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(wa[3 * dr + dc][ct], b, acc[r][ct], 0, 0, 0);
          }
        }
      }
    const int c = tc.c0 + lc;
#pragma unroll
    for (int r = 0; r < TR; ++r) {
      const int rr = tc.r0 + r;
      float v[NCT * 4];
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float s = acc[r][ct][e] + bs[ct][e];
          v[4 * ct + e] = relu ? fmaxf(s, 0.0f) : s;
        }
      if (rr >= tc.rows || c >= tc.cols) continue;
      const long long pix = tc.off + (long long)rr * tc.cols + c;
      if constexpr (OUTF) {
        if (lk == 0) *reinterpret_cast<f2u *>(static_cast<float *>(yv) + 2 * pix) = f2{v[0], v[1]};
      } else {
        uint16_t *yp = static_cast<uint16_t *>(yv) + pix * COUT + NCT * 4 * lk;
        if constexpr (NCT == 2) {
          const f8 o = {v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]};
          *reinterpret_cast<b8u *>(yp) = __builtin_convertvector(o, b8);
        } else {
          typedef __bf16 b4 __attribute__((ext_vector_type(4)));
          const f4 o = {v[0], v[1], v[2], v[3]};
          *reinterpret_cast<b4 *>(yp) = __builtin_convertvector(o, b4);
        }
      }
    }
    if (!more) break;
    tc = tl;
    wave_lds_sync();
  }
}

// Weight and bias gradients: dw[tap][co][ci] = G^T[co][pixels] X_tap[pixels][ci].
// A workgroup of four wavefronts sums its tiles in registers and writes one
// partial; sum_partials adds them in a fixed order.  Each wavefront owns one 16
// x 16 block of (co, ci) for all nine taps (36 sums per lane, and with two such
// blocks only, every second pair of tile rows), so that 4 workgroups fit on a
// CU.  The tile's gradient (64 pixels) and input with a one-pixel halo are
// staged in LDS transposed, [channel][pixel], two neighbouring pixels per write
// (lanes of neighbouring pixels swap half their channels), so that a lane's 8
// pixels of an operand are one 16-byte read, and the three column taps come
// from the same 10 pixels, shifted.  Two rows of a tile (32 pixels) make one
// v_mfma_f32_16x16x32_bf16.  The channel pitches (76 and 36 dwords) put the 16
// channels of a read on distinct banks.  The next tile's loads are issued
// before this one's products; two buffers, one barrier per tile.  The bias
// gradient is a product with ones.  Over 16 images of 256 x 256 (floor 28 us):
// 32 -> 32 channels 95 -> 58 us against one wavefront per workgroup with all
// blocks' sums in 144 registers and 2-byte LDS reads, 16 -> 32 69 -> 38, 32 -> 16
// 71 -> 42.  512 and 768 workgroups instead of at most 1024: 69 and 60 us, 1280: 69.
constexpr int GP = TR * TC + 8;                   // pitch of a channel of g
constexpr int XW = 24, XP = (TR + 2) * XW + 8;    // pitch of a row and of a channel of x

template <int CIN, int COUT>
__global__ void __launch_bounds__(256) k_conv_dw(const NTile *__restrict__ tiles, int ntiles,
                                                 const uint16_t *__restrict__ g,
                                                 const uint16_t *__restrict__ x, float *__restrict__ part) {
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  constexpr int NCI = CIN / 16, NCO = COUT / 16, NB = NCI * NCO, WB = 4 / NB;  // WB: wavefronts per (co, ci) block
  static_assert(TR == 4 && TC == 16 && (NB == 2 || NB == 4), "");
  constexpr int XC = TC + 2, GH = COUT / 8, XH = CIN / 8;
  constexpr int NG = TR * TC * GH, NX = (TR + 2) * XC * XH, LX = (NX + 255) / 256;
  constexpr int BUF = COUT * GP + CIN * XP, RED = WB == 2 ? 2 * 10 * 64 * 8 : 0;  // uint16
  __shared__ __align__(16) uint16_t sm[2 * BUF > RED ? 2 * BUF : RED];
  const int tid = threadIdx.x, lane = tid & 63, lc = lane & 15, lk = lane >> 4, wv = tid >> 6;
  const int co = wv % NCO, ci = (wv / NCO) % NCI, wr = wv / NB;
  f4 acc[9], accb = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int tap = 0; tap < 9; ++tap) acc[tap] = f4{0.0f, 0.0f, 0.0f, 0.0f};
  const short one = 0x3f80;
  typedef short s8 __attribute__((ext_vector_type(8)));
  const b8 ones = __builtin_bit_cast(b8, s8{one, one, one, one, one, one, one, one});

  u4 pg, pxr[LX];
  auto load = [&](const NTile &t) {
    const u4 z = {0, 0, 0, 0};
    if (NG == 256 || tid < NG) {
      const int px = tid / GH, ch = tid % GH;
      const int rr = t.r0 + px / TC, cc = t.c0 + px % TC;
      const bool ok = rr < t.rows && cc < t.cols;
      const b8 v = ld8(g + (t.off + (ok ? (long long)rr * t.cols + cc : 0)) * COUT + 8 * ch);
      pg = ok ? __builtin_bit_cast(u4, v) : z;
    } else {
      pg = z;
    }
#pragma unroll
    for (int l = 0; l < LX; ++l) {
      const int q = tid + 256 * l, px = q / XH, ch = q % XH;
      const int rr = t.r0 + px / XC - 1, cc = t.c0 + px % XC - 1;
      const bool ok = q < NX && rr >= 0 && rr < t.rows && cc >= 0 && cc < t.cols;
      const b8 v = ld8(x + (t.off + (ok ? (long long)rr * t.cols + cc : 0)) * CIN + 8 * ch);
      pxr[l] = ok ? __builtin_bit_cast(u4, v) : z;
    }
  };
  // 8 channels of pixel p (this lane) and of its neighbour p ^ 1 (lane ^ H) to
  // 4 channels of both: four dwords at d, d + pitch, ..
  auto put = [&](u4 v, int H, uint16_t *d, int pitch, bool odd, bool ok) {
    const uint32_t r0 = __shfl_xor(odd ? v[0] : v[2], H), r1 = __shfl_xor(odd ? v[1] : v[3], H);
    if (!ok) return;
    const uint32_t a0 = odd ? r0 : v[0], b0 = odd ? v[2] : r0, a1 = odd ? r1 : v[1], b1 = odd ? v[3] : r1;
    uint32_t *o = reinterpret_cast<uint32_t *>(d);
    o[0] = (a0 & 0xffffu) | (b0 << 16);
    o[pitch / 2] = (a0 >> 16) | (b0 & 0xffff0000u);
    o[pitch] = (a1 & 0xffffu) | (b1 << 16);
    o[3 * (pitch / 2)] = (a1 >> 16) | (b1 & 0xffff0000u);
  };

  // blocks b, b + 8, .. run on one XCD: each XCD takes a contiguous run of tiles
  const int nb = (int)gridDim.x, runs = nb % 8 == 0 ? 8 : 1, gx = (ntiles + runs - 1) / runs;
  int tix = ((int)blockIdx.x % runs) * gx + (int)blockIdx.x / runs;
  const int tend = min(ntiles, ((int)blockIdx.x % runs + 1) * gx);
  const int dt = nb / runs;
  NTile tn = tiles[min(tix + dt, ntiles - 1)];
  if (tix < tend) load(tiles[tix]);
  for (int k = 0; tix < tend; k ^= 1) {
    uint16_t *sg = sm + k * BUF, *sx = sg + COUT * GP;
    {
      const int px = tid / GH, ch = tid % GH, odd = px & 1;
      put(pg, GH, sg + (8 * ch + 4 * odd) * GP + (px & ~1), GP, odd, NG == 256 || tid < NG);
    }
#pragma unroll
    for (int l = 0; l < LX; ++l) {
      const int q = tid + 256 * l, px = q / XH, ch = q % XH, odd = px & 1;
      put(pxr[l], XH, sx + (8 * ch + 4 * odd) * XP + px / XC * XW + (px % XC & ~1), XP, odd, q < NX);
    }
    __syncthreads();
    tix += dt;
    if (tix < tend) {
      load(tn);
      tn = tiles[min(tix + dt, ntiles - 1)];
    }
#pragma unroll
    for (int rp = 0; rp < TR / 2; ++rp) {
      if (WB == 2 && rp != wr) continue;
      const b8 a = *reinterpret_cast<const b8 *>(sg + (co * 16 + lc) * GP + 32 * rp + 8 * lk);
      if (ci == 0) accb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, ones, accb, 0, 0, 0);
#pragma unroll
      for (int dr = 0; dr < 3; ++dr) {
        const uint16_t *p = sx + (ci * 16 + lc) * XP + (2 * rp + (lk >> 1) + dr) * XW + 8 * (lk & 1);
        const u4 w = *reinterpret_cast<const u4 *>(p);
        const uint32_t w4 = *reinterpret_cast<const uint32_t *>(p + 8);
        const u4 m = {__builtin_amdgcn_alignbit(w[1], w[0], 16), __builtin_amdgcn_alignbit(w[2], w[1], 16),
                      __builtin_amdgcn_alignbit(w[3], w[2], 16), __builtin_amdgcn_alignbit(w4, w[3], 16)};
        const u4 e = {w[1], w[2], w[3], w4};
        acc[3 * dr] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(b8, w), acc[3 * dr], 0, 0, 0);
        acc[3 * dr + 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(b8, m), acc[3 * dr + 1], 0, 0, 0);
        acc[3 * dr + 2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(b8, e), acc[3 * dr + 2], 0, 0, 0);
      }
    }
  }
  if constexpr (WB == 2) {  // the second half of the rows joins the first
    f4 *red = reinterpret_cast<f4 *>(sm) + (wv % NB) * 10 * 64 + lane;
    __syncthreads();
    if (wr == 1) {
#pragma unroll
      for (int tap = 0; tap < 9; ++tap) red[tap * 64] = acc[tap];
      red[9 * 64] = accb;
    }
    __syncthreads();
    if (wr == 1) return;
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) acc[tap] += red[tap * 64];
    accb += red[9 * 64];
  }
  constexpr int NW = 9 * COUT * CIN;
  float *P = part + (size_t)blockIdx.x * (NW + COUT);
#pragma unroll
  for (int tap = 0; tap < 9; ++tap)
#pragma unroll
    for (int e = 0; e < 4; ++e) P[(tap * COUT + co * 16 + 4 * lk + e) * CIN + ci * 16 + lc] = acc[tap][e];
  if (ci == 0 && lc == 0)
#pragma unroll
    for (int e = 0; e < 4; ++e) P[NW + co * 16 + 4 * lk + e] = accb[e];
}

// Sum of the workgroups' partials (up to 1024 of 9 cout cin + cout floats, 38
// MB for 32 -> 32 channels).  Bound by the latency of its loads: one thread
// per sum walking every partial took 202 us (190 GB/s, 37 workgroups); with
// SP_G groups of partials per sum and SP_U independent running sums per group
// it takes 5 to 8 us (train step, 16 images of 256 x 256: 3338 -> 1368 us).  The
// order is fixed: partial b goes to group b % SP_G, then the groups' sums are
// added in order.
constexpr int SP_Q = 64, SP_G = 16, SP_U = 4;
__global__ void __launch_bounds__(SP_Q *SP_G) k_sum_partials(int nblk, int n, const float *__restrict__ part,
                                                             float *__restrict__ dw, int nw, float *__restrict__ db) {
  __shared__ float red[SP_G][SP_Q];
  const int q = blockIdx.x * SP_Q + threadIdx.x, g = threadIdx.y;
  float s[SP_U] = {};
  if (q < n) {
    const float *p = part + q;
    int b = g;
    for (; b + (SP_U - 1) * SP_G < nblk; b += SP_U * SP_G)
#pragma unroll
      for (int u = 0; u < SP_U; ++u) s[u] += p[(size_t)(b + u * SP_G) * n];
    for (; b < nblk; b += SP_G) s[0] += p[(size_t)b * n];
  }
  red[g][threadIdx.x] = (s[0] + s[1]) + (s[2] + s[3]);
  __syncthreads();
  if (g != 0 || q >= n) return;
  float r = 0.0f;
#pragma unroll
  for (int k = 0; k < SP_G; ++k) r += red[k][threadIdx.x];
  if (q < nw) dw[q] = r;
  else db[q - nw] = r;
}

// ---------------------------------------------------------------------------
// pooling, upsampling and their backward passes (32 channels).  Two
// workgroups per tile, eight lanes per pixel (four channels each), so a
// wavefront reads and writes whole 64-byte channel vectors of 8 neighbouring
// pixels.
// ---------------------------------------------------------------------------
#define NET_PIXEL8(V)                                                 \
  const NTile t = V.tiles[blockIdx.x >> 1];                           \
  const int px = (int)(threadIdx.x >> 3), k = 4 * (int)(threadIdx.x & 7); \
  const int r = t.r0 + 2 * (int)(blockIdx.x & 1) + (px >> 4), c = t.c0 + (px & 15);

__global__ void __launch_bounds__(256) k_pool(LevelView F, LevelView C, const uint16_t *__restrict__ x,
                                              uint16_t *__restrict__ y) {
  NET_PIXEL8(C)
  const NImg fm = F.img[t.img];
  const NTile &cm = t;
  if (r >= cm.rows || c >= cm.cols) return;
  const long long q = cm.off + (long long)r * cm.cols + c;
  float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int fr = 2 * r + a, fc = 2 * c + b;
      if (fr < fm.rows && fc < fm.cols) {
        const s4 v = ld4(x + (fm.off + (long long)fr * fm.cols + fc) * 32 + k);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += bf2f((uint16_t)v[e]);
      }
    }
  s4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = (short)f2bf(0.25f * s[e]);
  st4(y + q * 32 + k, o);
}

__global__ void __launch_bounds__(256) k_upadd(LevelView F, LevelView C, const uint16_t *__restrict__ a,
                                               const uint16_t *__restrict__ b, uint16_t *__restrict__ y) {
  NET_PIXEL8(F)
  const NImg cm = C.img[t.img];
  const NTile &fm = t;
  if (r >= fm.rows || c >= fm.cols) return;
  const long long p = fm.off + (long long)r * fm.cols + c;
  const long long q = cm.off + (long long)(r >> 1) * cm.cols + (c >> 1);
  const s4 va = ld4(a + p * 32 + k), vb = ld4(b + q * 32 + k);
  s4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = (short)f2bf(bf2f((uint16_t)va[e]) + bf2f((uint16_t)vb[e]));
  st4(y + p * 32 + k, o);
}

__global__ void __launch_bounds__(256) k_gpool(LevelView F, LevelView C, const uint16_t *__restrict__ a,
                                               const uint16_t *__restrict__ pc, const uint16_t *__restrict__ yact,
                                               uint16_t *__restrict__ g) {
  NET_PIXEL8(F)
  const NTile &fm = t;
  if (r >= fm.rows || c >= fm.cols) return;
  const long long p = fm.off + (long long)r * fm.cols + c;
  const s4 ya = ld4(yact + p * 32 + k);
  s4 va = s4{0, 0, 0, 0}, vc = s4{0, 0, 0, 0};
  if (a) va = ld4(a + p * 32 + k);
  if (pc) {
    const NImg cm = C.img[t.img];
    vc = ld4(pc + (cm.off + (long long)(r >> 1) * cm.cols + (c >> 1)) * 32 + k);
  }
  s4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float s = bf2f((uint16_t)va[e]) + 0.25f * bf2f((uint16_t)vc[e]);
    o[e] = (bf2f((uint16_t)ya[e]) > 0.0f) ? (short)f2bf(s) : (short)0;
  }
  st4(g + p * 32 + k, o);
}

__global__ void __launch_bounds__(256) k_gup(LevelView F, LevelView C, const uint16_t *__restrict__ a,
                                             const uint16_t *__restrict__ yact, uint16_t *__restrict__ g) {
  NET_PIXEL8(C)
  const NImg fm = F.img[t.img];
  const NTile &cm = t;
  if (r >= cm.rows || c >= cm.cols) return;
  const long long q = cm.off + (long long)r * cm.cols + c;
  float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int da = 0; da < 2; ++da)
#pragma unroll
    for (int db = 0; db < 2; ++db) {
      const int fr = 2 * r + da, fc = 2 * c + db;
      if (fr < fm.rows && fc < fm.cols) {
        const s4 v = ld4(a + (fm.off + (long long)fr * fm.cols + fc) * 32 + k);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += bf2f((uint16_t)v[e]);
      }
    }
  const s4 ya = ld4(yact + q * 32 + k);
  s4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = (bf2f((uint16_t)ya[e]) > 0.0f) ? (short)f2bf(s[e]) : (short)0;
  st4(g + q * 32 + k, o);
}

// ---------------------------------------------------------------------------
// loss, optimiser, weight packing
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_loss(LevelView L, const float *__restrict__ out, const float *__restrict__ tg,
                                              const float *__restrict__ wt, float scale, uint16_t *__restrict__ g,
                                              double *__restrict__ partial) {
  __shared__ double red[256];
  double acc = 0.0;
  const int lane = threadIdx.x & 63;
  const int wid = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (wid < L.ntiles) {
    const NTile t = L.tiles[wid];
    const NTile &im = t;
    const int r = t.r0 + (lane >> 4), c = t.c0 + (lane & 15);
    if (r < im.rows && c < im.cols) {
      const long long p = im.off + (long long)r * im.cols + c;
      const float w = wt[p];
      const float d0 = out[2 * p] - tg[2 * p], d1 = out[2 * p + 1] - tg[2 * p + 1];
      acc = (double)w * ((double)d0 * d0 + (double)d1 * d1);
      const s4 z = s4{0, 0, 0, 0};
      s4 o = z;
      o[0] = (short)f2bf(2.0f * scale * w * d0);
      o[1] = (short)f2bf(2.0f * scale * w * d1);
      st4(g + p * IMAU_NET_OUT, o);
#pragma unroll
      for (int k = 4; k < IMAU_NET_OUT; k += 4) st4(g + p * IMAU_NET_OUT + k, z);
    }
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ void __launch_bounds__(256) k_adam(long long n, float *__restrict__ p, const float *__restrict__ g,
                                              float *__restrict__ m, float *__restrict__ v, float lr, float b1,
                                              float b2, float eps, float bc1, float bc2) {
  const long long q = (long long)blockIdx.x * 256 + threadIdx.x;
  if (q >= n) return;
  const float gq = g[q];
  const float mq = b1 * m[q] + (1.0f - b1) * gq;
  const float vq = b2 * v[q] + (1.0f - b2) * gq * gq;
  m[q] = mq;
  v[q] = vq;
  p[q] -= lr * (mq / bc1) / (sqrtf(vq / bc2) + eps);
}

__global__ void __launch_bounds__(256) k_pack(int cin, int cout, const float *__restrict__ w, uint16_t *__restrict__ wf,
                                              uint16_t *__restrict__ wt) {
  const int q = blockIdx.x * 256 + threadIdx.x;
  if (q >= 9 * cout * cin) return;
  const int tap = q / (cout * cin), co = (q / cin) % cout, ci = q % cin;
  wf[q] = f2bf(w[q]);
  wt[(tap * cin + ci) * cout + co] = f2bf(w[((8 - tap) * cout + co) * cin + ci]);
}

inline int nblk4(int ntiles) { return (ntiles + 3) / 4; }

}  // namespace

namespace imau {
namespace net {

bool conv(hipStream_t s, const LevelView &L, int cin, int cout, const uint16_t *x, const uint16_t *w,
          const float *bias, int relu, void *y, int yf32) {
  if (L.ntiles == 0) return true;
  // a multiple of 8 workgroups (one run of tiles per XCD), at most as many as
  // are resident at once (registers: two per CU for 32 -> 32 channels, else
  // three); more of them load the weights again: 32 -> 32 over 1.3 million
  // pixels took 40 us with 512, 46 with 768 and 1536, 16 -> 32 took 33 us with
  // 768, 39 with 512 and 1024
  const int nb = std::min((nblk4(L.ntiles) + 7) / 8 * 8, cin == 32 && cout == 32 ? 512 : 768);
#define CONV(CI, CO, F32)                                                                                        \
  hipLaunchKernelGGL((k_conv<CI, CO, F32>), dim3(nb), dim3(256), 0, s, L.tiles, L.ntiles, x, w, bias, relu, y)
  if (cin == 16 && cout == 32 && !yf32) CONV(16, 32, false);
  else if (cin == 32 && cout == 32 && !yf32) CONV(32, 32, false);
  else if (cin == 32 && cout == 16 && yf32) CONV(32, 16, true);
  else if (cin == 32 && cout == 16 && !yf32) CONV(32, 16, false);
  else return false;
#undef CONV
  return true;
}

int dw_blocks(const LevelView &L) { return std::max(1, std::min(L.ntiles, 1024)); }

bool conv_dw(hipStream_t s, const LevelView &L, int cin, int cout, const uint16_t *g, const uint16_t *x, float *dw,
             float *db, float *part) {
  const int nb = dw_blocks(L);
  const int n = 9 * cout * cin + cout;
  if (L.ntiles == 0) return false;
  if (cin == 16 && cout == 32)
    hipLaunchKernelGGL((k_conv_dw<16, 32>), dim3(nb), dim3(256), 0, s, L.tiles, L.ntiles, g, x, part);
  else if (cin == 32 && cout == 32)
    hipLaunchKernelGGL((k_conv_dw<32, 32>), dim3(nb), dim3(256), 0, s, L.tiles, L.ntiles, g, x, part);
  else if (cin == 32 && cout == 16)
    hipLaunchKernelGGL((k_conv_dw<32, 16>), dim3(nb), dim3(256), 0, s, L.tiles, L.ntiles, g, x, part);
  else
    return false;
  sum_partials(s, nb, n, part, dw, 9 * cout * cin, db);
  return true;
}

void sum_partials(hipStream_t s, int nblk, int n, const float *part, float *dw, int nw, float *db) {
  hipLaunchKernelGGL(k_sum_partials, dim3((n + SP_Q - 1) / SP_Q), dim3(SP_Q, SP_G), 0, s, nblk, n, part, dw, nw, db);
}

// two workgroups of 256 threads (32 pixels x 8 lanes) per 64-pixel tile
void pool(hipStream_t s, const LevelView &F, const LevelView &C, const uint16_t *x, uint16_t *y) {
  if (C.ntiles) hipLaunchKernelGGL(k_pool, dim3(2 * C.ntiles), dim3(256), 0, s, F, C, x, y);
}
void upadd(hipStream_t s, const LevelView &F, const LevelView &C, const uint16_t *a, const uint16_t *b, uint16_t *y) {
  if (F.ntiles) hipLaunchKernelGGL(k_upadd, dim3(2 * F.ntiles), dim3(256), 0, s, F, C, a, b, y);
}
void gpool(hipStream_t s, const LevelView &F, const LevelView &C, const uint16_t *a, const uint16_t *pc,
           const uint16_t *yact, uint16_t *g) {
  if (F.ntiles) hipLaunchKernelGGL(k_gpool, dim3(2 * F.ntiles), dim3(256), 0, s, F, C, a, pc, yact, g);
}
void gup(hipStream_t s, const LevelView &F, const LevelView &C, const uint16_t *a, const uint16_t *yact, uint16_t *g) {
  if (C.ntiles) hipLaunchKernelGGL(k_gup, dim3(2 * C.ntiles), dim3(256), 0, s, F, C, a, yact, g);
}
int loss_blocks(const LevelView &L) { return std::max(1, nblk4(L.ntiles)); }
void loss(hipStream_t s, const LevelView &L, const float *out, const float *t, const float *w, float scale,
          uint16_t *g, double *partial) {
  hipLaunchKernelGGL(k_loss, dim3(loss_blocks(L)), dim3(256), 0, s, L, out, t, w, scale, g, partial);
}
void adam(hipStream_t s, long long n, float *p, const float *g, float *m, float *v, float lr, float b1, float b2,
          float eps, float bc1, float bc2) {
  if (n > 0)
    hipLaunchKernelGGL(k_adam, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, p, g, m, v, lr, b1, b2, eps,
                       bc1, bc2);
}
void pack(hipStream_t s, int cin, int cout, const float *w, uint16_t *wf, uint16_t *wt) {
  const int n = 9 * cin * cout;
  hipLaunchKernelGGL(k_pack, dim3((n + 255) / 256), dim3(256), 0, s, cin, cout, w, wf, wt);
}

}  // namespace net
}  // namespace imau
