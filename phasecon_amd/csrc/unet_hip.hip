// unet_hip.hip -- learned warm start for the MBIR solver: a 3-level 3D U-Net
// (channels c / 2c / 4c, two 3x3x3 convolutions per level, average pooling,
// nearest up-sampling, concatenated skips, residual output) trained and run
// on the GPU with BF16 MFMA kernels and FP32 accumulation.
//
// The network has no counterpart in the reference: it maps the normalised
// back-projection  sum(w a y) / sum(w a^2)  of every voxel to the converged
// MBIR image, and the MBIR solver then starts from its output instead of from
// zero (it always runs to convergence).
//
// Layout: activations and their gradients are BF16, channels last,
// [n][z][y][x][channel stride]; a layer reads / writes a channel range
// (offset, count) of a buffer.  A decoder layer's input, the concatenation of
// an up-sampled half-resolution buffer and a skip, is read from both places
// and never written out (its gradient is).  Parameters, gradients and Adam
// moments: FP32, one buffer each, per layer [cout][27][cin] (tap = (dz+1)*9 +
// (dy+1)*3 + (dx+1)) then [cout]; BF16 copies of the weights in MFMA fragment order for the forward
// GEMM and, with taps flipped and channels swapped, the backward-data GEMM.
//
// Kernels
//   k_conv       implicit-GEMM 3x3x3 convolution, v_mfma_f32_16x16x32_bf16,
//                the tile's input with halo in LDS; forward (bias, ReLU) and
//                backward-data (flipped weights)
//   k_conv_dw    weight and bias gradient: 16 x 16 channels x 27 taps per
//                workgroup, reduced over voxel rows with MFMA, FP32 sums per
//                workgroup that k_dw_sum adds up in their order
//   k_pool / k_pool_bwd, k_up_bwd, k_relu_bwd, k_mse, k_adam, k_pack
//                elementwise / reduction helpers
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "copy_out.h"
#include "unet_hip.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16;

thread_local std::string g_err;
int fail(const std::string& m) {
  g_err = m;
  return -1;
}
#define HIP_OK(call)                                                      \
  do {                                                                    \
    hipError_t e_ = (call);                                               \
    if (e_ != hipSuccess)                                                 \
      return fail(std::string(#call) + ": " + hipGetErrorString(e_));     \
  } while (0)

// FP32 -> BF16, round to nearest even (NaN kept quiet)
__host__ __device__ inline u16 f2bf(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u16)((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (u16)(u >> 16);
}
__host__ __device__ inline float bf2f(u16 h) {
  uint32_t u = (uint32_t)h << 16;
  float f;
  memcpy(&f, &u, 4);
  return f;
}

// Two floats to a dword of BF16 (round to nearest even, v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t pk_bf16(float lo, float hi) {
  typedef float float2_t __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(float2_t{lo, hi}, bf16x2));
}

inline int rup(int a, int b) { return (a + b - 1) / b * b; }

// A channel range of a channels-last BF16 buffer.
struct Chan {
  u16* p;
  int cs, co;  // channel stride, first channel
};

// Input channels of a convolution: a channel range of one buffer, or (up)
// the concatenation [nearest 2x up-sampled range of a half-resolution buffer
// | range], which is then never written out.
struct ConvIn {
  const u16* p;
  int cs, co;
  const u16* up;  // may be null
  int cs_up, co_up, c_up;  // stride, first channel, channels (a multiple of 8)
};

struct ConvArgs {
  ConvIn in;
  const u16* w;  // fragments of k_pack
  const float* bias;
  u16* out;      // BF16 output channel range (may be null)
  int cs_out, co_out;
  float* out32;  // FP32 output [v][cout] (may be null)
  const float* add32;  // added to out32's channel 0 (may be null), stride cs_add
  int cs_add;
  int N, D, H, W;
  int cin_pad, cout, nt, relu;
  int lfx, lty, ltz;  // a workgroup's output tile: 16 fx x ty x tz voxels (log2)
  int ntx, ntz;       // tiles along x and z
  int by, bz;         // first tile of the launch along y and along (volume, z)
};

// Channels of the input staged at once: all of up to 32, else 32, or 24 where
// that leaves no remainder and 32 does (two tiles with their halo then fit a
// CU's LDS).
__host__ __device__ inline int conv_chunk(int cin_pad) {
  return cin_pad <= 32 ? cin_pad : (cin_pad % 32 != 0 && cin_pad % 24 == 0 ? 24 : 32);
}
// MFMA steps (4 groups of 8 channels of one tap) of a chunk of c channels.
__host__ __device__ inline int conv_steps(int c) { return (27 * (c / 8) + 3) / 4; }
__host__ __device__ inline int conv_steps_all(int cin_pad) {
  const int cc = conv_chunk(cin_pad), rest = cin_pad % cc;
  return cin_pad / cc * conv_steps(cc) + (rest ? conv_steps(rest) : 0);
}

// The 16-byte channel group cg of input voxel (n, z, y, x), in bounds.
__device__ __forceinline__ uint4 conv_load(const ConvIn& I, int n, int z, int y, int x, int D,
                                           int H, int W, int c) {
  const u16* p;
  if (c < I.c_up)
    p = I.up + (((long long)(n * (D >> 1) + (z >> 1)) * (H >> 1) + (y >> 1)) * (W >> 1) +
                (x >> 1)) * I.cs_up + I.co_up + c;
  else
    p = I.p + (((long long)(n * D + z) * H + y) * W + x) * I.cs + I.co + (c - I.c_up);
  return *reinterpret_cast<const uint4*>(p);
}

// 3x3x3 convolution, an implicit GEMM on v_mfma_f32_16x16x32_bf16.  A
// workgroup stages its output tile's input with a one-voxel halo (zeros
// outside the volume) in LDS once per channel chunk; its four wavefronts take
// MV fragments of 16 voxels each (along x) and the NT output channel tiles of
// 16 of its split (blockIdx.x counts splits, then tiles along x).  One step
// multiplies 4 groups of 8 input channels of one tap each (a lane's k group
// lane / 16) by weights that k_pack laid out in fragment order (1 KiB per step
// and channel tile): one LDS read of 16 bytes per voxel fragment and no bounds
// test.  Weights are the A operand, so
// a lane ends with 4 consecutive channels of one voxel.
// Bound by instruction issue around the MFMAs: staging, and at NT = 1 the LDS
// reads (1 KiB per MFMA).  Reading the fragments from global memory, with the
// taps' bounds and 64-bit addresses formed per step, spent ten times the
// MFMAs' cycles on that arithmetic.  16 volumes of 8x256x256, 16 base
// channels: the 11 layers 5.9 -> 2.45 ms (0.31 PFLOP/s, without writing the
// up-sampled halves: another 0.38 ms); 16 to 16 channels at full size 0.87 ->
// 0.33 ms, 48 to 16 1.9 -> 0.67 ms.
constexpr int kConvPre = 4;
template <int NT, int MV>
__global__ __launch_bounds__(256) void k_conv(ConvArgs a) {
  constexpr int kPre = NT <= 2 ? kConvPre : 2;
  constexpr int kRows = 6;  // rows of a wavefront at tile 32 x 4 x 2
  extern __shared__ uint4 s_in[];
  __shared__ int s_off[4 * 27];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, kg = lane >> 4;
  const int fx = 1 << a.lfx, HX = 16 * fx + 2, HY = (1 << a.lty) + 2, HZ = (1 << a.ltz) + 2;
  const unsigned bz = blockIdx.z + a.bz;
  const int split = blockIdx.x / a.ntx, n = bz / a.ntz;
  const int x0 = (blockIdx.x - split * a.ntx) * 16 * fx, y0 = (blockIdx.y + a.by) << a.lty;
  const int z0 = (bz - n * a.ntz) << a.ltz;
  const int t0 = split * NT;
  int fb[MV];  // staged voxel index of the fragment's tap (-1, -1, -1)
#pragma unroll
  for (int f = 0; f < MV; ++f) {
    const int q = wave * MV + f, qr = q >> a.lfx;
    fb[f] = ((qr >> a.lty) * HY + (qr & ((1 << a.lty) - 1))) * HX + (q & (fx - 1)) * 16 + m;
  }
  floatx4 acc[MV][NT];
#pragma unroll
  for (int f = 0; f < MV; ++f)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[f][t] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int CC = conv_chunk(a.cin_pad);
  const int invy = (65536 + HY - 1) / HY;  // row / HY = row invy >> 16 for row < 1000
  const uint4* wp = reinterpret_cast<const uint4*>(a.w) + (size_t)t0 * 64 + lane;
  for (int c0 = 0; c0 < a.cin_pad; c0 += CC) {
    const int cg = (a.cin_pad - c0 < CC ? a.cin_pad - c0 : CC) >> 3;
    const int inv = (65536 + cg - 1) / cg;  // i / cg = i inv >> 16 for i < 9000
    const int steps = conv_steps(8 * cg);
    if (c0) __syncthreads();
    for (int i = tid; i < 4 * steps; i += 256) {
      // a group past the last tap has zero weights: it reads the first one
      const int g = i < 27 * cg ? i : 0, tap = g / cg;
      s_off[i] = ((tap / 9 * HY + tap / 3 % 3) * HX + tap % 3) * cg + (g - tap * cg);
    }
    // the rows' 16 fx inner voxels: a wavefront takes whole rows, so that a
    // row's address and bounds are scalar; kRows rows in flight before their
    // LDS writes
    for (int i0 = 0; i0 < 16 * fx * cg; i0 += 64) {
      const int i = i0 + lane, v = (i * inv) >> 16, g = i - v * cg, c = c0 + 8 * g;
      const bool xok = i < 16 * fx * cg && x0 + v < a.W, up = c < a.in.c_up;
      const unsigned o1 = (unsigned)(v * a.in.cs + c - a.in.c_up) * 2u;
      const unsigned o2 = (unsigned)((v >> 1) * a.in.cs_up + c) * 2u;
      for (int r0 = wave; r0 < HY * HZ; r0 += 4 * kRows) {
        uint4 raw[kRows];
#pragma unroll
        for (int j = 0; j < kRows; ++j) {
          const int row = r0 + 4 * j, rz = (row * invy) >> 16;
          const int z = z0 + rz - 1, y = y0 + (row - rz * HY) - 1;
          raw[j] = make_uint4(0u, 0u, 0u, 0u);
          if (row < HY * HZ && z >= 0 && z < a.D && y >= 0 && y < a.H) {
            const char* p1 = reinterpret_cast<const char*>(
                a.in.p + ((long long)((n * a.D + z) * a.H + y) * a.W + x0) * a.in.cs + a.in.co);
            if (xok && !up) raw[j] = *reinterpret_cast<const uint4*>(p1 + o1);
            if (a.in.up != nullptr) {
              const char* p2 = reinterpret_cast<const char*>(
                  a.in.up + ((long long)((n * (a.D >> 1) + (z >> 1)) * (a.H >> 1) + (y >> 1)) *
                             (a.W >> 1) + (x0 >> 1)) * a.in.cs_up + a.in.co_up);
              if (xok && up) raw[j] = *reinterpret_cast<const uint4*>(p2 + o2);
            }
          }
        }
#pragma unroll
        for (int j = 0; j < kRows; ++j) {
          const int row = r0 + 4 * j;
          if (row < HY * HZ && i < 16 * fx * cg) s_in[(row * HX + v + 1) * cg + g] = raw[j];
        }
      }
    }
    // and their two halo voxels
    for (int i = tid; i < HY * HZ * 2 * cg; i += 256) {
      const int rs = (i * inv) >> 16, g = i - rs * cg, row = rs >> 1;
      const int rz = (row * invy) >> 16, z = z0 + rz - 1, y = y0 + (row - rz * HY) - 1;
      const int v = (rs & 1) * (HX - 1), x = x0 + v - 1;
      uint4 raw = make_uint4(0u, 0u, 0u, 0u);
      if (z >= 0 && z < a.D && y >= 0 && y < a.H && x >= 0 && x < a.W)
        raw = conv_load(a.in, n, z, y, x, a.D, a.H, a.W, c0 + 8 * g);
      s_in[(row * HX + v) * cg + g] = raw;
    }
    __syncthreads();
    // weights kPre steps ahead (the buffer holds kConvPre steps past the last)
    uint4 bw[kPre][NT];
#pragma unroll
    for (int p = 0; p < kPre; ++p)
#pragma unroll
      for (int t = 0; t < NT; ++t) bw[p][t] = wp[((size_t)p * a.nt + t) * 64];
    for (int s0 = 0; s0 < steps; s0 += kPre) {
#pragma unroll
      for (int p = 0; p < kPre; ++p) {
        if (s0 + p >= steps) break;
        uint4 bc[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          bc[t] = bw[p][t];
          bw[p][t] = wp[((size_t)(s0 + p + kPre) * a.nt + t) * 64];
        }
        const int off = s_off[4 * (s0 + p) + kg];
#pragma unroll
        for (int f = 0; f < MV; ++f) {
          const bf16x8 v = __builtin_bit_cast(bf16x8, s_in[fb[f] * cg + off]);
#pragma unroll
          for (int t = 0; t < NT; ++t)
            acc[f][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8, bc[t]), v, acc[f][t], 0, 0, 0);
        }
      }
    }
    wp += (size_t)steps * a.nt * 64;
  }
  // a lane's 4 channels of tile t: 16 (t0 + t) + 4 kg; the fragment's first
  // voxel is scalar, the lane's place in it is the same for all fragments
  float bias[NT][4];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int co = (t0 + t) * 16 + 4 * kg + j;
      bias[t][j] = a.bias && co < a.cout ? a.bias[co] : 0.f;
    }
  const int lo_out = m * a.cs_out + t0 * 16 + 4 * kg;
#pragma unroll
  for (int f = 0; f < MV; ++f) {
    const int q = wave * MV + f, qr = q >> a.lfx, xf = x0 + (q & (fx - 1)) * 16;
    const int y = y0 + (qr & ((1 << a.lty) - 1)), z = z0 + (qr >> a.lty);
    if (y >= a.H || z >= a.D || xf + m >= a.W) continue;
    const long long vf = ((long long)(n * a.D + z) * a.H + y) * a.W + xf;
    u16* const of = a.out + vf * a.cs_out + a.co_out;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int co = (t0 + t) * 16 + 4 * kg;
      if (co >= a.cout) continue;
      float o[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        o[j] = acc[f][t][j] + bias[t][j];
        if (a.relu) o[j] = fmaxf(o[j], 0.f);
      }
      if (a.out32) {
        const long long vo = vf + m;
        for (int j = 0; j < 4; ++j)
          if (co + j < a.cout)
            a.out32[vo * a.cout + co + j] =
                o[j] + (a.add32 && co + j == 0 ? a.add32[vo * a.cs_add] : 0.f);
      }
      if (!a.out) continue;
      u16* dst = of + lo_out + t * 16;
      const uint32_t lo = pk_bf16(o[0], o[1]), hi = pk_bf16(o[2], o[3]);
      if (co + 3 < a.cout) {
        *reinterpret_cast<uint2*>(dst) = make_uint2(lo, hi);
      } else {
        const u16 h[4] = {(u16)lo, (u16)(lo >> 16), (u16)hi, (u16)(hi >> 16)};
        for (int j = 0; j < 4; ++j)
          if (co + j < a.cout) dst[j] = h[j];
      }
    }
  }
}

struct DwArgs {
  const u16* g;  // output gradient channel range (the GEMM's M side)
  int cs_g, co_g, cg;  // cg: readable channels from co_g on (a multiple of 8)
  ConvIn in;     // layer input
  float* part;   // [workgroup along x][cout][27][cin] sums, then [..][cout] of g
  size_t stride; // floats per workgroup
  int N, D, H, W;
  int cin, cin_pad, cout;
  int ntx, nty, ntz, per;  // tiles per axis, tiles per workgroup
};

constexpr int kDwX = 32, kDwY = 4, kDwZ = 2;  // output rows of a tile: 8 of 32 voxels
constexpr int kDwIn = (kDwY + 2) * (kDwZ + 2);
// LDS strides of a channel's rows, in 16-byte units: odd, so that 16
// channels at one offset fall on different banks
constexpr int kDwSi = kDwIn * 4 + 1, kDwSg = kDwY * kDwZ * 4 + 1;

// 8 channels of two neighbouring voxels as 8 pairs (v0, v1), one dword each,
// into rows of stride `st` bytes.
__device__ __forceinline__ void dw_put(char* dst, int st, uint4 v0, uint4 v1) {
  const uint32_t a[4] = {v0.x, v0.y, v0.z, v0.w}, b[4] = {v1.x, v1.y, v1.z, v1.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    *reinterpret_cast<uint32_t*>(dst + (2 * i) * st) = (a[i] & 0xffffu) | (b[i] << 16);
    *reinterpret_cast<uint32_t*>(dst + (2 * i + 1) * st) = (a[i] >> 16) | (b[i] & 0xffff0000u);
  }
}

// dW[co][tap][ci] = sum over voxels of g[v][co] in[v + d_tap][ci], and
// db[co] = sum g[v][co], partial sums per workgroup: a workgroup takes 16
// output channels (blockIdx.z), 16 input channels (blockIdx.y) and `per` tiles
// of 8 output rows of 32 voxels; the MFMA's k runs over a row's 32 input
// voxels.  Per tile the input rows with their y and z halo and three copies of
// the gradient rows, shifted by -1, 0 and 1 voxels against them, go to LDS
// transposed (channel rows, voxels contiguous), so that every fragment is one
// aligned 16-byte read and the three x taps share the input fragment.  A
// wavefront takes two of the rows and all 27 taps: 9 input and 3 gradient
// fragments per 27 MFMAs, 112 accumulators with the bias's (AGPRs) beside 124
// VGPRs and 32 bytes of scratch per lane, two wavefronts per SIMD.  The
// wavefronts' sums meet in LDS, the workgroups' in k_dw_sum (1024 workgroups'
// atomics on one gradient took 160 of the 225 us of a 16-to-16-channel layer
// over 262144 voxels).  Bound by the LDS traffic (staging and fragments);
// gathering both operands voxel by voxel from global memory was bound by its
// 16 scalar 2-byte loads per MFMA.  8 volumes of 8x64x64, 16 base channels: the
// 11 layers 5.01 ms (and 0.24 ms for the bias sums) -> 0.24 ms; 16 to 16
// channels at full size 0.46 -> 0.019 ms.
__global__ __launch_bounds__(256) void k_conv_dw(DwArgs a) {
  __shared__ uint4 s_i[16 * kDwSi];
  __shared__ uint4 s_g[3 * 16 * kDwSg];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, kg = lane >> 4;
  const int ci0 = blockIdx.y * 16, co0 = blockIdx.z * 16;
  const bool bias = blockIdx.y == 0;
  float* part = a.part + blockIdx.x * a.stride;
  floatx4 acc[27], accb = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < 27; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
  const uint4 ones = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);
  const long long tiles = (long long)a.N * a.ntz * a.nty * a.ntx;
  const long long tb = (long long)blockIdx.x * a.per;
  const long long te = tb + a.per < tiles ? tb + a.per : tiles;
  for (long long tile = tb; tile < te; ++tile) {
    long long q = tile;
    const int x0 = (int)(q % a.ntx) * kDwX;
    q /= a.ntx;
    const int y0 = (int)(q % a.nty) * kDwY;
    q /= a.nty;
    const int z0 = (int)(q % a.ntz) * kDwZ, n = (int)(q / a.ntz);
    __syncthreads();  // the previous tile has been read
    // input rows: a thread takes two voxels (x, x + 1) of one channel group
    for (int i = tid; i < kDwIn * 2 * 16; i += 256) {
      const int px = i & 15, g = (i >> 4) & 1, row = i >> 5;
      const int rz = row / (kDwY + 2), z = z0 + rz - 1, y = y0 + row - rz * (kDwY + 2) - 1;
      const int x = x0 + 2 * px, c = ci0 + 8 * g;
      const bool ok = z >= 0 && z < a.D && y >= 0 && y < a.H && c < a.cin_pad;
      const uint4 v0 = ok && x < a.W ? conv_load(a.in, n, z, y, x, a.D, a.H, a.W, c) : zero;
      const uint4 v1 =
          ok && x + 1 < a.W ? conv_load(a.in, n, z, y, x + 1, a.D, a.H, a.W, c) : zero;
      dw_put(reinterpret_cast<char*>(s_i + 8 * g * kDwSi + row * 4) + 4 * px, 16 * kDwSi, v0, v1);
    }
    // gradient rows: copy d holds g(x' - (d - 1)) at input voxel x'
    for (int i = tid; i < kDwY * kDwZ * 2 * 16; i += 256) {
      const int px = i & 15, g = (i >> 4) & 1, row = i >> 5;
      const int z = z0 + row / kDwY, y = y0 + row % kDwY;
      const int x = x0 + 2 * px, c = co0 + 8 * g;
      const bool ok = z < a.D && y < a.H && c < a.cg;
      const u16* src = a.g + (((long long)(n * a.D + z) * a.H + y) * a.W) * a.cs_g + a.co_g + c;
      uint4 v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int xx = x + j - 1;
        v[j] = ok && xx >= 0 && xx < a.W
                   ? *reinterpret_cast<const uint4*>(src + (long long)xx * a.cs_g) : zero;
      }
      char* dst = reinterpret_cast<char*>(s_g + 8 * g * kDwSg + row * 4) + 4 * px;
      dw_put(dst, 16 * kDwSg, v[2], v[3]);                          // tap dx = -1: g(x' + 1)
      dw_put(dst + 16 * 16 * kDwSg, 16 * kDwSg, v[1], v[2]);        // dx = 0
      dw_put(dst + 2 * 16 * 16 * kDwSg, 16 * kDwSg, v[0], v[1]);    // dx = 1: g(x' - 1)
    }
    __syncthreads();
#pragma unroll
    for (int r2 = 0; r2 < kDwY * kDwZ / 4; ++r2) {
      const int row = wave + 4 * r2, rz = row / kDwY, ry = row % kDwY;
      bf16x8 gv[3];
#pragma unroll
      for (int d = 0; d < 3; ++d)
        gv[d] = __builtin_bit_cast(bf16x8, s_g[(d * 16 + m) * kDwSg + row * 4 + kg]);
      if (bias)
        accb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            gv[1], __builtin_bit_cast(bf16x8, ones), accb, 0, 0, 0);
#pragma unroll
      for (int p = 0; p < 9; ++p) {
        const bf16x8 iv = __builtin_bit_cast(
            bf16x8, s_i[m * kDwSi + ((rz + p / 3) * (kDwY + 2) + ry + p % 3) * 4 + kg]);
#pragma unroll
        for (int d = 0; d < 3; ++d)
          acc[3 * p + d] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(gv[d], iv, acc[3 * p + d], 0, 0, 0);
      }
    }
  }
  // the four wavefronts' sums, in wavefront order (9 taps at a time fit the
  // input rows' buffer), then the workgroup's into part; a lane holds input
  // channel ci0 + m of output channels co0 + 4 kg + 0..3
  float* red = reinterpret_cast<float*>(s_i);  // [9 taps][4][64], 4 wavefronts of it in turn
#pragma unroll
  for (int third = 0; third < 3; ++third) {
    for (int w = 0; w < 4; ++w) {
      __syncthreads();
      if (wave == w) {
#pragma unroll
        for (int p = 0; p < 9; ++p)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float* r = red + (p * 4 + q) * 64 + lane;
            *r = (w ? *r : 0.f) + acc[9 * third + p][q];
          }
      }
    }
    __syncthreads();
    for (int i = tid; i < 9 * 256; i += 256) {
      const int l = i & 63, q = (i >> 6) & 3, tap = 9 * third + (i >> 8);
      const int co = co0 + 4 * (l >> 4) + q, ci = ci0 + (l & 15);
      const float v = red[i];
      if (co < a.cout && ci < a.cin) part[((size_t)co * 27 + tap) * a.cin + ci] = v;
    }
  }
  // every column of accb holds the row sums of g
  if (bias) {
    for (int w = 0; w < 4; ++w) {
      __syncthreads();
      if (wave == w && m == 0)
#pragma unroll
        for (int q = 0; q < 4; ++q) red[4 * kg + q] = (w ? red[4 * kg + q] : 0.f) + accb[q];
    }
    __syncthreads();
    if (tid < 16 && co0 + tid < a.cout)
      part[(size_t)a.cout * 27 * a.cin + co0 + tid] = red[tid];
  }
}

// dw[i] := the sum of the workgroups' partials, in their order
__global__ void k_dw_sum(const float* __restrict__ part, int np, size_t n, float* dw) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float s = 0.f;
#pragma unroll 8
  for (int p = 0; p < np; ++p) s += part[p * n + i];
  dw[i] = s;
}

// 8 BF16 channels of one 16-byte group as floats, and back
__device__ __forceinline__ void unpack8(uint4 r, float f[8]) {
  const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = bf2f((u16)(w[i] & 0xffffu));
    f[2 * i + 1] = bf2f((u16)(w[i] >> 16));
  }
}
__device__ __forceinline__ uint4 pack8(const float f[8]) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = pk_bf16(f[2 * i], f[2 * i + 1]);
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// The helpers below take one thread per voxel and 8 channels (16-byte
// accesses; channel counts, strides and offsets are multiples of 8).

// 2x2x2 average pooling: out (D/2, H/2, W/2) channel range := mean of 8.
__global__ void k_pool(const u16* in, int cs_in, int co_in, u16* out, int cs_out, int co_out,
                       int C, int N, int D, int H, int W) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int D2 = D / 2, H2 = H / 2, W2 = W / 2, C8 = C / 8;
  const long long total = (long long)N * D2 * H2 * W2 * C8;
  if (i >= total) return;
  const int c = (int)(i % C8) * 8;
  long long v = i / C8;
  const long long dst = v * cs_out + co_out + c;
  const int x = (int)(v % W2);
  v /= W2;
  const int y = (int)(v % H2);
  v /= H2;
  const int z = (int)(v % D2);
  const long long n = v / D2;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    const long long src = ((n * D + 2 * z + (d >> 2)) * H + 2 * y + ((d >> 1) & 1)) * W + 2 * x + (d & 1);
    float f[8];
    unpack8(*reinterpret_cast<const uint4*>(in + src * cs_in + co_in + c), f);
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] += f[j];
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) s[j] *= 0.125f;
  *reinterpret_cast<uint4*>(out + dst) = pack8(s);
}

// gradient of the pooling: gin (D, H, W) channel range += gout / 8
__global__ void k_pool_bwd(const u16* gout, int cs_o, int co_o, u16* gin, int cs_i, int co_i,
                           int C, int N, int D, int H, int W) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int C8 = C / 8;
  const long long total = (long long)N * D * H * W * C8;
  if (i >= total) return;
  const int c = (int)(i % C8) * 8;
  long long v = i / C8;
  uint4* dst = reinterpret_cast<uint4*>(gin + v * cs_i + co_i + c);
  const int x = (int)(v % W);
  v /= W;
  const int y = (int)(v % H);
  v /= H;
  const int z = (int)(v % D);
  const long long n = v / D;
  const long long p = ((n * (D / 2) + z / 2) * (H / 2) + y / 2) * (W / 2) + x / 2;
  float a[8], b[8];
  unpack8(*dst, a);
  unpack8(*reinterpret_cast<const uint4*>(gout + p * cs_o + co_o + c), b);
#pragma unroll
  for (int j = 0; j < 8; ++j) a[j] += 0.125f * b[j];
  *dst = pack8(a);
}

// gradient of the nearest 2x up-sampling: gin (D, H, W) := sum of its 8
// children
__global__ void k_up_bwd(const u16* gout, int cs_o, int co_o, u16* gin, int cs_i, int co_i, int C,
                         int N, int D, int H, int W) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int C8 = C / 8;
  const long long total = (long long)N * D * H * W * C8;
  if (i >= total) return;
  const int c = (int)(i % C8) * 8;
  long long v = i / C8;
  const long long dst = v * cs_i + co_i + c;
  const int x = (int)(v % W);
  v /= W;
  const int y = (int)(v % H);
  v /= H;
  const int z = (int)(v % D);
  const long long n = v / D;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    const long long src =
        ((n * 2 * D + 2 * z + (d >> 2)) * 2 * H + 2 * y + ((d >> 1) & 1)) * 2 * W + 2 * x + (d & 1);
    float f[8];
    unpack8(*reinterpret_cast<const uint4*>(gout + src * cs_o + co_o + c), f);
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] += f[j];
  }
  *reinterpret_cast<uint4*>(gin + dst) = pack8(s);
}

// g := g where act > 0, else 0 (ReLU gradient through the stored output)
__global__ void k_relu_bwd(u16* g, int cs_g, int co_g, const u16* act, int cs_a, int co_a, int C,
                           long long V) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int C8 = C / 8;
  if (i >= V * C8) return;
  const int c = (int)(i % C8) * 8;
  const long long v = i / C8;
  uint4* dst = reinterpret_cast<uint4*>(g + v * cs_g + co_g + c);
  const uint4 r = *dst, a = *reinterpret_cast<const uint4*>(act + v * cs_a + co_a + c);
  const uint32_t rw[4] = {r.x, r.y, r.z, r.w}, aw[4] = {a.x, a.y, a.z, a.w};
  uint32_t o[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    o[j] = (bf2f((u16)(aw[j] & 0xffffu)) > 0.f ? rw[j] & 0xffffu : 0u) |
           (bf2f((u16)(aw[j] >> 16)) > 0.f ? rw[j] & 0xffff0000u : 0u);
  *dst = make_uint4(o[0], o[1], o[2], o[3]);
}

// pred = net + x (input channel 0 of cin); grad channel 0 := 2 (pred - t) / V
// (the other 7 zero); partial sums of (pred - t)^2 per block
__global__ void k_mse(const float* net, const float* x, int cin, const float* t, long long V,
                      u16* g, double* partial) {
  __shared__ double red[256];
  double s = 0.0;
  for (long long v = (long long)blockIdx.x * 256 + threadIdx.x; v < V; v += (long long)gridDim.x * 256) {
    const float d = net[v] + x[v * cin] - t[v];
    s += (double)d * d;
    *reinterpret_cast<uint4*>(g + v * 8) = make_uint4(f2bf(2.f * d / (float)V), 0u, 0u, 0u);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// x (FP32, [v][cin]) into channels 0 .. cin-1 of a BF16 buffer of stride 8
// (the others 0)
__global__ void k_in_pack(const float* x, int cin, long long V, u16* out) {
  const long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= V) return;
  float f[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) f[c] = c < cin ? x[v * cin + c] : 0.f;
  *reinterpret_cast<uint4*>(out + v * 8) = pack8(f);
}

__global__ void k_adam(float* p, const float* g, float* m, float* v, long long n, float lr,
                       float b1, float b2, float eps, float c1, float c2) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// Place of weight (tap, input channel c, output channel o) in the fragment
// order k_conv reads: steps of 4 groups of 8 channels, chunk by chunk.
__device__ __forceinline__ size_t frag_at(int tap, int c, int o, int cin_pad, int nt) {
  const int CC = conv_chunk(cin_pad), chunk = c / CC, cc = c - chunk * CC;
  const int left = cin_pad - chunk * CC, g8 = (left < CC ? left : CC) / 8;
  const int g = tap * g8 + cc / 8, step = chunk * conv_steps(CC) + g / 4;
  return (((size_t)step * nt + o / 16) * 64 + (g % 4) * 16 + o % 16) * 8 + cc % 8;
}

// BF16 fragments of up to kLayers layers' FP32 weights [cout][27][cin]:
// forward, and backward-data (taps flipped, channels swapped)
constexpr int kLayers = 11;
struct PackArgs {
  const float* w[kLayers];
  u16 *wf[kLayers], *wb[kLayers];
  int cin[kLayers], cout[kLayers];
};
__global__ void k_pack(PackArgs a) {
  const int l = blockIdx.y, cin = a.cin[l], cout = a.cout[l];
  const int nt = (cout + 15) / 16, ntT = (cin + 15) / 16;
  const int cin_pad = (cin + 7) / 8 * 8, cout_pad = (cout + 7) / 8 * 8;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < cout * 27 * cin;
       i += gridDim.x * blockDim.x) {
    const int ci = i % cin, tap = (i / cin) % 27, co = i / (27 * cin);
    const u16 h = f2bf(a.w[l][i]);
    a.wf[l][frag_at(tap, ci, co, cin_pad, nt)] = h;
    a.wb[l][frag_at(26 - tap, co, ci, cout_pad, ntT)] = h;
  }
}

// One wavefront: D = A B with A 16x32, B 32x16 (row-major FP32 in, rounded
// to BF16), through the lane layout k_conv and k_conv_dw use.
__global__ void k_mfma_probe(const float* A, const float* B, float* Dm) {
  const int lane = threadIdx.x, m = lane & 15, kg = lane >> 4;
  u16 a[8], b[8];
  for (int j = 0; j < 8; ++j) {
    a[j] = f2bf(A[m * 32 + kg * 8 + j]);
    b[j] = f2bf(B[(kg * 8 + j) * 16 + m]);
  }
  const bf16x8 av = __builtin_bit_cast(
      bf16x8, make_uint4(a[0] | (uint32_t)a[1] << 16, a[2] | (uint32_t)a[3] << 16,
                         a[4] | (uint32_t)a[5] << 16, a[6] | (uint32_t)a[7] << 16));
  const bf16x8 bv = __builtin_bit_cast(
      bf16x8, make_uint4(b[0] | (uint32_t)b[1] << 16, b[2] | (uint32_t)b[3] << 16,
                         b[4] | (uint32_t)b[5] << 16, b[6] | (uint32_t)b[7] << 16));
  floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, acc, 0, 0, 0);
  for (int q = 0; q < 4; ++q) Dm[(kg * 4 + q) * 16 + m] = acc[q];
}

template <typename T>
int dalloc(T** p, size_t n) {
  *p = nullptr;
  HIP_OK(hipMalloc((void**)p, (n ? n : 1) * sizeof(T)));
  HIP_OK(hipMemset(*p, 0, (n ? n : 1) * sizeof(T)));
  return 0;
}

unsigned blocks_for(long long n, int bs = 256) { return (unsigned)((n + bs - 1) / bs); }

// One 3x3x3 convolution layer: its weights' offset in the parameter buffer
// (the bias follows) and BF16 fragments.
struct Layer {
  int cin = 0, cout = 0, relu = 1;
  int cin_pad = 0, nt = 0;   // forward GEMM
  int cout_pad = 0, ntT = 0; // backward-data GEMM
  size_t off = 0;
  u16 *wf = nullptr, *wb = nullptr;
  size_t nw() const { return (size_t)cout * 27 * cin; }
  int init(int ci, int co, int r, size_t o) {
    cin = ci;
    cout = co;
    relu = r;
    off = o;
    cin_pad = rup(ci, 8);
    nt = rup(co, 16) / 16;
    cout_pad = rup(co, 8);
    ntT = rup(ci, 16) / 16;
    // kConvPre steps more than the layer has: k_conv prefetches past the last
    if (dalloc(&wf, (size_t)(conv_steps_all(cin_pad) + kConvPre) * nt * 512) ||
        dalloc(&wb, (size_t)(conv_steps_all(cout_pad) + kConvPre) * ntT * 512))
      return -1;
    return 0;
  }
  void release() {
    if (wf) (void)hipFree(wf);
    if (wb) (void)hipFree(wb);
    wf = wb = nullptr;
  }
};

int launch_pack(hipStream_t s, const Layer* L, int n, const float* params) {
  PackArgs a;
  memset(&a, 0, sizeof(a));
  size_t most = 1;
  for (int i = 0; i < n; ++i) {
    a.w[i] = params + L[i].off;
    a.wf[i] = L[i].wf;
    a.wb[i] = L[i].wb;
    a.cin[i] = L[i].cin;
    a.cout[i] = L[i].cout;
    most = std::max(most, L[i].nw());
  }
  const unsigned nb = std::min(64u, blocks_for((long long)most));
  hipLaunchKernelGGL(k_pack, dim3(nb, (unsigned)n), dim3(256), 0, s, a);
  HIP_OK(hipGetLastError());
  return 0;
}

ConvIn conv_in(const Chan& c) { return ConvIn{c.p, c.cs, c.co, nullptr, 0, 0, 0}; }
// the concatenation [up-sampled c_up channels of u | c]
ConvIn conv_cat(const Chan& u, int c_up, const Chan& c) {
  return ConvIn{c.p, c.cs, c.co, u.p, u.cs, u.co, c_up};
}

template <int NT>
void conv_kernel(hipStream_t s, const ConvArgs& a, int mv, dim3 g, size_t lds) {
  if (mv == 4)
    hipLaunchKernelGGL((k_conv<NT, 4>), g, dim3(256), lds, s, a);
  else if (mv == 2)
    hipLaunchKernelGGL((k_conv<NT, 2>), g, dim3(256), lds, s, a);
  else
    hipLaunchKernelGGL((k_conv<NT, 1>), g, dim3(256), lds, s, a);
}

// Output tile of 4 mv fragments of 16 voxels along x: of the shapes that give
// so many, the one that stages the fewest voxels over the volume.  Returns
// the workgroups per channel split and the tiles along y in nty.
long long conv_tile(ConvArgs& a, int mv, int* nty) {
  long long best = -1, wgs = 0;
  int lf = 2;
  while ((4 << (lf - 2)) < 4 * mv) ++lf;
  for (int lx = 0; lx <= 2; ++lx)
    for (int lz = 0; lz <= 2 && lx + lz <= lf; ++lz) {
      const int ly = lf - lx - lz;
      const int nx = (a.W + (16 << lx) - 1) >> (4 + lx), ny = (a.H + (1 << ly) - 1) >> ly,
                nz = (a.D + (1 << lz) - 1) >> lz;
      const long long n = (long long)nx * ny * nz;
      const long long cost = n * ((16 << lx) + 2) * ((1 << ly) + 2) * ((1 << lz) + 2);
      if (best >= 0 && cost >= best) continue;
      best = cost;
      wgs = n * a.N;
      a.lfx = lx;
      a.lty = ly;
      a.ltz = lz;
      a.ntx = nx;
      a.ntz = nz;
      *nty = ny;
    }
  return wgs;
}

int launch_conv(hipStream_t s, const ConvIn& in, const u16* w, int cin_pad, int nt,
                const float* bias, const Chan* out, float* out32, int cout, int relu, int N, int D,
                int H, int W, const float* add32 = nullptr, int cs_add = 0) {
  ConvArgs a;
  memset(&a, 0, sizeof(a));
  a.in = in;
  a.w = w;
  a.bias = bias;
  a.out = out ? out->p : nullptr;
  a.cs_out = out ? out->cs : 0;
  a.co_out = out ? out->co : 0;
  a.out32 = out32;
  a.add32 = add32;
  a.cs_add = cs_add;
  a.N = N;
  a.D = D;
  a.H = H;
  a.W = W;
  a.cin_pad = cin_pad;
  a.cout = cout;
  a.nt = nt;
  a.relu = relu;
  const long long V = (long long)N * D * H * W;
  if (V % 16) return fail("voxel count must be a multiple of 16");
  if (in.cs % 8 || in.co % 8 || (out && (out->cs < out->co + cout)))
    return fail("channel strides and offsets must be multiples of 8");
  if (out && (out->cs % 4 || out->co % 4))
    return fail("output channel strides and offsets must be multiples of 4");
  // 4 voxel fragments and up to 4 channel tiles (a divisor of their number)
  // per wavefront: 64 accumulator VGPRs (8 fragments measured slower, 2.54
  // against 2.45 ms for the layers of 16 volumes of 8x256x256); fewer
  // fragments, then fewer channel tiles, until the launch has two workgroups
  // per CU
  int NT = 4, mv = 4, nty = 0;
  while (nt % NT) --NT;
  long long wgs = conv_tile(a, mv, &nty) * (nt / NT);
  while (wgs < 512 && (mv > 1 || NT > 1)) {
    if (mv > 1)
      mv /= 2;
    else
      NT = NT % 2 ? 1 : NT / 2;  // still a divisor
    wgs = conv_tile(a, mv, &nty) * (nt / NT);
  }
  if (V >= (1LL << 31)) return fail("too many voxels");
  const size_t lds = (size_t)((16 << a.lfx) + 2) * ((1 << a.lty) + 2) * ((1 << a.ltz) + 2) *
                     (conv_chunk(cin_pad) / 8) * 16;
  // the y and z axes of a grid hold 65535 blocks: further tiles and volumes
  // are launches of their own (one axis for all of them cost 1.3 % in divisions)
  const int kAxis = 65535, ntnz = a.ntz * N;
  for (a.bz = 0; a.bz < ntnz; a.bz += kAxis)
    for (a.by = 0; a.by < nty; a.by += kAxis) {
      const dim3 g((unsigned)a.ntx * (nt / NT), (unsigned)std::min(kAxis, nty - a.by),
                   (unsigned)std::min(kAxis, ntnz - a.bz));
      switch (NT) {
        case 1: conv_kernel<1>(s, a, mv, g, lds); break;
        case 2: conv_kernel<2>(s, a, mv, g, lds); break;
        case 3: conv_kernel<3>(s, a, mv, g, lds); break;
        default: conv_kernel<4>(s, a, mv, g, lds); break;
      }
    }
  HIP_OK(hipGetLastError());
  return 0;
}

// Tiles of a weight gradient, and its workgroups over them: at most two per
// CU over all pairs of 16 channels, each ending with a 27 KiB partial.
long long dw_tiles(int N, int D, int H, int W) {
  return (long long)N * ((W + kDwX - 1) / kDwX) * ((H + kDwY - 1) / kDwY) *
         ((D + kDwZ - 1) / kDwZ);
}
int dw_groups(long long tiles, int cin, int cout) {
  const long long pairs = (long long)((cin + 15) / 16) * ((cout + 15) / 16);
  const long long want = std::max(1LL, 512 / pairs);
  const long long per = (tiles + want - 1) / want;
  return (int)((tiles + per - 1) / per);
}
size_t dw_partial(long long tiles, int cin, int cout) {
  return (size_t)dw_groups(tiles, cin, cout) * ((size_t)cout * 27 * cin + cout);
}

// dw [cout][27][cin] and the bias gradient behind it; part: dw_partial floats
int launch_dw(hipStream_t s, const Chan& g, const ConvIn& in, float* dw, float* part, int cin,
              int cout, int N, int D, int H, int W) {
  DwArgs a;
  memset(&a, 0, sizeof(a));
  a.g = g.p;
  a.cs_g = g.cs;
  a.co_g = g.co;
  a.cg = rup(cout, 8);
  a.in = in;
  a.part = part;
  a.stride = (size_t)cout * 27 * cin + cout;
  a.N = N;
  a.D = D;
  a.H = H;
  a.W = W;
  a.cin = cin;
  a.cin_pad = rup(cin, 8);
  a.cout = cout;
  a.ntx = (W + kDwX - 1) / kDwX;
  a.nty = (H + kDwY - 1) / kDwY;
  a.ntz = (D + kDwZ - 1) / kDwZ;
  const long long tiles = dw_tiles(N, D, H, W);
  const int ng = dw_groups(tiles, cin, cout);
  a.per = (int)((tiles + ng - 1) / ng);
  hipLaunchKernelGGL(k_conv_dw, dim3((unsigned)ng, (cin + 15) / 16, (cout + 15) / 16), dim3(256),
                     0, s, a);
  hipLaunchKernelGGL(k_dw_sum, dim3(blocks_for((long long)a.stride)), dim3(256), 0, s, part, ng,
                     a.stride, dw);
  HIP_OK(hipGetLastError());
  return 0;
}

}  // namespace

// ------------------------------------------------------------------ network
struct unet_ctx {
  phasecon::CopyOut copy_out;
  hipStream_t s = nullptr;
  int c = 16, cin = 1;  // base channels, input channels
  Layer L[kLayers];
  size_t np = 0;  // parameters, all layers
  float* dwpart = nullptr;  // the largest layer's weight-gradient partials
  float *par = nullptr, *grad = nullptr, *mom1 = nullptr, *mom2 = nullptr;
  // shape the activation buffers hold
  int N = 0, D = 0, H = 0, W = 0;
  long long V1 = 0, V2 = 0, V3 = 0;
  u16 *X0 = nullptr, *A1 = nullptr, *S1 = nullptr, *P1 = nullptr, *A2 = nullptr, *S2 = nullptr,
      *P2 = nullptr, *A3 = nullptr, *B3 = nullptr, *A4 = nullptr, *B4 = nullptr, *A5 = nullptr,
      *B5 = nullptr;
  u16 *GO = nullptr, *GB5 = nullptr, *GA5 = nullptr, *GC1 = nullptr, *GB4 = nullptr,
      *GA4 = nullptr, *GC2 = nullptr, *GB3 = nullptr, *GA3 = nullptr, *GP2 = nullptr,
      *GA2 = nullptr, *GP1 = nullptr, *GA1 = nullptr;
  float *x32 = nullptr, *t32 = nullptr, *o32 = nullptr;
  double* partial = nullptr;
  int step = 0;
  std::vector<void*> acts;
  void free_acts() {
    for (void* p : acts)
      if (p) (void)hipFree(p);
    acts.clear();
  }
};

namespace {

constexpr int kLossBlocks = 256;

template <typename T>
int alloc_act(unet_ctx* c, T** p, long long n) {
  const int rc = dalloc(p, (size_t)n);
  if (*p) c->acts.push_back(*p);
  return rc;
}

int alloc_shape(unet_ctx* c, int N, int D, int H, int W) {
  const long long V1 = (long long)N * D * H * W, V2 = V1 / 8, V3 = V1 / 64;
  const int c1 = c->c, c2 = 2 * c->c, c3 = 4 * c->c;
  u16** bufs1[] = {&c->A1, &c->A5, &c->B5, &c->GB5, &c->GA5, &c->GA1};
  for (u16** b : bufs1)
    if (alloc_act(c, b, V1 * c1)) return -1;
  if (alloc_act(c, &c->X0, V1 * 8) || alloc_act(c, &c->GO, V1 * 8) ||
      alloc_act(c, &c->S1, V1 * c1) || alloc_act(c, &c->GC1, V1 * (c2 + c1)))
    return -1;
  u16** bufs2[] = {&c->A2, &c->A4, &c->B4, &c->GB4, &c->GA4, &c->GA2};
  for (u16** b : bufs2)
    if (alloc_act(c, b, V2 * c2)) return -1;
  if (alloc_act(c, &c->P1, V2 * c1) || alloc_act(c, &c->GP1, V2 * c1) ||
      alloc_act(c, &c->S2, V2 * c2) || alloc_act(c, &c->GC2, V2 * (c3 + c2)))
    return -1;
  u16** bufs3[] = {&c->A3, &c->B3, &c->GB3, &c->GA3};
  for (u16** b : bufs3)
    if (alloc_act(c, b, V3 * c3)) return -1;
  if (alloc_act(c, &c->P2, V3 * c2) || alloc_act(c, &c->GP2, V3 * c2)) return -1;
  size_t part = 1;
  for (int i = 0; i < kLayers; ++i) {
    const int sh = i < 2 || i > 7 ? 0 : (i == 4 || i == 5 ? 2 : 1);  // the layer's level
    part = std::max(part, dw_partial(dw_tiles(N, D >> sh, H >> sh, W >> sh), c->L[i].cin,
                                     c->L[i].cout));
  }
  if (alloc_act(c, &c->dwpart, (long long)part)) return -1;
  float** f32s[] = {&c->x32, &c->t32, &c->o32};
  for (float** b : f32s)
    if (alloc_act(c, b, V1 * (b == &c->x32 ? c->cin : 1))) return -1;
  return 0;
}

// The activation buffers of a shape.  The context holds the shape only once
// all of them are there: a call after a failed one allocates again.
int set_shape(unet_ctx* c, int N, int D, int H, int W) {
  if (N == c->N && D == c->D && H == c->H && W == c->W) return 0;
  if (N < 1 || D < 4 || H < 4 || W < 64 || D % 4 || H % 4 || W % 64)
    return fail("volume must have D, H divisible by 4 and W divisible by 64");
  HIP_OK(hipStreamSynchronize(c->s));
  c->free_acts();
  c->N = 0;
  if (alloc_shape(c, N, D, H, W)) {
    c->free_acts();
    return -1;
  }
  c->N = N;
  c->D = D;
  c->H = H;
  c->W = W;
  c->V1 = (long long)N * D * H * W;
  c->V2 = c->V1 / 8;
  c->V3 = c->V1 / 64;
  return 0;
}

int conv_layer(unet_ctx* c, int li, const ConvIn& in, const Chan* out, float* out32, int lev,
               const float* add32 = nullptr, int cs_add = 0) {
  const Layer& l = c->L[li];
  const int sh = lev;  // spatial halving per level
  return launch_conv(c->s, in, l.wf, l.cin_pad, l.nt, c->par + l.off + l.nw(), out, out32, l.cout,
                     l.relu, c->N, c->D >> sh, c->H >> sh, c->W >> sh, add32, cs_add);
}

// o32 := net(x), plus x_0 when residual
int forward(unet_ctx* c, bool residual) {
  const int c1 = c->c, c2 = 2 * c->c, c3 = 4 * c->c;
  const int N = c->N, D = c->D, H = c->H, W = c->W;
  const Chan X0{c->X0, 8, 0}, A1{c->A1, c1, 0}, S1{c->S1, c1, 0}, P1{c->P1, c1, 0},
      A2{c->A2, c2, 0}, S2{c->S2, c2, 0}, P2{c->P2, c2, 0}, A3{c->A3, c3, 0},
      B3{c->B3, c3, 0}, A4{c->A4, c2, 0}, B4{c->B4, c2, 0}, A5{c->A5, c1, 0}, B5{c->B5, c1, 0};
  hipLaunchKernelGGL(k_in_pack, dim3(blocks_for(c->V1)), dim3(256), 0, c->s, c->x32, c->cin,
                     c->V1, c->X0);
  if (conv_layer(c, 0, conv_in(X0), &A1, nullptr, 0) ||
      conv_layer(c, 1, conv_in(A1), &S1, nullptr, 0))
    return -1;
  hipLaunchKernelGGL(k_pool, dim3(blocks_for(c->V2 * c1 / 8)), dim3(256), 0, c->s, S1.p, S1.cs,
                     S1.co, P1.p, P1.cs, P1.co, c1, N, D, H, W);
  if (conv_layer(c, 2, conv_in(P1), &A2, nullptr, 1) ||
      conv_layer(c, 3, conv_in(A2), &S2, nullptr, 1))
    return -1;
  hipLaunchKernelGGL(k_pool, dim3(blocks_for(c->V3 * c2 / 8)), dim3(256), 0, c->s, S2.p, S2.cs,
                     S2.co, P2.p, P2.cs, P2.co, c2, N, D / 2, H / 2, W / 2);
  if (conv_layer(c, 4, conv_in(P2), &A3, nullptr, 2) ||
      conv_layer(c, 5, conv_in(A3), &B3, nullptr, 2) ||
      conv_layer(c, 6, conv_cat(B3, c3, S2), &A4, nullptr, 1) ||
      conv_layer(c, 7, conv_in(A4), &B4, nullptr, 1) ||
      conv_layer(c, 8, conv_cat(B4, c2, S1), &A5, nullptr, 0) ||
      conv_layer(c, 9, conv_in(A5), &B5, nullptr, 0) ||
      conv_layer(c, 10, conv_in(B5), nullptr, c->o32, 0, residual ? c->x32 : nullptr, c->cin))
    return -1;
  HIP_OK(hipGetLastError());
  return 0;
}

// gradients of one layer: relu mask on g (when the layer has one), dW, db,
// and (when gin) the input gradient
int layer_bwd(unet_ctx* c, int li, const Chan& g, const Chan& act_out, const ConvIn& in,
              const Chan* gin, int lev) {
  const Layer& l = c->L[li];
  const int N = c->N, D = c->D >> lev, H = c->H >> lev, W = c->W >> lev;
  const long long V = (long long)N * D * H * W;
  if (l.relu)
    hipLaunchKernelGGL(k_relu_bwd, dim3(blocks_for(V * l.cout / 8)), dim3(256), 0, c->s, g.p, g.cs,
                       g.co, act_out.p, act_out.cs, act_out.co, l.cout, V);
  float* gw = c->grad + l.off;
  if (launch_dw(c->s, g, in, gw, c->dwpart, l.cin, l.cout, N, D, H, W)) return -1;
  if (gin && launch_conv(c->s, conv_in(g), l.wb, l.cout_pad, l.ntT, nullptr, gin, nullptr, l.cin,
                         0, N, D, H, W))
    return -1;
  HIP_OK(hipGetLastError());
  return 0;
}

int backward(unet_ctx* c, double* loss) {
  const int c1 = c->c, c2 = 2 * c->c, c3 = 4 * c->c;
  const int N = c->N, D = c->D, H = c->H, W = c->W;
  const Chan X0{c->X0, 8, 0}, A1{c->A1, c1, 0}, S1{c->S1, c1, 0}, P1{c->P1, c1, 0},
      A2{c->A2, c2, 0}, S2{c->S2, c2, 0}, P2{c->P2, c2, 0}, A3{c->A3, c3, 0},
      B3{c->B3, c3, 0}, A4{c->A4, c2, 0}, B4{c->B4, c2, 0}, A5{c->A5, c1, 0}, B5{c->B5, c1, 0};
  const Chan GO{c->GO, 8, 0}, GB5{c->GB5, c1, 0}, GA5{c->GA5, c1, 0}, GC1{c->GC1, c2 + c1, 0},
      GU1{c->GC1, c2 + c1, 0}, GS1{c->GC1, c2 + c1, c2}, GB4{c->GB4, c2, 0}, GA4{c->GA4, c2, 0},
      GC2{c->GC2, c3 + c2, 0}, GU2{c->GC2, c3 + c2, 0}, GS2{c->GC2, c3 + c2, c3},
      GB3{c->GB3, c3, 0}, GA3{c->GA3, c3, 0}, GP2{c->GP2, c2, 0}, GA2{c->GA2, c2, 0},
      GP1{c->GP1, c1, 0}, GA1{c->GA1, c1, 0};
  hipLaunchKernelGGL(k_mse, dim3(kLossBlocks), dim3(256), 0, c->s, c->o32, c->x32, c->cin,
                     c->t32, c->V1, c->GO, c->partial);
  if (layer_bwd(c, 10, GO, GO, conv_in(B5), &GB5, 0) ||
      layer_bwd(c, 9, GB5, B5, conv_in(A5), &GA5, 0) ||
      layer_bwd(c, 8, GA5, A5, conv_cat(B4, c2, S1), &GC1, 0))
    return -1;
  hipLaunchKernelGGL(k_up_bwd, dim3(blocks_for(c->V2 * c2 / 8)), dim3(256), 0, c->s, GU1.p, GU1.cs,
                     GU1.co, GB4.p, GB4.cs, GB4.co, c2, N, D / 2, H / 2, W / 2);
  if (layer_bwd(c, 7, GB4, B4, conv_in(A4), &GA4, 1) ||
      layer_bwd(c, 6, GA4, A4, conv_cat(B3, c3, S2), &GC2, 1))
    return -1;
  hipLaunchKernelGGL(k_up_bwd, dim3(blocks_for(c->V3 * c3 / 8)), dim3(256), 0, c->s, GU2.p, GU2.cs,
                     GU2.co, GB3.p, GB3.cs, GB3.co, c3, N, D / 4, H / 4, W / 4);
  if (layer_bwd(c, 5, GB3, B3, conv_in(A3), &GA3, 2) ||
      layer_bwd(c, 4, GA3, A3, conv_in(P2), &GP2, 2))
    return -1;
  hipLaunchKernelGGL(k_pool_bwd, dim3(blocks_for(c->V2 * c2 / 8)), dim3(256), 0, c->s, GP2.p,
                     GP2.cs, GP2.co, GS2.p, GS2.cs, GS2.co, c2, N, D / 2, H / 2, W / 2);
  if (layer_bwd(c, 3, GS2, S2, conv_in(A2), &GA2, 1) ||
      layer_bwd(c, 2, GA2, A2, conv_in(P1), &GP1, 1))
    return -1;
  hipLaunchKernelGGL(k_pool_bwd, dim3(blocks_for(c->V1 * c1 / 8)), dim3(256), 0, c->s, GP1.p,
                     GP1.cs, GP1.co, GS1.p, GS1.cs, GS1.co, c1, N, D, H, W);
  if (layer_bwd(c, 1, GS1, S1, conv_in(A1), &GA1, 0) ||
      layer_bwd(c, 0, GA1, A1, conv_in(X0), nullptr, 0))
    return -1;
  if (loss) {
    std::vector<double> part(kLossBlocks);
    HIP_OK(hipMemcpyAsync(part.data(), c->partial, kLossBlocks * sizeof(double),
                          hipMemcpyDeviceToHost, c->s));
    HIP_OK(hipStreamSynchronize(c->s));
    double s = 0.0;
    for (double v : part) s += v;
    *loss = s / (double)c->V1;
  }
  HIP_OK(hipGetLastError());
  return 0;
}

int upload_pair(unet_ctx* c, const float* x, const float* t) {
  HIP_OK(hipMemcpyAsync(c->x32, x, c->V1 * c->cin * sizeof(float), hipMemcpyHostToDevice, c->s));
  if (t) HIP_OK(hipMemcpyAsync(c->t32, t, c->V1 * sizeof(float), hipMemcpyHostToDevice, c->s));
  return 0;
}

}  // namespace

extern "C" {

const char* unet_last_error(void) { return g_err.c_str(); }

int unet_create(unet_ctx** out, int32_t channels, int32_t in_channels, uint32_t seed) {
  if (!out) return fail("null argument");
  *out = nullptr;
  if (channels < 8 || channels > 32 || channels % 8) return fail("channels must be 8, 16, 24 or 32");
  if (in_channels < 1 || in_channels > 8) return fail("in_channels must be in [1, 8]");
  unet_ctx* c = new unet_ctx();
  c->c = channels;
  c->cin = in_channels;
  const int c1 = channels, c2 = 2 * channels, c3 = 4 * channels;
  const int io[11][3] = {{in_channels, c1, 1},  {c1, c1, 1},      {c1, c2, 1}, {c2, c2, 1},
                         {c2, c3, 1}, {c3, c3, 1},      {c3 + c2, c2, 1}, {c2, c2, 1},
                         {c2 + c1, c1, 1}, {c1, c1, 1}, {c1, 1, 0}};
  if (hipStreamCreate(&c->s) != hipSuccess) {
    delete c;
    return fail("hipStreamCreate failed");
  }
  std::mt19937 rng(seed);
  for (int i = 0; i < kLayers; ++i) {
    if (c->L[i].init(io[i][0], io[i][1], io[i][2], c->np)) {
      unet_destroy(c);
      return -1;
    }
    c->np += c->L[i].nw() + c->L[i].cout;
  }
  if (dalloc(&c->par, c->np) || dalloc(&c->grad, c->np) || dalloc(&c->mom1, c->np) ||
      dalloc(&c->mom2, c->np)) {
    unet_destroy(c);
    return -1;
  }
  std::vector<float> par(c->np, 0.f);
  for (int i = 0; i < kLayers; ++i) {
    // He-normal initialisation (the output layer scaled down: the network
    // starts near the identity of its residual form)
    const float sd = std::sqrt(2.f / (27.f * io[i][0])) * (i == 10 ? 0.1f : 1.f);
    std::normal_distribution<float> nd(0.f, sd);
    for (size_t k = 0; k < c->L[i].nw(); ++k) par[c->L[i].off + k] = nd(rng);
  }
  if (hipMemcpy(c->par, par.data(), c->np * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
      launch_pack(c->s, c->L, kLayers, c->par)) {
    unet_destroy(c);
    return fail("weight upload failed");
  }
  if (dalloc(&c->partial, kLossBlocks)) {
    unet_destroy(c);
    return -1;
  }
  *out = c;
  return 0;
}

void unet_destroy(unet_ctx* c) {
  if (!c) return;
  if (c->s) (void)hipStreamSynchronize(c->s);
  c->free_acts();
  for (auto& l : c->L) l.release();
  float* ps[] = {c->par, c->grad, c->mom1, c->mom2};
  for (float* p : ps)
    if (p) (void)hipFree(p);
  if (c->partial) (void)hipFree(c->partial);
  if (c->s) (void)hipStreamDestroy(c->s);
  delete c;
}

int64_t unet_param_count(const unet_ctx* c) { return c ? (int64_t)c->np : -1; }

int unet_get_params(unet_ctx* c, float* buf) {
  if (!c || !buf) return fail("null argument");
  HIP_OK(hipMemcpy(buf, c->par, c->np * sizeof(float), hipMemcpyDeviceToHost));
  return 0;
}

int unet_set_params(unet_ctx* c, const float* buf) {
  if (!c || !buf) return fail("null argument");
  HIP_OK(hipStreamSynchronize(c->s));
  HIP_OK(hipMemcpy(c->par, buf, c->np * sizeof(float), hipMemcpyHostToDevice));
  if (launch_pack(c->s, c->L, kLayers, c->par)) return -1;
  HIP_OK(hipStreamSynchronize(c->s));
  return 0;
}

int unet_forward(unet_ctx* c, int32_t N, int32_t D, int32_t H, int32_t W, const float* x,
                 float* y) {
  if (!c || !x || !y) return fail("null argument");
  if (set_shape(c, N, D, H, W) || upload_pair(c, x, nullptr) || forward(c, true)) return -1;
  HIP_OK(c->copy_out(y, c->o32, c->V1 * sizeof(float), c->s));
  HIP_OK(hipStreamSynchronize(c->s));
  return 0;
}

int unet_gradients(unet_ctx* c, int32_t N, int32_t D, int32_t H, int32_t W, const float* x,
                   const float* t, float* grads, double* loss) {
  if (!c || !x || !t || !grads) return fail("null argument");
  if (set_shape(c, N, D, H, W) || upload_pair(c, x, t) || forward(c, false) || backward(c, loss))
    return -1;
  HIP_OK(hipMemcpy(grads, c->grad, c->np * sizeof(float), hipMemcpyDeviceToHost));
  return 0;
}

int unet_train_step(unet_ctx* c, int32_t N, int32_t D, int32_t H, int32_t W, const float* x,
                    const float* t, float lr, double* loss) {
  if (!c || !x || !t) return fail("null argument");
  if (set_shape(c, N, D, H, W) || upload_pair(c, x, t) || forward(c, false) || backward(c, loss))
    return -1;
  ++c->step;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float c1 = 1.f - std::pow(b1, (float)c->step), c2 = 1.f - std::pow(b2, (float)c->step);
  hipLaunchKernelGGL(k_adam, dim3(blocks_for((long long)c->np)), dim3(256), 0, c->s, c->par,
                     c->grad, c->mom1, c->mom2, (long long)c->np, lr, b1, b2, eps, c1, c2);
  if (launch_pack(c->s, c->L, kLayers, c->par)) return -1;
  HIP_OK(hipGetLastError());
  HIP_OK(hipStreamSynchronize(c->s));
  return 0;
}

// ---- single-layer entry points (parity tests of the kernels)
int unet_conv3d(int32_t mode, int32_t N, int32_t D, int32_t H, int32_t W, int32_t cin,
                int32_t cout, const float* in, const float* w, const float* bias, int32_t relu,
                const float* gout, float* out) {
  // mode 0: out [v][cout] = conv(in [v][cin]) (+ bias, ReLU);
  // mode 1: out [v][cin] = input gradient of conv for gout [v][cout];
  // mode 2: out [cout][27][cin] = weight gradient for gout and in.
  // in, gout and w are rounded to BF16 as the network stores them.
  if (mode < 0 || mode > 2 || !out || !w) return fail("bad argument");
  if (cin < 1 || cout < 1 || cin > 128 || cout > 128) return fail("bad channel count");
  const long long V = (long long)N * D * H * W;
  if (V <= 0 || V % 16) return fail("voxel count must be a positive multiple of 16");
  Layer l;
  float* par = nullptr;  // weights, then the bias
  if (l.init(cin, cout, relu, 0) || dalloc(&par, l.nw() + cout)) {
    l.release();
    return -1;
  }
  float* parb = par + l.nw();
  hipStream_t s = nullptr;
  HIP_OK(hipStreamCreate(&s));
  int rc = 0;
  u16 *din = nullptr, *dg = nullptr;
  float *o32 = nullptr, *dpart = nullptr;
  auto pack_act = [&](const float* src, int C, int cs, u16** dst) -> int {
    std::vector<u16> h((size_t)V * cs, 0);
    for (long long v = 0; v < V; ++v)
      for (int ch = 0; ch < C; ++ch) h[(size_t)v * cs + ch] = f2bf(src[(size_t)v * C + ch]);
    if (dalloc(dst, h.size())) return -1;
    HIP_OK(hipMemcpy(*dst, h.data(), h.size() * sizeof(u16), hipMemcpyHostToDevice));
    return 0;
  };
  do {
    if ((rc = (int)(hipMemcpy(par, w, l.nw() * sizeof(float), hipMemcpyHostToDevice) != hipSuccess))) {
      rc = fail("upload failed");
      break;
    }
    if (bias && hipMemcpy(parb, bias, cout * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) {
      rc = fail("upload failed");
      break;
    }
    if ((rc = launch_pack(s, &l, 1, par))) break;
    if (mode == 0) {
      if (!in) { rc = fail("null input"); break; }
      if ((rc = pack_act(in, cin, l.cin_pad, &din)) || (rc = dalloc(&o32, (size_t)V * cout))) break;
      if ((rc = launch_conv(s, conv_in(Chan{din, l.cin_pad, 0}), l.wf, l.cin_pad, l.nt,
                            bias ? parb : nullptr, nullptr, o32, cout, relu, N, D, H, W)))
        break;
      HIP_OK(hipStreamSynchronize(s));
      HIP_OK(hipMemcpy(out, o32, (size_t)V * cout * sizeof(float), hipMemcpyDeviceToHost));
    } else if (mode == 1) {
      if (!gout) { rc = fail("null gradient"); break; }
      if ((rc = pack_act(gout, cout, l.cout_pad, &dg)) || (rc = dalloc(&o32, (size_t)V * cin)))
        break;
      if ((rc = launch_conv(s, conv_in(Chan{dg, l.cout_pad, 0}), l.wb, l.cout_pad, l.ntT, nullptr,
                            nullptr, o32, cin, 0, N, D, H, W)))
        break;
      HIP_OK(hipStreamSynchronize(s));
      HIP_OK(hipMemcpy(out, o32, (size_t)V * cin * sizeof(float), hipMemcpyDeviceToHost));
    } else {
      if (!gout || !in) { rc = fail("null input"); break; }
      if ((rc = pack_act(in, cin, l.cin_pad, &din)) || (rc = pack_act(gout, cout, l.cout_pad, &dg)))
        break;
      if ((rc = dalloc(&o32, l.nw() + cout)) ||
          (rc = dalloc(&dpart, dw_partial(dw_tiles(N, D, H, W), cin, cout))) ||
          (rc = launch_dw(s, Chan{dg, l.cout_pad, 0}, conv_in(Chan{din, l.cin_pad, 0}), o32,
                          dpart, cin, cout, N, D, H, W)))
        break;
      HIP_OK(hipStreamSynchronize(s));
      HIP_OK(hipMemcpy(out, o32, l.nw() * sizeof(float), hipMemcpyDeviceToHost));
    }
  } while (0);
  (void)hipStreamSynchronize(s);
  void* ps[] = {din, dg, o32, dpart, par};
  for (void* p : ps)
    if (p) (void)hipFree(p);
  l.release();
  (void)hipStreamDestroy(s);
  return rc;
}

int unet_mfma_probe(const float* A, const float* B, float* Dm) {
  if (!A || !B || !Dm) return fail("null argument");
  float *dA, *dB, *dD;
  if (dalloc(&dA, 16 * 32) || dalloc(&dB, 32 * 16) || dalloc(&dD, 16 * 16)) return -1;
  HIP_OK(hipMemcpy(dA, A, 16 * 32 * sizeof(float), hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(dB, B, 32 * 16 * sizeof(float), hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_mfma_probe, dim3(1), dim3(64), 0, 0, dA, dB, dD);
  HIP_OK(hipGetLastError());
  HIP_OK(hipMemcpy(Dm, dD, 16 * 16 * sizeof(float), hipMemcpyDeviceToHost));
  (void)hipFree(dA);
  (void)hipFree(dB);
  (void)hipFree(dD);
  return 0;
}

}  // extern "C"
