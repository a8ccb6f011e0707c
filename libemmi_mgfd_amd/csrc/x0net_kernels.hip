// x0net_kernels.hip -- kernels of the initial-guess network (3D U-Net).
//
// Tensors are channel-last [Z][Y][X][C] with C a multiple of 16; network
// activations and gradients are BF16 (raw 16-bit storage), accumulation is
// FP32.  The 3x3x3 convolutions are implicit GEMMs on the gfx950 matrix cores
// (v_mfma_f32_16x16x32_bf16):
//   forward       y[v][co] = sum_{tap,ci} x[v+tap-1][ci] w[co][tap*Cin+ci]
//                 M = voxels, N = Cout, K = 27*Cin (padded to 32)
//   grad of input dx = the forward kernel applied to dy with the flipped,
//                 transposed weights w'[ci][tap'*Cout+co] = w[co][(26-tap')*Cin+ci]
//   grad of weight dw[co][tap*Cin+ci] = sum_v dy[v][co] x[v+tap-1][ci]
//                 M = Cout, N = Cin per tap, K = voxels, partial sums per
//                 slab of z-slices, then a fixed-order reduction
// Operand layout of the 16x16x32 instruction (one wave): lane l holds
// A[l%16][8(l/16)+j] and B[8(l/16)+j][l%16] (j < 8) and receives
// D[4(l/16)+i][l%16] (i < 4).
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <cstdint>
#include <algorithm>
#include <cmath>

#include "dynamic_lds.h"
#include "emmi_mgfd.h"
#include "timing.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t bf16;

__device__ __forceinline__ float bf2f(bf16 v) { return __uint_as_float(((uint32_t)v) << 16); }
__device__ __forceinline__ bf16 f2bf(float f) {
  // round to nearest even
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (bf16)(u >> 16);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16)(u >> 16);
}

__device__ __forceinline__ bf16x8 load8(const bf16* p) {
  const uint4 v = *reinterpret_cast<const uint4*>(p);
  return __builtin_bit_cast(bf16x8, v);
}
__device__ __forceinline__ bf16x8 zero8() { return __builtin_bit_cast(bf16x8, make_uint4(0, 0, 0, 0)); }

enum Epilogue { EPI_LEAKY = 0, EPI_LINEAR = 1, EPI_DACT = 2, EPI_LINEAR_BF16 = 3 };

// a wave's 16 MT voxels from x0 of row (z, y): with the weights as the first
// operand a lane holds voxel x0 + 16 m + l % 16, channels 16 n + 4 (l / 16) + i,
// so that it stores four channels at once and the wave's stores are contiguous
template <int MT, int NT>
__device__ __forceinline__ void conv_epilogue(const f32x4 (&acc)[MT][NT], int x0, int y, int z, int Y, int X,
                                              const float* __restrict__ bias, int epi, float slope,
                                              const bf16* __restrict__ act, bf16* __restrict__ out_bf,
                                              float* __restrict__ out_f, int Cout_store) {
  constexpr int Cout = 16 * NT;
  const int lane = threadIdx.x & 63, c4 = 4 * (lane >> 4);
  // four channels at once where the tensors' bases allow it (uniform)
  const bool vec = ((reinterpret_cast<uintptr_t>(out_bf) | reinterpret_cast<uintptr_t>(act)) & 7) == 0;
  auto pack = [](const f32x4& r) {
    return make_uint2((unsigned)f2bf(r[0]) | ((unsigned)f2bf(r[1]) << 16), (unsigned)f2bf(r[2]) | ((unsigned)f2bf(r[3]) << 16));
  };
#pragma unroll
  for (int m = 0; m < MT; m++) {
    const int xx = x0 + 16 * m + (lane & 15);
    if (xx >= X) continue;
    const long v = ((long)z * Y + y) * X + xx;
#pragma unroll
    for (int n = 0; n < NT; n++) {
      f32x4 r = acc[m][n];
      const int co = 16 * n + c4;
      if (epi == EPI_LEAKY || (epi == EPI_LINEAR && bias)) {
#pragma unroll
        for (int i = 0; i < 4; i++) r[i] += bias[co + i];
      }
      if (epi == EPI_LEAKY) {
#pragma unroll
        for (int i = 0; i < 4; i++) r[i] = r[i] > 0.f ? r[i] : slope * r[i];
      } else if (epi == EPI_DACT) {
        // gradient through the activation of the tensor this one feeds
        bf16 a4[4];
        if (vec) {
          const uint2 av = *reinterpret_cast<const uint2*>(act + v * Cout + co);
          a4[0] = (bf16)av.x; a4[1] = (bf16)(av.x >> 16); a4[2] = (bf16)av.y; a4[3] = (bf16)(av.y >> 16);
        } else {
#pragma unroll
          for (int i = 0; i < 4; i++) a4[i] = act[v * Cout + co + i];
        }
#pragma unroll
        for (int i = 0; i < 4; i++) r[i] = bf2f(a4[i]) > 0.f ? r[i] : slope * r[i];
      }
      if (epi == EPI_LINEAR) {
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (co + i < Cout_store) out_f[v * Cout_store + co + i] = r[i];
      } else if (vec) {
        *reinterpret_cast<uint2*>(out_bf + v * Cout + co) = pack(r);
      } else {
#pragma unroll
        for (int i = 0; i < 4; i++) out_bf[v * Cout + co + i] = f2bf(r[i]);
      }
    }
  }
}

// One wave: 16*MT consecutive voxels along x of row (z, y) and all 16*NT
// output channels.  Block: 4 waves on rows y0..y0+3.
// (Four waves per SIMD for one tile into 48 to 80 channels: at three, 33^3 needs
// a second, nearly empty round of blocks, 48 -> 48 channels 46 -> 54 us.)
template <int MT, int NT>
__global__ void __launch_bounds__(256, MT == 1 && NT >= 3 && NT <= 5 ? 4 : 1) k_conv_fwd(const bf16* __restrict__ x, int Z, int Y, int X, int Cin,
                                                  const bf16* __restrict__ w, int Kpad,
                                                  const float* __restrict__ bias, int epi, float slope,
                                                  const bf16* __restrict__ act, bf16* __restrict__ out_bf,
                                                  float* __restrict__ out_f, int Cout_store) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int x0 = blockIdx.x * 16 * MT;
  const int y = blockIdx.y * 4 + wave;
  const int z = blockIdx.z;
  if (y >= Y) return;
  f32x4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; m++)
#pragma unroll
    for (int n = 0; n < NT; n++) acc[m][n] = f32x4{0, 0, 0, 0};
  const int K27 = 27 * Cin;
  const int row = lane & 15, kq = (lane >> 4) * 8;
  // the next G steps' operands are in flight while a step is multiplied
  constexpr int G = MT + NT <= 4 ? 6 : MT + NT <= 6 && NT != 5 ? 4 : 3;
  bf16x8 a[G][MT], b[G][NT];
  auto fetch = [&](int q, int k0) {
    if (k0 >= Kpad) return;   // uniform
    const int k = k0 + kq;
    const int tap = k / Cin, ci = k - tap * Cin;
    const int dz = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dx = tap % 3 - 1;
    const int zz = z + dz, yy = y + dy;
    const bool zy_ok = k < K27 && zz >= 0 && zz < Z && yy >= 0 && yy < Y;
#pragma unroll
    for (int m = 0; m < MT; m++) {
      const int xx = x0 + 16 * m + row + dx;
      if (zy_ok && xx >= 0 && xx < X)
        a[q][m] = load8(x + (((long)zz * Y + yy) * X + xx) * Cin + ci);
      else
        a[q][m] = zero8();
    }
#pragma unroll
    for (int n = 0; n < NT; n++) b[q][n] = load8(w + (long)(16 * n + row) * Kpad + k);
  };
#pragma unroll
  for (int q = 0; q < G; q++) fetch(q, 32 * q);
  for (int k0 = 0; k0 < Kpad; k0 += 32 * G) {
#pragma unroll
    for (int q = 0; q < G; q++) {
      if (k0 + 32 * q < Kpad) {   // uniform
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
          for (int m = 0; m < MT; m++) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[q][n], a[q][m], acc[m][n], 0, 0, 0);
      }
      fetch(q, k0 + 32 * (G + q));
    }
  }
  conv_epilogue<MT, NT>(acc, x0, y, z, Y, X, bias, epi, slope, act, out_bf, out_f, Cout_store);
}

// The same sums from LDS: a block takes a tile of 32 x TY voxels, a wave per
// row of 32, and marches along z with three planes of the input (the tile and
// a voxel around it, zero outside the grid) in LDS, so every input voxel is
// loaded (TY + 2) 34 / (32 TY) times instead of 27, and with contiguous loads.
// The plane after next is loaded while a plane is computed.  Voxels stand
// 2 Cin + 16 bytes apart, so that the 16 voxels of an operand start in
// different banks.  A table holds, for each phase of the ring and each group of
// 8 k, the place of its tap and channels relative to the output voxel.  The
// instructions and their order are those of k_conv_fwd: the results are equal
// bit for bit.
//
// What bounds it: k_conv_fwd gathered every operand from 16 rows in L1 or L2
// (one 16-byte load a lane for each NT matrix instructions); here an operand is
// one LDS read.  At 96^3: 48 -> 16 channels 222 -> 118 us, 16 -> 48
// 183 -> 97 us (310 to 380 TFLOP/s); the weights come from LDS where they fit
// beside the planes -- read from memory, 16 rows apart, they were the bound
// (170 and 241 us).
template <int NT, int TY, int NP, bool WL>
__global__ void __launch_bounds__(64 * TY) k_conv_fwd_lds(const bf16* __restrict__ x, int Z, int Y, int X, int Cin,
                                                          const bf16* __restrict__ w, int Kpad,
                                                          const float* __restrict__ bias, int epi, float slope,
                                                          const bf16* __restrict__ act, bf16* __restrict__ out_bf,
                                                          float* __restrict__ out_f, int Cout_store, int zper) {
  constexpr int TX = 32, VX = TX + 2, NV = (TY + 2) * VX, BT = 64 * TY, MT = 2, G = WL ? 2 : NT <= 2 ? 8 : NT <= 4 ? 4 : 2;
  extern __shared__ __align__(16) char smem[];
  const int vs = 2 * Cin + 16, pb = NV * vs, pc = Cin / 8, np = NV * pc, ng = Kpad / 8;
  char* planes = smem;                                    // [3][NV][vs]
  int* tab = reinterpret_cast<int*>(smem + 3 * pb);       // [3][ng]
  const int ws = 2 * Kpad + 16;                           // bytes of a weight row (rows in different banks)
  char* wlds = smem + 3 * pb + (3 * ng * 4 + 15) / 16 * 16;   // WL: [16 NT][ws]
  if constexpr (WL) {
    for (int i = threadIdx.x; i < 16 * NT * ng; i += BT) {
      const int co = i / ng, k8 = i - co * ng;
      *reinterpret_cast<uint4*>(wlds + co * ws + 16 * k8) = *reinterpret_cast<const uint4*>(w + (long)co * Kpad + 8 * k8);
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int x0 = blockIdx.x * TX, y0 = blockIdx.y * TY, zs = blockIdx.z * zper, ze = min(Z, zs + zper);
  for (int i = threadIdx.x; i < 3 * ng; i += BT) {
    const int ph = i / ng, k = (i - ph * ng) * 8;
    int off = 0;
    if (k < 27 * Cin) {
      const int tap = k / Cin, ci = k - tap * Cin;
      const int dz = tap / 9, dy = (tap / 3) % 3, dx = tap % 3;
      off = ((ph + dz) % 3) * pb + (dy * VX + dx) * vs + 2 * ci;
    }
    tab[i] = off;   // (padding of K: masked)
  }
  // this thread's 16-byte pieces of a plane
  int go[NP], lo[NP];
#pragma unroll
  for (int i = 0; i < NP; i++) {
    const int idx = i * BT + (int)threadIdx.x, vox = idx / pc, piece = idx - vox * pc;
    const int gx = x0 + vox % VX - 1, gy = y0 + vox / VX - 1;
    lo[i] = idx < np ? vox * vs + 16 * piece : -1;
    go[i] = idx < np && gx >= 0 && gx < X && gy >= 0 && gy < Y ? (gy * X + gx) * Cin + 8 * piece : -1;
  }
  uint4 pre[NP];
  auto load = [&](int z) {
    const bool in = z >= 0 && z < Z;   // uniform
    const bf16* p = x + (long)z * Y * X * Cin;
#pragma unroll
    for (int i = 0; i < NP; i++)
      pre[i] = in && go[i] >= 0 ? *reinterpret_cast<const uint4*>(p + go[i]) : make_uint4(0, 0, 0, 0);
  };
  auto put = [&](int slot) {
#pragma unroll
    for (int i = 0; i < NP; i++)
      if (lo[i] >= 0) *reinterpret_cast<uint4*>(planes + slot * pb + lo[i]) = pre[i];
  };
  load(zs - 1);
  put(0);
  load(zs);
  put(1);
  load(zs + 1);
  const int row = lane & 15, kq = (lane >> 4) * 8, y = y0 + wave, K27 = 27 * Cin;
  const char* av = planes + (wave * VX + row) * vs;
  const bf16* wl = w + (long)row * Kpad + kq;
  int ph = 0;   // slot of plane z - 1
  for (int z = zs; z < ze; z++) {
    put(ph == 0 ? 2 : ph - 1);   // plane z + 1, where plane z - 2 was
    __syncthreads();
    if (z + 1 < ze) load(z + 2);
    if (y < Y) {   // uniform over the wave
      f32x4 acc[MT][NT];
#pragma unroll
      for (int m = 0; m < MT; m++)
#pragma unroll
        for (int n = 0; n < NT; n++) acc[m][n] = f32x4{0, 0, 0, 0};
      const int* tp = tab + ph * ng + (lane >> 4);
      // the next G steps' weights are in flight while a step is computed
      bf16x8 bw[G][NT];
      auto weights = [&](int q, int k0) {
        const int k = min(k0, Kpad - 32);
#pragma unroll
        for (int n = 0; n < NT; n++) {
          if constexpr (WL) bw[q][n] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(wlds + (16 * n + row) * ws + 2 * (k + kq)));
          else bw[q][n] = load8(wl + (long)16 * n * Kpad + k);
        }
      };
      auto step = [&](int q, int k0, bool tail) {
        const int off = tp[k0 / 8];
        bf16x8 a[MT];
#pragma unroll
        for (int m = 0; m < MT; m++) {
          a[m] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(av + off + 16 * m * vs));
          if (tail && k0 + kq >= K27) a[m] = zero8();   // the padding of K
        }
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
          for (int m = 0; m < MT; m++) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bw[q][n], a[m], acc[m][n], 0, 0, 0);
      };
#pragma unroll
      for (int q = 0; q < G; q++) weights(q, 32 * q);
      int k0 = 0;
      for (; k0 + 32 * G <= K27; k0 += 32 * G) {
#pragma unroll
        for (int q = 0; q < G; q++) {
          step(q, k0 + 32 * q, false);
          weights(q, k0 + 32 * (G + q));
        }
      }
#pragma unroll
      for (int q = 0; q < G; q++)
        if (k0 + 32 * q < Kpad) step(q, k0 + 32 * q, true);
      conv_epilogue<MT, NT>(acc, x0, y, z, Y, X, bias, epi, slope, act, out_bf, out_f, Cout_store);
    }
    __syncthreads();
    ph = ph == 2 ? 0 : ph + 1;
  }
}

// dw partials: a block takes the three taps of one (dz, dy) for up to NCI
// 16-channel input tiles and one 16-channel output tile, over the voxels of
// slab blockIdx.y; its waves take chunks of 32 voxels in turn, each in LDS of
// its own and without barriers.  A chunk's dy (32 voxels) and x (the same
// voxels displaced by dz and dy, and one more at either end) are loaded with
// contiguous 16-byte loads, stored voxel by voxel, and read back transposed
// (ds_read_b64_tr_b16), so that a lane holds 8 voxels of one channel, its
// share of an MFMA operand: the three taps read the same x tile at row offsets
// -1, 0 and 1.  Voxels whose tap falls outside the grid are masked in the
// operand (a chunk inside a row skips that).  The next chunk's loads are in
// flight while the current one is multiplied.
//
// What bounds it: with one tap and one input tile per block, every tile was
// stored element by element (16 two-byte LDS stores a voxel) for one matrix
// instruction per wave between two barriers; here five loads and five LDS
// stores serve nine.  48 -> 16 channels at 96^3: 560 -> 203 us (180 TFLOP/s).
// On small slabs the last phase, which adds the waves' sums, weighs more than
// the chunks: fewer waves there (conv_dw_waves).
constexpr int DW_CHUNK = 32;

typedef short s16x4 __attribute__((ext_vector_type(4)));
// transposed read of rows r0 .. r0 + 31 of a [voxel][16] tile: lane l receives
// channel l % 16 of voxels 4 (l / 16) + j and 16 + 4 (l / 16) + j (j < 4), an
// order of K that both operands share
__device__ __forceinline__ bf16x8 read_tr(const bf16* tile, int r0, int lane) {
  typedef __attribute__((address_space(3))) s16x4 lds4;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)(tile + 16 * r0 + 4 * lane));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)(tile + 16 * (r0 + 16) + 4 * lane));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int NCI, int DW_WAVES>
__global__ void __launch_bounds__(64 * DW_WAVES) k_conv_dw(const bf16* __restrict__ x, const bf16* __restrict__ dy,
                                                           int Z, int Y, int X, int Cin, int Cout, int zslab,
                                                           float* __restrict__ part) {
  constexpr int XR = DW_CHUNK + 2;             // voxels of an x tile
  constexpr int WT = (DW_CHUNK + NCI * XR) * 16;   // values of a wave's tiles
  constexpr int RED = DW_WAVES * NCI * 256;    // floats of one tap's sums
  __shared__ __align__(16) char smem[DW_WAVES * WT * 2 > RED * 4 ? DW_WAVES * WT * 2 : RED * 4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nci = Cin / 16, nco = Cout / 16, ng = (nci + NCI - 1) / NCI;
  const int t = blockIdx.x;
  const int zy = t / (ng * nco);   // 3 (dz + 1) + dy + 1
  const int c0 = ((t / nco) % ng) * NCI, co0 = (t % nco) * 16;
  const int nt = min(NCI, nci - c0);   // input tiles of this block
  const int dz = zy / 3 - 1, dyy = zy % 3 - 1;
  const int z0 = blockIdx.y * zslab, z1 = min(Z, z0 + zslab);
  // voxels of a slab fit 32-bit indices (the launcher checks the volume)
  const unsigned nv = (unsigned)(z1 - z0) * Y * X;
  const long base = (long)z0 * Y * X, vol = (long)Z * Y * X, shift = (long)(dz * Y + dyy) * X;
  bf16* A = reinterpret_cast<bf16*>(smem) + wave * WT;
  bf16* B = A + DW_CHUNK * 16;
  // coordinates of this lane's voxel of the chunk (lane % 32); a wave's next
  // chunk is DW_WAVES chunks on
  constexpr unsigned STEP = DW_WAVES * DW_CHUNK;
  unsigned v0 = wave * DW_CHUNK;   // the chunk's first voxel within the slab
  const unsigned vl = v0 + (lane & 31), uX = X, uY = Y;
  int xx = (int)(vl % uX), yy = (int)(vl / uX % uY), zz = z0 + (int)(vl / uX / uY);
  const int sx = (int)(STEP % uX), sy = (int)(STEP / uX % uY), sz = (int)(STEP / uX / uY);
  // loads: dy, voxel lane / 2; x, 16-byte piece i 64 + lane of the tile's
  // 34 voxels x 2 nt pieces
  constexpr int NX = (XR * 2 * NCI + 63) / 64;
  uint4 ra, rx[NX];
  unsigned m[3];   // voxels whose tap dx - 1 lies in the grid
  const int np = 2 * nt;
  int gx[NX], lx[NX], vx[NX];   // offset from the voxel before the chunk, place in the tiles, voxel
#pragma unroll
  for (int i = 0; i < NX; i++) {
    const int c = 64 * i + lane, piece = c % np;
    vx[i] = c / np;
    gx[i] = vx[i] * Cin + 16 * c0 + 8 * piece;
    lx[i] = (piece >> 1) * (XR * 16) + vx[i] * 16 + 8 * (piece & 1);
    if (vx[i] >= XR) vx[i] = 1 << 20;
  }
  auto load = [&]() {
    const bool in = v0 + (lane & 31) < nv;
    const int pz = zz + dz, py = yy + dyy;
    const bool ok = in && pz >= 0 && pz < Z && py >= 0 && py < Y;
    m[0] = (unsigned)__ballot(ok && xx > 0);
    m[1] = (unsigned)__ballot(ok);
    m[2] = (unsigned)__ballot(ok && xx < X - 1);
    const unsigned va = v0 + (lane >> 1);
    ra = va < nv ? *reinterpret_cast<const uint4*>(dy + (base + va) * Cout + co0 + 8 * (lane & 1)) : make_uint4(0, 0, 0, 0);
    // voxels of the x tile inside the tensor (the rest is masked anyway)
    const long f0 = base + shift - 1 + (long)__builtin_amdgcn_readfirstlane((int)v0);
    const int vlo = (int)max(0L, min(-f0, 1L << 20)), vhi = (int)max(0L, min((long)XR, vol - f0));
    const bf16* xp = x + f0 * Cin;
#pragma unroll
    for (int i = 0; i < NX; i++)
      rx[i] = vx[i] >= vlo && vx[i] < vhi ? *reinterpret_cast<const uint4*>(xp + gx[i]) : make_uint4(0, 0, 0, 0);
    v0 += STEP;
    xx += sx; yy += sy; zz += sz;
    if (xx >= X) { xx -= X; yy++; }
    if (yy >= Y) { yy -= Y; zz++; }
  };
  f32x4 acc[3][NCI];
#pragma unroll
  for (int k = 0; k < 3; k++)
#pragma unroll
    for (int n = 0; n < NCI; n++) acc[k][n] = f32x4{0, 0, 0, 0};
  if (v0 < nv) load();
  for (unsigned c = wave * DW_CHUNK; c < nv; c += STEP) {
    reinterpret_cast<uint4*>(A)[lane] = ra;
#pragma unroll
    for (int i = 0; i < NX; i++)
      if (vx[i] < XR) *reinterpret_cast<uint4*>(B + lx[i]) = rx[i];
    const unsigned mk[3] = {m[0], m[1], m[2]};
    if (c + STEP < nv) load();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // A = dy^T (rows co, cols voxels), B = x at the tap (rows voxels, cols ci)
    const bf16x8 a = read_tr(A, 0, lane);
#pragma unroll
    for (int k = 0; k < 3; k++) {
      if (mk[k] == 0) continue;   // uniform over the wave
      // 0xffff for the halves of the operand's voxels inside the grid
      uint4 keep = make_uint4(~0u, ~0u, ~0u, ~0u);
      if (mk[k] != ~0u) {
        const unsigned lo = mk[k] >> (4 * (lane >> 4)), hi = lo >> 16;
        auto two = [](unsigned bits) { return ((bits & 1) ? 0xffffu : 0u) | ((bits & 2) ? 0xffff0000u : 0u); };
        keep = make_uint4(two(lo), two(lo >> 2), two(hi), two(hi >> 2));
      }
#pragma unroll
      for (int n = 0; n < NCI; n++) {
        if (n >= nt) continue;   // uniform
        uint4 o = __builtin_bit_cast(uint4, read_tr(B + n * XR * 16, k, lane));
        if (mk[k] != ~0u) { o.x &= keep.x; o.y &= keep.y; o.z &= keep.z; o.w &= keep.w; }
        acc[k][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, o), acc[k][n], 0, 0, 0);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  // the waves' sums in a fixed order, one tap at a time in the tiles' memory
  float* red = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int k = 0; k < 3; k++) {
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NCI; n++)
#pragma unroll
      for (int i = 0; i < 4; i++) red[((wave * NCI + n) * 64 + lane) * 4 + i] = acc[k][n][i];
    __syncthreads();
    for (int e = threadIdx.x; e < nt * 256; e += 64 * DW_WAVES) {
      const int n = e / 256, ln = (e % 256) / 4, i = e % 4;
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < DW_WAVES; w++) sum += red[((w * NCI + n) * 64 + ln) * 4 + i];
      const int co = co0 + 4 * (ln >> 4) + i, ci = 16 * (c0 + n) + (ln & 15);
      part[((long)blockIdx.y * Cout + co) * (27L * Cin) + (long)(3 * zy + k) * Cin + ci] = sum;
    }
  }
}

__global__ void k_reduce_slabs(const float* __restrict__ part, int nslab, long n, float* __restrict__ dw) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  float s = 0.f;
  for (int q = 0; q < nslab; q++) s += part[q * n + i];
  dw[i] = s;
}

// bias gradient db[co] = sum over voxels of dy[v][co] (channels fastest), in
// two passes of fixed order: block b sums the voxels [b chunk, (b+1) chunk)
// of every channel, 256 / C voxels at a time with consecutive threads on
// consecutive (voxel, channel) elements, into part[b][co]; then the blocks'
// sums are added (a fixed tree per channel).  (C <= 256.)
__global__ void __launch_bounds__(256) k_bias_part(const bf16* __restrict__ dy, long nv, int C, long chunk,
                                                   float* __restrict__ part) {
  __shared__ float red[256];
  const int t = threadIdx.x, G = 256 / C, g = t / C, co = t % C;
  float s = 0.f;
  if (g < G) {
    const long v0 = (long)blockIdx.x * chunk, v1 = min(v0 + chunk, nv);
    for (long v = v0 + g; v < v1; v += G) s += bf2f(dy[v * C + co]);
  }
  red[t] = s;
  __syncthreads();
  if (t < C) {
    float a = 0.f;
    for (int k = 0; k < G; k++) a += red[k * C + t];
    part[(long)blockIdx.x * C + t] = a;
  }
}

// block co: the nb block sums of channel co, 256 at a time, then a tree
__global__ void __launch_bounds__(256) k_bias_sum(const float* __restrict__ part, int nb, int C,
                                                  float* __restrict__ db) {
  __shared__ float red[256];
  const int co = blockIdx.x, t = threadIdx.x;
  float a = 0.f;
  for (int b = t; b < nb; b += 256) a += part[(long)b * C + co];
  red[t] = a;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (t < o) red[t] += red[t + o];
    __syncthreads();
  }
  if (t == 0) db[co] = red[0];
}

// bf16 weights for the forward (w[co][Kpad]) and input-gradient
// (wt[ci][KpadT]) kernels from FP32 master weights m[co][27*Cin]
__global__ void k_prep_weights(const float* __restrict__ m, int Cin, int Cout, int Kpad, int KpadT,
                               bf16* __restrict__ w, bf16* __restrict__ wt) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const long nw = (long)Cout * Kpad, nt = (long)Cin * KpadT;
  if (i < nw) {
    const int co = (int)(i / Kpad), k = (int)(i % Kpad);
    w[i] = k < 27 * Cin ? f2bf(m[(long)co * 27 * Cin + k]) : (bf16)0;
  }
  if (i < nt) {
    const int ci = (int)(i / KpadT), k = (int)(i % KpadT);
    bf16 v = 0;
    if (k < 27 * Cout) {
      const int tp = k / Cout, co = k % Cout;
      v = f2bf(m[(long)co * 27 * Cin + (26 - tp) * Cin + ci]);
    }
    wt[i] = v;
  }
}

__global__ void k_pool2(const bf16* __restrict__ in, int Z, int Y, int X, int C, bf16* __restrict__ out) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const int Z2 = Z / 2, Y2 = Y / 2, X2 = X / 2;
  const long n = (long)Z2 * Y2 * X2 * C;
  if (i >= n) return;
  const int c = (int)(i % C);
  long v = i / C;
  const int x = (int)(v % X2), y = (int)((v / X2) % Y2), z = (int)(v / ((long)X2 * Y2));
  float s = 0.f;
  for (int q = 0; q < 8; q++) {
    const int zz = 2 * z + (q >> 2), yy = 2 * y + ((q >> 1) & 1), xx = 2 * x + (q & 1);
    s += bf2f(in[(((long)zz * Y + yy) * X + xx) * C + c]);
  }
  out[i] = f2bf(0.125f * s);
}

__global__ void k_pool2_bwd(const bf16* __restrict__ dout, int Z, int Y, int X, int C, bf16* __restrict__ din,
                            int accumulate) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const long n = (long)Z * Y * X * C;
  if (i >= n) return;
  const int c = (int)(i % C);
  long v = i / C;
  const int x = (int)(v % X), y = (int)((v / X) % Y), z = (int)(v / ((long)X * Y));
  const int Y2 = Y / 2, X2 = X / 2;
  float g = 0.125f * bf2f(dout[(((long)(z / 2) * Y2 + y / 2) * X2 + x / 2) * C + c]);
  if (accumulate) g += bf2f(din[i]);
  din[i] = f2bf(g);
}

// nearest 2x upsampling of `in` [Z/2][Y/2][X/2][C1] into channels [0, C1) of
// out [Z][Y][X][C1+C2]; channels [C1, C1+C2) take the skip tensor
__global__ void k_up2_cat(const bf16* __restrict__ in, const bf16* __restrict__ skip, int Z, int Y, int X, int C1,
                          int C2, bf16* __restrict__ out) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const int C = C1 + C2;
  const long n = (long)Z * Y * X * C;
  if (i >= n) return;
  const int c = (int)(i % C);
  const long v = i / C;
  if (c < C1) {
    const int x = (int)(v % X), y = (int)((v / X) % Y), z = (int)(v / ((long)X * Y));
    out[i] = in[(((long)(z / 2) * (Y / 2) + y / 2) * (X / 2) + x / 2) * C1 + c];
  } else {
    out[i] = skip[v * C2 + (c - C1)];
  }
}

// backward of k_up2_cat: din[parent][c] = sum over the 8 children; dskip is
// the gradient of the skip channels (added to dskip_acc when accumulate)
__global__ void k_up2_cat_bwd(const bf16* __restrict__ dout, int Z, int Y, int X, int C1, int C2,
                              bf16* __restrict__ din, bf16* __restrict__ dskip, int accumulate) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const int C = C1 + C2;
  const int Z2 = Z / 2, Y2 = Y / 2, X2 = X / 2;
  const long n1 = (long)Z2 * Y2 * X2 * C1, n2 = (long)Z * Y * X * C2;
  if (i < n1) {
    const int c = (int)(i % C1);
    const long v = i / C1;
    const int x = (int)(v % X2), y = (int)((v / X2) % Y2), z = (int)(v / ((long)X2 * Y2));
    float s = 0.f;
    for (int q = 0; q < 8; q++) {
      const int zz = 2 * z + (q >> 2), yy = 2 * y + ((q >> 1) & 1), xx = 2 * x + (q & 1);
      s += bf2f(dout[(((long)zz * Y + yy) * X + xx) * C + c]);
    }
    din[i] = f2bf(s);
  }
  if (i < n2) {
    const int c = (int)(i % C2);
    const long v = i / C2;
    float g = bf2f(dout[v * C + C1 + c]);
    if (accumulate) g += bf2f(dskip[i]);
    dskip[i] = f2bf(g);
  }
}

// g = g * (a > 0 ? 1 : slope): gradient through a LeakyReLU given its output
__global__ void k_dact(bf16* __restrict__ g, const bf16* __restrict__ a, long n, float slope) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float av = bf2f(a[i]);
  g[i] = f2bf(av > 0.f ? bf2f(g[i]) : slope * bf2f(g[i]));
}

// masked mean-square error between out [V][Cs] (FP32) and target [V][Cs];
// grad [V][16] BF16 = 2 (out - t) m / count (channels >= Cs zero); per-block
// partial sums of the squared error
__global__ void k_mse(const float* __restrict__ out, const float* __restrict__ tgt, const float* __restrict__ mask,
                      long nv, int Cs, float inv_count, bf16* __restrict__ grad, float* __restrict__ part) {
  __shared__ float red[256];
  const long v = blockIdx.x * (long)blockDim.x + threadIdx.x;
  float s = 0.f;
  if (v < nv) {
    for (int c = 0; c < 16; c++) {
      float g = 0.f;
      if (c < Cs) {
        const float m = mask[v * Cs + c];
        const float d = (out[v * Cs + c] - tgt[v * Cs + c]) * m;
        s += d * d;
        g = 2.f * d * inv_count;
      }
      grad[v * 16 + c] = f2bf(g);
    }
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m1,
                       float* __restrict__ m2, long n, float lr, float b1, float b2, float eps, float c1, float c2,
                       float clip) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  float gi = g[i];
  gi = fminf(fmaxf(gi, -clip), clip);
  const float a = b1 * m1[i] + (1.f - b1) * gi;
  const float b = b2 * m2[i] + (1.f - b2) * gi * gi;
  m1[i] = a;
  m2[i] = b;
  p[i] -= lr * (a / c1) / (sqrtf(b / c2) + eps);
}

// FP32 [V][C] -> BF16 [V][Cp] (channels >= C zero)
__global__ void k_pack_bf16(const float* __restrict__ in, long nv, int C, int Cp, bf16* __restrict__ out) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= nv * Cp) return;
  const int c = (int)(i % Cp);
  const long v = i / Cp;
  out[i] = c < C ? f2bf(in[v * C + c]) : (bf16)0;
}

// The network refines a field x1 (the field after one multigrid cycle): per
// component a it outputs three channels, a change of log-amplitude dL and a
// relative phasor (1 + q1) + i q2, and the refined field is
//   E_a = x1_a exp(dL) ((1 + q1) + i q2) / |(1 + q1) + i q2|.
// Zero outputs reproduce x1 exactly.

// Network output [n3][n2][n1][9] and x1 -> complex double edge vector x0
// [3][n3+1][n2+1][n1+1] (interior edges; others 0)
__global__ void k_out_to_edges(const float* __restrict__ o, const double2* __restrict__ x1, int n1, int n2, int n3,
                               double2* __restrict__ x0) {
  const long nc = (long)(n1 + 1) * (n2 + 1) * (n3 + 1);
  const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (t >= 3 * nc) return;
  const int a = (int)(t / nc);
  const long e = t % nc;
  const int i = (int)(e % (n1 + 1)), j = (int)((e / (n1 + 1)) % (n2 + 1)), k = (int)(e / ((long)(n1 + 1) * (n2 + 1)));
  const int p[3] = {i, j, k};
  const int n[3] = {n1, n2, n3};
  const int b = (a + 1) % 3, c = (a + 2) % 3;
  double2 v = make_double2(0.0, 0.0);
  if (p[a] < n[a] && p[b] >= 1 && p[b] <= n[b] - 1 && p[c] >= 1 && p[c] <= n[c] - 1) {
    const long cell = ((long)k * n2 + j) * n1 + i;
    const double dL = fmin(fmax((double)o[cell * 9 + 3 * a], -20.0), 20.0);
    const double qr = 1.0 + (double)o[cell * 9 + 3 * a + 1], qi = o[cell * 9 + 3 * a + 2];
    const double nrm = sqrt(qr * qr + qi * qi);
    const double2 u = x1[t];
    if (nrm > 1e-6) {
      const double s = exp(dL) / nrm;
      v.x = s * (u.x * qr - u.y * qi);
      v.y = s * (u.x * qi + u.y * qr);
    }
  }
  x0[t] = v;
}

// The same with the correction of each edge averaged over the four cells
// that share the edge, so the guess varies as smoothly as x1 between edges;
// cells whose conductivity s11 is below sig_air (the air) take no correction
// (s11 may be null: no cell is excluded).
__global__ void k_out_to_edges_avg(const float* __restrict__ o, const double2* __restrict__ x1,
                                   const float* __restrict__ s11, float sig_air, int n1, int n2, int n3,
                                   double2* __restrict__ x0) {
  const long nc = (long)(n1 + 1) * (n2 + 1) * (n3 + 1);
  const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (t >= 3 * nc) return;
  const int a = (int)(t / nc);
  const long e = t % nc;
  const int i = (int)(e % (n1 + 1)), j = (int)((e / (n1 + 1)) % (n2 + 1)), k = (int)(e / ((long)(n1 + 1) * (n2 + 1)));
  const int p[3] = {i, j, k};
  const int n[3] = {n1, n2, n3};
  const int b = (a + 1) % 3, c = (a + 2) % 3;
  double2 v = make_double2(0.0, 0.0);
  if (p[a] < n[a] && p[b] >= 1 && p[b] <= n[b] - 1 && p[c] >= 1 && p[c] <= n[c] - 1) {
    double dL = 0.0, qr = 0.0, qi = 0.0;
#pragma unroll
    for (int s = 0; s < 4; s++) {
      int q[3] = {p[0], p[1], p[2]};
      q[b] -= s & 1;
      q[c] -= s >> 1;
      const long cell = ((long)q[2] * n2 + q[1]) * n1 + q[0];
      if (s11 && s11[cell] < sig_air) continue;
      dL += 0.25 * fmin(fmax((double)o[cell * 9 + 3 * a], -20.0), 20.0);
      qr += 0.25 * (double)o[cell * 9 + 3 * a + 1];
      qi += 0.25 * (double)o[cell * 9 + 3 * a + 2];
    }
    qr += 1.0;
    const double nrm = sqrt(qr * qr + qi * qi);
    const double2 u = x1[t];
    if (nrm > 1e-6) {
      const double sc = exp(dL) / nrm;
      v.x = sc * (u.x * qr - u.y * qi);
      v.y = sc * (u.x * qi + u.y * qr);
    }
  }
  x0[t] = v;
}

// Training targets [V][9] for refining x1 towards the solved field E, and the
// loss weights: 1 on dL, wp on the phasor channels, where both |E_a| and
// |x1_a| exceed eref (elsewhere 0: the field is negligible there)
__global__ void k_edges_to_target(const double2* __restrict__ E, const double2* __restrict__ x1, int n1, int n2,
                                  int n3, double eref, float wp, float* __restrict__ tgt, float* __restrict__ mask) {
  const long ncell = (long)n1 * n2 * n3;
  const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (t >= ncell) return;
  const int i = (int)(t % n1), j = (int)((t / n1) % n2), k = (int)(t / ((long)n1 * n2));
  const int p[3] = {i, j, k};
  const int n[3] = {n1, n2, n3};
  const long es1 = n1 + 1, es2 = (long)(n1 + 1) * (n2 + 1), nc = es2 * (n3 + 1);
  for (int a = 0; a < 3; a++) {
    const int b = (a + 1) % 3, c = (a + 2) % 3;
    const bool in = p[b] >= 1 && p[b] <= n[b] - 1 && p[c] >= 1 && p[c] <= n[c] - 1;
    const long o = a * nc + i + es1 * j + es2 * k;
    const double2 v = in ? E[o] : make_double2(0.0, 0.0);
    const double2 u = in ? x1[o] : make_double2(0.0, 0.0);
    const double av = sqrt(v.x * v.x + v.y * v.y), au = sqrt(u.x * u.x + u.y * u.y);
    const bool ok = in && av > eref && au > eref;
    // relative phasor (E/|E|) conj(x1/|x1|)
    const double rr = ok ? (v.x * u.x + v.y * u.y) / (av * au) : 1.0;
    const double ri = ok ? (v.y * u.x - v.x * u.y) / (av * au) : 0.0;
    tgt[t * 9 + 3 * a] = ok ? (float)log(av / au) : 0.f;
    tgt[t * 9 + 3 * a + 1] = (float)(rr - 1.0);
    tgt[t * 9 + 3 * a + 2] = (float)ri;
    mask[t * 9 + 3 * a] = ok ? 1.f : 0.f;
    mask[t * 9 + 3 * a + 1] = ok ? wp : 0.f;
    mask[t * 9 + 3 * a + 2] = ok ? wp : 0.f;
  }
}

// Input features on the cells [n3][n2][n1][32]:
//   0 log10 sigma11, 1 log10 sigma33, 2..4 (x - xs)/delta per axis (clamped
//   to +-8), 5 log10(r/delta + 1e-3), 6 log10(cell size / delta),
//   7 source blob exp(-(r/h)^2) with h the source cell size, 8 constant 1,
//   9..17 when x1 is given: per component a of the field x1 after one
//   multigrid cycle, ln(max(|x1_a|, eref)/eref)/10 and its unit phasor
__global__ void k_features(const float* __restrict__ s11, const float* __restrict__ s33, const float* __restrict__ xs1,
                           const float* __restrict__ xs2, const float* __restrict__ xs3, const float* __restrict__ d1,
                           const float* __restrict__ d2, const float* __restrict__ d3, int n1, int n2, int n3,
                           float sx, float sy, float sz, float delta, float hsrc, const double2* __restrict__ x1,
                           double eref, bf16* __restrict__ feat) {
  const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const long nc = (long)n1 * n2 * n3;
  if (t >= nc) return;
  const int i = (int)(t % n1), j = (int)((t / n1) % n2), k = (int)(t / ((long)n1 * n2));
  float f[32];
  for (int c = 0; c < 32; c++) f[c] = 0.f;
  f[0] = log10f(fmaxf(s11[t], 1e-12f));
  f[1] = log10f(fmaxf(s33[t], 1e-12f));
  const float dx = xs1[i] - sx, dy = xs2[j] - sy, dz = xs3[k] - sz;
  f[2] = fminf(fmaxf(dx / delta, -8.f), 8.f);
  f[3] = fminf(fmaxf(dy / delta, -8.f), 8.f);
  f[4] = fminf(fmaxf(dz / delta, -8.f), 8.f);
  const float r = sqrtf(dx * dx + dy * dy + dz * dz);
  f[5] = log10f(r / delta + 1e-3f);
  f[6] = log10f(cbrtf(d1[i] * d2[j] * d3[k]) / delta);
  f[7] = expf(-(r / hsrc) * (r / hsrc));
  f[8] = 1.f;
  if (x1) {
    const int p[3] = {i, j, k};
    const int n[3] = {n1, n2, n3};
    const long es1 = n1 + 1, es2 = (long)(n1 + 1) * (n2 + 1), ncc = es2 * (n3 + 1);
    for (int a = 0; a < 3; a++) {
      const int b = (a + 1) % 3, c = (a + 2) % 3;
      const bool in = p[b] >= 1 && p[b] <= n[b] - 1 && p[c] >= 1 && p[c] <= n[c] - 1;
      const double2 v = in ? x1[a * ncc + i + es1 * j + es2 * k] : make_double2(0.0, 0.0);
      const double amp = sqrt(v.x * v.x + v.y * v.y);
      f[9 + 3 * a] = (float)(0.1 * log(fmax(amp, eref) / eref));
      f[10 + 3 * a] = amp > eref ? (float)(v.x / amp) : 0.f;
      f[11 + 3 * a] = amp > eref ? (float)(v.y / amp) : 0.f;
    }
  }
  for (int c = 0; c < 32; c++) feat[t * 32 + c] = f2bf(f[c]);
}

__global__ void k_fill_u32(uint32_t* __restrict__ p, long n, uint32_t v) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void k_scale(double2* __restrict__ v, long n, double s) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i < n) { v[i].x *= s; v[i].y *= s; }
}

inline unsigned blocks(long n, int b) { return (unsigned)((n + b - 1) / b); }
hipStream_t S(void* s) { return (hipStream_t)s; }

template <int MT>
void conv_fwd_mt(const bf16* x, int Z, int Y, int X, int Cin, const bf16* w, int Kpad, int Cout, const float* bias,
                 int epi, float slope, const bf16* act, bf16* ob, float* of, int cstore, hipStream_t s) {
  // the last tile of a row may be partial: loads and stores check x < X
  const dim3 g((X + 16 * MT - 1) / (16 * MT), (Y + 3) / 4, Z), b(256);
  hipEvent_t e0, e1;
  emmi::timing::kernel_events(emmi::timing::CONV, 54.0 * Cin * Cout * (double)Z * Y * X, &e0, &e1);
  switch (Cout / 16) {
#define CASE(NT)                                                                                                   \
  case NT:                                                                                                         \
    if (e0) hipExtLaunchKernelGGL((k_conv_fwd<MT, NT>), g, b, 0, s, e0, e1, 0, x, Z, Y, X, Cin, w, Kpad, bias, epi, \
                                  slope, act, ob, of, cstore);                                                     \
    else hipLaunchKernelGGL((k_conv_fwd<MT, NT>), g, b, 0, s, x, Z, Y, X, Cin, w, Kpad, bias, epi, slope, act, ob,  \
                            of, cstore);                                                                           \
    break;
    CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
  }
}

// LDS bytes of k_conv_fwd_lds for rows TY
size_t conv_lds(int TY, int Cin, int Kpad) {
  return 3 * (size_t)((TY + 2) * 34) * (2 * Cin + 16) + (3 * (Kpad / 8) * sizeof(int) + 15) / 16 * 16;
}

// planes that a block of k_conv_fwd_lds marches through: one where all tiles of
// all planes fill no more than the 256 CUs (two would double the serial time of
// a launch that leaves CUs idle: 8 x 9 x 33, 16 -> 16 channels 8.8 and 5.9 us),
// else enough for about two blocks a CU
int conv_planes(int Z, int Y, int X, int TY) {
  const long tiles = (long)((X + 31) / 32) * ((Y + TY - 1) / TY), n = Z * tiles;
  return n <= 256 ? 1 : (int)std::max(2L, n / 512);
}

// The rows that k_conv_fwd_lds takes, eight where the planes of the tile fit the
// LDS beside the table, four for more channels; 0: k_conv_fwd is the faster one.
// With the weights in LDS, or 16 outputs, the march wins (1.0x for a single 8 x 32
// plane of 16 -> 32 channels to 2.8x; the least of all sizes measured is 0.93,
// 32 -> 16 on 1000 planes of 9 x 33).  With weights from memory it is bound by their loads:
//  - where tiles leave CUs idle both are chains of latencies, and the march is
//    ahead with four rows and up to 48 outputs (128 x 128 plane, 80 -> 32
//    channels 32 and 24 us, 48 -> 64 28 and 33);
//  - where k_conv_fwd's waves hold one tile of 16 voxels (X no multiple of 32),
//    the march is about 1.9 (80 channels 1.8, 64, 96 and 112 2.1) times as fast
//    per voxel of its tiles, but wastes more of them at the grid's edges and in the last
//    round of blocks: it is taken by the ratio of the two fills (64 -> 64 at
//    80^3, ratio 0.65: 940 and 639 us; 48 -> 48 at 40^3, 0.59: 55 and 47, at 48^3,
//    0.42: 75 and 92);
//  - where they hold two or four tiles k_conv_fwd is ahead (48 -> 48 channels at
//    96^3 326 and 393 us, 64 -> 64 at 32^3 41 and 110) but for 96 channels and
//    more into up to 48 (112 -> 48 at 96^3 932 and 807).
int conv_rows(int Z, int Y, int X, int Cin, int Kpad, int Cout) {
  if (X < 32 || Y < 8 || Cin > 112 || (long)Y * X * Cin >= (1L << 31)) return 0;
  const int TY = Cin <= 64 && conv_lds(8, Cin, Kpad) <= (size_t)emmi::CU_LDS ? 8 : 4;
  if (conv_lds(TY, Cin, Kpad) > (size_t)emmi::CU_LDS) return 0;
  if (Cout == 16 || conv_lds(TY, Cin, Kpad) + (size_t)Cout * (2 * Kpad + 16) <= (size_t)emmi::CU_LDS) return TY;
  const int tx = (X + 31) / 32, ty = (Y + TY - 1) / TY, zper = conv_planes(Z, Y, X, TY);
  if (zper == 1) return TY == 4 && Cout <= 48 ? TY : 0;
  const double rounds = (double)(((long)tx * ty * ((Z + zper - 1) / zper) + 255) / 256);
  // voxels of the grid over those of the tile rows that the CUs' rounds hold, the same of k_conv_fwd's tiles
  const double fill = (double)Z * Y * X / (rounds * 256 * zper * 32 * TY);
  const double fill_fwd = (double)X / ((X + 15) / 16 * 16) * Y / ((Y + 3) / 4 * 4);
  const double least = X % 32 != 0 ? (Cin >= 64 && Cin != 80 ? 0.48 : 0.53) : Cin >= 96 && Cout <= 48 ? 0.6 : 2.0;
  return fill >= least * fill_fwd ? TY : 0;
}

// waves of a k_conv_dw block by the voxels of a slab: with sixteen, most of them
// have no chunk on a small slab, and two blocks fill a CU.  All launches of a
// weight and bias gradient, with 16, 8 and 4 waves (one wave per tile and tap,
// four per block, before): 64 -> 64 channels at 8^3 (slabs of 64 voxels) 21.5,
// 17.5 and 16.3 us (16.4); at 12^3 (144) 29.2, 22.7 and 20.5 (23.2); at 31^3 (961)
// 78.5, 56.7 and 53.2 (114.7); 16 -> 16 at 31^3 26.2, 23.3 and 24.5 (24.2), at 32^3
// (2048) 20.0, 21.0 and 26.4 (23.7).
int conv_dw_waves(long nv) { return nv <= 2 * DW_CHUNK ? 4 : nv <= 32 * DW_CHUNK ? 8 : 16; }

template <int TY, int NP>
bool conv_fwd_lds(const bf16* x, int Z, int Y, int X, int Cin, const bf16* w, int Kpad, int Cout, const float* bias,
                  int epi, float slope, const bf16* act, bf16* ob, float* of, int cstore, hipStream_t s) {
  const int zper = conv_planes(Z, Y, X, TY);
  const dim3 g((X + 31) / 32, (Y + TY - 1) / TY, (Z + zper - 1) / zper), b(64 * TY);
  // the weights join the planes where they fit
  const size_t planes = conv_lds(TY, Cin, Kpad), wl = (size_t)Cout * (2 * Kpad + 16);
  const bool in_lds = planes + wl <= (size_t)emmi::CU_LDS;
  const size_t lds = in_lds ? planes + wl : planes;
  hipEvent_t e0, e1;
  emmi::timing::kernel_events(emmi::timing::CONV, 54.0 * Cin * Cout * (double)Z * Y * X, &e0, &e1);
  auto go = [&](auto kernel) {
    if (lds > 64 * 1024 && emmi::allow_lds(reinterpret_cast<const void*>(kernel)) != hipSuccess) return false;
    if (e0) hipExtLaunchKernelGGL(kernel, g, b, lds, s, e0, e1, 0, x, Z, Y, X, Cin, w, Kpad, bias, epi, slope, act, ob, of, cstore, zper);
    else hipLaunchKernelGGL(kernel, g, b, lds, s, x, Z, Y, X, Cin, w, Kpad, bias, epi, slope, act, ob, of, cstore, zper);
    return true;
  };
  switch (Cout / 16) {
#define CASE(NT) case NT: return in_lds ? go(k_conv_fwd_lds<NT, TY, NP, true>) : go(k_conv_fwd_lds<NT, TY, NP, false>);
    CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
  }
  return true;
}

}  // namespace

extern "C" {

int emmi_x0_kpad(int cin) { return (27 * cin + 31) / 32 * 32; }

int emmi_x0_conv_route(int Z, int Y, int X, int Cin, int Cout) {
  if (Cin % 16 || Cout % 16 || Cout > 128 || Cin <= 0 || Cout <= 0 || X <= 0 || Y <= 0 || Z <= 0) return -1;
  return conv_rows(Z, Y, X, Cin, emmi_x0_kpad(Cin), Cout);
}

int emmi_x0_conv_fwd(const void* x, int Z, int Y, int X, int Cin, const void* w, int Cout, const float* bias, int epi,
                     float slope, const void* act, void* out_bf16, float* out_f32, int cout_store, void* stream) {
  if (Cin % 16 || Cout % 16 || Cout > 128 || Cin <= 0 || X <= 0 || Y <= 0 || Z <= 0) return -1;
  const int Kpad = emmi_x0_kpad(Cin);
  const bf16* xb = (const bf16*)x;
  const bf16* wb = (const bf16*)w;
  const int TY = conv_rows(Z, Y, X, Cin, Kpad, Cout);
  bool ok = true;
  if (TY == 8)
    ok = conv_fwd_lds<8, 6>(xb, Z, Y, X, Cin, wb, Kpad, Cout, bias, epi, slope, (const bf16*)act, (bf16*)out_bf16, out_f32, cout_store, S(stream));
  else if (TY == 4)
    ok = conv_fwd_lds<4, 12>(xb, Z, Y, X, Cin, wb, Kpad, Cout, bias, epi, slope, (const bf16*)act, (bf16*)out_bf16, out_f32, cout_store, S(stream));
  else if (X % 64 == 0) conv_fwd_mt<4>(xb, Z, Y, X, Cin, wb, Kpad, Cout, bias, epi, slope, (const bf16*)act, (bf16*)out_bf16, out_f32, cout_store, S(stream));
  else if (X % 32 == 0) conv_fwd_mt<2>(xb, Z, Y, X, Cin, wb, Kpad, Cout, bias, epi, slope, (const bf16*)act, (bf16*)out_bf16, out_f32, cout_store, S(stream));
  else conv_fwd_mt<1>(xb, Z, Y, X, Cin, wb, Kpad, Cout, bias, epi, slope, (const bf16*)act, (bf16*)out_bf16, out_f32, cout_store, S(stream));
  return ok && hipGetLastError() == hipSuccess ? 0 : -1;
}

int emmi_x0_conv_dw(const void* x, const void* dy, int Z, int Y, int X, int Cin, int Cout, float* part, int zslab,
                    float* dw, float* db, void* stream) {
  if (Cin % 16 || Cout % 16 || Cout > 256 || zslab < 1 || Z < 1 || Y < 1 || X < 1) return -1;
  if ((long)Z * Y * X >= (1L << 31)) return -1;   // the kernel indexes voxels in 32 bits
  const int nslab = (Z + zslab - 1) / zslab;
  // input tiles per block: up to three, one where single tiles do not fill the
  // CUs (48 -> 16 channels at 8^3 14.4 and 13.0 us)
  const int nci = Cin / 16, NCI = 9L * nci * (Cout / 16) * nslab <= 256 ? 1 : nci == 4 ? 2 : std::min(nci, 3);
  const int waves = conv_dw_waves((long)std::min(zslab, Z) * Y * X);
  const dim3 g(9 * ((nci + NCI - 1) / NCI) * (Cout / 16), nslab), b(64 * waves);
  hipEvent_t e0, e1;
  emmi::timing::kernel_events(emmi::timing::CONV_DW, 54.0 * Cin * Cout * (double)Z * Y * X, &e0, &e1);
  auto go = [&](auto kernel) {
    if (e0) hipExtLaunchKernelGGL(kernel, g, b, 0, S(stream), e0, e1, 0, (const bf16*)x, (const bf16*)dy, Z, Y, X, Cin,
                                  Cout, zslab, part);
    else hipLaunchKernelGGL(kernel, g, b, 0, S(stream), (const bf16*)x, (const bf16*)dy, Z, Y, X, Cin, Cout, zslab, part);
  };
#define CASE(W)                             \
  case W:                                   \
    if (NCI == 1) go(k_conv_dw<1, W>);      \
    else if (NCI == 2) go(k_conv_dw<2, W>); \
    else go(k_conv_dw<3, W>);               \
    break;
  switch (waves) { CASE(4) CASE(8) CASE(16) }
#undef CASE
  const long n = 27L * Cin * Cout;
  hipLaunchKernelGGL(k_reduce_slabs, dim3(blocks(n, 256)), dim3(256), 0, S(stream), part, nslab, n, dw);
  if (db) {
    // the bias partials reuse part once the slab reduction has read it (same
    // stream): nb Cout floats, nb <= nslab 27 Cin
    const long nv = (long)Z * Y * X;
    const long nbl = std::min<long>(std::min<long>(1024, (long)nslab * 27 * Cin), nv);
    const long chunk = (nv + nbl - 1) / nbl;
    const int nb = (int)((nv + chunk - 1) / chunk);
    hipLaunchKernelGGL(k_bias_part, dim3(nb), dim3(256), 0, S(stream), (const bf16*)dy, nv, Cout, chunk, part);
    hipLaunchKernelGGL(k_bias_sum, dim3(Cout), dim3(256), 0, S(stream), (const float*)part, nb, Cout, db);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int emmi_x0_prep_weights(const float* master, int Cin, int Cout, void* w, void* wt, void* stream) {
  const int Kpad = emmi_x0_kpad(Cin), KpadT = emmi_x0_kpad(Cout);
  const long n = std::max((long)Cout * Kpad, (long)Cin * KpadT);
  hipLaunchKernelGGL(k_prep_weights, dim3(blocks(n, 256)), dim3(256), 0, S(stream), master, Cin, Cout, Kpad, KpadT,
                     (bf16*)w, (bf16*)wt);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int emmi_x0_pool2(const void* in, int Z, int Y, int X, int C, void* out, void* stream) {
  const long n = (long)(Z / 2) * (Y / 2) * (X / 2) * C;
  hipLaunchKernelGGL(k_pool2, dim3(blocks(n, 256)), dim3(256), 0, S(stream), (const bf16*)in, Z, Y, X, C, (bf16*)out);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int emmi_x0_pool2_bwd(const void* dout, int Z, int Y, int X, int C, void* din, int accumulate, void* stream) {
  const long n = (long)Z * Y * X * C;
  hipLaunchKernelGGL(k_pool2_bwd, dim3(blocks(n, 256)), dim3(256), 0, S(stream), (const bf16*)dout, Z, Y, X, C, (bf16*)din,
                     accumulate);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int emmi_x0_up2_cat(const void* in, const void* skip, int Z, int Y, int X, int C1, int C2, void* out, void* stream) {
  const long n = (long)Z * Y * X * (C1 + C2);
  hipLaunchKernelGGL(k_up2_cat, dim3(blocks(n, 256)), dim3(256), 0, S(stream), (const bf16*)in, (const bf16*)skip, Z, Y,
                     X, C1, C2, (bf16*)out);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int emmi_x0_up2_cat_bwd(const void* dout, int Z, int Y, int X, int C1, int C2, void* din, void* dskip, int accumulate,
                        void* stream) {
  const long n = std::max((long)(Z / 2) * (Y / 2) * (X / 2) * C1, (long)Z * Y * X * C2);
  hipLaunchKernelGGL(k_up2_cat_bwd, dim3(blocks(n, 256)), dim3(256), 0, S(stream), (const bf16*)dout, Z, Y, X, C1, C2,
                     (bf16*)din, (bf16*)dskip, accumulate);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int emmi_x0_dact(void* g, const void* a, long n, float slope, void* stream) {
  hipLaunchKernelGGL(k_dact, dim3(blocks(n, 256)), dim3(256), 0, S(stream), (bf16*)g, (const bf16*)a, n, slope);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int emmi_x0_mse(const float* out, const float* tgt, const float* mask, long nv, int cs, float inv_count, void* grad,
                float* part, void* stream) {
  hipLaunchKernelGGL(k_mse, dim3(blocks(nv, 256)), dim3(256), 0, S(stream), out, tgt, mask, nv, cs, inv_count,
                     (bf16*)grad, part);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int emmi_x0_adam(float* p, const float* g, float* m1, float* m2, long n, float lr, float b1, float b2, float eps,
                 int step, float clip, void* stream) {
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(k_adam, dim3(blocks(n, 256)), dim3(256), 0, S(stream), p, g, m1, m2, n, lr, b1, b2, eps, c1, c2,
                     clip);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int emmi_x0_pack_bf16(const float* in, long nv, int C, int Cp, void* out, void* stream) {
  hipLaunchKernelGGL(k_pack_bf16, dim3(blocks(nv * Cp, 256)), dim3(256), 0, S(stream), in, nv, C, Cp, (bf16*)out);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int emmi_x0_out_to_edges(const float* o, const void* x1, int n1, int n2, int n3, void* x0, void* stream) {
  const long n = 3L * (n1 + 1) * (n2 + 1) * (n3 + 1);
  hipLaunchKernelGGL(k_out_to_edges, dim3(blocks(n, 256)), dim3(256), 0, S(stream), o, (const double2*)x1, n1, n2, n3,
                     (double2*)x0);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int emmi_x0_out_to_edges_avg(const float* o, const void* x1, const float* s11, float sig_air, int n1, int n2, int n3,
                             void* x0, void* stream) {
  const long n = 3L * (n1 + 1) * (n2 + 1) * (n3 + 1);
  hipLaunchKernelGGL(k_out_to_edges_avg, dim3(blocks(n, 256)), dim3(256), 0, S(stream), o, (const double2*)x1, s11,
                     sig_air, n1, n2, n3, (double2*)x0);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int emmi_x0_edges_to_target(const void* E, const void* x1, int n1, int n2, int n3, double eref, float wp, float* tgt,
                            float* mask, void* stream) {
  const long n = (long)n1 * n2 * n3;
  hipLaunchKernelGGL(k_edges_to_target, dim3(blocks(n, 256)), dim3(256), 0, S(stream), (const double2*)E,
                     (const double2*)x1, n1, n2, n3, eref, wp, tgt, mask);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int emmi_x0_features(const float* s11, const float* s33, const float* xs1, const float* xs2, const float* xs3,
                     const float* d1, const float* d2, const float* d3, int n1, int n2, int n3, float sx, float sy,
                     float sz, float delta, float hsrc, const void* x1, double eref, void* feat, void* stream) {
  const long n = (long)n1 * n2 * n3;
  hipLaunchKernelGGL(k_features, dim3(blocks(n, 256)), dim3(256), 0, S(stream), s11, s33, xs1, xs2, xs3, d1, d2, d3,
                     n1, n2, n3, sx, sy, sz, delta, hsrc, (const double2*)x1, eref, (bf16*)feat);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int emmi_x0_fill(void* p, long nwords, unsigned value, void* stream) {
  hipLaunchKernelGGL(k_fill_u32, dim3(blocks(nwords, 256)), dim3(256), 0, S(stream), (uint32_t*)p, nwords, value);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int emmi_x0_scale(void* v, long n, double s, void* stream) {
  hipLaunchKernelGGL(k_scale, dim3(blocks(n, 256)), dim3(256), 0, S(stream), (double2*)v, n, s);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // extern "C"
