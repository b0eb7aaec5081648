// Neural-operator kernels for gfx950: BF16 MFMA (v_mfma_f32_32x32x16_bf16)
// with FP32 accumulation.
//
// The operator that warm-starts particle loading is a stack of 3-D
// convolutions on the 64x32x32 simulation grid. Activations are BF16,
// channels-last ([B][Z][Y][X][C], C a multiple of 16); weights are BF16
// [taps][Cout][Cin] (K-contiguous per output channel) with FP32 master
// copies; gradients are FP32.
//
//  * conv_fwd: implicit GEMM, M = voxels, N = Cout, K = taps*Cin. Each wave
//    owns 32 voxels and all Cout (Cout/32 MFMA tiles); A fragments are
//    16-byte loads of 8 channels of the tap's neighbour voxel (zero outside
//    the grid), B fragments 16-byte LDS reads of the K-contiguous weights,
//    which the workgroup stages one tap ahead.
//    Epilogue: bias, optional ReLU, optional residual add, BF16 or FP32 out.
//  * the data gradient is conv_fwd on mirrored, transposed weights
//    (weight_flip), applied to the ReLU-masked output gradient.
//  * conv_bwd_w: per tap a GEMM M = Cout, N = Cin, K = voxels. A chunk of
//    voxels is staged transposed in LDS ([C][k], k contiguous) so both MFMA
//    operands are 16-byte LDS reads; each chunk writes an FP32 partial that
//    reduce_partials sums in a fixed order (deterministic).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

typedef __bf16 bf16;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

namespace {

constexpr int kWaves = 4;
constexpr int kMaxNTiles = 4;   // Cout <= 128
constexpr int kChunk = 128;     // voxels staged per LDS round in conv_bwd_w (two per lane)
constexpr int kLdk = kChunk + 8;  // LDS row length of the staged operands
constexpr int kMaxC = 128;
constexpr int kWRegs = kMaxC * kMaxC / 8 / 256;  // 16-byte weight pieces per thread when staging a tap

__device__ __forceinline__ void tap_offset(int t, int taps, int dil, int& dz, int& dy, int& dx) {
  if (taps == 1) {
    dz = dy = dx = 0;
  } else {
    dz = (t / 9 - 1) * dil;
    dy = ((t / 3) % 3 - 1) * dil;
    dx = (t % 3 - 1) * dil;
  }
}

__device__ __forceinline__ float bf2f(bf16 v) { return (float)v; }

}  // namespace

struct NoConvArgs {
  const bf16* x;
  const bf16* w;
  const float* bias;
  const bf16* res;
  bf16* y;
  float* y32;
  bf16* h;
  int B, Z, Y, X, Cin, Cout, taps, dil, relu;
};

__global__ void __launch_bounds__(256) k_no_conv_fwd(NoConvArgs a) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int V = a.Z * a.Y * a.X;
  const long M = (long)a.B * V;
  const long m = ((long)blockIdx.x * kWaves + wave) * 32 + (lane & 31);
  const int kg = lane >> 5;  // which 8 of the 16 K values this lane supplies
  const int ntiles = a.Cout >> 5;
  f32x16 acc[kMaxNTiles];
#pragma unroll
  for (int j = 0; j < kMaxNTiles; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[j][i] = 0.0f;
  int b = 0, z = 0, y = 0, x = 0;
  const bool valid = m < M;
  if (valid) {
    b = (int)(m / V);
    int r = (int)(m - (long)b * V);
    z = r / (a.Y * a.X);
    r -= z * a.Y * a.X;
    y = r / a.X;
    x = r - y * a.X;
  }
  // The workgroup's four waves share each tap's weights: they are staged in
  // LDS ([Cout][Cin + 8], two buffers), tap t + 1's copied in while tap t is
  // computed, so the B fragments are LDS reads instead of a per-wave reload
  // through L1.
  extern __shared__ __align__(16) bf16 sw[];
  const int ldw = a.Cin + 8;
  const int wchunks = a.Cout * (a.Cin >> 3);  // 16-byte pieces of one tap's weights
  bf16x8 wreg[kWRegs];
  auto fetch_w = [&](int t) {
    const bf16* src = a.w + (long)t * a.Cout * a.Cin;
#pragma unroll
    for (int r = 0; r < kWRegs; ++r) {
      const int q = threadIdx.x + r * 256;
      if (q < wchunks) wreg[r] = *reinterpret_cast<const bf16x8*>(src + (long)q * 8);
    }
  };
  auto store_w = [&](int buf) {
    bf16* dst = sw + (long)buf * a.Cout * ldw;
#pragma unroll
    for (int r = 0; r < kWRegs; ++r) {
      const int q = threadIdx.x + r * 256;
      if (q < wchunks) {
        const int co = q / (a.Cin >> 3), c8 = q - co * (a.Cin >> 3);
        *reinterpret_cast<bf16x8*>(dst + co * ldw + c8 * 8) = wreg[r];
      }
    }
  };
  fetch_w(0);
  store_w(0);
  __syncthreads();
  for (int t = 0; t < a.taps; ++t) {
    if (t + 1 < a.taps) fetch_w(t + 1);
    int dz, dy, dx;
    tap_offset(t, a.taps, a.dil, dz, dy, dx);
    const int zz = z + dz, yy = y + dy, xx = x + dx;
    const bool in = valid && zz >= 0 && zz < a.Z && yy >= 0 && yy < a.Y && xx >= 0 && xx < a.X;
    const bf16* xp = a.x + ((((long)b * a.Z + zz) * a.Y + yy) * a.X + xx) * a.Cin;
    const bf16* wl = sw + (long)(t & 1) * a.Cout * ldw;
    for (int c0 = 0; c0 < a.Cin; c0 += 16) {
      bf16x8 av;
      if (in) {
        av = *reinterpret_cast<const bf16x8*>(xp + c0 + kg * 8);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) av[e] = (bf16)0.0f;
      }
#pragma unroll
      for (int j = 0; j < kMaxNTiles; ++j) {
        if (j < ntiles) {
          const int co = j * 32 + (lane & 31);
          const bf16x8 bv = *reinterpret_cast<const bf16x8*>(wl + co * ldw + c0 + kg * 8);
          acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, acc[j], 0, 0, 0);
        }
      }
    }
    if (t + 1 < a.taps) store_w((t + 1) & 1);  // that buffer was last read in tap t - 1
    __syncthreads();
  }
  // epilogue: lane holds D[row][col], col = lane % 32,
  // row = 8 * (i / 4) + 4 * (lane / 32) + i % 4
  const long mbase = ((long)blockIdx.x * kWaves + wave) * 32;
#pragma unroll
  for (int j = 0; j < kMaxNTiles; ++j) {
    if (j >= ntiles) continue;
    const int co = j * 32 + (lane & 31);
    const float bias = a.bias ? a.bias[co] : 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const long mr = mbase + 8 * (i / 4) + 4 * kg + (i % 4);
      if (mr >= M) continue;
      float v = acc[j][i] + bias;
      if (a.relu) v = v > 0.0f ? v : 0.0f;
      const long o = mr * a.Cout + co;
      if (a.h) a.h[o] = (bf16)v;
      if (a.res) v += bf2f(a.res[o]);
      if (a.y32) a.y32[o] = v;
      if (a.y) a.y[o] = (bf16)v;
    }
  }
}

// ---------------------------------------------------------------- 3x3x3 conv
// conv_fwd for 27 taps: the same sums in the same order as k_no_conv_fwd
// (taps outer, channels inner, so the results are the same bits), with the
// operands' traffic cut to what the LDS can deliver beside the matrix cores.
//
// A wave owns 32 R consecutive voxels and all Cout channels. The three taps
// of one (dz, dy) read the same run of voxel rows, shifted by the dilation:
// the wave copies that run (32 R + 2 dil rows) into LDS of its own once and
// reads it three times, so x is fetched 9 times instead of 27, and no
// barrier is needed for it; the next run travels to registers while this
// one is computed. A voxel whose neighbour lies outside the grid reads a row
// of zeros instead. The weights of a tap are staged for the whole workgroup,
// one tap ahead, with one barrier per tap in its middle: with three buffers
// no wave waits for another at a tap's edge (where only two fit, a second
// barrier guards the buffer that is written). The operands of each step are
// read from LDS during the step before, also across taps.
//
// Workgroups are persistent (as many as the chip holds) and flow from one
// tile of voxels into the next: its first run and weights are fetched during
// the last taps of the tile before, and the output stores drain beside its
// first ones. XCD w mod 8 takes a contiguous eighth of the tiles, so that
// the neighbouring rows which its workgroups share sit in one L2.
//
// 96 -> 96 channels, 524288 voxels: 594 -> 298 us (440 -> 876 TFLOP/s; a
// large library product reaches 1220 here).
constexpr int kConvMaxDil = 8;  // the staged runs are sized for dilations up to this
constexpr int kConvLds = 160 * 1024;
constexpr int kCus = 256;

template <int KS, int NT, int R>
struct ConvShape {
  static constexpr int kCin = KS * 16, kCout = NT * 32;
  static constexpr int kLd = kCin + 8;      // LDS row length: 16 bytes of padding spread the rows over the banks
  static constexpr int kPieces = KS * 2;    // 16-byte pieces per row
  static constexpr int kRun = ((32 * R + 2 * kConvMaxDil) * kPieces + 63) / 64;  // pieces per lane of a staged run
  static constexpr int kRows = (kRun * 64 + kPieces - 1) / kPieces;             // LDS rows of a wave's run
  static constexpr int kW = (kCout * kPieces + 255) / 256;                       // weight pieces per thread
  static constexpr int kBufs = (kWaves * kRows + 3 * kCout + 1) * kLd * 2 <= kConvLds ? 3 : 2;
  static constexpr int kLds = (kWaves * kRows + kBufs * kCout + 1) * kLd * 2;    // bytes
};

// Exchanges the upper half-wave of a with the lower half-wave of b.
__device__ __forceinline__ void half_swap(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  bf16x2 p;
  p[0] = (bf16)lo;
  p[1] = (bf16)hi;
  return __builtin_bit_cast(uint32_t, p);
}

// Bias, ReLU, residual and stores of 32 voxels. A lane holds voxel m and, per
// group q of four values of tile j, channels j * 32 + 8 q + 4 kg + (0..3);
// the half-waves exchange groups so that a lane moves eight consecutive
// channels (16 bytes): those of group 2 p for kg = 0, of 2 p + 1 for kg = 1.
template <int NT>
__device__ __forceinline__ void conv_store(const NoConvArgs& a, int m, int M, int kg, f32x16 (&acc)[NT]) {
  constexpr int kCout = NT * 32;
  const long row = (long)(m < M ? m : 0) * kCout + 8 * kg;
  uint4 res[NT][2];
  if (a.res) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int p = 0; p < 2; ++p) res[j][p] = *reinterpret_cast<const uint4*>(a.res + row + j * 32 + 16 * p);
  }
  if (a.bias)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[j][i] += a.bias[j * 32 + 8 * (i / 4) + 4 * kg + i % 4];
  if (a.relu)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[j][i] = acc[j][i] > 0.0f ? acc[j][i] : 0.0f;
  auto store_bf16 = [&](bf16* dst) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const f32x16& v = acc[j];
        uint4 o = make_uint4(pack_bf16(v[8 * p], v[8 * p + 1]), pack_bf16(v[8 * p + 2], v[8 * p + 3]),
                             pack_bf16(v[8 * p + 4], v[8 * p + 5]), pack_bf16(v[8 * p + 6], v[8 * p + 7]));
        half_swap(o.x, o.z);
        half_swap(o.y, o.w);
        if (m < M) *reinterpret_cast<uint4*>(dst + row + j * 32 + 16 * p) = o;
      }
  };
  if (a.h) store_bf16(a.h);
  if (a.res) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        uint4 o = res[j][p];
        half_swap(o.x, o.z);
        half_swap(o.y, o.w);
        const uint32_t w[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc[j][8 * p + 2 * e] += __uint_as_float(w[e] << 16);
          acc[j][8 * p + 2 * e + 1] += __uint_as_float(w[e] & 0xFFFF0000u);
        }
      }
  }
  if (a.y32 && m < M) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[j][4 * q + e];
        *reinterpret_cast<f32x4*>(a.y32 + (long)m * kCout + j * 32 + 8 * q + 4 * kg) = v;
      }
  }
  if (a.y) store_bf16(a.y);
}

template <int KS, int NT, int R>
__global__ void __launch_bounds__(256, 1) k_no_conv27(NoConvArgs a, int tiles) {
  using S = ConvShape<KS, NT, R>;
  constexpr int Ld = S::kLd, kBufs = S::kBufs;
  __shared__ __align__(16) bf16 lds[S::kLds / 2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 31, kg = lane >> 5;
  bf16* const sx = lds + wave * S::kRows * Ld;
  bf16* const sw = lds + kWaves * S::kRows * Ld;
  bf16* const zero = sw + kBufs * S::kCout * Ld;
  const int V = a.Z * a.Y * a.X;
  const int M = a.B * V;
  const uint32_t bytes = (uint32_t)M * (S::kCin * 2);
  // this workgroup's tiles: tile0, tile0 + step, ... below tile_end
  int tile0 = blockIdx.x, step = gridDim.x, tile_end = tiles;
  if (gridDim.x % 8u == 0u) {
    const int q = blockIdx.x % 8u;
    tile0 = (int)((long)tiles * q / 8) + blockIdx.x / 8u;
    tile_end = (int)((long)tiles * (q + 1) / 8);
    step = gridDim.x / 8u;
  }
  if (tile0 >= tile_end) return;
  if (threadIdx.x < Ld / 8) {
    bf16x8 z;
#pragma unroll
    for (int e = 0; e < 8; ++e) z[e] = (bf16)0.0f;
    *reinterpret_cast<bf16x8*>(zero + threadIdx.x * 8) = z;
  }
  // coordinates of the lane's voxel in each of the wave's R voxel tiles
  int vx[R], vy[R], vz[R];
  auto locate = [&](int m0) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int m = m0 + r * 32 + col;
      int q = m % V;
      vz[r] = m < M ? q / (a.Y * a.X) : -(1 << 20);  // past the end: every neighbour is outside
      q %= a.Y * a.X;
      vy[r] = q / a.X;
      vx[r] = q % a.X;
    }
  };
  bf16x8 px[S::kRun], pw[S::kW];
  const char* const xb = reinterpret_cast<const char*>(a.x);
  // the run of (dz, dy): rows m0 + (dz Y + dy) X - dil onwards, contiguous in
  // memory; pieces outside the tensor are read from its start and never used
  auto fetch_x = [&](int m0, int g, int i0, int i1) {
    const int off = ((g / 3 - 1) * a.Y + (g % 3 - 1)) * a.dil * a.X - a.dil;
    const int start = (m0 + off) * (S::kCin * 2) + lane * 16;
#pragma unroll
    for (int i = i0; i < i1; ++i) {
      const uint32_t o = (uint32_t)(start + i * 1024);
      px[i] = *reinterpret_cast<const bf16x8*>(xb + (o < bytes ? o : 0u));
    }
  };
  auto store_x = [&]() {
#pragma unroll
    for (int i = 0; i < S::kRun; ++i) {
      const int q = i * 64 + lane;
      *reinterpret_cast<bf16x8*>(sx + (q / S::kPieces) * Ld + (q % S::kPieces) * 8) = px[i];
    }
  };
  // piece i of this thread; past the last one threads repeat earlier pieces
  auto w_piece = [&](int i) {
    constexpr int n = S::kCout * S::kPieces;
    const int q = i * 256 + threadIdx.x;
    return n < 256 ? q % n : (q < n ? q : q - 256);
  };
  auto fetch_w = [&](int t) {
    const bf16* src = a.w + (long)t * (S::kCout * S::kCin);
#pragma unroll
    for (int i = 0; i < S::kW; ++i) pw[i] = *reinterpret_cast<const bf16x8*>(src + w_piece(i) * 8);
  };
  auto store_w = [&](int buf) {
    bf16* dst = sw + buf * S::kCout * Ld;
#pragma unroll
    for (int i = 0; i < S::kW; ++i) {
      const int q = w_piece(i);
      *reinterpret_cast<bf16x8*>(dst + (q / S::kPieces) * Ld + (q % S::kPieces) * 8) = pw[i];
    }
  };
  bf16x8 xf[2][R], wf[2][NT];  // operands of this step and the next
  const bf16* xr[R];
  auto aim = [&](int g, int s) {  // the lane's voxels at tap (g, s): their rows in the run, or the zeros
    const int dz = (g / 3 - 1) * a.dil, dy = (g % 3 - 1) * a.dil;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int zz = vz[r] + dz, yy = vy[r] + dy, xx = vx[r] + (s - 1) * a.dil;
      const bool in = (unsigned)zz < (unsigned)a.Z && (unsigned)yy < (unsigned)a.Y && (unsigned)xx < (unsigned)a.X;
      xr[r] = (in ? sx + (r * 32 + col + s * a.dil) * Ld : zero) + kg * 8;
    }
  };
  auto load_step = [&](int k, int buf) {
    const bf16* wr = sw + buf * S::kCout * Ld + col * Ld + kg * 8;
#pragma unroll
    for (int r = 0; r < R; ++r) xf[k & 1][r] = *reinterpret_cast<const bf16x8*>(xr[r] + k * 16);
#pragma unroll
    for (int j = 0; j < NT; ++j) wf[k & 1][j] = *reinterpret_cast<const bf16x8*>(wr + j * 32 * Ld + k * 16);
  };
  f32x16 acc[R][NT];
  int m0 = (tile0 * kWaves + wave) * (32 * R);
  fetch_x(m0, 0, 0, S::kRun);
  fetch_w(0);
  store_x();
  store_w(0);
  fetch_w(1);
  __syncthreads();
  locate(m0);
  aim(0, 0);
  load_step(0, 0);
  int wbuf = 0;  // two buffers: the one that holds this tap's weights
  for (int tile = tile0; tile < tile_end; tile += step) {  // uniform over the workgroup
    const int m_next = tile + step < tile_end ? m0 + step * (kWaves * 32 * R) : m0;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[r][j][i] = 0.0f;
    for (int g = 0; g < 9; ++g) {
      const int gn = g < 8 ? g + 1 : 0, mn = g < 8 ? m0 : m_next;
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        const int t = 3 * g + s;
        const int cur = kBufs == 3 ? s : wbuf, nxt = kBufs == 3 ? (s + 1) % 3 : wbuf ^ 1;
        // weights of tap t + 1. Three buffers: theirs was last read in tap
        // t - 2, and every wave is past that one since tap t - 1's barrier
        if (kBufs == 2) __syncthreads();
        store_w(nxt);
        fetch_w(t < 25 ? t + 2 : t - 25);
        fetch_x(mn, gn, s * S::kRun / 3, (s + 1) * S::kRun / 3);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < KS; ++k) {
          if (k + 1 < KS) {
            load_step(k + 1, cur);
          } else {
            // the next tap's first operands; after the third tap the next run
            // takes this one's place (LDS operations of a wave stay in order:
            // only the compiler needs telling that other lanes read it)
            if (s == 2) {
              asm volatile("" ::: "memory");
              store_x();
              asm volatile("" ::: "memory");
              if (g == 8) locate(m_next);
            }
            aim(s < 2 ? g : gn, (s + 1) % 3);
            load_step(0, nxt);
          }
#pragma unroll
          for (int r = 0; r < R; ++r)
#pragma unroll
            for (int j = 0; j < NT; ++j)
              acc[r][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[k & 1][j], xf[k & 1][r], acc[r][j], 0, 0, 0);
          // one LDS read between two matrix instructions
#pragma unroll
          for (int i = 0; i < R * NT; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
          if (k == KS / 2 - 1) __syncthreads();
        }
        wbuf ^= 1;
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) conv_store<NT>(a, m0 + r * 32 + col, M, kg, acc[r]);
    m0 = m_next;
  }
}

// conv_fwd for one tap: reading x and writing y bound it. A wave keeps the
// weights in registers and walks over tiles of 32 voxels, the next tile's
// rows on their way while this one is multiplied. Same sums as k_no_conv_fwd.
// 524288 voxels: 96 -> 32 channels 50 -> 22 us, 32 -> 96 75 -> 26 us.
template <int KS, int NT>
__global__ void __launch_bounds__(256) k_no_conv1(NoConvArgs a, int tiles) {
  constexpr int kCin = KS * 16;
  const int lane = threadIdx.x & 63;
  const int col = lane & 31, kg = lane >> 5;
  const int M = a.B * a.Z * a.Y * a.X;
  const int waves = gridDim.x * kWaves;
  int tile = blockIdx.x * kWaves + (threadIdx.x >> 6);
  if (tile >= tiles) return;
  bf16x8 wf[KS][NT], xf[KS];
#pragma unroll
  for (int k = 0; k < KS; ++k)
#pragma unroll
    for (int j = 0; j < NT; ++j)
      wf[k][j] = *reinterpret_cast<const bf16x8*>(a.w + (j * 32 + col) * kCin + k * 16 + kg * 8);
  auto fetch = [&](int t) {
    const int m = min(t * 32 + col, M - 1);
#pragma unroll
    for (int k = 0; k < KS; ++k) xf[k] = *reinterpret_cast<const bf16x8*>(a.x + (long)m * kCin + k * 16 + kg * 8);
  };
  fetch(tile);
  for (; tile < tiles; tile += waves) {
    f32x16 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[j][i] = 0.0f;
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[k][j], xf[k], acc[j], 0, 0, 0);
    fetch(min(tile + waves, tiles - 1));
    conv_store<NT>(a, tile * 32 + col, M, kg, acc);
  }
}

// wb[t'][ci][co] = w[t][co][ci] with t' the mirrored tap (offset -d): the
// data gradient of conv(x, w) is conv(dy, wb).
__global__ void k_no_weight_flip(const bf16* w, bf16* wb, int taps, int Cout, int Cin) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long n = (long)taps * Cout * Cin;
  if (i >= n) return;
  int ci = (int)(i % Cin);
  int co = (int)((i / Cin) % Cout);
  int t = (int)(i / ((long)Cin * Cout));
  int tm = taps - 1 - t;  // (dz,dy,dx) -> (-dz,-dy,-dx)
  wb[((long)tm * Cin + ci) * Cout + co] = w[i];
}

struct NoBwdWArgs {
  const bf16* x;   // conv input [M][Cin]
  const bf16* dy;  // output gradient [M][Cout]
  float* part;     // [n_chunks][taps][Cout][Cin]
  int B, Z, Y, X, Cin, Cout, taps, dil, chunk;  // voxels per block
};

__global__ void __launch_bounds__(256) k_no_conv_bwd_w(NoBwdWArgs a) {
  // dy and the shifted x of kChunk voxels, transposed: [Cout][kLdk] then
  // [cin][kLdk] (dynamic LDS sized by the call's channel counts)
  extern __shared__ __align__(16) bf16 sbw[];
  bf16* const sdy = sbw;
  bf16* const sx = sbw + (long)a.Cout * kLdk;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int kg = lane >> 5;
  const int t = blockIdx.y;
  const int V = a.Z * a.Y * a.X;
  const long M = (long)a.B * V;
  const long m0 = (long)blockIdx.x * a.chunk;
  int dz, dyo, dx;
  tap_offset(t, a.taps, a.dil, dz, dyo, dx);
  const int cin = a.Cin / gridDim.z, c0 = blockIdx.z * cin;  // this workgroup's input channels
  const int tm = a.Cout >> 5, tn = cin >> 5;
  const int ntile = tm * tn;
  f32x16 acc[kMaxNTiles];
#pragma unroll
  for (int j = 0; j < kMaxNTiles; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[j][i] = 0.0f;
  const int cgy = a.Cout / 8, cgx = cin / 8;
  const long m_end = m0 + a.chunk < M ? m0 + a.chunk : M;  // this workgroup's voxels: [m0, m_end)
  for (long k0 = m0; k0 < m_end; k0 += kChunk) {
    __syncthreads();
    // stage dy and the shifted x of kChunk voxels, transposed to [c][k]:
    // lane l takes voxels 2l and 2l + 1, so a channel's two values form one
    // 32-bit LDS word and consecutive lanes write consecutive words (no bank
    // conflicts); each lane works out its voxels' sources once, and the
    // waves share out the 8-channel groups
    {
      static_assert(kChunk == 128, "two staged voxels per lane of a wavefront");
      long mm[2], src[2];  // the voxels, and the voxels x is read from for this tap (-1: outside)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        mm[h] = k0 + 2 * lane + h;
        src[h] = -1;
        if (mm[h] < m_end) {
          const int b = (int)(mm[h] / V);
          int r = (int)(mm[h] - (long)b * V);
          const int z = r / (a.Y * a.X);
          r -= z * a.Y * a.X;
          const int y = r / a.X;
          const int x = r - y * a.X;
          const int zz = z + dz, yy = y + dyo, xx = x + dx;
          if (zz >= 0 && zz < a.Z && yy >= 0 && yy < a.Y && xx >= 0 && xx < a.X)
            src[h] = (((long)b * a.Z + zz) * a.Y + yy) * a.X + xx;
        }
      }
      for (int g = wave; g < cgy + cgx; g += kWaves) {
        bf16x8 v[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[h][e] = (bf16)0.0f;
          if (g < cgy) {
            if (mm[h] < m_end) v[h] = *reinterpret_cast<const bf16x8*>(a.dy + mm[h] * a.Cout + g * 8);
          } else if (src[h] >= 0) {
            v[h] = *reinterpret_cast<const bf16x8*>(a.x + src[h] * a.Cin + c0 + (g - cgy) * 8);
          }
        }
        bf16* row = g < cgy ? sdy + (long)(g * 8) * kLdk : sx + (long)((g - cgy) * 8) * kLdk;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          bf16x2 pr;
          pr[0] = v[0][e];
          pr[1] = v[1][e];
          *reinterpret_cast<bf16x2*>(row + (long)e * kLdk + 2 * lane) = pr;
        }
      }
    }
    __syncthreads();
    // tiles assigned round-robin to the waves
#pragma unroll
    for (int j = 0; j < kMaxNTiles; ++j) {
      const int tile = wave + j * kWaves;
      if (tile >= ntile) continue;
      const int co = (tile / tn) * 32 + (lane & 31);
      const int ci = (tile % tn) * 32 + (lane & 31);
#pragma unroll
      for (int kc = 0; kc < kChunk; kc += 16) {
        bf16x8 av = *reinterpret_cast<const bf16x8*>(sdy + (long)co * kLdk + kc + kg * 8);
        bf16x8 bv = *reinterpret_cast<const bf16x8*>(sx + (long)ci * kLdk + kc + kg * 8);
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, acc[j], 0, 0, 0);
      }
    }
  }
  float* out = a.part + ((long)blockIdx.x * a.taps + t) * a.Cout * a.Cin;
#pragma unroll
  for (int j = 0; j < kMaxNTiles; ++j) {
    const int tile = wave + j * kWaves;
    if (tile >= ntile) continue;
    const int ci = c0 + (tile % tn) * 32 + (lane & 31);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int co = (tile / tn) * 32 + 8 * (i / 4) + 4 * kg + (i % 4);
      out[(long)co * a.Cin + ci] = acc[j][i];
    }
  }
}

// ------------------------------------------------- 3x3x3 weight gradient
// conv_bwd_w for 27 taps: dw[t] = dy^T x(shifted by tap t), K = voxels, so
// both operands need the voxel index innermost while memory has the channel
// innermost. Rows are staged in LDS as they come (16-byte copies) and read
// with the transposing LDS load: of 16 lanes, lane 4 r + q names the four
// channels 4 q of row r, and lane c receives channel c of rows 0..3.
//
// A workgroup takes four consecutive taps, one per wave, and a range of
// voxels: a wave keeps its tap's whole Cout x Cin product in registers, so
// dy is read once per voxel for the four taps, and the runs of x rows of the
// (at most two) (dz, dy) that they belong to serve the taps that share them.
// A row whose neighbour lies outside the grid is read as zeros: per block of
// voxels each wave makes a bit mask of its tap's inside voxels. Blocks flow
// through three LDS buffers: while one is multiplied, the next is stored and
// the one after that is on its way to registers, with one barrier per block.
//
// LDS traffic bounds it: (TM + TN) KB read per TM TN MFMAs of 32 cycles and
// wave (85 B per cycle and CU for 96 x 96 channels) and about 36 B written.
// With blocks of 32 voxels two workgroups share a CU and cover each other's
// waits; with 64 there is one. The sums and their order are those of
// k_no_conv_bwd_w (16 voxels per MFMA, in order within a chunk), so the
// results are the same bits. 96 x 96 channels, 524288 voxels: 1212 -> 310 us
// (750 TFLOP/s with the reduction); longer chunks that filled the chip evenly
// were 5% faster, but lengthen the chains of additions.
template <int TM, int TN, bool PAIR>
struct BwdShape {
  static constexpr int kCo = TM * 32, kCi = TN * 32;
  // row lengths that put four consecutive rows' 64-byte pieces in different banks (16 or 48 words modulo 64)
  static constexpr int ld(int c) { return c == 64 ? 96 : c == 128 ? 160 : c; }
  static constexpr int kLdY = ld(kCo), kLdX = ld(kCi);
  static constexpr int buf(int kb) { return kb * kLdY + 2 * (kb + 2 * kConvMaxDil) * kLdX; }
  static constexpr bool kPairs = TM * TN <= 9;  // registers for two waves per SIMD
  static constexpr int kB = !PAIR && (3 * buf(64) + kLdX) * 2 <= kConvLds ? 64 : 32;  // voxels per block
  static constexpr int kRunX = kB + 2 * kConvMaxDil;                          // rows of a run of x
  static constexpr int kBuf = buf(kB);
  static constexpr int kPY = kCo / 8, kPX = kCi / 8;                          // 16-byte pieces per row
  static constexpr int kNY = (kB * kPY + 255) / 256, kNX = (2 * kRunX * kPX + 255) / 256;  // pieces per thread
  static constexpr int kLds = (3 * kBuf + kLdX) * 2;
};

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) bf16 lds_bf16;

// rows r..r+3 of the lane's 16-lane group, transposed (see above)
__device__ __forceinline__ s16x4 lds_tr(const lds_bf16* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p);
}

template <int TM, int TN, bool PAIR>
__global__ void __launch_bounds__(256, PAIR ? 2 : 1) k_no_conv27_bwd_w(NoBwdWArgs a) {
  using S = BwdShape<TM, TN, PAIR>;
  constexpr int kB = S::kB;
  __shared__ __align__(16) bf16 lds[S::kLds / 2];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = lane >> 5;
  const int M = a.B * a.Z * a.Y * a.X;
  // XCD b mod 8 takes a contiguous share of the (chunk, tap group) list, tap
  // groups fastest: the groups of a chunk share its rows in one L2
  const unsigned T = gridDim.x, q8 = blockIdx.x % 8u;
  const unsigned item = q8 * (T / 8u) + min(q8, T % 8u) + blockIdx.x / 8u;
  const int chunk = item / 7u, t0 = (item % 7u) * 4;
  const int t = t0 + wave;  // this wave's tap (27: none, the wave only stages)
  const int b0 = chunk * (a.chunk / kB), b1 = min(b0 + a.chunk / kB, (M + kB - 1) / kB);  // the chunk's blocks
  lds_bf16* const base = (lds_bf16*)lds;
  lds_bf16* const zero = base + 3 * S::kBuf;
  if (threadIdx.x < S::kLdX) lds[3 * S::kBuf + threadIdx.x] = (bf16)0.0f;

  // staging: pieces of dy and of the two runs of x, at fixed places per thread
  const int gA = t0 / 3, gB = min((t0 + 3) / 3, 8);
  const int offA = ((gA / 3 - 1) * a.Y + (gA % 3 - 1)) * a.dil * a.X - a.dil;
  const int offB = ((gB / 3 - 1) * a.Y + (gB % 3 - 1)) * a.dil * a.X - a.dil;
  const uint32_t ybytes = (uint32_t)M * (S::kCo * 2), xbytes = (uint32_t)M * (S::kCi * 2);
  const char* const yb = reinterpret_cast<const char*>(a.dy);
  const char* const xb = reinterpret_cast<const char*>(a.x);
  bf16x8 py[S::kNY], px[S::kNX];
  auto piece = [&](int i, int n) {  // piece i of this thread; past the last one threads repeat earlier pieces
    const int q = i * 256 + threadIdx.x;
    return n < 256 ? q % n : (q < n ? q : q - 256);
  };
  auto fetch = [&](int b) {
#pragma unroll
    for (int i = 0; i < S::kNY; ++i) {
      const uint32_t o = (uint32_t)(b * kB) * (S::kCo * 2) + piece(i, kB * S::kPY) * 16;
      py[i] = *reinterpret_cast<const bf16x8*>(yb + (o < ybytes ? o : 0u));
    }
#pragma unroll
    for (int i = 0; i < S::kNX; ++i) {
      constexpr int n = S::kRunX * S::kPX;
      const int q = piece(i, 2 * n);
      const uint32_t o = (uint32_t)((b * kB + (q < n ? offA : offB)) * (S::kCi * 2) + (q < n ? q : q - n) * 16);
      px[i] = *reinterpret_cast<const bf16x8*>(xb + (o < xbytes ? o : 0u));
    }
  };
  auto store = [&](int b, lds_bf16* buf) {
#pragma unroll
    for (int i = 0; i < S::kNY; ++i) {
      const int q = piece(i, kB * S::kPY), row = q / S::kPY;
      bf16x8 v = py[i];
      if (b * kB + row >= M)  // rows past the end meet rows of zeros, but may not be infinite
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (bf16)0.0f;
      *reinterpret_cast<__attribute__((address_space(3))) bf16x8*>(buf + row * S::kLdY + (q % S::kPY) * 8) = v;
    }
#pragma unroll
    for (int i = 0; i < S::kNX; ++i) {
      const int q = piece(i, 2 * S::kRunX * S::kPX);
      *reinterpret_cast<__attribute__((address_space(3))) bf16x8*>(buf + kB * S::kLdY + (q / S::kPX) * S::kLdX +
                                                                    (q % S::kPX) * 8) = px[i];
    }
  };
  // the lane's voxel of the block (kB = 32: lanes 32.. repeat), advanced by kB voxels per block
  int dz, dyo, dx;
  tap_offset(min(t, 26), 27, a.dil, dz, dyo, dx);
  int m = b0 * kB + (lane & (kB - 1));
  int vx = m % a.X, vy = m / a.X % a.Y, vz = m / (a.X * a.Y) % a.Z;
  const int ax = kB % a.X, ay = kB / a.X % a.Y, az = kB / (a.X * a.Y) % a.Z;
  uint64_t inside = 0;  // bit v: voxel v of the block has its neighbour inside the grid
  auto look = [&]() {
    const int zz = vz + dz, yy = vy + dyo, xx = vx + dx;
    inside = __ballot(m < M && (unsigned)zz < (unsigned)a.Z && (unsigned)yy < (unsigned)a.Y &&
                      (unsigned)xx < (unsigned)a.X);
    m += kB;
    vx += ax;
    if (vx >= a.X) vx -= a.X, ++vy;
    vy += ay;
    if (vy >= a.Y) vy -= a.Y, ++vz;
    vz += az;
    if (vz >= a.Z) vz -= a.Z;
  };
  // the lane's part of a transposing read: row (kg * 8 + (lane % 16) / 4) of
  // the step's 16, channels 16 ((lane / 16) % 2) + 4 (lane % 4)
  const int rrow = kg * 8 + (lane & 15) / 4, rcol = (lane & 16) + (lane & 3) * 4;
  const int xrow = ((t / 3 == gA ? 0 : S::kRunX) + (t % 3) * a.dil);  // the tap's first row in the staged runs
  bf16x8 fy[2][TM], fx[2][TN];
  auto load_step = [&](int k, const lds_bf16* buf) {
    const lds_bf16* y = buf + (k * 16 + rrow) * S::kLdY + rcol;
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      const s16x4 lo = lds_tr(y + j * 32), hi = lds_tr(y + 4 * S::kLdY + j * 32);
      fy[k & 1][j] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
    const lds_bf16* x = buf + kB * S::kLdY + (xrow + k * 16 + rrow) * S::kLdX;
    const uint32_t bits = (uint32_t)(inside >> (k * 16)) >> rrow;
    const lds_bf16* x0 = ((bits & 1u) ? x : zero) + rcol;
    const lds_bf16* x1 = ((bits & 16u) ? x + 4 * S::kLdX : zero) + rcol;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const s16x4 lo = lds_tr(x0 + j * 32), hi = lds_tr(x1 + j * 32);
      fx[k & 1][j] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  };
  lds_bf16 *cur = base, *nxt = base + S::kBuf, *far = base + 2 * S::kBuf;
  fetch(b0);
  store(b0, cur);
  fetch(b0 + 1 < b1 ? b0 + 1 : b0);
  __syncthreads();
  look();
  load_step(0, cur);
  constexpr int kSteps = kB / 16;
  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  for (int b = b0; b < b1; ++b) {  // uniform over the workgroup
    // block b + 1 goes to the buffer last read for block b - 2, which every
    // wave is past since block b - 1's barrier
    store(b + 1 < b1 ? b + 1 : b, nxt);
    fetch(b + 2 < b1 ? b + 2 : b);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < kSteps; ++k) {
      if (k + 1 < kSteps) {
        load_step(k + 1, cur);
      } else {
        look();
        load_step(0, nxt);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fy[k & 1][i], fx[k & 1][j], acc[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < TM * TN; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (k == kSteps / 2 - 1) __syncthreads();
    }
    lds_bf16* const p = cur;
    cur = nxt;
    nxt = far;
    far = p;
  }
  if (t >= 27) return;
  float* const out = a.part + ((long)chunk * 27 + t) * (S::kCo * S::kCi) + 4 * kg * S::kCi + (lane & 31);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) out[(i * 32 + 8 * (e / 4) + e % 4) * S::kCi + j * 32] = acc[i][j][e];
}

// out[i] (+)= sum over chunks of part[c][i], in the chunks' order: one value
// per thread, the loads of kRedLoads chunks in flight.
constexpr int kRedLoads = 16;

__global__ void __launch_bounds__(256) k_no_reduce_partials(const float* part, long n, int chunks, float* out,
                                                            int accumulate) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float s = 0.0f;
  int c = 0;
  for (; c + kRedLoads <= chunks; c += kRedLoads) {
    float v[kRedLoads];
#pragma unroll
    for (int k = 0; k < kRedLoads; ++k) v[k] = part[(c + k) * n + i];
#pragma unroll
    for (int k = 0; k < kRedLoads; ++k) s += v[k];
  }
  for (; c < chunks; ++c) s += part[c * n + i];
  out[i] = accumulate ? out[i] + s : s;
}

// db[co] partial sums: part[b][co] sums voxels [b * kBiasChunk, (b + 1) *
// kBiasChunk). A thread takes eight channels (16 bytes) and every eighth
// voxel, and the eight voxel lanes are added in a fixed order; a workgroup of
// 256 threads takes 256 / Cout chunks. FUSE: dz = dy * (h > 0) is formed and
// stored on the way, and its sums taken. 524288 x 96: 69 -> 20 us for the sums
// alone; with the ReLU 54 us in place of 136 + 69.
constexpr int kBiasChunk = 512;

template <bool FUSE, bool VEC>
__global__ void __launch_bounds__(256) k_no_bias_grad(const bf16* dy, const bf16* h, bf16* dz, long M, int Cout,
                                                      float* part) {
  __shared__ float red[8][256];
  const int t = threadIdx.x, pieces = Cout / 8;
  const int sub = t / Cout, vl = t % Cout / pieces, pc = t % pieces;  // chunk of the workgroup, voxel lane, channels 8 pc..
  const int per = 256 / Cout;
  const long chunk = (long)blockIdx.x * per + sub;
  const long m0 = chunk * kBiasChunk;
  if (sub < per) {
    float s[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) s[e] = 0.0f;
    auto load = [](const bf16* p) {
      bf16x8 v;
      if (VEC) {
        v = *reinterpret_cast<const bf16x8*>(p);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = p[e];
      }
      return v;
    };
    auto batch = [&](int i, auto whole) {  // voxels i, i + 8, ... i + 56; whole: all of them exist
      bf16x8 v[8], act[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {  // past the end: the last voxel's values, not used
        const long m = m0 + i + 8 * k;
        const long at = (whole() ? m : min(m, M - 1)) * Cout + pc * 8;
        v[k] = load(dy + at);
        if (FUSE) act[k] = load(h + at);
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const long m = m0 + i + 8 * k;
        const bool in = whole() || m < M;
        if (FUSE) {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[k][e] = bf2f(act[k][e]) > 0.0f ? v[k][e] : (bf16)0.0f;
          bf16* const o = dz + m * Cout + pc * 8;
          if (VEC) {
            if (in) *reinterpret_cast<bf16x8*>(o) = v[k];
          } else if (in) {
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = v[k][e];
          }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] += in ? bf2f(v[k][e]) : 0.0f;  // (adding zero leaves every sum as it is)
      }
    };
    // one form per wave: with 32 channels a wave has two chunks, and a ragged
    // second one would have it run both (1000 voxels: 17 -> 11 us)
    if (__all(m0 + kBiasChunk <= M)) {
      for (int i = vl; i < kBiasChunk; i += 64) batch(i, std::true_type{});
    } else {
      for (int i = vl; i < kBiasChunk && m0 + i < M; i += 64) batch(i, std::false_type{});
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) red[vl][sub * Cout + pc * 8 + e] = s[e];
  }
  __syncthreads();
  if (sub < per && m0 < M) {
    float s = 0.0f;
    for (int v = 0; v < 8; ++v) s += red[v][t];
    part[chunk * Cout + t % Cout] = s;
  }
}

// out[i] (+)= sum over c of part[c][i] for many partial rows: a workgroup
// per output, the rows split over its threads and added in a fixed order.
__global__ void __launch_bounds__(256) k_no_reduce_rows(const float* part, int n, int rows, float* out,
                                                        int accumulate) {
  __shared__ float red[256];
  const int i = blockIdx.x, t = threadIdx.x;
  float s = 0.0f;
  for (int c = t; c < rows; c += 256) s += part[(long)c * n + i];
  red[t] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (t < h) red[t] += red[t + h];
    __syncthreads();
  }
  if (t == 0) out[i] = accumulate ? out[i] + red[0] : red[0];
}

// dz = dy * (h > 0)  (ReLU backward through the stored activation), eight
// values per thread (16 bytes) where the arrays are 16-byte aligned (50M
// values: 136 -> 48 us; one value per thread keeps too few bytes in flight)
template <int W>
__global__ void k_no_relu_bwd(const bf16* dy, const bf16* h, bf16* dz, long n) {
  const long i = ((long)blockIdx.x * blockDim.x + threadIdx.x) * W;
  if (i >= n) return;
  if (W == 8 && i + W <= n) {
    bf16x8 g = *reinterpret_cast<const bf16x8*>(dy + i);
    const bf16x8 a = *reinterpret_cast<const bf16x8*>(h + i);
#pragma unroll
    for (int e = 0; e < 8; ++e) g[e] = bf2f(a[e]) > 0.0f ? g[e] : (bf16)0.0f;
    *reinterpret_cast<bf16x8*>(dz + i) = g;
    return;
  }
  for (long q = i; q < n && q < i + W; ++q) dz[q] = bf2f(h[q]) > 0.0f ? dy[q] : (bf16)0.0f;
}

// c = a + b
__global__ void k_no_add(const bf16* a, const bf16* b, bf16* c, long n) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  c[i] = (bf16)(bf2f(a[i]) + bf2f(b[i]));
}

// Masked mean-squared error of pred [M][C] (FP32, only the first Cf channels
// are fields) against target [M][Cf]; dpred = 2 (pred - target) mask / count,
// written as BF16 [M][C] (zero in the padding channels); per-block loss sums.
// A wave takes the 256 elements of a block, four per lane; only the field
// channels of pred are read. 524288 x 32: 49 -> 26 us (64-bit divisions per
// element before).
__global__ void __launch_bounds__(256) k_no_mse(const float* pred, const float* target, const float* mask, long M,
                                                int C, int Cf, float inv_count, bf16* dpred, float* loss_part) {
  const long n = M * C;
  const long block = (long)blockIdx.x * 4 + threadIdx.x / 64;
  const long i0 = block * 256 + (threadIdx.x & 63) * 4;
  if (block * 256 >= n) return;
  float l = 0.0f;
  long m = i0 < (1L << 32) ? (long)((uint32_t)i0 / (uint32_t)C) : i0 / C;
  int c = (int)(i0 - m * C);
  bf16x4 out;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    float g = 0.0f;
    if (i0 + k < n && c < Cf) {
      const float w = mask ? mask[m] : 1.0f;
      const float d = (pred[i0 + k] - target[m * Cf + c]) * w;
      l += d * d * inv_count;
      g = 2.0f * d * inv_count;
    }
    out[k] = (bf16)g;
    if (++c == C) c = 0, ++m;
  }
  if (i0 + 4 <= n && (reinterpret_cast<uintptr_t>(dpred) & 7u) == 0u)
    *reinterpret_cast<bf16x4*>(dpred + i0) = out;
  else
    for (int k = 0; k < 4 && i0 + k < n; ++k) dpred[i0 + k] = out[k];
  for (int off = 32; off > 0; off >>= 1) l += __shfl_down(l, off);
  if ((threadIdx.x & 63) == 0) loss_part[block] = l;
}

// Adam on FP32 master weights, BF16 copy refreshed.
__global__ void k_no_adam(float* w, const float* g, float* m1, float* m2, bf16* wbf, long n, float lr, float b1,
                          float b2, float eps, float c1, float c2, float wd) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float gi = g[i] + wd * w[i];
  float a = b1 * m1[i] + (1.0f - b1) * gi;
  float b = b2 * m2[i] + (1.0f - b2) * gi * gi;
  m1[i] = a;
  m2[i] = b;
  float upd = (a / c1) / (sqrtf(b / c2) + eps);
  float nw = w[i] - lr * upd;
  w[i] = nw;
  if (wbf) wbf[i] = (bf16)nw;
}

__global__ void k_no_f32_to_bf16(const float* a, bf16* b, long n) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = (bf16)a[i];
}

// Per-voxel input features of the operator: x, y, z in [-1, 1], signed
// distance to the sphere surface in units of the box height, and the five
// normalised freestream/body parameters broadcast (p[b][5]); channels
// 9..C-1 are zero. sphere[b] = {cx, cy, cz, r} in metres, box = {xmin, ymin,
// zmin, xmax, ymax, zmax}.
__global__ void k_no_inputs(const float* p, const float* sphere, const float* box, int B, int Z, int Y, int X, int C,
                            bf16* out) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long V = (long)Z * Y * X;
  if (i >= (long)B * V) return;
  int b = (int)(i / V);
  int r = (int)(i - (long)b * V);
  int z = r / (Y * X);
  r -= z * Y * X;
  int y = r / X;
  int x = r - y * X;
  float fx = (x + 0.5f) / X, fy = (y + 0.5f) / Y, fz = (z + 0.5f) / Z;
  float px = box[0] + fx * (box[3] - box[0]);
  float py = box[1] + fy * (box[4] - box[1]);
  float pz = box[2] + fz * (box[5] - box[2]);
  const float* s = sphere + 4 * b;
  float dx = px - s[0], dy = py - s[1], dz = pz - s[2];
  float sd = (sqrtf(dx * dx + dy * dy + dz * dz) - s[3]) / (box[4] - box[1]);
  bf16* o = out + i * C;
  float f[9] = {2.0f * fx - 1.0f, 2.0f * fy - 1.0f, 2.0f * fz - 1.0f, sd, p[5 * b], p[5 * b + 1], p[5 * b + 2],
                p[5 * b + 3], p[5 * b + 4]};
  for (int c = 0; c < C; ++c) o[c] = (bf16)(c < 9 ? f[c] : 0.0f);
}

// ------------------------------------------------------------------ C ABI
static inline unsigned nb(long n, int t) { return (unsigned)((n + t - 1) / t); }
static inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0u; }
#define NO_EMPTY(n) \
  if ((n) <= 0) return 0

namespace {

template <int KS, int NT, int R>
void conv27_launch(const NoConvArgs& a, long M, hipStream_t st) {
  // persistent workgroups: one resident set
  static const int per_cu = [] {
    int n = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_no_conv27<KS, NT, R>, 256, 0);
    return e == hipSuccess && n > 0 ? n : 1;
  }();
  const unsigned tiles = nb(M, 32 * R * kWaves);
  const unsigned grid = std::min(tiles, (unsigned)(kCus * per_cu));
  hipLaunchKernelGGL((k_no_conv27<KS, NT, R>), dim3(grid), dim3(256), 0, st, a, (int)tiles);
}

template <int KS, int NT>
void conv27_r(const NoConvArgs& a, long M, hipStream_t st) {
  // Two voxel tiles per wave; one where that leaves half the CUs without a
  // workgroup (M <= 32768: 1008 voxels of 128 -> 128 channels 35 us against
  // 56). Three or four per wave need fewer LDS reads per matrix instruction,
  // but their registers cost more than that gains (96 -> 96 channels, 524288
  // voxels: 304 us with two, 326 with three, 505 with four, which spills).
  if (M <= kCus / 2 * 64 * kWaves) return conv27_launch<KS, NT, 1>(a, M, st);
  return conv27_launch<KS, NT, 2>(a, M, st);
}

template <int KS>
void conv27_n(const NoConvArgs& a, long M, hipStream_t st) {
  switch (a.Cout / 32) {
    case 1: return conv27_r<KS, 1>(a, M, st);
    case 2: return conv27_r<KS, 2>(a, M, st);
    case 3: return conv27_r<KS, 3>(a, M, st);
    default: return conv27_r<KS, 4>(a, M, st);
  }
}

template <int KS>
void conv1_n(const NoConvArgs& a, long M, hipStream_t st) {
  const unsigned tiles = nb(M, 32);
  const dim3 grid(std::min(nb(tiles, kWaves), 4u * kCus));  // four workgroups per CU
  switch (a.Cout / 32) {
    case 1: hipLaunchKernelGGL((k_no_conv1<KS, 1>), grid, dim3(256), 0, st, a, (int)tiles); break;
    case 2: hipLaunchKernelGGL((k_no_conv1<KS, 2>), grid, dim3(256), 0, st, a, (int)tiles); break;
    case 3: hipLaunchKernelGGL((k_no_conv1<KS, 3>), grid, dim3(256), 0, st, a, (int)tiles); break;
    default: hipLaunchKernelGGL((k_no_conv1<KS, 4>), grid, dim3(256), 0, st, a, (int)tiles); break;
  }
}

// The staged kernels are made for whole groups of channels and a grid; calls
// without (no output channel, negative extents) stay with the general ones.
bool conv_sizes(int B, int Z, int Y, int X, int Cin, int Cout) {
  return B > 0 && Z > 0 && Y > 0 && X > 0 && Cin > 0 && Cout > 0;
}

// The staged kernels move 16 bytes at a time; arrays that start elsewhere
// (views at odd offsets) go to the general ones.
bool conv_aligned(const NoConvArgs& a) {
  return aligned16(a.x) && aligned16(a.w) && aligned16(a.res) && aligned16(a.y) && aligned16(a.y32) && aligned16(a.h);
}

bool conv1(const NoConvArgs& a, long M, hipStream_t st) {
  if (a.taps != 1 || M >= (1L << 31) - 64 || !conv_sizes(a.B, a.Z, a.Y, a.X, a.Cin, a.Cout) || !conv_aligned(a))
    return false;
  switch (a.Cin) {
    case 32: conv1_n<2>(a, M, st); return true;
    case 64: conv1_n<4>(a, M, st); return true;
    case 96: conv1_n<6>(a, M, st); return true;
    case 128: conv1_n<8>(a, M, st); return true;
    default: return false;
  }
}

// The staged kernel for the shapes that it covers; false: not covered.
bool conv27(const NoConvArgs& a, long M, hipStream_t st) {
  // byte offsets into x, from a run's start before the first voxel to past the last workgroup's voxels, fit an int
  const long reach = M + 1024 + (long)kConvMaxDil * (a.Y + 2) * a.X;
  if (a.taps != 27 || a.dil < 0 || a.dil > kConvMaxDil || reach * a.Cin * 2 >= (1L << 31) ||
      !conv_sizes(a.B, a.Z, a.Y, a.X, a.Cin, a.Cout) || !conv_aligned(a))
    return false;
  switch (a.Cin) {
    case 32: conv27_n<2>(a, M, st); return true;
    case 64: conv27_n<4>(a, M, st); return true;
    case 96: conv27_n<6>(a, M, st); return true;
    case 128: conv27_n<8>(a, M, st); return true;
    default: return false;
  }
}

// Items are (chunk, tap group); two workgroups per CU where there are items
// for both and the registers allow it.
template <int TM, int TN>
void conv27_bwd_w_launch(const NoBwdWArgs& a, int chunks, hipStream_t st) {
  if constexpr (BwdShape<TM, TN, true>::kPairs) {
    if (chunks * 7 > kCus) {
      hipLaunchKernelGGL((k_no_conv27_bwd_w<TM, TN, true>), dim3(chunks * 7), dim3(256), 0, st, a);
      return;
    }
  }
  hipLaunchKernelGGL((k_no_conv27_bwd_w<TM, TN, false>), dim3(chunks * 7), dim3(256), 0, st, a);
}

template <int TM>
void conv27_bwd_w_n(const NoBwdWArgs& a, int chunks, hipStream_t st) {
  switch (a.Cin / 32) {
    case 1: return conv27_bwd_w_launch<TM, 1>(a, chunks, st);
    case 2: return conv27_bwd_w_launch<TM, 2>(a, chunks, st);
    case 3: return conv27_bwd_w_launch<TM, 3>(a, chunks, st);
    default: return conv27_bwd_w_launch<TM, 4>(a, chunks, st);
  }
}

// The staged weight gradient where it applies; false: not covered.
bool conv27_bwd_w(const NoBwdWArgs& a, long M, int chunks, hipStream_t st) {
  const long reach = M + 1024 + (long)kConvMaxDil * (a.Y + 2) * a.X;
  if (a.taps != 27 || a.dil < 0 || a.dil > kConvMaxDil || reach * std::max(a.Cin, a.Cout) * 2 >= (1L << 31) ||
      !conv_sizes(a.B, a.Z, a.Y, a.X, a.Cin, a.Cout) || !aligned16(a.x) || !aligned16(a.dy))
    return false;
  switch (a.Cout / 32) {
    case 1: conv27_bwd_w_n<1>(a, chunks, st); return true;
    case 2: conv27_bwd_w_n<2>(a, chunks, st); return true;
    case 3: conv27_bwd_w_n<3>(a, chunks, st); return true;
    default: conv27_bwd_w_n<4>(a, chunks, st); return true;
  }
}

template <bool FUSE>
int bias_grad(const void* dy, const void* h, void* dz, long M, int Cout, float* db, float* part, long part_floats,
              int accumulate, hipStream_t st) {
  NO_EMPTY(M);
  if (Cout % 32 || Cout <= 0 || Cout > kMaxC) return -1;
  const int chunks = (int)nb(M, kBiasChunk);
  if ((long)chunks * Cout > part_floats) return -5;
  const dim3 grid(nb(chunks, 256 / Cout));
  if (aligned16(dy) && aligned16(h) && aligned16(dz))
    hipLaunchKernelGGL((k_no_bias_grad<FUSE, true>), grid, dim3(256), 0, st, (const bf16*)dy, (const bf16*)h, (bf16*)dz,
                       M, Cout, part);
  else
    hipLaunchKernelGGL((k_no_bias_grad<FUSE, false>), grid, dim3(256), 0, st, (const bf16*)dy, (const bf16*)h,
                       (bf16*)dz, M, Cout, part);
  hipLaunchKernelGGL(k_no_reduce_rows, dim3(Cout), dim3(256), 0, st, part, Cout, chunks, db, accumulate);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace

extern "C" {

int dsmc_no_conv_fwd(const void* x, const void* w, const float* bias, const void* res, void* y, float* y32,
                     void* h, int B, int Z, int Y, int X, int Cin, int Cout, int taps, int dil, int relu,
                     void* stream) {
  if (Cin % 16 || Cin > kMaxC || Cout % 32 || Cout > 32 * kMaxNTiles || (taps != 1 && taps != 27) || B <= 0)
    return -1;
  NoConvArgs a{(const bf16*)x, (const bf16*)w, bias, (const bf16*)res, (bf16*)y, y32, (bf16*)h,
               B, Z, Y, X, Cin, Cout, taps, dil, relu};
  long M = (long)B * Z * Y * X;
  NO_EMPTY(M);
  if (conv27(a, M, (hipStream_t)stream) || conv1(a, M, (hipStream_t)stream)) return hipGetLastError() == hipSuccess ? 0 : -3;
  const size_t lds = 2ull * Cout * (Cin + 8) * sizeof(bf16);  // two taps of weights
  hipLaunchKernelGGL(k_no_conv_fwd, dim3(nb(M, 32 * kWaves)), dim3(256), lds, (hipStream_t)stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int dsmc_no_weight_flip(const void* w, void* wb, int taps, int Cout, int Cin, void* stream) {
  long n = (long)taps * Cout * Cin;
  NO_EMPTY(n);
  hipLaunchKernelGGL(k_no_weight_flip, dim3(nb(n, 256)), dim3(256), 0, (hipStream_t)stream, (const bf16*)w,
                     (bf16*)wb, taps, Cout, Cin);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int dsmc_no_conv_bwd_w(const void* x, const void* dy, float* dw, float* part, long part_floats, int B, int Z,
                       int Y, int X, int Cin, int Cout, int taps, int dil, int chunk, int accumulate, void* stream) {
  if (Cin % 32 || Cout % 32 || Cin > kMaxC || Cout > kMaxC || chunk <= 0 || chunk % 64 || (taps != 1 && taps != 27))
    return -1;
  if ((Cout / 32) * (Cin / 32) > kWaves * kMaxNTiles) return -1;
  long M = (long)B * Z * Y * X;
  NO_EMPTY(M);
  if (Cin <= 0 || Cout <= 0) return -1;
  int chunks = (int)nb(M, chunk);
  long n = (long)taps * Cout * Cin;
  if ((long)chunks * n > part_floats) return -5;
  NoBwdWArgs a{(const bf16*)x, (const bf16*)dy, part, B, Z, Y, X, Cin, Cout, taps, dil, chunk};
  if (!conv27_bwd_w(a, M, chunks, (hipStream_t)stream)) {
    // One tap is too few workgroups for the chip, each waiting for its own
    // loads: up to 1024 of them, one per 32 input channels. The sums stay as
    // they are (96 -> 32 channels, 524288 voxels: 140 -> 101 us).
    const int parts = taps == 1 && chunks * (Cin / 32) <= 1024 ? Cin / 32 : 1;
    const size_t lds = (size_t)(Cout + Cin / parts) * kLdk * sizeof(bf16);
    hipLaunchKernelGGL(k_no_conv_bwd_w, dim3(chunks, taps, parts), dim3(256), lds, (hipStream_t)stream, a);
  }
  hipLaunchKernelGGL(k_no_reduce_partials, dim3(nb(n, 256)), dim3(256), 0, (hipStream_t)stream, part, n, chunks,
                     dw, accumulate);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int dsmc_no_bias_grad(const void* dy, long M, int Cout, float* db, float* part, long part_floats, int accumulate,
                      void* stream) {
  return bias_grad<false>(dy, nullptr, nullptr, M, Cout, db, part, part_floats, accumulate, (hipStream_t)stream);
}

int dsmc_no_relu_bias_bwd(const void* dy, const void* h, void* dz, long M, int Cout, float* db, float* part,
                          long part_floats, int accumulate, void* stream) {
  return bias_grad<true>(dy, h, dz, M, Cout, db, part, part_floats, accumulate, (hipStream_t)stream);
}

int dsmc_no_relu_bwd(const void* dy, const void* h, void* dz, long n, void* stream) {
  NO_EMPTY(n);
  if (aligned16(dy) && aligned16(h) && aligned16(dz))
    hipLaunchKernelGGL(k_no_relu_bwd<8>, dim3(nb(n, 256 * 8)), dim3(256), 0, (hipStream_t)stream, (const bf16*)dy,
                       (const bf16*)h, (bf16*)dz, n);
  else
    hipLaunchKernelGGL(k_no_relu_bwd<1>, dim3(nb(n, 256)), dim3(256), 0, (hipStream_t)stream, (const bf16*)dy,
                       (const bf16*)h, (bf16*)dz, n);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int dsmc_no_add(const void* a, const void* b, void* c, long n, void* stream) {
  NO_EMPTY(n);
  hipLaunchKernelGGL(k_no_add, dim3(nb(n, 256)), dim3(256), 0, (hipStream_t)stream, (const bf16*)a,
                     (const bf16*)b, (bf16*)c, n);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int dsmc_no_mse(const float* pred, const float* target, const float* mask, long M, int C, int Cf, float inv_count,
                void* dpred, float* loss_part, void* stream) {
  NO_EMPTY(M * C);
  hipLaunchKernelGGL(k_no_mse, dim3(nb(M * C, 1024)), dim3(256), 0, (hipStream_t)stream, pred, target, mask, M, C,
                     Cf, inv_count, (bf16*)dpred, loss_part);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int dsmc_no_adam(float* w, const float* g, float* m1, float* m2, void* wbf, long n, float lr, float b1, float b2,
                 float eps, float c1, float c2, float wd, void* stream) {
  NO_EMPTY(n);
  hipLaunchKernelGGL(k_no_adam, dim3(nb(n, 256)), dim3(256), 0, (hipStream_t)stream, w, g, m1, m2, (bf16*)wbf, n,
                     lr, b1, b2, eps, c1, c2, wd);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int dsmc_no_f32_to_bf16(const float* a, void* b, long n, void* stream) {
  NO_EMPTY(n);
  hipLaunchKernelGGL(k_no_f32_to_bf16, dim3(nb(n, 256)), dim3(256), 0, (hipStream_t)stream, a, (bf16*)b, n);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int dsmc_no_inputs(const float* p, const float* sphere, const float* box, int B, int Z, int Y, int X, int C,
                   void* out, void* stream) {
  if (C < 9) return -1;
  long n = (long)B * Z * Y * X;
  NO_EMPTY(n);
  hipLaunchKernelGGL(k_no_inputs, dim3(nb(n, 256)), dim3(256), 0, (hipStream_t)stream, p, sphere, box, B, Z, Y, X,
                     C, (bf16*)out);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // extern "C"
