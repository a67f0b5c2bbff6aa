// Weight-streaming matrix products of decode batches for gfx950:
// y[M, N] = x[M, K] W[N, K]^T, M <= 64 (128 for partial sums), bf16 with fp32
// sums.
//
// What bounds it: every weight is used once, so the time is that of streaming
// W from HBM, and a read-only stream only reaches the memory's rate if each
// load instruction asks for whole 128-byte lines and enough of them are in
// flight (measured on 235 MB that no cache holds: 16 rows x 64 bytes per
// instruction 6.0 TB/s, 8 rows x 128 bytes without temporal hint 6.6).
//   - W goes from memory to the registers that the matrix core reads, without
//     LDS in between. 8 rows x 128 bytes are not the 16 rows x 64 bytes of an A
//     operand; taken as one all the same, its rows 0..7 are the W rows' first
//     half lines and its rows 8..15 their second halves. Two products, one with
//     x's first half line and one with its second, therefore hold what is
//     wanted in their rows 0..7 and 8..15; the other halves are left over. The
//     matrix cores have that to spare (31% busy at M = 64), and exchanging
//     registers between lanes instead would cost vector instructions per byte.
//   - x passes through LDS, a slice of 256 k at a time for the 128 rows of W of
//     a workgroup's 8 waves (read by every wave from L2 instead it took longer
//     than W: 106 us where this takes 50). The next slice of x and W is asked
//     for before the present one is multiplied, x first, so that storing x
//     leaves W in flight across the barrier.
//   - matrices of few rows split the reduction over workgroups until the chip
//     is full; whoever reads the result next adds the partial sums up.
// Measured, M = 8 / 32 / 64, weights from HBM, in us (hipBLASLt beside it):
//   28672 x 4096   44 / 45 / 52   (62 / 51 / 52), with the activation
//   4096 x 14336   20 / 22 / 27   (28 / 32 / 40)
//   6144 x 4096    11 / 13 / 16   (21 / 19 / 19)
//   4096 x 4096     8 /  9 / 11   (21 / 19 / 19)
//   8192 x 28672   72 / 76 / 93   (92 / 102 / 140)
//   32000 x 8192   92 / 99 / 104  (126 / 138 / 116)
// The ends: bf16 rows; silu(gate) up of W's two halves, both in fp32; fp32
// partial sums for the residual norm or the rotary embedding that follows.
//
// Fragment maps (pinned by tests/test_ops_gpu.py), v_mfma_f32_16x16x32_bf16:
//   A[16x32k]: lane l -> row = l&15, k = 8*(l>>4) + j   (j = 0..7)
//   B[32kx16]: lane l -> col = l&15, k = 8*(l>>4) + j
//   C/D:       lane l -> col = l&15, row = 4*(l>>4) + r (r = 0..3)
#include "common.h"
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

namespace kukeon {
namespace {

typedef __attribute__((__vector_size__(8 * sizeof(short)))) short frag_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float acc_t;
typedef __attribute__((__vector_size__(4 * sizeof(unsigned int)))) unsigned int
    word4_t;

enum End { ROWS, SILU, SUMS };

// MT: 16-row tiles of x; RT: tiles of W per wave, of 8 rows as above or, with
// HALF, of 16 rows read half a line at a time; NW: waves; KS: k per slice; OCC:
// waves per SIMD that the registers have to allow
template <int MT, int RT, int NW, int KS, int OCC, int END, bool HALF>
__global__ __launch_bounds__(NW * WAVE, OCC) void stream_gemm_kernel(
    unsigned short* __restrict__ out,      // [M, N] bf16; SILU: [M, N / 2]
    float* __restrict__ sums,              // [splits, M, N] (SUMS)
    const unsigned short* __restrict__ x,  // [M, K]
    const unsigned short* __restrict__ w,  // [N, K]
    int M, int N, long K) {
  constexpr int NT = NW * WAVE;
  constexpr int ST = KS / 64;                  // steps per slice
  constexpr int TR = HALF ? 16 : 8;            // rows of W per tile
  constexpr int LW = HALF ? 2 : 1;             // loads per tile and step
  constexpr int XP = MT * 16 * KS / 8;         // 16-byte pieces of x per slice
  constexpr int XC = (XP + NT - 1) / NT;       // of them per thread
  __shared__ __align__(16) unsigned short xbuf[2][MT * 16 * KS];
  const int wid = threadIdx.x / WAVE;
  const int lane = threadIdx.x & (WAVE - 1);
  const int g = lane >> 4, c16 = lane & 15;
  const int slices = (int)(K / KS);

  // with SILU the first half of a wave's tiles are gate rows, the others the
  // up rows of the same outputs
  const int first =
      (blockIdx.x * NW + wid) * (END == SILU ? RT * TR / 2 : RT * TR);
  const unsigned short* wp[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int tile_row = END != SILU ? first + i * TR
                         : i < RT / 2 ? first + i * TR
                                      : N / 2 + first + (i - RT / 2) * TR;
    wp[i] = w + (long)(tile_row + (lane & (TR - 1))) * K +
            (HALF ? g : g + ((lane >> 3) & 1) * 4) * 8;
  }

  acc_t lo[RT][MT], hi[RT][MT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int m = 0; m < MT; ++m) lo[i][m] = hi[i][m] = acc_t{};

  word4_t xr[XC];
  auto load_x = [&](int s) {
#pragma unroll
    for (int i = 0; i < XC; ++i) {
      const int p = threadIdx.x + i * NT;
      if (XP % NT && p >= XP) break;
      const int row = p / (KS / 8);
      xr[i] = *reinterpret_cast<const word4_t*>(
          x + (long)min(M - 1, row) * K + (long)s * KS + (p % (KS / 8)) * 8);
    }
  };
  auto store_x = [&](int b) {
#pragma unroll
    for (int i = 0; i < XC; ++i) {
      const int p = threadIdx.x + i * NT;
      if (XP % NT && p >= XP) break;
      const int row = p / (KS / 8);
      *reinterpret_cast<word4_t*>(
          reinterpret_cast<char*>(xbuf[b]) + row * KS * 2 +
          (((p % (KS / 8)) * 16) ^ ((row & 15) << 4))) = xr[i];
    }
  };
  auto load_w = [&](int s, word4_t (&wv)[ST][RT][LW]) {
#pragma unroll
    for (int u = 0; u < ST; ++u)
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int h = 0; h < LW; ++h) {
          const auto* p = reinterpret_cast<const word4_t*>(
              wp[i] + (long)s * KS + u * 64 + h * 32);
          // half a line is better off kept for its other half
          wv[u][i][h] = HALF ? *p : __builtin_nontemporal_load(p);
        }
  };
  auto multiply = [&](int b, const word4_t (&wv)[ST][RT][LW]) {
#pragma unroll
    for (int u = 0; u < ST; ++u)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const char* row =
            reinterpret_cast<const char*>(xbuf[b]) + (m * 16 + c16) * KS * 2;
        const frag_t x0 = *reinterpret_cast<const frag_t*>(
            row + ((u * 128 + g * 16) ^ (c16 << 4)));
        const frag_t x1 = *reinterpret_cast<const frag_t*>(
            row + ((u * 128 + 64 + g * 16) ^ (c16 << 4)));
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          auto& other = HALF ? lo[i][m] : hi[i][m];
          lo[i][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(frag_t, wv[u][i][0]), x0, lo[i][m], 0, 0, 0);
          other = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(frag_t, wv[u][i][LW - 1]), x1, other, 0, 0,
              0);
        }
      }
  };

  const int step = gridDim.y;
  int s = blockIdx.y;
  word4_t wa[ST][RT][LW], wb[ST][RT][LW];
  load_x(s);
  load_w(s, wa);
  store_x(0);
  __syncthreads();
  // x of the next slice is asked for ahead of its weights, so that waiting
  // for it leaves the weights in flight
  for (;;) {
    const int n1 = s + step;
    if (n1 < slices) { load_x(n1); load_w(n1, wb); }
    multiply(0, wa);
    if (n1 >= slices) break;
    store_x(1);
    __syncthreads();
    s = n1 + step;
    if (s < slices) { load_x(s); load_w(s, wa); }
    multiply(1, wb);
    if (s >= slices) break;
    store_x(0);
    __syncthreads();
  }

  // With HALF a lane holds rows 4 * g + r of tile i. Otherwise W row
  // 4 * (g & 1) + r: lanes below 32 hold its first half lines' sum, lanes above
  // its second half lines'
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    float v[RT][4];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[i][r] = HALF || g < 2 ? lo[i][m][r] : hi[i][m][r];
        if (!HALF) v[i][r] += __shfl_xor(v[i][r], 32, WAVE);
      }
    const int row = m * 16 + c16;
    if ((!HALF && g >= 2) || row >= M) continue;
#pragma unroll
    for (int i = 0; i < (END == SILU ? RT / 2 : RT); ++i) {
      const int n = first + i * TR + g * 4;
      if (END == SUMS) {
        *reinterpret_cast<float4*>(
            sums + ((long)blockIdx.y * M + row) * N + n) =
            float4{v[i][0], v[i][1], v[i][2], v[i][3]};
        continue;
      }
      if (END == SILU)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[i][r] = v[i][r] / (1.f + __expf(-v[i][r])) * v[RT / 2 + i][r];
      *reinterpret_cast<uint2*>(out + row * (long)(END == SILU ? N / 2 : N) +
                                n) =
          uint2{cvtpk_bf16(v[i][0], v[i][1]), cvtpk_bf16(v[i][2], v[i][3])};
    }
  }
}

// residual += sums of all splits; normed = rmsnorm(residual) * weight.
// Workgroup per row, four entries per thread and pass, everything in registers
// between the one read and the one write.
template <int PER>
__global__ __launch_bounds__(1024) void sums_add_rmsnorm_kernel(
    unsigned short* __restrict__ normed, unsigned short* __restrict__ residual,
    const float* __restrict__ sums, const unsigned short* __restrict__ nw,
    int N, int splits, float eps) {
  __shared__ float red[16];
  const long row = (long)blockIdx.x * N;
  const long slab = (long)gridDim.x * N;
  float v[PER][4];
  float sq = 0.f;
  uint2 wv[PER];
#pragma unroll
  for (int c = 0; c < PER; ++c) {
    const int n = (c * blockDim.x + threadIdx.x) * 4;
    const uint2 r = *reinterpret_cast<const uint2*>(residual + row + n);
    wv[c] = *reinterpret_cast<const uint2*>(nw + n);
    float4 a = *reinterpret_cast<const float4*>(sums + row + n);
#pragma unroll 8
    for (int s = 1; s < splits; ++s) {
      const float4 b =
          *reinterpret_cast<const float4*>(sums + s * slab + row + n);
      a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
    }
    const uint2 t{cvtpk_bf16(us2f(r.x & 0xffff) + a.x,
                             us2f(r.x >> 16) + a.y),
                  cvtpk_bf16(us2f(r.y & 0xffff) + a.z,
                             us2f(r.y >> 16) + a.w)};
    *reinterpret_cast<uint2*>(residual + row + n) = t;
    // the norm is that of the rounded residual
    v[c][0] = us2f(t.x & 0xffff); v[c][1] = us2f(t.x >> 16);
    v[c][2] = us2f(t.y & 0xffff); v[c][3] = us2f(t.y >> 16);
#pragma unroll
    for (int j = 0; j < 4; ++j) sq = fmaf(v[c][j], v[c][j], sq);
  }
  sq = block_reduce(sq, red, SumOp{}, 0.f);
  const float rs = __frsqrt_rn(sq / N + eps);
#pragma unroll
  for (int c = 0; c < PER; ++c) {
    const int n = (c * blockDim.x + threadIdx.x) * 4;
    *reinterpret_cast<uint2*>(normed + row + n) =
        uint2{cvtpk_bf16(v[c][0] * rs * us2f(wv[c].x & 0xffff),
                         v[c][1] * rs * us2f(wv[c].x >> 16)),
              cvtpk_bf16(v[c][2] * rs * us2f(wv[c].y & 0xffff),
                         v[c][3] * rs * us2f(wv[c].y >> 16))};
  }
}

// out = bf16 of the sums of all splits
__global__ __launch_bounds__(256) void sums_rows_kernel(
    unsigned short* __restrict__ out, const float* __restrict__ sums,
    long total, int splits) {
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= total) return;
  float4 a = *reinterpret_cast<const float4*>(sums + i);
#pragma unroll 8
  for (int s = 1; s < splits; ++s) {
    const float4 b = *reinterpret_cast<const float4*>(sums + s * total + i);
    a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
  }
  *reinterpret_cast<uint2*>(out + i) =
      uint2{cvtpk_bf16(a.x, a.y), cvtpk_bf16(a.z, a.w)};
}

constexpr int ROWS_PER_WG = 128;   // 8 waves x 2 tiles of 8 rows
constexpr int SLICE = 256;

template <int END>
void launch(unsigned short* out, float* sums, int splits,
            const torch::Tensor& x, const torch::Tensor& w) {
  const int M = x.size(0), N = w.size(0);
  const long K = x.size(1);
  auto stream = c10::hip::getCurrentHIPStream().stream();
#define SG_LAUNCH(MT_, RT_, NW_, KS_, OCC_, HALF_)                           \
  stream_gemm_kernel<MT_, RT_, NW_, KS_, OCC_, END, HALF_>                   \
      <<<dim3(N / (RT_ * NW_ * (HALF_ ? 16 : 8)), splits), NW_ * WAVE, 0,    \
         stream>>>(                                                          \
          out, sums, reinterpret_cast<const unsigned short*>(x.data_ptr()),  \
          reinterpret_cast<const unsigned short*>(w.data_ptr()), M, N, K)
  const int MT = (M + 15) / 16;
  if constexpr (END == SUMS) {
    // The matrix cores have nothing to spare any more: whole tiles of 16 rows
    // (4096 x 14336: 33 us at M = 96, 35 at 128; hipBLASLt 65 and 76).
    if (M > 64) {
      if (M <= 96) { SG_LAUNCH(6, 1, 8, 256, 2, true); }
      else { SG_LAUNCH(8, 1, 8, 256, 2, true); }
      HIP_CHECK_KERNEL();
      return;
    }
  } else {
    // Without parts it is the rows that have to fill the chip: 7 waves to a
    // workgroup where that makes more workgroups than 8 do and not more than
    // there are CUs (28672 x 4096: 256 instead of 224, with the activation 44.4
    // -> 43.5 us at 8 rows and 48.3 -> 45.2 at 32; 57344 x 8192 167.8 -> 159.8).
    const auto seven = [&](int rt) {
      return N > 256 * 64 && N % (rt * 56) == 0 && N / (rt * 56) <= 256;
    };
    // Twice the rows per workgroup halve the passes of x through LDS, where
    // that leaves most CUs one workgroup and none a second (57344 x 8192: M = 8
    // 166 -> 156 us, 32 178 -> 159, 64 200 -> 183; but 128256 x 4096, M = 8
    // 179 -> 203)
    const bool wide = N % 256 == 0 && N >= 200 * 256 && N <= 256 * 256;
#define SG_WIDE(NW_)                                                         \
  switch (MT) {                                                              \
    case 1: SG_LAUNCH(1, 4, NW_, 256, 2, false); break;                      \
    case 2: SG_LAUNCH(2, 4, NW_, 256, 2, false); break;                      \
    case 3: SG_LAUNCH(3, 4, NW_, 128, 2, false); break;                      \
    default: SG_LAUNCH(4, 4, NW_, 128, 2, false); break;                     \
  }
    if (wide || seven(2)) {
      if (wide && seven(4)) {
        SG_WIDE(7)
      } else if (wide) {
        SG_WIDE(8)
      } else {
        switch (MT) {
          case 1: SG_LAUNCH(1, 2, 7, 256, 4, false); break;
          case 2: SG_LAUNCH(2, 2, 7, 256, 2, false); break;
          case 3: SG_LAUNCH(3, 2, 7, 256, 2, false); break;
          default: SG_LAUNCH(4, 2, 7, 256, 2, false); break;
        }
      }
      HIP_CHECK_KERNEL();
      return;
    }
#undef SG_WIDE
  }
  if constexpr (END == SILU) {
    // the activation cannot be split into parts: few rows take half as many
    // waves to a workgroup (14336 x 4096, 8 rows: 38.4 -> 28.5 us)
    if (N <= 256 * 64) {
      switch (MT) {
        case 1: SG_LAUNCH(1, 2, 4, 256, 2, false); break;
        case 2: SG_LAUNCH(2, 2, 4, 256, 2, false); break;
        case 3: SG_LAUNCH(3, 2, 4, 256, 2, false); break;
        default: SG_LAUNCH(4, 2, 4, 256, 2, false); break;
      }
      HIP_CHECK_KERNEL();
      return;
    }
  }
  switch (MT) {
    case 1: SG_LAUNCH(1, 2, 8, 256, 4, false); break;
    case 2: SG_LAUNCH(2, 2, 8, 256, 2, false); break;
    case 3: SG_LAUNCH(3, 2, 8, 256, 2, false); break;
    default: SG_LAUNCH(4, 2, 8, 256, 2, false); break;
  }
#undef SG_LAUNCH
  HIP_CHECK_KERNEL();
}

void check(const torch::Tensor& x, const torch::Tensor& w) {
  TORCH_CHECK(x.is_cuda() && w.is_cuda() && x.device() == w.device());
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1));
  TORCH_CHECK(x.scalar_type() == torch::kBFloat16 &&
              w.scalar_type() == torch::kBFloat16);
  TORCH_CHECK(x.is_contiguous() && w.is_contiguous());
  TORCH_CHECK(x.size(0) >= 1 && x.size(0) <= 128 && w.size(0) > 0 &&
              w.size(0) % ROWS_PER_WG == 0 && x.size(1) > 0 &&
              x.size(1) % SLICE == 0);
  TORCH_CHECK(reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0);
}

// Workgroups of the same rows that share their reduction: one for each of 256
// CUs. The registers of one tile of x would let two share a CU, and the product
// alone is then 1 us faster (4096 x 14336, M = 8: 20.4 us in 16 parts, 21.5 in
// 8), but twice the parts cost who reads them more: with the norm 28.1 us and
// 26.7, 8192 x 28672 96.8 and 86.2.
int splits_of(const torch::Tensor& x, const torch::Tensor& w) {
  const long rows = w.size(0) / ROWS_PER_WG;
  if (rows >= 192 && x.size(0) <= 64) return 1;
  const long room = 256;
  return (int)std::max(1L, std::min(room / rows, (long)x.size(1) / SLICE));
}

torch::Tensor partial_sums(const torch::Tensor& x, const torch::Tensor& w) {
  const int splits = splits_of(x, w);
  auto sums = torch::empty({splits, x.size(0), w.size(0)},
                           x.options().dtype(torch::kFloat32));
  launch<SUMS>(nullptr, sums.data_ptr<float>(), splits, x, w);
  return sums;
}

unsigned short* bf16_rows(const torch::Tensor& t, long rows, long cols) {
  TORCH_CHECK(t.scalar_type() == torch::kBFloat16 && t.is_contiguous() &&
              t.dim() == 2 && t.size(0) == rows && t.size(1) == cols &&
              t.is_cuda() &&
              reinterpret_cast<uintptr_t>(t.data_ptr()) % 8 == 0);
  return reinterpret_cast<unsigned short*>(t.data_ptr());
}

}  // namespace

// out = x W^T
void stream_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w) {
  check(x, w);
  auto* op = bf16_rows(out, x.size(0), w.size(0));
  if (x.size(0) <= 64 && splits_of(x, w) == 1) {
    launch<ROWS>(op, nullptr, 1, x, w);
    return;
  }
  const auto sums = partial_sums(x, w);
  const long total = out.numel();
  sums_rows_kernel<<<(unsigned)((total / 4 + 255) / 256), 256, 0,
                     c10::hip::getCurrentHIPStream().stream()>>>(
      op, sums.data_ptr<float>(), total, (int)sums.size(0));
  HIP_CHECK_KERNEL();
}

// [splits, M, N]: fp32 parts of x W^T
torch::Tensor stream_gemm_sums(torch::Tensor x, torch::Tensor w) {
  check(x, w);
  return partial_sums(x, w);
}

// out [M, N / 2] = silu(x W[:N/2]^T) * (x W[N/2:]^T)
void stream_gemm_silu(torch::Tensor out, torch::Tensor x, torch::Tensor w) {
  check(x, w);
  TORCH_CHECK(x.size(0) <= 64);
  launch<SILU>(bf16_rows(out, x.size(0), w.size(0) / 2), nullptr, 1, x, w);
}

// residual += x W^T; normed = rmsnorm(residual) * nw
void stream_gemm_norm(torch::Tensor normed, torch::Tensor x, torch::Tensor w,
                      torch::Tensor residual, torch::Tensor nw, double eps) {
  check(x, w);
  const int M = x.size(0), N = w.size(0);
  TORCH_CHECK(N % 2048 == 0 && N <= 8192);
  auto* np = bf16_rows(normed, M, N);
  auto* rp = bf16_rows(residual, M, N);
  TORCH_CHECK(nw.scalar_type() == torch::kBFloat16 && nw.is_contiguous() &&
              nw.numel() == N &&
              reinterpret_cast<uintptr_t>(nw.data_ptr()) % 8 == 0);
  const auto sums = partial_sums(x, w);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const auto* wp = reinterpret_cast<const unsigned short*>(nw.data_ptr());
  if (N <= 4096)
    sums_add_rmsnorm_kernel<1><<<M, N / 4, 0, stream>>>(
        np, rp, sums.data_ptr<float>(), wp, N, (int)sums.size(0), (float)eps);
  else
    sums_add_rmsnorm_kernel<2><<<M, N / 8, 0, stream>>>(
        np, rp, sums.data_ptr<float>(), wp, N, (int)sums.size(0), (float)eps);
  HIP_CHECK_KERNEL();
}

}  // namespace kukeon
