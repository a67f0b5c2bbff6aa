// Fused top-k / top-p / temperature sampling for gfx950 — wide-parallel.
//
// Key observations driving the design (see profiles/r01_bench8_kernel_stats):
//  * logits are bf16, so their monotonic integer map has only 16 bits —
//    TWO 8-bit radix levels give an EXACT threshold (no 3rd pass, no ties
//    below the representable precision),
//  * one workgroup per row leaves a 256-CU chip almost idle at B<=64: every
//    pass here is split over grid (B, S) chunks of the vocab with
//    LDS-local histograms merged by global atomics,
//  * the categorical draw is Gumbel-max over the masked set (single packed
//    64-bit atomicMax, deterministic: ties resolve to the lowest index).
//
// Pipeline (7 small kernels, all hipGraph-capturable; ws row = 528 floats):
//  memset ws -> K1 max (+invT)  -> K2 level-0 count/weight hists + Z
//  -> K3 walk0 (+ hist re-zero) -> K4 level-1 hists -> K5 walk1 (threshold)
//  -> K6 masked gumbel argmax   -> K7 finalize token + bump seed.
//
// ws[b] layout (floats, reinterpreted per slot):
//  [0] row max (mapped u32)   [1] Z (f32)        [2] invT (f32)
//  [3] threshold (f32)        [4] prefix_k (u32) [5] prefix_p (u32)
//  [6..7] packed argmax (u64, 8-byte aligned: 528*4 % 8 == 0)
//  [8]  need_k (f32)          [9] need_p (f32)
//  [16..271] hist_count (u32) [272..527] hist_weight (f32)
#include <algorithm>

#include "common.h"
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

namespace kukeon {

constexpr int WS_ROW = 528;

DEV_INLINE unsigned int map16(unsigned short us) {
  return (us & 0x8000u) ? (unsigned int)(~us & 0xffffu)
                        : (unsigned int)(us | 0x8000u);
}
DEV_INLINE float unmap16_f(unsigned int mu) {
  unsigned short us = (mu & 0x8000u) ? (unsigned short)(mu & 0x7fffu)
                                     : (unsigned short)(~mu & 0xffffu);
  return us2f(us);
}
DEV_INLINE unsigned int map_f32(float f) {
  unsigned int b = __builtin_bit_cast(unsigned int, f);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

DEV_INLINE unsigned long long splitmix64(unsigned long long x) {
  x += 0x9e3779b97f4a7c15ull;
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
  return x ^ (x >> 31);
}
DEV_INLINE float uniform01(unsigned long long seed, unsigned int row,
                           unsigned int idx) {
  unsigned long long h =
      splitmix64(seed ^ ((unsigned long long)row << 32) ^ idx);
  return ((h >> 40) + 1.f) * (1.f / 16777217.f);
}

// Calls f(index, value) for this thread's share of chunk s of a row. With
// VEC (rows that start on 16 bytes) a thread takes 8 neighbours per load; a
// chunk is a multiple of 8 entries either way.
template <bool VEC, typename F>
DEV_INLINE void for_chunk(const unsigned short* __restrict__ row, int V,
                          int splits, int s, F f) {
  const int per = ((V + splits - 1) / splits + 7) / 8 * 8;
  const int lo = min(V, s * per), hi = min(V, lo + per);
  if (VEC) {
    for (int i = lo + (int)threadIdx.x * 8; i < hi; i += blockDim.x * 8) {
      const bf16x8 v = load_bf16x8(row + i);
#pragma unroll
      for (int j = 0; j < 8; ++j) f(i + j, v.us(j));
    }
  } else {
    for (int i = lo + (int)threadIdx.x; i < hi; i += blockDim.x) f(i, row[i]);
  }
}

// Histograms in LDS, one copy for every 16th lane: a row's logits fall into a
// handful of the 256 bins, and with one copy all lanes of a wave queue at the
// same address (this pass took 212 of the 500 us that 256 rows of 128256 took
// in all; with copies, wide loads and the walks in LDS all passes take 233, 8
// rows 33 instead of 50). Copies start 8 banks apart.
constexpr int COPIES = 16;
constexpr int COPY = 256 + 8;
struct Hists {
  unsigned int count[COPIES * COPY];
  float weight[COPIES * COPY];
};
DEV_INLINE void clear(Hists& h) {
  for (int i = threadIdx.x; i < COPIES * COPY; i += blockDim.x) {
    h.count[i] = 0;
    h.weight[i] = 0.f;
  }
}
DEV_INLINE void merge(const Hists& h, float* wsb) {
  unsigned int* gc = reinterpret_cast<unsigned int*>(wsb + 16);
  float* gw = wsb + 272;
  for (int i = threadIdx.x; i < 256; i += blockDim.x) {
    unsigned int n = 0;
    float w = 0.f;
#pragma unroll
    for (int c = 0; c < COPIES; ++c) {
      n += h.count[c * COPY + i];
      w += h.weight[c * COPY + i];
    }
    if (n) atomicAdd(&gc[i], n);
    if (w != 0.f) atomicAdd(&gw[i], w);
  }
}

// From the top bin down, the first at which the sum reaches `need` (or bin 0);
// *cum gets the sum above it. One thread, in this order (the sums are floats);
// the bins are in LDS and read 8 at a time, ahead of the additions. (Read
// from memory one by one they took 10 to 19 us.)
DEV_INLINE int walk(const float* bins, float need, float* cum) {
  float sum = 0.f;
  for (int b0 = 255; b0 >= 0; b0 -= 8) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = bins[b0 - j];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (sum + v[j] >= need || b0 - j == 0) {
        *cum = sum;
        return b0 - j;
      }
      sum += v[j];
    }
  }
  *cum = sum;
  return 0;
}

// ---- K0: zero the workspace rows. A kernel, NOT hipMemsetAsync: a
// memset captured inside a hipGraph was observed not to replay (ROCm 7.2),
// which let Z/argmax state accumulate across replays. ----
__global__ void k0_zero(float* __restrict__ ws) {
  float* wsb = ws + (long)blockIdx.x * WS_ROW;
  for (int i = threadIdx.x; i < WS_ROW; i += blockDim.x) wsb[i] = 0.f;
}

// ---- K1: row max (mapped) + invT ----
template <bool VEC>
__global__ void k1_max(float* __restrict__ ws,
                       const unsigned short* __restrict__ logits,
                       const float* __restrict__ temps, int V, int splits) {
  const int b = blockIdx.x;
  unsigned int mx = 0;
  for_chunk<VEC>(logits + (long)b * V, V, splits, blockIdx.y,
                 [&](int, unsigned short us) { mx = max(mx, map16(us)); });
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    mx = max(mx, (unsigned)__shfl_xor((int)mx, off, WAVE));
  __shared__ unsigned int red[16];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) red[wid] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < (blockDim.x + 63) / 64; ++w) mx = max(mx, red[w]);
    atomicMax(reinterpret_cast<unsigned int*>(ws + (long)b * WS_ROW), mx);
    if (blockIdx.y == 0) {
      const float T = temps[b];
      ws[(long)b * WS_ROW + 2] = T > 0.f ? 1.f / T : 1.f;
    }
  }
}

// ---- K2: level-0 histograms (count + exp-weight) + Z ----
template <bool VEC>
__global__ void k2_hist0(float* __restrict__ ws,
                         const unsigned short* __restrict__ logits, int V,
                         int splits) {
  __shared__ Hists h;
  __shared__ float redf[16];
  const int b = blockIdx.x;
  float* wsb = ws + (long)b * WS_ROW;
  clear(h);
  __syncthreads();
  const float mx = unmap16_f(
      *reinterpret_cast<const unsigned int*>(wsb + 0));
  const float invT = wsb[2];
  const int copy = (threadIdx.x & (COPIES - 1)) * COPY;
  float z = 0.f;
  for_chunk<VEC>(logits + (long)b * V, V, splits, blockIdx.y,
                 [&](int, unsigned short us) {
                   const unsigned int mu = map16(us);
                   const float e = __expf((us2f(us) - mx) * invT);
                   z += e;
                   atomicAdd(&h.count[copy + (mu >> 8)], 1u);
                   if (e != 0.f) atomicAdd(&h.weight[copy + (mu >> 8)], e);
                 });
  z = block_reduce(z, redf, SumOp{}, 0.f);
  if (threadIdx.x == 0) atomicAdd(wsb + 1, z);
  __syncthreads();
  merge(h, wsb);
}

// The 256 counts (as floats) and weights of a row, from memory to LDS.
DEV_INLINE void stage_bins(const float* wsb, float* counts, float* weights) {
  for (int i = threadIdx.x; i < 256; i += blockDim.x) {
    counts[i] = (float)reinterpret_cast<const unsigned int*>(wsb + 16)[i];
    weights[i] = wsb[272 + i];
  }
  __syncthreads();
}

// ---- K3: walk level 0 for both constraints, then re-zero the hists ----
__global__ void k3_walk0(float* __restrict__ ws,
                         const int* __restrict__ top_k,
                         const float* __restrict__ top_p, int V) {
  __shared__ float counts[256], weights[256];
  const int b = blockIdx.x;
  float* wsb = ws + (long)b * WS_ROW;
  stage_bins(wsb, counts, weights);
  // the two walks run in different waves
  if (threadIdx.x == 0) {
    const int k = top_k[b];
    unsigned int sel = 0xffffffffu;
    if (k > 0 && k < V) {
      float cum;
      sel = (unsigned)walk(counts, (float)k, &cum);
      wsb[8] = (float)k - cum;
    }
    *reinterpret_cast<unsigned int*>(wsb + 4) = sel;
  } else if (threadIdx.x == WAVE) {
    const float p = top_p[b];
    unsigned int sel = 0xffffffffu;
    if (p > 0.f && p < 1.f) {
      const float need = p * wsb[1];
      float cum;
      sel = (unsigned)walk(weights, need, &cum);
      wsb[9] = need - cum;
    }
    *reinterpret_cast<unsigned int*>(wsb + 5) = sel;
  }
  for (int i = threadIdx.x; i < 512; i += blockDim.x) wsb[16 + i] = 0.f;
}

// ---- K4: level-1 histograms restricted to the selected level-0 bins ----
template <bool VEC>
__global__ void k4_hist1(float* __restrict__ ws,
                         const unsigned short* __restrict__ logits, int V,
                         int splits) {
  __shared__ Hists h;
  const int b = blockIdx.x;
  float* wsb = ws + (long)b * WS_ROW;
  const unsigned int pk = *reinterpret_cast<const unsigned int*>(wsb + 4);
  const unsigned int pp = *reinterpret_cast<const unsigned int*>(wsb + 5);
  if (pk == 0xffffffffu && pp == 0xffffffffu) return;
  clear(h);
  __syncthreads();
  const float mx = unmap16_f(*reinterpret_cast<const unsigned int*>(wsb));
  const float invT = wsb[2];
  const int copy = (threadIdx.x & (COPIES - 1)) * COPY;
  for_chunk<VEC>(logits + (long)b * V, V, splits, blockIdx.y,
                 [&](int, unsigned short us) {
                   const unsigned int mu = map16(us);
                   const unsigned int hi8 = mu >> 8;
                   if (hi8 == pk)
                     atomicAdd(&h.count[copy + (mu & 0xffu)], 1u);
                   if (hi8 == pp)
                     atomicAdd(&h.weight[copy + (mu & 0xffu)],
                               __expf((us2f(us) - mx) * invT));
                 });
  __syncthreads();
  merge(h, wsb);
}

// ---- K5: walk level 1 -> final logit threshold ----
__global__ void k5_walk1(float* __restrict__ ws, int V) {
  __shared__ float counts[256], weights[256];
  __shared__ float th[2];
  const int b = blockIdx.x;
  float* wsb = ws + (long)b * WS_ROW;
  const unsigned int pk = *reinterpret_cast<const unsigned int*>(wsb + 4);
  const unsigned int pp = *reinterpret_cast<const unsigned int*>(wsb + 5);
  stage_bins(wsb, counts, weights);
  float cum;
  if (threadIdx.x == 0)
    th[0] = pk == 0xffffffffu
                ? -INFINITY
                : unmap16_f((pk << 8) | (unsigned)walk(counts, wsb[8], &cum));
  if (threadIdx.x == WAVE)
    th[1] = pp == 0xffffffffu
                ? -INFINITY
                : unmap16_f((pp << 8) | (unsigned)walk(weights, wsb[9],
                                                       &cum));
  __syncthreads();
  if (threadIdx.x == 0) wsb[3] = fmaxf(fmaxf(-INFINITY, th[0]), th[1]);
}

// ---- K6: masked Gumbel argmax, packed 64-bit atomic merge ----
template <bool VEC>
__global__ void k6_draw(float* __restrict__ ws,
                        const unsigned short* __restrict__ logits,
                        const float* __restrict__ temps,
                        const unsigned long long* __restrict__ seed, int V,
                        int splits) {
  const int b = blockIdx.x;
  float* wsb = ws + (long)b * WS_ROW;
  const float T = temps[b];
  const bool greedy = T <= 0.f;
  const float mx = unmap16_f(*reinterpret_cast<const unsigned int*>(wsb));
  const float invT = wsb[2];
  const float th = wsb[3];
  const unsigned long long sd = seed[0];
  float best = -INFINITY;
  int besti = 0;
  for_chunk<VEC>(
      logits + (long)b * V, V, splits, blockIdx.y,
      [&](int i, unsigned short us) {
        const float l = us2f(us);
        if (l < th) return;
        float key;
        if (greedy) {
          key = l;
        } else {
          key = (l - mx) * invT -
                __logf(-__logf(uniform01(sd, (unsigned)b, (unsigned)i)));
        }
        if (key > best || (key == best && i < besti)) {
          best = key;
          besti = i;
        }
      });
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float ov = __shfl_xor(best, off, WAVE);
    const int oi = __shfl_xor(besti, off, WAVE);
    if (ov > best || (ov == best && oi < besti)) { best = ov; besti = oi; }
  }
  __shared__ float rv[16];
  __shared__ int ri[16];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) { rv[wid] = best; ri[wid] = besti; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < (blockDim.x + 63) / 64; ++w)
      if (rv[w] > best || (rv[w] == best && ri[w] < besti)) {
        best = rv[w];
        besti = ri[w];
      }
    if (best != -INFINITY) {
      // pack: key (mapped f32) in the high word, ~idx low (ties -> min idx)
      const unsigned long long packed =
          ((unsigned long long)map_f32(best) << 32) |
          (unsigned)(~(unsigned)besti);
      atomicMax(reinterpret_cast<unsigned long long*>(wsb + 6), packed);
    }
  }
}

// ---- K7: finalize tokens + bump the seed ----
__global__ void k7_finalize(int* __restrict__ tokens,
                            const float* __restrict__ ws,
                            unsigned long long* __restrict__ seed, int B) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < B) {
    const unsigned long long packed =
        *reinterpret_cast<const unsigned long long*>(ws + (long)b * WS_ROW + 6);
    tokens[b] = (int)(~(unsigned)(packed & 0xffffffffu));
  }
  if (b == 0) seed[0] += 1;
}

// ---- self-advancing decode support: after sampling, feed the token back
// as the next step's input, advance the device-side cursors, and append to
// the ring buffer — so a micro-batch of decode steps replays with no host
// round-trip (one sync per micro-batch).
__global__ void decode_advance_kernel(int* __restrict__ ids,
                                      int* __restrict__ pos,
                                      int* __restrict__ seq_lens,
                                      const int* __restrict__ tokens,
                                      int* __restrict__ ring,
                                      int* __restrict__ counter, int B) {
  const int step = counter[0];
  // all waves have the step before one of them moves it on: a wave that came
  // late wrote its tokens to the next step's line (more than 64 rows)
  __syncthreads();
  for (int b = threadIdx.x; b < B; b += blockDim.x) {
    if (seq_lens[b] > 0) {  // active rows only (padded rows stay parked)
      ids[b] = tokens[b];
      pos[b] += 1;
      seq_lens[b] += 1;
      ring[step * B + b] = tokens[b];
    }
  }
  if (threadIdx.x == 0) counter[0] = step + 1;
}

void decode_advance(torch::Tensor ids, torch::Tensor pos,
                    torch::Tensor seq_lens, torch::Tensor tokens,
                    torch::Tensor ring, torch::Tensor counter) {
  const int B = ids.size(0);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  // one workgroup: the step counter is read and moved on within it
  decode_advance_kernel<<<1, std::max(64, std::min(1024, (B + 63) / 64 * 64)),
                          0, stream>>>(
      ids.data_ptr<int>(), pos.data_ptr<int>(), seq_lens.data_ptr<int>(),
      tokens.data_ptr<int>(), ring.data_ptr<int>(), counter.data_ptr<int>(),
      B);
  HIP_CHECK_KERNEL();
}

void sample(torch::Tensor tokens, torch::Tensor logits, torch::Tensor temps,
            torch::Tensor top_k, torch::Tensor top_p, torch::Tensor seed,
            torch::Tensor workspace) {
  const int B = logits.size(0);
  if (B == 0) return;
  const int V = logits.size(1);
  TORCH_CHECK(logits.scalar_type() == torch::kBFloat16 &&
              logits.is_contiguous());
  TORCH_CHECK(tokens.scalar_type() == torch::kInt32);
  TORCH_CHECK(workspace.numel() >= (long)B * WS_ROW,
              "sampling workspace must be at least [B, 528] floats");
  TORCH_CHECK(reinterpret_cast<uintptr_t>(workspace.data_ptr()) % 8 == 0);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const auto* lp = reinterpret_cast<const unsigned short*>(logits.data_ptr());
  float* ws = workspace.data_ptr<float>();
  // as many workgroups as fit with their histograms (34 KB each, 4 to a CU)
  const int splits = max(1, min(64, 1024 / B));
  dim3 wide(B, splits);
  k0_zero<<<B, 256, 0, stream>>>(ws);
  auto* sp = reinterpret_cast<unsigned long long*>(seed.data_ptr());
#define SAMPLE_PASS(VEC_)                                                    \
  k1_max<VEC_><<<wide, 256, 0, stream>>>(ws, lp, temps.data_ptr<float>(), V, \
                                         splits);                            \
  k2_hist0<VEC_><<<wide, 256, 0, stream>>>(ws, lp, V, splits);               \
  k3_walk0<<<B, 256, 0, stream>>>(ws, top_k.data_ptr<int>(),                 \
                                  top_p.data_ptr<float>(), V);               \
  k4_hist1<VEC_><<<wide, 256, 0, stream>>>(ws, lp, V, splits);               \
  k5_walk1<<<B, 256, 0, stream>>>(ws, V);                                    \
  k6_draw<VEC_><<<wide, 256, 0, stream>>>(ws, lp, temps.data_ptr<float>(),   \
                                          sp, V, splits)
  if (V % 8 == 0 && reinterpret_cast<uintptr_t>(lp) % 16 == 0) {
    SAMPLE_PASS(true);
  } else {
    SAMPLE_PASS(false);
  }
#undef SAMPLE_PASS
  k7_finalize<<<(B + 255) / 256, 256, 0, stream>>>(
      tokens.data_ptr<int>(), ws, sp, B);
  HIP_CHECK_KERNEL();
}

}  // namespace kukeon
