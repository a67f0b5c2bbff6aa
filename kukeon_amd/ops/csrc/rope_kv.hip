// Fused rotary embedding (NEOX / Llama half-rotation style) + paged-KV-cache
// append for gfx950.
//
// Operates in place on the fused qkv projection output [T, (Hq+2*Hk)*D]
// (avoids materializing contiguous q/k/v copies), rotates q and k, and
// scatters the rotated k and raw v into the paged caches
// k_cache/v_cache [num_blocks, Hk, BLOCK, D].
//
// cos/sin are host-precomputed per guide Appendix B (trig on device turns
// memory-bound into VALU-bound): table [max_pos, D] f32 with cos in [0, D/2)
// and sin in [D/2, D).
#include "common.h"
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

namespace kukeon {

torch::Tensor stream_gemm_sums(torch::Tensor x, torch::Tensor w);

// A thread takes 8 pairs of one head (queries, then keys) or 8 entries of a
// value row; the three kinds are numbered through, so that a decode batch does
// them side by side. SUMS: the projection arrives as fp32 parts [splits, T,
// row] that are added up here; queries go to qkv rounded once, keys and values
// to their pages only.
template <bool FP8, bool SUMS>
__global__ void rope_kv_kernel(
    unsigned short* __restrict__ qkv,        // [T, (Hq+2Hk)*D]
    const float* __restrict__ sums, int splits,
    void* __restrict__ k_cache,              // [NB, Hk, BS, D] bf16|fp8
    void* __restrict__ v_cache,
    const float* __restrict__ cos_sin,       // [max_pos, D]
    const int* __restrict__ positions,       // [T]
    const int* __restrict__ slot_mapping,    // [T] flat slot = block*BS + off
    const int* __restrict__ block_table,     // [T, max_blocks] decode mode:
    int max_blocks,                          //   slot derived on device
    int Hq, int Hk, int D, int BS) {
  const long t = blockIdx.x;
  // grid.y splits the per-token chunk loops so small decode batches still
  // put >=256 workgroups on the chip
  const int yoff = blockIdx.y * blockDim.x + threadIdx.x;
  const int ystride = gridDim.y * blockDim.x;
  const int half = D / 2;
  const long row_stride = (long)(Hq + 2 * Hk) * D;
  unsigned short* row = qkv + t * row_stride;
  const int pos = positions[t];
  if (pos < 0) return;  // inactive decode row: no rotate, no KV write
  int slot;
  if (block_table != nullptr) {
    // decode: the device owns the sequence cursor (self-advancing graph)
    slot = block_table[t * (long)max_blocks + pos / BS] * BS + pos % BS;
  } else {
    slot = slot_mapping[t];
  }
  const float* cs = cos_sin + (long)pos * D;
  const long cache_tok_base =
      slot >= 0 ? ((long)(slot / BS) * Hk * BS + (long)(slot % BS)) * D : 0;

  auto load8 = [&](int col, float* f) {
    if (SUMS) {
      const float* p = sums + t * row_stride + col;
      const long slab = (long)gridDim.x * row_stride;
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = 0.f;
#pragma unroll 4
      for (int s = 0; s < splits; ++s) {
        const float4 a = *reinterpret_cast<const float4*>(p + s * slab);
        const float4 b = *reinterpret_cast<const float4*>(p + s * slab + 4);
        f[0] += a.x; f[1] += a.y; f[2] += a.z; f[3] += a.w;
        f[4] += b.x; f[5] += b.y; f[6] += b.z; f[7] += b.w;
      }
    } else {
      const bf16x8 v = load_bf16x8(row + col);
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = v.f(j);
    }
  };
  auto page_write = [&](void* cache, long off, const float* f, uint4 packed) {
    if (FP8)
      *reinterpret_cast<uint2*>(reinterpret_cast<unsigned char*>(cache) +
                                off) = pack_fp8x8(f);
    else
      *reinterpret_cast<uint4*>(reinterpret_cast<unsigned short*>(cache) +
                                off) = packed;
  };

  const int pair_chunks = D / 16;                  // per head
  const int k_first = Hq * pair_chunks;
  const int v_first = k_first + Hk * pair_chunks;
  const int total = v_first + Hk * (D / 8);
  for (int c = yoff; c < total; c += ystride) {
    if (c < v_first) {
      const int h = c / pair_chunks;               // keys follow the queries
      const int d0 = (c % pair_chunks) * 8;
      float x[8], y[8], xo[8], yo[8];
      load8(h * D + d0, x);
      load8(h * D + half + d0, y);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float co = cs[d0 + j], si = cs[half + d0 + j];
        xo[j] = x[j] * co - y[j] * si;
        yo[j] = y[j] * co + x[j] * si;
      }
      const uint4 px = pack_bf16x8(xo), py = pack_bf16x8(yo);
      if (!SUMS || c < k_first) {
        *reinterpret_cast<uint4*>(row + (long)h * D + d0) = px;
        *reinterpret_cast<uint4*>(row + (long)h * D + half + d0) = py;
      }
      if (c >= k_first && slot >= 0) {
        const long off = cache_tok_base + (long)(h - Hq) * BS * D;
        page_write(k_cache, off + d0, xo, px);
        page_write(k_cache, off + half + d0, yo, py);
      }
    } else if (slot >= 0) {
      const int h = (c - v_first) / (D / 8);
      const int d0 = ((c - v_first) % (D / 8)) * 8;
      float f[8];
      load8((Hq + Hk + h) * D + d0, f);
      page_write(v_cache, cache_tok_base + (long)h * BS * D + d0, f,
                 pack_bf16x8(f));
    }
  }
}

// `sums`: undefined, or the projection's parts
static void rope_kv(torch::Tensor qkv, const torch::Tensor& sums,
                    torch::Tensor k_cache, torch::Tensor v_cache,
                    torch::Tensor cos_sin, torch::Tensor positions,
                    torch::Tensor slot_mapping, int64_t num_q_heads,
                    int64_t num_kv_heads, int64_t head_dim,
                    torch::Tensor block_table) {
  TORCH_CHECK(qkv.is_contiguous() && qkv.scalar_type() == torch::kBFloat16);
  TORCH_CHECK(cos_sin.scalar_type() == torch::kFloat32);
  TORCH_CHECK(positions.scalar_type() == torch::kInt32);
  TORCH_CHECK(slot_mapping.scalar_type() == torch::kInt32);
  const long T = qkv.size(0);
  if (T == 0) return;
  const int D = (int)head_dim;
  TORCH_CHECK(D % 16 == 0, "head_dim must be a multiple of 16");
  TORCH_CHECK(qkv.size(1) == (num_q_heads + 2 * num_kv_heads) * D);
  const int BS = (int)k_cache.size(2);
  TORCH_CHECK(k_cache.size(1) == num_kv_heads && k_cache.size(3) == D);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const bool table_mode = block_table.dim() == 2;
  const int* bt = table_mode ? block_table.data_ptr<int>() : nullptr;
  const int mb = table_mode ? (int)block_table.size(1) : 0;
  const bool fp8 = k_cache.scalar_type() == torch::kUInt8;
  const unsigned ysplit = T <= 128 ? 4 : 1;
  const bool parts = sums.defined();
  const float* sp = parts ? sums.data_ptr<float>() : nullptr;
  const int splits = parts ? (int)sums.size(0) : 0;
#define RK_LAUNCH(FP8_, SUMS_)                                               \
  rope_kv_kernel<FP8_, SUMS_><<<dim3((unsigned)T, ysplit), 256, 0, stream>>>(\
      reinterpret_cast<unsigned short*>(qkv.data_ptr()), sp, splits,         \
      k_cache.data_ptr(), v_cache.data_ptr(), cos_sin.data_ptr<float>(),     \
      positions.data_ptr<int>(), slot_mapping.data_ptr<int>(), bt, mb,       \
      (int)num_q_heads, (int)num_kv_heads, D, BS)
  if (parts) {
    if (fp8) { RK_LAUNCH(true, true); } else { RK_LAUNCH(false, true); }
  } else {
    if (fp8) { RK_LAUNCH(true, false); } else { RK_LAUNCH(false, false); }
  }
#undef RK_LAUNCH
  HIP_CHECK_KERNEL();
}

void rope_kv_append(torch::Tensor qkv, torch::Tensor k_cache,
                    torch::Tensor v_cache, torch::Tensor cos_sin,
                    torch::Tensor positions, torch::Tensor slot_mapping,
                    int64_t num_q_heads, int64_t num_kv_heads,
                    int64_t head_dim, torch::Tensor block_table) {
  rope_kv(qkv, torch::Tensor(), k_cache, v_cache, cos_sin, positions,
          slot_mapping, num_q_heads, num_kv_heads, head_dim, block_table);
}

// The projection qkv = x W^T and rope_kv_append in one: the projection's parts
// go straight to the rotary kernel. Only the query columns of qkv are written.
void qkv_rope_append(torch::Tensor qkv, torch::Tensor x, torch::Tensor w,
                     torch::Tensor k_cache, torch::Tensor v_cache,
                     torch::Tensor cos_sin, torch::Tensor positions,
                     torch::Tensor slot_mapping, int64_t num_q_heads,
                     int64_t num_kv_heads, int64_t head_dim,
                     torch::Tensor block_table) {
  TORCH_CHECK(qkv.dim() == 2 && qkv.size(0) == x.size(0) &&
              qkv.size(1) == w.size(0));
  rope_kv(qkv, stream_gemm_sums(x, w), k_cache, v_cache, cos_sin, positions,
          slot_mapping, num_q_heads, num_kv_heads, head_dim, block_table);
}

}  // namespace kukeon
