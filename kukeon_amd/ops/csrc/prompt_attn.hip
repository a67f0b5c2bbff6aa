// Varlen causal attention of prompt portions over paged keys and values
// (MFMA, bf16) for gfx950.
//
// What bounds it: one wave owns 32 query rows of one head. Per 64 keys it
// issues 32 v_mfma_f32_32x32x16_bf16 (1024 matrix-core cycles) against about
// as many cycles of softmax on the vector ALU (64 exponentials at quarter rate
// among them) and 32 KB of LDS reads, so all three pipes are close to even and
// what matters is that they overlap: two waves share a SIMD, and a workgroup
// has one barrier per 64 keys.
//   - workgroup = 8 waves = 4 query heads of one kv head x 2 blocks of 32
//     rows (4 waves = one block where sequences bring no more than that): a
//     K/V tile is staged in LDS once for all of them.
//   - two LDS tiles in turn: the next tile's global loads are issued before
//     the present tile's arithmetic and written to the other buffer after its
//     softmax.
//   - swapped S^T = K Q^T, so that a lane owns one query row's scores; the
//     score registers are the B operand of O^T = V^T P^T as they stand if the
//     PV product counts its keys in the order of the score rows (lane half
//     hi, entry j of chunk c is key 16 c + 4 hi + (j & 3) + 8 (j >> 2)).
//   - V stays row-major in LDS: ds_read_b64_tr_b16 hands each lane four keys
//     of its value entry. (Staging V transposed cost a 16-way bank conflict
//     per store.) Both images are swizzled: K by 16-byte pieces with row & 15,
//     V by pairs of 32-byte pieces with row & 3.
//   - exponents in base 2 with the scale folded into one fma; the running
//     maximum only moves when a row's scores pass it by 2^8, so that most
//     tiles rescale nothing; the mask is applied to tiles on the diagonal
//     only.
//   - few query rows against a long context leave the chip idle: the key
//     tiles of a workgroup are then split over several, their unnormalised
//     sums merged in split order by a second kernel.
// Measured (32 query heads, 8 kv heads, bf16; before: 32-key tiles, one row
// block per workgroup, V staged transposed): one prompt of 12037 tokens 3330 ->
// 1200 us (990 TFLOP/s), 64 prompts of 257 on contexts of 513 to 3201 1780 ->
// 753 us, one of 333 on 2900 210 -> 47 us, 30 of 390 to 701 299 -> 183 us.
// Without any loads it would take 1020 us on the first: the rest is the two
// waves' products and softmax not overlapping, which neither staggered waves
// nor wave priorities changed.
// Workgroups are numbered kv head first: consecutive ones go to different
// XCDs, so with 8 kv heads an XCD's L2 holds one head's pages.
//
// Fragment maps (pinned by tests/test_ops_gpu.py):
//   A[32x16k]: lane l -> row = l&31, k = 8*(l>>5) + j   (j = 0..7, bf16x8)
//   B[16kx32]: lane l -> col = l&31, k = 8*(l>>5) + j
//   C/D:       lane l -> col = l&31, row = (r&3) + 8*(r>>2) + 4*(l>>5)
//   ds_read_b64_tr_b16, per 16 lanes: lane i gives the address of row i>>2,
//   entries 4*(i&3)..+3, and gets entry i of rows 0..3
#include "common.h"
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

namespace kukeon {
namespace {

typedef __attribute__((__vector_size__(8 * sizeof(short)))) short frag8_t;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short frag4_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float acc16_t;
typedef __attribute__((address_space(3))) frag4_t lds_frag4_t;

constexpr int D = 128;
constexpr int BS = 16;          // tokens per page
constexpr int KVT = 64;         // keys per tile
constexpr float NONE = -3.0e38f;  // running maximum before any key

struct frag_words { unsigned int x[4]; };
struct frag_pair { frag4_t lo, hi; };

// four keys of this lane's value entry, from row-major rows in LDS
DEV_INLINE frag4_t read_tr(const char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (lds_frag4_t*)(__attribute__((address_space(3))) void*)p);
}

// Order of a block of N matrix instructions with R LDS reads each: the reads
// run AHEAD instructions in front (left to itself the compiler issues them
// two at a time and waits out the LDS latency every time).
template <int N, int AHEAD, int R>
DEV_INLINE void interleave() {
  __builtin_amdgcn_sched_group_barrier(0x100, AHEAD * R, 0);
#pragma unroll
  for (int i = 0; i < N - AHEAD; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, R, 0);
  }
  __builtin_amdgcn_sched_group_barrier(0x008, AHEAD, 0);
}

// NW waves: (NW / 4) blocks of 32 rows x 4 heads
template <int NW, bool FP8, bool SPLIT>
__global__ __launch_bounds__(NW * WAVE, 2) void prompt_attn_kernel(
    unsigned short* __restrict__ out,       // [T, Hq*D]
    float* __restrict__ part_o,             // [splits, T, Hq, D] (SPLIT)
    float* __restrict__ part_ml,            // [splits, T, Hq, 2]
    const unsigned short* __restrict__ q,   // [T, q_stride] fused qkv rows
    const void* __restrict__ k_cache,       // [NB, Hk, BS, D] bf16|fp8
    const void* __restrict__ v_cache,
    const int* __restrict__ block_table,    // [nseq, max_blocks]
    const int* __restrict__ seq_lens,       // [nseq] total ctx after append
    const int* __restrict__ q_starts,       // [nseq, 2] = (abs_start, row0)
    const int* __restrict__ qb_seq,         // [nqb]
    const int* __restrict__ qb_start,       // [nqb] local q offset
    long q_stride, long q_offset, long out_stride, long T, int nqb, int Hq,
    int Hk, int max_blocks, int splits, float scale) {
  constexpr int NT = NW * WAVE;
  constexpr int CH = KVT * D / 8 / NT;      // 16-byte pieces per thread
  __shared__ __align__(16) unsigned short kbuf[2][KVT * D];
  __shared__ __align__(16) unsigned short vbuf[2][KVT * D];

  // The last blocks of a sequence have the most keys: they go first. With
  // pairs, every second block only hands over to the one before it: as
  // workgroups go round the shader engines in turn, idle ones in alternation
  // would leave every second engine empty, so the even entries come first.
  int e = nqb - 1 - (int)(blockIdx.x / Hk);
  if (NW == 8) {
    const int odd = nqb / 2;
    e = e < odd ? 2 * e + 1 : 2 * (e - odd);
  }
  const int hk = blockIdx.x % Hk;
  const int zs = (int)blockIdx.y / splits;       // group of 4 query heads
  const int split = (int)blockIdx.y % splits;
  const int s = qb_seq[e];
  const int qb0 = qb_start[e];
  int rows_max = 32;
  if (NW == 8) {
    // a block at 32 mod 64 belongs to the workgroup of the one before it
    if (qb0 % 64 == 32 && e > 0 && qb_seq[e - 1] == s &&
        qb_start[e - 1] == qb0 - 32)
      return;
    if (qb0 % 64 == 0 && e + 1 < nqb && qb_seq[e + 1] == s &&
        qb_start[e + 1] == qb0 + 32)
      rows_max = 64;
  }
  const int ctx = seq_lens[s];
  const int abs_start = q_starts[2 * s];
  const int row0 = q_starts[2 * s + 1] + qb0;
  const int qn = min(rows_max, ctx - abs_start - qb0);
  if (qn <= 0) return;
  const int G = Hq / Hk;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x & (WAVE - 1);
  const int hi = lane >> 5;
  const int col = lane & 31;
  const int h_local = zs * 4 + (wid & 3);
  const int r0 = (wid >> 2) * 32;                // this wave's first row
  const bool active = h_local < G && r0 < qn;
  const int head = hk * G + (h_local < G ? h_local : 0);
  const int my_row = min(r0 + col, qn - 1);      // clamped for padding
  const int q_abs = abs_start + qb0 + my_row;
  const int wave_first = abs_start + qb0 + r0;
  const int wave_last = abs_start + qb0 + min(r0 + 32, qn) - 1;

  unsigned int qf[8][4];
  {
    const unsigned short* qp =
        q + (row0 + my_row) * q_stride + q_offset + (long)head * D;
    // a negative scale is a positive one on negated queries
    const unsigned int flip = scale < 0.f ? 0x80008000u : 0u;
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      const uint4 v = *reinterpret_cast<const uint4*>(qp + st * 16 + hi * 8);
      qf[st][0] = v.x ^ flip; qf[st][1] = v.y ^ flip;
      qf[st][2] = v.z ^ flip; qf[st][3] = v.w ^ flip;
    }
  }
  const float c2 = fabsf(scale) * 1.44269504088896340736f;

  // key tiles of this workgroup
  const int ntiles = (abs_start + qb0 + qn + KVT - 1) / KVT;
  int t_begin = 0, t_end = ntiles;
  if (SPLIT) {
    const int per = (ntiles + splits - 1) / splits;
    t_begin = split * per;
    t_end = min(ntiles, t_begin + per);
  }
  const int last_page = (ctx + BS - 1) / BS - 1;
  const int* table = block_table + (long)s * max_blocks;

  // staging: piece i of a thread is entries d0.. of row st_row + i * NT / 16
  const int st_row = threadIdx.x >> 4;
  const int d0 = (threadIdx.x & 15) * 8;
  uint4 kreg[CH], vreg[CH];
  // page ids of the pieces, fetched a tile ahead of the rows themselves
  int pk[CH];
  auto pages = [&](int t) {
#pragma unroll
    for (int i = 0; i < CH; ++i)
      pk[i] = table[min((t * KVT + st_row + i * (NT / 16)) / BS, last_page)];
  };
  auto row_at = [&](int page, int i) {
    return (((long)page * Hk + hk) * BS + ((st_row + i * (NT / 16)) % BS)) *
               D + d0;
  };
  auto load8 = [&](const void* cache, long off) {
    if (FP8) {
      const uint2 w = *reinterpret_cast<const uint2*>(
          reinterpret_cast<const unsigned char*>(cache) + off);
      return uint4{w.x, w.y, 0, 0};
    }
    return *reinterpret_cast<const uint4*>(
        reinterpret_cast<const unsigned short*>(cache) + off);
  };
  auto widen = [&](uint4 w) {
    return FP8 ? fp8x8_to_bf16x8(uint2{w.x, w.y}) : w;
  };
  auto fetch_k = [&](int t) {
    if (t < t_end)
#pragma unroll
      for (int i = 0; i < CH; ++i) kreg[i] = load8(k_cache, row_at(pk[i], i));
  };
  auto fetch_v = [&](int t) {
    if (t < t_end)
#pragma unroll
      for (int i = 0; i < CH; ++i) vreg[i] = load8(v_cache, row_at(pk[i], i));
  };
  auto store_k = [&](int t) {
    if (t < t_end)
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const int row = st_row + i * (NT / 16);
        *reinterpret_cast<uint4*>(
            reinterpret_cast<char*>(kbuf[(t - t_begin) & 1]) + row * 256 +
            ((d0 * 2) ^ ((row & 15) << 4))) = widen(kreg[i]);
      }
  };
  auto store_v = [&](int t) {
    if (t < t_end)
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const int row = st_row + i * (NT / 16);
        uint4 vv = widen(vreg[i]);
        // no value of a row past the context: 0 * NaN would poison the sum
        if (t * KVT + row >= ctx) vv = uint4{0, 0, 0, 0};
        *reinterpret_cast<uint4*>(
            reinterpret_cast<char*>(vbuf[(t - t_begin) & 1]) + row * 256 +
            ((d0 * 2) ^ ((row & 3) << 6))) = vv;
      }
  };

  float mc = NONE, l_acc = 0.f;     // running maximum times c2; lane's sum
  acc16_t oacc[4] = {{}, {}, {}, {}};
  acc16_t sc[2];
  unsigned int pw[2][8];

  // per-lane LDS offsets
  const int k_row = col * 256;
  const int k_swz = (col & 15) << 4;
  const int v_row = 4 * hi + ((lane & 15) >> 2);         // + 16 c (+ 8)
  const int v_col = ((lane >> 4) & 1) * 32 + (lane & 3) * 8;   // bytes
  const int v_swz = (v_row & 3) << 6;

  // S^T = K Q^T of tile t
  auto scores = [&](int t) {
    if (!active || t * KVT > wave_last) return;
    const char* kb = reinterpret_cast<const char*>(kbuf[(t - t_begin) & 1]);
    sc[0] = acc16_t{};
    sc[1] = acc16_t{};
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      const int byte = k_row + ((st * 32 + hi * 16) ^ k_swz);
      const frag8_t qv = __builtin_bit_cast(
          frag8_t,
          frag_words{{qf[st][0], qf[st][1], qf[st][2], qf[st][3]}});
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        const uint4 kf =
            *reinterpret_cast<const uint4*>(kb + kt * 32 * 256 + byte);
        sc[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            __builtin_bit_cast(frag8_t, kf), qv, sc[kt], 0, 0, 0);
      }
    }
    interleave<16, 6, 1>();
  };
  // weights of tile t from its scores
  auto softmax = [&](int t) {
    const int kvbase = t * KVT;
    if (!active || kvbase > wave_last) return;
    if (kvbase + KVT - 1 > wave_first) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int kvpos = kvbase + kt * 32 + (r & 3) + 8 * (r >> 2) + 4 * hi;
          if (kvpos > q_abs) sc[kt][r] = -INFINITY;
        }
    }
    float mx = sc[0][0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, sc[0][r]);
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[1][r]);
    // the other half of the wave holds the row's other keys
    {
      const auto sw = __builtin_amdgcn_permlane32_swap(
          __builtin_bit_cast(unsigned int, mx),
          __builtin_bit_cast(unsigned int, mx), false, false);
      mx = fmaxf(__builtin_bit_cast(float, (unsigned int)sw[0]),
                 __builtin_bit_cast(float, (unsigned int)sw[1]));
    }
    if (__any(fmaf(mx, c2, -mc) > 8.f)) {
      const float mn = fmaxf(mc, mx * c2);
      const float alpha = __builtin_amdgcn_exp2f(mc - mn);
      mc = mn;
      l_acc *= alpha;
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[db][r] *= alpha;
    }
    float ls[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float p0 = __builtin_amdgcn_exp2f(fmaf(sc[kt][r], c2, -mc));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(sc[kt][r + 1], c2, -mc));
        ls[r & 2] += p0;
        ls[(r & 2) + 1] += p1;
        pw[kt][r >> 1] = cvtpk_bf16(p0, p1);
      }
    l_acc += (ls[0] + ls[1]) + (ls[2] + ls[3]);
  };
  // O^T += V^T P^T of tile t
  auto values = [&](int t) {
    if (!active || t * KVT > wave_last) return;
    const char* vb = reinterpret_cast<const char*>(vbuf[(t - t_begin) & 1]);
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const frag8_t pf = __builtin_bit_cast(
            frag8_t, frag_words{{pw[kt][4 * c], pw[kt][4 * c + 1],
                                 pw[kt][4 * c + 2], pw[kt][4 * c + 3]}});
        const char* vp = vb + (kt * 32 + c * 16 + v_row) * 256;
#pragma unroll
        for (int db = 0; db < 4; ++db) {
          const int byte = (db * 64 + v_col) ^ v_swz;
          const frag_pair vf{read_tr(vp + byte), read_tr(vp + 8 * 256 + byte)};
          oacc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              __builtin_bit_cast(frag8_t, vf), pf, oacc[db], 0, 0, 0);
        }
      }
    interleave<16, 6, 2>();
  };

  if (t_begin < t_end) {
    pages(t_begin);
    fetch_k(t_begin);
    fetch_v(t_begin);
    pages(t_begin + 1);
    store_k(t_begin);
    store_v(t_begin);
    __syncthreads();
    for (int t = t_begin; t < t_end; ++t) {
      fetch_k(t + 1);
      fetch_v(t + 1);
      pages(t + 2);
      scores(t);
      softmax(t);
      store_k(t + 1);
      store_v(t + 1);
      values(t);
      __syncthreads();
    }
  }

  if (!active) return;
  l_acc += __shfl_xor(l_acc, 32, WAVE);
  if (r0 + col >= qn) return;
  const long row = row0 + r0 + col;
  if (SPLIT) {
    const long at = ((long)split * T + row) * Hq + head;
    if (hi == 0)
      *reinterpret_cast<float2*>(part_ml + at * 2) = float2{mc, l_acc};
    if (t_begin >= t_end) return;
    float* po = part_o + at * D;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd)
        *reinterpret_cast<float4*>(po + db * 32 + qd * 8 + 4 * hi) =
            float4{oacc[db][qd * 4], oacc[db][qd * 4 + 1],
                   oacc[db][qd * 4 + 2], oacc[db][qd * 4 + 3]};
    return;
  }
  const float inv = l_acc != 0.f ? 1.f / l_acc : 0.f;
  unsigned short* orow = out + row * out_stride + (long)head * D;
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int qd = 0; qd < 4; ++qd)
      *reinterpret_cast<uint2*>(orow + db * 32 + qd * 8 + 4 * hi) =
          uint2{cvtpk_bf16(oacc[db][qd * 4] * inv, oacc[db][qd * 4 + 1] * inv),
                cvtpk_bf16(oacc[db][qd * 4 + 2] * inv,
                           oacc[db][qd * 4 + 3] * inv)};
}

// Sums of the key splits, in split order. A wave per (row of a 32-row block,
// head), two entries per lane. A split without a visible key (sum 0) holds no
// values.
__global__ __launch_bounds__(256) void prompt_attn_merge_kernel(
    unsigned short* __restrict__ out, const float* __restrict__ part_o,
    const float* __restrict__ part_ml, const int* __restrict__ seq_lens,
    const int* __restrict__ q_starts, const int* __restrict__ qb_seq,
    const int* __restrict__ qb_start, long out_stride, long T, int Hq,
    int splits) {
  const int s = qb_seq[blockIdx.x];
  const int r = qb_start[blockIdx.x] + blockIdx.y;
  const int head = blockIdx.z * 4 + threadIdx.x / WAVE;
  if (r >= seq_lens[s] - q_starts[2 * s] || head >= Hq) return;
  const long row = q_starts[2 * s + 1] + r;
  const int d = (threadIdx.x & (WAVE - 1)) * 2;
  float m = NONE;
  for (int p = 0; p < splits; ++p)
    m = fmaxf(m, part_ml[(((long)p * T + row) * Hq + head) * 2]);
  float l = 0.f, a0 = 0.f, a1 = 0.f;
  for (int p = 0; p < splits; ++p) {
    const long at = ((long)p * T + row) * Hq + head;
    const float2 ml = *reinterpret_cast<const float2*>(part_ml + at * 2);
    if (ml.y == 0.f) continue;
    const float w = __builtin_amdgcn_exp2f(ml.x - m);
    const float2 o = *reinterpret_cast<const float2*>(part_o + at * D + d);
    l += w * ml.y;
    a0 += w * o.x;
    a1 += w * o.y;
  }
  const float inv = l != 0.f ? 1.f / l : 0.f;
  *reinterpret_cast<unsigned int*>(out + row * out_stride + (long)head * D +
                                   d) = cvtpk_bf16(a0 * inv, a1 * inv);
}

}  // namespace

void prefill_attention(torch::Tensor out, torch::Tensor q,
                       torch::Tensor k_cache, torch::Tensor v_cache,
                       torch::Tensor block_table, torch::Tensor seq_lens,
                       torch::Tensor q_starts, torch::Tensor qb_seq,
                       torch::Tensor qb_start, int64_t q_offset, double scale) {
  const int Hk = k_cache.size(1);
  const int Hq = out.size(1) / D;
  const int G = Hq / Hk;
  const int nqb = qb_seq.size(0);
  if (nqb == 0) return;
  TORCH_CHECK(k_cache.size(3) == D, "only head_dim=128 supported");
  TORCH_CHECK(k_cache.size(2) == BS, "kv block size must be 16");
  TORCH_CHECK(q_starts.dim() == 2 && q_starts.size(1) == 2);
  TORCH_CHECK(qb_seq.scalar_type() == torch::kInt32);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const long T = q.size(0);
  const int max_blocks = block_table.size(1);
  const bool fp8 = k_cache.scalar_type() == torch::kUInt8;
  // Two row blocks per workgroup halve the staging per query row, where
  // sequences bring more than one block at all.
  const bool pairs = 4 * (long)nqb > 5 * block_table.size(0);
  // The chip holds 256 workgroups of 8 waves or 512 of 4 at a time. Splitting
  // the key tiles fills it where there are fewer, and evens out the last round
  // where there are few rounds. A tile takes about 2 us; the merge writes and
  // reads the partial sums (about 4 TB/s) and is one more launch. Below 4
  // tiles (256 keys) per split the walk is no longer what takes the time.
  // (333 rows on 2900 keys: 210 us unsplit before, 5 splits 47 us.)
  const int groups = (G + 3) / 4;
  const long units = (pairs ? (nqb + 1L) / 2 : nqb) * Hk * groups;
  const long room = pairs ? 256 : 512;
  const long tiles = ((long)max_blocks * BS + KVT - 1) / KVT;
  int splits = 1;
  double least = 0;
  for (int sp = 1; sp <= 16 && (sp == 1 || tiles >= 4 * sp); ++sp) {
    const double rounds = (double)((units * sp + room - 1) / room);
    const double us =
        rounds * ((tiles + sp - 1) / sp) * 2.0 +
        (sp > 1 ? 4.0 + 2.0 * sp * T * Hq * (D + 2) * 4 / 4e6 : 0.0);
    if (sp == 1 || us < least) {
      least = us;
      splits = sp;
    }
  }
  torch::Tensor ws;
  float *po = nullptr, *pml = nullptr;
  if (splits > 1) {
    ws = torch::empty({splits * T * Hq * (D + 2)},
                      q.options().dtype(torch::kFloat32));
    po = ws.data_ptr<float>();
    pml = po + splits * T * Hq * D;
  }
  dim3 grid((unsigned)Hk * nqb, groups * splits);
  auto* op = reinterpret_cast<unsigned short*>(out.data_ptr());
#define PA_LAUNCH(NW_, FP8_, SP_)                                            \
  prompt_attn_kernel<NW_, FP8_, SP_><<<grid, NW_ * WAVE, 0, stream>>>(       \
      op, po, pml, reinterpret_cast<const unsigned short*>(q.data_ptr()),    \
      k_cache.data_ptr(), v_cache.data_ptr(), block_table.data_ptr<int>(),   \
      seq_lens.data_ptr<int>(), q_starts.data_ptr<int>(),                    \
      qb_seq.data_ptr<int>(), qb_start.data_ptr<int>(), q.stride(0),         \
      q_offset, out.stride(0), T, nqb, Hq, Hk, max_blocks, splits,           \
      (float)scale)
#define PA_LAUNCH2(NW_, SP_)                                                 \
  if (fp8) { PA_LAUNCH(NW_, true, SP_); } else { PA_LAUNCH(NW_, false, SP_); }
  if (pairs) {
    if (splits > 1) { PA_LAUNCH2(8, true) } else { PA_LAUNCH2(8, false) }
  } else {
    if (splits > 1) { PA_LAUNCH2(4, true) } else { PA_LAUNCH2(4, false) }
  }
#undef PA_LAUNCH2
#undef PA_LAUNCH
  HIP_CHECK_KERNEL();
  if (splits > 1) {
    prompt_attn_merge_kernel<<<dim3(nqb, 32, (Hq + 3) / 4), 256, 0, stream>>>(
        op, po, pml, seq_lens.data_ptr<int>(), q_starts.data_ptr<int>(),
        qb_seq.data_ptr<int>(), qb_start.data_ptr<int>(), out.stride(0), T,
        Hq, splits);
    HIP_CHECK_KERNEL();
  }
}

}  // namespace kukeon
