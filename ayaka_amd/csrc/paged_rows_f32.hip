// Multi-row attention for fp32 models (prompts and prefill chunks) on MI355X (gfx950): the
// rows of a request share each key and value read, and both products run on the matrix cores.
//
// Semantics: the decode entry point's over rows that carry positions (row n attends to
// positions [0, len_n) of its request; reference python/ayaka/ops/backends/torch/attention.py:
// 209-234 in fp32), scores, softmax and the value sum in fp32, the output written in fp32.
//
// Row by row (paged_attention_f32_kernel) a prompt of n rows reads its context n times and runs
// four FMAs per lane, key and head on the VALU. Here a workgroup serves one key/value head and a
// tile of PT x 16 (row, query head) pairs, consecutive in the order (row, head of the group); the
// tile's rows are walked request by request, each wave taking every W-th 16-position step of the
// context, and the waves' states meet in LDS in wave order. Both contractions are
// v_mfma_f32_16x16x4f32 (fp32 products and sums), so nothing is rounded to a shorter type. What
// bounds it: the chain of each wave's steps. A step of 16 positions takes 1.6 us at head_dim 64,
// 2.8 at 128 and 3.3 at 256 with 16 pairs, 2.6 and 3.1 with 32, of which the products' own rate
// (64 flops a cycle and SIMD, 157 TFLOP/s; a large fp32 product reaches 150 here) is about half at
// 64 with 16 pairs; large steps reach 54-65 TFLOP/s. A tile of prompts spans one request or two, but
// one of one-row requests up to 16 PT, each with its own pass over all columns, two barriers and a
// merge (3-5 us): such steps are left to the row kernel by the caller's launch model.
//
// Measured, us, row by row -> here: 2 prompts of 592 and 491 rows, 9/3 heads of 64, 54 -> 23; 32/8
// heads of 64, one chunk of 300 rows over 3000 positions, 364 -> 108 (65 TFLOP/s), 1000-row prompt
// 225 -> 71; 32/8 heads of 128, the same prompt, 504 -> 134; 16/8 heads of 256, 980 -> 152.
//
//  * No operand goes through LDS. S^T = K Q^T: the contraction index is free to permute, so lane
//    (mt, mq) of the key operand loads 16 contiguous bytes of position mt (dims 16 u + 4 mq + e)
//    and its four floats are four k-steps; q is held in the same order. A load instruction covers
//    64 contiguous bytes of each of 16 positions.
//  * O^T += V^T P^T: the scores of lane (mt, mq) are positions 4 mq + i of pair mt, which is the B
//    operand of k-step i when the contraction runs over positions 4 mq + i; the value operand's
//    rows are permuted (row mt of product t is dim 4 mt + t), so that a lane's 16-byte load feeds
//    four products, a load instruction covers whole 256-byte rows, and the lane's outputs are 16
//    contiguous dims.
//  * The sums of q.k run over 8 dims at a time, added pairwise, and each step's 16
//    positions of P.V are summed by themselves before they join the output: as exact as the row
//    kernel's tree over lanes and its partitions.
//
// A position that some pairs of the tile see and others do not may hold any value, infinities and
// NaN included, and 0 x inf is NaN: where a masked step holds such a value its positions are
// folded one at a time and each pair keeps the positions that it sees.

#include "attention_common.h"

namespace ayk {

// q.k over 8-dim pieces [LO, HI) of a lane's order (two products of four dims each), halves added
// pairwise.
template <int LO, int HI, int KU>
__device__ __forceinline__ f32x4 dims_sum(const f32x4 (&k)[KU], const f32x4 (&q)[KU]) {
  if constexpr (HI - LO > 1) {
    constexpr int MID = (LO + HI) / 2;
    return dims_sum<LO, MID>(k, q) + dims_sum<MID, HI>(k, q);
  } else {
    constexpr int u = LO / 2, e = LO % 2 * 2;
    const f32x4 a = __builtin_amdgcn_mfma_f32_16x16x4f32(k[u][e], q[u][e], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(k[u][e + 1], q[u][e + 1], a, 0, 0, 0);
  }
}

template <int D, int PT, int W>
__global__ __launch_bounds__(W * kWave) void paged_rows_f32_kernel(const AttnParams p) {
  constexpr int KU = D / 16;   // 16-byte key loads per lane and step
  constexpr int VC = D / 64;   // 16-byte value loads per lane and position
  constexpr int CH = rows_f32_step();
  constexpr int PAIRS = 16 * PT;
  __shared__ uint32_t s_tbl[kTableCap];
  __shared__ f32x4 s_o[W - 1][PT][VC * 4][kWave];
  __shared__ float s_m[W - 1][PAIRS], s_l[W - 1][PAIRS];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int mt = lane % 16, mq = lane / 16;
  const int kv_heads = p.num_heads / p.group;
  const int kvh = blockIdx.x % kv_heads;
  // the last rows (of a prompt, those with the longest contexts) start first
  const int tile = gridDim.x / kv_heads - 1 - blockIdx.x / kv_heads;
  const int first_pair = tile * PAIRS;
  const int n_pairs = p.n_rows * p.group;  // of one key/value head (the host keeps it below 2^31)

  int prow[PT], phead[PT], preq[PT], plen[PT];
  bool left[PT];  // pairs not yet computed
#pragma unroll
  for (int j = 0; j < PT; ++j) {
    const int pair = first_pair + j * 16 + mt;
    left[j] = pair < n_pairs;
    const int at = left[j] ? pair : n_pairs - 1;
    prow[j] = at / p.group;
    phead[j] = kvh * p.group + (at - prow[j] * p.group);
    row_context(p, prow[j], preq[j], plen[j]);
  }
  // q in the keys' k-order: dims 16 u + 4 mq + e of pair mt
  f32x4 qv[PT][KU];
#pragma unroll
  for (int j = 0; j < PT; ++j)
#pragma unroll
    for (int u = 0; u < KU; ++u)
      qv[j][u] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(p.q) +
                                                 ((int64_t)prow[j] * p.num_heads + phead[j]) * D + 16 * u + 4 * mq);

  const int seg_len = segment_positions(p, CH);
  const uint32_t token_stride = (uint32_t)p.token_stride;
  const float scale_log2 = p.scale_log2;
  const float* kbase = reinterpret_cast<const float*>(p.k_cache) + (int64_t)kvh * p.head_stride + 4 * mq;
  const float* vbase = reinterpret_cast<const float*>(p.v_cache) + (int64_t)kvh * p.head_stride + 4 * mt;

  for (;;) {
    // the next request with pairs left (the first left pair's), the same in every wave
    uint64_t waiting = 0;
    int group_of = 0;
#pragma unroll
    for (int j = PT - 1; j >= 0; --j) {
      const uint64_t b = __builtin_amdgcn_ballot_w64(left[j]);
      if (b) {
        waiting = b;
        group_of = j;
      }
    }
    if (!waiting) break;
    int req = 0;
#pragma unroll
    for (int j = 0; j < PT; ++j)
      if (group_of == j) req = __builtin_amdgcn_readlane(preq[j], __builtin_ctzll(waiting));
    bool mine[PT];
    int lim[PT];  // positions a pair of this request sees
    int t_end = 0, all_see = INT32_MAX;
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      mine[j] = left[j] && preq[j] == req;
      lim[j] = mine[j] ? plen[j] : 0;
      t_end = imax(t_end, lim[j]);
      if (mine[j]) all_see = imin(all_see, lim[j]);
    }
#pragma unroll
    for (int st = 1; st < kWave; st <<= 1) {
      t_end = imax(t_end, __shfl_xor(t_end, st));
      all_see = imin(all_see, __shfl_xor(all_see, st));
    }
    t_end = __builtin_amdgcn_readfirstlane(t_end);
    all_see = __builtin_amdgcn_readfirstlane(all_see);

    float m[PT], l[PT];
    f32x4 o[PT][VC * 4];
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      m[j] = kNoScore;
      l[j] = 0.f;
#pragma unroll
      for (int c = 0; c < VC * 4; ++c) o[j][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const int32_t* tbl = p.block_table + (int64_t)req * p.table_stride;
    for (int s0 = 0; s0 < t_end; s0 += seg_len) {
      const int s1 = imin(t_end, s0 + seg_len);
      const int b0 = stage_table(p, tbl, s_tbl, s0, s1, tid, W * kWave);
      const int nch = (s1 - s0 + CH - 1) / CH;
      auto load_keys = [&](int ci, f32x4(&k)[KU]) {
        const float* at = kbase + kv_offset(p, s_tbl, b0, chunk_position(s0, s1, ci, CH, 0, CH, mt), token_stride);
#pragma unroll
        for (int u = 0; u < KU; ++u) k[u] = *reinterpret_cast<const f32x4*>(at + 16 * u);
      };
      auto fold = [&](int ci, const f32x4(&k)[KU]) {
        const int tb = s0 + ci * CH;
        f32x4 v[4][VC];
        uint32_t off[4];
        prefill_offsets<4>(p, s_tbl, b0, tb + 4 * mq, s1, 0, token_stride, off);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int c = 0; c < VC; ++c) v[i][c] = *reinterpret_cast<const f32x4*>(vbase + off[i] + 64 * c);
        f32x4 s[PT];
#pragma unroll
        for (int j = 0; j < PT; ++j) {
          s[j] = dims_sum<0, 2 * KU>(k, qv[j]);
        }
        const bool whole = tb + CH <= all_see && tb + CH <= s1;  // uniform: every pair of the request sees the step
        bool grow = false;
        float mx[PT];
#pragma unroll
        for (int j = 0; j < PT; ++j) {
          mx[j] = -INFINITY;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            s[j][i] *= scale_log2;
            if (!whole && tb + 4 * mq + i >= lim[j]) s[j][i] = -INFINITY;
            mx[j] = fmaxf(mx[j], s[j][i]);
          }
          grow |= mx[j] > m[j] + kRescaleSlack;
        }
        if (__builtin_amdgcn_ballot_w64(grow)) {
#pragma unroll
          for (int j = 0; j < PT; ++j) {
            const float mn = fmaxf(m[j], column_max(mx[j]));
            const float alpha = fast_exp2(m[j] - mn);
            l[j] *= alpha;
#pragma unroll
            for (int c = 0; c < VC * 4; ++c) o[j][c] *= alpha;
            m[j] = mn;
          }
        }
#pragma unroll
        for (int j = 0; j < PT; ++j) {
#pragma unroll
          for (int i = 0; i < 4; ++i) s[j][i] = fast_exp2(s[j][i] - m[j]);
          l[j] += (s[j][0] + s[j][1]) + (s[j][2] + s[j][3]);
        }
        bool odd = false;  // a masked step with a value that is not finite
        if (!whole) {
          float z = 0.f;
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int c = 0; c < VC; ++c)
#pragma unroll
              for (int t = 0; t < 4; ++t) z = fmaf(v[i][c][t], 0.f, z);
          odd = __builtin_amdgcn_ballot_w64(z != 0.f) != 0;  // finite values leave 0
        }
        if (!odd) {
          // a step's 16 positions are summed by themselves and added once
#pragma unroll
          for (int c = 0; c < VC; ++c) {
            f32x4 part[PT][4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int j = 0; j < PT; ++j)
                  part[j][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                      v[i][c][t], s[j][i], i == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : part[j][t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
              for (int j = 0; j < PT; ++j) o[j][c * 4 + t] += part[j][t];
          }
        } else {
          // one position per product: the other three k-slots hold zeros on both sides
#pragma unroll 1
          for (int g = 0; g < 4; ++g) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int c = 0; c < VC; ++c)
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                  for (int j = 0; j < PT; ++j) {
                    const f32x4 was = o[j][c * 4 + t];
                    const f32x4 now = __builtin_amdgcn_mfma_f32_16x16x4f32(mq == g ? v[i][c][t] : 0.f,
                                                                            mq == g ? s[j][i] : 0.f, was, 0, 0, 0);
                    o[j][c * 4 + t] = tb + 4 * g + i < lim[j] ? now : was;
                  }
          }
        }
      };
      if (wave < nch) {
        const int last = last_chunk_of_slice(nch, wave, W);
        f32x4 ka[KU];
        if constexpr (D == 256) {  // (two steps' keys would not fit the registers)
          for (int ci = wave; ci <= last; ci += W) {
            load_keys(ci, ka);
            fold(ci, ka);
          }
        } else {
          // the next step's keys are in flight while the current step is folded
          f32x4 kb[KU];
          int ci = wave;
          load_keys(ci, ka);
          for (;;) {
            load_keys(imin(ci + W, last), kb);
            fold(ci, ka);
            ci += W;
            if (ci > last) break;
            load_keys(imin(ci + W, last), ka);
            fold(ci, kb);
            ci += W;
            if (ci > last) break;
          }
        }
      }
    }
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      l[j] += __shfl_xor(l[j], 16);
      l[j] += __shfl_xor(l[j], 32);
    }
    __syncthreads();  // the previous request's states have been read
    if (wave > 0) {
#pragma unroll
      for (int j = 0; j < PT; ++j) {
#pragma unroll
        for (int c = 0; c < VC * 4; ++c) s_o[wave - 1][j][c][lane] = o[j][c];
        if (mq == 0) {
          s_m[wave - 1][j * 16 + mt] = m[j];
          s_l[wave - 1][j * 16 + mt] = l[j];
        }
      }
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int j = 0; j < PT; ++j) {
        float mn = m[j];
#pragma unroll
        for (int w = 0; w < W - 1; ++w) mn = fmaxf(mn, s_m[w][j * 16 + mt]);
        const float a0 = fast_exp2(m[j] - mn);
        float lsum = l[j] * a0;
#pragma unroll
        for (int c = 0; c < VC * 4; ++c) o[j][c] *= a0;
        for (int w = 0; w < W - 1; ++w) {
          const float a = fast_exp2(s_m[w][j * 16 + mt] - mn);
          lsum += s_l[w][j * 16 + mt] * a;
#pragma unroll
          for (int c = 0; c < VC * 4; ++c) o[j][c] += s_o[w][j][c][lane] * a;
        }
        const float inv = (lsum > 0.f ? 1.0f / lsum : 0.f) * p.v_scale;
        if (mine[j]) {
          float* out = static_cast<float*>(p.out) + ((int64_t)prow[j] * p.num_heads + phead[j]) * D + 16 * mq;
#pragma unroll
          for (int c = 0; c < VC; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              *reinterpret_cast<f32x4*>(out + 64 * c + 4 * i) = f32x4{o[j][c * 4][i] * inv, o[j][c * 4 + 1][i] * inv,
                                                                       o[j][c * 4 + 2][i] * inv, o[j][c * 4 + 3][i] * inv};
        }
      }
    }
#pragma unroll
    for (int j = 0; j < PT; ++j) left[j] = left[j] && !mine[j];
  }
}

template <int D, int PT, int W>
static hipError_t launch_rows_f32_typed(const AttnParams& p, int64_t tiles, hipStream_t stream) {
  hipLaunchKernelGGL((paged_rows_f32_kernel<D, PT, W>), dim3((unsigned)(tiles * (p.num_heads / p.group))),
                     dim3(W * kWave), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_rows_f32(const AttnParams& p, int head_dim, int compute_units, hipStream_t stream) {
  const int pt = rows_f32_groups(p, head_dim, compute_units);
  const int64_t tiles = rows_f32_tiles(p, pt);
  switch (head_dim) {
    case 64:
      return pt == 2 ? launch_rows_f32_typed<64, 2, rows_f32_waves(64, 2)>(p, tiles, stream)
                     : launch_rows_f32_typed<64, 1, rows_f32_waves(64, 1)>(p, tiles, stream);
    case 128:
      return pt == 2 ? launch_rows_f32_typed<128, 2, rows_f32_waves(128, 2)>(p, tiles, stream)
                     : launch_rows_f32_typed<128, 1, rows_f32_waves(128, 1)>(p, tiles, stream);
    case 256: return launch_rows_f32_typed<256, 1, rows_f32_waves(256, 1)>(p, tiles, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ayk
