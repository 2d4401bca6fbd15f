// Chunked-prefill attention tiles on CDNA4 matrix cores in fp32 (head_dim 64 and 128).
//
// A work item is (request, kv head, query tile of up to 16 QW virtual rows, KV split); virtual row
// rho is query token qb + rho / n_rep of query head h * n_rep + rho % n_rep. The four waves of a
// workgroup share the item's rows and split its keys (16 at a time, in turn); their (m, l, O) merge
// in LDS at the end, so that short prompts, a few hundred keys and a few hundred tiles, still
// put four waves on every SIMD pair.
//
// Everything stays fp32: products and sums on v_mfma_f32_16x16x4_f32, whose operands hold one
// value a lane. No operand passes through LDS: the contraction indexes are permuted so that a 16-
// byte load is four operands.
//   * S^T = K Q^T: lane (key r = lane % 16, g = lane / 16) loads dims 16 j + 4 g .. + 3 of its key,
//     element e being the A operand of step (j, e); Q is held the same way.
//   * O^T += V^T P^T: step i contracts keys {4 g + i}. Lane (r, g) loads dims 4 r .. + 3 of key
//     4 g + i, element t being the A operand of output tile t (dims 4 r + t); the probability of
//     key 4 g + i is S register i of the same lane.
// Keys without a valid block load zeros (out-of-range buffer offsets) and are masked.
//
// Bound by the fp32 matrix rate (64 FLOP a cycle and SIMD, 157 TFLOP/s on the chip) once the chip
// is full, by the length of one wave's chain of chunks below that. 9/3 heads of 64, two prompts of
// 300 tokens at 300 and 511 keys with 4 decodes: step 675 us on the row kernel -> 30 us; two 512-token slices, 32/8
// heads of 128, at 2,048 and 4,096 keys 524 us (90 TFLOP/s).
#include "attention_merge.h"
#include "attention_plan.h"

namespace edgerag {
namespace {

using namespace plan;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * kWave;
constexpr int kKeys = 16;            // keys per chunk
constexpr float kRescaleLog2 = 8.f;  // the reference max moves when a score beats it by 2^8
constexpr uint32_t kOutOfRange = 0xFFFFF000u;  // byte offset past any head's slice

struct Slice {
  const void* base;
  uint32_t bytes;
};

// 16 bytes at byte offset `off` of the slice, zeros past its end.
__device__ __forceinline__ f32x4 load_slice(Slice s, uint32_t off) {
  return __builtin_bit_cast(
      f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                 __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(s.base), 0, s.bytes,
                                                   0x00020000),
                 off, 0, 0));
}

// max of v over the four lanes that differ in lane / 16: the swaps pair rows of 16 lanes, then
// halves of the wave, in VALU ops.
__device__ __forceinline__ float groups_max(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float groups_sum(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

template <int D, int QW>
__global__ __launch_bounds__(kThreads) void attn_prefill_f32_kernel(
    const int32_t* __restrict__ plan, int32_t item_base, int32_t bs_shift,
    const int32_t* __restrict__ qsl, const int32_t* __restrict__ ctx,
    const int32_t* __restrict__ block_tables, int64_t bt_stride, int32_t num_blocks,
    int32_t n_q_heads, const float* __restrict__ q, int64_t q_st, int64_t q_sh,
    const float* __restrict__ kpool, const float* __restrict__ vpool, int32_t n_kv_heads,
    float scale_log2, float* __restrict__ out, int64_t o_st, int64_t o_sh,
    float2* __restrict__ part_ml, float* __restrict__ part_acc) {
  // Sums per 16 dims of a score, and per output element: shorter chains of fp32 additions. Error
  // of the outputs against float64 (300 tokens at 300 / 511 keys, head_dim 64; the row kernel
  // 1.50e-7): one chain each 1.6e-7, two sums 1.5e-7, two outputs as well 1.36e-7 (15.8 against
  // 14.6 us). At head_dim 128 one of each is below the row kernel already (2.2e-7 against 3.0e-7).
  constexpr int kSums = D == 64 ? 2 : 1, kOut = D == 64 ? 2 : 1;
  constexpr int kKj = D / 16;  // 16-byte loads of K per lane and chunk
  constexpr int kVu = D / 64;  // 16-byte loads of V per lane and key
  constexpr int kRows = 16 * QW;
  __shared__ uint32_t sblk[kMaxTileBlocks];  // byte offset of each block in the head's slice
  __shared__ float sm[kWaves][kRows], sl[kWaves][kRows];
  __shared__ __align__(16) float so[kWaves][kRows][D + 4];

  const int32_t* it = plan + plan[H_ITEM_OFF] + int64_t(item_base + blockIdx.x) * kItemWords;
  const int r = it[I_REQ], h = it[I_HEAD], qb = it[I_QBEGIN], qc = it[I_QCOUNT];
  const int kb = it[I_KVBEGIN], ke = it[I_KVEND], split = it[I_SPLIT];
  const int32_t* rq = plan + plan[H_REQ_OFF] + r * kReqWords;
  const int nsplit = rq[R_NSPLIT], part_off = rq[R_PARTOFF], pstride = rq[R_PSTRIDE];
  const int q0 = qsl[r], c = qsl[r + 1] - q0, L = ctx[r];
  const int n_rep = n_q_heads / n_kv_heads;
  const int32_t* table = block_tables + int64_t(r) * bt_stride;
  const int64_t head_base = int64_t(h) * num_blocks;
  const int bs_mask = (1 << bs_shift) - 1, blk0 = kb >> bs_shift;
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int g = lane / 16, col = lane % 16;
  const int nrows = qc * n_rep;

  int any_bad = 0;
  {
    const int nblk = min(((ke - 1) >> bs_shift) - blk0 + 1, kMaxTileBlocks);
    for (int i = tid; i < nblk; i += kThreads) {
      const int32_t b = table[blk0 + i];
      const bool ok = b >= 0 && b < num_blocks;
      sblk[i] = ok ? (uint32_t(b) << bs_shift) * uint32_t(D * 4) : kOutOfRange;
      any_bad |= ok ? 0 : 1;
    }
  }
  const bool item_has_bad = __syncthreads_or(any_bad) != 0;

  int lim[QW];         // last visible key position of this lane's row
  f32x4 qop[QW][kKj];  // dims 16 j + 4 g .. + 3, times scale * log2(e) as in the row kernel
#pragma unroll
  for (int w = 0; w < QW; ++w) {
    const int rho = 16 * w + col;
    const bool active = rho < nrows;
    const int t = qb + (active ? rho / n_rep : 0);
    const int hq = h * n_rep + (active ? rho % n_rep : 0);
    lim[w] = active ? L - c + (t - q0) : -1;
    const float* qp = q + int64_t(t) * q_st + int64_t(hq) * q_sh + 4 * g;
#pragma unroll
    for (int j = 0; j < kKj; ++j)
      qop[w][j] = active ? *reinterpret_cast<const f32x4*>(qp + 16 * j) * scale_log2 : f32x4{};
  }
  const int min_lim = L - c + (qb - q0);  // chunks ending at or below it need no causal mask
  f32x4 o[QW][kOut][4 * kVu];
  float m[QW], l[QW], nm[QW];
#pragma unroll
  for (int w = 0; w < QW; ++w) {
#pragma unroll
    for (int n = 0; n < kOut * 4 * kVu; ++n) o[w][n / (4 * kVu)][n % (4 * kVu)] = f32x4{};
    m[w] = -INFINITY;
    l[w] = nm[w] = 0.f;
  }
  const uint32_t head_bytes = uint32_t((int64_t(num_blocks) << bs_shift) * D * 4);
  const Slice ks{kpool + (head_base << bs_shift) * D, head_bytes};
  const Slice vs{vpool + (head_base << bs_shift) * D, head_bytes};

  // Byte offset of key position pos in the head's slice (past it for a key without a block).
  auto row_offset = [&](int pos) {
    const uint32_t blk = sblk[min((pos >> bs_shift) - blk0, kMaxTileBlocks - 1)];
    return pos < ke ? __builtin_elementwise_add_sat(blk, uint32_t(pos & bs_mask) * uint32_t(D * 4))
                    : kOutOfRange;
  };
  auto load_chunk = [&](int k0, f32x4 (&kr)[kKj], f32x4 (&vr)[4][kVu]) {
    const uint32_t ko = row_offset(k0 + col);
#pragma unroll
    for (int j = 0; j < kKj; ++j)
      kr[j] = load_slice(ks, __builtin_elementwise_add_sat(ko, uint32_t(64 * j + 16 * g)));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t vo = row_offset(k0 + 4 * g + i);
#pragma unroll
      for (int u = 0; u < kVu; ++u)
        vr[i][u] = load_slice(vs, __builtin_elementwise_add_sat(vo, uint32_t(256 * u + 16 * col)));
    }
  };
  auto chunk = [&](int k0, const f32x4 (&kr)[kKj], const f32x4 (&vr)[4][kVu]) {
    // One sum per 16 (or 8) dims, added in pairs: no MFMA waits for the one before it.
    f32x4 sj[QW][kKj * kSums];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int j = 0; j < kKj; ++j)
#pragma unroll
        for (int w = 0; w < QW; ++w) {
          f32x4& d = sj[w][j * kSums + e % kSums];
          d = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[j][e], qop[w][j][e],
                                                   e < kSums ? f32x4{} : d, 0, 0, 0);
        }
    f32x4 s[QW];
#pragma unroll
    for (int w = 0; w < QW; ++w) {
#pragma unroll
      for (int n = kKj * kSums / 2; n > 0; n /= 2)
#pragma unroll
        for (int j = 0; j < n; ++j) sj[w][j] += sj[w][j + n];
      s[w] = sj[w][0];
      // log2-domain scores relative to the reference max; register i holds key 4 g + i.
#pragma unroll
      for (int i = 0; i < 4; ++i) s[w][i] += nm[w];
      if (k0 + kKeys - 1 > min_lim || k0 + kKeys > ke || item_has_bad) {
        const int vis_end = min(ke, lim[w] + 1) - k0 - 4 * g;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          bool hide = i >= vis_end;
          if (item_has_bad)
            hide |= sblk[min((min(k0 + 4 * g + i, ke - 1) >> bs_shift) - blk0,
                             kMaxTileBlocks - 1)] == kOutOfRange;
          if (hide) s[w][i] = -INFINITY;
        }
      }
      const float tmax =
          groups_max(fmaxf(fmaxf(s[w][0], s[w][1]), fmaxf(s[w][2], s[w][3])));
      const bool first = m[w] == -INFINITY;
      const bool up = first ? tmax != -INFINITY : tmax > kRescaleLog2;
      if (__any(up)) {
        const float shift = up ? tmax : 0.f;
        const float alpha = first ? (up ? 0.f : 1.f) : exp2_fast(-shift);
        if (up) m[w] = first ? tmax : m[w] + tmax;
        nm[w] = m[w] == -INFINITY ? 0.f : -m[w];
        l[w] *= alpha;
#pragma unroll
        for (int n = 0; n < kOut * 4 * kVu; ++n) o[w][n / (4 * kVu)][n % (4 * kVu)] *= alpha;
#pragma unroll
        for (int i = 0; i < 4; ++i) s[w][i] -= shift;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[w][i] = exp2_fast(s[w][i]);
        l[w] += s[w][i];
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int u = 0; u < kVu; ++u)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int w = 0; w < QW; ++w)
            o[w][i % kOut][4 * u + t] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                vr[i][u][t], s[w][i], o[w][i % kOut][4 * u + t], 0, 0, 0);
  };

  // The next chunk's loads are in flight while a chunk is computed (past the split they load
  // zeros).
  f32x4 k0r[kKj], v0r[4][kVu], k1r[kKj], v1r[4][kVu];
  constexpr int kStep = kWaves * kKeys;
  load_chunk(kb + wave * kKeys, k0r, v0r);
  for (int k0 = kb + wave * kKeys; k0 < ke; k0 += 2 * kStep) {
    load_chunk(k0 + kStep, k1r, v1r);
    issue_fence();
    chunk(k0, k0r, v0r);
    if (k0 + kStep >= ke) break;
    load_chunk(k0 + 2 * kStep, k0r, v0r);
    issue_fence();
    chunk(k0 + kStep, k1r, v1r);
  }

  // Merge of the waves. Register i of O tile 4 u + t holds dim 64 u + 16 g + 4 i + t.
#pragma unroll
  for (int w = 0; w < QW; ++w) {
    const float lw = groups_sum(l[w]);
#pragma unroll
    for (int n = 1; n < kOut; ++n)
#pragma unroll
      for (int t = 0; t < 4 * kVu; ++t) o[w][0][t] += o[w][n][t];
    if (g == 0) {
      sm[wave][16 * w + col] = m[w];
      sl[wave][16 * w + col] = lw;
    }
#pragma unroll
    for (int u = 0; u < kVu; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<f32x4*>(&so[wave][16 * w + col][64 * u + 16 * g + 4 * i]) =
            f32x4{o[w][0][4 * u][i], o[w][0][4 * u + 1][i], o[w][0][4 * u + 2][i],
                  o[w][0][4 * u + 3][i]};
  }
  __syncthreads();
  const bool vec_out =
      (reinterpret_cast<uintptr_t>(out) & 15) == 0 && o_st % 4 == 0 && o_sh % 4 == 0;
  for (int i = tid; i < kRows * (D / 4); i += kThreads) {
    const int rho = i / (D / 4), d = i % (D / 4) * 4;
    if (rho >= nrows) break;
    float mx = -INFINITY, lsum = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) mx = fmaxf(mx, sm[w][rho]);
    f32x4 acc = {};
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float mw = sm[w][rho];
      const float wgt = mw == -INFINITY ? 0.f : exp2_fast(mw - mx);
      lsum = __builtin_fmaf(wgt, sl[w][rho], lsum);
      const f32x4 v = *reinterpret_cast<const f32x4*>(&so[w][rho][d]);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(wgt, v[e], acc[e]);
    }
    const int t = qb + rho / n_rep, hq = h * n_rep + rho % n_rep;
    // A key that a row does not see has p = 0, and 0 times a NaN or infinite V is NaN: a later
    // token's V must not reach the rows before it. Where one did, the row's keys are summed again.
    const float odd = (acc[0] + acc[1] + acc[2] + acc[3]) * 0.f;
    if (odd != 0.f) {
      const int seen = min(ke, L - c + (t - q0) + 1);
      bool hidden = false;
      for (int pos = max(kb, seen); pos < ke; ++pos) {
        const f32x4 v = load_slice(vs, __builtin_elementwise_add_sat(row_offset(pos), uint32_t(4 * d)));
        for (int e = 0; e < 4; ++e) hidden |= !(__builtin_fabsf(v[e]) < INFINITY);
      }
      if (hidden) {
        const float* qp = q + int64_t(t) * q_st + int64_t(hq) * q_sh;
        acc = f32x4{};
        for (int pos = kb; pos < seen; ++pos) {
          const uint32_t off = row_offset(pos);
          if (off >= head_bytes) continue;
          float dot = 0.f;
          for (int e = 0; e < D; e += 4) {
            const f32x4 k = load_slice(ks, off + uint32_t(4 * e));
            for (int x = 0; x < 4; ++x) dot = __builtin_fmaf(qp[e + x] * scale_log2, k[x], dot);
          }
          const float p = exp2_fast(dot - mx);
          const f32x4 v = load_slice(vs, off + uint32_t(4 * d));
          for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(p, v[e], acc[e]);
        }
      }
    }
    if (nsplit == 1) {
      const float inv = 1.f / fmaxf(lsum, 1.17549435e-38f);
      float* dst = out + int64_t(t) * o_st + int64_t(hq) * o_sh + d;
      if (vec_out) {
        *reinterpret_cast<f32x4*>(dst) = acc * inv;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[e] = acc[e] * inv;
      }
    } else {
      const int64_t idx = int64_t(part_off) + (int64_t(t - q0) * n_q_heads + hq) * pstride + split;
      if (d == 0) part_ml[idx] = make_float2(mx, lsum);
      *reinterpret_cast<f32x4*>(part_acc + idx * D + d) = acc;
    }
  }
}

template <int D, int QW>
void launch(const AttnLaunch& a, int item_base, int count) {
  hipLaunchKernelGGL((attn_prefill_f32_kernel<D, QW>), dim3(count), dim3(kThreads), 0, a.s,
                     a.plan, item_base, log2_exact(a.bs), a.qsl, a.ctx, a.bt, a.bt_stride, a.nb,
                     a.hq, static_cast<const float*>(a.q), a.q_st, a.q_sh,
                     static_cast<const float*>(a.kp), static_cast<const float*>(a.vp), a.hkv,
                     a.scale_log2, static_cast<float*>(a.out), a.o_st, a.o_sh, a.ml, a.pacc);
}

}  // namespace

bool prefill_f32_supported(int32_t num_blocks, int32_t block_size, int32_t head_dim) {
  // Power-of-two blocks (shift addressing); one kv head's slice of a pool below kOutOfRange.
  return (head_dim == 64 || head_dim == 128) && log2_exact(block_size) >= 0 &&
         int64_t(num_blocks) * block_size * head_dim * 4 < int64_t(kOutOfRange);
}

void launch_prefill_f32(const AttnLaunch& a, int32_t head_dim, int rows, int item_base, int count) {
  if (head_dim == 64) {
    if (rows <= 16) launch<64, 1>(a, item_base, count);
    else launch<64, 2>(a, item_base, count);
  } else {
    if (rows <= 16) launch<128, 1>(a, item_base, count);
    else launch<128, 2>(a, item_base, count);
  }
}

}  // namespace edgerag
