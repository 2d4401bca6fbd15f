// Decode rows of grouped-query attention on CDNA4 matrix cores (fp16 and bf16, head_dim 64 and 128).
//
// A row item is (request, kv head, keys) with 2 to 8 query vectors (new tokens x heads of the
// group). The VALU kernel (attn_decode_kernel) spends 2 D operations per key, value and query
// vector, so past one vector its time goes to arithmetic instead of to the stream of K and V. Here
// a wave takes 32 keys a step:
//   * S^T = K Q^T with v_mfma_f32_16x16x32: K goes from the pool to the A operand in registers
//     (lane (key, g = lane / 16) loads dims 32 ks + 8 g .. + 7); Q is held as B, the up to 8
//     vectors in columns 0-7 and again in 8-15 (bf16, up to 4 vectors: in each 4 columns).
//   * softmax in the log2 domain, the reference max raised lazily (Elem::kRaiseLog2).
//   * O^T += V^T P^T with the same MFMA. The columns left over hold the rest of each p: fp16 takes
//     two parts (8 columns each: at least 22 bits down to the floor beside kTopLog2), bf16 three, the
//     24 bits of fp32: of up to 4 vectors in 4 columns each, of 5 to 8 in 8 columns each and a
//     second MFMA for the third part. The parts of O add up at the end; l sums the fp32 p. V goes
//     from the pool straight into a buffer of the wave in LDS (no staging registers) and is read
//     transposed (ds_read_b64_tr_b16).
// The next step's K (registers) and V (the other LDS buffer) are in flight while a step is
// computed (as compiled, the exit in the middle of the loop and the branches that the block offsets
// become make a wave wait for some of those K loads early); waves do not wait for each other before
// the merge. Items are run as attn_decode_kernel
// runs them: one wave per KV split, or a workgroup whose waves split the item's keys and merge in
// LDS. A fused append stores the item's new rows to their slots first and reads them back from the
// pool, unless a slot is not the row's place in the block table (a padded token's negative slot):
// the item's new rows then come from the caller's rows, key by key after the others.
//
// Bound by the K/V stream at large batches (bf16 32/8 heads of 128, 48 requests of 256-8,192
// tokens, 870 MB, append, rows and merge in a stream of steps: 175.5 -> 156.9 us, 5.5 TB/s; the rows'
// launch replayed alone from a graph 213 -> 159), by the chain of one wave's steps in small ones (one
// request of 2,048 tokens 18.0 -> 9.6 us, 32 requests with 9/3 heads of 64 44.8 -> 25.2 us).
#include "attention_merge.h"
#include "attention_plan.h"

namespace edgerag {
namespace {

using namespace plan;

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kVecs = 8;             // query vectors of an item
constexpr int kKeys = 32;            // keys per step: two 16-key MFMA tiles
constexpr uint32_t kOutOfRange = 0xFFFFF000u;

// Cache policy of the K and V loads: non-temporal, a launch reads each byte once (48 requests,
// 870 MB: 171 -> 159 us; batches small enough to stay in the last-level cache between launches,
// which a model's layers do not, lose 2 to 4%).
constexpr int kStream = 2;

struct Slice {
  const void* base;
  uint32_t bytes;
};
__device__ __forceinline__ u32x4 load_slice(Slice s, uint32_t off) {
  return __builtin_bit_cast(
      u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                 __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(s.base), 0, s.bytes,
                                                   0x00020000),
                 off, 0, kStream));
}
// 16 bytes a lane from byte offset `off` of the slice (zeros past its end) to dst + 16 lane in LDS.
__device__ __forceinline__ void load_lds16(Slice s, char* dst, uint32_t off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(s.base), 0, s.bytes, 0x00020000),
      (__attribute__((address_space(3))) void*)dst, 16, off, 0, 0, kStream);
}

template <typename T>
struct Elem;
template <>
struct Elem<f16> {
  typedef h8 v8;
  // log2 of the p of a vector's largest score, and of the p past which its reference moves. fp16
  // subnormals end at 2^-24, so hi + lo is off by up to 2^-25 however small p is: 2^-36 of the
  // largest p here, with at least 22 bits of every p above 2^-14 of it. (Held at 2^0, keys below
  // 2^-25 of the largest dropped out of O while l counted them.)
  static constexpr float kTopLog2 = 11.f, kRaiseLog2 = 15.f;
  static __device__ __forceinline__ f32x4 mfma(v8 a, v8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t round2(float a, float b) {
    return __builtin_bit_cast(uint32_t, h2{_Float16(a), _Float16(b)});
  }
  static __device__ __forceinline__ float lo(uint32_t w) {
    return float(__builtin_bit_cast(h2, w)[0]);
  }
  static __device__ __forceinline__ float hi(uint32_t w) {
    return float(__builtin_bit_cast(h2, w)[1]);
  }
};
template <>
struct Elem<bf16> {
  typedef b8 v8;
  static constexpr float kTopLog2 = 0.f, kRaiseLog2 = 8.f;  // the exponents of fp32
  static __device__ __forceinline__ f32x4 mfma(v8 a, v8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

constexpr uint32_t kUpper = 0xFFFF0000u;
// v less the part of it in the bits of the mask.
__device__ __forceinline__ float less_upper(float v, uint32_t mask) {
  return v - __uint_as_float(__float_as_uint(v) & mask);
}
// The upper halves of a and b in one word.
__device__ __forceinline__ uint32_t uppers(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302);
}

// max / sum over the four lanes that differ in lane / 16.
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
// v of the lane N places on in the same row of 16 (row_shl; 0 past its end).
template <int N>
__device__ __forceinline__ float row_ahead(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x100 + N, 0xF, 0xF,
                                                    true));
}

// Slot of chunk c of key k in a V buffer row is c ^ v_swizzle(k): 32 lanes of a transposing read
// take 32 bytes (2 chunks) of each of 8 consecutive rows, which must cover all 256 bytes of banks
// (rows of head_dim 64 alternate between the two halves already).
template <int D>
__device__ __forceinline__ int v_swizzle(int key) {
  return D == 64 ? ((key >> 1) & 3) << 1 : (key & 7) << 1;
}

// NW: waves per workgroup (1: one wave per item). VC: columns of a part of the probabilities, 8, or 4
// for bf16 rows of up to 4 vectors.
template <typename T, int D, int NW, int VC>
__global__ __launch_bounds__(NW * kWave) __attribute__((amdgpu_waves_per_eu(2)))
void attn_decode_gqa_kernel(
    const int32_t* __restrict__ plan, int32_t item_base, int32_t limit_word,
    const int32_t* __restrict__ qsl, const int32_t* __restrict__ ctx,
    const int32_t* __restrict__ block_tables, int64_t bt_stride, int32_t num_blocks,
    int32_t block_size, const T* __restrict__ q, int64_t q_st, int64_t q_sh,
    const T* kpool, const T* vpool, int32_t n_q_heads, int32_t n_kv_heads, float scale_log2,
    T* __restrict__ out, int64_t o_st, int64_t o_sh, float2* __restrict__ part_ml,
    float* __restrict__ part_acc, const T* __restrict__ nk, const T* __restrict__ nv,
    int64_t n_st, int64_t n_sh, const int32_t* __restrict__ slots, T* kdst, T* vdst) {
  using E = Elem<T>;
  typedef typename E::v8 v8;
  constexpr bool kThree = __is_same(T, bf16);  // probabilities in three parts
  constexpr int kKs = D / 32, kDt = D / 16, kCh = D / 8;
  constexpr int kKpi = kWave / kCh;        // keys a V load covers
  constexpr int kVLoads = kKeys / kKpi;
  constexpr int kBuf = kKeys * D * 2;      // bytes of a V buffer
  static_assert(kVecs * D * 4 <= kBuf, "the merge reuses a wave's V buffer");
  // Two arrays, not one with an index: a load into one is then known not to alias the other.
  __shared__ __align__(16) char sv0[NW * kBuf], sv1[NW * kBuf];
  __shared__ float sml[NW][kVecs][2];

  const int64_t idx = int64_t(item_base) + blockIdx.x;
  if (idx >= plan[limit_word]) return;
  const int32_t* it = plan + kHeaderWords + idx * kItemWords;
  const int r = it[I_REQ], h = it[I_HEAD], qb = it[I_QBEGIN], qc = it[I_QCOUNT];
  int kb = it[I_KVBEGIN], ke = it[I_KVEND];
  const int split = it[I_SPLIT];
  const int32_t* rq = plan + plan[H_REQ_OFF] + r * kReqWords;
  const int lane = threadIdx.x % kWave;
  const int wave = NW > 1 ? __builtin_amdgcn_readfirstlane(int(threadIdx.x / kWave)) : 0;
  if constexpr (NW > 1) {
    // This wave's part: equal parts of whole blocks, empty for waves past the end.
    const int per = (ke - kb + NW - 1) / NW;
    const int part = (per + block_size - 1) / block_size * block_size;
    const int b0 = min(ke, kb + wave * part);
    ke = min(ke, b0 + part);
    kb = b0;
  }
  // Block ids of the wave's keys, one per lane.
  const int nblk = (ke - kb + block_size - 1) / block_size;
  int32_t my_blk = -1;
  if (nblk > 0)
    my_blk = block_tables[int64_t(r) * bt_stride + kb / block_size + min(lane, nblk - 1)];
  const int nsplit = rq[R_NSPLIT], part_off = rq[R_PARTOFF], pstride = rq[R_PSTRIDE];
  const int q0 = qsl[r], c = qsl[r + 1] - q0, L = ctx[r];
  if (lane >= nblk || my_blk >= num_blocks) my_blk = -1;
  const int n_rep = n_q_heads / n_kv_heads;
  const int nvec = qc * n_rep;
  const int g = lane / 16, col = lane % 16;
  // This lane's column holds part `part` of the probabilities of vector `vec`.
  const int part = col / VC, vec = col % VC;
  const bool active = vec < nvec;
  const uint32_t mask1 = part >= 1 ? kUpper : 0, mask2 = part >= 2 ? kUpper : 0;
  const uint32_t third_mask = part == 0 ? ~0u : 0;
  const int t = qb + (active ? vec / n_rep : 0);
  const int hq = h * n_rep + (active ? vec % n_rep : 0);
  const int lim = active ? L - c + (t - q0) : -1;
  const int min_lim = L - c + (qb - q0);

  const int64_t head_base = int64_t(h) * num_blocks * block_size;
  const uint32_t head_bytes = uint32_t(int64_t(num_blocks) * block_size * D * 2);
  const Slice ks{kpool + head_base * D, head_bytes}, vs{vpool + head_base * D, head_bytes};

  bool detached = false;   // a new row's slot is not its place in the block table
  const int ke_new = ke;
  if (nk != nullptr && ke > L - c && kb < ke) {
    // The new rows among this wave's keys go to their slots, and are read back below (same wave,
    // after the stores are done).
    for (int pos = max(kb, L - c); pos < ke; ++pos) {
      const int64_t tok = q0 + (pos - (L - c));
      const int64_t slot = slots[tok];
      if (lane < 2 * kCh && slot >= 0 && slot < int64_t(num_blocks) * block_size) {
        const T* src = (lane < kCh ? nk : nv) + tok * n_st + int64_t(h) * n_sh + lane % kCh * 8;
        T* dst = (lane < kCh ? kdst : vdst) + (head_base + slot) * D + lane % kCh * 8;
        store16(dst, load16(src));
      }
      const int bi = (pos - kb) / block_size;
      const int blk = __builtin_amdgcn_readlane(my_blk, bi);
      detached |= blk >= 0 && slot != int64_t(blk) * block_size + (pos - kb - bi * block_size);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (detached) ke = max(kb, L - c);  // the loop takes the keys before the new rows
  }

  v8 qop[kKs];
  {
    const T* qp = q + int64_t(t) * q_st + int64_t(hq) * q_sh + 8 * g;
#pragma unroll
    for (int s = 0; s < kKs; ++s)
      qop[s] = active ? *reinterpret_cast<const v8*>(qp + 32 * s) : v8{};
  }
  f32x4 o[kDt];
#pragma unroll
  for (int dt = 0; dt < kDt; ++dt) o[dt] = f32x4{};
  float m = -INFINITY, l = 0.f, nm = 0.f;

  // The load cursor: block index and row in the block of the next 16-key tile.
  int cur_blk = 0, cur_row = 0;
  // Byte offset of row `key` of the tile at tile_row (invalid or past the split: out of range).
  auto next_tile = [&](int& blk, int& row) {
    blk = __builtin_amdgcn_readlane(my_blk, min(cur_blk, kWave - 1));
    row = blk * block_size + cur_row;
    cur_row += 16;
    if (cur_row >= block_size) {
      cur_row = 0;
      ++cur_blk;
    }
  };
  auto load_step = [&](int k0, u32x4 (&kr)[2][kKs], char* sv) {
    int blk[2], row[2];
    next_tile(blk[0], row[0]);
    next_tile(blk[1], row[1]);
#pragma unroll
    for (int tl = 0; tl < 2; ++tl) {
      const uint32_t off = blk[tl] >= 0 && k0 + 16 * tl + col < ke
                               ? uint32_t(row[tl] + col) * uint32_t(D * 2) + uint32_t(16 * g)
                               : kOutOfRange;
#pragma unroll
      for (int s = 0; s < kKs; ++s) kr[tl][s] = load_slice(ks, off + uint32_t(64 * s));
    }
#pragma unroll
    for (int j = 0; j < kVLoads; ++j) {
      const int tl = kKpi * j / 16;
      const int key = kKpi * j + lane / kCh;  // in the step
      const int chunk = (lane % kCh) ^ v_swizzle<D>(key);
      const uint32_t off = blk[tl] >= 0 && k0 + key < ke
                               ? uint32_t(row[tl] + key % 16) * uint32_t(D * 2) + uint32_t(16 * chunk)
                               : kOutOfRange;
      load_lds16(vs, sv + j * 1024, off);
    }
  };
  auto read_v = [&](const char* sv, int dt) {
    union {
      s4 half[2];
      v8 all;
    } u;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int key = 16 * i + 4 * g + col / 4;
      const int dim = 16 * dt + 4 * (col % 4);
      u.half[i] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s4*)(sv + key * (D * 2) +
                                                  16 * ((dim / 8) ^ v_swizzle<D>(key)) +
                                                  2 * (dim % 8)));
    }
    return u.all;
  };
  auto step = [&](int k0, const u32x4 (&kr)[2][kKs], const char* sv) {
    f32x4 s[2] = {};
#pragma unroll
    for (int n = 0; n < kKs; ++n)
#pragma unroll
      for (int tl = 0; tl < 2; ++tl)
        s[tl] = E::mfma(__builtin_bit_cast(v8, kr[tl][n]), qop[n], s[tl]);
    // Register i of tile tl is key 16 tl + 4 g + i.
    const bool bad = __any(my_blk < 0 && lane < nblk);
#pragma unroll
    for (int tl = 0; tl < 2; ++tl)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[tl][i] = __builtin_fmaf(s[tl][i], scale_log2, nm);
    if (k0 + kKeys - 1 > min_lim || k0 + kKeys > ke || bad) {
      const int vis_end = min(ke, lim + 1) - k0 - 4 * g;
#pragma unroll
      for (int tl = 0; tl < 2; ++tl) {
        const bool gone =
            bad && __builtin_amdgcn_readlane(
                       my_blk, min((k0 - kb + 16 * tl) / block_size, kWave - 1)) < 0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (gone || 16 * tl + i >= vis_end) s[tl][i] = -INFINITY;
      }
    }
    float tmax = s[0][0];
#pragma unroll
    for (int tl = 0; tl < 2; ++tl)
#pragma unroll
      for (int i = 0; i < 4; ++i) tmax = fmaxf(tmax, s[tl][i]);
    tmax = groups_max(tmax);
    const bool first = m == -INFINITY;
    const bool up = first ? tmax != -INFINITY : tmax > E::kRaiseLog2;
    if (__any(up)) {
      const float shift = up ? tmax - E::kTopLog2 : 0.f;
      const float alpha = first ? (up ? 0.f : 1.f) : exp2_fast(-shift);
      if (up) m = first ? shift : m + shift;
      nm = m == -INFINITY ? 0.f : -m;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < kDt; ++dt) o[dt] *= alpha;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[0][i] -= shift;
        s[1][i] -= shift;
      }
    }
    u32x4 pw, third;  // (third: of 5 to 8 vectors in bf16)
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float p0 = exp2_fast(s[w / 2][2 * (w % 2)]), p1 = exp2_fast(s[w / 2][2 * (w % 2) + 1]);
      l += p0 + p1;
      if constexpr (kThree) {
        // The upper half of a float is its first 8 bits in bf16, and what is left is exact.
        const float a0 = less_upper(p0, mask1), a1 = less_upper(p1, mask1);
        pw[w] = uppers(less_upper(a0, mask2), less_upper(a1, mask2));
        if constexpr (VC == 8)
          third[w] = uppers(less_upper(less_upper(p0, kUpper), kUpper),
                            less_upper(less_upper(p1, kUpper), kUpper)) & third_mask;
      } else {
        const uint32_t head = E::round2(p0, p1);
        const uint32_t rest = E::round2(p0 - E::lo(head), p1 - E::hi(head));
        pw[w] = part != 0 ? rest : head;
      }
    }
    const v8 p = __builtin_bit_cast(v8, pw);
    // This step's V has landed when only the loads of the next step, issued after it, are left.
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kKs + kVLoads) : "memory");
#pragma unroll
    for (int dt = 0; dt < kDt; ++dt) o[dt] = E::mfma(read_v(sv, dt), p, o[dt]);
    if constexpr (kThree && VC == 8) {
#pragma unroll
      for (int dt = 0; dt < kDt; ++dt)
        o[dt] = E::mfma(read_v(sv, dt), __builtin_bit_cast(v8, third), o[dt]);
    }
  };

  char* const buf0 = sv0 + wave * kBuf;
  char* const buf1 = sv1 + wave * kBuf;
  u32x4 k0r[2][kKs], k1r[2][kKs];
  if (kb < ke) load_step(kb, k0r, buf0);
  for (int k0 = kb; k0 < ke; k0 += 2 * kKeys) {
    load_step(k0 + kKeys, k1r, buf1);
    issue_fence();
    step(k0, k0r, buf0);
    if (k0 + kKeys >= ke) break;
    load_step(k0 + 2 * kKeys, k0r, buf0);
    issue_fence();
    step(k0 + kKeys, k1r, buf1);
  }
  // Loads past the keys may still be on their way into this wave's buffers.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  l = groups_sum(l);
#pragma unroll
  for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v = o[dt][i];
      o[dt][i] += VC == 4 ? row_ahead<4>(v) + row_ahead<8>(v) : row_ahead<8>(v);
    }
  if (detached) {
    for (int pos = ke; pos < ke_new; ++pos) {
      if (__builtin_amdgcn_readlane(my_blk, (pos - kb) / block_size) < 0) continue;
      const int64_t row = int64_t(q0 + pos - (L - c)) * n_st + int64_t(h) * n_sh;
      float s = 0.f;
#pragma unroll
      for (int n = 0; n < kKs; ++n) {
        const v8 k = *reinterpret_cast<const v8*>(nk + row + 32 * n + 8 * g);
#pragma unroll
        for (int e = 0; e < 8; ++e) s = __builtin_fmaf(float(qop[n][e]), float(k[e]), s);
      }
      s = groups_sum(s) * scale_log2;
      if (pos > lim) s = -INFINITY;
      const float top = fmaxf(m, s);
      const float alpha = m == -INFINITY ? 0.f : exp2_fast(m - top);
      const float p = s == -INFINITY ? 0.f : exp2_fast(s - top);
      m = top;
      l = __builtin_fmaf(l, alpha, p);
#pragma unroll
      for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          o[dt][i] = __builtin_fmaf(o[dt][i], alpha,
                                    p * to_f32<T>(nv[row + 16 * dt + 4 * g + i]));
    }
  }

  // Register i of O tile dt holds dim 16 dt + 4 g + i of vector `vec`.
  const int64_t row0 = int64_t(part_off) + (int64_t(t - q0) * n_q_heads + hq) * pstride;
  if constexpr (NW == 1) {
    if (!active || part != 0) return;
    if (nsplit == 1) {
      const float inv = 1.f / fmaxf(l, 1.17549435e-38f);
      T* op = out + int64_t(t) * o_st + int64_t(hq) * o_sh;
#pragma unroll
      for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) op[16 * dt + 4 * g + i] = from_f32<T>(o[dt][i] * inv);
    } else {
      if (g == 0) part_ml[row0 + split] = make_float2(m, l);
      float* pa = part_acc + (row0 + split) * D;
#pragma unroll
      for (int dt = 0; dt < kDt; ++dt)
        *reinterpret_cast<f32x4*>(pa + 16 * dt + 4 * g) = o[dt];
    }
  } else {
    // The waves' (m, l, O) meet in their own V buffers; the workgroup merges and writes.
    float* acc0 = reinterpret_cast<float*>(buf0);
    if (active && part == 0) {
#pragma unroll
      for (int dt = 0; dt < kDt; ++dt)
        *reinterpret_cast<f32x4*>(acc0 + vec * D + 16 * dt + 4 * g) = o[dt];
      if (g == 0) {
        sml[wave][vec][0] = m;
        sml[wave][vec][1] = l;
      }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < nvec * D; e += NW * kWave) {
      const int v = e / D, d = e % D;
      float mx = -INFINITY, lsum = 0.f, a = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) mx = fmaxf(mx, sml[w][v][0]);
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float mw = sml[w][v][0];
        const float wgt = mw == -INFINITY ? 0.f : exp2_fast(mw - mx);
        lsum = __builtin_fmaf(wgt, sml[w][v][1], lsum);
        a = __builtin_fmaf(wgt, reinterpret_cast<const float*>(sv0 + w * kBuf)[v * D + d], a);
      }
      const int tv = qb + v / n_rep, hv = h * n_rep + v % n_rep;
      if (pstride == 1) {
        out[int64_t(tv) * o_st + int64_t(hv) * o_sh + d] =
            from_f32<T>(a * (1.f / fmaxf(lsum, 1.17549435e-38f)));
      } else {
        const int64_t rv = int64_t(part_off) + (int64_t(tv - q0) * n_q_heads + hv) * pstride;
        if (d == 0) part_ml[rv + split] = make_float2(mx, lsum);
        // The last part marks the unused slots of a slotted row empty.
        if (split == nsplit - 1 && nsplit + d < pstride)
          part_ml[rv + nsplit + d] = make_float2(-INFINITY, 0.f);
        part_acc[(rv + split) * D + d] = a;
      }
    }
  }
}

template <typename T, int D, int NW, int VC>
void launch_kernel(const AttnLaunch& a, int base, int count, int limit_word) {
  hipLaunchKernelGGL((attn_decode_gqa_kernel<T, D, NW, VC>), dim3(count), dim3(NW * kWave), 0, a.s,
                     a.plan, base, limit_word, a.qsl, a.ctx, a.bt, a.bt_stride, a.nb, a.bs,
                     static_cast<const T*>(a.q), a.q_st, a.q_sh, static_cast<const T*>(a.kp),
                     static_cast<const T*>(a.vp), a.hq, a.hkv, a.scale_log2,
                     static_cast<T*>(a.out), a.o_st, a.o_sh, a.ml, a.pacc,
                     static_cast<const T*>(a.nk), static_cast<const T*>(a.nv), a.n_st, a.n_sh,
                     a.slots, static_cast<T*>(const_cast<void*>(a.kp)),
                     static_cast<T*>(const_cast<void*>(a.vp)));
}

template <typename T, int D, int NW>
void launch(const AttnLaunch& a, int base, int count, int limit_word, int vecs) {
  if (__is_same(T, bf16) && vecs <= 4)
    launch_kernel<T, D, NW, __is_same(T, bf16) ? 4 : 8>(a, base, count, limit_word);
  else
    launch_kernel<T, D, NW, 8>(a, base, count, limit_word);
}

// Waves of a workgroup row this kernel is built for: those the planner gives rows of the head_dim.
bool row_waves_built(int32_t head_dim, int waves) {
  return waves == 0 || (head_dim == 64 ? waves == 8 || waves == 16 : waves == kGqaWaves);
}

template <typename T, int D>
void launch_waves(const AttnLaunch& a, int base, int count, int limit_word, int vecs, int waves) {
  if (waves == 0) {
    launch<T, D, 1>(a, base, count, limit_word, vecs);
  } else if constexpr (D == 64) {
    if (waves == 8) launch<T, D, 8>(a, base, count, limit_word, vecs);
    else launch<T, D, 16>(a, base, count, limit_word, vecs);
  } else {
    launch<T, D, kGqaWaves>(a, base, count, limit_word, vecs);
  }
}

}  // namespace

bool decode_gqa_shape(int32_t dtype, int32_t head_dim, int vecs, int32_t block_size) {
  return (dtype == EDGERAG_F16 || dtype == EDGERAG_BF16) && (head_dim == 64 || head_dim == 128) &&
         vecs >= 2 && vecs <= kVecs && block_size % 16 == 0;
}

// Rows of two vectors as KV splits, one wave an item in batches large enough to be bound by the
// stream, stay on attn_decode_kernel, whose loads run further ahead, but for bf16 at head_dim 64,
// whose fp32 query registers bind it there. Here / there, us: fp16 16/8 heads of 128, 32 requests of
// 256-7,472 tokens 100.7 / 95.4, 48 of 4,000 133.1 / 128.8; bf16 32/16 of 128, 48 of 4,000 259.0 /
// 249.3; fp16 64/32 of 64, 48 of 4,000 260.9 / 247.8, 32/16 of 64, 32 of 256-7,472 96.2 / 95.1; bf16
// 32/16 of 64 96.3 / 106.9. (fp16 32/16 of 64, 32 of 2,000: 46.4 / 48.6, the one the other way.)
// After or beside prefill tiles (tiles) the arithmetic of attn_decode_kernel takes longer than alone:
// head_dim 128 then stays here (two 512-token slices and 30 decodes of 4,096, 32/16 heads of 128,
// bf16 231 / 274, fp16 232 / 240; four slices and 40 of 512-7,472, 16/8 188 / 227, 189 / 201).
// Workgroup rows are bound by a wave's chain: fp16 32/16 of 64, 8 requests of 256-3,000 16.1 / 22.5.
// Three vectors: fp16 24/8 of 128, 64 of 256-4,096 105.4 / 109.7.
bool decode_gqa_supported(const AttnLaunch& a, int32_t dtype, int32_t head_dim, int vecs,
                          int waves, bool tiles) {
  if (vecs == 2 && waves == 0 && (head_dim == 128 ? !tiles : dtype == EDGERAG_F16)) return false;
  return decode_gqa_shape(dtype, head_dim, vecs, a.bs) && row_waves_built(head_dim, waves) &&
         int64_t(a.nb) * a.bs * head_dim * 2 < int64_t(kOutOfRange);
}

unsigned decode_gqa_lds(int32_t head_dim, int waves) {
  return unsigned(waves > 4 ? waves : 4) * 2 * kKeys * head_dim * 2;
}

void launch_decode_gqa(const AttnLaunch& a, int32_t dtype, int32_t head_dim, int base, int count,
                       int limit_word, int vecs, int waves) {
  const bool half = dtype == EDGERAG_F16;
  if (head_dim == 64) {
    if (half) launch_waves<f16, 64>(a, base, count, limit_word, vecs, waves);
    else launch_waves<bf16, 64>(a, base, count, limit_word, vecs, waves);
  } else {
    if (half) launch_waves<f16, 128>(a, base, count, limit_word, vecs, waves);
    else launch_waves<bf16, 128>(a, base, count, limit_word, vecs, waves);
  }
}

}  // namespace edgerag
