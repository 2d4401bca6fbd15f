// Chunked-prefill attention tiles on CDNA4 matrix cores (fp16 and bf16, head_dim 64 and 128).
//
// A work item is (request, kv head, query tile of up to kMfmaTileRows virtual rows, KV split).
// Virtual row rho is query token qb + rho / n_rep of query head h * n_rep + rho % n_rep, so all
// heads of a GQA group share every K/V tile. Each wave owns 32 rows.
//
// Per 64-key tile:
//   * K and V rows go from the paged pool straight into LDS (buffer_load ... lds, 16 bytes a lane):
//     no staging registers and no LDS write instructions. A lane chooses which 16-byte chunk of
//     its row it fetches, so the rows land XOR-swizzled and the operand reads are free of bank
//     conflicts. Keys without a valid block get an out-of-range offset and zeros land. Two buffers
//     of each: K of tile i + 2 and V of tile i + 1 are in flight while tile i is computed, with one
//     barrier per tile.
//   * S^T = K Q^T with v_mfma_f32_32x32x16: A = 32 keys x 16 dims from LDS, B = Q^T from registers
//     (loaded once per item): per lane, 16 keys of one query.
//   * online softmax in the log2 domain, p = exp2(s * scale * log2(e) - m). The max m is only
//     raised when a score beats it by 2^8 (lazy rescale). Masks (causal k <= L - c + i, split end,
//     invalid blocks) are applied only on tiles that need them.
//   * O^T += V^T P^T with the same MFMA: the probabilities are already in the B-operand layout
//     once the contraction index is permuted; the A operand is V read transposed out of its
//     row-major LDS tile (ds_read_b64_tr_b16), four keys of one dim a lane and read.
//   * fp16 at head_dim 64 rounds p to fp16 (l sums the same rounded p). The other shapes hold p
//     as hi + lo, both halves in the 16-bit type, two MFMAs per step, and l sums the fp32 p: 16
//     bits of p in bf16 (error 2^-16 of it), 22 in fp16 (2^-22, down to the floor beside
//     kTopLog2), where the output is rounded to 8 and 11.
// A wave computes the scores of tile i + 1 while it exponentiates those of tile i, and scales and
// reduces them while it accumulates P V of tile i: at head_dim 64, matrix and VALU work that do not
// depend on each other alternate in the instruction stream, and issue bounds a tile: at two waves
// per SIMD a wave's 64-key tile takes ~1,600 cycles (130 VALU instructions of ~4 cycles, 32 of them
// exponentials, and 16 MFMAs of 32 cycles); taking out the loads, the exponentials or the P V
// products each gains about 10%. At head_dim 128 (48 MFMAs) the 256 registers do not hold it all: 15
// are spilled, and in every second tile their reloads share the load counter with the prefetch just
// issued, so the wave waits for it; a tile takes ~6,500 cycles (87 us for items of 32
// tiles), twice what its instructions need.
// Measured: bf16, 32/8 heads of 128, two 512-token slices at 2,048 and 4,096 keys beside 7 decodes
// 4,387 us on the row kernel -> 111 us a step in a stream of steps (append, tiles, rows and merge; the
// tiles 87); four such slices at 4,096 keys, 129 GFLOP, 195 us (660 TFLOP/s). fp16 head_dim 64 against
// staging through registers with a transposing LDS write: a decoder's prefill iteration (4
// layers) 880 -> 864 us.
// The output is O / l or, for split items, fp32 partials merged by attn_combine_kernel.
#include "attention_plan.h"

namespace edgerag {
namespace {

using namespace plan;

typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef __bf16 b4 __attribute__((ext_vector_type(4)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

#ifndef EDGERAG_ATTN_SHARED_PAD_KB
#define EDGERAG_ATTN_SHARED_PAD_KB 48  // dynamic LDS of a shared-mode tile workgroup
#endif
#ifndef EDGERAG_TILE_PRIO
// Issue priority (s_setprio) of the tile waves. Beside the decode rows (shared mode) the VALU-
// bound tiles then win the SIMDs' issue slots and the memory-bound row waves fill the gaps:
// config 3 227-229 -> 220-221 us (priority 1: 221-224, 3: 221-223; two tile workgroups per CU
// instead of one, at priority 2: 253 us).
#define EDGERAG_TILE_PRIO 2
#endif
constexpr unsigned kSharedLdsPad = EDGERAG_ATTN_SHARED_PAD_KB * 1024;
constexpr int kKeys = 64;            // keys per LDS tile
constexpr float kRescaleLog2 = 8.f;  // lazy rescale: p may grow to 2^8 before the max moves
constexpr int kWaves = kMfmaTileRows / 32;
constexpr int kThreads = kWaves * kWave;

// Byte offset handed to buffer loads for keys with no valid block: beyond num_records (with any
// chunk offset added), so zeros land without a branch (the launcher keeps a head's pool slice
// below it).
constexpr uint32_t kOutOfRange = 0xFFFFF000u;

constexpr unsigned tile_lds(int d) { return 4 * kKeys * d * 2 + kMaxTileBlocks * 4 + 24; }
static_assert(tile_lds(64) + kSharedLdsPad <= 160 * 1024 &&
                  2 * (tile_lds(64) + kSharedLdsPad) > 160 * 1024 &&
                  tile_lds(128) + kSharedLdsPad <= 160 * 1024 &&
                  2 * (tile_lds(128) + kSharedLdsPad) > 160 * 1024,
              "shared mode: the pad must leave room for exactly one tile workgroup per CU");

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// max / sum of v and its value in lane (lane ^ 32) in every lane: v_permlane32_swap exchanges
// the wave's halves in a VALU op, where a shuffle goes through LDS (ds_bpermute, a round trip).
// The swap leaves lane i with (v[i], v[i + 32]) and lane i + 32 with (v[i], v[i + 32]).
__device__ __forceinline__ float halves_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float halves_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The 16-bit element type of a tile kernel: vectors, matrix product, packing of probabilities.
template <typename T>
struct Elem;
template <>
struct Elem<f16> {
  typedef h8 v8;
  typedef h4 v4;
  static __device__ __forceinline__ f32x16 mfma(v8 a, v8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ v4 pack4(float a, float b, float c, float d) {
    return v4{_Float16(a), _Float16(b), _Float16(c), _Float16(d)};
  }
  // The shapes that hold p as hi + lo hold the p of a row's largest score at 2^kTopLog2 and let it
  // grow to 2^kRaiseLog2. fp16 subnormals end at 2^-24, so hi + lo is off by up to 2^-25 however
  // small p is: 2^-36 of the largest p here, with at least 22 bits of every p above 2^-14 of it.
  // (Held at 2^0, the tail behind one dominant key, thousands of keys of 2^-16 to 2^-24 of it, came
  // out 1% short.)
  static constexpr float kTopLog2 = 11.f, kRaiseLog2 = 15.f;
  // p[0], p[1] as two 16-bit words (round towards zero; the one word of fp16 at head_dim 64).
  static __device__ __forceinline__ uint32_t head_rtz(f2 p) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(p[0], p[1]));
  }
  // The same rounded to nearest, and what that left of each, rounded to nearest too: rounding
  // towards zero would take from every key of a long tail what l still counts.
  static __device__ __forceinline__ uint32_t head(f2 p) {
    uint32_t w = __builtin_bit_cast(uint32_t, h2{_Float16(p[0]), _Float16(p[1])});
    asm("" : "+v"(w));  // one packed conversion: else each half is converted again for rest()
    return w;
  }
  static __device__ __forceinline__ uint32_t rest(f2 p, uint32_t hi) {
    const h2 h = __builtin_bit_cast(h2, hi);
    return __builtin_bit_cast(uint32_t, h2{_Float16(__builtin_fmaf(-float(h[0]), 1.f, p[0])),
                                           _Float16(__builtin_fmaf(-float(h[1]), 1.f, p[1]))});
  }
};
template <>
struct Elem<bf16> {
  typedef b8 v8;
  typedef b4 v4;
  static __device__ __forceinline__ f32x16 mfma(v8 a, v8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ v4 pack4(float a, float b, float c, float d) {
    return v4{__bf16(a), __bf16(b), __bf16(c), __bf16(d)};
  }
  static constexpr float kTopLog2 = 0.f, kRaiseLog2 = kRescaleLog2;  // the exponents of fp32
  static __device__ __forceinline__ uint32_t head(f2 p) {
    return __builtin_bit_cast(uint32_t, b2{__bf16(p[0]), __bf16(p[1])});
  }
  static __device__ __forceinline__ uint32_t rest(f2 p, uint32_t hi) {
    return head(f2{p[0] - __uint_as_float(hi << 16), p[1] - __uint_as_float(hi & 0xFFFF0000u)});
  }
};

// The LDS tile layouts. A row holds one key's D elements as D / 8 16-byte chunks; chunk c of key
// k sits at slot c ^ swizzle(k). LDS serves 256 bytes (64 banks) a cycle, 16 slots: K operands are
// read 16 bytes a lane down consecutive rows, so 16 consecutive rows (8 pairs of 128-byte rows,
// or 16 of 256) must take different slots; V operands are read by ds_read_b64_tr_b16, where 32
// lanes read 64 bytes (4 chunks) of each of 4 consecutive rows. (With only 8 slots told apart
// the K reads of head_dim 64 and all reads of 128 took twice the LDS cycles.)
template <int D>
__device__ __forceinline__ int k_swizzle(int key) {
  return D == 64 ? (key >> 1) & 7 : key & 15;
}
template <int D>
__device__ __forceinline__ int v_swizzle(int key) {
  return D == 64 ? (key & 3) << 1 : (key & 3) << 2;
}

template <bool B>
struct Flag {
  static constexpr bool value = B;
};

struct Geometry {
  int kb, ke, blk0, bs_shift, bs_mask;
};

// One kv head's slice of a pool.
struct Slice {
  const void* base;
  uint32_t bytes;
};

// 16 bytes a lane from byte offset `off` of the slice (zeros past its end) to dst + 16 lane in LDS.
__device__ __forceinline__ void load_lds16(Slice s, char* dst, uint32_t off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(s.base), 0, s.bytes, 0x00020000),
      (__attribute__((address_space(3))) void*)dst, 16, off, 0, 0, 0);
}

// 16 bytes of the slice at byte offset row + in_row (zeros past its end).
__device__ __forceinline__ u32x4 load16(Slice s, uint32_t row, int in_row) {
  return __builtin_bit_cast(
      u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                 __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(s.base), 0, s.bytes,
                                                   0x00020000),
                 __builtin_elementwise_add_sat(row, uint32_t(in_row)), 0, 0));
}

// One wave's share of a tile: load j fills the 64 / (D / 8) rows at dst + 1024 j lane by lane,
// slot lane % (D / 8) of key lkey + 64 / (D / 8) j.
template <int D, bool V, int N>
__device__ __forceinline__ void fetch_tile(Slice s, char* dst, int lane, int lkey,
                                           const uint32_t (&off)[N]) {
  constexpr int kCh = D / 8;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int key = lkey + kWave / kCh * j;
    const int chunk = (lane % kCh) ^ (V ? v_swizzle<D>(key) : k_swizzle<D>(key));
    load_lds16(s, dst + j * 1024, __builtin_elementwise_add_sat(off[j], uint32_t(16 * chunk)));
  }
}

// Two waves per SIMD: the register budget (256 per lane) keeps two tiles' scores, O and Q in VGPRs,
// at head_dim 128 but for 15 of them.
template <typename T, int D>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attn_prefill_mfma_kernel(
    const int32_t* __restrict__ plan, int32_t item_base, int32_t bs_shift,
    const int32_t* __restrict__ qsl, const int32_t* __restrict__ ctx,
    const int32_t* __restrict__ block_tables, int64_t bt_stride, int32_t num_blocks,
    int32_t n_q_heads, const T* __restrict__ q, int64_t q_st, int64_t q_sh,
    const T* __restrict__ kpool, const T* __restrict__ vpool, int32_t n_kv_heads,
    float scale_log2, T* __restrict__ out,
    int64_t o_st, int64_t o_sh, float2* __restrict__ part_ml, float* __restrict__ part_acc) {
  using E = Elem<T>;
  typedef typename E::v8 v8;
  constexpr bool kSplit = !(__is_same(T, f16) && D == 64);  // p as hi + lo (see above)
  // log2 of the p of a row's largest score, and of the p past which its reference moves.
  constexpr float kTop = kSplit ? E::kTopLog2 : 0.f;
  constexpr float kRaise = kSplit ? E::kRaiseLog2 : kRescaleLog2;
  constexpr int kCh = D / 8;                                 // 16-byte chunks of a row
  constexpr int kKpi = kWave / kCh;                          // keys one wave load covers
  constexpr int kLoads = kKeys / kKpi / kWaves;              // wave loads of a tile per wave
  constexpr int kKs = D / 16;                                // 16-dim steps of S
  constexpr int kDt = D / 32;                                // 32-dim tiles of O
  // Separate arrays, not one with a buffer index: a load into one of them is then known not to
  // alias reads of the others, so no read waits for the loads in flight.
  __shared__ __align__(16) char sk0[kKeys * D * 2], sk1[kKeys * D * 2];
  __shared__ __align__(16) char sv0[kKeys * D * 2], sv1[kKeys * D * 2];
  __shared__ uint32_t sblk[kMaxTileBlocks];  // byte offset of each block in the head's slice
  __shared__ struct {
    const T* q;
    int64_t st, sh;
  } sq;  // q again, for the rare sum after the last tile: no register holds it across the loop

  if (EDGERAG_TILE_PRIO > 0) __builtin_amdgcn_s_setprio(EDGERAG_TILE_PRIO);
  const int32_t* it = plan + plan[H_ITEM_OFF] + int64_t(item_base + blockIdx.x) * kItemWords;
  const int r = it[I_REQ], h = it[I_HEAD], qb = it[I_QBEGIN], qc = it[I_QCOUNT];
  const int kb = it[I_KVBEGIN], ke = it[I_KVEND], split = it[I_SPLIT];
  const int32_t* rq = plan + plan[H_REQ_OFF] + r * kReqWords;
  const int nsplit = rq[R_NSPLIT], part_off = rq[R_PARTOFF], pstride = rq[R_PSTRIDE];
  const int q0 = qsl[r], c = qsl[r + 1] - q0, L = ctx[r];
  const int n_rep = n_q_heads / n_kv_heads;
  const int32_t* table = block_tables + int64_t(r) * bt_stride;
  const int64_t head_base = int64_t(h) * num_blocks;
  const int block_size = 1 << bs_shift;

  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int g = lane / 32, col = lane % 32;
  const int nrows = qc * n_rep;
  const int rho = wave * 32 + col;
  const bool active = rho < nrows;
  const int t = qb + (active ? rho / n_rep : 0);
  const int hq = h * n_rep + (active ? rho % n_rep : 0);
  const int lim = active ? L - c + (t - q0) : -1;  // last visible key position of this row
  const bool wave_live = wave * 32 < nrows;
  // Smallest causal limit among the wave's rows: tiles ending at or below it need no mask.
  const int first_row = min(wave * 32, nrows - 1);
  const int wave_min_lim = L - c + (qb + first_row / n_rep - q0);

  Geometry geo;
  geo.kb = kb;
  geo.ke = ke;
  geo.blk0 = kb >> bs_shift;
  geo.bs_shift = bs_shift;
  geo.bs_mask = block_size - 1;
  // Block ids of the whole split, once (the planner caps a split at kMaxTileBlocks blocks).
  // Whether any of them is invalid (never in a well-formed table) decides once per item whether
  // tiles check for invalid keys.
  int any_bad = 0;
  if (tid == 0) {
    sq.q = q;
    sq.st = q_st;
    sq.sh = q_sh;
  }
  {
    const int nblk = min(((ke - 1) >> bs_shift) - geo.blk0 + 1, kMaxTileBlocks);
    for (int i = tid; i < nblk; i += kThreads) {
      const int32_t b = table[geo.blk0 + i];
      const bool ok = b >= 0 && b < num_blocks;
      sblk[i] = ok ? (uint32_t(b) << bs_shift) * uint32_t(D * 2) : kOutOfRange;
      any_bad |= ok ? 0 : 1;
    }
  }
  const bool item_has_bad = __syncthreads_or(any_bad) != 0;

  // Q^T as the B operand: k-step ks covers dims 16*ks + 8*g .. +7 of this lane's query, as
  // given. The scale (times log2 e) multiplies the fp32 dot products afterwards, like the decode
  // rows: scaling q first would round every q * scale to fp16, a score error that grows with the
  // score (scores of tens of nats, as with attention sinks, moved outputs by 3e-2).
  v8 qop[kKs];
  {
    const T* qp = q + int64_t(t) * q_st + int64_t(hq) * q_sh;
#pragma unroll
    for (int ks = 0; ks < kKs; ++ks)
      qop[ks] = active ? *reinterpret_cast<const v8*>(qp + 16 * ks + 8 * g) : v8{};
  }
  f32x16 o[kDt];  // O^T dims 32 dt + .. of this lane's query
#pragma unroll
  for (int dt = 0; dt < kDt; ++dt) o[dt] = f32x16{};
  float m = -INFINITY;  // reference max of the log2-domain scores
  float l = 0.f;        // this lane half's keys only: the halves are added after the last tile
  float nm = 0.f;       // -m (0 while m is -inf)

  const uint32_t head_bytes = uint32_t(int64_t(num_blocks) * block_size * D * 2);
  const Slice krs{kpool + head_base * block_size * D, head_bytes};
  const Slice vrs{vpool + head_base * block_size * D, head_bytes};

  // Staging: wave load j of wave w fills LDS rows kKpi (w kLoads + j) .. + kKpi - 1, lane by lane
  // in order: key lkey + kKpi j of the tile, slot lane % kCh.
  const int lkey = kKpi * kLoads * wave + lane / kCh, wave_lds = wave * kLoads * 1024;
  // Row offsets of this thread's keys of the tile at k0 (a multiple of kKeys) in the head's pool
  // slice: its block's, and the row in the block, which splits into a part of the thread and (for
  // blocks of more than kKeys) a part of the tile. Sums past kOutOfRange saturate.
  auto row_offsets = [&](int k0, uint32_t (&off)[kLoads]) {
    const int i0 = (k0 >> bs_shift) - geo.blk0;
    const uint32_t in_block = uint32_t(k0 & geo.bs_mask) * uint32_t(D * 2);
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int key = lkey + kKpi * j;
      // Looked up in any case (the index clamped) and checked after: no branch around the read.
      const uint32_t blk = sblk[min(i0 + (key >> bs_shift), kMaxTileBlocks - 1)];
      const uint32_t row = uint32_t(key & geo.bs_mask) * uint32_t(D * 2) + in_block;
      off[j] = key < ke - k0 ? __builtin_elementwise_add_sat(blk, row) : kOutOfRange;
    }
  };

  // S^T operand: keys 32 kt + col, dims 16 ks + 8 g .. + 7.
  auto read_k = [&](const char* skb, int ks, int kt) {
    const int key = 32 * kt + col;
    return *reinterpret_cast<const v8*>(skb + key * (D * 2) +
                                        16 * ((2 * ks + g) ^ k_swizzle<D>(key)));
  };
  // V^T operand of k-step st (keys 16 st + {0-3, 8-11} + 4 g) and dim tile dt: two transposing
  // reads of 4 keys x 16 dims per 16 lanes.
  auto read_v = [&](const char* svb, int st, int dt) {
    union {
      s4 half[2];
      v8 all;
    } u;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int key = 16 * st + 8 * i + 4 * g + (lane % 16) / 4;
      const int dim = 32 * dt + 16 * ((lane / 16) % 2) + 4 * (lane % 4);
      u.half[i] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s4*)(svb + key * (D * 2) +
                                                  16 * ((dim / 8) ^ v_swizzle<D>(key)) +
                                                  2 * (dim % 8)));
    }
    return u.all;
  };

  // Masks of the scores of the tile at k0 (already relative to m); their new maximum.
  auto masked_max = [&](f32x16 (&s)[2], int k0, float tmax) {
    const int key_end = min(ke - k0, kKeys);  // keys of this tile inside the split
    if (k0 + kKeys - 1 <= wave_min_lim && key_end == kKeys && !item_has_bad) return tmax;
    // Register i of tile kt holds key 32kt + (i%4) + 8(i/4) + 4g.
    // Keys [0, vis_end + 4g) are visible: compared with constants, so that no key index of a
    // lane is held in a register across the loop.
    const int vis_end = min(key_end, lim - k0 + 1) - 4 * g;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (32 * kt + (i & 3) + 8 * (i >> 2) >= vis_end) s[kt][i] = -INFINITY;
    // Keys whose block id is invalid (never in a well-formed table): masked too.
    uint64_t bad = 0;
    if (item_has_bad) {
      const int bi =
          min(((k0 + min(lane, key_end - 1)) >> bs_shift) - geo.blk0, kMaxTileBlocks - 1);
      bad = __ballot(lane < key_end && sblk[bi] == kOutOfRange);
    }
    if (bad != 0) {
      // Lane group g's keys of tile kt are bits (i%4) + 8(i/4) of (bad_kt >> 4g).
      const uint32_t b0 = uint32_t(bad) >> (4 * g), b1 = uint32_t(bad >> 32) >> (4 * g);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int bit = (i & 3) + 8 * (i >> 2);
        if ((b0 >> bit) & 1u) s[0][i] = -INFINITY;
        if ((b1 >> bit) & 1u) s[1][i] = -INFINITY;
      }
    }
    tmax = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) tmax = fmaxf(tmax, s[kt][i]);
    return tmax;
  };

  // Lazy rescale before the tile whose scores (relative to m) are s with this lane half's
  // maximum tmax: the reference m (the max less kTop) only moves when a p would pass 2^kRaise
  // (before the first visible score, m is -inf and s is absolute).
  auto rescale = [&](f32x16 (&s)[2], float tmax) {
    tmax = halves_max(tmax);  // the other 16 keys of each 32-key tile
    const bool first = m == -INFINITY;
    const bool up = first ? tmax != -INFINITY : tmax > kRaise;
    if (__any(up)) {
      const float shift = up ? tmax - kTop : 0.f;
      const float alpha = first ? (up ? 0.f : 1.f) : exp2_fast(-shift);
      if (up) m = first ? shift : m + shift;
      nm = m == -INFINITY ? 0.f : -m;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < kDt; ++dt) o[dt] *= alpha;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        s[0][i] -= shift;
        s[1][i] -= shift;
      }
    }
  };

  // One tile: s holds its scores (masked, relative to m); with NEXT the scores of the tile at
  // kn = k0 + kKeys are computed into sn on the way.
  const f32x16 zero16 = {};
  const h2 ones = {_Float16(1.f), _Float16(1.f)};
  constexpr int kKAhead = 1, kAhead = 2;  // K steps / V operands read ahead of their MFMAs
  auto tile = [&](auto next, const char* skb, const char* svb, f32x16 (&s)[2], f32x16 (&sn)[2],
                  int kn) {
    constexpr bool kNext = decltype(next)::value;
    constexpr int kSteps = kNext ? kKs : 4;   // chunks of the first phase
    constexpr int kPer = 32 / kSteps;         // probabilities exponentiated per chunk
    uint32_t hi[16], lo[kSplit ? 16 : 1];     // P of k-step st: words 4 st .. 4 st + 3
    float ls[2] = {0.f, 0.f};
    v8 ka[kKAhead + 1][2];
    if constexpr (kNext) {
#pragma unroll
      for (int c = 0; c < kKAhead; ++c) {
        ka[c][0] = read_k(skb, c, 0);
        ka[c][1] = read_k(skb, c, 1);
      }
    }
#pragma unroll
    for (int c = 0; c < kSteps; ++c) {
      if constexpr (kNext) {
        if (c + kKAhead < kKs) {
          ka[(c + kKAhead) % (kKAhead + 1)][0] = read_k(skb, c + kKAhead, 0);
          ka[(c + kKAhead) % (kKAhead + 1)][1] = read_k(skb, c + kKAhead, 1);
        }
        sn[0] = E::mfma(ka[c % (kKAhead + 1)][0], qop[c], c == 0 ? zero16 : sn[0]);
      }
#pragma unroll
      for (int w = c * kPer / 2; w < (c + 1) * kPer / 2; ++w) {
        const int kt = w / 8, i = 2 * (w % 8);
        const f2 p = {exp2_fast(s[kt][i]), exp2_fast(s[kt][i + 1])};
        if constexpr (kSplit) {
          hi[w] = E::head(p);
          ls[0] += p[0];
          ls[1] += p[1];
          lo[w] = E::rest(p, hi[w]);
        } else {
          hi[w] = E::head_rtz(p);
          ls[w & 1] = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, hi[w]), ones, ls[w & 1], false);
        }
        if constexpr (kNext)
          if (w == c * kPer / 2 + kPer / 4) sn[1] = E::mfma(ka[c % (kKAhead + 1)][1], qop[c], c == 0 ? zero16 : sn[1]);
      }
    }
    l += ls[0] + ls[1];
    asm volatile("" : "+v"(l));  // summed here: sunk below, it would keep every p alive
    // O^T += V^T P^T, and the next tile's scores scaled and reduced.
    float tmax = -INFINITY;
    v8 va[kAhead + 1];
#pragma unroll
    for (int n = 0; n < kAhead; ++n) va[n] = read_v(svb, n / kDt, n % kDt);
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      union {
        uint32_t w[4];
        v8 v;
      } ph, pl;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        ph.w[j] = hi[4 * st + j];
        if constexpr (kSplit) pl.w[j] = lo[4 * st + j];
      }
#pragma unroll
      for (int dt = 0; dt < kDt; ++dt) {
        const int n = st * kDt + dt;
        if (n + kAhead < 4 * kDt)
          va[(n + kAhead) % (kAhead + 1)] = read_v(svb, (n + kAhead) / kDt, (n + kAhead) % kDt);
        o[dt] = E::mfma(va[n % (kAhead + 1)], ph.v, o[dt]);
        if constexpr (kSplit) o[dt] = E::mfma(va[n % (kAhead + 1)], pl.v, o[dt]);
        if constexpr (kNext) {
          // log2-domain scores relative to the reference max: q.k * scale * log2(e) - m.
#pragma unroll
          for (int e = 8 / kDt * dt; e < 8 / kDt * (dt + 1); ++e) {
            const int kt = st / 2, i = 8 * (st % 2) + e;
            sn[kt][i] = __builtin_fmaf(sn[kt][i], scale_log2, nm);
            tmax = fmaxf(tmax, sn[kt][i]);
          }
        }
      }
    }
    if constexpr (kNext) rescale(sn, masked_max(sn, kn, tmax));
  };
  // The scores of the first tile alone.
  auto first_scores = [&](const char* skb, f32x16 (&s)[2]) {
#pragma unroll
    for (int ks = 0; ks < kKs; ++ks)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
        s[kt] = E::mfma(read_k(skb, ks, kt), qop[ks], ks == 0 ? zero16 : s[kt]);
    float tmax = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        s[kt][i] = __builtin_fmaf(s[kt][i], scale_log2, nm);
        tmax = fmaxf(tmax, s[kt][i]);
      }
    rescale(s, masked_max(s, kb, tmax));
  };

  // This wave's loads have landed; after the barrier, every wave's have, and every wave is done
  // with the buffers of the tile before.
  auto landed = [&]() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };
  // Even tiles use buffers 0 and offsets off0, odd tiles buffers 1 and off1. While tile i is
  // computed, K of tile i + 2 and V of tile i + 1 are on their way (tiles past the split load
  // zeros).
  uint32_t off0[kLoads], off1[kLoads];
  auto advance_even = [&](int k0) {
    landed();
    fetch_tile<D, false>(krs, sk0 + wave_lds, lane, lkey, off0);
    fetch_tile<D, true>(vrs, sv1 + wave_lds, lane, lkey, off1);
    row_offsets(k0 + 3 * kKeys, off1);
  };
  auto advance_odd = [&](int k0) {
    landed();
    fetch_tile<D, false>(krs, sk1 + wave_lds, lane, lkey, off1);
    fetch_tile<D, true>(vrs, sv0 + wave_lds, lane, lkey, off0);
    row_offsets(k0 + 3 * kKeys, off0);
  };
  row_offsets(kb, off0);
  fetch_tile<D, false>(krs, sk0 + wave_lds, lane, lkey, off0);
  row_offsets(kb + kKeys, off1);
  landed();
  fetch_tile<D, false>(krs, sk1 + wave_lds, lane, lkey, off1);
  fetch_tile<D, true>(vrs, sv0 + wave_lds, lane, lkey, off0);
  row_offsets(kb + 2 * kKeys, off0);
  const int last = kb + (ke - kb - 1) / kKeys * kKeys;  // first key of the last tile
  if (!wave_live) {  // this wave only stages
    for (int k0 = kb; k0 <= last; k0 += 2 * kKeys) {
      advance_even(k0);
      if (k0 < last) advance_odd(k0 + kKeys);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return;
  }
  f32x16 s0[2], s1[2];
  first_scores(sk0, s0);
  int k0 = kb;
  const char* svl = sv0;  // V of the last tile
  for (; k0 < last; k0 += 2 * kKeys) {
    advance_even(k0);
    tile(Flag<true>{}, sk1, sv0, s0, s1, k0 + kKeys);
    if (k0 + kKeys >= last) {
      s0[0] = s1[0];
      s0[1] = s1[1];
      svl = sv1;
      break;
    }
    advance_odd(k0 + kKeys);
    tile(Flag<true>{}, sk0, sv1, s1, s0, k0 + 2 * kKeys);
  }
  landed();
  tile(Flag<false>{}, sk0, svl, s0, s1, 0);
  // No load may still be on its way into this workgroup's LDS when the workgroup ends.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  l = halves_sum(l);

  // A key that a row does not see has p = 0, and 0 times a NaN or infinite V is NaN: a later token's
  // V must not reach the rows before it. Where one did, the rows are summed again key by key.
  float any_odd = 0.f;
#pragma unroll
  for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) any_odd = __builtin_fmaf(o[dt][i], 0.f, any_odd);
  if (__any(active && any_odd != 0.f)) {
    // (Loads through the descriptors of the main loop, and indexes of this lane formed here: nothing
    // of this is held in registers across the loop.)
    int ln = lane;
    asm volatile("" : "+v"(ln));
    auto row_of = [&](int pos) {  // byte offset of key pos in the head's slice
      return __builtin_elementwise_add_sat(sblk[(pos >> bs_shift) - geo.blk0],
                                           uint32_t(pos & geo.bs_mask) * uint32_t(D * 2));
    };
    bool hidden = false;  // a non-finite V among the keys that some row of the wave does not see
    for (int pos = max(kb, wave_min_lim + 1) + ln / kCh; pos < ke; pos += kKpi) {
      const v8 v = __builtin_bit_cast(v8, load16(vrs, row_of(pos), 16 * (ln % kCh)));
#pragma unroll
      for (int e = 0; e < 8; ++e) hidden |= !(__builtin_fabsf(float(v[e])) < INFINITY);
    }
    if (__any(hidden)) {
      const T* qp = sq.q + int64_t(t) * sq.st + int64_t(hq) * sq.sh + 8 * (ln / 32);
#pragma unroll
      for (int dt = 0; dt < kDt; ++dt) o[dt] = f32x16{};
      for (int pos = kb; pos < ke; ++pos) {
        const uint32_t off = row_of(pos);
        if (off >= krs.bytes) continue;
        float s = 0.f;
#pragma unroll
        for (int ks = 0; ks < kKs; ++ks) {
          const v8 k = __builtin_bit_cast(v8, load16(krs, off, 32 * ks + 16 * (ln / 32)));
          const v8 qk = *reinterpret_cast<const v8*>(qp + 16 * ks);
#pragma unroll
          for (int e = 0; e < 8; ++e) s = __builtin_fmaf(float(qk[e]), float(k[e]), s);
        }
        float p = exp2_fast(__builtin_fmaf(halves_sum(s), scale_log2, nm));
        if constexpr (!kSplit)
          p = float(__builtin_bit_cast(h2, E::head_rtz(f2{p, 0.f}))[0]);
        if (pos > lim) continue;
        // Dims 32 dt + 8 qd + 0-3 (lanes of the lower half) and + 4-7 (of the upper).
#pragma unroll
        for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
          for (int qd = 0; qd < 4; ++qd) {
            const v8 v = __builtin_bit_cast(v8, load16(vrs, off, 64 * dt + 16 * qd));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float ve = ln < 32 ? float(v[e]) : float(v[4 + e]);
              o[dt][4 * qd + e] = __builtin_fmaf(p, ve, o[dt][4 * qd + e]);
            }
          }
      }
    }
  }

  if (!active) return;
  // O^T register i of dim tile dt holds dim 32dt + (i%4) + 8(i/4) + 4g of this lane's query.
  if (nsplit == 1) {
    const float inv = 1.f / fmaxf(l, 1.17549435e-38f);
    T* op = out + int64_t(t) * o_st + int64_t(hq) * o_sh;
    const bool vec_out =
        (reinterpret_cast<uintptr_t>(out) & 7) == 0 && o_st % 4 == 0 && o_sh % 4 == 0;
#pragma unroll
    for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        T* dst = op + 32 * dt + 8 * qd + 4 * g;
        const typename E::v4 v = E::pack4(o[dt][4 * qd] * inv, o[dt][4 * qd + 1] * inv,
                                          o[dt][4 * qd + 2] * inv, o[dt][4 * qd + 3] * inv);
        if (vec_out) {
          *reinterpret_cast<typename E::v4*>(dst) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) dst[e] = __builtin_bit_cast(T, v[e]);
        }
      }
  } else {
    // Partials carry the max in the log2 domain, like the decode kernels'.
    const int64_t idx = int64_t(part_off) + (int64_t(t - q0) * n_q_heads + hq) * pstride + split;
    if (g == 0) part_ml[idx] = make_float2(m, l);
    float* pa = part_acc + idx * D;
#pragma unroll
    for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd)
        *reinterpret_cast<float4*>(pa + 32 * dt + 8 * qd + 4 * g) =
            make_float4(o[dt][4 * qd], o[dt][4 * qd + 1], o[dt][4 * qd + 2], o[dt][4 * qd + 3]);
  }
}

template <typename T, int D>
void launch_tiles(const AttnLaunch& a, int item_base, int count, bool shared, unsigned row_lds) {
  // Shared mode reserves unused dynamic LDS so that a second workgroup no longer fits a CU's
  // 160 KiB (the static arrays take 34 or 66 KiB): the tiles then hold one of each SIMD's two
  // register halves and decode waves keep the other. Rows on the grouped kernel need LDS of
  // their own (row_lds, for a wave per SIMD): where that does not fit beside tile and pad, the pad
  // would hold the place of a second tile for rows that cannot use it, and is left out (the rows
  // then fill in as tiles end). Slices beside decodes, us with the pad / without: bf16 32/8 heads
  // of 128, two at 4,096 keys with 24 of 4,096 tokens 194 / 158, with 60 of 1,200 168 / 143, with 40
  // of 2,000 145 / 151; 32/8 of 64, three with 32 of 8,000 (rows of 16 waves) 195 / 161. Where
  // it fits (rows of 8 waves or one wave at 64): three with 20 of 8,192 115 / 131, with 48 of
  // 4,096 132 / 140, of 8,000 211 / 199.
  const bool fits = tile_lds(D) + kSharedLdsPad + row_lds <= 160 * 1024;
  const unsigned pad = shared && fits ? kSharedLdsPad : 0;
  hipLaunchKernelGGL((attn_prefill_mfma_kernel<T, D>), dim3(count), dim3(kThreads), pad, a.s,
                     a.plan, item_base, log2_exact(a.bs), a.qsl, a.ctx, a.bt, a.bt_stride, a.nb,
                     a.hq, static_cast<const T*>(a.q), a.q_st, a.q_sh,
                     static_cast<const T*>(a.kp), static_cast<const T*>(a.vp), a.hkv,
                     a.scale_log2, static_cast<T*>(a.out), a.o_st, a.o_sh, a.ml, a.pacc);
}
}  // namespace

bool prefill_tile_shape(int32_t dtype, int32_t head_dim) {
  return (dtype == EDGERAG_F16 || dtype == EDGERAG_BF16) && (head_dim == 64 || head_dim == 128);
}

bool prefill_tiles_supported(int32_t num_blocks, int32_t block_size, int32_t head_dim) {
  // Power-of-two blocks of at least 4 keys (shift addressing), and one kv head's slice of a pool
  // must fit a buffer resource, below kOutOfRange.
  return log2_exact(block_size) >= 2 &&
         int64_t(num_blocks) * block_size * head_dim * 2 < int64_t(kOutOfRange);
}

void launch_prefill_tiles(const AttnLaunch& a, int32_t dtype, int32_t head_dim, int item_base,
                          int count, bool shared, unsigned row_lds) {
  const bool half = dtype == EDGERAG_F16;
  if (head_dim == 64) {
    if (half) launch_tiles<f16, 64>(a, item_base, count, shared, row_lds);
    else launch_tiles<bf16, 64>(a, item_base, count, shared, row_lds);
  } else {
    if (half) launch_tiles<f16, 128>(a, item_base, count, shared, row_lds);
    else launch_tiles<bf16, 128>(a, item_base, count, shared, row_lds);
  }
}

}  // namespace edgerag
