// K2 for prefill rows of any context, column tiles (fp16 / bf16): the attention of a
// sequence's new rows over its whole context (reference src/tinybatch/model.py:130-147:
// gather, repeat_interleave, the mask of model.py:139-146 and SDPA).
//
// Work: the new rows of a sequence and the rep query heads of a kv head make
// n * rep columns, column = row * rep + head; a workgroup takes NW * 32 consecutive
// columns (every head of NW * 32 / rep rows), wave w its columns 32 w .. 32 w + 31. So all
// of a workgroup's columns read the same K/V rows, whatever rep is, with no padded
// columns but the sequence's last ones, and its rows lie close together, so that few
// scores past the diagonal are computed. The workgroup walks its positions in chunks of
// 64.
//
// Loads. A chunk's K and V rows go to LDS by direct global->LDS loads (1 KiB of
// consecutive pool bytes per instruction) through a ring of two chunks: the next chunk is
// issued as a chunk's computation starts, so one wait (for the wave's own loads) and one
// barrier per chunk are all the synchronisation. Rows past the workgroup's last position
// repeat the last one: their scores are masked.
//
// Math per chunk, the wave's 32 columns as the 32 MFMA columns:
//   S^T[pos][col] = K[pos][:] . q[col][:]         v_mfma_f32_32x32x16, A = K rows (LDS)
//   O^T[d][col]  += V^T[d][pos] . P^T[pos][col]   v_mfma_f32_32x32x16, A = V^T (LDS
//                                                  transpose reads), B = the S^T registers
// so that each K or V value read from LDS meets 32 columns, and the online softmax state
// of column l % 32 lives in lanes l and l ^ 32. A masked score weighs 0, also against what is
// not finite: an infinite or NaN value of a new row makes the earlier rows of its workgroup NaN
// (in the reference's masked product all rows of the sequence); a key's reaches none.
//
// What bounds it and what it measured (bf16, us per layer, against the 64-row tiles of
// tb_attention.hip): three prompts of 5300..7333 tokens at 32 / 8 heads of 128: 1100 us =
// 985 TFLOP/s once the clock has settled (1150 to 1500 in the first twenty launches after idle)
// against 3260 + 290 for the merge of split rows; four of 1746..3738 at 14 / 2
// heads of 64: 86 us = 670 TFLOP/s against 122 + 14. (A plain 8192^3 library product
// reaches 1232 TFLOP/s on this card.) At head dim 128 two chunks of a CU take 4200 cycles of the
// launch (counters; workgroup starts and ends in it), 2040 of them MFMA on each SIMD, at a
// shader clock of 1.5 to 1.9 GHz; at 64 (2.2 GHz, MFMA busy 28%)
// the softmax (32 exponentials, FMAs and packs a chunk) and its issue bound it. Measured
// and not kept: 256 columns in eight waves (one workgroup per CU at head dim 128, whose
// start and end, 9 us of 65 by marks in a timing copy, nothing then overlaps: 1140 us); the two
// waves of a SIMD held half a chunk apart by barriers (930 against 911 us on six prompts of 4096);
// the next chunk's scores computed under this chunk's exponentials (spills at head dim 128); a
// chunk's loads spread between its products (the same); row sums on the matrix unit (5%
// slower at head dim 64).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <exception>
#include <vector>

#include "tb_stream.h"

namespace tb {

typedef float float16_t __attribute__((ext_vector_type(16)));

template <typename Tag>
struct cmath;
template <>
struct cmath<f16_t> {
  typedef shalf8_t vec8_t;
  static __device__ __forceinline__ float16_t mfma(su32x4_t a, su32x4_t b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(shalf8_t, a), __builtin_bit_cast(shalf8_t, b), c,
                                                   0, 0, 0);
  }
  // acc + the two halves of p (times one each); subnormal halves count, as in the products
  // (measured: thousands of weights of 2^-16 .. 2^-22 beside one of 1)
  static __device__ __forceinline__ float add2(uint32_t p, uint32_t ones, float acc) {
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, p), __builtin_bit_cast(half2_t, ones), acc, false);
  }
  static constexpr uint32_t ONES = 0x3C003C00u;
};
template <>
struct cmath<bf16_t> {
  typedef sbf168_t vec8_t;
  static __device__ __forceinline__ float16_t mfma(su32x4_t a, su32x4_t b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(sbf168_t, a), __builtin_bit_cast(sbf168_t, b),
                                                    c, 0, 0, 0);
  }
  static __device__ __forceinline__ float add2(uint32_t p, uint32_t ones, float acc) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf162_t, p), __builtin_bit_cast(bf162_t, ones), acc, false);
  }
  static constexpr uint32_t ONES = 0x3F803F80u;
};

struct cols_args {
  const char* q;               // [T][Hq][D] rows of the step
  int64_t q_row_bytes;
  const char* pool;            // [NB][2][Hkv][BS][D]
  int64_t num_blocks;
  char* out;                   // [T][Hq*D]
  int64_t out_row_bytes;
  const int32_t* block_tables; // [B][max_nb]
  int32_t max_nb;
  const int4* work;            // two per workgroup: (row0, seq, pos0, nrows), (first column, kv head, part, part chunks)
  const int32_t* row_part_off; // partial slots of the step's rows
  float* ws_acc;               // [parts][Hq][D]
  float* ws_ml;                // [parts][Hq][2]
  int32_t num_heads, num_kv_heads, rep;
  int32_t log2_bs;             // block size: a power of two >= 16
  float scale_log2e;           // > 0: the scale's size times log2(e), or 1 for a scale of 0
  float q_sign;                // 1, -1 or 0 (NaN: a NaN scale): multiplies q, so that masked scores stay -inf
  rope_tables rope;
};

template <int D>
struct cshape {
  static constexpr int NW = 4;                  // waves per workgroup
  static constexpr int RB = 2 * D;              // bytes per K or V row
  static constexpr int TB = 16 * RB;            // bytes of a 16-position K (or V) tile
  static constexpr int CK = 64;                 // positions per chunk
  static constexpr int HALF = CK * RB;          // bytes of a chunk's K (or V) rows
  static constexpr int SLOT = 2 * HALF;         // K then V
  static constexpr int RING = 2;              // chunks in LDS: two or three workgroups on a CU
  static constexpr int VCOLS = RB / 16;         // 16-byte pieces per row
  static constexpr int RPL = 64 / VCOLS;        // rows per direct load
  static constexpr int TLD = TB / 1024;         // direct loads per 16-position tile
  static constexpr int KS = D / 16;             // q.k slices of 16 dims
  static constexpr int NB = D / 32;             // O^T blocks of 32 dims
  static constexpr int COLS = 32 * NW;          // columns per workgroup
  static_assert(CK == 16 * NW, "wave w loads tile w of a chunk");
  // K row r keeps its 16-byte piece c in slot c ^ kswz(r): the 16 rows that 16 lanes of an
  // operand read touch then cover all 64 banks (rows 2 apart share banks at D = 64)
  static __device__ __forceinline__ int kswz(int r) { return D == 64 ? (r & 7) ^ ((r >> 3) & 1) : r & 15; }
  // V row r keeps piece c in slot c ^ vswz(r): the transpose reads of 32 lanes (4 rows x
  // 64 bytes) cover all 64 banks
  static __device__ __forceinline__ int vswz(int r) {
    return D == 64 ? 2 * (r & 3) : (0xCA60 >> (4 * (r & 3))) & 15;
  }
};

// SP = 2: two sets of NW waves on the same columns, set sp taking chunks sp, sp + 2, ... of
// the range through a ring of its own; their states merge in LDS at the end. SIGNED: a scale of
// zero or below, whose sign goes into q (a branch on it in every launch cost 1% of short ones).
template <typename Tag, int D, int SP, bool SIGNED>
__global__ __launch_bounds__(64 * cshape<D>::NW * SP, 2) void paged_prefill_columns_kernel(const cols_args a) {
  using S = cshape<D>;
  using M = cmath<Tag>;
  typedef typename smath<Tag>::scalar_t scalar_t;
  constexpr int RB = S::RB, TB = S::TB, CK = S::CK, KS = S::KS, NB = S::NB;
  __shared__ __align__(1024) char lds_all[SP * S::RING * S::SLOT];

  const int wave_id = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wave = wave_id % S::NW, sp = wave_id / S::NW;   // the wave's columns, its set of chunks
  char* const lds = lds_all + sp * (S::RING * S::SLOT);
  const int lane = threadIdx.x & 63, lcol = lane & 31, half = lane >> 5;
  const int4 w0 = a.work[2 * blockIdx.x], w1 = a.work[2 * blockIdx.x + 1];
  const int row0 = w0.x, seq = w0.y, pos0 = w0.z, nrows = w0.w;
  if (nrows == 0) return;                       // a padding entry (whole workgroup)
  const int col0 = w1.x, kvh = w1.y, part = w1.z, part_chunks = w1.w;
  const int rep = a.rep, ncols = nrows * rep;

  // this lane's column: query row my_row of the sequence's new rows, head hd
  const int col = col0 + 32 * wave + lcol;
  const bool mine = col < ncols;
  const int ccol = mine ? col : ncols - 1;
  const int my_row = ccol / rep, hd = kvh * rep + ccol - my_row * rep;
  const int my_pos = pos0 + my_row;             // sees positions 0 .. my_pos
  // wave-uniform: the positions of the wave's first and last column, the workgroup's positions
  const int wcol = min(col0 + 32 * wave, ncols - 1);
  const bool wave_busy = col0 + 32 * wave < ncols;
  const int wave_first = pos0 + wcol / rep;
  const int wave_last = pos0 + min(col0 + 32 * wave + 31, ncols - 1) / rep;
  const int limit = pos0 + min(col0 + S::COLS - 1, ncols - 1) / rep + 1;
  const int c_begin = part * part_chunks;
  const int c_end = min(c_begin + part_chunks, (limit + CK - 1) / CK);

  // ---- q (B operand: lane holds dims 16 s + 8 half .. of its column) ----
  vec16 qv[KS];
  {
    const char* qrow = a.q + (int64_t)(row0 + my_row) * a.q_row_bytes + (int64_t)hd * RB + 16 * half;
#pragma unroll
    for (int s = 0; s < KS; ++s) qv[s] = ld16(qrow + 32 * s);
  }

  // ---- direct loads: pair i of this wave is tile lt[i] of the chunk, K or V ----
  const int64_t head_bytes = ((int64_t)1 << a.log2_bs) * RB;     // one kv head's K (or V) rows of a block
  const int64_t blk_bytes = 2 * (int64_t)a.num_kv_heads * head_bytes;
  const int64_t v_off = a.num_kv_heads * head_bytes;
  const int sub_mask = (1 << (a.log2_bs - 4)) - 1;                // 16-position tiles per block - 1
  const int32_t* const table = a.block_tables + (int64_t)seq * a.max_nb;
  const char* const pool_kvh = a.pool + kvh * head_bytes;
  const int last_tile = (limit - 1) >> 4;
  const int lt = wave;                          // the tile of a chunk this wave loads, K and V
  const int lrow = lane / S::VCOLS, lpiece = lane % S::VCOLS;
  // lane j: the block of this wave's tile in chunk id0 + j
  int id0 = c_begin + sp;
  auto load_ids = [&](int c) {
    const int t = min(4 * (c + lane) + lt, last_tile);
    int b = table[(t << 4) >> a.log2_bs];
    return (b < 0 || b >= a.num_blocks) ? 0 : b;   // host validates; stay inside the pool
  };
  int ids = load_ids(id0);
  auto issue = [&](int c, int slot) {
    if (c - id0 >= 64) {                        // uniform, once per 64 chunks
      id0 = c;
      ids = load_ids(id0);
    }
    const int t = min(4 * c + lt, last_tile);
    const int rmax = limit - 1 - 16 * t;        // rows past it repeat the workgroup's last position
    const int64_t b = __builtin_amdgcn_readlane(ids, c - id0);
    const char* const base = pool_kvh + b * blk_bytes + (int64_t)(t & sub_mask) * TB;
    char* const dst = lds + slot * S::SLOT + lt * TB;
#pragma unroll
    for (int i = 0; i < S::TLD; ++i) {
      const int r = S::RPL * i + lrow;
      const uint32_t row = (uint32_t)(min(r, rmax) * RB);
      s_dma16_l2(row + 16 * (lpiece ^ S::kswz(r)), base, dst + 1024 * i);
      s_dma16_l2(row + 16 * (lpiece ^ S::vswz(r)), base + v_off, dst + S::HALF + 1024 * i);
    }
  };
  asm volatile("" : "+v"(ids));                 // the block ids have landed: no wait inside the loop
  if (c_begin + sp < c_end) issue(c_begin + sp, 0);

  // ---- q rotated (RoPE at the column's position), complete here ----
  if (a.rope.cos) {
    const int64_t r = a.rope.row(my_pos, D / 2) + 8 * half;
#pragma unroll
    for (int s = 0; s < KS / 2; ++s)            // slices s and s + KS/2 pair (dims i and i + D/2)
      rope_pair<scalar_t>(qv[s], qv[s + KS / 2], a.rope.cos + r + 16 * s, a.rope.sin + r + 16 * s);
  }
  if constexpr (SIGNED) {
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      typename M::vec8_t x = __builtin_bit_cast(typename M::vec8_t, qv[s]);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = (scalar_t)((float)x[e] * a.q_sign);
      qv[s] = __builtin_bit_cast(vec16, x);
    }
  }
  su32x4_t q[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    q[s] = __builtin_bit_cast(su32x4_t, qv[s]);
    asm volatile("" : "+v"(q[s]));
  }

  uint32_t ones = M::ONES;                      // in a register: as a literal the bf16 dot product read it wrong
  asm volatile("" : "+v"(ones));
  float m = -INFINITY, l = 0.f;                 // reference max (scaled, base-2) and this lane's share of the sum
  float16_t acc[NB];                            // O^T[32 b + 8 (r / 4) + 4 half + r % 4][col]
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[b][r] = 0.f;

  // operand addresses of this lane in a ring slot
  uint32_t ka[KS], va[NB];
#pragma unroll
  for (int s = 0; s < KS; ++s) ka[s] = (uint32_t)(lcol * RB + 16 * ((2 * s + half) ^ S::kswz(lcol)));
  {
    const int li = lane & 15, rv = 4 * half + (li >> 2);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int c = 4 * b + 2 * ((lane >> 4) & 1) + ((li & 3) >> 1);
      va[b] = (uint32_t)(S::HALF + rv * RB + 16 * (c ^ S::vswz(rv)) + 8 * (li & 1));
    }
  }
  const float sl2e = a.scale_log2e;

  float16_t sc[2];                              // S^T: positions 64 c + 32 t + 8 (r / 4) + 4 half + r % 4 of column lcol
  su32x4_t pb[4];                               // P of a chunk: B operands of 16 positions each
  // S^T = K.q of the chunk in a slot
  auto scores = [&](int slot) {
    const char* const base = lds + slot * S::SLOT;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) sc[t][r] = 0.f;
    // operands read KG slices ahead of their products, pinned by the scheduling barriers:
    // left to itself the compiler keeps one slice in flight and every product waits out
    // an LDS latency
    constexpr int KG = 2;
    su32x4_t kf[2][KG][2];
    auto read = [&](int g) {
#pragma unroll
      for (int i = 0; i < KG; ++i)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          kf[g & 1][i][t] = *reinterpret_cast<const su32x4_t*>(base + ka[KG * g + i] + 32 * t * RB);
    };
    read(0);
#pragma unroll
    for (int g = 0; g < KS / KG; ++g) {
      if (g + 1 < KS / KG) read(g + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < KG; ++i)
#pragma unroll
        for (int t = 0; t < 2; ++t) sc[t] = M::mfma(kf[g & 1][i][t], q[KG * g + i], sc[t]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // the online softmax of chunk c: sc -> pb, and the state's rescale
  auto softmax = [&](int c) {
    if (CK * c + CK - 1 > wave_first) {         // the chunk crosses the diagonal of some column
      // kept a branch (most chunks skip it): folded into selects it cost every chunk 96
      // vector instructions beside the 150 it needs
      asm volatile("");
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (CK * c + 32 * t + 8 * (r >> 2) + 4 * half + (r & 3) > my_pos) sc[t][r] = -INFINITY;
    }
    float cm = max_f32(sc[0][0], sc[0][1]);
#pragma unroll
    for (int e = 2; e < 32; e += 2) cm = max3_f32(cm, sc[e >> 4][e & 15], sc[e >> 4][(e & 15) + 1]);
    cm *= sl2e;
    // the reference max moves only when some column outgrows it by 8 (p <= 2^8)
    if (__any(cm > m + 8.f)) {
      const float m_new = fmaxf(m, max_xor32(cm));
      const float alpha = fast_exp2(m - (m_new == -INFINITY ? 0.f : m_new));   // 0 while m = -inf
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[b] *= alpha;
    }
    const float neg_m = m == -INFINITY ? 0.f : -m;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      // k index 8 half + j <-> position 16 w + 4 half + j (j < 4) or 8 further
      float p[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) p[j] = fast_exp2(fmaf(sc[w >> 1][8 * (w & 1) + j], sl2e, neg_m));
      pb[w] = smath<Tag>::pack8(p);
#pragma unroll
      for (int j = 0; j < 4; ++j) l = M::add2(pb[w][j], ones, l);   // of the rounded P that multiplies V
    }
  };
  // O^T += V^T.P of the chunk in a slot
  auto values = [&](int slot) {
    const char* const base = lds + slot * S::SLOT;
    uint2 vf[2][NB][2];
    auto read = [&](int w) {
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const char* const vp = base + va[b] + 16 * w * RB;
        vf[w & 1][b][0] = lds_read_tr16(vp);
        vf[w & 1][b][1] = lds_read_tr16(vp + 8 * RB);
      }
    };
    read(0);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (w + 1 < 4) read(w + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const uint2 lo = vf[w & 1][b][0], hi = vf[w & 1][b][1];
        acc[b] = M::mfma(su32x4_t{lo.x, lo.y, hi.x, hi.y}, pb[w], acc[b]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // The set's chunk k, c_begin + SP k + sp, lies in slot k % RING of its ring.
  const int n = (c_end - c_begin + SP - 1) / SP;
  const int c_wave = wave_busy ? min(c_end - 1, wave_last / CK) : -1;   // this wave's last chunk
  for (int k = 0; k < n; ++k) {
    // the wave's loads of chunk k have landed and its LDS reads of chunk k - 1 are done:
    // behind the barrier all of chunk k is in LDS and the slot of chunk k - 1 is free
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int c = c_begin + SP * k + sp;
    if (c + SP < c_end) issue(c + SP, (k + 1) % S::RING);
    if (c <= c_wave) {
      const int slot = k % S::RING;
      scores(slot);
      softmax(c);
      values(slot);
    }
  }

  if constexpr (SP == 2) {                      // set 1's state to set 0 (log-sum-exp)
    float* const slot = reinterpret_cast<float*>(lds_all) + wave * (64 * (16 * NB + 2)) + lane;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // every read of the chunks is done
    if (sp == 1) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) slot[64 * (16 * b + r)] = acc[b][r];
      slot[64 * 16 * NB] = m;
      slot[64 * (16 * NB + 1)] = l;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (sp == 1) return;
    const float m1 = slot[64 * 16 * NB], l1 = slot[64 * (16 * NB + 1)];
    const float m_new = fmaxf(m, m1), m_safe = m_new == -INFINITY ? 0.f : m_new;
    const float f0 = fast_exp2(m - m_safe), f1 = fast_exp2(m1 - m_safe);   // 0 for a set that saw nothing
    m = m_new;
    l = l * f0 + l1 * f1;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[b][r] = acc[b][r] * f0 + slot[64 * (16 * b + r)] * f1;
  }

  l = sum_xor32(l);
  if (!mine) return;
  const int row = row0 + my_row;
  const int pbeg = a.row_part_off[row], nparts = a.row_part_off[row + 1] - pbeg;
  if (part >= nparts) return;                   // the row ends before this part
  if (nparts == 1) {                            // the whole row: final output
    const float inv = 1.f / l;
    char* const orow = a.out + (int64_t)row * a.out_row_bytes + (int64_t)hd * RB + 8 * half;
    typedef scalar_t s4_t __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        s4_t o;
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = (scalar_t)(acc[b][4 * g + j] * inv);
        st8_through(orow + 64 * b + 16 * g, o);
      }
  } else {                                      // partial of a split row
    const int64_t slot_i = (int64_t)(pbeg + part) * a.num_heads + hd;
    float* const dst = a.ws_acc + slot_i * D + 4 * half;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4_t*>(dst + 32 * b + 8 * g) =
            float4_t{acc[b][4 * g], acc[b][4 * g + 1], acc[b][4 * g + 2], acc[b][4 * g + 3]};
    if (half == 0) *reinterpret_cast<float2*>(a.ws_ml + slot_i * 2) = make_float2(m, l);
  }
}

// ---------------------------------------------------------------------------
// The same work in fp32: v_mfma_f32_32x32x2_f32 (fp32 products and sums), chunks of
// 32 positions. k index half of a product stands for dim 8 c + 4 half + i of the K rows and
// q (whole 16-byte loads, component by component), and for position 8 (r / 4) + 4 half +
// r % 4 of V and P, whose B operand is then register r of the scores as it is. A
// score's dims are summed in 16 chains, and a chunk's P.V in two, apart from the chunks
// before it, so that rounding stays below the row-by-row kernel's (distance from 64-bit
// results 1.30e-7 against 1.45e-7; 2.2e-7 with two chains and one running sum).
//
// Bound by the fp32 matrix rate (154 TFLOP/s for a library product here). us per
// layer for six prompts of 201..687 tokens at 14 / 2 heads of 64: 47 to 50 with the append,
// against 119 for one work item per row.
template <int D>
struct fshape {
  static constexpr int RB = 4 * D;
  static constexpr int TB = 16 * RB;
  static constexpr int CK = 32;                 // positions per chunk
  static constexpr int HALF = CK * RB;
  static constexpr int SLOT = 2 * HALF;
  static constexpr int PPR = RB / 16;           // 16-byte pieces per row
  static constexpr int RPL = 64 / PPR;          // rows per direct load
  static constexpr int TLD = TB / 1024;
  static constexpr int KC = D / 8;              // 16-byte K chunks of a lane
  static constexpr int NB = D / 32;
  // 16 lanes of a K read touch 16 rows of one piece: spread over the 16 pieces of 64 banks
  static __device__ __forceinline__ int kswz(int r) { return r & 15; }
};

template <int D>
__global__ __launch_bounds__(256, D == 64 ? 2 : 1) void paged_prefill_columns_f32_kernel(const cols_args a) {
  using S = fshape<D>;
  constexpr int RB = S::RB, TB = S::TB, CK = S::CK, KC = S::KC, NB = S::NB, COLS_ = 128;
  extern __shared__ __align__(1024) char flds[];   // two chunks

  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, lcol = lane & 31, half = lane >> 5;
  const int4 w0 = a.work[2 * blockIdx.x], w1 = a.work[2 * blockIdx.x + 1];
  const int row0 = w0.x, seq = w0.y, pos0 = w0.z, nrows = w0.w;
  if (nrows == 0) return;                       // a padding entry (whole workgroup)
  const int col0 = w1.x, kvh = w1.y, part = w1.z, part_chunks = 2 * w1.w;   // the list counts chunks of 64
  const int rep = a.rep, ncols = nrows * rep;
  const int col = col0 + 32 * wave + lcol;
  const bool mine = col < ncols;
  const int ccol = mine ? col : ncols - 1;
  const int my_row = ccol / rep, hd = kvh * rep + ccol - my_row * rep;
  const int my_pos = pos0 + my_row;
  const int wcol = min(col0 + 32 * wave, ncols - 1);
  const bool wave_busy = col0 + 32 * wave < ncols;
  const int wave_first = pos0 + wcol / rep;
  const int wave_last = pos0 + min(col0 + 32 * wave + 31, ncols - 1) / rep;
  const int limit = pos0 + min(col0 + COLS_ - 1, ncols - 1) / rep + 1;
  const int c_begin = part * part_chunks;
  const int c_end = min(c_begin + part_chunks, (limit + CK - 1) / CK);

  vec16 q[KC];                                  // dims 8 c + 4 half .. of the column
  {
    const char* qrow = a.q + (int64_t)(row0 + my_row) * a.q_row_bytes + (int64_t)hd * RB + 16 * half;
#pragma unroll
    for (int c = 0; c < KC; ++c) q[c] = ld16(qrow + 32 * c);
  }
  // ---- direct loads: a chunk's K tiles by waves 0, 1 and its V tiles by waves 2, 3 ----
  const int64_t head_bytes = ((int64_t)1 << a.log2_bs) * RB;
  const int64_t blk_bytes = 2 * (int64_t)a.num_kv_heads * head_bytes;
  const int64_t v_off = a.num_kv_heads * head_bytes;
  const int sub_mask = (1 << (a.log2_bs - 4)) - 1;
  const int32_t* const table = a.block_tables + (int64_t)seq * a.max_nb;
  const int last_tile = (limit - 1) >> 4;
  const int lt = wave & 1;
  const bool is_v = wave >= 2;
  const char* const pool_src = a.pool + kvh * head_bytes + (is_v ? v_off : 0);
  const int lrow = lane / S::PPR, lpiece = lane % S::PPR;
  int id0 = c_begin;
  auto load_ids = [&](int c) {                  // lane j: the block of this wave's tile in chunk c + j
    const int t = min(2 * (c + lane) + lt, last_tile);
    int b = table[(t << 4) >> a.log2_bs];
    return (b < 0 || b >= a.num_blocks) ? 0 : b;   // host validates; stay inside the pool
  };
  int ids = load_ids(id0);
  auto issue = [&](int c, int slot) {
    if (c - id0 >= 64) {
      id0 = c;
      ids = load_ids(id0);
    }
    const int t = min(2 * c + lt, last_tile);
    const int rmax = limit - 1 - 16 * t;
    const int64_t b = __builtin_amdgcn_readlane(ids, c - id0);
    const char* const base = pool_src + b * blk_bytes + (int64_t)(t & sub_mask) * TB;
    char* const dst = flds + slot * S::SLOT + (is_v ? S::HALF : 0) + lt * TB;
#pragma unroll
    for (int i = 0; i < S::TLD; ++i) {
      const int r = S::RPL * i + lrow;
      s_dma16_l2((uint32_t)(min(r, rmax) * RB + 16 * (is_v ? lpiece : lpiece ^ S::kswz(r))), base, dst + 1024 * i);
    }
  };
  asm volatile("" : "+v"(ids));
  if (c_begin < c_end) issue(c_begin, 0);
  if (a.rope.cos) {                             // chunk c pairs with chunk c + KC/2 (dims i and i + D/2)
    const int64_t r = a.rope.row(my_pos, D / 2) + 4 * half;
#pragma unroll
    for (int c = 0; c < KC / 2; ++c)
      rope_pair<float>(q[c], q[c + KC / 2], a.rope.cos + r + 8 * c, a.rope.sin + r + 8 * c);
  }
  if (a.q_sign != 1.f) {
#pragma unroll
    for (int c = 0; c < KC; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) q[c].w[i] = __float_as_uint(bits_to_f32(q[c].w[i]) * a.q_sign);
  }
#pragma unroll
  for (int c = 0; c < KC; ++c)
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(q[c].w[i]));

  float m = -INFINITY, l = 0.f;
  float16_t acc[NB];                            // O^T[32 b + 8 (r / 4) + 4 half + r % 4][col]
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[b][r] = 0.f;
  const float sl2e = a.scale_log2e;
  const int n = c_end - c_begin;
  const int n_wave = wave_busy ? min(c_end - 1, wave_last / CK) - c_begin + 1 : 0;
  for (int k = 0; k < n; ++k) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");   // as the 16-bit kernel
    if (k + 1 < n) issue(c_begin + k + 1, (k + 1) & 1);
    if (k >= n_wave) continue;
    const int c = c_begin + k;
    const char* const base = flds + (k & 1) * S::SLOT;
    float16_t sh[4];                            // chains of D / 16 dims, added pairwise
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      float16_t d4[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) d4[i][r] = 0.f;
#pragma unroll
      for (int cc = h * KC / 4; cc < (h + 1) * KC / 4; ++cc) {
        const vec16 kv = ld16(base + lcol * RB + 16 * ((2 * cc + half) ^ S::kswz(lcol)));
#pragma unroll
        for (int i = 0; i < 4; ++i)
          d4[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(bits_to_f32(kv.w[i]), bits_to_f32(q[cc].w[i]), d4[i], 0, 0, 0);
      }
      sh[h] = (d4[0] + d4[1]) + (d4[2] + d4[3]);
    }
    float16_t sc = (sh[0] + sh[1]) + (sh[2] + sh[3]);
    if (CK * c + CK - 1 > wave_first) {         // the chunk crosses the diagonal of some column
      asm volatile("");
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (CK * c + 8 * (r >> 2) + 4 * half + (r & 3) > my_pos) sc[r] = -INFINITY;
    }
    float cm = max_f32(sc[0], sc[1]);
#pragma unroll
    for (int e = 2; e < 16; e += 2) cm = max3_f32(cm, sc[e], sc[e + 1]);
    cm = max_xor32(cm) * sl2e;
    if (__any(cm > m)) {
      const float m_new = fmaxf(m, cm);
      const float alpha = fast_exp2(m - (m_new == -INFINITY ? 0.f : m_new));   // 0 while m = -inf
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[b] *= alpha;
    }
    const float m_safe = m == -INFINITY ? 0.f : m;
#pragma unroll
    for (int r = 0; r < 16; ++r) sc[r] = fast_exp2(sc[r] * sl2e - m_safe);
    l += (((sc[0] + sc[1]) + (sc[2] + sc[3])) + ((sc[4] + sc[5]) + (sc[6] + sc[7]))) +
         (((sc[8] + sc[9]) + (sc[10] + sc[11])) + ((sc[12] + sc[13]) + (sc[14] + sc[15])));
    const char* const vb = base + S::HALF + 4 * half * RB + 4 * lcol;
    // the chunk's own sums, in two chains: shorter than one over all positions
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      float16_t pv[2];
#pragma unroll
      for (int r = 0; r < 16; ++r) pv[0][r] = pv[1][r] = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        pv[r & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(
            *reinterpret_cast<const float*>(vb + (8 * (r >> 2) + (r & 3)) * RB + 128 * b), sc[r], pv[r & 1], 0, 0, 0);
      acc[b] += pv[0] + pv[1];
    }
  }

  l = sum_xor32(l);
  if (!mine) return;
  const int row = row0 + my_row;
  const int pbeg = a.row_part_off[row], nparts = a.row_part_off[row + 1] - pbeg;
  if (part >= nparts) return;                   // the row ends before this part
  if (nparts == 1) {
    const float inv = 1.f / l;
    char* const orow = a.out + (int64_t)row * a.out_row_bytes + (int64_t)hd * RB + 16 * half;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        st_through(orow + 128 * b + 32 * g, float4_t{acc[b][4 * g], acc[b][4 * g + 1], acc[b][4 * g + 2], acc[b][4 * g + 3]} * inv);
  } else {
    const int64_t slot_i = (int64_t)(pbeg + part) * a.num_heads + hd;
    float* const dst = a.ws_acc + slot_i * D + 4 * half;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4_t*>(dst + 32 * b + 8 * g) =
            float4_t{acc[b][4 * g], acc[b][4 * g + 1], acc[b][4 * g + 2], acc[b][4 * g + 3]};
    if (half == 0) *reinterpret_cast<float2*>(a.ws_ml + slot_i * 2) = make_float2(m, l);
  }
}

}  // namespace tb

// ---------------------------------------------------------------------------
// Host side: the work list (no device call) and the launch.

namespace {

constexpr int COLS = tb::cshape<64>::COLS, CHUNK = tb::cshape<64>::CK;
static_assert(COLS == tb::cshape<128>::COLS && CHUNK == tb::cshape<128>::CK, "one work list for both head dims");

struct col_entry {
  int seq, kvh, col0, part, chunks;
};

bool columns_args_ok(const int32_t* pos0, const int32_t* new_rows, int32_t num_seqs, int32_t num_heads,
                     int32_t num_kv_heads) {
  if (num_seqs < 0 || num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads) return false;
  if (num_seqs > 0 && (!pos0 || !new_rows)) return false;
  for (int i = 0; i < num_seqs; ++i)
    if (pos0[i] < 0 || new_rows[i] <= 0 || (int64_t)pos0[i] + new_rows[i] > (1 << 30) ||
        (int64_t)new_rows[i] * (num_heads / num_kv_heads) > (1 << 28))
      return false;
  return true;
}

// The positions the last row of the columns from col0 on sees.
int columns_limit(int pos0, int new_rows, int rep, int col0) {
  return pos0 + std::min(col0 + COLS - 1, new_rows * rep - 1) / rep + 1;
}

// The column tiles of a step by their chunks: reach[n - 1] tiles (of one kv head) have n or
// more, so that a partition length is priced in longest / length steps.
struct column_tiles {
  std::vector<int32_t> reach;
  int64_t chunks = 0;
  int longest = 0;

  column_tiles(const int32_t* pos0, const int32_t* new_rows, int32_t num_seqs, int rep) {
    auto each = [&](auto&& f) {
      for (int i = 0; i < num_seqs; ++i)
        for (int c = 0; c < new_rows[i] * rep; c += COLS)
          f((columns_limit(pos0[i], new_rows[i], rep, c) + CHUNK - 1) / CHUNK);
    };
    each([&](int n) { longest = std::max(longest, n); });
    reach.assign(longest + 1, 0);
    each([&](int n) { ++reach[n - 1], chunks += n; });
    for (int n = longest - 1; n > 0; --n) reach[n - 1] += reach[n];
  }
  int64_t entries(int part) const {   // of `part` chunks or fewer
    int64_t n = 0;
    for (int64_t at = 0; at < longest; at += part) n += reach[at];
    return n;
  }
};

}  // namespace

namespace {

// What a step of column tiles costs, in us: a workgroup alone on its CU takes 1.0 (head
// dim 64) or 1.6 us a chunk, a full CU 0.65 or 1.05 us per chunk of its workgroups (fp32, at
// the matrix rate either way: 4 or 8 and 3.6 or 7.2, to the proportion that counts here: with
// the sums in short chains they measure 1.5 times that); a split
// adds the merge's launch (5 us) and its rows' partials, written and read (4 bytes/ps).
struct columns_price {
  const column_tiles& tiles;
  bool f32;
  int hkv, cus;
  double alone, full, share, slot_bytes;

  columns_price(const column_tiles& t, int num_heads, int num_kv_heads, int head_dim, int32_t dtype, int num_cus)
      : tiles(t), f32(dtype == TB_DTYPE_F32), hkv(num_kv_heads), cus(num_cus) {
    const bool d64 = head_dim == 64;
    alone = f32 ? (d64 ? 4.0 : 8.0) : d64 ? 1.0 : 1.6;
    full = f32 ? (d64 ? 3.6 : 7.2) : d64 ? 0.65 : 1.05;
    share = full * (double)(tiles.chunks * hkv) / num_cus;
    slot_bytes = (double)num_heads * (head_dim + 2) * 4;
  }
  double one(int chunks) const {   // us a chunk takes the longest workgroup
    const bool two_sets = !f32 && tiles.entries(chunks) * hkv <= cus;   // as launch_columns
    return two_sets ? 0.66 * alone : alone;
  }
  // rows unsplit (chunks == tiles.longest) or in parts of `chunks`, without the merge
  double span(int chunks) const { return std::max(one(chunks) * chunks, share + 0.5 * full * chunks); }
  // the merge of rows in parts of `chunks`, of which `partials` are written and read: it reads
  // eight partials at a time, and each eight more are another round trip
  double merge(int chunks, int64_t partials) const {
    return 5.0 + 3.0 * ((tiles.longest - 1) / chunks / 8) + 2 * partials * slot_bytes / 4e6;
  }
};

// The partitions of a step's rows in parts of `tokens` positions: of split rows, of all rows.
void count_partitions(const int32_t* pos0, const int32_t* new_rows, int num_seqs, int64_t tokens, int64_t* split,
                      int64_t* all) {
  *split = *all = 0;
  for (int i = 0; i < num_seqs; ++i) {
    // rows of k partitions: positions (k - 1) tokens .. k tokens - 1
    const int64_t first = pos0[i], last = first + new_rows[i];
    for (int64_t k = first / tokens + 1; (k - 1) * tokens < last; ++k) {
      const int64_t rows_k = std::min(last, k * tokens) - std::max(first, (k - 1) * tokens);
      *all += k * rows_k;
      if (k > 1) *split += k * rows_k;
    }
  }
}

// The partition of least cost in chunks (past the longest context: no row is split). Measured
// in a graph with the append, bf16, 14 / 2 heads of 64, us per layer: 16 prefix hits
// of 100 rows after 3008 positions 41.4 (45.4 when split at 512 positions), 4 of 30 after
// 704 14.2 (16.9), one fresh prompt of 600 unsplit 16.8 (17.7).
int best_partition(const columns_price& price, const int32_t* pos0, const int32_t* new_rows, int num_seqs,
                   int64_t other_partitions) {
  const int longest = price.tiles.longest;
  int best = longest + 1;
  double cost = price.span(longest);
  for (int part = 4; part < longest; part += part < 16 ? 2 : part < 64 ? 8 : 32) {
    int64_t split, all;
    count_partitions(pos0, new_rows, num_seqs, (int64_t)part * CHUNK, &split, &all);
    // a call without a workspace still finds room: shorter than the tiles' 1024 positions only
    // while the step's partials fit the static scratch
    if (part < 16 && (all + other_partitions) * price.slot_bytes > TB_NOALLOC_SCRATCH_BYTES) continue;
    const double c = price.span(part) + price.merge(part, split);
    if (c < 0.95 * cost) cost = c, best = part;
  }
  return best;
}

bool columns_shape_ok(int32_t head_dim, int32_t dtype) {
  return (head_dim == 64 || head_dim == 128) &&
         (dtype == TB_DTYPE_F32 || dtype == TB_DTYPE_F16 || dtype == TB_DTYPE_BF16);
}

}  // namespace

extern "C" int32_t tb_prefill_columns_partition(const int32_t* pos0, const int32_t* new_rows, int32_t num_seqs,
                                                int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
                                                int32_t dtype, int32_t num_cus, int32_t other_partitions) {
  if (!columns_args_ok(pos0, new_rows, num_seqs, num_heads, num_kv_heads) || num_cus <= 0 || other_partitions < 0)
    return TB_ERR_INVALID_ARG;
  if (!columns_shape_ok(head_dim, dtype)) return TB_ERR_INVALID_ARG;
  try {
    const column_tiles tiles(pos0, new_rows, num_seqs, num_heads / num_kv_heads);
    const columns_price price(tiles, num_heads, num_kv_heads, head_dim, dtype, num_cus);
    return best_partition(price, pos0, new_rows, num_seqs, other_partitions) * CHUNK;
  } catch (const std::exception&) {   // no memory for a step of this size
    return TB_ERR_INVALID_ARG;
  }
}

// The two routes priced, in us without the launch and append they share. Fitted to times in a
// graph of both routes for 1128 steps (1 to 16 prompts of 16 to 4000 rows after 0 to 8000
// positions, alone and beside 4 to 40 decode rows, 1 to 8 heads per kv head, head dims 64 and
// 128); the route taken is then within 5% of the better one for 97% of them. What it comes to,
// us per layer with the append:
// - beside other rows the column tiles are a launch of their own, where tiles and work items
//   share one: bf16, 14 / 2 heads of 64, 4 decode rows: a prompt of 40 18.5 (tiles 11.5), of 3000
//   50.1 (49.6), 4 of 1500 43.5 (51.6), 8 of 1500 70.6 (95.8);
// - at head dim 64, fresh prompts the tiles take whole (1024 positions): 4 of 700 20.3
//   (19.2), 16 of 700 40.7 (43.8); with one head per kv head 16 of 850 56.8 (51.4);
// - fp32: prompts of 16 to 200 rows 11.8..30.7 (work items 8.5..15.7), 16 of 100 21 (31).
static int32_t columns_pay(const int32_t* pos0, const int32_t* new_rows, int32_t num_seqs, int32_t num_heads,
                           int32_t num_kv_heads, int32_t head_dim, int32_t dtype, int32_t num_cus,
                           int32_t tiles_served, int32_t beside_others) {
  if (!columns_args_ok(pos0, new_rows, num_seqs, num_heads, num_kv_heads) || num_cus <= 0) return TB_ERR_INVALID_ARG;
  if (!columns_shape_ok(head_dim, dtype)) return TB_ERR_INVALID_ARG;
  if (num_seqs == 0) return 0;
  const bool d64 = head_dim == 64, f32 = dtype == TB_DTYPE_F32;
  const int rep = num_heads / num_kv_heads;
  const column_tiles tiles(pos0, new_rows, num_seqs, rep);
  const columns_price price(tiles, num_heads, num_kv_heads, head_dim, dtype, num_cus);
  const int part = best_partition(price, pos0, new_rows, num_seqs, 0), chunks = std::min(part, tiles.longest);
  const bool split = part <= tiles.longest;
  int64_t split_parts = 0, all_parts = 0;
  if (split) count_partitions(pos0, new_rows, num_seqs, (int64_t)part * CHUNK, &split_parts, &all_parts);
  double columns = split ? price.merge(part, split_parts) : 0.0;
  // a launch of its own, while the merge is there anyway (fp32: the others' chain is the longer one)
  if (beside_others) columns += !split ? 6.0 : !f32 ? 1.0 : d64 ? 5.0 : 8.0;
  double other = 0.0;
  if (f32) {
    // in the kernel's own chunks of 32, by the waves that have columns
    int64_t longest_half = 0, busy = 0;
    for (int i = 0; i < num_seqs; ++i)
      for (int c = 0; c < new_rows[i] * rep; c += COLS) {
        const int64_t n = (columns_limit(pos0[i], new_rows[i], rep, c) + 31) / 32;
        longest_half = std::max(longest_half, n);
        busy += n * ((std::min(COLS, new_rows[i] * rep - c) + 31) / 32);
      }
    columns += 1.0 + std::max((d64 ? 3.1 : 5.3) * (split ? 2 * chunks : longest_half),
                              (d64 ? 2.9 : 6.0) * (0.25 * busy * num_kv_heads / num_cus + chunks));
    int64_t longest_ctx = 0, items = 0, reads = 0, kv = 0;   // work items, positions they read, the pool's positions
    for (int i = 0; i < num_seqs; ++i) {
      const int64_t n = new_rows[i], c = (int64_t)pos0[i] + n;
      longest_ctx = std::max(longest_ctx, c);
      items += n * ((c + 255) / 256);
      reads += n * pos0[i] + n * (n + 1) / 2;
      kv += c;
    }
    int group = d64 ? 14 : 15;                         // heads per workgroup (tb_paged_attention)
    while (rep % group) --group;
    const double wgs = (double)items * num_kv_heads * (rep / group), kr = 1e-3 * reads * num_kv_heads * (rep / group);
    const bool brief = longest_ctx <= 64 && !beside_others;
    if (group <= (brief ? 8 : 5) && wgs >= (brief ? 128 : 320) * group) {   // the VALU kernel
      const double chain = (9.0 + 4.0 * group) * (beside_others ? 1.0 : std::min<int64_t>(longest_ctx, 256) / 256.0);
      other = (d64 ? 1.0 : 2.0) * (0.6 * chain + 0.00025 * (1 + group) * wgs + (0.0058 + 0.0087 * group) * kr) +
              0.35e-3 * std::max(0.0, (double)kv * num_kv_heads - (d64 ? 50e3 : 25e3));   // K/V past the L2s
    } else {
      other = d64 ? 0.0045 * wgs + 0.058 * kr : 0.0055 * wgs + 0.12 * kr;
    }
    if (longest_ctx > 256 && !beside_others) other += 5.0;
    return columns < 0.92 * other;
  }
  // columns: a workgroup's rows cross the diagonal over rows / 64 chunks, of which its waves
  // use a part
  const double cross = 2.0 * COLS / rep / 64;
  const double share = price.share + price.full * cross * (double)tiles.entries(tiles.longest) * num_kv_heads / num_cus;
  columns += 2.0 + std::max(price.one(part) * (chunks + cross), share + 0.5 * price.full * chunks);
  // 64-row tiles of one head in parts of 1024 positions; longer tails as work items
  int group = 16;
  while (rep % group) --group;
  const int rows_per_item = std::max(1, 16 / group);
  int64_t tile_chunks = 0, items = 0, partials = 0;
  int longest = 0;
  bool merge = false;
  for (int i = 0; i < num_seqs; ++i) {
    const int64_t n = new_rows[i], c = (int64_t)pos0[i] + n;
    if (!tiles_served || (c > 4096 && c > 16 * n)) {   // metadata.tiles_sequence
      items += (n + rows_per_item - 1) / rows_per_item * ((c + 255) / 256) * num_kv_heads * (rep / group);
      partials += n * ((c + 255) / 256);
      merge |= c > 256;
      continue;
    }
    for (int64_t r = 0; r < n; r += 64) {
      const int64_t end = pos0[i] + std::min<int64_t>(n, r + 64), whole = end / 1024, rest = end % 1024;
      tile_chunks += whole * 16 + (rest + 63) / 64;
      longest = std::max(longest, whole ? 16 : (int)((rest + 63) / 64));
      if (end > 1024) partials += 64 * ((end + 1023) / 1024), merge = true;
    }
  }
  const double tile_alone = d64 ? 0.82 : 3.1, tile_full = d64 ? 0.61 : 1.6;
  const double tile_share = tile_full * (double)(tile_chunks * num_heads) / num_cus;
  if (longest > 0)
    other += std::max(tile_alone * longest + (d64 ? 0.3 : 0.75) * tile_share, tile_share + 0.3 * tile_full * longest);
  other += (d64 ? 0.0135 : 0.028) * items + partials * price.slot_bytes / 4e6;
  if (merge && !beside_others) other += 5.0;
  return columns < 0.97 * other;
}

extern "C" int32_t tb_prefill_columns_pay(const int32_t* pos0, const int32_t* new_rows, int32_t num_seqs,
                                          int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, int32_t dtype,
                                          int32_t num_cus, int32_t tiles_served, int32_t beside_others) {
  try {
    return columns_pay(pos0, new_rows, num_seqs, num_heads, num_kv_heads, head_dim, dtype, num_cus, tiles_served,
                       beside_others);
  } catch (const std::exception&) {
    return TB_ERR_INVALID_ARG;
  }
}

static int32_t build_columns_work(const int32_t* first_row, const int32_t* seq_index, const int32_t* pos0,
                                  const int32_t* new_rows, int32_t num_seqs, int32_t num_heads, int32_t num_kv_heads,
                                  int32_t partition_tokens, int32_t num_xcds, int32_t num_cus, int32_t* work,
                                  int32_t capacity, int32_t* count) {
  if (!columns_args_ok(pos0, new_rows, num_seqs, num_heads, num_kv_heads) || !count || num_xcds <= 0 || num_cus <= 0)
    return TB_ERR_INVALID_ARG;
  if (num_seqs > 0 && (!first_row || !seq_index)) return TB_ERR_INVALID_ARG;
  if (partition_tokens < CHUNK || partition_tokens % CHUNK) return TB_ERR_INVALID_ARG;
  for (int i = 0; i < num_seqs; ++i)
    if (first_row[i] < 0 || seq_index[i] < 0) return TB_ERR_INVALID_ARG;
  const int rep = num_heads / num_kv_heads, pc = partition_tokens / CHUNK;
  std::vector<col_entry> entries;
  int64_t total = 0;
  for (int h = 0; h < num_kv_heads; ++h)
    for (int i = 0; i < num_seqs; ++i)
      for (int c = 0; c < new_rows[i] * rep; c += COLS) {
        const int n = (columns_limit(pos0[i], new_rows[i], rep, c) + CHUNK - 1) / CHUNK;
        for (int p = 0; p * pc < n; ++p) {
          entries.push_back({i, h, c, p, std::min(pc, n - p * pc)});
          total += entries.back().chunks + 2;            // + 2: a workgroup's start and end
        }
      }
  // Entry g runs on XCD g % num_xcds: the entries in (kv head, sequence) order are cut into
  // runs of equal work, one per XCD, so that few K/V ranges pass through each L2; up to one
  // entry per CU, into runs of equal length (every entry then has a CU).
  const bool one_each = (int64_t)entries.size() <= num_cus;
  if (one_each) total = (int64_t)entries.size();
  const int X = num_xcds, per = std::max(1, num_cus / X);
  std::vector<std::vector<col_entry>> bins(X);
  int64_t at = 0;
  for (const col_entry& e : entries) {
    const int64_t w = one_each ? 1 : e.chunks + 2;
    bins[std::min<int64_t>(X - 1, (2 * at + w) * X / (2 * total))].push_back(e);
    at += w;
  }
  size_t rounds = 0;
  for (auto& b : bins) {
    // longest first, and every second round of one entry per CU reversed: a CU holds two or
    // three workgroups at once, and its long first one then has a short second one
    std::stable_sort(b.begin(), b.end(), [](const col_entry& x, const col_entry& y) { return x.chunks > y.chunks; });
    for (size_t r = per; r + per <= b.size(); r += 2 * per) std::reverse(b.begin() + r, b.begin() + r + per);
    rounds = std::max(rounds, b.size());
  }
  const int64_t n = (int64_t)rounds * X;
  if (n > INT32_MAX) return TB_ERR_INVALID_ARG;
  *count = (int32_t)n;
  if (!work) return TB_OK;                             // the count alone
  if (n > capacity) return TB_ERR_INVALID_ARG;
  for (size_t r = 0; r < rounds; ++r)
    for (int x = 0; x < X; ++x) {
      int32_t* w = work + 8 * (r * X + x);
      if (r >= bins[x].size()) {
        std::fill(w, w + 8, 0);                          // no rows: the workgroup ends at once
        continue;
      }
      const col_entry& e = bins[x][r];
      w[0] = first_row[e.seq];
      w[1] = seq_index[e.seq];
      w[2] = pos0[e.seq];
      w[3] = new_rows[e.seq];
      w[4] = e.col0;
      w[5] = e.kvh;
      w[6] = e.part;
      w[7] = pc;
    }
  return TB_OK;
}

extern "C" int32_t tb_build_prefill_columns_work(const int32_t* first_row, const int32_t* seq_index, const int32_t* pos0,
                                                 const int32_t* new_rows, int32_t num_seqs, int32_t num_heads,
                                                 int32_t num_kv_heads, int32_t partition_tokens, int32_t num_xcds,
                                                 int32_t num_cus, int32_t* work, int32_t capacity, int32_t* count) {
  try {
    return build_columns_work(first_row, seq_index, pos0, new_rows, num_seqs, num_heads, num_kv_heads,
                              partition_tokens, num_xcds, num_cus, work, capacity, count);
  } catch (const std::exception&) {
    return TB_ERR_INVALID_ARG;
  }
}

namespace {

// The CUs of the current device (asked once; 256 where that fails).
int device_cus() {
  constexpr int MAX_DEVICES = 64;
  static std::atomic<int> cus[MAX_DEVICES];
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return 256;
  if ((n = cus[dev].load(std::memory_order_relaxed)) > 0) return n;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
  cus[dev].store(n, std::memory_order_relaxed);
  return n;
}

// At most one workgroup per CU: two sets of waves share its chunks, which then take
// 0.66 us each instead of 1.0 (head dim 64). Twelve prefix hits of 40..400 rows after
// 600..3600 positions, 4 fp16 layers with the append: 149 us unsplit against 162 for one set
// of waves and rows split at 896 positions. Past one per CU (256) one set each leaves room
// for a second workgroup on the CU, whose start and end then overlap.
template <typename Tag, int D, bool SIGNED>
void launch_columns_sets(const tb::cols_args& a, int num_work, hipStream_t stream) {
  constexpr int T = 64 * tb::cshape<D>::NW;
  if (num_work <= device_cus())
    hipLaunchKernelGGL((tb::paged_prefill_columns_kernel<Tag, D, 2, SIGNED>), dim3(num_work), dim3(2 * T), 0, stream, a);
  else
    hipLaunchKernelGGL((tb::paged_prefill_columns_kernel<Tag, D, 1, SIGNED>), dim3(num_work), dim3(T), 0, stream, a);
}

template <typename Tag, int D>
void launch_columns(const tb::cols_args& a, int num_work, hipStream_t stream) {
  a.q_sign == 1.f ? launch_columns_sets<Tag, D, false>(a, num_work, stream)
                  : launch_columns_sets<Tag, D, true>(a, num_work, stream);
}

}  // namespace

extern "C" int32_t tb_paged_prefill_columns(const void* q, int64_t q_row_stride, const void* pool, int64_t num_blocks,
                                            void* out, int64_t out_row_stride, const int32_t* block_tables,
                                            int32_t max_blocks_per_seq, const int32_t* work, int32_t num_work,
                                            const int32_t* row_part_offsets, int32_t num_rows,
                                            const int32_t* split_rows, int32_t num_split_rows,
                                            int32_t max_parts_per_row, int32_t total_partitions, int32_t num_heads,
                                            int32_t num_kv_heads, int32_t head_dim, int32_t block_size, float scale,
                                            int32_t dtype, void* workspace, size_t workspace_bytes,
                                            const float* rope_cos, const float* rope_sin, int32_t rope_max_position,
                                            hipStream_t stream) {
  using namespace tb;
  TB_CHECK_ARG(num_work >= 0 && num_rows >= 0 && num_split_rows >= 0 && num_split_rows <= num_rows);
  TB_CHECK_ARG(num_heads > 0 && num_kv_heads > 0 && num_heads % num_kv_heads == 0);
  if (num_work == 0) return TB_OK;
  const int eb = dtype == TB_DTYPE_F32 ? 4 : dtype == TB_DTYPE_F16 || dtype == TB_DTYPE_BF16 ? 2 : 0;
  TB_CHECK_ARG(eb > 0);
  if (head_dim != 64 && head_dim != 128) return TB_ERR_UNSUPPORTED;
  if (block_size < 16 || (block_size & (block_size - 1))) return TB_ERR_UNSUPPORTED;
  TB_CHECK_ARG(q && pool && out && block_tables && work && row_part_offsets && num_rows > 0);
  TB_CHECK_ARG(num_blocks > 0 && max_blocks_per_seq > 0 && max_parts_per_row >= 0 && total_partitions >= 0);
  TB_CHECK_ARG(q_row_stride >= (int64_t)num_heads * head_dim && out_row_stride >= (int64_t)num_heads * head_dim);
  TB_CHECK_ARG((((uintptr_t)q | (uintptr_t)pool | (uintptr_t)out | (uintptr_t)work) & 15u) == 0);
  TB_CHECK_ARG((q_row_stride * eb) % 16 == 0 && (out_row_stride * eb) % 16 == 0);
  TB_CHECK_ARG(num_split_rows == 0 || (split_rows && max_parts_per_row > 1));
  TB_CHECK_ARG(((uintptr_t)split_rows & 15u) == 0);
  TB_CHECK_ARG(!rope_cos == !rope_sin && (!rope_cos || rope_max_position > 0));
  TB_CHECK_ARG((((uintptr_t)rope_cos | (uintptr_t)rope_sin) & 15u) == 0);
  void* ws = nullptr;
  if (max_parts_per_row > 1) {
    const size_t need = tb_paged_attention_workspace_bytes(total_partitions, num_heads, head_dim);
    ws = workspace;
    if (!ws) {                                           // the library's static scratch
      if (need > (size_t)TB_NOALLOC_SCRATCH_BYTES) return TB_ERR_SCRATCH;
      const int32_t st = noalloc_scratch(stream, &ws);
      if (st != TB_OK) return st;
    } else {
      TB_CHECK_ARG(workspace_bytes >= need && ((uintptr_t)ws & 15u) == 0);
    }
  }
  cols_args a{};
  a.q = static_cast<const char*>(q);
  a.q_row_bytes = q_row_stride * eb;
  a.pool = static_cast<const char*>(pool);
  a.num_blocks = num_blocks;
  a.out = static_cast<char*>(out);
  a.out_row_bytes = out_row_stride * eb;
  a.block_tables = block_tables;
  a.max_nb = max_blocks_per_seq;
  a.work = reinterpret_cast<const int4*>(work);
  a.row_part_off = row_part_offsets;
  a.ws_acc = static_cast<float*>(ws);
  a.ws_ml = ws ? a.ws_acc + (size_t)total_partitions * num_heads * head_dim : nullptr;
  a.num_heads = num_heads;
  a.num_kv_heads = num_kv_heads;
  a.rep = num_heads / num_kv_heads;
  while ((1 << a.log2_bs) < block_size) ++a.log2_bs;
  a.scale_log2e = scale > 0.f || scale < 0.f ? fabsf(scale) * 1.4426950408889634f : 1.f;
  a.q_sign = scale > 0.f ? 1.f : scale < 0.f ? -1.f : scale * 0.f;
  a.rope = rope_tables{rope_cos, rope_sin, rope_max_position};
  const bool d64 = head_dim == 64;
  if (dtype == TB_DTYPE_F32) {
    const dim3 grid(num_work), block(256);
    if (d64) hipLaunchKernelGGL((paged_prefill_columns_f32_kernel<64>), grid, block, 2 * fshape<64>::SLOT, stream, a);
    else hipLaunchKernelGGL((paged_prefill_columns_f32_kernel<128>), grid, block, 2 * fshape<128>::SLOT, stream, a);
  } else if (dtype == TB_DTYPE_F16) {
    d64 ? launch_columns<f16_t, 64>(a, num_work, stream) : launch_columns<f16_t, 128>(a, num_work, stream);
  } else {
    d64 ? launch_columns<bf16_t, 64>(a, num_work, stream) : launch_columns<bf16_t, 128>(a, num_work, stream);
  }
  if (num_split_rows > 0)
    combine_split_rows(dtype, head_dim, num_heads, out, out_row_stride * eb, split_rows, num_split_rows, a.ws_acc, a.ws_ml,
                       stream);
  TB_RETURN_LAUNCH_STATUS();
}
