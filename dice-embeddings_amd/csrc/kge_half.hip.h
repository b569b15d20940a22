// The fp32 contractions of a training step on the fp16 MFMA (gfx950).
//
// A value x of an operand whose largest magnitude lies below 2^(15 - s) is kept as
//   x 2^s = h + l 2^-11,   h = fp16(x 2^s),   l = fp16((x 2^s - h) 2^11)       (both to nearest even)
// and a product is taken as the three leading part products, in two fp32 accumulators:
//   main += h h'       cross += h l' + l h'       x x' = (main + cross 2^-11) 2^-(s + s')
// l is as large as h, so neither loses places to fp16's narrow range before the other: a value keeps 22 - 23 bits down to
// 2^-29 of its operand's largest, and below that an absolute 2^-50 of it.  The dropped l l' and the rounding of l are each
// below 2^-22 of x x'; what the six bf16 products of ksplit_kernel add to their exact parts is the rounding of six
// accumulations per K step, where this has one in `main` and two, 2^-11 as heavy, in `cross`.
//
// Used where a result is the sum of many products and is not compared bit for bit with another kernel's: the score gradients
// and the two gradient products of a BCE step.  Scores that are ranked or returned keep the bf16 chain.
//
// Operands are matrices of split rows: 32 columns of a row are one line of 128 bytes, their 32 h, then their 32 l; a row is
// padded with zeros to whole lines (the table and the queries are split once per step, the score gradients are written so by
// the kernel that forms them).  What reads them then converts nothing: lines go global -> LDS and fragments LDS -> MFMA.
#pragma once
#include "kge_contract.hip.h"

namespace kge {

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) _Float16 f16x4;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;

using host::HALF_SLOTS;
constexpr int HALF_TOP = 14;  // the largest magnitude of a scaled operand lies in [2^14, 2^15)

// The power of two (its exponent) that brings magnitudes up to `bits` below 2^15; between 2^-113 and 2^116, so that it and
// 2^11 times it are normal numbers.
__device__ __forceinline__ int half_exponent(uint32_t bits) {
  const int e = HALF_TOP + 127 - (int)(bits >> 23);
  return e < 116 ? e : 116;
}
__device__ __forceinline__ float pow2f(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }

// Where a launch's exponents come from: the step's (written by half_split_kernel), or null: the given ones.
struct HalfArgs {
  const int32_t* exp_e;
  const int32_t* exp_q;
  int fixed_e, fixed_q;
  // StoreTEpi: the workgroups from tail_first on take the chunks from tail_chunk (= a.n_chunks) on, tail_splits of them a tile, each a range of
  // K; their sums go to tail + range * tail_stride (host::half_tail)
  int64_t tail_first, tail_chunk, tail_stride;
  int tail_splits, tail_len;
  float* tail;
  int k_splits;  // StoreEpi: the ranges K is summed in
};

// h and l of one value x whose product with `up` = 2^s lies below 2^15 (up_2k: 2^(s + 11)); the residual and its factor 2^11
// are one exact fused multiply-add
__device__ __forceinline__ void half_parts(float x, float up, float up_2k, _Float16& h, _Float16& l) {
  h = (_Float16)(x * up);
  l = (_Float16)__builtin_fmaf((float)h, -2048.f, x * up_2k);
}

// ---- before the contractions: the largest magnitudes, then the split rows --------------------------------------------
// One slot per workgroup: the first HALF_SLOTS workgroups take E, the rest Q (rows are whole 16-byte pieces, values that are
// not finite do not count); beside that what bce_init_kernel clears, and in the workgroups
// behind those a step's preparations.
constexpr int HALF_MAX_THREADS = 512;
__global__ void __launch_bounds__(HALF_MAX_THREADS) half_max_kernel(const float* E, int64_t n_e, const float* Q, int64_t n_q,
                                                                   uint32_t* slots, double* sums, int n_sums, float* dbias,
                                                                   int64_t B, StepPrepare prep) {
  if (blockIdx.x >= 2 * HALF_SLOTS) {
    step_prepare(prep, blockIdx.x - 2 * HALF_SLOTS, gridDim.x - 2 * HALF_SLOTS);
    return;
  }
  const int64_t gid = (int64_t)blockIdx.x * HALF_MAX_THREADS + threadIdx.x;
  if (gid < n_sums) sums[gid] = 0.0;
  if (dbias)
    for (int64_t i = gid; i < B; i += (int64_t)2 * HALF_SLOTS * HALF_MAX_THREADS) dbias[i] = 0.f;
  const bool second = blockIdx.x >= HALF_SLOTS;
  const f32x4* x = (const f32x4*)(second ? Q : E);
  const int64_t n = (second ? n_q : n_e) >> 2;
  constexpr int U = 8;
  constexpr int64_t STRIDE = (int64_t)HALF_SLOTS * HALF_MAX_THREADS;
  uint32_t m = 0;
  auto take = [&](f32x4 v) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t u = __float_as_uint(v[j]) & 0x7fffffffu;
      u = u < 0x7f800000u ? u : 0u;
      m = m > u ? m : u;
    }
  };
  int64_t i = (int64_t)(blockIdx.x & (HALF_SLOTS - 1)) * HALF_MAX_THREADS + threadIdx.x;
  for (; i + (U - 1) * STRIDE < n; i += U * STRIDE) {
    f32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = x[i + u * STRIDE];
#pragma unroll
    for (int u = 0; u < U; ++u) take(v[u]);
  }
  for (; i < n; i += STRIDE) take(x[i]);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const uint32_t other = (uint32_t)__shfl_xor((int)m, o, 64);
    m = m > other ? m : other;
  }
  __shared__ uint32_t part[HALF_MAX_THREADS / 64];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < HALF_MAX_THREADS / 64; ++w) m = m > part[w] ? m : part[w];
    slots[blockIdx.x] = m;
  }
}

// rows x cols fp32 -> split rows of `lines` lines, zeros from `rows` up to rows_padded; a workgroup is 32 groups of eight lanes,
// a group takes a line at a time, a lane four columns of it.
struct HalfSplit {
  const float* x;
  unsigned char* out;
  int64_t rows, rows_padded;
  int cols, lines;
};
__global__ void __launch_bounds__(256) half_split_kernel(HalfSplit e, HalfSplit q, unsigned blocks_e, const uint32_t* slots,
                                                       int32_t* exps) {
  const bool second = blockIdx.x >= blocks_e;
  const HalfSplit s = second ? q : e;
  const int lane = threadIdx.x & 63;
  const u32x4 v4 = *(const u32x4*)(slots + (second ? HALF_SLOTS : 0) + 4 * lane);
  static_assert(HALF_SLOTS == 256, "four slots per lane");
  uint32_t m = v4[0] > v4[1] ? v4[0] : v4[1];
  m = m > v4[2] ? m : v4[2];
  m = m > v4[3] ? m : v4[3];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const uint32_t other = (uint32_t)__shfl_xor((int)m, o, 64);
    m = m > other ? m : other;
  }
  const int ex = half_exponent(m);
  if (threadIdx.x == 0 && (blockIdx.x == 0 || blockIdx.x == blocks_e)) exps[second ? 1 : 0] = ex;
  const float up = pow2f(ex), up_2k = pow2f(ex + 11);
  const unsigned blk = second ? blockIdx.x - blocks_e : blockIdx.x, blks = second ? gridDim.x - blocks_e : blocks_e;
  const uint32_t n = (uint32_t)(s.rows_padded * s.lines);  // (host::half_pays keeps it below 2^31)
  const int sub = threadIdx.x & 7;
  constexpr int U = 4;
  const uint32_t stride = blks * 32;
  for (uint32_t i0 = blk * 32 + (threadIdx.x >> 3); i0 < n; i0 += U * stride) {
    f32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i = i0 + u * stride, row = i / (uint32_t)s.lines;
      const int col = (int)(i - row * (uint32_t)s.lines) * 32 + 4 * sub;
      const bool in = i < n && row < s.rows && col < s.cols;
      v[u] = *(const f32x4*)(s.x + (in ? (int64_t)row * s.cols + col : 0));
#pragma unroll
      for (int j = 0; j < 4; ++j) v[u][j] = in ? v[u][j] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i = i0 + u * stride;
      if (i >= n) break;
      f16x4 h, l;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        _Float16 hh, ll;
        half_parts(v[u][j], up, up_2k, hh, ll);
        h[j] = hh;
        l[j] = ll;
      }
      unsigned char* to = s.out + (int64_t)i * 128 + sub * 8;
      *(f16x4*)to = h;
      *(f16x4*)(to + 64) = l;
    }
  }
}

// ---- the score gradients -----------------------------------------------------------------------------------------------
// GradEpi's sums, and its gradients as split rows of ldG columns: zeros in the columns past N of the last line, and in the
// rows past B up to the next 32.  What bounds the kernel is the vector instructions of this epilogue beside the matrix cores (2048 x 40,943,
// d = 256: 154k of a SIMD's cycles against 123k of MFMAs), so the scale of the scores and their bias are two fused
// multiply-adds, the gradient is formed at its scale, and a row's address is a scalar.
struct GradSplitArgs {
  const float* bias;
  double* sums;      // as BceArgs::sums
  unsigned char* G;
  float* dbias;      // [B], zero-initialised; read by GradSplitBiasEpi only
  int64_t ldG;
  float c, uniform;  // gradient / 2^-s = c sigmoid - uniform (c: upstream gradient / (B N) times 2^s)
  float down;        // 2^-s
  int32_t want_s;
};
template <int NQT, bool DBIAS>
struct GradSplitEpiT {
  static constexpr bool SWAP = true;
  static constexpr bool STAGE_HOOK = false;
  static constexpr bool DEFER = false;
  __device__ void stage_mark() {}
  __device__ void stage_end() {}
  using Args = GradSplitArgs;
  struct Shared {
    float bias[8 * 32 * NQT];
  };
  Args a;
  const float* lb;
  float rowsum[DBIAS ? NQT : 1][16];
  double sp, ss;
  int64_t q0, B;
  int c, hf;
  __device__ void init(const Args& args, int64_t q0_, int c_, int hf_, int64_t B_) {
    a = args; q0 = q0_; c = c_; hf = hf_; B = B_;
    sp = 0.0; ss = 0.0;
#pragma unroll
    for (int t = 0; t < (DBIAS ? NQT : 1); ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) rowsum[t][i] = 0.f;
  }
  __device__ void bind(Shared* sh) {
    float* mine = sh->bias + (threadIdx.x >> 6) * (32 * NQT);
    for (int j = (threadIdx.x & 63); j < 32 * NQT; j += 64) {
      const int64_t q = q0 + j;
      mine[j] = (a.bias && q < B) ? a.bias[q] : 0.f;
    }
    lb = mine;
    __syncthreads();
  }
  // acc[i], cross[i]: query row_of(i, hf) of tile qt, entity e_base + c; score = acc up + cross up_2k + bias
  __device__ __forceinline__ void tile_split(int qt, const f32x16& acc, const f32x16& cross, float up, float up_2k,
                                             int64_t e_base, int64_t limit) {
    tile_of(qt, e_base, limit, [&](int i, float b) { return __builtin_fmaf(acc[i], up, __builtin_fmaf(cross[i], up_2k, b)); });
  }
  // the same behind ksplit_kernel
  template <bool HAS_SCALE>
  __device__ __forceinline__ void tile(int qt, const f32x16& acc, const float*, float, int64_t e_base, int64_t limit) {
    static_assert(!HAS_SCALE, "fp32 tables only");
    tile_of(qt, e_base, limit, [&](int i, float b) { return acc[i] + b; });
  }
  template <class Score>
  __device__ __forceinline__ void tile_of(int qt, int64_t e_base, int64_t limit, Score score) {
    if (q0 + 32 * qt >= B) return;
    const bool full = q0 + 32 * qt + 32 <= B && e_base + 32 <= limit;  // the same for the wave: one branch
    const bool col_ok = e_base + c < limit;
    const int64_t pitch = 4 * a.ldG;  // bytes
    unsigned char* row0 = a.G + (q0 + 32 * qt) * pitch + 4 * e_base;             // the same for the wave
    // Stores: a lane's element is two bytes of each part; lanes c and c ^ 1 exchange theirs of two rows, so that the even one
    // stores both columns of the first row, the odd one of the second, four bytes each.
    const uint32_t in_row = (uint32_t)((4 * hf + (c & 1)) * (int)pitch + 4 * (c >> 1));
    const uint32_t pick = (c & 1) ? 0x03020706u : 0x05040100u;  // of {the other's two rows, mine}
    float tpos = 0.f, tss = 0.f, prod = 1.f;  // one logarithm for the sixteen elements, as in BceEpi
    auto body = [&](auto masked) {
      constexpr bool MASKED = decltype(masked)::value;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 b4 = *(const f32x4*)(lb + 32 * qt + 8 * g + 4 * hf);
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
          f16x2 h, l;
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int i = 4 * g + r + j;
            const float v = score(i, b4[r + j]);
            const bool ok = !MASKED || (col_ok && q0 + 32 * qt + row_of(i, hf) < B);
            const float ex = __expf(-fabsf(v));                       // in (0, 1]
            const float sig = quotient_1_2(v >= 0.f ? 1.0f : ex, 1.0f + ex);  // sigmoid without overflow
            float gr = __builtin_fmaf(sig, a.c, -a.uniform);
            if (MASKED) gr = ok ? gr : 0.f;
            prod = __builtin_fmaf(prod, ok ? ex : 0.f, prod);
            tpos += ok ? fmaxf(v, 0.f) : 0.f;
            tss += ok ? v : 0.f;
            if constexpr (DBIAS) rowsum[qt][i] += gr;
            h[j] = (_Float16)gr;
            l[j] = (_Float16)__builtin_fmaf((float)h[j], -2048.f, gr * 2048.f);
          }
          unsigned char* to = row0 + (8 * g + r) * pitch + in_row;
          auto put = [&](f16x2 mine, int part) {
            const uint32_t m = __builtin_bit_cast(uint32_t, mine);
            const uint32_t other = (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0xB1, 0xf, 0xf, false);  // lanes 1, 0, 3, 2
            __builtin_nontemporal_store(__builtin_amdgcn_perm(other, m, pick), (uint32_t*)(to + 64 * part));  // (the table stays in L2)
          };
          put(h, 0);
          put(l, 1);
        }
      }
    };
    if (full) body(std::false_type{});
    else body(std::true_type{});
    sp += (double)(tpos + __logf(prod));
    ss += (double)tss;
  }
  __device__ void finish() {
    double x = sp, y = ss;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      x += __shfl_xor(x, o, 64);
      y += __shfl_xor(y, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
      const int slot = (int)((blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) & (BCE_SLOTS - 1));
      atomicAdd(&a.sums[slot], x);
      if (a.want_s) atomicAdd(&a.sums[BCE_SLOTS + slot], y);
    }
    if constexpr (DBIAS) {
#pragma unroll
      for (int t = 0; t < NQT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          float v = rowsum[t][i];
#pragma unroll
          for (int o = 16; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);  // over the 32 entity columns of this half
          const int64_t q = q0 + 32 * t + 8 * (i >> 2) + 4 * hf + (i & 3);
          if (c == 0 && q < B) atomicAdd(&a.dbias[q], v * a.down);
        }
    }
  }
};
template <int NQT>
using GradSplitEpi = GradSplitEpiT<NQT, false>;
template <int NQT>
using GradSplitBiasEpi = GradSplitEpiT<NQT, true>;  // with the row sums of the gradient

// ---- the contraction ---------------------------------------------------------------------------------------------------
// 128 x 128 scores per workgroup of 4 waves, 64 x 64 per wave, K in chunks of 32 columns: a line per row.  Two LDS buffers of
// 32 KB, two workgroups per CU, so that one's epilogue and waits run beside the other's products; a chunk's lines are requested
// while the chunk before is multiplied; one barrier per chunk.  Per chunk a wave reads 16 fragments for 24 MFMAs.  (256 entities
// per workgroup of 8 waves, three buffers, a chunk two ahead: 258 / 151 / 217 us for the three products of a step of 2048 x 40,943,
// d = 256, against 236 / 147 / 169.)
//
// a.E / a.Q are split rows of pitch lde / ldq columns; K is a.d columns (a multiple of 32), zeros past the operands' own in at
// least one of them.  Nothing is clamped: the rows of either operand are allocated up to whole tiles, what lies past the valid
// ones is read into scores that no epilogue stores (host::bwd_plan lays the workspace out so).
// KMAJ (bit 0: the entity operand, bit 1: the query operand): the operand is K-major, X[k][row] with its rows along the lines.
//
// LDS, row-major operand: row r is its line, 8 pieces of 16 bytes, piece p kept at p ^ (r & 7).  K-major: k after k, the lines of
// the tile's rows, 32-byte segment s of a line (two of h, two of l) at s ^ (k & 3); a fragment is two transposing reads, and the four
// k a read touches lie in four different segments.
constexpr int HALF_ROWS = host::HALF_ROWS, HALF_THREADS = 256;
template <template <int> class EpiT, int KMAJ>
__global__ void __launch_bounds__(HALF_THREADS, 2) half_kernel(ContractArgs a, HalfArgs hs, typename EpiT<KS_NQT>::Args ea) {
  using Epi = EpiT<KS_NQT>;
  constexpr bool KE = (KMAJ & 1) != 0, KQ = (KMAJ & 2) != 0;
  constexpr int ROWS = HALF_ROWS, WAVES = HALF_THREADS / 64;
  constexpr int E_BYTES = ROWS * 128, Q_BYTES = KS_WG_QUERIES * 128, STAGE_BYTES = E_BYTES + Q_BYTES;
  constexpr int EL = E_BYTES / 1024 / WAVES, QL = Q_BYTES / 1024 / WAVES;  // loads of a wave per chunk, 1 KB each
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * STAGE_BYTES];

  int qg, k_range = 0, k_off = 0, k_end = a.d;  // this workgroup's columns of K
  int64_t chunk, wg_flat = blockIdx.x;
  constexpr bool STORE_T = std::is_same<Epi, StoreTEpi<KS_NQT>>::value;
  bool tail = false;
  if constexpr (STORE_T) tail = wg_flat >= hs.tail_first;
  if (tail) {
    const int64_t rest = wg_flat - hs.tail_first, tile = rest / hs.tail_splits;
    k_range = (int)(rest % hs.tail_splits);
    k_off = k_range * hs.tail_len;
    k_end = a.d - k_off > hs.tail_len ? k_off + hs.tail_len : a.d;
    qg = (int)(tile % a.n_qgroups);
    chunk = a.n_chunks + tile / a.n_qgroups;
  } else {
    if (hs.k_splits > 1) {
      k_range = (int)blockIdx.y;
      if (a.k_split_xcd) {  // flat grid: consecutive ids go round the XCDs, and an XCD keeps to its K ranges
        const int64_t per_range = a.n_chunks * a.n_qgroups, slot = wg_flat >> 3;
        k_range = (int)(wg_flat & 7) + 8 * (int)(slot / per_range);
        wg_flat = slot % per_range;
      }
      const int64_t chunks = a.d / KS_KC;  // whole chunks, as equal as they go
      k_off = (int)(chunks * k_range / hs.k_splits) * KS_KC;
      k_end = (int)(chunks * (k_range + 1) / hs.k_splits) * KS_KC;
    }
    if (!decompose_wg(a, qg, chunk, wg_flat)) return;
  }
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, hf = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int we = wave >> 1, wq = wave & 1;
  const int d = k_end - k_off;
  const int64_t q_base = (int64_t)qg * KS_WG_QUERIES;
  const int64_t r0 = a.e_begin + chunk * a.chunk_rows;
  const int64_t r1 = (r0 + a.chunk_rows < a.e_end) ? r0 + a.chunk_rows : a.e_end;
  const int nkc = d / KS_KC;
  const int n_et = (int)((r1 - r0 + ROWS - 1) / ROWS);
  const int n_it = n_et * nkc;
  const int64_t pitch_e = 4 * (int64_t)a.lde, pitch_q = 4 * (int64_t)a.ldq;  // bytes

  // This lane's share of a load of 1 KB.  Row-major: eight rows, lane / 8 and the piece that its LDS place holds.  K-major: a tile
  // row of R rows is R / 32 lines, R * 4 bytes of LDS.
  auto row_offset = [&](int64_t pitch) { return (uint32_t)((lane >> 3) * (int)pitch + (((lane & 7) ^ (lane >> 3)) << 4)); };
  auto kmaj_offset = [&](int R, int64_t pitch, int load) {  // load: its number in the tile
    const int byte = load * 1024 + lane * 16, k = byte / (R * 4), in = byte % (R * 4);
    const int k_in = k - load * 1024 / (R * 4);  // k rows behind the load's first
    return (uint32_t)(k_in * (int)pitch + (in & ~127) + (((((in >> 5) & 3) ^ (k & 3)) << 5) | (in & 31)));
  };
  uint32_t off_e[KE ? EL : 1], off_q[KQ ? QL : 1];
  if constexpr (KE) {
#pragma unroll
    for (int j = 0; j < EL; ++j) off_e[j] = kmaj_offset(ROWS, pitch_e, wave * EL + j);
  } else {
    off_e[0] = row_offset(pitch_e);
  }
  if constexpr (KQ) {
#pragma unroll
    for (int j = 0; j < QL; ++j) off_q[j] = kmaj_offset(KS_WG_QUERIES, pitch_q, wave * QL + j);
  } else {
    off_q[0] = row_offset(pitch_q);
  }
  // scalar bases of this wave's first load of a chunk, and how far the next loads and the next chunk lie from it
  const unsigned char* e_base0 = (const unsigned char*)a.E + (KE ? (int64_t)k_off * pitch_e : 4 * (int64_t)k_off);
  const unsigned char* q_base0 = (const unsigned char*)a.Q + (KQ ? (int64_t)k_off * pitch_q + 4 * q_base : 4 * (int64_t)k_off + q_base * pitch_q);
  constexpr int KE_PER = 1024 / (ROWS * 4), KQ_PER = 1024 / (KS_WG_QUERIES * 4);  // K-major: k rows of a load
  const int64_t e_step = KE ? KE_PER * pitch_e : 8 * pitch_e, q_step = KQ ? KQ_PER * pitch_q : 8 * pitch_q;
  const int64_t e_next = KE ? KS_KC * pitch_e : 128, q_next = KQ ? KS_KC * pitch_q : 128;
  e_base0 += wave * EL * e_step;
  q_base0 += wave * QL * q_step;
  int ld_kc = 0, ld_left = n_it;  // K chunk of the next loads, chunks not yet requested
  int64_t ld_row = r0;
  const unsigned char* e_at = e_base0 + (KE ? 4 * ld_row : ld_row * pitch_e);
  const unsigned char* q_at = q_base0;
  // (Written in assembly so that the compiler does not see LDS change behind the fragment reads, before which it would wait for
  // every load in flight; the waits are the ones at the loop's top.  Nothing is returned to a register, and nothing else here uses m0.)
  auto load_line = [&](uint32_t to, const unsigned char* base, uint32_t off) {
    asm volatile("s_mov_b32 m0, %0\ns_nop 0\nglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(off), "s"(base) : "memory");
  };
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
  auto issue = [&](int buffer) {  // (after the last chunk: that chunk again, which nobody reads)
    uint32_t dst = lds0 + buffer * STAGE_BYTES + wave * (EL * 1024);
#pragma unroll
    for (int j = 0; j < EL; ++j) load_line(dst + j * 1024, e_at + j * e_step, off_e[KE ? j : 0]);
    dst = lds0 + buffer * STAGE_BYTES + E_BYTES + wave * (QL * 1024);
#pragma unroll
    for (int j = 0; j < QL; ++j) load_line(dst + j * 1024, q_at + j * q_step, off_q[KQ ? j : 0]);
    if (--ld_left > 0) {
      if (++ld_kc == nkc) {
        ld_kc = 0;
        ld_row += ROWS;
        e_at = e_base0 + (KE ? 4 * ld_row : ld_row * pitch_e);
        q_at = q_base0;
      } else {
        e_at += e_next;
        q_at += q_next;
      }
    }
  };
  if (n_it > 0) issue(0);
  // (the first loads are under way)
  Epi epi;
  epi.init(ea, q_base + 64 * wq, c, hf, a.B);
  if constexpr (std::is_same<Epi, StoreEpi<KS_NQT>>::value) {
    if (a.k_split_xcd) epi.a.S += (int64_t)k_range * epi.a.split_stride;  // (blockIdx.y is 0 in a flat grid)
  }
  if constexpr (STORE_T) {
    if (tail) epi.a.S = hs.tail + (int64_t)k_range * hs.tail_stride;
  }
  __shared__ typename Epi::Shared epi_sh;
  epi.bind(&epi_sh);
  const int down = -((hs.exp_e ? *hs.exp_e : hs.fixed_e) + (hs.exp_q ? *hs.exp_q : hs.fixed_q));
  // The scores' factor, for the gradients: past the ends of fp32's range a score is the bias or saturates either way.
  constexpr bool GRAD = std::is_same<Epi, GradSplitEpi<KS_NQT>>::value || std::is_same<Epi, GradSplitBiasEpi<KS_NQT>>::value;
  const float up = pow2f(down < -126 ? -126 : down > 127 ? 127 : down), up_2k = up * (1.f / 2048.f);

  // fragments of this lane: row-major, row c of a tile of 32 rows, part and K step give the piece; K-major, its address for the
  // transposing reads (within 16 lanes: k (lane % 16) / 4, rows 4 (lane % 4) .. of a segment)
  const int tr_k = 8 * hf + ((lane & 15) >> 2), tr_half = (lane >> 4) & 1, tr_in = (lane & 3) << 3;
  auto fragment = [&](const unsigned char* from, bool kmaj, int R, int row0, int part, int ks) -> f16x8 {
    if (!kmaj) return *(const f16x8*)(from + (row0 + c) * 128 + (((4 * part + 2 * ks + hf) ^ (c & 7)) << 4));
    typedef __attribute__((ext_vector_type(4))) short s16x4;
    typedef __attribute__((ext_vector_type(8))) short s16x8;
    const unsigned char* p0 = from + (16 * ks + tr_k) * (R * 4) + row0 * 4 + (((2 * part + tr_half) ^ (tr_k & 3)) << 5) + tr_in;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p0));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p0 + 4 * (R * 4)));
    return __builtin_bit_cast(f16x8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  f32x16 acc[2][2], cross[2][2];
  auto clear = [&]() {
#pragma unroll
    for (int te = 0; te < 2; ++te)
#pragma unroll
      for (int tq = 0; tq < 2; ++tq)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[te][tq][i] = cross[te][tq][i] = 0.f;
  };
  clear();
  struct Step {  // the fragments of a K step of 16
    f16x8 e[2][2], q[2][2];
  };
  auto read_step = [&](const unsigned char* from, int ks, Step& f) {
#pragma unroll
    for (int part = 0; part < 2; ++part)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        f.e[part][t] = fragment(from, KE, ROWS, 64 * we + 32 * t, part, ks);
        f.q[part][t] = fragment(from + E_BYTES, KQ, KS_WG_QUERIES, 64 * wq + 32 * t, part, ks);
      }
  };
  auto mfma = [](f16x8 x, f16x8 y, f32x16 z) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(x, y, z, 0, 0, 0); };
  auto multiply = [&](const Step& f) {
#pragma unroll
    for (int m = 0; m < 12; ++m) {
      const int p = m / 4, te = (m >> 1) & 1, tq = m & 1;
      const f16x8 e = f.e[p == 2 ? 1 : 0][te], q = f.q[p == 1 ? 1 : 0][tq];
      f32x16& to = p == 0 ? acc[te][tq] : cross[te][tq];
      to = Epi::SWAP ? mfma(q, e, to) : mfma(e, q, to);
    }
  };

  int kc = 0;
  bool landed = false;  // the next chunk's lines have been waited for already
  int64_t et0 = r0;
  for (int it = 0; it < n_it; ++it) {
    // this chunk has landed for every wave, and everyone is done with the buffer that is filled next
    if (!landed) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    landed = false;
    asm volatile("s_waitcnt lgkmcnt(0)\ns_barrier" ::: "memory");
    const unsigned char* cur = lds + (it & 1) * STAGE_BYTES;
    issue((it & 1) ^ 1);
    Step f[2];
    read_step(cur, 0, f[0]);
    read_step(cur, 1, f[1]);
    multiply(f[0]);
    multiply(f[1]);
    // the first step's fragments, then the second's under its products
    constexpr int READS = 4 * (KE ? 2 : 1) + 4 * (KQ ? 2 : 1);
    __builtin_amdgcn_sched_group_barrier(0x100, READS, 0);
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, READS / 8, 0);
      if (READS % 8 && (m & 1)) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 16, 0);
    if (++kc == nkc) {  // this entity tile is complete
      // (waited for here, in front of the epilogue's stores, which the next wait would otherwise have to see finished)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      landed = true;
#pragma unroll
      for (int te = 0; te < 2; ++te) {
        const int64_t e_base = et0 + 64 * we + 32 * te;
        if (e_base < r1) {
#pragma unroll
          for (int tq = 0; tq < 2; ++tq) {
            if constexpr (GRAD) {
              epi.tile_split(tq, acc[te][tq], cross[te][tq], up, up_2k, e_base, r1);
            } else {
              float sc16[16];
#pragma unroll
              for (int i = 0; i < 16; ++i)
                acc[te][tq][i] = __builtin_amdgcn_ldexpf(__builtin_fmaf(cross[te][tq][i], 1.f / 2048.f, acc[te][tq][i]), down);
              epi.template tile<false>(tq, acc[te][tq], sc16, 1.f, e_base, r1);
            }
          }
        }
      }
      clear();
      kc = 0;
      et0 += ROWS;
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load may land in LDS after the workgroup has gone
  epi.finish();
}

}  // namespace kge
