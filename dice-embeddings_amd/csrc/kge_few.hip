// Few queries against the whole table (gfx950): the scan of kge_topk and the store of kge_scores for batches of at most
// 128 queries.
//
// The main loops of kge_contract.hip.h give every wave its own queries and every workgroup all of a chunk's rows: 512
// queries (256 / 128) per workgroup, so that a batch of 32 multiplies sixteen times the rows it needs, for padding
// queries, and runs at the matrix rate of the padding (bf16 d = 128, N = 2.5M, B = 32: 2.9 TB/s of table).  Here all waves
// hold the SAME queries, as MFMA fragments in LDS, and share out the entity rows, which go as whole lines through
// registers and a wave's own LDS into operands (few_scan_kernel): what bounds the scan is the table's bytes.
// Measured, whole calls: top-10 of 32 queries, bf16 d = 128, N = 2.5M 408 -> 180 us; top-10 of one question by name, fp32
// d = 256, N = 41k 284 -> 131 us (the rounds of the large-batch form were four to seven scans and selections, and a
// read-back).
//
// Scores are formed by the chain every kernel uses (K steps of 16 ascending; fp32 operands as three bf16 parts, six
// products in SPLIT order), so they carry the same bits.
#include "kge_contract.hip.h"

#include <algorithm>
#include <type_traits>

namespace kge {
namespace {

using host::FEW_LDS_KB;
using host::FEW_MAX_K;
using host::FEW_TILES_DIRECT;

struct FewArgs {
  const float* Q;
  const void* E;
  const float* scale;
  const float* bias;  // FEW_STORE only
  float* out;         // FEW_STORE: scores [B, ldo]; else the maximum over every 32-row tile [B, ldo]
  float* runs;        // FEW_MAX with tpw = 8: the maximum over every run of eight tiles [B, ldo / 8]
  float* raw;         // FEW_MAX_RAW: the scores themselves too, without a bias [B, ldr], whole tiles
  int64_t ldo, ldr, N, n_tiles;
  int B, d, nks;
  int tpw;   // consecutive tiles a wave takes at a time
  int n_qg;  // query groups: 32 * QT queries each, as many as LDS holds fragments of
  int n_wg;  // workgroups of a group, a multiple of 8
  GradArgs grad;  // FEW_GRAD only
};

// One wave at a time: chunks of a 32-row tile, 128 (bf16: 256) bytes of every row, loaded as whole lines into registers
// (eight or sixteen lanes per row), put into the wave's own LDS (16-byte piece p of row r at p ^ (r & 7 or 15)) and read back as MFMA
// operands; the next chunk's loads are in flight while a chunk is multiplied, across tiles, and no wave waits for another.
// (Operands loaded straight from memory, each lane its 16 or 32 bytes of a row: every request touches 32 lines, four
// requests share them, and a CU's waves push each other's lines out of the L1 in between: bf16 d = 128, N = 2.5M 152 us against 143, int8 N = 10M
// whole calls of 32 queries 507 against 382.)
constexpr int few_stage_bytes(int edt) { return edt == KGE_BF16 ? 8192 : 4096; }
// FEW_GRAD: GradEpi's gradients, loss sums and bias gradient in the place of the scores (fp32 tables)
enum FewMode { FEW_MAX, FEW_MAX_RAW, FEW_STORE, FEW_GRAD };
constexpr int FEW_RUN = 8;  // tiles of a run whose maxima go out together
template <int EDT, int QT, int MODE>
__global__ void __launch_bounds__(256, QT > 1 ? 2 : EDT == KGE_F32 ? 3 : 4) few_scan_kernel(FewArgs a) {
  constexpr int PARTS = EDT == KGE_F32 ? 3 : 1;
  constexpr int CH = EDT == KGE_F32 ? 2 : 8;            // K steps per chunk: a line of an fp32 or int8 row, two of a bf16 row
  constexpr int PIECES = EDT == KGE_BF16 ? 16 : 8;       // 16-byte pieces of a row's chunk
  constexpr int RPL = 64 / PIECES, NLD = 32 / RPL;       // rows per wave-wide load, loads per chunk
  constexpr int PER_PIECE = EDT == KGE_F32 ? 4 : EDT == KGE_BF16 ? 8 : 16;  // elements
  constexpr bool GRAD = MODE == FEW_GRAD;
  constexpr bool STORE = MODE == FEW_STORE || GRAD;  // accumulator columns are entities
  extern __shared__ __attribute__((aligned(16))) unsigned char fq_lds[];
  __shared__ __attribute__((aligned(16))) float s_bias[STORE ? 32 * QT : 1];
  __shared__ __attribute__((aligned(16))) float s_max[MODE == FEW_MAX ? 4 * 32 * QT * FEW_RUN : 4];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, hf = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // The query groups of a batch walk the table side by side, a row's groups on one XCD (ids go round the eight of them): the
  // first to come loads it, the others find it in that L2.  (One group after the other, each reads the whole table: fp32
  // d = 256, N = 2M, 128 queries 1565 us; side by side 1196.)
  const int slot = (int)blockIdx.x >> 3, qg = slot % a.n_qg, wg = slot / a.n_qg * 8 + ((int)blockIdx.x & 7);
  const int q0 = qg * (32 * QT);
  const int nks = a.nks, d = a.d;
  for (int i = tid; i < QT * nks * 64; i += 256) {
    const int l = i & 63, s = (i >> 6) % nks, t = (i >> 6) / nks;
    const int q = q0 + 32 * t + (l & 31), k = 16 * s + 8 * (l >> 5);
    f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = {0.f, 0.f, 0.f, 0.f};
    if (q < a.B) {
      const float* src = a.Q + (int64_t)q * d + k;
      if (k + 4 <= d) lo = *(const f32x4*)src;  // (d is a multiple of 4)
      if (k + 8 <= d) hi = *(const f32x4*)(src + 4);
    }
    unsigned char* dst = fq_lds + (size_t)(t * nks + s) * PARTS * 1024 + l * 16;
    if constexpr (EDT == KGE_F32) {
      bf16x8 p[3];
      split3_bf16x8(lo, hi, p);
#pragma unroll
      for (int part = 0; part < 3; ++part) *(bf16x8*)(dst + part * 1024) = p[part];
    } else {
      *(bf16x8*)dst = cvt_bf16x8(lo, hi);
    }
  }
  if (STORE) {
    for (int i = tid; i < 32 * QT; i += 256) s_bias[i] = (a.bias && q0 + i < a.B) ? a.bias[q0 + i] : 0.f;
  }
  __syncthreads();

  unsigned char* stage = fq_lds + (size_t)QT * nks * PARTS * 1024 + wave * few_stage_bytes(EDT);
  u32x4 staged[NLD];
  f32x4 next_sc[EDT == KGE_I8 ? 4 : 1], sc[EDT == KGE_I8 ? 4 : 1];  // int8: row scales of the chunk loaded, multiplied
  const int l_row = lane / PIECES, l_piece = lane % PIECES;
  const int nch = (nks + CH - 1) / CH;
  int64_t unit = wg, tile = (unit * 4 + wave) * a.tpw;
  int ch = 0, in_unit = 0;
  // the position after (tile, ch); past the end: tile >= n_tiles
  auto advance = [&]() {
    if (++ch < nch) return;
    ch = 0;
    ++tile;
    if (++in_unit == a.tpw) {
      in_unit = 0;
      unit += a.n_wg;
      tile = (unit * 4 + wave) * a.tpw;
    }
  };
  constexpr int64_t ELEM = EDT == KGE_F32 ? 4 : EDT == KGE_BF16 ? 2 : 1;
  auto load = [&]() {
    int k = ch * CH * 16 + l_piece * PER_PIECE;
    k = k < d ? k : 0;  // (pieces past the row's end: any valid address, their columns are zeroed below)
    const unsigned char* base = (const unsigned char*)a.E + k * ELEM;
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      int64_t row = tile * 32 + i * RPL + l_row;
      row = row < a.N ? row : a.N - 1;  // rows past the end repeat the last one; the epilogues ignore them
      staged[i] = *(const u32x4*)(base + row * d * ELEM);
    }
    if constexpr (EDT == KGE_I8) {
      if (ch == nch - 1) {
        if (STORE) {
          next_sc[0][0] = a.scale[tile * 32 + c < a.N ? tile * 32 + c : a.N - 1];
        } else {
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const int64_t e = tile * 32 + 8 * g + 4 * hf;
#pragma unroll
            for (int j = 0; j < 4; ++j) next_sc[g][j] = a.scale[e + j < a.N ? e + j : a.N - 1];
          }
        }
      }
    }
  };
  auto store = [&]() {
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const int row = i * RPL + l_row;
      *(u32x4*)(stage + (row * PIECES + (l_piece ^ (row & (PIECES - 1)))) * 16) = staged[i];
    }
    if constexpr (EDT == KGE_I8) {
#pragma unroll
      for (int g = 0; g < 4; ++g) sc[g] = next_sc[g];
    }
  };
  auto piece = [&](int p) -> const unsigned char* { return stage + (c * PIECES + (p ^ (c & (PIECES - 1)))) * 16; };
  f32x16 acc[QT];
  float run_max[QT];  // FEW_MAX with tpw = FEW_RUN
  std::conditional_t<GRAD, GradEpi<QT>, int> epi;
  if constexpr (GRAD) {
    epi.init(a.grad, q0, c, hf, a.B);
    epi.lb = s_bias;
  }
  auto multiply = [&](int64_t t_tile, int t_ch) {
    if (t_ch == 0) {
#pragma unroll
      for (int t = 0; t < QT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int s = t_ch * CH + u;
      if (s < nks) {  // uniform
        const int k = 16 * s + 8 * hf;
        bf16x8 fe[PARTS];
        if constexpr (EDT == KGE_F32) {
          f32x4 lo = *(const f32x4*)piece(4 * u + 2 * hf), hi = *(const f32x4*)piece(4 * u + 2 * hf + 1);
          if (16 * s + 16 > d) {  // the row's last, partial step: its columns past d are zeros, whatever was read
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              lo[j] = k + j < d ? lo[j] : 0.f;
              hi[j] = k + 4 + j < d ? hi[j] : 0.f;
            }
          }
          bf16x8 p[3];
          split3_bf16x8(lo, hi, p);
#pragma unroll
          for (int part = 0; part < 3; ++part) fe[part] = p[part];
        } else {
          u32x4 w;
          if constexpr (EDT == KGE_I8) {
            const u32x2 b = *(const u32x2*)(piece(u) + 8 * hf);
            w = i8x8_to_bf16x8(b[0], b[1]);
          } else {
            w = *(const u32x4*)piece(2 * u + hf);
          }
          if (16 * s + 16 > d && k >= d) w = u32x4{0u, 0u, 0u, 0u};
          fe[0] = __builtin_bit_cast(bf16x8, w);
        }
#pragma unroll
        for (int t = 0; t < QT; ++t) {
          const unsigned char* src = fq_lds + (size_t)(t * nks + s) * PARTS * 1024 + lane * 16;
          bf16x8 fq[PARTS];
#pragma unroll
          for (int part = 0; part < PARTS; ++part) fq[part] = *(const bf16x8*)(src + part * 1024);
          if constexpr (EDT == KGE_F32) {
#pragma unroll
            for (int p = 0; p < SPLIT_PRODUCTS; ++p)
              acc[t] = STORE ? mfma_bf16(fq[SPLIT_B[p]], fe[SPLIT_A[p]], acc[t])
                             : mfma_bf16(fe[SPLIT_A[p]], fq[SPLIT_B[p]], acc[t]);
          } else {
            acc[t] = STORE ? mfma_bf16(fq[0], fe[0], acc[t]) : mfma_bf16(fe[0], fq[0], acc[t]);
          }
        }
      }
    }
    if (t_ch != nch - 1) return;
    if constexpr (GRAD) {
#pragma unroll
      for (int t = 0; t < QT; ++t) epi.template tile<false>(t, acc[t], nullptr, 1.f, t_tile * 32, a.N);
    } else if constexpr (STORE) {
      const int64_t e = t_tile * 32 + c;
      if (e < a.N) {
#pragma unroll
        for (int t = 0; t < QT; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int r = 32 * t + row_of(i, hf);
            if (q0 + r < a.B) {
              const float v = EDT == KGE_I8 ? acc[t][i] * sc[0][0] : acc[t][i];
              a.out[(int64_t)(q0 + r) * a.ldo + e] = v + s_bias[r];
            }
          }
      }
    } else {
      const bool whole = t_tile * 32 + 32 <= a.N;
      const bool in_runs = MODE == FEW_MAX && a.tpw == FEW_RUN;
      const int at = (int)(t_tile & (FEW_RUN - 1));
#pragma unroll
      for (int t = 0; t < QT; ++t) {
        float m = __uint_as_float(0xff800000u);  // (a NaN score never becomes the maximum)
        const int q = q0 + 32 * t + c;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          f32x4 v;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            v[r] = acc[t][4 * g + r];
            if constexpr (EDT == KGE_I8) v[r] *= sc[g][r];
            if (!whole && t_tile * 32 + 8 * g + 4 * hf + r >= a.N) v[r] = __uint_as_float(0xff800000u);
            m = __builtin_fmaxf(m, v[r]);
          }
          if constexpr (MODE == FEW_MAX_RAW) {
            if (q < a.B) *(f32x4*)(a.raw + (int64_t)q * a.ldr + t_tile * 32 + 8 * g + 4 * hf) = v;
          }
        }
        m = __builtin_fmaxf(m, __shfl_xor(m, 32, 64));
        if (in_runs) {
          if (hf == 0) s_max[(wave * 32 * QT + 32 * t + c) * FEW_RUN + at] = m;
          run_max[t] = at == 0 ? m : __builtin_fmaxf(run_max[t], m);
        } else if (hf == 0 && q < a.B) {
          a.out[(int64_t)q * a.ldo + t_tile] = m;
        }
      }
      if constexpr (MODE == FEW_MAX) {
        // a run's maxima together, 32 bytes per query (one by one, 4 bytes to each of 32 rows, they cost a sixth of the
        // scan); what lies past the last tile is never read
        if (in_runs && (at == FEW_RUN - 1 || t_tile == a.n_tiles - 1)) {
          wave_sync();
          const int64_t run = t_tile / FEW_RUN;
          for (int i = lane; i < 32 * QT * 2; i += 64) {
            const int q = q0 + (i >> 1);
            const f32x4 v = *(const f32x4*)(s_max + (wave * 32 * QT + (i >> 1)) * FEW_RUN + 4 * (i & 1));
            if (q < a.B) *(f32x4*)(a.out + (int64_t)q * a.ldo + run * FEW_RUN + 4 * (i & 1)) = v;
          }
#pragma unroll
          for (int t = 0; t < QT; ++t)
            if (hf == 0 && q0 + 32 * t + c < a.B) a.runs[(int64_t)(q0 + 32 * t + c) * (a.ldo / FEW_RUN) + run] = run_max[t];
          wave_sync();
        }
      }
    }
  };
  if (tile >= a.n_tiles) return;
  load();
  for (;;) {
    store();
    wave_sync();
    const int64_t t_tile = tile;
    const int t_ch = ch;
    advance();
    const bool more = tile < a.n_tiles;
    if (more) load();
    multiply(t_tile, t_ch);
    wave_sync();
    if (!more) break;
  }
  if constexpr (GRAD) epi.finish();
}

// ---- the best k from the tile maxima ----------------------------------------------------------------------
// The best k entities (score descending, id ascending) lie in the best k tiles (maximum descending, tile ascending): if a
// tile is not among them, k tiles hold an entity each that ranks above everything in it (a higher score, or the same
// score at a lower id).  So one workgroup per query picks the k best tiles, forms their 32 k scores again and picks the
// k best of those: no thresholds, no candidate buffers that could overflow, nothing read back.  Tables of more than
// FEW_TILES_DIRECT tiles go through the maxima of 32 tiles first, by the same argument.
constexpr int FEW_THREADS = 1024;
constexpr int SELECT_GROUPS = FEW_THREADS / 4, SELECT_CAP = 512;
// This many entities are ranked without being picked first (each against all: 320 of them cost 7 us more than their selection)
constexpr int FEW_DIRECT = 160;
struct SelectShared {
  unsigned long long cnt[16];
  union {
    uint32_t scan[256];           // block_select_bits
    __attribute__((aligned(16))) uint32_t top[SELECT_GROUPS];  // the largest value of every four threads (t, t + 256, ..)
  };
  int rank[SELECT_GROUPS];
  __attribute__((aligned(16))) unsigned long long cand[SELECT_CAP];  // (value, then the lower position) as one key, zeros behind them
  int picked[FEW_MAX_K];
  int n_cand, n_above;
  uint32_t bound, least;
};

__device__ __forceinline__ uint32_t score_key(float v) {
  return v > __uint_as_float(0xff800000u) ? f32_to_ordered(v) : 0u;  // NaN and -inf are never ranked
}

// The positions of the k largest of vals[0 .. M) (ties: the lower positions; zeros never), ascending, into pos; returns
// how many.  M <= 16 * FEW_THREADS.  (Loops that are not unrolled: a launch is one pass of a few workgroups through the code, and
// what the code's length costs in fetches is more than what its loops cost; selections of two, four and sixteen values per
// thread in registers, the steps below otherwise alike, made the kernel 27.7 us where the bits alone took 24.8.)
//
// block_select_bits: the k-th largest value is found two bits at a time, three counts per step, by the whole workgroup; a step
// that splits off exactly k ends the search.  known: it is that value, no search.
__device__ __forceinline__ int block_select_bits(const uint32_t* vals, int M, int k, int* pos, SelectShared& sh, uint32_t known) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int V = (M + FEW_THREADS - 1) / FEW_THREADS;
  auto value = [&](int j) { return j * FEW_THREADS + tid < M ? vals[j * FEW_THREADS + tid] : 0u; };
  __syncthreads();
  if (tid < 16) sh.cnt[tid] = 0;
  __syncthreads();
  uint32_t th = known;
  bool exact = false;  // exactly k values are >= th
#pragma unroll 1
  for (int b = 30; b >= 0 && !exact && !known; b -= 2) {
    const uint32_t t1 = th | (1u << b), t2 = th | (2u << b), t3 = th | (3u << b);
    int c1 = 0, c2 = 0, c3 = 0;
#pragma unroll 1
    for (int j = 0; j < V; ++j) {
      const uint32_t v = value(j);
      c1 += __builtin_popcountll(__builtin_amdgcn_ballot_w64(v >= t1));
      c2 += __builtin_popcountll(__builtin_amdgcn_ballot_w64(v >= t2));
      c3 += __builtin_popcountll(__builtin_amdgcn_ballot_w64(v >= t3));
    }
    if (lane == 0)
      atomicAdd(&sh.cnt[b >> 1], (unsigned long long)c1 | ((unsigned long long)c2 << 20) | ((unsigned long long)c3 << 40));
    __syncthreads();
    const unsigned long long n = sh.cnt[b >> 1];
    const int n1 = (int)(n & 0xfffff), n2 = (int)((n >> 20) & 0xfffff), n3 = (int)(n >> 40);
    if (n3 >= k) {
      th = t3;
      exact = n3 == k;
    } else if (n2 >= k) {
      th = t2;
      exact = n2 == k;
    } else if (n1 >= k) {
      th = t1;
      exact = n1 == k;
    }
  }
  // above: selected whatever the ties do; at: values equal to the k-th largest, taken in order until there are k
  const uint32_t above = exact ? th - 1 : th;  // (exact only with th > 0)
  const uint32_t at = exact ? 0u : th;         // 0: none
#pragma unroll 1
  for (int j = 0; j < V; ++j) {
    const uint32_t v = value(j);
    const int ng = __builtin_popcountll(__builtin_amdgcn_ballot_w64(v > above));
    const int ne = __builtin_popcountll(__builtin_amdgcn_ballot_w64(at != 0 && v == at));
    if (lane == 0) sh.scan[j * 16 + wave] = (uint32_t)ng | ((uint32_t)ne << 16);
  }
  __syncthreads();
  uint32_t total = 0;
  if (wave == 0) {
    uint32_t x[4], sum = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[i] = (4 * lane + i < 16 * V) ? sh.scan[4 * lane + i] : 0u;
      sum += x[i];
    }
    uint32_t run = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(run, o, 64);
      if (lane >= o) run += y;
    }
    total = __shfl(run, 63, 64);
    run -= sum;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (4 * lane + i < 16 * V) sh.scan[4 * lane + i] = run;
      run += x[i];
    }
    if (lane == 0) sh.cnt[0] = total;
  }
  __syncthreads();
  total = (uint32_t)sh.cnt[0];
  const int n_gt = (int)(total & 0xffff), n_eq = (int)(total >> 16);
  const int need = n_eq < k - n_gt ? n_eq : k - n_gt;
  const unsigned long long below_lane = (1ull << lane) - 1;
#pragma unroll 1
  for (int j = 0; j < V; ++j) {
    const uint32_t v = value(j);
    const unsigned long long bg = __builtin_amdgcn_ballot_w64(v > above);
    const unsigned long long be = __builtin_amdgcn_ballot_w64(at != 0 && v == at);
    const uint32_t base = sh.scan[j * 16 + wave];
    const int g = (int)(base & 0xffff) + __builtin_popcountll(bg & below_lane);
    const int e = (int)(base >> 16) + __builtin_popcountll(be & below_lane);
    if (v > above || (at != 0 && v == at && e < need)) pos[g + (e < need ? e : need)] = j * FEW_THREADS + tid;
  }
  __syncthreads();
  return n_gt + need;
}
// block_select: what bounds it is its chain of steps, so it has few, and none waits for one LDS read at a time.  The k-th
// largest of 256 maxima, of the values at every 256th position each, is a lower bound of the k-th largest value, and hardly more
// than k values reach it; those are gathered and ranked by counting.  Where more than SELECT_CAP reach it, either one
// value repeated is the k-th largest, or the bits decide.  Best 10 of 1280 and then of 320, with the loads: 24.9 -> 8.5 us; of 2442,
// 320 and 320, with the scores formed again: 36.5 -> 19.6; of 14,541 values: 23.5 -> 8.2.
__device__ __forceinline__ int block_select(const uint32_t* vals, int M, int k, int* pos, SelectShared& sh) {
  const int tid = threadIdx.x, lane = tid & 63;
  __syncthreads();  // sh and pos are free
  if (tid < SELECT_CAP) sh.cand[tid] = 0;
  if (tid < SELECT_GROUPS) {
    sh.rank[tid] = 0;
    sh.top[tid] = 0;
  }
  static_assert(SELECT_GROUPS == 256, "a group's number is a byte");
  if (tid == 0) {
    sh.n_cand = sh.n_above = 0;
    sh.least = 0xffffffffu;
    sh.bound = 1;  // (where fewer than k groups have a value: every value)
  }
  __syncthreads();  // vals is complete
  uint32_t top = 0;
#pragma unroll 2
  for (int p = tid; p < M; p += FEW_THREADS) top = vals[p] > top ? vals[p] : top;
  if (top) atomicMax(&sh.top[tid & (SELECT_GROUPS - 1)], (top & ~0xffu) | (uint32_t)(tid & (SELECT_GROUPS - 1)));
  __syncthreads();
  const int g = tid & (SELECT_GROUPS - 1), seg = tid / SELECT_GROUPS * 64;  // a quarter of the maxima against maximum g
  // (the last byte gives way to the group's number: no two are equal, and one comparison orders them)
  const uint32_t mine = sh.top[g];
  int above = 0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    u32x4 x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = *(const u32x4*)(sh.top + seg + 32 * h + 4 * i);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) above += x[i][j] > mine ? 1 : 0;
  }
  if (above) atomicAdd(&sh.rank[g], above);
  __syncthreads();
  if (tid < SELECT_GROUPS && sh.rank[tid] == k - 1 && mine > 0xff) sh.bound = mine & ~0xffu;
  __syncthreads();
  const uint32_t bound = sh.bound;
#pragma unroll 2
  for (int p = tid; p < M; p += FEW_THREADS) {  // (lanes past the end sit out: a ballot counts the others)
    const uint32_t v = vals[p];
    const unsigned long long b = __builtin_amdgcn_ballot_w64(v >= bound);
    if (v >= bound) {
      int at = 0;
      if (lane == __builtin_ctzll(b)) at = atomicAdd(&sh.n_cand, (int)__builtin_popcountll(b));
      at = __builtin_amdgcn_readfirstlane(at) + __builtin_popcountll(b & ((1ull << lane) - 1));
      if (at < SELECT_CAP) sh.cand[at] = ((unsigned long long)v << 32) | (0xffffffffu - (uint32_t)p);
    }
  }
  __syncthreads();
  const int C = sh.n_cand;
  if (C > SELECT_CAP) {
    // one value repeated?  The least of those that reach the bound, if fewer than k lie above it
    uint32_t least = 0xffffffffu;
#pragma unroll 2
    for (int p = tid; p < M; p += FEW_THREADS) least = vals[p] >= bound && vals[p] < least ? vals[p] : least;
    atomicMin(&sh.least, least);
    __syncthreads();
    least = sh.least;
    int n_above = 0;
#pragma unroll 2
    for (int p = tid; p < M; p += FEW_THREADS) n_above += vals[p] > least ? 1 : 0;
    if (n_above) atomicAdd(&sh.n_above, n_above);
    __syncthreads();
    return block_select_bits(vals, M, k, pos, sh, sh.n_above < k ? least : 0u);
  }
  const int n = C < k ? C : k;
  if (tid < C) {
    typedef __attribute__((ext_vector_type(2))) unsigned long long u64x2;
    const unsigned long long key = sh.cand[tid];
    int rank = 0;
    for (int i = 0; i < C; i += 16) {
      u64x2 x[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = *(const u64x2*)(sh.cand + i + 2 * j);
#pragma unroll
      for (int j = 0; j < 8; ++j) rank += (x[j][0] > key ? 1 : 0) + (x[j][1] > key ? 1 : 0);
    }
    if (rank < k) sh.picked[rank] = (int)(0xffffffffu - (uint32_t)key);
  }
  __syncthreads();
  if (tid < n) {
    const int p = sh.picked[tid];
    int below = 0;
#pragma unroll 8
    for (int i = 0; i < n; ++i) below += sh.picked[i] < p ? 1 : 0;
    pos[below] = p;
  }
  __syncthreads();
  return n;
}

struct FewFinishArgs {
  const float* Q;
  const void* E;
  const float* scale;
  const float* bias;
  const float* maxima;  // [B, ldm]
  const float* runs;    // [B, ldm / FEW_RUN], where there are more tiles than one workgroup selects from
  const float* raw;     // [B, ldr] the scores, or null: formed again
  int64_t ldm, ldr, N, n_tiles;
  int d, k, sigmoid;
  float* out_scores;
  int64_t* out_idx;
};

// RAW: the scores are at hand (a form of its own: the code that forms scores again is not in a launch's way then)
template <int EDT, bool RAW>
__global__ void __launch_bounds__(FEW_THREADS) few_finish_kernel(FewFinishArgs a) {
  __shared__ __attribute__((aligned(16))) uint32_t vals[16 * FEW_THREADS];
  __shared__ int pos[FEW_MAX_K], groups[FEW_MAX_K];
  __shared__ int64_t tiles[FEW_MAX_K];
  __shared__ unsigned long long keys[FEW_MAX_K];
  __shared__ SelectShared sh;
  __shared__ __attribute__((aligned(16))) unsigned char s_query[RAW ? 16 : query_lds_bytes(EDT, QUERY_LDS_MAX_D)];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, hf = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t q = blockIdx.x;
  const float* mx = a.maxima + q * a.ldm;
  const int T = (int)a.n_tiles, k = a.k;
  const float bias = a.bias ? a.bias[q] : 0.f;  // (asked for long before it is needed)
  // fill vals[0 .. M) from memory, four loads of a thread in flight
  auto fill = [&](int M, auto load, auto key) {
    for (int i0 = tid; i0 < M; i0 += 4 * FEW_THREADS) {
      float x[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) x[u] = i0 + u * FEW_THREADS < M ? load(i0 + u * FEW_THREADS) : 0.f;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (i0 + u * FEW_THREADS < M) vals[i0 + u * FEW_THREADS] = key(i0 + u * FEW_THREADS, x[u]);
    }
  };
  // Three levels, groups of 32 tiles (where there are too many tiles), tiles, entities: the candidates' keys into vals, the
  // best k of them picked.  (One loop, so that the selection is in the code once: the kernel runs a few microseconds, and
  // every copy of it would be fetched cold.)
  const bool grouped = T > FEW_TILES_DIRECT;
  int n = 0;
  bool picked = false;  // the entities: else they are few enough to be ranked all
  // Every tile is among the best k: nothing to pick (k = 100, N = 1000, d = 32, 64 queries: 10 us of the call).
  const bool all = T <= k;
  if (all) {
    n = T;
    if (tid < n) tiles[tid] = tid;
    __syncthreads();
  }
  for (int level = grouped ? 0 : all ? 2 : 1; level < 3; ++level) {
    int M;
    if (level == 0) {
      M = (T + 31) / 32;
      fill(M, [&](int g) {
        const f32x4 x = *(const f32x4*)(a.runs + q * (a.ldm / FEW_RUN) + 4 * (int64_t)g);  // 4 runs: 32 tiles
        float m = x[0];
#pragma unroll
        for (int i = 1; i < 4; ++i)
          if (FEW_RUN * (4 * g + i) < T) m = __builtin_fmaxf(m, x[i]);
        return m;
      }, [&](int, float m) { return score_key(m); });
    } else if (level == 1) {
      M = grouped ? 32 * n : T;
      auto tile_at = [&](int i) { return grouped ? 32 * groups[i >> 5] + (i & 31) : i; };
      fill(M, [&](int i) { return mx[tile_at(i) < T ? tile_at(i) : 0]; },
           [&](int i, float m) { return tile_at(i) < T ? score_key(m) : 0u; });
    } else {
      // the tiles' scores: kept by the scan, or formed again (every column of the result tile holds this query, lane
      // c < 16 keeps accumulator c)
      M = 32 * n;
      if constexpr (RAW) {
        fill(M, [&](int i) { return a.raw[q * a.ldr + tiles[i >> 5] * 32 + (i & 31)]; },  // (rows past the end: -inf)
             [&](int, float x) { return score_key(x); });
      } else {
        query_to_lds<EDT>(a.Q + q * a.d, a.d, s_query, tid, FEW_THREADS);
        __syncthreads();
        for (int j = wave; j < n; j += FEW_THREADS / 64) {
          const int64_t row = tiles[j] * 32 + c;
          const f32x16 acc = chain_one_query<EDT>(a.E, a.d, row < a.N ? row : -1, s_query, hf);
          float v = 0.f;
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (i == c) v = acc[i];
          if (c < 16) {
            const int r = row_of(c, hf);
            const int64_t e = tiles[j] * 32 + r;
            if constexpr (EDT == KGE_I8) v *= a.scale[e < a.N ? e : a.N - 1];
            vals[32 * j + r] = e < a.N ? score_key(v) : 0u;
          }
        }
      }
    }
    if (level == 2 && M <= FEW_DIRECT) break;
    n = block_select(vals, M, k, pos, sh);
    picked = level == 2;
    if (level == 0) {
      for (int j = tid; j < n; j += FEW_THREADS) groups[j] = pos[j];
    } else if (level == 1) {
      for (int j = tid; j < n; j += FEW_THREADS)
        tiles[j] = grouped ? 32 * (int64_t)groups[pos[j] >> 5] + (pos[j] & 31) : (int64_t)pos[j];
    } else {
      break;
    }
    __syncthreads();
  }
  auto put = [&](int at, uint32_t key, int64_t e) {  // key 0: fewer than k could be ranked
    float s = __uint_as_float(0x7fc00000u);
    if (key) {
      s = ordered_to_f32(key);
      if (a.bias) s += bias;
      if (a.sigmoid) s = 1.0f / (1.0f + expf(-s));
    }
    a.out_scores[q * k + at] = s;
    a.out_idx[q * k + at] = key ? e : -1;
  };
  if (32 * n <= FEW_DIRECT && !picked) {
    // few enough: one value per thread, whose rank is the number of values above it (equal ones at lower positions count as above)
    const int M = 32 * n;
    __syncthreads();
    const uint32_t mine = tid < M ? vals[tid] : 0u;
    int at = 0;
    if (wave * 64 < M) {
      for (int j = 0; j < M; j += 32) {
        u32x4 v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = *(const u32x4*)(vals + j + 4 * u);
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) at += (v[u][i] > mine || (v[u][i] == mine && j + 4 * u + i < tid)) ? 1 : 0;
      }
    }
    const int ranked = __syncthreads_count(mine != 0);
    if (mine != 0 && at < k) put(at, mine, tiles[tid >> 5] * 32 + (tid & 31));
    for (int j = ranked + tid; j < k; j += FEW_THREADS) put(j, 0u, 0);
    return;
  }
  for (int j = tid; j < n; j += FEW_THREADS)
    keys[j] = ((unsigned long long)vals[pos[j]] << 32) | (0xffffffffull - (unsigned long long)(tiles[pos[j] >> 5] * 32 + (pos[j] & 31)));
  __syncthreads();
  for (int j = tid; j < k; j += FEW_THREADS) {
    if (j >= n) {
      put(j, 0u, 0);
      continue;
    }
    const unsigned long long key = keys[j];
    int at = 0;
#pragma unroll 8
    for (int i = 0; i < n; ++i) at += keys[i] > key ? 1 : 0;
    put(at, (uint32_t)(key >> 32), (int64_t)(0xffffffffu - (uint32_t)(key & 0xffffffffull)));
  }
}

// ---- the best k of a vector of values (descending, equal values by position, NaN first: a stable descending sort cut at k) --
__device__ __forceinline__ uint32_t value_key(float v) {
  return v != v ? 0xffffffffu : f32_to_ordered(v + 0.f);  // (-0 and 0 are equal); never 0
}
// the largest key of every 32 values
__global__ void __launch_bounds__(256) value_tiles_kernel(const float* values, int N, uint32_t* tiles, int n_tiles) {
  const int t = blockIdx.x * 8 + (threadIdx.x >> 5), i = 32 * t + (threadIdx.x & 31);
  uint32_t k = i < N ? value_key(values[i]) : 0u;
#pragma unroll
  for (int o = 16; o >= 1; o >>= 1) {
    const uint32_t y = __shfl_xor(k, o, 64);
    k = y > k ? y : k;
  }
  if ((threadIdx.x & 31) == 0 && t < n_tiles) tiles[t] = k;
}
// One workgroup: latency, not work, is what this costs.  tiles: null where the workgroup selects from the values
// themselves.  (The hop of a query answered by the library's device sort was seven launches for ten values.)
__global__ void __launch_bounds__(FEW_THREADS) topk_values_kernel(const float* values, int N, const uint32_t* tiles,
                                                                  int n_tiles, int k, float* out_values, int64_t* out_idx,
                                                                  int64_t idx_stride, int64_t relation) {
  __shared__ __attribute__((aligned(16))) uint32_t vals[16 * FEW_THREADS];
  __shared__ int pos[FEW_MAX_K], best[FEW_MAX_K];
  __shared__ unsigned long long keys[FEW_MAX_K];
  __shared__ SelectShared sh;
  const int tid = threadIdx.x;
  int M = N, n = 0;
  if (tiles) {
#pragma unroll 4
    for (int t = tid; t < n_tiles; t += FEW_THREADS) vals[t] = tiles[t];
    n = block_select(vals, n_tiles, k, best, sh);
    M = 32 * n;
  }
  for (int i0 = tid; i0 < M; i0 += 8 * FEW_THREADS) {  // (eight loads of a thread in flight)
    float x[8];
    int at[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = i0 + u * FEW_THREADS;
      at[u] = i >= M ? N : tiles ? 32 * best[i >> 5] + (i & 31) : i;
      x[u] = values[at[u] < N ? at[u] : 0];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (i0 + u * FEW_THREADS < M) vals[i0 + u * FEW_THREADS] = at[u] < N ? value_key(x[u]) : 0u;
  }
  const bool all = M <= FEW_MAX_K;  // few enough to be ranked without being picked first
  if (all) {
    __syncthreads();
    n = M;
  } else {
    n = block_select(vals, M, k, pos, sh);  // k <= N: there are k
  }
  for (int j = tid; j < n; j += FEW_THREADS) {
    const int p = all ? j : pos[j], at = tiles ? 32 * best[p >> 5] + (p & 31) : p;
    keys[j] = ((unsigned long long)vals[p] << 32) | (0xffffffffu - (uint32_t)at);
  }
  __syncthreads();
  for (int j = tid; j < n; j += FEW_THREADS) {
    const unsigned long long key = keys[j];
    int rank = 0;
#pragma unroll 8
    for (int i = 0; i < n; ++i) rank += keys[i] > key ? 1 : 0;
    if (rank >= k) continue;
    const uint32_t at = 0xffffffffu - (uint32_t)(key & 0xffffffffull);
    out_values[rank] = values[at];
    out_idx[rank * idx_stride] = (int64_t)at;
    if (idx_stride == 2) out_idx[rank * 2 + 1] = relation;  // (the pairs of the next hop's queries)
  }
}

template <int MODE>
int launch_few_scan(int dtype, FewArgs a, hipStream_t st) {
  const int parts = dtype == KGE_F32 ? 3 : 1;
  a.nks = (a.d + 15) / 16;
  a.n_tiles = (a.N + 31) / 32;
  const int qt = host::few_query_tiles(dtype, a.B, a.d, MODE >= FEW_STORE ? 2 : 4);
  a.n_qg = (a.B + 32 * qt - 1) / (32 * qt);
  // workgroups, as many per CU as registers and LDS allow, walk units of 4 * tpw tiles, each about the same number of them; runs of
  // eight tiles where there are more tiles than the selection reads one by one
  a.tpw = a.n_tiles > FEW_TILES_DIRECT ? FEW_RUN : 1;
  const size_t lds = (size_t)qt * a.nks * parts * 1024 + 4 * few_stage_bytes(dtype);
  const size_t own = (lds + (MODE == FEW_MAX ? 4096 * qt : MODE >= FEW_STORE ? 128 * qt : 0) + 1279) / 1280 * 1280;  // (granules of 1280)
  const size_t room = 163840 / own;
  const int64_t slots = 256 * std::max<int64_t>(1, std::min<int64_t>(room, qt > 1 ? 2 : dtype == KGE_F32 ? 3 : 4));
  const int64_t units = (a.n_tiles + 4 * a.tpw - 1) / (4 * a.tpw);
  // In a long scan every slot has a workgroup, also where fewer would take as many units each: CUs that hold three beside others
  // with two end last (32 queries, k = 10, N = 2.5M, the call: bf16 d = 128 616 workgroups 160 us, 768 150; int8 d = 128 816
  // workgroups 116, 1024 98).  In a short one the start of the others costs more (fp32 d = 256, N = 200k: 392 workgroups
  // 53.5 us, 512 55.3).
  const bool fill = MODE == FEW_MAX && a.tpw > 1;
  // one to four rounds of them: the fewest units in turn on a slot, a workgroup's start counted as one (several query groups
  // rarely divide one round: int8 d = 1024, N = 41k, 96 queries, one round 89 us, the best of four 65)
  int64_t best = -1;
  for (int64_t r = 1; r <= (a.n_qg > 1 ? 4 : 1); ++r) {
    const int64_t share = slots * r / a.n_qg / 8 * 8, each = (units + share - 1) / share;
    const int64_t n_wg = ((fill ? std::min(share, units) : (units + each - 1) / each) + 7) / 8 * 8;
    const int64_t rounds = (n_wg * a.n_qg + slots - 1) / slots;
    if (best < 0 || rounds * (each + 1) < best) {
      best = rounds * (each + 1);
      a.n_wg = (int)n_wg;
    }
  }
  const dim3 grid((unsigned)(a.n_wg * a.n_qg)), block(256);
  auto go = [&](auto edt) {
    constexpr int EDT = decltype(edt)::value;
    if (qt == 1) hipLaunchKernelGGL((few_scan_kernel<EDT, 1, MODE>), grid, block, lds, st, a);
    else if (qt == 2) hipLaunchKernelGGL((few_scan_kernel<EDT, 2, MODE>), grid, block, lds, st, a);
    else if constexpr (MODE < FEW_STORE) hipLaunchKernelGGL((few_scan_kernel<EDT, 4, MODE>), grid, block, lds, st, a);
  };
  if (dtype == KGE_F32) go(std::integral_constant<int, KGE_F32>{});
  else if constexpr (MODE != FEW_GRAD) {
    if (dtype == KGE_BF16) go(std::integral_constant<int, KGE_BF16>{});
    else go(std::integral_constant<int, KGE_I8>{});
  }
  KGE_LAUNCH_CHECK("few_scan_kernel");
  return KGE_OK;
}
}  // namespace

int few_scores_launch(const float* Q, const float* bias, const void* E, int dtype, const float* scale, int64_t B, int64_t d,
                      int64_t N, float* out, int64_t ldo, hipStream_t st) {
  FewArgs a{Q, E, scale, bias, out, nullptr, nullptr, ldo, 0, N, 0, (int)B, (int)d, 0, 0, 0, 0, {}};
  return launch_few_scan<FEW_STORE>(dtype, a, st);
}

int few_grad_launch(const float* Q, const float* E, int64_t B, int64_t d, int64_t N, const GradArgs& grad, hipStream_t st) {
  FewArgs a{Q, E, nullptr, grad.bias, nullptr, nullptr, nullptr, 0, 0, N, 0, (int)B, (int)d, 0, 0, 0, 0, grad};
  return launch_few_scan<FEW_GRAD>(KGE_F32, a, st);
}

int few_topk_launch(const float* Q, const float* bias, const void* E, int dtype, const float* scale, int64_t B, int64_t d,
                    int64_t N, int64_t k, float* out_scores, int64_t* out_idx, int apply_sigmoid, void* workspace,
                    hipStream_t st) {
  const host::FewTopkWs w = host::few_topk_ws(B, N);
  float* maxima = (float*)workspace;
  float* runs = w.runs ? maxima + w.runs : nullptr;
  float* raw = w.raw ? maxima + w.raw : nullptr;
  FewArgs a{Q, E, scale, nullptr, maxima, runs, raw, w.ldm, w.ldr, N, 0, (int)B, (int)d, 0, 0, 0, 0, {}};
  const int rc = raw ? launch_few_scan<FEW_MAX_RAW>(dtype, a, st) : launch_few_scan<FEW_MAX>(dtype, a, st);
  if (rc) return rc;
  FewFinishArgs f{Q, E, scale, bias, maxima, runs, raw, w.ldm, w.ldr, N, (N + 31) / 32, (int)d, (int)k, apply_sigmoid,
                  out_scores, out_idx};
  const dim3 grid((unsigned)B), block(FEW_THREADS);
  if (raw) hipLaunchKernelGGL((few_finish_kernel<KGE_F32, true>), grid, block, 0, st, f);  // (whatever the table's type)
  else if (dtype == KGE_F32) hipLaunchKernelGGL((few_finish_kernel<KGE_F32, false>), grid, block, 0, st, f);
  else if (dtype == KGE_BF16) hipLaunchKernelGGL((few_finish_kernel<KGE_BF16, false>), grid, block, 0, st, f);
  else hipLaunchKernelGGL((few_finish_kernel<KGE_I8, false>), grid, block, 0, st, f);
  KGE_LAUNCH_CHECK("few_finish_kernel");
  return KGE_OK;
}
}  // namespace kge

extern "C" size_t kge_topk_values_workspace_bytes(int64_t N) {
  return N > kge::host::FEW_TILES_DIRECT ? (size_t)((N + 31) / 32) * 4 : 0;
}

namespace kge {
namespace {
int topk_values_impl(const float* values, int64_t N, int64_t k, float* out_values, int64_t* out_idx, int64_t idx_stride,
                     int64_t relation, void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  KGE_REQUIRE(N >= 1 && N <= 32LL * FEW_TILES_DIRECT, KGE_ERR_UNSUPPORTED, "kge_topk_values: N=%lld outside [1, %lld]",
              (long long)N, 32LL * FEW_TILES_DIRECT);
  KGE_REQUIRE(k >= 1 && k <= N && k <= FEW_MAX_K, KGE_ERR_UNSUPPORTED, "kge_topk_values: k=%lld outside [1, min(N, %d)]",
              (long long)k, FEW_MAX_K);
  KGE_REQUIRE(values && out_values && out_idx, KGE_ERR_INVALID, "kge_topk_values: null pointer argument");
  const size_t need = ::kge_topk_values_workspace_bytes(N);
  KGE_REQUIRE(need == 0 || (workspace && workspace_bytes >= need && ((uintptr_t)workspace & 3) == 0), KGE_ERR_WORKSPACE,
              "kge_topk_values: workspace of %zu bytes, need %zu, 4-byte aligned", workspace_bytes, need);
  hipStream_t st = (hipStream_t)stream;
  const int n_tiles = (int)((N + 31) / 32);
  uint32_t* tiles = need ? (uint32_t*)workspace : nullptr;
  if (tiles) {
    hipLaunchKernelGGL(value_tiles_kernel, dim3((unsigned)((n_tiles + 7) / 8)), dim3(256), 0, st, values, (int)N, tiles, n_tiles);
    KGE_LAUNCH_CHECK("value_tiles_kernel");
  }
  hipLaunchKernelGGL(topk_values_kernel, dim3(1), dim3(FEW_THREADS), 0, st, values, (int)N, tiles, n_tiles, (int)k, out_values,
                     out_idx, idx_stride, relation);
  KGE_LAUNCH_CHECK("topk_values_kernel");
  return KGE_OK;
}

// out[n] = the largest of t(weight[j], S[j, n]) over the substitutions j: a thread per entity, four rows' loads in flight
template <bool MIN>
__global__ void __launch_bounds__(256) hop_scores_kernel(const float* weight, const float* S, int k, int64_t N, int64_t ldS, float* out) {
  const int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (n >= N) return;
  float best = 0.f;
#pragma unroll 4
  for (int j = 0; j < k; ++j) {
    const float w = weight[j], s = S[j * ldS + n];
    const float v = MIN ? (w != w ? w : s < w || s != s ? s : w) : w * s;
    best = j == 0 || v > best || v != v ? v : best;  // (a NaN stays: nothing is greater)
  }
  out[n] = best;
}
}  // namespace
}  // namespace kge

extern "C" int kge_topk_values(const float* values, int64_t N, int64_t k, float* out_values, int64_t* out_idx,
                               void* workspace, size_t workspace_bytes, void* stream) {
  return kge::topk_values_impl(values, N, k, out_values, out_idx, 1, 0, workspace, workspace_bytes, stream);
}

extern "C" int kge_topk_values_pairs(const float* values, int64_t N, int64_t k, int64_t relation, float* out_values,
                                     int64_t* out_pairs, void* workspace, size_t workspace_bytes, void* stream) {
  return kge::topk_values_impl(values, N, k, out_values, out_pairs, 2, relation, workspace, workspace_bytes, stream);
}

extern "C" int kge_hop_scores(const float* weight, const float* S, int64_t k, int64_t N, int64_t ldS, int tnorm, float* out,
                              void* stream) {
  using namespace kge;
  clear_error();
  KGE_REQUIRE(k >= 1 && k <= 0x7fffffff && N >= 1 && N <= 0x7fffffffLL * 256 && ldS >= N && (tnorm == 0 || tnorm == 1), KGE_ERR_INVALID,
              "kge_hop_scores: k=%lld N=%lld ldS=%lld tnorm=%d", (long long)k, (long long)N, (long long)ldS, tnorm);
  KGE_REQUIRE(weight && S && out, KGE_ERR_INVALID, "kge_hop_scores: null pointer argument");
  const dim3 grid((unsigned)((N + 255) / 256)), block(256);
  if (tnorm) hipLaunchKernelGGL((hop_scores_kernel<true>), grid, block, 0, (hipStream_t)stream, weight, S, (int)k, N, ldS, out);
  else hipLaunchKernelGGL((hop_scores_kernel<false>), grid, block, 0, (hipStream_t)stream, weight, S, (int)k, N, ldS, out);
  KGE_LAUNCH_CHECK("hop_scores_kernel");
  return KGE_OK;
}
