// Few queries against the whole table (gfx950): the scan of kge_topk and the store of kge_scores for batches of at most
// 128 queries.
//
// The main loops of kge_contract.hip.h give every wave its own queries and every workgroup all of a chunk's rows: 512
// queries (256 / 128) per workgroup, so that a batch of 32 multiplies sixteen times the rows it needs, for padding
// queries, and runs at the matrix rate of the padding (bf16 d = 128, N = 2.5M, B = 32: 2.9 TB/s of table).  Here all waves
// hold the SAME queries, as MFMA fragments in LDS, and share out the entity rows, which go from global memory straight
// into fragment registers: what bounds the scan is the table's bytes.
// Measured, whole calls: top-10 of 32 queries, bf16 d = 128, N = 2.5M 408 -> 193 us; top-10 of one question by name, fp32
// d = 256, N = 41k 284 -> 141 us (the rounds of the large-batch form were four to seven scans and selections, and a
// read-back).
//
// Scores are formed by the chain every kernel uses (K steps of 16 ascending; fp32 operands as three bf16 parts, six
// products in SPLIT order), so they carry the same bits.
#include "kge_contract.hip.h"

#include <algorithm>

namespace kge {
namespace {

using host::FEW_LDS_KB;
using host::FEW_MAX_K;
using host::FEW_TILES_DIRECT;

struct FewArgs {
  const float* Q;
  const void* E;
  const float* scale;
  const float* bias;  // STORE only
  float* out;         // STORE: scores [B, ldo]; else the maximum over every 32-row tile [B, ldo]
  int64_t ldo, N, n_tiles;
  int B, d, nks;
  int tpw;  // consecutive tiles a wave takes at a time
};

// One wave at a time: 32-row tiles, their rows as MFMA operands straight from memory (lane (c, hf) reads its 16 or 32
// bytes of row c; four K steps of a bf16 row, two of an fp32 row make a 128-byte line, requested back to back), the
// loads of one chunk of K steps in flight while the chunk before is multiplied, across tiles.
template <int EDT, int QT, bool STORE>
__global__ void __launch_bounds__(256, QT > 1 ? 2 : EDT == KGE_F32 ? 3 : 4) few_scan_kernel(FewArgs a) {
  constexpr int PARTS = EDT == KGE_F32 ? 3 : 1;
  constexpr int CH = EDT == KGE_F32 ? 4 : 8;  // K steps per chunk: eight 16-byte loads (int8: eight of 8 bytes)
  extern __shared__ __attribute__((aligned(16))) unsigned char fq_lds[];
  __shared__ float s_bias[32 * QT];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, hf = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q0 = (int)blockIdx.y * (32 * QT);
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

  struct Chunk {
    u32x4 v[CH * (EDT == KGE_F32 ? 2 : 1)];  // (int8: the low halves)
    f32x4 sc[EDT == KGE_I8 ? 4 : 1];
  };
  const int nch = (nks + CH - 1) / CH;
  int64_t unit = blockIdx.x, tile = (unit * 4 + wave) * a.tpw;
  int ch = 0, in_unit = 0;
  // the position after (tile, ch); past the end: tile >= n_tiles
  auto advance = [&]() {
    if (++ch < nch) return;
    ch = 0;
    ++tile;
    if (++in_unit == a.tpw) {
      in_unit = 0;
      unit += gridDim.x;
      tile = (unit * 4 + wave) * a.tpw;
    }
  };
  auto load = [&](Chunk& x) {
    int64_t row = tile * 32 + c;
    row = row < a.N ? row : a.N - 1;  // rows past the end repeat the last one; the epilogues ignore them
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int k = (ch * CH + u) * 16 + 8 * hf;
      if constexpr (EDT == KGE_F32) {
        const float* p = (const float*)a.E + row * d;
        x.v[2 * u] = *(const u32x4*)(p + (k < d ? k : 0));
        x.v[2 * u + 1] = *(const u32x4*)(p + (k + 4 < d ? k + 4 : 0));
      } else if constexpr (EDT == KGE_BF16) {
        x.v[u] = *(const u32x4*)((const uint16_t*)a.E + row * d + (k < d ? k : 0));
      } else {
        const u32x2 w = *(const u32x2*)((const int8_t*)a.E + row * d + (k < d ? k : 0));
        x.v[u][0] = w[0];
        x.v[u][1] = w[1];
      }
    }
    if constexpr (EDT == KGE_I8) {
      if (STORE) {
        x.sc[0][0] = a.scale[row];
      } else if (ch == nch - 1) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int64_t e = tile * 32 + 8 * g + 4 * hf;
#pragma unroll
          for (int j = 0; j < 4; ++j) x.sc[g][j] = a.scale[e + j < a.N ? e + j : a.N - 1];
        }
      }
    }
  };
  f32x16 acc[QT];
  auto multiply = [&](Chunk& x, int64_t t_tile, int t_ch) {
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
          f32x4 lo = __builtin_bit_cast(f32x4, x.v[2 * u]), hi = __builtin_bit_cast(f32x4, x.v[2 * u + 1]);
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
          u32x4 w = x.v[u];
          if constexpr (EDT == KGE_I8) w = i8x8_to_bf16x8(w[0], w[1]);
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
    if constexpr (STORE) {
      const int64_t e = t_tile * 32 + c;
      if (e < a.N) {
#pragma unroll
        for (int t = 0; t < QT; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int r = 32 * t + row_of(i, hf);
            if (q0 + r < a.B) {
              const float v = EDT == KGE_I8 ? acc[t][i] * x.sc[0][0] : acc[t][i];
              a.out[(int64_t)(q0 + r) * a.ldo + e] = v + s_bias[r];
            }
          }
      }
    } else {
      const bool whole = t_tile * 32 + 32 <= a.N;
#pragma unroll
      for (int t = 0; t < QT; ++t) {
        float m = __uint_as_float(0xff800000u);  // (a NaN score never becomes the maximum)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          float v = acc[t][i];
          if constexpr (EDT == KGE_I8) v *= x.sc[i >> 2][i & 3];
          if (!whole && t_tile * 32 + row_of(i, hf) >= a.N) v = __uint_as_float(0xff800000u);
          m = __builtin_fmaxf(m, v);
        }
        m = __builtin_fmaxf(m, __shfl_xor(m, 32, 64));
        const int q = q0 + 32 * t + c;
        if (hf == 0 && q < a.B) a.out[(int64_t)q * a.ldo + t_tile] = m;
      }
    }
  };
  if (tile >= a.n_tiles) return;
  Chunk x0, x1;
  load(x0);
  for (;;) {
    int64_t t_tile = tile;
    int t_ch = ch;
    advance();
    const bool more1 = tile < a.n_tiles;
    if (more1) load(x1);
    multiply(x0, t_tile, t_ch);
    if (!more1) break;
    t_tile = tile;
    t_ch = ch;
    advance();
    const bool more0 = tile < a.n_tiles;
    if (more0) load(x0);
    multiply(x1, t_tile, t_ch);
    if (!more0) break;
  }
}

// ---- the best k from the tile maxima ----------------------------------------------------------------------
// The best k entities (score descending, id ascending) lie in the best k tiles (maximum descending, tile ascending): if a
// tile is not among them, k tiles hold an entity each that ranks above everything in it (a higher score, or the same
// score at a lower id).  So one workgroup per query picks the k best tiles, forms their 32 k scores again and picks the
// k best of those: no thresholds, no candidate buffers that could overflow, nothing read back.  Tables of more than
// FEW_TILES_DIRECT tiles go through the maxima of 32 tiles first, by the same argument.
struct SelectShared {
  unsigned long long cnt[16];
  uint32_t scan[256];
};
constexpr int FEW_THREADS = 1024;

__device__ __forceinline__ uint32_t score_key(float v) {
  return v > __uint_as_float(0xff800000u) ? f32_to_ordered(v) : 0u;  // NaN and -inf are never ranked
}

// The positions of the k largest of vals[0 .. M) (ties: the lower positions; zeros never), ascending, into pos; returns
// how many.  M <= 16 * FEW_THREADS.  The k-th largest value is found two bits at a time, three counts per step, by the
// whole workgroup; a step that splits off exactly k ends the search.
__device__ int block_select(const uint32_t* vals, int M, int k, int* pos, SelectShared& sh) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int V = (M + FEW_THREADS - 1) / FEW_THREADS;
  __syncthreads();  // vals is complete; sh and pos are free
  if (tid < 16) sh.cnt[tid] = 0;
  uint32_t v[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    v[j] = 0;
    if (j < V) {
      const int p = j * FEW_THREADS + tid;
      if (p < M) v[j] = vals[p];
    }
  }
  __syncthreads();
  uint32_t th = 0;
  bool exact = false;  // exactly k values are >= th
  for (int b = 30; b >= 0 && !exact; b -= 2) {
    const uint32_t t1 = th | (1u << b), t2 = th | (2u << b), t3 = th | (3u << b);
    int c1 = 0, c2 = 0, c3 = 0;
#pragma unroll
    for (int j = 0; j < 16; ++j)
      if (j < V) {
        c1 += __builtin_popcountll(__builtin_amdgcn_ballot_w64(v[j] >= t1));
        c2 += __builtin_popcountll(__builtin_amdgcn_ballot_w64(v[j] >= t2));
        c3 += __builtin_popcountll(__builtin_amdgcn_ballot_w64(v[j] >= t3));
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
#pragma unroll
  for (int j = 0; j < 16; ++j)
    if (j < V) {
      const int ng = __builtin_popcountll(__builtin_amdgcn_ballot_w64(v[j] > above));
      const int ne = __builtin_popcountll(__builtin_amdgcn_ballot_w64(at != 0 && v[j] == at));
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
#pragma unroll
  for (int j = 0; j < 16; ++j)
    if (j < V) {
      const unsigned long long bg = __builtin_amdgcn_ballot_w64(v[j] > above);
      const unsigned long long be = __builtin_amdgcn_ballot_w64(at != 0 && v[j] == at);
      const uint32_t base = sh.scan[j * 16 + wave];
      const int g = (int)(base & 0xffff) + __builtin_popcountll(bg & below_lane);
      const int e = (int)(base >> 16) + __builtin_popcountll(be & below_lane);
      if (v[j] > above || (at != 0 && v[j] == at && e < need)) pos[g + (e < need ? e : need)] = j * FEW_THREADS + tid;
    }
  __syncthreads();
  return n_gt + need;
}

struct FewFinishArgs {
  const float* Q;
  const void* E;
  const float* scale;
  const float* bias;
  const float* maxima;  // [B, ldm]
  int64_t ldm, N, n_tiles;
  int d, k, sigmoid;
  float* out_scores;
  int64_t* out_idx;
};

template <int EDT>
__global__ void __launch_bounds__(FEW_THREADS) few_finish_kernel(FewFinishArgs a) {
  __shared__ uint32_t vals[16 * FEW_THREADS];
  __shared__ int pos[FEW_MAX_K], groups[FEW_MAX_K];
  __shared__ int64_t tiles[FEW_MAX_K];
  __shared__ unsigned long long keys[FEW_MAX_K];
  __shared__ SelectShared sh;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, hf = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t q = blockIdx.x;
  const float* mx = a.maxima + q * a.ldm;
  const int T = (int)a.n_tiles, k = a.k;
  int n;
  if (T <= FEW_TILES_DIRECT) {
    for (int t = tid; t < T; t += FEW_THREADS) vals[t] = score_key(mx[t]);
    n = block_select(vals, T, k, pos, sh);
    for (int j = tid; j < n; j += FEW_THREADS) tiles[j] = pos[j];
  } else {
    const int G = (T + 31) / 32;
    for (int g = tid; g < G; g += FEW_THREADS) {
      float m = __uint_as_float(0xff800000u);
      if (32 * g + 32 <= T) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const f32x4 x = *(const f32x4*)(mx + 32 * (int64_t)g + 4 * i);
          m = __builtin_fmaxf(__builtin_fmaxf(__builtin_fmaxf(m, x[0]), __builtin_fmaxf(x[1], x[2])), x[3]);
        }
      } else {
        for (int t = 32 * g; t < T; ++t) m = __builtin_fmaxf(m, mx[t]);
      }
      vals[g] = score_key(m);
    }
    const int ng = block_select(vals, G, k, groups, sh);
    for (int i = tid; i < 32 * ng; i += FEW_THREADS) {
      const int t = 32 * groups[i >> 5] + (i & 31);
      vals[i] = t < T ? score_key(mx[t]) : 0u;
    }
    n = block_select(vals, 32 * ng, k, pos, sh);
    for (int j = tid; j < n; j += FEW_THREADS) tiles[j] = 32 * (int64_t)groups[pos[j] >> 5] + (pos[j] & 31);
  }
  __syncthreads();
  // the tiles' scores again: every column of the result tile holds this query, lane c < 16 keeps accumulator c
  for (int j = wave; j < n; j += FEW_THREADS / 64) {
    const int64_t row = tiles[j] * 32 + c;
    const f32x16 acc = chain_direct<EDT>(a.E, a.d, row < a.N ? row : -1, a.Q, q, hf);
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
  n = block_select(vals, 32 * n, k, pos, sh);
  for (int j = tid; j < n; j += FEW_THREADS)
    keys[j] = ((unsigned long long)vals[pos[j]] << 32) | (0xffffffffull - (unsigned long long)(tiles[pos[j] >> 5] * 32 + (pos[j] & 31)));
  __syncthreads();
  for (int j = tid; j < k; j += FEW_THREADS) {
    int at = j;
    float s = __uint_as_float(0x7fc00000u);
    int64_t e = -1;
    if (j < n) {
      const unsigned long long key = keys[j];
      at = 0;
      for (int i = 0; i < n; ++i) at += keys[i] > key ? 1 : 0;
      s = ordered_to_f32((uint32_t)(key >> 32));
      e = (int64_t)(0xffffffffu - (uint32_t)(key & 0xffffffffull));
      if (a.bias) s += a.bias[q];
      if (a.sigmoid) s = 1.0f / (1.0f + expf(-s));
    }
    a.out_scores[q * k + at] = s;
    a.out_idx[q * k + at] = e;
  }
}

template <bool STORE>
int launch_few_scan(int dtype, FewArgs a, hipStream_t st) {
  const int parts = dtype == KGE_F32 ? 3 : 1;
  a.nks = (a.d + 15) / 16;
  a.n_tiles = (a.N + 31) / 32;
  // as many query tiles per wave as the batch has and LDS holds fragments of: every tile reads the table's rows once
  int qt = 1;
  while (qt < (STORE ? 2 : 4) && 32 * qt < a.B && 2 * qt * a.nks * parts <= FEW_LDS_KB) qt *= 2;
  const int n_qg = (a.B + 32 * qt - 1) / (32 * qt);
  // four workgroups per CU walk units of 4 * tpw tiles; the longest runs that leave each of them four units
  a.tpw = 8;
  while (a.tpw > 1 && a.n_tiles < (int64_t)4 * a.tpw * 4096) a.tpw /= 2;
  const int64_t units = (a.n_tiles + 4 * a.tpw - 1) / (4 * a.tpw);
  const dim3 grid((unsigned)std::min<int64_t>(units, 1024), (unsigned)n_qg), block(256);
  const size_t lds = (size_t)qt * a.nks * parts * 1024;
  auto go = [&](auto edt) {
    constexpr int EDT = decltype(edt)::value;
    if (qt == 1) hipLaunchKernelGGL((few_scan_kernel<EDT, 1, STORE>), grid, block, lds, st, a);
    else if (qt == 2) hipLaunchKernelGGL((few_scan_kernel<EDT, 2, STORE>), grid, block, lds, st, a);
    else if constexpr (!STORE) hipLaunchKernelGGL((few_scan_kernel<EDT, 4, STORE>), grid, block, lds, st, a);
  };
  if (dtype == KGE_F32) go(std::integral_constant<int, KGE_F32>{});
  else if (dtype == KGE_BF16) go(std::integral_constant<int, KGE_BF16>{});
  else go(std::integral_constant<int, KGE_I8>{});
  KGE_LAUNCH_CHECK("few_scan_kernel");
  return KGE_OK;
}
}  // namespace

int few_scores_launch(const float* Q, const float* bias, const void* E, int dtype, const float* scale, int64_t B, int64_t d,
                      int64_t N, float* out, int64_t ldo, hipStream_t st) {
  FewArgs a{Q, E, scale, bias, out, ldo, N, 0, (int)B, (int)d, 0, 0};
  return launch_few_scan<true>(dtype, a, st);
}

int few_topk_launch(const float* Q, const float* bias, const void* E, int dtype, const float* scale, int64_t B, int64_t d,
                    int64_t N, int64_t k, float* out_scores, int64_t* out_idx, int apply_sigmoid, void* workspace,
                    hipStream_t st) {
  const int64_t ldm = host::few_maxima_pitch(N);
  FewArgs a{Q, E, scale, nullptr, (float*)workspace, ldm, N, 0, (int)B, (int)d, 0, 0};
  int rc = launch_few_scan<false>(dtype, a, st);
  if (rc) return rc;
  FewFinishArgs f{Q, E, scale, bias, (const float*)workspace, ldm, N, (N + 31) / 32, (int)d, (int)k, apply_sigmoid,
                  out_scores, out_idx};
  const dim3 grid((unsigned)B), block(FEW_THREADS);
  if (dtype == KGE_F32) hipLaunchKernelGGL((few_finish_kernel<KGE_F32>), grid, block, 0, st, f);
  else if (dtype == KGE_BF16) hipLaunchKernelGGL((few_finish_kernel<KGE_BF16>), grid, block, 0, st, f);
  else hipLaunchKernelGGL((few_finish_kernel<KGE_I8>), grid, block, 0, st, f);
  KGE_LAUNCH_CHECK("few_finish_kernel");
  return KGE_OK;
}
}  // namespace kge
