// Products for the layouts that the tiled kernels do not take: K or N off the 64 grid, ranks
// off 8, rows or pointers that are not 16-byte aligned. Same arithmetic contract as the other
// paths: fp32 accumulation, T = bf16(s * x.A^T) rounded once, y = bf16((x.W^T) * w_scale + T.B^T).
//
// One kernel, c[i][j] = bf16(scale * sum over k of P(i, k) Q(j, k)), on v_mfma_f32_32x32x16_bf16.
// Each operand stores either k along its rows (x, W, A, gy in the forward products) or k as its
// rows ("token-major": gy, x, T, U in the weight gradients, W and A in the input gradient). Both
// are loaded as rows of 8-element chunks, bounds-checked against the operand's own extent (one
// 16-byte load a chunk, whatever its alignment), staged through LDS with zeros past the edges, and read back as MFMA
// fragments (plain reads, or gfx950's transposing reads for a token-major operand). So no
// operand is copied or padded in memory.
//
// A workgroup of four waves owns a BT x BT tile and walks k in steps of KT (64 x 128 tiles of
// both operands, or 128 x 64), the next two steps' loads in flight in registers while this
// one is multiplied, LDS double-buffered with one barrier a step. 128-wide tiles where they alone fill
// the 256 CUs, else 64-wide: these products are small, and their time is the chain of loads
// (steps x a memory round trip), which the longer k steps of the 64-wide tile shorten.
//
// Measured at 777 x 1500 x 1000, r = 12: forward 204 us a scalar kernel per element before, 30 now;
// input gradient 38, both factor gradients 45 (a training step 1202 us before, 2 launches more).
#include <algorithm>

#include "wsl_common.h"

namespace wsl {
namespace {

typedef short v4i16_t __attribute__((ext_vector_type(4)));

constexpr int GP_T = 256;               // threads: 2 x 2 waves
constexpr int GP_TILE = 16384;          // bytes of one operand's tile, BT * KT * 2
constexpr int GP_CH = GP_TILE / 16 / GP_T;  // 16-byte chunks per thread, operand and step

// One product. `p` is [I, K] (or [K, I] token-major), `q` [J, K] (or [K, J]); a second segment
// (K2 > 0) adds P2 . Q2^T after the first segment's sums are multiplied by cscale[column].
struct GenericJob {
  const uint16_t* p; int64_t ldp;
  const void* q; int64_t ldq;
  int64_t K;
  const uint16_t* p2; int64_t ldp2;
  const uint16_t* q2; int64_t ldq2;
  int64_t K2;
  const int64_t* gather; int64_t gather_rows;  // row i of p is row gather[i] of a [gather_rows, ldp] table
  const float* cscale;
  RowMap qmap;                                 // row of q (and cscale) by output column
  int64_t I, J;
  float scale;
  uint16_t* c; int64_t ldc;
  int64_t tiles_j, tiles;
};
constexpr int GP_JOBS = 3;
struct GenericJobs {
  GenericJob job[GP_JOBS];
  int n;
};


// The GP_CH chunks that a thread holds of one operand's next tile, as loaded. Each is one
// unconditional load, so that all of a step's loads are in flight together and nothing waits for
// them before they are written to LDS: a chunk outside the operand loads its first elements, and
// one that the rows' end cuts loads the row's last eight. What is to be done about that is kept
// as four bits a chunk (elements to shift out, or kOutside) and done on the way to LDS. Operands
// with rows of fewer than eight elements are loaded element by element, in kernels of their own
// (SHORT: with both ways in one kernel, every use of a loaded register would wait for all of them).
constexpr uint32_t kOutside = 8;
struct Chunks {
  u32x4_t v[GP_CH];
  uint32_t code;
};
// The addresses of a thread's chunks of one operand, moved along k step by step. The step's
// chunks are tile rows of CH chunks: rows of the operand over columns k (plain), or rows k over
// the operand's columns (TOK).
template <int CH, int KT, bool TOK, bool F8, bool SHORT>
struct Loader {
  const char* at[GP_CH];  // this step's chunk, its columns moved back inside the row
  uint32_t fixed;         // codes of what is the same in every step: rows past the end, TOK: columns
  int64_t step;           // bytes from one step to the next
  int64_t ld, len;        // bytes between operand rows, elements of an operand row
  static constexpr int ES = F8 ? 1 : 2;

  // row(u): operand row of chunk u (plain; < 0: outside). c0: first column (TOK). n: k in all
  // (TOK: operand rows), cols: elements of an operand row.
  template <class Row>
  __device__ __forceinline__ void init(const void* base, int64_t ld_elems, int tid, int64_t c0, int64_t cols, Row row) {
    ld = ld_elems * ES;
    len = cols;
    step = TOK ? KT * ld : KT * ES;
    fixed = 0;
#pragma unroll
    for (int u = 0; u < GP_CH; ++u) {
      const int idx = tid + GP_T * u;
      const int64_t r = TOK ? (int64_t)(idx / CH) : row(u);
      int64_t c = (TOK ? c0 : 0) + (idx % CH) * 8;
      uint32_t code = 0;
      if (TOK) {
        if (c >= cols) code = kOutside;
        else if (c + 8 > cols) code = (uint32_t)(c + 8 - cols);
        if (code != 0) c = cols - 8;
      } else if (r < 0) {
        code = kOutside;
      }
      fixed |= code << (4 * u);
      at[u] = reinterpret_cast<const char*>(base) + (r < 0 ? 0 : r) * ld + c * ES;
    }
  }
  // The next step's loads; `rem`: k left from this step's start.
  __device__ __forceinline__ void load(Chunks& ch, int tid, int64_t rem) {
    const char* p[GP_CH];
    ch.code = fixed;
#pragma unroll
    for (int u = 0; u < GP_CH; ++u) p[u] = at[u];
    if (rem < KT) {  // the last step of the segment
      const int left = (int)rem;
#pragma unroll
      for (int u = 0; u < GP_CH; ++u) {
        const int k = TOK ? (tid + GP_T * u) / CH : ((tid + GP_T * u) % CH) * 8;
        uint32_t code = 0;
        int64_t back;
        if (TOK) {
          code = k >= left ? kOutside : 0;
          back = k >= left ? (int64_t)(k - left + 1) * ld : 0;
        } else {
          const int over = k + 8 - left;  // elements past the row's end
          code = over >= 8 ? kOutside : over > 0 ? (uint32_t)over : 0;
          back = over > 0 ? (int64_t)over * ES : 0;
        }
        p[u] -= back;
        const uint32_t f = fixed >> (4 * u) & 15;
        ch.code = (ch.code & ~(15u << (4 * u))) | ((f == kOutside ? f : code | (TOK && code == 0 ? f : 0)) << (4 * u));
      }
    }
    if (!SHORT || len >= 8) {
#pragma unroll
      for (int u = 0; u < GP_CH; ++u) {
        if (F8) {
          uint2 q;
          __builtin_memcpy(&q, p[u], 8);
          ch.v[u][0] = q.x;
          ch.v[u][1] = q.y;
        } else {
          __builtin_memcpy(&ch.v[u], p[u], 16);
        }
      }
      return;
    }
    // rows of fewer than eight elements: only their first chunk is inside, moved back by 8 - len
#pragma unroll
    for (int u = 0; u < GP_CH; ++u) {
      ch.v[u] = zero_u32x4();
      const uint32_t code = ch.code >> (4 * u) & 15;
      if (code == kOutside) continue;
      ch.code &= ~(15u << (4 * u));
      const char* r = p[u] + (8 - len) * ES;
#pragma unroll
      for (int e = 0; e < 7; ++e) {
        if (e >= len) break;
        if (F8) ch.v[u][e >> 2] |= (uint32_t)(uint8_t)r[e] << ((e & 3) * 8);
        else ch.v[u][e >> 1] |= (uint32_t)reinterpret_cast<const uint16_t*>(r)[e] << ((e & 1) * 16);
      }
    }
  }
  __device__ __forceinline__ void advance() {
#pragma unroll
    for (int u = 0; u < GP_CH; ++u) at[u] += step;
  }
};
template <bool F8>
__device__ __forceinline__ u32x4_t chunk(const Chunks& ch, int u) {
  const uint32_t code = ch.code >> (4 * u) & 15;
  if (code == kOutside) return zero_u32x4();
  uint64_t lo = (uint64_t)ch.v[u][1] << 32 | ch.v[u][0], hi = (uint64_t)ch.v[u][3] << 32 | ch.v[u][2];
  if (F8) {
    lo >>= 8 * code;
    return fp8x8_to_bf16x8((uint32_t)lo, (uint32_t)(lo >> 32));
  }
  if (code != 0) {
    const int n = 16 * (int)code;
    lo = n >= 64 ? hi >> (n - 64) : lo >> n | hi << (64 - n);
    hi = n >= 64 ? 0 : hi >> n;
  }
  return u32x4_t{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}

// Byte offset of 16-byte chunk c of a tile row of RB bytes. Plain fragments read 16 rows at one
// chunk index, transposed ones 4 rows of 4 chunks: each spreads over all the banks.
template <int RB, bool TOK>
__device__ __forceinline__ int tile_off(int row, int c) {
  int s;
  if (TOK) s = RB == 256 ? (row & 3) << 2 : ((row >> 1) & 1) << 2;
  else s = RB == 256 ? row & 15 : (row >> 1) & 7;
  return row * RB + ((c ^ s) << 4);
}

__device__ __forceinline__ uint2 read_tr4(const char* p) {
  const v4i16_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4i16_t*)p);
  return uint2{(uint32_t)(uint16_t)v[0] | ((uint32_t)(uint16_t)v[1] << 16),
               (uint32_t)(uint16_t)v[2] | ((uint32_t)(uint16_t)v[3] << 16)};
}
__device__ __forceinline__ f32x16_t mfma16(u32x4_t a, u32x4_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}

// Workgroup barrier after this wave's LDS accesses; loads in flight into registers are not waited
// for (the release fence of __syncthreads() would wait for them).
__device__ __forceinline__ void tile_barrier() {
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0); vmcnt, expcnt unconstrained
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The MFMA operand of tile rows f0..f0+31 over k 16 ks + 8 (lane / 32) + 0..7.
template <int BT, int KT, bool TOK>
__device__ __forceinline__ u32x4_t frag(const char* tile, int f0, int ks, int lane) {
  const int h = lane >> 5;
  if (!TOK) {
    const int row = f0 + (lane & 31);
    return *reinterpret_cast<const u32x4_t*>(tile + tile_off<KT * 2, false>(row, 2 * ks + h));
  }
  const int j = lane & 15, col = f0 + 16 * ((lane >> 4) & 1) + 4 * (j & 3);
  u32x4_t v;
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    const int row = 16 * ks + 8 * h + 4 * half + (j >> 2);
    const uint2 t = read_tr4(tile + tile_off<BT * 2, true>(row, col >> 3) + (j & 1) * 8);
    v[2 * half] = t.x;
    v[2 * half + 1] = t.y;
  }
  return v;
}

// PT, QT: p, q token-major. Q8: q holds e4m3 (plain layout only). SHORT: an operand's rows have
// fewer than eight elements.
template <int BT, int KT, bool PT, bool QT, bool Q8, bool SHORT>
__global__ void __launch_bounds__(GP_T, 2) generic_product_kernel(const GenericJobs jobs) {
  constexpr int WT = BT / 2, NB = WT / 32;  // wave tile, its MFMA blocks per side
  __shared__ __attribute__((aligned(1024))) char smem[2][2][GP_TILE];
  int64_t b = blockIdx.x;
  int ji = 0;
  while (ji + 1 < jobs.n && b >= jobs.job[ji].tiles) b -= jobs.job[ji++].tiles;
  const GenericJob& J = jobs.job[ji];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t i0 = (b / J.tiles_j) * BT, j0 = (b % J.tiles_j) * BT;
  const int wi = (wave >> 1) * WT, wj = (wave & 1) * WT;

  constexpr int PC = PT ? BT / 8 : KT / 8, QC = QT ? BT / 8 : KT / 8;  // chunks per tile row
  Loader<PC, KT, PT, false, SHORT> pl;
  Loader<QC, KT, QT, false, SHORT> ql;
  Loader<QC, KT, QT, true, SHORT> ql8;  // an e4m3 q (the first segment's)
  const int64_t s1 = (J.K + KT - 1) / KT, steps = s1 + (J.K2 + KT - 1) / KT;
  int64_t at = s1 > 0 ? 0 : s1, rem = 0;  // the step that the loaders stand at, and k from it on
  auto segment = [&](bool two) {
    rem = two ? J.K2 : J.K;
    pl.init(two ? J.p2 : J.p, two ? J.ldp2 : J.ldp, tid, i0, PT ? J.I : rem, [&](int u) {
      const int64_t i = i0 + (tid + GP_T * u) / PC;
      if (i >= J.I) return (int64_t)-1;
      if (two || J.gather == nullptr) return i;
      const int64_t id = J.gather[i];
      return id >= 0 && id < J.gather_rows ? id : (int64_t)-1;
    });
    auto qrow = [&](int u) {
      const int64_t j = j0 + (tid + GP_T * u) / QC;
      return j >= J.J ? (int64_t)-1 : two ? j : (int64_t)map_row((int)j, J.qmap);
    };
    if (Q8 && !two) ql8.init(J.q, J.ldq, tid, j0, rem, qrow);
    else ql.init(two ? (const void*)J.q2 : J.q, two ? J.ldq2 : J.ldq, tid, j0, QT ? J.J : rem, qrow);
  };
  Chunks pr[2], qr[2];  // two steps' loads: a step's are issued two steps before they are written to LDS
  // The loads of the step that the loaders stand at, and on to the next (the last is loaded again).
  auto load = [&](Chunks& pc, Chunks& qc) {
    pl.load(pc, tid, rem);
    if (Q8 && at < s1) ql8.load(qc, tid, rem);
    else ql.load(qc, tid, rem);
    if (at + 1 < steps) {
      if (++at == s1) {
        segment(true);
      } else {
        rem -= KT;
        pl.advance();
        if (Q8 && at < s1) ql8.advance();
        else ql.advance();
      }
    }
  };
  f32x16_t acc[NB][NB];
#pragma unroll
  for (int x = 0; x < NB; ++x)
#pragma unroll
    for (int y = 0; y < NB; ++y)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[x][y][e] = 0.f;
  const int64_t jl = j0 + wj + (lane & 31);  // this lane's column in block column 0
  auto scale_cols = [&]() {
#pragma unroll
    for (int y = 0; y < NB; ++y) {
      const int64_t j = jl + 32 * y;
      const float f = j < J.J ? J.cscale[map_row((int)j, J.qmap)] : 0.f;
#pragma unroll
      for (int x = 0; x < NB; ++x)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[x][y][e] *= f;
    }
  };

  auto step = [&](int64_t t, char* pt, char* qt, Chunks& pc, Chunks& qc) {
#pragma unroll
    for (int u = 0; u < GP_CH; ++u) {
      const int idx = tid + GP_T * u;
      *reinterpret_cast<u32x4_t*>(pt + tile_off<PC * 16, PT>(idx / PC, idx % PC)) = chunk<false>(pc, u);
      *reinterpret_cast<u32x4_t*>(qt + tile_off<QC * 16, QT>(idx / QC, idx % QC)) =
          Q8 && t < s1 ? chunk<true>(qc, u) : chunk<false>(qc, u);
    }
    tile_barrier();  // the other buffer's readers are a step behind this barrier's last one
    load(pc, qc);
    if (t == s1 && J.cscale != nullptr) scale_cols();
#pragma unroll
    for (int ks = 0; ks < KT / 16; ++ks) {
      u32x4_t pf[NB], qf[NB];
#pragma unroll
      for (int x = 0; x < NB; ++x) {
        pf[x] = frag<BT, KT, PT>(pt, wi + 32 * x, ks, lane);
        qf[x] = frag<BT, KT, QT>(qt, wj + 32 * x, ks, lane);
      }
#pragma unroll
      for (int x = 0; x < NB; ++x)
#pragma unroll
        for (int y = 0; y < NB; ++y) acc[x][y] = mfma16(pf[x], qf[y], acc[x][y]);
    }
  };
  if (steps > 0) {
    segment(s1 == 0);
    load(pr[0], qr[0]);
    load(pr[1], qr[1]);
    for (int64_t t = 0;;) {
      step(t, smem[0][0], smem[0][1], pr[0], qr[0]);
      if (++t == steps) break;
      step(t, smem[1][0], smem[1][1], pr[1], qr[1]);
      if (++t == steps) break;
    }
  }
  if (J.cscale != nullptr && J.K2 == 0) scale_cols();
  // element e of block (x, y): row 8 (e / 4) + 4 (lane / 32) + e % 4, column lane % 32
#pragma unroll
  for (int x = 0; x < NB; ++x)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int64_t i = i0 + wi + 32 * x + 8 * (e / 4) + 4 * (lane >> 5) + e % 4;
      if (i >= J.I) continue;
#pragma unroll
      for (int y = 0; y < NB; ++y)
        if (jl + 32 * y < J.J) J.c[i * J.ldc + jl + 32 * y] = f32_to_bf16_bits(J.scale * acc[x][y][e]);
    }
}

template <int BT, int KT, bool SHORT>
hipError_t launch_tiles(GenericJobs& jobs, bool pt, bool qt, bool q8, hipStream_t st) {
  int64_t total = 0;
  for (int i = 0; i < jobs.n; ++i) {
    GenericJob& j = jobs.job[i];
    j.tiles_j = (j.J + BT - 1) / BT;
    j.tiles = j.tiles_j * ((j.I + BT - 1) / BT);
    total += j.tiles;
  }
  if (total > 0x7fffffff) return hipErrorInvalidValue;
  const dim3 grid((unsigned)total), block(GP_T);
  if (q8) generic_product_kernel<BT, KT, false, false, true, SHORT><<<grid, block, 0, st>>>(jobs);
  else if (pt) generic_product_kernel<BT, KT, true, true, false, SHORT><<<grid, block, 0, st>>>(jobs);
  else if (qt) generic_product_kernel<BT, KT, false, true, false, SHORT><<<grid, block, 0, st>>>(jobs);
  else generic_product_kernel<BT, KT, false, false, false, SHORT><<<grid, block, 0, st>>>(jobs);
  return hipGetLastError();
}

// The jobs of one layout as one launch. 128-wide tiles where they give every CU one.
hipError_t launch_jobs(GenericJobs& jobs, bool pt, bool qt, bool q8, hipStream_t st) {
  if (jobs.n == 0) return hipSuccess;
  int64_t big = 0;
  bool is_short = false;
  for (int i = 0; i < jobs.n; ++i) {
    const GenericJob& j = jobs.job[i];
    big += ((j.I + 127) / 128) * ((j.J + 127) / 128);
    const int64_t k = j.K2 > 0 && (j.K == 0 || j.K2 < j.K) ? j.K2 : j.K;
    is_short |= (pt ? j.I : k) < 8 || (qt ? j.J : k) < 8;
  }
  if (is_short)
    return big >= 256 ? launch_tiles<128, 64, true>(jobs, pt, qt, q8, st)
                      : launch_tiles<64, 128, true>(jobs, pt, qt, q8, st);
  return big >= 256 ? launch_tiles<128, 64, false>(jobs, pt, qt, q8, st)
                    : launch_tiles<64, 128, false>(jobs, pt, qt, q8, st);
}

GenericJob make_job(const void* p, int64_t ldp, const void* q, int64_t ldq, int64_t I, int64_t J, int64_t K,
                    float scale, void* c, int64_t ldc) {
  GenericJob j{};
  j.p = reinterpret_cast<const uint16_t*>(p); j.ldp = ldp;
  j.q = q; j.ldq = ldq;
  j.I = I; j.J = J; j.K = K;
  j.scale = scale;
  j.c = reinterpret_cast<uint16_t*>(c); j.ldc = ldc;
  return j;
}

hipError_t launch_one(const GenericJob& j, bool pt, bool qt, bool q8, hipStream_t st) {
  GenericJobs jobs{};
  jobs.job[0] = j;
  jobs.n = 1;
  return launch_jobs(jobs, pt, qt, q8, st);
}

}  // namespace

hipError_t launch_generic(const LoraArgs& p) {
  uint16_t* t = reinterpret_cast<uint16_t*>(p.ws);
  if (p.r > 0) {
    const hipError_t e = launch_one(make_job(p.x, p.ldx, p.a, p.lda, p.M, p.r, p.K, p.scale, t, p.r), false, false,
                                    false, p.stream);
    if (e != hipSuccess) return e;
  }
  GenericJob j = make_job(p.x, p.ldx, p.w, p.ldw, p.M, p.N, p.w != nullptr ? p.K : 0, 1.f, p.y, p.ldy);
  if (p.gather != nullptr && p.gather_rows < 1) j.K = 0;  // an empty table: every row reads as zeros
  j.gather = p.gather;
  j.gather_rows = p.gather_rows;
  j.cscale = p.w != nullptr ? p.w_scale : nullptr;
  j.qmap = p.wmap;
  j.p2 = t; j.ldp2 = p.r;
  j.q2 = reinterpret_cast<const uint16_t*>(p.b); j.ldq2 = p.ldb;
  j.K2 = p.r;
  return launch_one(j, false, false, p.w != nullptr && p.w_dtype == kFP8, p.stream);
}

// T = bf16(s x . A^T) and U = bf16(s gy . B) into `t` [M, r] and `u` [M, r], then dW = gy^T . x,
// dB = gy^T . T and dA = U^T . x over the tokens in one launch (null outputs left out).
hipError_t launch_weight_grads_generic(const LoraArgs& p, const void* gy, int64_t ldg, void* dw, int64_t lddw,
                                       void* da, int64_t ldda, void* db, int64_t lddb, int64_t r, uint16_t* t,
                                       uint16_t* u) {
  hipError_t e = hipSuccess;
  GenericJobs jobs{};
  if (dw != nullptr) jobs.job[jobs.n++] = make_job(gy, ldg, p.x, p.ldx, p.N, p.K, p.M, 1.f, dw, lddw);
  if (db != nullptr) {
    e = launch_one(make_job(p.x, p.ldx, p.a, p.lda, p.M, r, p.K, p.scale, t, r), false, false, false, p.stream);
    if (e != hipSuccess) return e;
    jobs.job[jobs.n++] = make_job(gy, ldg, t, r, p.N, r, p.M, 1.f, db, lddb);
  }
  if (da != nullptr) {
    e = launch_one(make_job(gy, ldg, p.b, p.ldb, p.M, r, p.N, p.scale, u, r), false, true, false, p.stream);
    if (e != hipSuccess) return e;
    jobs.job[jobs.n++] = make_job(u, r, p.x, p.ldx, r, p.K, p.M, 1.f, da, ldda);
  }
  return launch_jobs(jobs, true, true, false, p.stream);
}

namespace {
// SPREAD: rank q of a group's rp takes row q % r of A, and the copies of one rank share its column
// of B in powers of two that sum to one (1; 1/2, 1/2; 1/2, 1/4, 1/4; ..). Zeros instead would make
// T's padding Inf . 0 = NaN in a row of x that holds an infinity, and with it the whole row of y;
// a copy's product with its share has the sign of the rank it copies, so y keeps its infinities.
template <bool SPREAD>
__global__ void __launch_bounds__(256) pad_rank_kernel(const uint16_t* __restrict__ a, int64_t lda,
                                                      const uint16_t* __restrict__ b, int64_t ldb, int64_t na,
                                                      int64_t nb, int64_t r, int64_t rp, int64_t K,
                                                      uint16_t* __restrict__ a_out, uint16_t* __restrict__ b_out) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e < na) {
    const int64_t row = e / K, k = e % K, j = row % rp;
    a_out[e] = SPREAD || j < r ? a[(row / rp * r + j % r) * lda + k] : 0;
  } else if (e - na < nb) {
    const int64_t n = (e - na) / rp, q = (e - na) % rp, j = q % r;
    if (SPREAD) {
      const int copy = (int)(q / r), last = (int)(rp / r) - (j < rp % r ? 0 : 1);
      b_out[e - na] = f32_to_bf16_bits(ldexpf(bf16_bits_to_f32(b[n * ldb + j]), -min(copy + 1, last)));
    } else {
      b_out[e - na] = q < r ? b[n * ldb + j] : 0;
    }
  }
}
}  // namespace

hipError_t launch_pad_rank(const void* a, int64_t lda, const void* b, int64_t ldb, int groups, int64_t r, int64_t rp,
                           int64_t K, int64_t N, void* a_out, void* b_out, bool spread, hipStream_t st) {
  const int64_t na = groups * rp * K, nb = N * rp, blocks = (na + nb + 255) / 256;
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  const auto kernel = spread ? pad_rank_kernel<true> : pad_rank_kernel<false>;
  kernel<<<dim3((unsigned)blocks), dim3(256), 0, st>>>(
      reinterpret_cast<const uint16_t*>(a), lda, reinterpret_cast<const uint16_t*>(b), ldb, na, nb, r, rp, K,
      reinterpret_cast<uint16_t*>(a_out), reinterpret_cast<uint16_t*>(b_out));
  return hipGetLastError();
}

// dX = gy . W + U . A with U = bf16(s gy . B) into `u` [M, r]: W [N, K] and A [r, K] as they lie,
// their rows the reduction (p as launch_bwd_input takes it).
hipError_t launch_bwd_input_generic(const LoraArgs& p, uint16_t* u) {
  if (p.r > 0) {
    const hipError_t e = launch_one(make_job(p.x, p.ldx, p.b, p.ldb, p.M, p.r, p.N, p.scale, u, p.r), false, true,
                                    false, p.stream);
    if (e != hipSuccess) return e;
  }
  GenericJob j = make_job(p.x, p.ldx, p.w, p.ldw, p.M, p.K, p.N, 1.f, p.y, p.ldy);
  j.p2 = u; j.ldp2 = p.r;
  j.q2 = reinterpret_cast<const uint16_t*>(p.a); j.ldq2 = p.lda;
  j.K2 = p.r;
  return launch_one(j, false, true, false, p.stream);
}

}  // namespace wsl
