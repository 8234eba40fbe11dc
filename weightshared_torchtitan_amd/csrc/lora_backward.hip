// Weight gradients of the fused LoRA linear (y = x . W^T + s (x . A^T) . B^T) on gfx950:
//
//   dW = gy^T . x            [N, K]
//   dA = s (gy . B)^T . x    [r, K]
//   dB = s gy^T . (x . A^T)  [N, r]
//
// dW reduces over the M tokens of two operands that store tokens as rows. The fused kernel's
// tile loop takes them in that form (TN: the tiles go into LDS as they lie and each MFMA
// fragment is read with gfx950's transposing LDS reads), so neither operand is copied. An
// output too small to fill the 256 CUs splits the token reduction into equal parts (fp32
// partials) that a reduce kernel sums in split order (deterministic), rounding once to bf16.
//
// With dW at hand, dA and dB follow from it by associativity, as products over K or N
// instead of over the tokens:
//
//   dB = s (gy^T . x) . A^T = s dW . A^T        dA = s B^T . (gy^T . x) = s B^T . dW
//
// 2 N K r multiply-adds each instead of 2 M r (N + K) for the rank projections T = x . A^T,
// U = gy . B and their products: both read the bf16 dW (dA through its transpose) and
// nothing of size M. Without dW (a frozen base) they take the token route instead:
// T = bf16(s x . A^T) and U = bf16(s gy . B) from the forward's rank pre-pass, then
// dB = gy^T . T and dA = U^T . x as token-major products.
//
// The reference has no backward of its own: torch autograd differentiates LoRAModule.forward
// (torchtitan/models/llama3/model/model.py:189-192) and the base nn.Linear (:257-273)
// composed by broadcast_add (:392-398); the trainer runs it at torchtitan/train.py:456.
#include <algorithm>

#include "wsl_common.h"

namespace wsl {

namespace {

constexpr int TT = 64;       // transpose tile: 64 rows x 64 columns
constexpr int TS = TT + 2;   // its LDS row stride in bf16 (odd word count: spread banks)

// dst[c][i] = src[i][c] for i < R and 0 for R <= i < Rp, c < C (B^T and dW^T here, Rp = R).
// 16-byte global accesses both ways (C % 8 == 0, Rp % 8 == 0, 16-byte aligned rows).
struct TransposeJob {
  const uint16_t* src;
  int64_t lds_, R, C;
  uint16_t* dst;
  int64_t ldd, Rp;
};

// The 64 x 64 tile (bx, by) of one job, staged through `tile`.
__device__ __forceinline__ void transpose_tile(const TransposeJob& j, int64_t bx, int64_t by, uint32_t* tile) {
  const uint16_t* __restrict__ src = j.src;
  uint16_t* __restrict__ dst = j.dst;
  const int64_t lds_ = j.lds_, R = j.R, C = j.C, ldd = j.ldd, Rp = j.Rp;
  const uint16_t* t16 = reinterpret_cast<const uint16_t*>(tile);
  const int64_t r0 = by * TT, c0 = bx * TT;
  const int tid = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int idx = tid + 256 * i, row = idx >> 3, ch = idx & 7;
    const int64_t r = r0 + row, c = c0 + ch * 8;
    u32x4_t v = u32x4_t{0u, 0u, 0u, 0u};
    if (r < R && c < C) v = *reinterpret_cast<const u32x4_t*>(src + r * lds_ + c);
    uint32_t* d = tile + (row * TS + ch * 8) / 2;  // TS even, ch * 8 even: word aligned
    d[0] = v[0]; d[1] = v[1]; d[2] = v[2]; d[3] = v[3];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int idx = tid + 256 * i, q = idx & 7, c = idx >> 3;  // 8 lanes: one 128-byte output row piece
    if (c0 + c >= C || r0 + q * 8 >= Rp) continue;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      w[j] = (uint32_t)t16[(q * 8 + 2 * j) * TS + c] | ((uint32_t)t16[(q * 8 + 2 * j + 1) * TS + c] << 16);
    *reinterpret_cast<u32x4_t*>(dst + (c0 + c) * ldd + r0 + q * 8) = u32x4_t{w[0], w[1], w[2], w[3]};
  }
}

__global__ void __launch_bounds__(256) transpose_pad_kernel(const TransposeJob j) {
  __shared__ uint32_t tile[TT * TS / 2];
  transpose_tile(j, blockIdx.x, blockIdx.y, tile);
}

// Two jobs in one launch (blockIdx.z picks the job; tiles past a job's extent exit).
__global__ void __launch_bounds__(256) transpose_pair_kernel(const TransposeJob j0, const TransposeJob j1) {
  __shared__ uint32_t tile[TT * TS / 2];
  const TransposeJob& j = blockIdx.z == 0 ? j0 : j1;
  if ((int64_t)blockIdx.x * TT >= j.C || (int64_t)blockIdx.y * TT >= j.Rp) return;
  transpose_tile(j, blockIdx.x, blockIdx.y, tile);
}

// Four bf16 of row-major `d` (8-byte pieces when `vec`).
__device__ __forceinline__ void store4(uint16_t* d, f32x4_t v, bool vec) {
  if (vec) {
    *reinterpret_cast<uint2*>(d) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
  } else {
    d[0] = f32_to_bf16_bits(v[0]); d[1] = f32_to_bf16_bits(v[1]);
    d[2] = f32_to_bf16_bits(v[2]); d[3] = f32_to_bf16_bits(v[3]);
  }
}

// sum over q of p[q * slice .. + 4) in split order, four loads in flight at a time (16-byte
// aligned p, slice % 4 == 0).
__device__ __forceinline__ f32x4_t sum_splits(const float* p, int64_t slice, int splits) {
  const f32x4_t* pv = reinterpret_cast<const f32x4_t*>(p);
  const int64_t sv = slice / 4;
  f32x4_t a = pv[0];
  int q = 1;
  for (; q + 4 <= splits; q += 4) {
    const f32x4_t a0 = pv[q * sv], a1 = pv[(q + 1) * sv], a2 = pv[(q + 2) * sv], a3 = pv[(q + 3) * sv];
    a += a0; a += a1; a += a2; a += a3;
  }
  for (; q < splits; ++q) a += pv[q * sv];
  return a;
}

// dst = bf16(scale * sum over the splits of part[s]) for an fp32 [splits][rows][cols] partial
// product, splits in order; four consecutive columns per thread (cols % 4 == 0).
__global__ void __launch_bounds__(256) split_sum_kernel(const float* __restrict__ part, int splits, int64_t rows,
                                                       int64_t cols, float scale, uint16_t* __restrict__ dst,
                                                       int64_t ldd, int vec) {
  const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  const int64_t slice = rows * cols;
  if (e >= slice) return;
  store4(dst + (e / cols) * ldd + e % cols, sum_splits(part + e, slice, splits) * scale, vec != 0);
}

// dW = bf16(sum over the splits of part[s]) ([splits][N][K] fp32, splits in order) to the
// caller's dw (row stride lddw, 8-byte pieces when `vec`), to the contiguous copy dwc
// [N][K] when given, and transposed to dwt [K][N] when given. 64 x 64 tiles (N % 64 ==
// K % 64 == 0); the transpose goes through LDS as in transpose_pad_kernel.
__global__ void __launch_bounds__(256) dw_reduce_kernel(const float* __restrict__ part, int splits, int64_t N,
                                                       int64_t K, uint16_t* __restrict__ dw, int64_t lddw, int vec,
                                                       uint16_t* __restrict__ dwc, uint16_t* __restrict__ dwt) {
  __shared__ uint32_t tile[TT * TS / 2];
  const uint16_t* t16 = reinterpret_cast<const uint16_t*>(tile);
  const int64_t n0 = (int64_t)blockIdx.y * TT, k0 = (int64_t)blockIdx.x * TT;
  const int tid = threadIdx.x;
  const int64_t slice = N * K;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = tid / 16 + 16 * i, col = (tid % 16) * 4;
    const int64_t e = (n0 + row) * K + k0 + col;
    const f32x4_t v = sum_splits(part + e, slice, splits);
    store4(dw + (n0 + row) * lddw + k0 + col, v, vec != 0);
    const uint32_t lo = pack_bf16x2(v[0], v[1]), hi = pack_bf16x2(v[2], v[3]);
    if (dwc != nullptr) *reinterpret_cast<uint2*>(dwc + e) = uint2{lo, hi};
    uint32_t* d = tile + (row * TS + col) / 2;
    d[0] = lo; d[1] = hi;
  }
  if (dwt == nullptr) return;  // uniform over the workgroup
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int idx = tid + 256 * i, q = idx & 7, c = idx >> 3;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      w[j] = (uint32_t)t16[(q * 8 + 2 * j) * TS + c] | ((uint32_t)t16[(q * 8 + 2 * j + 1) * TS + c] << 16);
    *reinterpret_cast<u32x4_t*>(dwt + (k0 + c) * N + n0 + q * 8) = u32x4_t{w[0], w[1], w[2], w[3]};
  }
}

hipError_t transpose_pad(const void* src, int64_t lds_, int64_t R, int64_t C, uint16_t* dst, int64_t ldd,
                         int64_t Rp, hipStream_t st) {
  if (C == 0 || Rp == 0) return hipSuccess;
  const dim3 grid((unsigned)((C + TT - 1) / TT), (unsigned)((Rp + TT - 1) / TT));
  transpose_pad_kernel<<<grid, dim3(256), 0, st>>>(TransposeJob{reinterpret_cast<const uint16_t*>(src), lds_, R, C,
                                                                dst, ldd, Rp});
  return hipGetLastError();
}

// Both transposes of the input gradient's rank factors in one launch.
hipError_t transpose_pair(const TransposeJob& j0, const TransposeJob& j1, hipStream_t st) {
  const int64_t gx = std::max((j0.C + TT - 1) / TT, (j1.C + TT - 1) / TT);
  const int64_t gy = std::max((j0.Rp + TT - 1) / TT, (j1.Rp + TT - 1) / TT);
  transpose_pair_kernel<<<dim3((unsigned)gx, (unsigned)gy, 2), dim3(256), 0, st>>>(j0, j1);
  return hipGetLastError();
}

size_t a256(size_t v) { return (v + 255) & ~(size_t)255; }
bool al16(const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15u) == 0; }

// Workspace plan. It depends on the sizes only, so the workspace query needs no flags: the
// union of both routes' buffers.
struct Plan {
  int sw;          // token splits of the dW product
  bool sw_big;     // dW over 256 x 256 tiles
  int sb, sa;      // token route: token splits of the dB and dA products
  int sdb, sda;    // dW route: splits of dB = s dW . A^T (over K) and dA = s B^T . dW (over N)
  size_t off_t, off_u, off_bt, off_dwc, off_dwt, off_part, total;
};

Plan make_plan(int64_t M, int64_t N, int64_t K, int64_t r) {
  Plan L{};
  const int64_t nk = (M + 63) / 64;
  const TnSplit tw = product_tn_splits(N, K, nk);
  L.sw = tw.splits;
  L.sw_big = tw.big;
  L.sb = r > 0 ? product_splits(N, r, nk, false) : 1;
  L.sa = r > 0 ? product_splits(r, K, nk, false) : 1;
  L.sdb = r > 0 ? product_splits(N, r, K / 64, true) : 1;
  L.sda = r > 0 ? product_splits(r, K, N / 64, true) : 1;
  size_t off = 0;
  L.off_t = off;   off = a256(off + (r > 0 ? rank_prepass_bytes(M, K, r) : 0));
  L.off_u = off;   off = a256(off + (r > 0 ? rank_prepass_bytes(M, N, r) : 0));
  L.off_bt = off;  off = a256(off + (size_t)r * N * 2);
  L.off_dwc = off; off = a256(off + (r > 0 ? (size_t)N * K * 2 : 0));
  L.off_dwt = off; off = a256(off + (r > 0 ? (size_t)N * K * 2 : 0));
  L.off_part = off;
  size_t part = (size_t)L.sw * N * K;  // worst case: any product may go through partials
  const size_t cand[4] = {(size_t)L.sb * N * r, (size_t)L.sa * r * K, (size_t)L.sdb * N * r, (size_t)L.sda * r * K};
  for (size_t c : cand) part = c > part ? c : part;
  L.total = a256(off + part * 4);
  return L;
}

}  // namespace

// Shapes and layouts the tile kernels of the weight-gradient path take: K and N on the
// 64-element tile grid (the reductions of the dA and dB products and of the token route's
// pre-passes), ranks in multiples of 8, 16-byte aligned rows, and sizes within the tile
// kernel's int range. Every other layout takes the token route on the generic products
// (csrc/lora_generic.hip).
bool weight_grads_supported(const LoraArgs& p, const void* gy, int64_t ldg) {
  if (p.M < 1 || p.K % 64 != 0 || p.N % 64 != 0 || p.r % 8 != 0) return false;
  if (p.M > ((int64_t)1 << 22) - 2048 || p.N > ((int64_t)1 << 22) || p.K > ((int64_t)1 << 22)) return false;
  if (!al16(p.x) || p.ldx % 8 != 0 || !al16(gy) || ldg % 8 != 0) return false;
  if (p.ldx > ((int64_t)1 << 22) || ldg > ((int64_t)1 << 22)) return false;
  if (p.r > 0 && (!al16(p.a) || p.lda % 8 != 0 || !al16(p.b) || p.ldb % 8 != 0 || p.lda > ((int64_t)1 << 22)))
    return false;
  return true;
}

size_t weight_grads_workspace_bytes(int64_t M, int64_t N, int64_t K, int64_t r, bool need_w, bool need_ab) {
  (void)need_w;
  return make_plan(M, N, K, need_ab ? r : 0).total;
}

// ---- Input gradient: dX = dY . W + s (dY . B) . A, W read where it lies ----
// The forward-shaped problem of dX (x' = dY, reduction K' = N, N' = K output columns) runs
// on the prefill kernel's WT form: W's rows are the reduction, so its tiles go into LDS as
// they lie and its fragments are transposing reads; no copy of W. The rank factors take the
// places of the forward's: A' = B^T [r, N] and B' = A^T [K, r], transposed into the
// workspace after the prefill scratch (r (N + K) bf16).
namespace {
LoraArgs wt_problem(const LoraArgs& p) {
  LoraArgs q = p;
  q.K = p.N;
  q.N = p.K;
  return q;
}
size_t a256b(size_t v) { return (v + 255) & ~(size_t)255; }
}  // namespace

bool bwd_input_supported(const LoraArgs& p) {
  if (p.r > 0 && (p.N % 8 != 0 || p.K % 8 != 0 || !al16(p.a) || p.lda % 8 != 0 || !al16(p.b) || p.ldb % 8 != 0))
    return false;
  LoraArgs q = wt_problem(p);
  // the transposed factors stand in for a and b (aligned, tight leading dimensions)
  static char kAligned[16] __attribute__((aligned(16))) = {0};
  q.a = p.r > 0 ? kAligned : nullptr;
  q.lda = p.N;
  q.b = p.r > 0 ? kAligned : nullptr;
  q.ldb = p.r;
  return prefill_wt_supported(q);
}

size_t bwd_input_workspace_bytes(int64_t M, int64_t N, int64_t K, int64_t r) {
  return a256b(prefill_workspace_bytes(M, K, N, r, kBF16)) + a256b((size_t)r * N * 2) + (size_t)K * r * 2;
}

hipError_t launch_bwd_input(const LoraArgs& p) {
  LoraArgs q = wt_problem(p);
  hipError_t e = hipSuccess;
  if (p.r > 0) {
    char* base = reinterpret_cast<char*>(p.ws) + a256b(prefill_workspace_bytes(p.M, p.K, p.N, p.r, kBF16));
    uint16_t* bt = reinterpret_cast<uint16_t*>(base);
    uint16_t* at = reinterpret_cast<uint16_t*>(base + a256b((size_t)p.r * p.N * 2));
    // B [N, r] -> B^T [r, N] and A [r, K] -> A^T [K, r], one launch
    e = transpose_pair(TransposeJob{reinterpret_cast<const uint16_t*>(p.b), p.ldb, p.N, p.r, bt, p.N, p.N},
                       TransposeJob{reinterpret_cast<const uint16_t*>(p.a), p.lda, p.r, p.K, at, p.r, p.r}, p.stream);
    q.a = bt;
    q.lda = p.N;
    q.b = at;
    q.ldb = p.r;
  }
  if (e == hipSuccess) e = launch_prefill_wt(q);
  return e;
}

hipError_t launch_weight_grads(const LoraArgs& p, const void* gy, int64_t ldg, void* dw, int64_t lddw, void* da,
                               int64_t ldda, void* db, int64_t lddb) {
  const int64_t M = p.M, N = p.N, K = p.K;
  const int64_t r = (da != nullptr || db != nullptr) ? p.r : 0;
  if (r == 0) da = db = nullptr;
  if (dw == nullptr && r == 0) return hipSuccess;
  const Plan L = make_plan(M, N, K, r);
  char* ws = reinterpret_cast<char*>(p.ws);
  uint16_t* T = reinterpret_cast<uint16_t*>(ws + L.off_t);
  uint16_t* U = reinterpret_cast<uint16_t*>(ws + L.off_u);
  if (!weight_grads_supported(p, gy, ldg))
    return launch_weight_grads_generic(p, gy, ldg, dw, lddw, da, ldda, db, lddb, r, T, U);
  uint16_t* Bt = reinterpret_cast<uint16_t*>(ws + L.off_bt);
  uint16_t* dwc = reinterpret_cast<uint16_t*>(ws + L.off_dwc);
  uint16_t* dwt = reinterpret_cast<uint16_t*>(ws + L.off_dwt);
  float* part = reinterpret_cast<float*>(ws + L.off_part);
  const hipStream_t st = p.stream;
  const int64_t nkt = (M + 63) / 64;  // 64-token K tiles
  hipError_t e = hipSuccess;

  auto vec_ok = [](const void* dst, int64_t ldd) { return (reinterpret_cast<uintptr_t>(dst) & 7u) == 0 && ldd % 4 == 0; };
  // dst = bf16(scale * sum_s part[s]) [rows, cols] from the partial products
  auto reduce = [&](int splits, int64_t rows, int64_t cols, float scale, void* dst, int64_t ldd, bool vec) {
    const int64_t n4 = rows * cols / 4;
    split_sum_kernel<<<dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, st>>>(
        part, splits, rows, cols, scale, reinterpret_cast<uint16_t*>(dst), ldd, vec ? 1 : 0);
    return hipGetLastError();
  };
  // y' = scale * x' . W'^T, x' and W' rows `red` long: straight to bf16 when unsplit and the
  // destination takes the tile store's 8-byte pieces, else through fp32 partials
  auto product = [&](const void* xa, int64_t ldxa, int64_t rows, const void* wb, int64_t ldwb, int64_t cols,
                     int64_t red, int splits, float scale, void* dst, int64_t ldd) -> hipError_t {
    LoraArgs q = p;
    q.x = xa; q.ldx = ldxa; q.w = wb; q.ldw = ldwb; q.M = rows; q.N = cols; q.yscale = scale;
    const bool vec = vec_ok(dst, ldd);
    if (splits == 1 && vec) {
      q.K = red; q.y = dst; q.ldy = ldd;
      return launch_product(q, nullptr, 1);
    }
    q.K = red / splits;
    const hipError_t err = launch_product(q, part, splits);
    return err != hipSuccess ? err : reduce(splits, rows, cols, scale, dst, ldd, vec);
  };
  // Token splits as launched: equal whole 64-token tiles, none starting past the tokens.
  auto tn_splits = [&](int splits, int64_t* per) {
    const int64_t kt = (nkt + splits - 1) / splits;
    *per = kt * 64;
    return (int)((nkt + kt - 1) / kt);
  };
  // the same over the tokens with token-major operands: x'[m][t] = xa[t * ldxa + m],
  // W'[n][t] = wb[t * ldwb + n]
  auto product_tn = [&](const void* xa, int64_t ldxa, int64_t rows, const void* wb, int64_t ldwb, int64_t cols,
                        int splits, float scale, void* dst, int64_t ldd) -> hipError_t {
    LoraArgs q = p;
    q.x = xa; q.ldx = ldxa; q.w = wb; q.ldw = ldwb; q.M = rows; q.N = cols; q.yscale = scale;
    const int s = tn_splits(splits, &q.K);
    const bool vec = vec_ok(dst, ldd);
    if (s == 1 && vec) {
      q.y = dst; q.ldy = ldd;
      return launch_product_tn(q, M, nullptr, 1);
    }
    const hipError_t err = launch_product_tn(q, M, part, s);
    return err != hipSuccess ? err : reduce(s, rows, cols, scale, dst, ldd, vec);
  };

  if (dw != nullptr) {
    // ---- dW route: dW over the tokens, then dB = s dW . A^T and dA = s B^T . dW ----
    int64_t per = 0;
    const int sw = tn_splits(L.sw, &per);
    const bool direct = sw == 1 && al16(dw) && lddw % 8 == 0;
    const uint16_t* dws = reinterpret_cast<const uint16_t*>(dw);  // bf16 dW rows for dB
    int64_t ldws = lddw;
    if (direct) {
      e = product_tn(gy, ldg, N, p.x, p.ldx, K, 1, 1.f, dw, lddw);
      if (e == hipSuccess && da != nullptr) e = transpose_pad(dw, lddw, N, K, dwt, N, N, st);
    } else {
      LoraArgs q = p;
      q.x = gy; q.ldx = ldg; q.w = p.x; q.ldw = p.ldx; q.M = N; q.N = K; q.K = per;
      e = launch_product_tn(q, M, part, sw, L.sw_big);
      if (e == hipSuccess) {
        dw_reduce_kernel<<<dim3((unsigned)(K / TT), (unsigned)(N / TT)), dim3(256), 0, st>>>(
            part, sw, N, K, reinterpret_cast<uint16_t*>(dw), lddw, vec_ok(dw, lddw) ? 1 : 0,
            db != nullptr ? dwc : nullptr, da != nullptr ? dwt : nullptr);
        e = hipGetLastError();
      }
      dws = dwc;
      ldws = K;
    }
    if (e == hipSuccess && db != nullptr) e = product(dws, ldws, N, p.a, p.lda, r, K, L.sdb, p.scale, db, lddb);
    if (e == hipSuccess && da != nullptr) {
      e = transpose_pad(p.b, p.ldb, N, r, Bt, N, N, st);
      if (e == hipSuccess) e = product(Bt, N, r, dwt, N, K, N, L.sda, p.scale, da, ldda);
    }
    return e;
  }

  // ---- token route (no dW): T, U by the rank pre-pass, token-major products ----
  if (db != nullptr) {  // dB = gy^T . T, T = bf16(s x . A^T)
    LoraArgs q = p;
    q.groups = 1;
    e = rank_prepass(q, T);
    if (e == hipSuccess) e = product_tn(gy, ldg, N, T, r, r, L.sb, 1.f, db, lddb);
    if (e != hipSuccess) return e;
  }
  if (da != nullptr) {  // dA = U^T . x, U = bf16(s gy . B) with B^T [r, N] in the place of A
    e = transpose_pad(p.b, p.ldb, N, r, Bt, N, N, st);
    if (e != hipSuccess) return e;
    LoraArgs q = p;
    q.x = gy; q.ldx = ldg; q.K = N; q.a = Bt; q.lda = N; q.groups = 1;
    e = rank_prepass(q, U);
    if (e == hipSuccess) e = product_tn(U, r, r, p.x, p.ldx, K, L.sa, 1.f, da, ldda);
  }
  return e;
}

// ---- Shared-base backward ----
// One base W [base_n, K] under `groups` projections of N columns, output column c of each on base
// row c' = map_row(c) (RowMap). With gy_b [M, base_n] the sums of gy's columns by base row and Bd
// the block-diagonal [G N, G r] form of B,
//
//   dX = gy_b . W + U . A      U = bf16(s gy . Bd)     dW = gy_b^T . x
//   dA = U^T . x               dB_j = gy_j^T . T_j     T = bf16(s x . A^T)
//
// U is computed once for dX and dA. Kernels of this part: the column sums (one read of gy), and the
// factors in the layouts that the products take (Bd^T and A^T, one launch); dB's diagonal blocks
// are picked out as the token splits of the [G N, G r] product are summed. As torch operators
// (casts, a 5-d sum, block copies, transposes, a separate delta product and its addition) this
// work was 22 launches and 125 of 307 us of the backward at M = 4096, q|k|v on 2048 x 2048, r = 32;
// forward and backward there 433 -> 305 us (dX's delta joins its base product's accumulators, so
// dX is rounded once, not three times), 436 -> 107 us on small sizes, which the launches bounded.
namespace {
// gyb[m][n] = bf16(sum of gy[m][c] over the columns c of every group whose base row is n), groups
// then heads in order; eight consecutive base rows per thread (the template width D is a multiple
// of 8, so they are consecutive columns in every head). Bound by reading gy.
__global__ void __launch_bounds__(256) fold_columns_kernel(const uint16_t* __restrict__ gy, int64_t ldg, int64_t M,
                                                          int base_n, int N, int groups, RowMap wmap,
                                                          uint16_t* __restrict__ gyb) {
  const int per = base_n / 8;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t m = idx / per;
  if (m >= M) return;
  const int n = (int)(idx % per) * 8;
  // base row n of template n / D is column (n / D) S + h D + n % D of head h, h < S / D
  const int c0 = n / wmap.D * wmap.S + n % wmap.D, heads = wmap.S / wmap.D;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int j = 0; j < groups; ++j)
    for (int h = 0; h < heads; ++h) {
      const u32x4_t v = ld_global_16(gy + m * ldg + (int64_t)j * N + c0 + h * wmap.D);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += bf16_bits_to_f32((v[e >> 1] >> ((e & 1) * 16)) & 0xffffu);
    }
  u32x4_t o;
#pragma unroll
  for (int q = 0; q < 4; ++q) o[q] = pack_bf16x2(acc[2 * q], acc[2 * q + 1]);
  *reinterpret_cast<u32x4_t*>(gyb + m * base_n + n) = o;
}

// bt [G r, G N] = Bd^T (zeros off the diagonal blocks) and at [K, G r] = A^T, one element a thread.
__global__ void __launch_bounds__(256) bcast_factors_kernel(const uint16_t* __restrict__ a, int64_t lda,
                                                           const uint16_t* __restrict__ b, int64_t ldb, int64_t K,
                                                           int64_t N, int64_t r, int groups,
                                                           uint16_t* __restrict__ bt, uint16_t* __restrict__ at) {
  const int64_t gr = groups * r, gn = groups * N, nb = gr * gn;
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e < nb) {
    const int64_t q = e / gn, c = e % gn;
    bt[e] = c / N == q / r ? b[c * ldb + q % r] : 0;
  } else if (e - nb < K * gr) {
    const int64_t k = (e - nb) / gr, q = (e - nb) % gr;
    at[e - nb] = a[q * lda + k];
  }
}

// db[c][q] = bf16(sum over the splits of part[s][c][(c / N) r + q]), splits in order: four
// consecutive ranks per thread.
__global__ void __launch_bounds__(256) diag_sum_kernel(const float* __restrict__ part, int splits, int64_t gn, int64_t N,
                                                      int64_t r, int64_t gr, uint16_t* __restrict__ db) {
  const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (e >= gn * r) return;
  const int64_t c = e / r, q = e % r;
  const f32x4_t v = sum_splits(part + c * gr + c / N * r + q, gn * gr, splits);
  *reinterpret_cast<uint2*>(db + e) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

struct BcastPlan {
  int sw, sb, sa;  // token splits of the dW, dB and dA products
  bool sw_big;     // dW's over 256 x 256 tiles
  size_t off_gyb, off_bt, off_at, off_u, off_t, off_part, total;
};
BcastPlan make_bcast_plan(int64_t M, int64_t N, int64_t K, int64_t r, int64_t base_n, int groups) {
  BcastPlan L{};
  const int64_t nk = (M + 63) / 64, gn = groups * N, gr = groups * r;
  const TnSplit tw = product_tn_splits(base_n, K, nk);
  L.sw = tw.splits;
  L.sw_big = tw.big;
  L.sb = r > 0 ? product_splits(gn, gr, nk, false) : 1;
  L.sa = r > 0 ? product_splits(gr, K, nk, false) : 1;
  size_t off = 0;
  L.off_gyb = off; off = a256(off + (size_t)M * base_n * 2);
  L.off_bt = off;  off = a256(off + (size_t)(gr * gn) * 2);
  L.off_at = off;  off = a256(off + (size_t)(K * gr) * 2);
  L.off_u = off;   off = a256(off + (r > 0 ? rank_prepass_bytes(M, gn, gr) : 0));
  L.off_t = off;   off = a256(off + (r > 0 ? rank_prepass_bytes(M, K, gr) : 0));
  L.off_part = off;
  size_t part = (size_t)L.sw * base_n * K;
  part = std::max({part, (size_t)(L.sb * gn * gr), (size_t)(L.sa * gr * K)});
  L.total = a256(off + part * 4);
  return L;
}
}  // namespace

bool bcast_bwd_supported(const LoraArgs& p, const void* gy, int64_t ldg) {
  const int64_t gn = p.groups * p.N, gr = p.groups * p.r, base_n = p.wrows, lim = (int64_t)1 << 22;
  if (p.M < 1 || p.M > lim - 2048 || gn > lim || p.K > lim || p.ldx > lim || ldg > lim || p.ldw > lim || p.lda > lim)
    return false;
  if (p.K % 64 != 0 || gn % 64 != 0 || base_n % 64 != 0 || p.wmap.D % 8 != 0 || p.r % 8 != 0 || gr > WSL_MAX_RANK)
    return false;
  if (p.w == nullptr || p.w_dtype != kBF16 || !al16(p.w) || p.ldw % 8 != 0) return false;
  if (!al16(p.x) || p.ldx % 8 != 0 || !al16(gy) || ldg % 8 != 0) return false;
  if (p.r > 0 && (!al16(p.a) || p.lda % 8 != 0)) return false;  // b goes through its rearranged copy
  return p.M * base_n / 8 / 256 < 0x7fffffff;
}

size_t bcast_bwd_workspace_bytes(int64_t M, int64_t N, int64_t K, int64_t r, int64_t base_n, int groups) {
  return make_bcast_plan(M, N, K, r, base_n, groups).total;
}

hipError_t launch_bcast_bwd(const LoraArgs& p, const void* gy, int64_t ldg, void* dx, void* dw, void* da, void* db) {
  const int64_t M = p.M, K = p.K, N = p.N, r = p.r, base_n = p.wrows;
  const int64_t gn = p.groups * N, gr = p.groups * r;
  const hipStream_t st = p.stream;
  const BcastPlan L = make_bcast_plan(M, N, K, r, base_n, p.groups);
  char* ws = reinterpret_cast<char*>(p.ws);
  uint16_t* gyb = reinterpret_cast<uint16_t*>(ws + L.off_gyb);
  uint16_t* bt = reinterpret_cast<uint16_t*>(ws + L.off_bt);
  uint16_t* at = reinterpret_cast<uint16_t*>(ws + L.off_at);
  uint16_t* U = reinterpret_cast<uint16_t*>(ws + L.off_u);
  uint16_t* T = reinterpret_cast<uint16_t*>(ws + L.off_t);
  float* part = reinterpret_cast<float*>(ws + L.off_part);
  const int64_t nkt = (M + 63) / 64;
  hipError_t e = hipSuccess;
  LoraArgs base = p;  // a plain problem of this stream; its operands are set per product
  base.groups = 1; base.wmap = RowMap{}; base.gather = nullptr; base.gather_rows = 0;

  // part[s] [rows, cols] = the token splits of xa^T . wb; how many there are
  auto token_product = [&](const void* xa, int64_t ldxa, int64_t rows, const void* wb, int64_t ldwb, int64_t cols,
                           int splits, bool big, int* used, void* direct) -> hipError_t {
    LoraArgs q = base;
    q.x = xa; q.ldx = ldxa; q.w = wb; q.ldw = ldwb; q.M = rows; q.N = cols; q.yscale = 1.f;
    const int64_t kt = (nkt + splits - 1) / splits;
    q.K = kt * 64;
    *used = (int)((nkt + kt - 1) / kt);
    if (direct != nullptr && *used == 1) {
      q.y = direct; q.ldy = cols;
      *used = 0;
      return launch_product_tn(q, M, nullptr, 1);
    }
    return launch_product_tn(q, M, part, *used, big);
  };
  auto sum_to = [&](int splits, int64_t rows, int64_t cols, void* dst) {
    const int64_t n4 = rows * cols / 4;
    split_sum_kernel<<<dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, st>>>(
        part, splits, rows, cols, 1.f, reinterpret_cast<uint16_t*>(dst), cols, 1);
    return hipGetLastError();
  };

  const void* gb = gy;  // gy by base row
  int64_t ldgb = ldg;
  if ((dx != nullptr || dw != nullptr) && !(p.groups == 1 && base_n == N)) {
    const int64_t blocks = (M * (base_n / 8) + 255) / 256;
    fold_columns_kernel<<<dim3((unsigned)blocks), dim3(256), 0, st>>>(reinterpret_cast<const uint16_t*>(gy), ldg, M,
                                                                     (int)base_n, (int)N, p.groups, p.wmap, gyb);
    e = hipGetLastError();
    gb = gyb;
    ldgb = base_n;
  }
  if (e == hipSuccess && r > 0 && (dx != nullptr || da != nullptr)) {
    const int64_t blocks = (gr * gn + K * gr + 255) / 256;
    bcast_factors_kernel<<<dim3((unsigned)blocks), dim3(256), 0, st>>>(
        reinterpret_cast<const uint16_t*>(p.a), p.lda, reinterpret_cast<const uint16_t*>(p.b), p.ldb, K, N, r,
        p.groups, bt, at);
    e = hipGetLastError();
    if (e == hipSuccess) {
      LoraArgs q = base;
      q.x = gy; q.ldx = ldg; q.K = gn; q.a = bt; q.lda = gn; q.r = gr;
      e = rank_prepass(q, U);
    }
  }
  if (e == hipSuccess && dx != nullptr) {
    LoraArgs q = base;
    q.x = gb; q.ldx = ldgb; q.K = base_n; q.N = K; q.wrows = 0;
    q.a = bt; q.lda = gn; q.b = at; q.ldb = gr; q.r = gr; q.y = dx; q.ldy = K;
    e = launch_prefill_wt(q, r > 0 ? U : nullptr, gr);
  }
  int s = 0;
  if (e == hipSuccess && dw != nullptr) {
    e = token_product(gb, ldgb, base_n, p.x, p.ldx, K, L.sw, L.sw_big, &s, dw);
    if (e == hipSuccess && s > 0) e = sum_to(s, base_n, K, dw);
  }
  if (e == hipSuccess && r > 0 && da != nullptr) {
    e = token_product(U, gr, gr, p.x, p.ldx, K, L.sa, false, &s, nullptr);
    if (e == hipSuccess) e = sum_to(s, gr, K, da);
  }
  if (e == hipSuccess && r > 0 && db != nullptr) {
    LoraArgs q = base;
    q.r = gr;
    e = rank_prepass(q, T);
    if (e == hipSuccess) e = token_product(gy, ldg, gn, T, gr, gr, L.sb, false, &s, nullptr);
    if (e == hipSuccess) {
      diag_sum_kernel<<<dim3((unsigned)((gn * r / 4 + 255) / 256)), dim3(256), 0, st>>>(
          part, s, gn, N, r, gr, reinterpret_cast<uint16_t*>(db));
      e = hipGetLastError();
    }
  }
  return e;
}

}  // namespace wsl
