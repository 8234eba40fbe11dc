// Prompt (prefill) kernels of the weight-shared Qwen3 harness for gfx950: the work between
// the fused LoRA projections of a whole-sequence forward from position 0.
//
//   kv_rope_kernel            per (token, kv head): k RMS-normed over head_dim and rotated, k and
//                             v written into the KV cache at the token's position.
//   prefill_attention_kernel  causal GQA attention over the cache's first `seq` positions, the
//                             q RMSNorm and RoPE applied as the query rows are loaded.
//
// Attention on the matrix cores. A workgroup of NW waves owns 32 query rows per wave: HPW heads
// of one kv head's group (their rows share every K/V tile) by 32 * NW / HPW positions. It walks
// the keys in tiles of 64 through two LDS buffers filled by global_load_lds_dwordx4, the next
// tile's fill in flight while this one is multiplied. Scores are computed transposed,
// S^T = K . Q^T (v_mfma_f32_32x32x16_bf16, K rows as the A operand), so a lane holds 32 of the
// tile's 64 scores of ONE query: the softmax state is two registers a lane, and its reductions
// are in-lane but for one exchange with the lane's other half. The output accumulates
// transposed too, O^T = V^T . P^T: the score registers, rounded to bf16, are the B operand as
// they lie (a reduction does not care in which order it meets the keys, so V^T takes the keys
// in the order the score layout has them), and V^T is read from the row-major V tile with
// gfx950's transposing LDS reads. Nothing moves between lanes but the two softmax reductions.
//
// Measured at 8 sequences of 512, 16 heads on 8 kv heads of 128 (per layer, rocprofv3 trace):
// attention 28.4 us (310 TFLOP/s of causal work) with the q norm and rotation in it, against 75.7
// for the flash kernel torch takes, on keys and values repeated per head by copies; k norm,
// rotation and cache write 10 us. Norms, rotations, repeats and copies as torch ops took 380 us.
// The attention is bound by its LDS reads (a wave reads every K and V tile for 32 rows, 128
// bytes a cycle and CU at full matrix rate) and by the softmax between the two products.
//
// Arithmetic is fp32 with one rounding to bf16 of the rotated q and k, of the probabilities
// and of the output, as flash attention over bf16 tensors has it. Reference semantics:
// torchtitan/experiments/qwen3/model/model.py:20-36,73-90 (RoPE), :167-218 (q/k norm, GQA).
#include "../../include/wsl_decode.h"
#include "wsl_common.h"

namespace wsl {
namespace {

__device__ __forceinline__ float bf(uint32_t h) { return bf16_bits_to_f32(h & 0xffffu); }
__device__ __forceinline__ float bf_at(const u32x4_t& v, int e) { return bf(v[e >> 1] >> ((e & 1) * 16)); }

// cos and sin of the 8 elements from j on; a row of the table is cos [HD] | sin [HD].
struct Rot8 {
  float c[8], s[8];
  __device__ __forceinline__ void load(const float* row, int hd, int j) {
    const float* r[2] = {row + j, row + hd + j};
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const f32x4_t cv = *reinterpret_cast<const f32x4_t*>(r[0] + 4 * q);
      const f32x4_t sv = *reinterpret_cast<const f32x4_t*>(r[1] + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        c[4 * q + e] = cv[e];
        s[4 * q + e] = sv[e];
      }
    }
  }
};

// ----------------------------------------------------------- k norm + RoPE + cache write
// HD / 8 lanes per (token, kv head) row, 8 elements a lane; the rotation partner of a lane's
// elements is HD / 16 lanes away. Bound by memory: k and v in, k and v out.
template <int HD>
__global__ void __launch_bounds__(256) kv_rope_kernel(const uint16_t* __restrict__ k, int64_t ldk,
                                                     const uint16_t* __restrict__ v, int64_t ldv, int seq, int nkv,
                                                     int64_t rows, const uint16_t* __restrict__ kw, float eps,
                                                     const float* __restrict__ rope, uint16_t* __restrict__ kc,
                                                     uint16_t* __restrict__ vc, int64_t cache_len) {
  constexpr int LPR = HD / 8;
  const int64_t row = (int64_t)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
  if (row >= rows) return;  // the LPR lanes of a row leave together
  const int l = threadIdx.x % LPR;
  const int64_t t = row / nkv;
  const int kh = (int)(row % nkv);
  const int64_t b = t / seq;
  const int pos = (int)(t % seq);
  const u32x4_t kv = ld_global_16(k + t * ldk + (int64_t)kh * HD + 8 * l);
  const u32x4_t vv = ld_global_16(v + t * ldv + (int64_t)kh * HD + 8 * l);
  const u32x4_t wv = ld_global_16(kw + 8 * l);
  Rot8 rot;
  rot.load(rope + (int64_t)pos * 2 * HD, HD, 8 * l);
  float x[8], ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    x[e] = bf_at(kv, e);
    ss += x[e] * x[e];
  }
#pragma unroll
  for (int o = LPR / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
  const float inv = rsqrtf(ss / (float)HD + eps);
  u32x4_t ov;
  float o8[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float n = x[e] * inv * bf_at(wv, e);
    const float partner = __shfl_xor(n, LPR / 2, 64);
    o8[e] = n * rot.c[e] + (l < LPR / 2 ? -partner : partner) * rot.s[e];
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) ov[q] = pack_bf16x2(o8[2 * q], o8[2 * q + 1]);
  const int64_t dst = ((b * nkv + kh) * cache_len + pos) * HD + 8 * l;
  *reinterpret_cast<u32x4_t*>(kc + dst) = ov;
  *reinterpret_cast<u32x4_t*>(vc + dst) = vv;
}

// ----------------------------------------------------------------------- attention
typedef __attribute__((address_space(3))) void lds_void_t;
typedef short v4i16_t __attribute__((ext_vector_type(4)));

constexpr int PA_KT = 64;  // keys per tile

// One wave instruction: lane i's 16 bytes at `src` land at the wave-uniform `dst` + 16 i.
__device__ __forceinline__ void fill16(const uint16_t* src, char* dst) {
  __builtin_amdgcn_global_load_lds(src, (lds_void_t*)dst, 16, 0, 0);
}
// Transposing LDS read: if lane j of a 16-lane group addresses row r0 + j / 4 at column
// f0 + 4 (j % 4) of a row-major bf16 matrix, lane i receives rows r0 .. r0 + 3 of column f0 + i.
__device__ __forceinline__ uint2 read_tr4(const char* p) {
  const v4i16_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4i16_t*)p);
  return uint2{(uint32_t)(uint16_t)v[0] | ((uint32_t)(uint16_t)v[1] << 16),
               (uint32_t)(uint16_t)v[2] | ((uint32_t)(uint16_t)v[3] << 16)};
}
__device__ __forceinline__ f32x16_t mfma16(u32x4_t a, u32x4_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}
__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }

// s_waitcnt vmcnt(N), N < 64, the other counters unconstrained
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
}
// Barrier between a tile's reads and the next fill of its buffer: this wave's LDS reads are
// done (lgkmcnt(0)), the fills in flight are not waited for.
__device__ __forceinline__ void tile_barrier() {
  __builtin_amdgcn_s_waitcnt(0xc07f);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Swizzles of the 16-byte chunks of a row. K rows are read 16 at a time at one chunk index:
// 16 rows must spread over the 16 bank groups. V rows are read 4 at a time, 4 chunks each.
template <int HD>
__device__ __forceinline__ int k_swz(int row) { return HD == 128 ? (row & 15) : ((row >> 1) & 7); }
template <int HD>
__device__ __forceinline__ int v_swz(int row) { return HD == 128 ? ((row & 3) << 2) : (((row >> 1) & 1) << 2); }

// out[b, pos, head] = softmax(q . K^T * scale over keys <= pos) . V. `log2s` = scale * log2(e).
// Grid: ceil(seq / QT) query tiles (the longest first) x batch * n_kv_heads * (rep / HPW).
template <int HD, int HPW, int NW>
__global__ void __launch_bounds__(NW * 64, NW / 2)
prefill_attention_kernel(const uint16_t* __restrict__ q, int64_t ldq, const uint16_t* __restrict__ qw, float eps,
                         const float* __restrict__ rope, const uint16_t* __restrict__ kc,
                         const uint16_t* __restrict__ vc, int64_t cache_len, int seq, int nh, int nkv, int groups,
                         float log2s, uint16_t* __restrict__ out, int64_t ldo) {
  constexpr int WPH = NW / HPW;        // waves per head
  constexpr int QT = 32 * WPH;         // positions per workgroup
  constexpr int ST = HD / 16;          // k steps of S
  constexpr int DB = HD / 32;          // 32-row blocks of O^T
  constexpr int RB = HD * 2;           // bytes of an LDS row
  constexpr int CPR = HD / 8;          // chunks per row
  constexpr int TB = PA_KT * RB;       // bytes of a K or V tile
  constexpr int RPI = 1024 / RB;       // rows per fill instruction
  constexpr int NF = TB / 1024 / NW;   // fill instructions of K (and of V) per wave and tile
  __shared__ __attribute__((aligned(1024))) char smem[4 * TB];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, h = lane >> 5;
  const int nqt = (seq + QT - 1) / QT;
  const int qt = nqt - 1 - (int)(blockIdx.x / (unsigned)groups);
  const int grp = (int)(blockIdx.x % (unsigned)groups);
  const int rep = nh / nkv, subs = rep / HPW;
  const int pair = grp / subs;         // batch * nkv + kv head
  const int b = pair / nkv, kvh = pair % nkv;
  const int head = kvh * rep + (grp % subs) * HPW + wave / WPH;
  const int q0 = qt * QT + (wave % WPH) * 32;  // this wave's first position
  const int qp = q0 + col;                     // this lane's query position

  const uint16_t* kbase = kc + (int64_t)pair * cache_len * HD;
  const uint16_t* vbase = vc + (int64_t)pair * cache_len * HD;
  auto fill = [&](int t, int buf) {
    char* kt = smem + buf * 2 * TB;
    char* vt = kt + TB;
#pragma unroll
    for (int i = 0; i < NF; ++i) {
      const int f = wave * NF + i;
      const int row = f * RPI + lane / CPR, slot = lane % CPR;
      const int64_t src = (int64_t)min(t * PA_KT + row, seq - 1) * HD;  // past the last key: masked, read in range
      fill16(kbase + src + (slot ^ k_swz<HD>(row)) * 8, kt + f * 1024);
      fill16(vbase + src + (slot ^ v_swz<HD>(row)) * 8, vt + f * 1024);
    }
  };

  fill(0, 0);  // in flight while the queries are loaded and rotated
  // ---- query rows: RMSNorm, RoPE, bf16; lane (col, h) holds elements 16 st + 8 h + 0..7 ----
  u32x4_t qf[ST];
  {
    const uint16_t* qr = q + ((int64_t)b * seq + min(qp, seq - 1)) * ldq + (int64_t)head * HD + 8 * h;
#pragma unroll
    for (int st = 0; st < ST; ++st) qf[st] = ld_global_16(qr + 16 * st);
    float ss = 0.f;
#pragma unroll
    for (int st = 0; st < ST; ++st)
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += bf_at(qf[st], e) * bf_at(qf[st], e);
    ss += __shfl_xor(ss, 32, 64);
    const float inv = rsqrtf(ss / (float)HD + eps);
    const float* rrow = rope + (int64_t)min(qp, seq - 1) * 2 * HD;
#pragma unroll
    for (int st = 0; st < ST / 2; ++st) {
      const int j = 16 * st + 8 * h;
      Rot8 r1, r2;
      r1.load(rrow, HD, j);
      r2.load(rrow, HD, HD / 2 + j);
      const u32x4_t w1 = ld_global_16(qw + j), w2 = ld_global_16(qw + HD / 2 + j);
      float a[8], c[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float n1 = bf_at(qf[st], e) * inv * bf_at(w1, e);
        const float n2 = bf_at(qf[st + ST / 2], e) * inv * bf_at(w2, e);
        a[e] = n1 * r1.c[e] - n2 * r1.s[e];
        c[e] = n2 * r2.c[e] + n1 * r2.s[e];
      }
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        qf[st][p] = pack_bf16x2(a[2 * p], a[2 * p + 1]);
        qf[st + ST / 2][p] = pack_bf16x2(c[2 * p], c[2 * p + 1]);
      }
    }
  }

  f32x16_t o[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] = 0.f;
  float m = -INFINITY, lsum = 0.f;

  const int nkt = (min(qt * QT + QT, seq) + PA_KT - 1) / PA_KT;
  for (int t = 0; t < nkt; ++t) {
    if (t + 1 < nkt) {
      fill(t + 1, (t + 1) & 1);
      wait_vm<2 * NF>();  // this tile's fills have landed, the next one's are in flight
    } else {
      wait_vm<0>();
    }
    tile_barrier();
    const int t0 = t * PA_KT;
    if (t0 <= q0 + 31) {  // else every key of the tile is after every query of the wave
      const char* kt = smem + (t & 1) * 2 * TB;
      const char* vt = kt + TB;
      f32x16_t s[2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
        for (int i = 0; i < 16; ++i) s[kb][i] = 0.f;
        const int row = kb * 32 + col;
#pragma unroll
        for (int st = 0; st < ST; ++st) {
          const u32x4_t kf = *reinterpret_cast<const u32x4_t*>(kt + row * RB + (((2 * st + h) ^ k_swz<HD>(row)) << 4));
          s[kb] = mfma16(kf, qf[st], s[kb]);
        }
      }
      // score i of block kb: key t0 + 32 kb + 8 (i / 4) + 4 h + i % 4, query qp
      if (t0 + PA_KT - 1 > q0) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (t0 + 32 * kb + 8 * (i / 4) + 4 * h + i % 4 > qp) s[kb][i] = -INFINITY;
      }
      float mx = s[0][0];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[kb][i]);
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float mn = fmaxf(m, mx);  // finite from the first tile on: key 0 is visible to every query
      if (__ballot(mn != m) != 0) {
        const float corr = exp2_hw((m - mn) * log2s);
        lsum *= corr;
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[d][i] *= corr;
        m = mn;
      }
      const float ms = m * log2s;
      u32x4_t pf[4];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
          const float p0 = exp2_hw(s[kb][i] * log2s - ms);
          const float p1 = exp2_hw(s[kb][i + 1] * log2s - ms);
          lsum += p0 + p1;
          pf[2 * kb + i / 8][(i % 8) / 2] = pack_bf16x2(p0, p1);
        }
      }
      // O^T += V^T . P^T, 16 keys a step: lane half h takes keys 16 st + 4 h + 0..3 and + 8
      const int j = lane & 15, dg = (lane >> 4) & 1;
#pragma unroll
      for (int st = 0; st < 4; ++st) {
#pragma unroll
        for (int d = 0; d < DB; ++d) {
          u32x4_t vf;
#pragma unroll
          for (int half = 0; half < 2; ++half) {
            const int row = 16 * st + 8 * half + 4 * h + j / 4;
            const int ch = 4 * d + 2 * dg + (j % 4) / 2;
            const int off = row * RB + ((ch ^ v_swz<HD>(row)) << 4) + (j & 1) * 8;
            const uint2 v = read_tr4(vt + off);
            vf[2 * half] = v.x;
            vf[2 * half + 1] = v.y;
          }
          o[d] = mfma16(vf, pf[st], o[d]);
        }
      }
    }
    tile_barrier();  // every wave is done with this buffer: the next iteration refills it
  }

  // ---- output: whole rows through this wave's share of the LDS ----
  lsum += __shfl_xor(lsum, 32, 64);
  const float inv_l = 1.f / lsum;
  char* ob = smem + wave * 32 * RB;
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<uint2*>(ob + col * RB + (((4 * d + g) ^ (col & (CPR - 1))) << 4) + 8 * h) =
          uint2{pack_bf16x2(o[d][4 * g] * inv_l, o[d][4 * g + 1] * inv_l),
                pack_bf16x2(o[d][4 * g + 2] * inv_l, o[d][4 * g + 3] * inv_l)};
#pragma unroll
  for (int it = 0; it < 32 / RPI; ++it) {
    const int row = it * RPI + lane / CPR, c = lane % CPR;
    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(ob + row * RB + ((c ^ (row & (CPR - 1))) << 4));
    if (q0 + row < seq)
      *reinterpret_cast<u32x4_t*>(out + ((int64_t)b * seq + q0 + row) * ldo + (int64_t)head * HD + c * 8) = v;
  }
}

// ----------------------------------------------------------------------- SwiGLU
// out = bf16(silu(g) * u), rows of g and u apart (two projections' own outputs).
__global__ void __launch_bounds__(256) swiglu_pair_kernel(const uint16_t* __restrict__ g, int64_t ldg,
                                                         const uint16_t* __restrict__ u, int64_t ldu, int64_t rows,
                                                         int chunks, uint16_t* __restrict__ out, int64_t ldo) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = idx / chunks;
  const int c = (int)(idx % chunks);
  if (row >= rows) return;
  const u32x4_t gv = ld_global_16(g + row * ldg + c * 8), uv = ld_global_16(u + row * ldu + c * 8);
  u32x4_t ov;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    float r[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float gg = bf_at(gv, 2 * p + e);
      r[e] = gg / (1.f + __expf(-gg)) * bf_at(uv, 2 * p + e);
    }
    ov[p] = pack_bf16x2(r[0], r[1]);
  }
  *reinterpret_cast<u32x4_t*>(out + row * ldo + c * 8) = ov;
}

bool a16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

struct AttnArgs {
  const uint16_t* q; int64_t ldq; const uint16_t* qw; float eps; const float* rope;
  const uint16_t* kc; const uint16_t* vc; int64_t cache_len;
  int seq, nh, nkv; int64_t batch; float log2s; uint16_t* out; int64_t ldo; hipStream_t st;
};

template <int HD, int HPW, int NW>
hipError_t launch_attention(const AttnArgs& a) {
  const int64_t groups = a.batch * a.nkv * (a.nh / a.nkv / HPW);
  const int qt = 32 * (NW / HPW);
  const int64_t blocks = groups * ((a.seq + qt - 1) / qt);
  if (groups > 0x7fffffff || blocks > 0x7fffffff) return hipErrorInvalidValue;
  prefill_attention_kernel<HD, HPW, NW><<<dim3((unsigned)blocks), dim3(NW * 64), 0, a.st>>>(
      a.q, a.ldq, a.qw, a.eps, a.rope, a.kc, a.vc, a.cache_len, a.seq, a.nh, a.nkv, (int)groups, a.log2s, a.out, a.ldo);
  return hipGetLastError();
}

// Heads per workgroup: as many of a kv head's group as divide it, up to the waves (they share
// the K/V tiles): 8 x 512, 16 heads on 4 of 128: 25.6 / 25.7 / 26.5 us with 4 / 2 / 1 heads; 64
// wide, 32 heads on 4: 23.2 / 23.2 / 24.1. Two waves where four would leave CUs without a
// workgroup, below 1024 row blocks (graphs of 20, us, two waves against four, 16 heads on 8):
// 1 x 64 7.9 / 9.4, 1 x 128 9.4 / 10.6, 1 x 256 12.6 / 13.3, even at 256 and 512 blocks (19.1 /
// 18.8, 19.5 / 19.0), 768 22.0 / 19.4, 1024 22.5 / 20.1, 8 x 512 30.5 / 25.6: past 512 blocks the
// line is late.
template <int HD>
hipError_t launch_attention_hd(const AttnArgs& a) {
  const int rep = a.nh / a.nkv;
  const int64_t rows = a.batch * a.nh * (((int64_t)a.seq + 31) / 32);  // 32-row query blocks
  const bool four = rows >= 4 * 256;
  if (rep % 4 == 0 && four) return launch_attention<HD, 4, 4>(a);
  if (rep % 2 == 0) return four ? launch_attention<HD, 2, 4>(a) : launch_attention<HD, 2, 2>(a);
  return four ? launch_attention<HD, 1, 4>(a) : launch_attention<HD, 1, 2>(a);
}

}  // namespace
int decode_fail(int code, const char* msg);  // decode_step.hip: sets wsl_decode_last_error()
}  // namespace wsl

using namespace wsl;

extern "C" {

int wsl_kv_norm_rope_fwd(const void* k, int64_t ldk, const void* v, int64_t ldv, int64_t batch, int64_t seq,
                         int64_t n_kv_heads, int64_t head_dim, const void* k_norm_w, float eps, const float* rope,
                         void* k_cache, void* v_cache, int64_t cache_len, void* stream) {
  decode_fail(WSL_OK, "");
  if (batch < 0 || seq < 0 || n_kv_heads < 1 || n_kv_heads > 0x7fffffff || cache_len < 1 || seq > cache_len ||
      seq > 0x7fffffff)
    return decode_fail(WSL_E_SHAPE, "kv_norm_rope: bad sizes (seq must fit the cache)");
  if (head_dim != 64 && head_dim != 128) return decode_fail(WSL_E_SHAPE, "kv_norm_rope: head_dim must be 64 or 128");
  if (ldk < n_kv_heads * head_dim || ldv < n_kv_heads * head_dim)
    return decode_fail(WSL_E_SHAPE, "kv_norm_rope: leading dimension too small");
  if (batch == 0 || seq == 0) return WSL_OK;
  if (!k || !v || !k_norm_w || !rope || !k_cache || !v_cache)
    return decode_fail(WSL_E_INVALID_ARG, "kv_norm_rope: null pointer");
  if (!a16(k) || !a16(v) || !a16(k_norm_w) || !a16(rope) || !a16(k_cache) || !a16(v_cache) || ldk % 8 || ldv % 8)
    return decode_fail(WSL_E_ALIGN, "kv_norm_rope: pointers must be 16-byte aligned, leading dims multiples of 8");
  const int64_t rows = batch * seq * n_kv_heads;
  const int64_t per = 256 / (head_dim / 8);
  if ((rows + per - 1) / per > 0x7fffffff) return decode_fail(WSL_E_SHAPE, "kv_norm_rope: too many rows");
  const dim3 grid((unsigned)((rows + per - 1) / per));
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
#define WSL_KV(HD)                                                                                              \
  kv_rope_kernel<HD><<<grid, dim3(256), 0, st>>>((const uint16_t*)k, ldk, (const uint16_t*)v, ldv, (int)seq,    \
                                                 (int)n_kv_heads, rows, (const uint16_t*)k_norm_w, eps, rope,    \
                                                 (uint16_t*)k_cache, (uint16_t*)v_cache, cache_len)
  if (head_dim == 64) WSL_KV(64);
  else WSL_KV(128);
#undef WSL_KV
  return hipGetLastError() == hipSuccess ? WSL_OK : decode_fail(WSL_E_LAUNCH, "kv_norm_rope: launch failed");
}

int wsl_prefill_attention_fwd(const void* q, int64_t ldq, int64_t batch, int64_t seq, int64_t n_heads,
                              int64_t n_kv_heads, int64_t head_dim, const void* q_norm_w, float eps,
                              const float* rope, const void* k_cache, const void* v_cache, int64_t cache_len,
                              float scale, void* out, int64_t ldo, void* stream) {
  decode_fail(WSL_OK, "");
  if (batch < 0 || seq < 0 || n_heads < 1 || n_kv_heads < 1 || n_heads % n_kv_heads != 0 || n_heads > 0x7fffffff ||
      cache_len < 1 || seq > cache_len || seq > 0x7fffffff - 256)
    return decode_fail(WSL_E_SHAPE, "prefill_attention: bad sizes (seq must fit the cache, n_heads a multiple of n_kv_heads)");
  if (head_dim != 64 && head_dim != 128)
    return decode_fail(WSL_E_SHAPE, "prefill_attention: head_dim must be 64 or 128");
  if (ldq < n_heads * head_dim || ldo < n_heads * head_dim)
    return decode_fail(WSL_E_SHAPE, "prefill_attention: leading dimension too small");
  if (!(scale > 0.f)) return decode_fail(WSL_E_INVALID_ARG, "prefill_attention: scale must be positive");
  if (batch == 0 || seq == 0) return WSL_OK;
  if (!q || !q_norm_w || !rope || !k_cache || !v_cache || !out)
    return decode_fail(WSL_E_INVALID_ARG, "prefill_attention: null pointer");
  if (!a16(q) || !a16(q_norm_w) || !a16(rope) || !a16(k_cache) || !a16(v_cache) || !a16(out) || ldq % 8 || ldo % 8)
    return decode_fail(WSL_E_ALIGN, "prefill_attention: pointers must be 16-byte aligned, leading dims multiples of 8");
  const AttnArgs a{(const uint16_t*)q, ldq, (const uint16_t*)q_norm_w, eps, rope, (const uint16_t*)k_cache,
                   (const uint16_t*)v_cache, cache_len, (int)seq, (int)n_heads, (int)n_kv_heads, batch,
                   scale * 1.4426950408889634f, (uint16_t*)out, ldo, reinterpret_cast<hipStream_t>(stream)};
  const hipError_t e = head_dim == 64 ? launch_attention_hd<64>(a) : launch_attention_hd<128>(a);
  if (e == hipErrorInvalidValue) return decode_fail(WSL_E_SHAPE, "prefill_attention: too many query tiles");
  return e == hipSuccess ? WSL_OK : decode_fail(WSL_E_LAUNCH, "prefill_attention: launch failed");
}

int wsl_swiglu_pair_fwd(const void* gate, int64_t ldg, const void* up, int64_t ldu, int64_t rows, int64_t ffn,
                        void* out, int64_t ldo, void* stream) {
  decode_fail(WSL_OK, "");
  if (rows < 0 || ffn < 8 || ffn % 8 != 0 || ffn > 0x7fffffff)
    return decode_fail(WSL_E_SHAPE, "swiglu_pair: ffn must be a positive multiple of 8, rows >= 0");
  if (ldg < ffn || ldu < ffn || ldo < ffn) return decode_fail(WSL_E_SHAPE, "swiglu_pair: leading dimension below ffn");
  if (rows == 0) return WSL_OK;
  if (!gate || !up || !out) return decode_fail(WSL_E_INVALID_ARG, "swiglu_pair: null pointer");
  if (!a16(gate) || !a16(up) || !a16(out) || ldg % 8 || ldu % 8 || ldo % 8)
    return decode_fail(WSL_E_ALIGN, "swiglu_pair: pointers must be 16-byte aligned, leading dims multiples of 8");
  const int64_t blocks = (rows * (ffn / 8) + 255) / 256;
  if (blocks > 0x7fffffff) return decode_fail(WSL_E_SHAPE, "swiglu_pair: too many elements");
  swiglu_pair_kernel<<<dim3((unsigned)blocks), dim3(256), 0, reinterpret_cast<hipStream_t>(stream)>>>(
      (const uint16_t*)gate, ldg, (const uint16_t*)up, ldu, rows, (int)(ffn / 8), (uint16_t*)out, ldo);
  return hipGetLastError() == hipSuccess ? WSL_OK : decode_fail(WSL_E_LAUNCH, "swiglu_pair: launch failed");
}

}  // extern "C"
