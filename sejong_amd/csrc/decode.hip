// The blocks' products for a few rows: the KV-cache path's decode steps
// (Model::forward_cached, model lib.rs:362-372; architecture.rs:474-533) and
// chunks of up to 8 tokens, bf16.
//
// A tiled product gives a row-starved call N / 64 workgroups that each stream
// 64 weight rows through LDS stages behind barriers: at one token (d 384)
// 10 workgroups and 5.6-7.7 us a product, nearly all of it latency.  Here one
// wave owns 16 output columns and all the rows (one MFMA tile): its weight
// rows come straight from the transposed mirror into registers, 16 k-steps
// in flight, requested before anything else; the RMSNorm that precedes a
// product runs in every wave on the few rows meanwhile (its row is read once
// from cache) and leaves the normed rows in LDS, so a layer is five launches
// instead of seven and no normed row travels through memory.  The bound is
// one weight read's latency plus the launch.  25 calls (a prompt of 200 and
// 24 tokens, 6 layers, d 384): 7.2 -> 4.8 ms (the rest is launches: 32 a token,
// about 4 us of host time each, one read-back).
//
// The rows' norms run one after another in every wave, so each further row
// adds a latency per product where the tiled path's time stays: a call of
// 1 / 4 / 8 / 12 / 16 tokens takes 158 / 206 / 255 / 305 / 350 us (6 layers,
// d 384; tiled 272 / 272 / 279 / 291 / 297) and 423 / 548 / 680 / 808 / 930
// (12 layers, d 1024; tiled 763 / 786 / 806 / 830 / 847).  Hence 8 rows.
//
// Every product keeps the k order, the MFMA shape and the roundings of the
// tiled one (k_gemm_fast, k_rms_fwd_t), so the logits keep their bits: a
// cached call equals the full forward.
#include <math.h>

#include "common.h"

using namespace sj;

namespace {

constexpr int DR = sjh::DECODE_ROWS;  // at most the 16 of one MFMA tile
constexpr int U = 8;                  // k-steps (32) per register group, two groups in flight
enum { D_QKV = 0, D_RESID = 1, D_GATEUP = 2, D_HEAD = 3 };

struct DArgs {
  int n, N, K;             // rows, output columns, contraction
  const bf16_t* x;         // rows [n][ldx]
  long ldx;
  const bf16_t* wn;        // norm weight (NORM)
  float eps;
  const bf16_t *w0, *w1;   // [N][ldw]; w1: up (gate/up) or the lo plane (head)
  long ldw;
  // embedding lookup as the rows (nullable): row r is table[ids[r]], also
  // written to xout [n][K] by the first workgroup
  const bf16_t* table;
  bf16_t* xout;
  int ids[DR];
  // outputs
  bf16_t *c0, *c1, *c2;    // QKV: q, k, v; residual / gate-up: c0
  long ldc0, ldc1;         // q (or c0), k and v row strides
  int n1, n2;              // QKV: first column of k and of v
  const float* rope;       // QKV: table row r is row r's position
  int hd;
  const bf16_t* r;         // residual
  long ldr;
  float *f0, *f1;          // head: fp32 logits (f1 nullable)
};

__device__ __forceinline__ bf16x8 zfrag() { return __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u}); }

template <int EPI>
__global__ __launch_bounds__(64) void k_decode(DArgs p) {
  constexpr bool NORM = EPI != D_RESID, DUAL = EPI == D_GATEUP || EPI == D_HEAD;
  constexpr int NB = DUAL ? 2 : 1;
  extern __shared__ __attribute__((aligned(16))) bf16_t rows[];  // NORM: [n][K + 8]
  const int lane = threadIdx.x, j = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16, K = p.K, nk = (K + 31) / 32;
  const int col = n0 + j, brow = col < p.N ? col : p.N - 1;
  const bf16_t* b0 = p.w0 + (long)brow * p.ldw + 8 * g;
  const bf16_t* b1 = DUAL ? p.w1 + (long)brow * p.ldw + 8 * g : nullptr;
  const int ar = j < p.n ? j : p.n - 1;  // rows past n repeat the last: their results are not stored
  const bf16_t* ga = NORM ? nullptr : p.x + (long)ar * p.ldx + 8 * g;
  // k-steps [s0, s0 + U) of this lane's weight row(s) (and row operand); a
  // chunk past K (the last step of a ragged K) is zero
  auto load = [&](int s0, u32x4 (&wb)[NB][U], u32x4 (&wa)[U]) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = 32 * (s0 + u);
      const bool in = k + 8 * g < K;
      wb[0][u] = in ? *(const u32x4*)(b0 + k) : u32x4{0u, 0u, 0u, 0u};
      if constexpr (DUAL) wb[NB - 1][u] = in ? *(const u32x4*)(b1 + k) : u32x4{0u, 0u, 0u, 0u};
      if constexpr (!NORM) wa[u] = in ? *(const u32x4*)(ga + k) : u32x4{0u, 0u, 0u, 0u};
    }
  };
  u32x4 wb[2][NB][U], wa[2][U];
  load(0, wb[0], wa[0]);
  load(U, wb[1], wa[1]);

  if constexpr (NORM) {
    // RMSNorm of the rows (k_rms_fwd_t's sums and roundings): a lane holds
    // column pairs lane + 64 i
    const int pairs = K >> 1;
    for (int r = 0; r < p.n; r++) {
      const bf16_t* x = p.table ? p.table + (long)p.ids[r] * K : p.x + (long)r * p.ldx;
      uint32_t xw[8], ww[8];
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int q = lane + 64 * i;
        xw[i] = q < pairs ? *(const uint32_t*)(x + 2 * q) : 0u;
        ww[i] = q < pairs ? *(const uint32_t*)(p.wn + 2 * q) : 0u;
      }
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float a = bf2f((bf16_t)(xw[i] & 0xffffu)), b = bf2f((bf16_t)(xw[i] >> 16));
        s += a * a + b * b;
      }
      s = wave_sum(s);
      const float inv = 1.f / sqrtf(s / (float)(long)K + p.eps);
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int q = lane + 64 * i;
        if (q >= pairs) continue;
        const float a = bf2f((bf16_t)(xw[i] & 0xffffu)), b = bf2f((bf16_t)(xw[i] >> 16));
        const float wx = bf2f((bf16_t)(ww[i] & 0xffffu)), wy = bf2f((bf16_t)(ww[i] >> 16));
        *(uint32_t*)(rows + (long)r * (K + 8) + 2 * q) = pack2(f2bf(a * inv * wx), f2bf(b * inv * wy));
        if (p.xout && blockIdx.x == 0) *(uint32_t*)(p.xout + (long)r * K + 2 * q) = xw[i];
      }
    }
    __syncthreads();
  }

  f32x4 acc[EPI == D_GATEUP ? 2 : 1];
  acc[0] = f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (EPI == D_GATEUP) acc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto steps = [&](int s0, const u32x4 (&b)[NB][U], const u32x4 (&a)[U]) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = 32 * (s0 + u);
      if (k >= K) break;
      bf16x8 af;
      if constexpr (NORM)
        af = k + 8 * g < K ? __builtin_bit_cast(bf16x8, *(const u32x4*)(rows + (long)ar * (K + 8) + k + 8 * g)) : zfrag();
      else
        af = __builtin_bit_cast(bf16x8, a[u]);
      acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, __builtin_bit_cast(bf16x8, b[0][u]), acc[0], 0, 0, 0);
      if constexpr (EPI == D_GATEUP)
        acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, __builtin_bit_cast(bf16x8, b[1][u]), acc[1], 0, 0, 0);
      if constexpr (EPI == D_HEAD)  // hi, then lo plane of the weight
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, __builtin_bit_cast(bf16x8, b[1][u]), acc[0], 0, 0, 0);
    }
  };
  for (int s0 = 0; s0 < nk; s0 += 2 * U) {
    steps(s0, wb[0], wa[0]);
    if (s0 + 2 * U < nk) load(s0 + 2 * U, wb[0], wa[0]);
    if (s0 + U < nk) steps(s0 + U, wb[1], wa[1]);
    if (s0 + 3 * U < nk) load(s0 + 3 * U, wb[1], wa[1]);
  }

  // acc[.][i] = C[4 g + i][n0 + j]
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int row = 4 * g + i;
    const bool ok = row < p.n && col < p.N;
    const float v = acc[0][i];
    if constexpr (EPI == D_QKV) {
      const float a = round_bf(v), y = __shfl_xor(a, 1, 64);  // the pair partner's column
      float o = a;
      const int seg = col >= p.n2 ? 2 : col >= p.n1 ? 1 : 0;
      const int cl = col - (seg == 2 ? p.n2 : seg == 1 ? p.n1 : 0);
      if (seg < 2 && ok) {
        const float2 cs = *(const float2*)(p.rope + 2 * ((long)row * (p.hd >> 1) + ((cl % p.hd) >> 1)));
        o = (cl & 1) ? fmaf(a, cs.x, mul_rn(y, cs.y)) : fmaf(a, cs.x, -mul_rn(y, cs.y));
      }
      if (ok) {
        if (seg == 0) p.c0[(long)row * p.ldc0 + cl] = f2bf(o);
        else (seg == 1 ? p.c1 : p.c2)[(long)row * p.ldc1 + cl] = f2bf(o);
      }
    } else if constexpr (EPI == D_RESID) {
      if (ok) p.c0[(long)row * p.ldc0 + col] = f2bf(bf2f(p.r[(long)row * p.ldr + col]) + round_bf(v));
    } else if constexpr (EPI == D_GATEUP) {
      const float gt = round_bf(v), up = round_bf(acc[1][i]);
      const float sg = 1.f / (1.f + expf(-gt));
      if (ok) p.c0[(long)row * p.ldc0 + col] = f2bf(gt * sg * up);
    } else {
      if (ok) {
        p.f0[col] = v;
        if (p.f1) p.f1[col] = v;
      }
    }
  }
}

template <int EPI>
int launch(hipStream_t s, const DArgs& p, const char* what) {
  const size_t lds = EPI == D_RESID ? 0 : sizeof(bf16_t) * (size_t)p.n * (size_t)(p.K + 8);
  hipLaunchKernelGGL(k_decode<EPI>, dim3((unsigned)((p.N + 15) / 16)), dim3(64), lds, s, p);
  SJ_LAUNCH_CHECK(what);
  return SJ_OK;
}

bool al16(const void* q) { return ((uintptr_t)q & 15) == 0; }

}  // namespace

namespace sjh {

// n rows of width d (a multiple of 8, at most 1024: the lanes' column pairs)
bool decode_rows_ok(long n, long d) { return n >= 1 && n <= DECODE_ROWS && d % 8 == 0 && d <= 1024; }

int decode_qkv(hipStream_t s, const uint16_t* x, const uint16_t* table, const int32_t* ids, uint16_t* xout,
               const uint16_t* wn, float eps, long n, long d, const uint16_t* wqkv_t, long kv, uint16_t* q, uint16_t* k,
               uint16_t* v, const float* rope, long head_dim) {
  SJ_REQUIRE(decode_rows_ok(n, d) && al16(wqkv_t) && wn && (x || (table && ids)) && rope && head_dim % 2 == 0 &&
                 d % head_dim == 0 && kv % head_dim == 0,
             "project_qkv (few rows): rows %ld width %ld", n, d);
  DArgs p = {};
  p.n = (int)n; p.N = (int)(d + 2 * kv); p.K = (int)d;
  p.x = x; p.ldx = d; p.wn = wn; p.eps = eps; p.w0 = wqkv_t; p.ldw = d;
  p.table = table; p.xout = xout;
  for (long i = 0; i < n && ids; i++) p.ids[i] = ids[i];
  p.c0 = q; p.c1 = k; p.c2 = v; p.ldc0 = d; p.ldc1 = kv; p.n1 = (int)d; p.n2 = (int)(d + kv);
  p.rope = rope; p.hd = (int)head_dim;
  return launch<D_QKV>(s, p, "project_qkv (few rows)");
}

int decode_residual(hipStream_t s, const uint16_t* a, long n, long K, const uint16_t* w_t, long N, const uint16_t* r,
                    uint16_t* y) {
  SJ_REQUIRE(n >= 1 && n <= DECODE_ROWS && K % 8 == 0 && al16(a) && al16(w_t), "linear_residual (few rows): rows %ld", n);
  DArgs p = {};
  p.n = (int)n; p.N = (int)N; p.K = (int)K;
  p.x = a; p.ldx = K; p.w0 = w_t; p.ldw = K;
  p.c0 = y; p.ldc0 = N; p.r = r; p.ldr = N;
  return launch<D_RESID>(s, p, "linear_residual (few rows)");
}

int decode_gate_up(hipStream_t s, const uint16_t* x, const uint16_t* wn, float eps, long n, long d, const uint16_t* wg_t,
                   const uint16_t* wu_t, long F, uint16_t* h) {
  SJ_REQUIRE(decode_rows_ok(n, d) && al16(wg_t) && al16(wu_t), "gate_up (few rows): rows %ld width %ld", n, d);
  DArgs p = {};
  p.n = (int)n; p.N = (int)F; p.K = (int)d;
  p.x = x; p.ldx = d; p.wn = wn; p.eps = eps; p.w0 = wg_t; p.w1 = wu_t; p.ldw = d;
  p.c0 = h; p.ldc0 = F;
  return launch<D_GATEUP>(s, p, "gate_up (few rows)");
}

int decode_head(hipStream_t s, const uint16_t* x, const uint16_t* wn, float eps, long d, const uint16_t* w_hi,
                const uint16_t* w_lo, long N, float* logits, float* logits2) {
  SJ_REQUIRE(decode_rows_ok(1, d) && al16(w_hi) && al16(w_lo), "head (one row): width %ld", d);
  DArgs p = {};
  p.n = 1; p.N = (int)N; p.K = (int)d;
  p.x = x; p.ldx = d; p.wn = wn; p.eps = eps; p.w0 = w_hi; p.w1 = w_lo; p.ldw = d;
  p.f0 = logits; p.f1 = logits2;
  return launch<D_HEAD>(s, p, "head (one row)");
}

}  // namespace sjh
