// INT8 on gfx950: the quantizers of src/scratch_llm/quant/int8.py bit-exact with the reference (which
// computes in the input's dtype: every fp32 intermediate is rounded back to bf16 / fp16 exactly where
// torch rounds it), w8a8_linear on int8 MFMA with exact int32 accumulation, and the int8 weight-only
// linear as a policy of the shared GEMV.
//
// Reductions see the input as [A, B, C] with B the kept axis (A = product of the dims before it,
// C = product of the dims after it); per-tensor is A = C = 1, B = 1 over all n elements.
//
// Tiled int8 layout (the weight-only linear): block (t, kb) = 1 KiB covering 16 rows x 64 columns;
// lane L owns the 16 codes of row 16t + (L & 15), columns kb*64 + 16(L >> 4) + e, stored as
// u = q + 128 in byte e. Per-row fp32 scales are read in the epilogue.
#include "sqx_quant.h"
#include "sqx_skinny.h"

namespace sqx {

template <int DT>
__device__ inline float rd(float v) {  // round an fp32 result to the working dtype
  if (DT == SQX_DTYPE_BF16) return bf16_bits_to_f32(f32_to_bf16_bits(v));
  if (DT == SQX_DTYPE_F16) return f16_bits_to_f32(f32_to_f16_bits(v));
  return v;
}

template <int DT>
__device__ inline void store_dt(void* p, int64_t i, float v) {  // v already representable in DT
  if (DT == SQX_DTYPE_F32)
    static_cast<float*>(p)[i] = v;
  else if (DT == SQX_DTYPE_BF16)
    static_cast<uint16_t*>(p)[i] = f32_to_bf16_bits(v);
  else
    static_cast<uint16_t*>(p)[i] = f32_to_f16_bits(v);
}

// NaN-propagating reductions (torch amax / amin propagate NaN)
__device__ inline float nmax(float m, float v) { return (v > m || v != v) ? v : m; }
__device__ inline float nmin(float m, float v) { return (v < m || v != v) ? v : m; }

// ----------------------------------------------------------------------------------------------
// Per-slice statistics. OP 0: amax of |x| -> symmetric scale; OP 1: min and max -> affine scale and
// zero-point. The scale math (int8.py:119-124, 163-170), in the working dtype DT:
//   symmetric: s = max(rd(amax / 127), rd(eps))
//   affine:    lo = min(xmin, 0), hi = max(xmax, 0); s = max(rd(rd(hi - lo) / 255), rd(eps));
//              z = clamp(rint(rd(-lo / s)), 0, 255)
// ----------------------------------------------------------------------------------------------
template <int DT, int OP>
__device__ inline void slice_params(float a, float b, float eps, float& s, float& z) {
  const float e = rd<DT>(eps);
  z = 0.0f;
  if (OP == 0) {
    s = rd<DT>(__fdiv_rn(a, 127.0f));
    if (s < e) s = e;
  } else {
    const float lo = a < 0.0f || a != a ? a : 0.0f;  // torch.minimum(x, 0) propagates NaN
    const float hi = b > 0.0f || b != b ? b : 0.0f;
    s = rd<DT>(__fdiv_rn(rd<DT>(hi - lo), 255.0f));
    if (s < e) s = e;
    z = __builtin_rintf(rd<DT>(__fdiv_rn(-lo, s)));
    z = fminf(fmaxf(z, 0.0f), 255.0f);
  }
}
template <int DT, int OP>
__device__ inline void finish_stats(float a, float b, float eps, void* s_out, void* z_out, int64_t i) {
  float s, z;
  slice_params<DT, OP>(a, b, eps, s, z);
  store_dt<DT>(s_out, i, s);
  if (OP == 1) store_dt<DT>(z_out, i, z);
}

// One workgroup per kept index b (C >= 32 or A*C large): reduces x[a, b, c] over a and c.
template <int DT, int OP>
__global__ __launch_bounds__(256) void stats_wg_kernel(const void* __restrict__ x, int64_t A, int64_t B, int64_t C,
                                                       float eps, void* __restrict__ s_out,
                                                       void* __restrict__ z_out) {
  __shared__ float ra[256], rb[256];
  const int64_t b = blockIdx.x;
  float m0 = OP == 0 ? 0.0f : INFINITY, m1 = -INFINITY;
  const int64_t per = A * C;
  for (int64_t j = threadIdx.x; j < per; j += blockDim.x) {
    const int64_t a = j / C, c = j - a * C;
    const float v = load_as_f32(x, DT, (a * B + b) * C + c);
    if (OP == 0) m0 = nmax(m0, fabsf(v));
    else { m0 = nmin(m0, v); m1 = nmax(m1, v); }
  }
  ra[threadIdx.x] = m0;
  rb[threadIdx.x] = m1;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) {
      if (OP == 0) ra[threadIdx.x] = nmax(ra[threadIdx.x], ra[threadIdx.x + s]);
      else {
        ra[threadIdx.x] = nmin(ra[threadIdx.x], ra[threadIdx.x + s]);
        rb[threadIdx.x] = nmax(rb[threadIdx.x], rb[threadIdx.x + s]);
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) finish_stats<DT, OP>(ra[0], rb[0], eps, s_out, z_out, b);
}

// One thread per kept index b (small C): coalesced across b.
template <int DT, int OP>
__global__ __launch_bounds__(256) void stats_thread_kernel(const void* __restrict__ x, int64_t A, int64_t B,
                                                           int64_t C, float eps, void* __restrict__ s_out,
                                                           void* __restrict__ z_out) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  float m0 = OP == 0 ? 0.0f : INFINITY, m1 = -INFINITY;
  for (int64_t a = 0; a < A; ++a)
    for (int64_t c = 0; c < C; ++c) {
      const float v = load_as_f32(x, DT, (a * B + b) * C + c);
      if (OP == 0) m0 = nmax(m0, fabsf(v));
      else { m0 = nmin(m0, v); m1 = nmax(m1, v); }
    }
  finish_stats<DT, OP>(m0, m1, eps, s_out, z_out, b);
}

// Per-tensor: grid-stride partials, then one workgroup finishes.
static constexpr int kStatParts = 512;

template <int DT, int OP>
__global__ __launch_bounds__(256) void stats_partial_kernel(const void* __restrict__ x, int64_t n,
                                                            float* __restrict__ part) {
  __shared__ float ra[256], rb[256];
  float m0 = OP == 0 ? 0.0f : INFINITY, m1 = -INFINITY;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float v = load_as_f32(x, DT, i);
    if (OP == 0) m0 = nmax(m0, fabsf(v));
    else { m0 = nmin(m0, v); m1 = nmax(m1, v); }
  }
  ra[threadIdx.x] = m0;
  rb[threadIdx.x] = m1;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) {
      if (OP == 0) ra[threadIdx.x] = nmax(ra[threadIdx.x], ra[threadIdx.x + s]);
      else {
        ra[threadIdx.x] = nmin(ra[threadIdx.x], ra[threadIdx.x + s]);
        rb[threadIdx.x] = nmax(rb[threadIdx.x], rb[threadIdx.x + s]);
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = ra[0];
    part[2 * blockIdx.x + 1] = rb[0];
  }
}

template <int DT, int OP>
__global__ __launch_bounds__(256) void stats_final_kernel(const float* __restrict__ part, int parts, float eps,
                                                          void* __restrict__ s_out, void* __restrict__ z_out) {
  __shared__ float ra[256], rb[256];
  float m0 = OP == 0 ? 0.0f : INFINITY, m1 = -INFINITY;
  for (int i = threadIdx.x; i < parts; i += blockDim.x) {
    if (OP == 0) m0 = nmax(m0, part[2 * i]);
    else { m0 = nmin(m0, part[2 * i]); m1 = nmax(m1, part[2 * i + 1]); }
  }
  ra[threadIdx.x] = m0;
  rb[threadIdx.x] = m1;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) {
      if (OP == 0) ra[threadIdx.x] = nmax(ra[threadIdx.x], ra[threadIdx.x + s]);
      else {
        ra[threadIdx.x] = nmin(ra[threadIdx.x], ra[threadIdx.x + s]);
        rb[threadIdx.x] = nmax(rb[threadIdx.x], rb[threadIdx.x + s]);
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) finish_stats<DT, OP>(ra[0], rb[0], eps, s_out, z_out, 0);
}

// ----------------------------------------------------------------------------------------------
// Elementwise quantize / dequantize with the scale of slice b = (i / C) % B
// ----------------------------------------------------------------------------------------------
// symmetric: q = clamp(rint(rd(x / s)), -127, 127); affine: q = clamp(rint(rd(rd(x / s) + z)), 0, 255)
template <int DT, int OP>
__global__ __launch_bounds__(256) void quantize_kernel(const void* __restrict__ x, int64_t n, int64_t B, int64_t C,
                                                       const void* __restrict__ s, const void* __restrict__ z,
                                                       uint8_t* __restrict__ q) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t b = (i / C) % B;
  const float v = load_as_f32(x, DT, i);
  const float sv = load_as_f32(s, DT, b);
  if (OP == 0) {
    const float r = fminf(fmaxf(__builtin_rintf(rd<DT>(__fdiv_rn(v, sv))), -127.0f), 127.0f);
    q[i] = static_cast<uint8_t>(static_cast<int8_t>(r == r ? r : 0.0f));
  } else {
    const float r = fminf(fmaxf(__builtin_rintf(rd<DT>(rd<DT>(__fdiv_rn(v, sv)) + load_as_f32(z, DT, b))), 0.0f), 255.0f);
    q[i] = static_cast<uint8_t>(r == r ? r : 0.0f);
  }
}

// The same two steps for the rows of a [B, C] matrix (A = 1), in one pass: the row stays in registers between
// its statistics and its codes. 256 threads a row, 8 consecutive elements per thread and chunk (chunk c of the
// row is thread c % 256's). w8a8_linear quantizes both operands on every call: 14336 x 4096 in bf16 took 184 us in
// two passes (element loads, 64-bit divisions for the slice index, an IEEE division per element), 37.7 us (4.7 TB/s)
// in one. Rows from B1 on come from a second matrix x2 of the same width, so w8a8_linear's two operands take one
// launch.
template <int DT>
__device__ inline float rd_fast(float v) {  // rd without its NaN case (NaN stays NaN)
  if (DT == SQX_DTYPE_BF16) return bf16_lo(ActBF16::pack_rne(v, 0.0f));
  return rd<DT>(v);
}

template <int DT, int OP, int NCH>
__global__ __launch_bounds__(256) void quantize_rows_kernel(const void* __restrict__ x, const void* __restrict__ x2,
                                                            int64_t B1, int64_t C, float eps,
                                                            void* __restrict__ s_out, void* __restrict__ z_out,
                                                            uint8_t* __restrict__ q) {
  __shared__ float red[2][4];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x;
  const int nch = static_cast<int>(C / 8);
  float v[NCH][8];
  float m0 = OP == 0 ? 0.0f : INFINITY, m1 = -INFINITY;
  const void* src = row < B1 ? x : x2;
  const int64_t src0 = (row < B1 ? row : row - B1) * C;
#pragma unroll
  for (int i = 0; i < NCH; ++i)
    if (tid + 256 * i < nch) load8_f32(src, DT, src0 + 8 * (tid + 256 * i), v[i]);
#pragma unroll
  for (int i = 0; i < NCH; ++i)
    if (tid + 256 * i < nch) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (OP == 0) m0 = nmax(m0, fabsf(v[i][e]));
        else m0 = nmin(m0, v[i][e]), m1 = nmax(m1, v[i][e]);
      }
    }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    if (OP == 0) m0 = nmax(m0, __shfl_xor(m0, o, 64));
    else m0 = nmin(m0, __shfl_xor(m0, o, 64)), m1 = nmax(m1, __shfl_xor(m1, o, 64));
  }
  if ((tid & 63) == 0) red[0][tid >> 6] = m0, red[1][tid >> 6] = m1;
  __syncthreads();
  m0 = red[0][0], m1 = red[1][0];
#pragma unroll
  for (int w = 1; w < 4; ++w) {
    if (OP == 0) m0 = nmax(m0, red[0][w]);
    else m0 = nmin(m0, red[0][w]), m1 = nmax(m1, red[1][w]);
  }
  float sv, zv;
  slice_params<DT, OP>(m0, m1, eps, sv, zv);
  if (tid == 0) {
    store_dt<DT>(s_out, row, sv);
    if (OP == 1) store_dt<DT>(z_out, row, zv);
  }
  const SharedDiv sd = shared_div(sv);
#pragma unroll
  for (int i = 0; i < NCH; ++i)
    if (tid + 256 * i < nch) {
      uint32_t w[2] = {0u, 0u};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float t = rd_fast<DT>(div_by(sd, v[i][e]));
        float r;
        if (OP == 0) r = fminf(fmaxf(__builtin_rintf(t), -127.0f), 127.0f);
        else r = fminf(fmaxf(__builtin_rintf(rd_fast<DT>(t + zv)), 0.0f), 255.0f);
        const int c = static_cast<int>(r == r ? r : 0.0f);
        w[e >> 2] |= (static_cast<uint32_t>(c) & 0xffu) << (8 * (e & 3));
      }
      *reinterpret_cast<u32x2v_t*>(q + row * C + 8 * (tid + 256 * i)) = u32x2v_t{w[0], w[1]};
    }
}

// symmetric: rd(q * s); affine: rd(rd(q - z) * s) (int8.py:127-129, 174-176), in the scale dtype.
template <int DT, int OP>
__global__ __launch_bounds__(256) void dequantize_kernel(const uint8_t* __restrict__ q, int64_t n, int64_t B,
                                                         int64_t C, const void* __restrict__ s,
                                                         const void* __restrict__ z, void* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t b = (i / C) % B;
  const float sv = load_as_f32(s, DT, b);
  float v;
  if (OP == 0) v = rd<DT>(static_cast<float>(static_cast<int8_t>(q[i])) * sv);
  else v = rd<DT>(rd<DT>(static_cast<float>(q[i]) - load_as_f32(z, DT, b)) * sv);
  store_dt<DT>(out, i, v);
}

// ----------------------------------------------------------------------------------------------
// w8a8_linear (int8.py:189-213): acc = q_x @ q_w^T in int32 (exact), y = fp32(acc) * (s_x[m] * s_w[n])
// with the scale product in the promoted scale dtype PD, on v_mfma_i32_16x16x64_i8.
//
// A workgroup of four waves owns a T x T output tile (T = 64 or 128), each wave a quarter. A stage covers 128 k of
// the T rows of either operand, 128 bytes a row, copied by buffer loads that write LDS directly into a ring of NS
// stages; 16-byte chunk c of row r lies at slot c ^ (r & 7), so the 16 rows of a fragment read touch distinct
// banks. w is the MFMA's first operand: a lane's four accumulators are four consecutive columns of one row.
// The 64-row tile takes grids that 128-row tiles would leave below one workgroup per CU. A form without LDS,
// one 16 x 16 tile a wave, took 61 us for 256 x 4096 x 4096. The linear with both quantizers: 132 us so and 29 now
// at that size (39 before w8a8_tile_of below and the one quantizer launch); at 2048 x 4096 x 4096 536 and 94 us, at
// 1024 x 14336 x 4096 976 and 192, both before those two.
// ----------------------------------------------------------------------------------------------
typedef int i32x4_t __attribute__((__vector_size__(4 * sizeof(int))));

// Output tile (tm, tn) of workgroup `bid`. Workgroup b runs on XCD b % 8, each with its own L2: an XCD takes a
// contiguous range of the walk, which goes through column tiles in groups of kW8GroupM row tiles, so the 32 CUs of an
// XCD share their rows of x and of w (4 x 8 or 8 x 4 tiles; with workgroup b on tile b an XCD held one row tile and 32
// column tiles, and every row of w went to four L2s). The product alone, 256 / 500 x 4096 x 4096: 22.3 -> 15.5 and
// 25.1 -> 18.3 us. A single row tile shares no row of w: there the walk in order is the better one
// (64 x 28672 x 4096: 32.4 us against 33.1).
constexpr int kW8GroupM = 8;
__device__ inline void w8a8_tile_of(int bid, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int total = tiles_m * tiles_n, per = total >> 3, rem = total & 7, xcd = bid & 7;
  // the first `rem` XCDs have one tile more
  const int lin = tiles_m == 1 ? bid : xcd * per + min(xcd, rem) + (bid >> 3);
  const int per_group = kW8GroupM * tiles_n;
  const int g = lin / per_group, r = lin - g * per_group;
  const int gm = min(tiles_m - g * kW8GroupM, kW8GroupM);
  tm = g * kW8GroupM + r % gm;
  tn = r / gm;
}

template <int PD, int T, int NS>
__global__ __launch_bounds__(256, 2) void w8a8_kernel(const int8_t* __restrict__ qx, const int8_t* __restrict__ qw,
                                                   const void* __restrict__ sx, int sx_dt, const void* __restrict__ sw,
                                                   int sw_dt, float* __restrict__ y, int M, int N, int K, int tiles_m,
                                                   int tiles_n) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem8[];
  constexpr int kStage = 2 * T * 128;   // x rows, then w rows
  constexpr int CPW = 2 * T / 8 / 4;    // 1 KiB copies (8 rows) per wave and stage
  constexpr int F = T / 32;             // 16-row fragments of either operand per wave
  constexpr uint32_t kNone = 0x80000000u;  // past either buffer (both below 2 GiB): zeros, no memory traffic
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int tm, tn;
  w8a8_tile_of(static_cast<int>(blockIdx.x), tiles_m, tiles_n, tm, tn);
  const int m0 = tm * T, n0 = tn * T;
  const rsrc_t xr = make_rsrc(qx, (uint32_t)M * (uint32_t)K);
  const rsrc_t wr = make_rsrc(qw, (uint32_t)N * (uint32_t)K);
  const bool is_w = wave >= 2;  // waves 0, 1 copy x's rows, 2, 3 w's
  const rsrc_t cr = is_w ? wr : xr;
  const int lim = is_w ? N - n0 : M - m0;
  const uint32_t row_base = (uint32_t)(is_w ? n0 : m0) * (uint32_t)K;
  const int S = (K + 127) / 128;
  auto issue = [&](int s, int slot) {
    uint8_t* dst = smem8 + slot * kStage + wave * CPW * 1024;
#pragma unroll
    for (int j = 0; j < CPW; ++j) {
      const int r = ((wave & 1) * CPW + j) * 8 + (lane >> 3);
      const int c = 128 * s + 16 * ((lane & 7) ^ (r & 7));
      const uint32_t off = (r < lim) & (c < K) ? row_base + (uint32_t)r * (uint32_t)K + (uint32_t)c : kNone;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(cr, (lds_void*)(dst + j * 1024), 16, off, 0, 0, 0);
    }
  };
  i32x4_t acc[F][F];
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) acc[i][j] = i32x4_t{0, 0, 0, 0};
  const int wm = (wave >> 1) * (T / 2), wn = (wave & 1) * (T / 2);
  const int r = lane & 15, g = lane >> 4;
#pragma unroll
  for (int s = 0; s < NS - 1; ++s)
    if (s < S) issue(s, s);
  int slot = 0;
  for (int s = 0; s < S; ++s) {
    // stage s has landed for this wave (the NS - 2 after it may be in flight), then for all; every wave has also
    // read stage s - 1 (its MFMAs waited for the reads), whose slot the next copies take
    if (s + NS - 2 < S) wait_vmcnt<CPW * (NS - 2)>();
    else wait_vmcnt<0>();
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (s + NS - 1 < S) issue(s + NS - 1, slot == 0 ? NS - 1 : slot - 1);
    const uint8_t* xb = smem8 + slot * kStage;
    const uint8_t* wb = xb + T * 128;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u32x4_t a[F], b[F];
      const int sl = ((4 * h + g) ^ (r & 7)) * 16;
#pragma unroll
      for (int i = 0; i < F; ++i) a[i] = *reinterpret_cast<const u32x4_t*>(xb + (wm + 16 * i + r) * 128 + sl);
#pragma unroll
      for (int i = 0; i < F; ++i) b[i] = *reinterpret_cast<const u32x4_t*>(wb + (wn + 16 * i + r) * 128 + sl);
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4_t, b[j]),
                                                            __builtin_bit_cast(i32x4_t, a[i]), acc[i][j], 0, 0, 0);
    }
    slot = slot == NS - 1 ? 0 : slot + 1;
  }
  // acc[i][j][e] is y[m0 + wm + 16i + (l & 15)][n0 + wn + 16j + 4(l >> 4) + e]
  const bool vec = N % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
#pragma unroll
  for (int i = 0; i < F; ++i) {
    const int m = m0 + wm + 16 * i + r;
    if (m >= M) continue;
    const float sm = load_as_f32(sx, sx_dt, m);
#pragma unroll
    for (int j = 0; j < F; ++j) {
      const int n = n0 + wn + 16 * j + 4 * g;
      if (n >= N) continue;
      f32x4_t v;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[e] = static_cast<float>(acc[i][j][e]) * rd<PD>(sm * load_as_f32(sw, sw_dt, min(n + e, N - 1)));
      float* dst = y + (int64_t)m * N + n;
      if (vec) {
        *reinterpret_cast<f32x4_t*>(dst) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) dst[e] = v[e];
      }
    }
  }
}

// The same product for rows that are not a multiple of 16 bytes: one wave per 16 x 16 tile, element loads.
template <int PD>
__global__ __launch_bounds__(256) void w8a8_ragged_kernel(const int8_t* __restrict__ qx, const int8_t* __restrict__ qw,
                                                          const void* __restrict__ sx, int sx_dt,
                                                          const void* __restrict__ sw, int sw_dt, float* __restrict__ y,
                                                          int M, int N, int K) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int m0 = blockIdx.y * 32 + (wave >> 1) * 16;
  const int n0 = blockIdx.x * 32 + (wave & 1) * 16;
  const int r = lane & 15, g = lane >> 4;
  const int am = m0 + r, bn = n0 + r;
  i32x4_t acc = {0, 0, 0, 0};
  for (int k0 = 0; k0 < K; k0 += 64) {
    const int kk = k0 + 16 * g;
    uint32_t av[4] = {0u, 0u, 0u, 0u}, bv[4] = {0u, 0u, 0u, 0u};
    for (int e = 0; e < 16; ++e) {
      if (kk + e < K) {
        if (am < M) av[e >> 2] |= static_cast<uint32_t>(static_cast<uint8_t>(qx[(int64_t)am * K + kk + e])) << (8 * (e & 3));
        if (bn < N) bv[e >> 2] |= static_cast<uint32_t>(static_cast<uint8_t>(qw[(int64_t)bn * K + kk + e])) << (8 * (e & 3));
      }
    }
    const u32x4_t a = {av[0], av[1], av[2], av[3]}, b = {bv[0], bv[1], bv[2], bv[3]};
    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4_t, a), __builtin_bit_cast(i32x4_t, b), acc,
                                                0, 0, 0);
  }
  const int n = n0 + r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + 4 * g + i;
    if (m < M && n < N) {
      const float p = rd<PD>(load_as_f32(sx, sx_dt, m) * load_as_f32(sw, sw_dt, n));
      y[(int64_t)m * N + n] = static_cast<float>(acc[i]) * p;
    }
  }
}

// ----------------------------------------------------------------------------------------------
// Int8 weight-only linear: the GEMV policy
// ----------------------------------------------------------------------------------------------
struct WInt8 {
  static constexpr int KBLK = 64, STEPS = 2;
  struct Args {
    const uint8_t* wt;
    const float* scale;  // [rows] fp32
  };
  struct Ctx {
    rsrc_t wr;
    uint32_t wvo;
  };
  struct P {};
  __device__ static Ctx ctx(const Args& a, int t, int KB, int lane) {
    return Ctx{make_rsrc(a.wt + (int64_t)t * KB * 1024, (uint32_t)KB * 1024u), (uint32_t)lane * 16u};
  }
  __device__ static void load(const Ctx& c, int kb, u32x4_t& w, P&) { w = bload128<2>(c.wr, c.wvo, (uint32_t)kb * 1024u); }
  __device__ static int xk(int i, int jg) { return 16 * jg + 8 * i; }
  template <class A, int MCH>
  __device__ static void mma(const u32x4_t& w, const P&, const u32x4_t (&xv)[MCH][STEPS], f32x4_t (&yacc)[MCH]) {
    const uint32_t off = A::pair_from_f32(-128.0f);
    const u32x4_t boff = u32x4_t{off, off, off, off};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t d0 = w[2 * i], d1 = w[2 * i + 1];
      const u32x4_t b = {A::pack_exact(ubyte_f32<0>(d0), ubyte_f32<1>(d0)), A::pack_exact(ubyte_f32<2>(d0), ubyte_f32<3>(d0)),
                         A::pack_exact(ubyte_f32<0>(d1), ubyte_f32<1>(d1)), A::pack_exact(ubyte_f32<2>(d1), ubyte_f32<3>(d1))};
#pragma unroll
      for (int c = 0; c < MCH; ++c) {
        yacc[c] = A::mfma(xv[c][i], b, yacc[c]);
        yacc[c] = A::mfma(xv[c][i], boff, yacc[c]);
      }
    }
  }
  // One activation row (the GEMV's ONE form): the code chains only, with the offset -128 charged
  // through the block's activation sum sig[0].
  static constexpr bool kSumOffset = true;
  static constexpr int NG = 1;
  template <class A>
  __device__ static void mma_one(const u32x4_t& w, const P&, const u32x4_t (&xv)[STEPS], const float (&sig)[NG],
                                 float& y0) {
    f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t d0 = w[2 * i], d1 = w[2 * i + 1];
      const u32x4_t b = {A::pack_exact(ubyte_f32<0>(d0), ubyte_f32<1>(d0)), A::pack_exact(ubyte_f32<2>(d0), ubyte_f32<3>(d0)),
                         A::pack_exact(ubyte_f32<0>(d1), ubyte_f32<1>(d1)), A::pack_exact(ubyte_f32<2>(d1), ubyte_f32<3>(d1))};
      acc = A::mfma(xv[i], b, acc);
    }
    y0 += fmaf(-128.0f, sig[0], acc[0]);
  }
  __device__ static float out_scale(const Args& a, int n) { return a.scale[n]; }

  // The row-tiled kernels' hooks (sqx_skinny.h): the codes as their signed values, exact in bf16 and fp16, so a
  // block's MFMAs chain straight into the output sums.
  static constexpr int MPG = STEPS;
  static constexpr bool kPlainBlocks = true, kConstOffset = true;
  __device__ static Ctx ctx_tiles(const Args& a, int t, int nt, int KB, int lane) {
    return Ctx{make_rsrc(a.wt + (int64_t)t * KB * 1024, (uint32_t)nt * (uint32_t)KB * 1024u), (uint32_t)lane * 16u};
  }
  template <class A>
  __device__ static u32x4_t bfrag(const u32x4_t& w, int i) {
    const uint32_t d0 = w[2 * i] ^ 0x80808080u, d1 = w[2 * i + 1] ^ 0x80808080u;  // q + 128 -> two's complement
    return u32x4_t{A::pack_exact(sbyte_f32<0>(d0), sbyte_f32<1>(d0)), A::pack_exact(sbyte_f32<2>(d0), sbyte_f32<3>(d0)),
                   A::pack_exact(sbyte_f32<0>(d1), sbyte_f32<1>(d1)), A::pack_exact(sbyte_f32<2>(d1), sbyte_f32<3>(d1))};
  }
  template <class A>
  __device__ static float const_offset() { return 0.0f; }
  template <class A>
  __device__ static float offset(const P&, int) { return 0.0f; }
  __device__ static float scale(const P&, int) { return 1.0f; }
  static const float* out_scales(const Args& a) { return a.scale; }
};

// One thread per output dword of the tiled int8 weight. vec: the four codes are one aligned dword.
__global__ __launch_bounds__(256) void int8_tile_kernel(const int8_t* __restrict__ q, int64_t rows, int64_t cols,
                                                        int64_t KB, int64_t n_dwords, uint32_t* __restrict__ wt, int vec) {
  const int64_t d = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= n_dwords) return;
  const int i = static_cast<int>(d & 3);
  const int L = static_cast<int>((d >> 2) & 63);
  const uint32_t blk = static_cast<uint32_t>(d >> 8);  // blocks of 1 KiB: below 2**32
  const int64_t t = blk / static_cast<uint32_t>(KB);
  const int64_t kb = blk - t * KB;
  const int64_t r = 16 * t + (L & 15);
  const int64_t c0 = kb * 64 + 16 * (L >> 4) + 4 * i;
  uint32_t word = 0;
  if (vec && r < rows && c0 + 4 <= cols) {
    word = *reinterpret_cast<const uint32_t*>(q + r * cols + c0) ^ 0x80808080u;  // q + 128 in every byte
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t c = c0 + e;
      const uint32_t u = (r < rows && c < cols) ? static_cast<uint32_t>(q[r * cols + c] + 128) : 128u;
      word |= (u & 0xffu) << (8 * e);
    }
  }
  wt[d] = word;
}

// The inverse re-layout: one thread per tiled dword writes its 4 codes back to q [rows, cols].
__global__ __launch_bounds__(256) void int8_untile_kernel(const uint32_t* __restrict__ wt, int64_t rows, int64_t cols,
                                                          int64_t KB, int64_t n_dwords, int8_t* __restrict__ q) {
  const int64_t d = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= n_dwords) return;
  const int i = static_cast<int>(d & 3);
  const int L = static_cast<int>((d >> 2) & 63);
  const int64_t blk = d >> 8;
  const int64_t t = blk / KB;
  const int64_t kb = blk - t * KB;
  const int64_t r = 16 * t + (L & 15);
  if (r >= rows) return;
  const int64_t c0 = kb * 64 + 16 * (L >> 4) + 4 * i;
  const uint32_t word = wt[d];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int64_t c = c0 + e;
    if (c < cols) q[r * cols + c] = static_cast<int8_t>(static_cast<int>((word >> (8 * e)) & 0xffu) - 128);
  }
}

}  // namespace sqx

using namespace sqx;

// ==============================================================================================
// extern "C" entry points
// ==============================================================================================
static bool is_float_dtype(int d) { return d == SQX_DTYPE_F32 || d == SQX_DTYPE_BF16 || d == SQX_DTYPE_F16; }
static dim3 grid_for(int64_t n) { return dim3(static_cast<unsigned>(ceil_div(n, 256))); }

template <int OP>
static int int8_stats(const void* x, int dtype, int64_t A, int64_t B, int64_t C, float eps, void* s, void* z,
                      void* workspace, int64_t workspace_bytes, hipStream_t st, const char* fn) {
  const int64_t n = A * B * C;
  const bool per_tensor = B == 1;
  if (per_tensor) {
    SQX_REQUIRE(workspace && workspace_bytes >= (int64_t)kStatParts * 8, SQX_E_SPACE,
                "%s: a per-tensor scale needs a workspace of %d bytes", fn, kStatParts * 8);
    const int parts = n == 0 ? 1 : static_cast<int>(std::min<int64_t>(kStatParts, ceil_div(n, 256)));
    float* part = static_cast<float*>(workspace);
#define SQX_PT(DT)                                                                                                   \
  do {                                                                                                               \
    if (n > 0) hipLaunchKernelGGL((stats_partial_kernel<DT, OP>), dim3(parts), dim3(256), 0, st, x, n, part);        \
    hipLaunchKernelGGL((stats_final_kernel<DT, OP>), dim3(1), dim3(256), 0, st, part, n > 0 ? parts : 0, eps, s, z); \
  } while (0)
    if (dtype == SQX_DTYPE_F32) SQX_PT(SQX_DTYPE_F32);
    else if (dtype == SQX_DTYPE_BF16) SQX_PT(SQX_DTYPE_BF16);
    else SQX_PT(SQX_DTYPE_F16);
#undef SQX_PT
    return SQX_OK;
  }
  const bool wg = C >= 32 || A * C >= 4096;
#define SQX_AX(DT)                                                                                                   \
  do {                                                                                                               \
    if (wg) hipLaunchKernelGGL((stats_wg_kernel<DT, OP>), dim3(static_cast<unsigned>(B)), dim3(256), 0, st, x, A, B, \
                               C, eps, s, z);                                                                        \
    else hipLaunchKernelGGL((stats_thread_kernel<DT, OP>), grid_for(B), dim3(256), 0, st, x, A, B, C, eps, s, z);   \
  } while (0)
  if (dtype == SQX_DTYPE_F32) SQX_AX(SQX_DTYPE_F32);
  else if (dtype == SQX_DTYPE_BF16) SQX_AX(SQX_DTYPE_BF16);
  else SQX_AX(SQX_DTYPE_F16);
#undef SQX_AX
  return SQX_OK;
}

extern "C" int64_t sqx_int8_workspace_bytes(void) { return (int64_t)kStatParts * 8; }

// One pass over the B rows of x (from row B1 on: of x2), for rows of whole 8-element chunks that fit a workgroup's
// registers. A workgroup a row pays from 64 columns on (the affine form, with its two statistics, from 128), and for
// as few rows as the chip holds workgroups at once: more rows that are shorter leave most lanes idle (bf16, one pass
// against two: 300000 x 16 230 and 22 us, 65536 x 32 51 and 49, 262144 x 64 201 and 215, affine 275 and 261;
// 1000 x 24 4.2 and 6.4). A launch holds fewer than 2**32 threads.
constexpr int64_t kQuantRowsMaxC = 16 * 2048;
static bool quantize_rows_fits(int64_t B, int64_t C, bool affine) {
  return C % 8 == 0 && C <= kQuantRowsMaxC && B < ((int64_t)1 << 24) && (C >= (affine ? 128 : 64) || B <= 2048);
}
template <int OP>
static void launch_quantize_rows(const void* x, const void* x2, int64_t B1, int64_t B, int dtype, int64_t C, float eps,
                                 uint8_t* q, void* s, void* z, hipStream_t st) {
  const dim3 grid(static_cast<unsigned>(B));
#define SQX_QR(DT, N) \
  hipLaunchKernelGGL((quantize_rows_kernel<DT, OP, N>), grid, dim3(256), 0, st, x, x2, B1, C, eps, s, z, q)
#define SQX_QRN(DT)                     \
  do {                                  \
    if (C <= 2048) SQX_QR(DT, 1);       \
    else if (C <= 4096) SQX_QR(DT, 2);  \
    else if (C <= 8192) SQX_QR(DT, 4);  \
    else if (C <= 16384) SQX_QR(DT, 8); \
    else SQX_QR(DT, 16);                \
  } while (0)
  if (dtype == SQX_DTYPE_F32) SQX_QRN(SQX_DTYPE_F32);
  else if (dtype == SQX_DTYPE_BF16) SQX_QRN(SQX_DTYPE_BF16);
  else SQX_QRN(SQX_DTYPE_F16);
#undef SQX_QRN
#undef SQX_QR
}

template <int OP>
static int int8_quantize(const void* x, int dtype, int64_t A, int64_t B, int64_t C, float eps, uint8_t* q, void* s,
                         void* z, void* workspace, int64_t workspace_bytes, sqx_stream_t stream, const char* fn) {
  SQX_REQUIRE(is_float_dtype(dtype), SQX_E_ARG, "%s: unsupported dtype %d", fn, dtype);
  SQX_REQUIRE(A >= 1 && B >= 1 && C >= 1 && A * B * C < ((int64_t)1 << 40), SQX_E_ARG, "%s: bad view [%lld, %lld, %lld]",
              fn, (long long)A, (long long)B, (long long)C);
  SQX_REQUIRE(x && q && s && (OP == 0 || z), SQX_E_ARG, "%s: null pointer", fn);
  SQX_REQUIRE(B == 1 || B < ((int64_t)1 << 31), SQX_E_ARG, "%s: kept axis too long", fn);
  hipStream_t st = as_stream(stream);
  if (A == 1 && B > 1 && quantize_rows_fits(B, C, OP == 1) && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
      reinterpret_cast<uintptr_t>(q) % 8 == 0) {
    launch_quantize_rows<OP>(x, nullptr, B, B, dtype, C, eps, q, s, z, st);
    SQX_LAUNCH_CHECK(fn);
    return SQX_OK;
  }
  int rc = int8_stats<OP>(x, dtype, A, B, C, eps, s, z, workspace, workspace_bytes, st, fn);
  if (rc) return rc;
  const int64_t n = A * B * C;
  if (n > 0) {
    if (dtype == SQX_DTYPE_F32)
      hipLaunchKernelGGL((quantize_kernel<SQX_DTYPE_F32, OP>), grid_for(n), dim3(256), 0, st, x, n, B, C, s, z, q);
    else if (dtype == SQX_DTYPE_BF16)
      hipLaunchKernelGGL((quantize_kernel<SQX_DTYPE_BF16, OP>), grid_for(n), dim3(256), 0, st, x, n, B, C, s, z, q);
    else
      hipLaunchKernelGGL((quantize_kernel<SQX_DTYPE_F16, OP>), grid_for(n), dim3(256), 0, st, x, n, B, C, s, z, q);
  }
  SQX_LAUNCH_CHECK(fn);
  return SQX_OK;
}

extern "C" int sqx_int8_quantize_sym(const void* x, int dtype, int64_t A, int64_t B, int64_t C, float eps,
                                     int8_t* q, void* s, void* workspace, int64_t workspace_bytes,
                                     sqx_stream_t stream) {
  return int8_quantize<0>(x, dtype, A, B, C, eps, reinterpret_cast<uint8_t*>(q), s, nullptr, workspace,
                          workspace_bytes, stream, "sqx_int8_quantize_sym");
}

extern "C" int sqx_int8_quantize_affine(const void* x, int dtype, int64_t A, int64_t B, int64_t C, float eps,
                                        uint8_t* q, void* s, void* z, void* workspace, int64_t workspace_bytes,
                                        sqx_stream_t stream) {
  return int8_quantize<1>(x, dtype, A, B, C, eps, q, s, z, workspace, workspace_bytes, stream,
                          "sqx_int8_quantize_affine");
}

template <int OP>
static int int8_dequantize(const uint8_t* q, int64_t A, int64_t B, int64_t C, const void* s, const void* z, int dtype,
                           void* out, sqx_stream_t stream, const char* fn) {
  SQX_REQUIRE(is_float_dtype(dtype), SQX_E_ARG, "%s: unsupported dtype %d", fn, dtype);
  SQX_REQUIRE(A >= 1 && B >= 1 && C >= 1, SQX_E_ARG, "%s: bad view", fn);
  const int64_t n = A * B * C;
  SQX_REQUIRE(q && s && out && (OP == 0 || z), SQX_E_ARG, "%s: null pointer", fn);
  hipStream_t st = as_stream(stream);
  if (dtype == SQX_DTYPE_F32)
    hipLaunchKernelGGL((dequantize_kernel<SQX_DTYPE_F32, OP>), grid_for(n), dim3(256), 0, st, q, n, B, C, s, z, out);
  else if (dtype == SQX_DTYPE_BF16)
    hipLaunchKernelGGL((dequantize_kernel<SQX_DTYPE_BF16, OP>), grid_for(n), dim3(256), 0, st, q, n, B, C, s, z, out);
  else
    hipLaunchKernelGGL((dequantize_kernel<SQX_DTYPE_F16, OP>), grid_for(n), dim3(256), 0, st, q, n, B, C, s, z, out);
  SQX_LAUNCH_CHECK(fn);
  return SQX_OK;
}

extern "C" int sqx_int8_dequantize_sym(const int8_t* q, int64_t A, int64_t B, int64_t C, const void* s, int dtype,
                                       void* out, sqx_stream_t stream) {
  return int8_dequantize<0>(reinterpret_cast<const uint8_t*>(q), A, B, C, s, nullptr, dtype, out, stream,
                            "sqx_int8_dequantize_sym");
}

extern "C" int sqx_int8_dequantize_affine(const uint8_t* q, int64_t A, int64_t B, int64_t C, const void* s,
                                          const void* z, int dtype, void* out, sqx_stream_t stream) {
  return int8_dequantize<1>(q, A, B, C, s, z, dtype, out, stream, "sqx_int8_dequantize_affine");
}

extern "C" int sqx_w8a8_gemm(const int8_t* qx, const void* sx, int sx_dtype, const int8_t* qw, const void* sw,
                             int sw_dtype, float* y, int64_t m, int64_t n, int64_t k, sqx_stream_t stream) {
  SQX_REQUIRE(is_float_dtype(sx_dtype) && is_float_dtype(sw_dtype), SQX_E_ARG, "sqx_w8a8_gemm: bad scale dtype");
  SQX_REQUIRE(m >= 0 && n >= 0 && k >= 1 && m * k < ((int64_t)1 << 31) && n * k < ((int64_t)1 << 31), SQX_E_ARG,
              "sqx_w8a8_gemm: bad shape m=%lld n=%lld k=%lld", (long long)m, (long long)n, (long long)k);
  SQX_REQUIRE(ceil_div(m, 64) * ceil_div(n, 64) < ((int64_t)1 << 31), SQX_E_ARG, "sqx_w8a8_gemm: too many output tiles");
  SQX_REQUIRE(k <= 131072, SQX_E_ARG, "sqx_w8a8_gemm: k=%lld may overflow the int32 accumulator", (long long)k);
  if (m == 0 || n == 0) return SQX_OK;
  SQX_REQUIRE(qx && sx && qw && sw && y, SQX_E_ARG, "sqx_w8a8_gemm: null pointer");
  SQX_REQUIRE(k % 16 != 0 || (reinterpret_cast<uintptr_t>(qx) % 16 == 0 && reinterpret_cast<uintptr_t>(qw) % 16 == 0),
              SQX_E_ARG, "sqx_w8a8_gemm: qx and qw must be 16-byte aligned");
  // the scale product is taken in the promoted dtype of the two scales (torch type promotion)
  const int pd = sx_dtype == sw_dtype ? sx_dtype : SQX_DTYPE_F32;
  hipStream_t st = as_stream(stream);
  const int M = static_cast<int>(m), N = static_cast<int>(n), K = static_cast<int>(k);
  hipError_t e = hipSuccess;
  auto go = [&](auto kern, int T, int stages) {
    const int64_t tm = ceil_div(m, T), tn = ceil_div(n, T);
    const int lds = stages * 2 * T * 128;
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e == hipSuccess)
      hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(tm * tn)), dim3(256), static_cast<size_t>(lds), st, qx, qw, sx,
                         sx_dtype, sw, sw_dtype, y, M, N, K, static_cast<int>(tm), static_cast<int>(tn));
  };
  // 128 x 128 tiles once they fill the 256 CUs (1024 x 4096 x 4096), 64 x 64 below
  const bool big = ceil_div(m, 128) * ceil_div(n, 128) >= 256;
#define SQX_W8(PD)                                                                                                    \
  do {                                                                                                                \
    if (k % 16 != 0)                                                                                                  \
      hipLaunchKernelGGL(w8a8_ragged_kernel<PD>,                                                                       \
                         dim3(static_cast<unsigned>(ceil_div(n, 32)), static_cast<unsigned>(ceil_div(m, 32))), dim3(256), \
                         0, st, qx, qw, sx, sx_dtype, sw, sw_dtype, y, M, N, K);                                       \
    else if (big) go(w8a8_kernel<PD, 128, 4>, 128, 4);                                                                 \
    else go(w8a8_kernel<PD, 64, 4>, 64, 4);                                                                            \
  } while (0)
  if (pd == SQX_DTYPE_F32) SQX_W8(SQX_DTYPE_F32);
  else if (pd == SQX_DTYPE_BF16) SQX_W8(SQX_DTYPE_BF16);
  else SQX_W8(SQX_DTYPE_F16);
#undef SQX_W8
  SQX_REQUIRE(e == hipSuccess, SQX_E_HIP, "sqx_w8a8_gemm: launch failed: %s", hipGetErrorString(e));
  SQX_LAUNCH_CHECK("sqx_w8a8_gemm");
  return SQX_OK;
}

extern "C" int64_t sqx_w8a8_workspace_bytes(int64_t m, int64_t n, int64_t k) {
  // int8 rows of x, then of w, then their scales (at most fp32)
  return k > 0 && k % 16 == 0 && m > 0 && n > 0 && quantize_rows_fits(m + n, k, false) && m * k < ((int64_t)1 << 31) &&
                 n * k < ((int64_t)1 << 31)
             ? (m + n) * (k + 4)
             : -1;
}

extern "C" int sqx_w8a8_linear(const void* x, const void* w, int dtype, float eps, float* y, int64_t m, int64_t n, int64_t k,
                               void* ws, int64_t ws_bytes, sqx_stream_t stream) {
  SQX_REQUIRE(is_float_dtype(dtype), SQX_E_ARG, "sqx_w8a8_linear: unsupported dtype %d", dtype);
  const int64_t need = sqx_w8a8_workspace_bytes(m, n, k);
  SQX_REQUIRE(need > 0, SQX_E_ARG, "sqx_w8a8_linear: bad shape m=%lld n=%lld k=%lld (sqx_w8a8_workspace_bytes is -1)",
              (long long)m, (long long)n, (long long)k);
  SQX_REQUIRE(x && w && y && ws, SQX_E_ARG, "sqx_w8a8_linear: null pointer");
  SQX_REQUIRE(ws_bytes >= need, SQX_E_SPACE, "sqx_w8a8_linear: the workspace needs %lld bytes", (long long)need);
  SQX_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(ws) % 16 == 0,
              SQX_E_ARG, "sqx_w8a8_linear: x, w and the workspace must be 16-byte aligned");
  auto* q = static_cast<uint8_t*>(ws);
  uint8_t* s = q + (m + n) * k;
  launch_quantize_rows<0>(x, w, m, m + n, dtype, k, eps, q, s, nullptr, as_stream(stream));
  SQX_LAUNCH_CHECK("sqx_w8a8_linear");
  return sqx_w8a8_gemm(reinterpret_cast<const int8_t*>(q), s, dtype, reinterpret_cast<const int8_t*>(q + m * k),
                       s + m * (dtype == SQX_DTYPE_F32 ? 4 : 2), dtype, y, m, n, k, stream);
}

extern "C" int64_t sqx_int8_tiled_weight_bytes(int64_t rows, int64_t cols) {
  if (rows < 0 || cols < 0) return -1;
  return ceil_div(rows, 16) * ceil_div(cols, 64) * 1024;
}

extern "C" int sqx_int8_tile(const int8_t* q, int64_t rows, int64_t cols, uint8_t* wt, sqx_stream_t stream) {
  SQX_REQUIRE(rows > 0 && cols > 0 && rows <= ((int64_t)1 << 30) && cols <= ((int64_t)1 << 30), SQX_E_ARG,
              "sqx_int8_tile: bad shape");
  SQX_REQUIRE(q && wt, SQX_E_ARG, "sqx_int8_tile: null pointer");
  const int64_t KB = ceil_div(cols, 64);
  const int64_t nd = ceil_div(rows, 16) * KB * 256;
  hipLaunchKernelGGL(int8_tile_kernel, grid_for(nd), dim3(256), 0, as_stream(stream), q, rows, cols, KB, nd,
                     reinterpret_cast<uint32_t*>(wt), cols % 4 == 0 && reinterpret_cast<uintptr_t>(q) % 4 == 0);
  SQX_LAUNCH_CHECK("sqx_int8_tile");
  return SQX_OK;
}

extern "C" int sqx_int8_untile(const uint8_t* wt, int64_t rows, int64_t cols, int8_t* q, sqx_stream_t stream) {
  SQX_REQUIRE(rows > 0 && cols > 0 && rows <= ((int64_t)1 << 30) && cols <= ((int64_t)1 << 30), SQX_E_ARG,
              "sqx_int8_untile: bad shape");
  SQX_REQUIRE(q && wt, SQX_E_ARG, "sqx_int8_untile: null pointer");
  const int64_t KB = ceil_div(cols, 64);
  const int64_t nd = ceil_div(rows, 16) * KB * 256;
  hipLaunchKernelGGL(int8_untile_kernel, grid_for(nd), dim3(256), 0, as_stream(stream),
                     reinterpret_cast<const uint32_t*>(wt), rows, cols, KB, nd, q);
  SQX_LAUNCH_CHECK("sqx_int8_untile");
  return SQX_OK;
}

extern "C" int sqx_int8_linear(const uint8_t* wt, const float* scale, const void* x, int act_dtype, void* y,
                               const void* bias, int64_t m, int64_t rows, int64_t cols, int k_slices,
                               sqx_stream_t stream) {
  SQX_REQUIRE(m >= 0 && rows > 0 && cols > 0, SQX_E_ARG, "sqx_int8_linear: bad shape");
  SQX_REQUIRE(act_dtype == SQX_DTYPE_BF16 || act_dtype == SQX_DTYPE_F16, SQX_E_ARG,
              "sqx_int8_linear: activations must be BF16 or F16");
  SQX_REQUIRE(rows < ((int64_t)1 << 31) && ceil_div(cols, 64) * 1024 < ((int64_t)1 << 31) && 64 * cols * 2 < ((int64_t)1 << 31),
              SQX_E_ARG, "sqx_int8_linear: shape too large for 32-bit buffer offsets");
  SQX_REQUIRE(cols % 8 == 0, SQX_E_ARG, "sqx_int8_linear: cols=%lld must be a multiple of 8", (long long)cols);
  SQX_REQUIRE(k_slices <= 16, SQX_E_ARG, "sqx_int8_linear: k_slices %d > 16", k_slices);
  if (m == 0) return SQX_OK;
  SQX_REQUIRE(wt && scale && x && y, SQX_E_ARG, "sqx_int8_linear: null pointer");
  SQX_REQUIRE(reinterpret_cast<uintptr_t>(wt) % 16 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0, SQX_E_ARG,
              "sqx_int8_linear: wt and x must be 16-byte aligned");
  const WInt8::Args a{wt, scale};
  hipError_t e;
  if (act_dtype == SQX_DTYPE_BF16)
    e = gemv_launch<ActBF16, WInt8, 4, 2, false>(a, static_cast<const uint16_t*>(x), y,
                                                 static_cast<const uint16_t*>(bias), nullptr, m, rows, cols, k_slices,
                                                 as_stream(stream));
  else
    e = gemv_launch<ActF16, WInt8, 4, 2, false>(a, static_cast<const uint16_t*>(x), y,
                                                static_cast<const uint16_t*>(bias), nullptr, m, rows, cols, k_slices,
                                                as_stream(stream));
  SQX_REQUIRE(e == hipSuccess, SQX_E_HIP, "sqx_int8_linear: launch failed: %s", hipGetErrorString(e));
  return SQX_OK;
}

// The launch for 2..64 rows: FP8's, but for 257..383 tiles to K = 12288 in one piece of 2 tiles x 8 waves (4096 -> 5120 at
// m = 16: 12.3 us with the GEMV, 9.9 so) and for the shapes where the call is the faster one with the GEMV. FP8 quantizes
// its rows in a launch of its own first and its GEMV has no such head start, so its lines are not int8's. A call from
// Python takes no less than its host time, 13 us with the GEMV and 17.6 us with a split (the workspace and the second
// launch), so the lines compare max(host, kernel) first and the kernels alone second. From a sweep of bf16 activations at
// 2..64 rows, 512..28672 weight rows and 512..14336 columns (kernels, us, GEMV and row-tiled): 512 -> 512 at m = 17 / 64
// 4.0 / 5.9 and 7.5 / 9.8; 1536 -> 3072 at m = 33 6.9 and 13.4; 4096 -> 16384 at m = 2 13.0 and 16.0; 2048 -> 2048 at
// m = 64 10.4 and 9.7, a split; 4096 -> 4096 at m = 24 / 64 9.8 / 18.2 and 10.1 / 15.4.
static constexpr GemvUntil kInt8Gemv[] = {
    { 128, {kG, kG, kG, kG, kG, kG, 28, 22, 18, 11, 10}},
    { 256, {kG, kG, kG, kG, kG, kG, 28, 22, 16, 16, 11}},
    { 383, {kG, kG, 24, 24, 12,  5,  5,  3,  3,  2,  0}},
    { 512, {kG, kG, kG, kG, 20,  5,  4,  3,  2,  2,  0}},
    { 639, {kG, kG, 10,  3,  3,  3,  3,  3,  3,  3,  3}},
    { 895, {kG, kG,  5,  4,  4,  4,  4,  3,  3,  4,  3}},
    {1023, {18, 14,  3,  3,  3,  2,  2,  2,  0,  2,  2}},
    {1199, {kG, kG, kG, kG,  5, kG,  7,  5,  3,  3,  2}},
    {1343, {kG, kG,  4,  3,  2, kG,  4,  4,  3,  3,  2}},
    {1919, {16,  5,  2,  2,  2,  3,  3,  2,  2,  0,  0}},
    {kAllTiles, { 2,  2,  0,  0,  0,  0,  0,  2,  0,  0,  0}}};
static SkinnyShape int8_default_shape(int64_t m, int64_t rows, int64_t cols) {
  SkinnyShape sh = skinny64_default_shape(m, rows, cols);
  const int64_t T = ceil_div(rows, 16);
  if (m >= 2 && m <= 64 && T > 256 && T < 384 && cols < 12288) sh = SkinnyShape{0, 2, 8, 1, false};
  if (gemv_ahead(kInt8Gemv, m, rows, cols)) sh.gemv = true;
  return sh;
}

extern "C" int64_t sqx_int8_skinny_workspace_bytes(int64_t m, int64_t rows, int64_t cols, int splits) {
  if (m <= 0 || m > 64 || rows <= 0 || cols <= 0) return 0;
  const SkinnyShape sh = int8_default_shape(m, rows, cols);
  const int S = splits > 0 ? splits : sh.gemv ? 1 : sh.S;
  return skinny_workspace_bytes(m, rows, skinny_splits(ceil_div(cols, 64), S));
}

extern "C" int sqx_int8_skinny_gemv(int64_t m, int64_t rows, int64_t cols) {
  return m > 0 && m <= 64 && rows > 0 && cols > 0 && int8_default_shape(m, rows, cols).gemv;
}

extern "C" int sqx_int8_skinny(const uint8_t* wt, const float* scale, const void* x, int act_dtype, void* y,
                               const void* bias, int64_t m, int64_t rows, int64_t cols, int tiles, int waves,
                               int splits, void* ws, int64_t ws_bytes, sqx_stream_t stream) {
  const char* fn = "sqx_int8_skinny";
  const bool choose = tiles <= 0 && waves <= 0 && splits <= 0;
  SkinnyShape sh = int8_default_shape(m, rows, cols);
  const int64_t KB = ceil_div(cols, 64);
  // the GEMV: the library's choice for the shape, or a row tile group beyond the 32-bit offsets
  if ((choose && sh.gemv) || 4 * KB * 1024 >= ((int64_t)1 << 31))
    return sqx_int8_linear(wt, scale, x, act_dtype, y, bias, m, rows, cols, 0, stream);
  if (!choose) sh = SkinnyShape{0, tiles > 0 ? tiles : 2, waves > 0 ? waves : 8, splits > 0 ? splits : 1, false};
  SQX_REQUIRE(m >= 1 && m <= 64 && rows > 0 && cols > 0 && cols % 8 == 0, SQX_E_ARG,
              "%s: bad shape m=%lld rows=%lld cols=%lld (1..64 rows, cols %% 8 == 0)", fn, (long long)m, (long long)rows,
              (long long)cols);
  SQX_REQUIRE(act_dtype == SQX_DTYPE_BF16 || act_dtype == SQX_DTYPE_F16, SQX_E_ARG, "%s: activations must be BF16 or F16",
              fn);
  SQX_REQUIRE(rows < ((int64_t)1 << 31) && 64 * cols * 2 < ((int64_t)1 << 31), SQX_E_ARG,
              "%s: shape too large for 32-bit buffer offsets", fn);
  SQX_REQUIRE(wt && scale && x && y, SQX_E_ARG, "%s: null pointer", fn);
  SQX_REQUIRE(reinterpret_cast<uintptr_t>(wt) % 16 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0, SQX_E_ARG,
              "%s: wt and x must be 16-byte aligned", fn);
  SQX_REQUIRE((sh.R == 2 || sh.R == 4) && sh.waves >= 1 && sh.waves <= kSkinnyMaxWaves, SQX_E_ARG,
              "%s: bad launch shape (tiles %d, waves %d, splits %d)", fn, sh.R, sh.waves, sh.S);
  const int S = skinny_splits(KB, sh.S);
  if (choose && S > 1 && (ws == nullptr || ws_bytes < skinny_workspace_bytes(m, rows, S))) sh.S = 1;
  else
    SQX_REQUIRE(S == 1 || (ws && ws_bytes >= skinny_workspace_bytes(m, rows, S)), SQX_E_SPACE,
                "%s: %d splits need a workspace of %lld bytes", fn, S, (long long)skinny_workspace_bytes(m, rows, S));
  const WInt8::Args a{wt, scale};
  const auto* xp = static_cast<const uint16_t*>(x);
  const auto* b16 = static_cast<const uint16_t*>(bias);
  auto* y16 = static_cast<uint16_t*>(y);
  auto* part = static_cast<float*>(ws);
  const hipError_t e =
      act_dtype == SQX_DTYPE_BF16
          ? skinny_launch<ActBF16, WInt8>(a, xp, y16, b16, m, rows, cols, sh, part, ws_bytes, as_stream(stream))
          : skinny_launch<ActF16, WInt8>(a, xp, y16, b16, m, rows, cols, sh, part, ws_bytes, as_stream(stream));
  SQX_REQUIRE(e == hipSuccess, SQX_E_HIP, "%s: launch failed: %s", fn, hipGetErrorString(e));
  return SQX_OK;
}
