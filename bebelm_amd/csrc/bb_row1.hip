// bb_row1.hip — one token's projections with what stands before and after them in the same launch.
//
// A decode step is a chain of small launches, each waiting for the one before: a layer boundary
// (residual, rmsnorm, Q8), a projection, the conv, its Q8, another projection. Each costs a launch
// and a memory round trip or two, about 4 us, whatever it computes. Here every block of a projection
// prepares the whole activation row itself while its weight rows are on their way (the row is 8 to
// 28 KB, read from L2; the weights come from HBM), so these launches fall away:
//   before   the residual add and rmsnorm of k_residual_norm (model.rs:105-130) and quantize_q8
//            (kernels/matmul.rs:141-160), or quantize_q8 alone
//   after    the short conv of the token's channels and its state (model.rs:399-427), or SwiGLU
//            (model.rs:464-466)
// One decode step of a six-layer model with its 128,000-row head: 401 -> 357 us (57 -> 40 launches);
// the conv operator alone 4 launches -> 2, 20.8 -> 12.5 us of kernels; gate/up with its boundary 9.8
// us against 4.2 + 7.4, down with its Q8 7.5 against 3.8 + 5.1.
// The launch is bound by latency, not bytes: 2 to 8 weight rows a wave (256 to 900 blocks for the
// model's matrices) time alike within 5%, one row or four 10% worse.
// Arithmetic and order are those of the kernels named: k_residual_norm's f64 sum (thread j's
// elements j, j + 256, ..., a butterfly, the four waves in a tree), k_rows_q8w's row values and
// left-to-right sum from -0.0 (one token: matvec, matmul.rs:850), k_conv_q8's conv.
#include "bb_device.h"
#include "bb_internal.h"

namespace bb {

namespace {

enum : int { KIND_ROWS = 0, KIND_CONV, KIND_SWIGLU };

// A lane's bytes of one row's super-block as loaded, so that nothing waits for them before the
// activations are ready: Q4_K as RowDot's, Q6_K the aligned dwords around its 2-byte aligned fields.
template <int DT>
struct Raw;
template <>
struct Raw<DT_Q4_K> {
  Q4kLane v;
  __device__ __forceinline__ void load(const uint8_t* block, int p) { v = q4k_load(block, p); }
  __device__ __forceinline__ Q4kLane lane() const { return v; }
};
template <>
struct Raw<DT_Q6_K> {
  uint32_t a[3], b[3], h[3], sc[3], d, sh;
  __device__ __forceinline__ void load(const uint8_t* block, int p) {
    const int n = p >> 2, l0 = 8 * (p & 3);
    const uintptr_t at = reinterpret_cast<uintptr_t>(block);  // every field starts 4k bytes after it
    const uint32_t* w = reinterpret_cast<const uint32_t*>(at & ~uintptr_t(3));
    sh = (uint32_t)(at & 3);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      a[k] = w[(64 * n + l0) / 4 + k];
      b[k] = w[(64 * n + 32 + l0) / 4 + k];
      h[k] = w[(128 + 32 * n + l0) / 4 + k];
      sc[k] = w[(192 + 8 * n) / 4 + k];
    }
    d = *reinterpret_cast<const uint16_t*>(block + 208);
  }
  __device__ __forceinline__ uint2 align(const uint32_t (&w)[3]) const {
    return make_uint2(__builtin_amdgcn_alignbyte(w[1], w[0], sh), __builtin_amdgcn_alignbyte(w[2], w[1], sh));
  }
  __device__ __forceinline__ Q6kLane lane() const { return {align(a), align(b), align(h), align(sc), d}; }
};

constexpr int R1_WAVES = 4;

// n <= NB * 256 activations in LDS. NORM rows also pass through f.
template <int NB>
struct Act {
  int8_t q[NB * QK];
  float sx[NB];
  int32_t sums[NB * 8];
};

__device__ __forceinline__ void quantize_lds(float4 v, int b, int8_t* q, float* sx, int32_t* sums) {
  const int lane = threadIdx.x & 63;
  float amax;
  int sum4;
  reinterpret_cast<uint32_t*>(q + b * QK)[lane] = wave_quantize(v, amax, sum4);
  const int s = sum8(sum4);
  if ((lane & 7) == 0) sums[b * 8 + (lane >> 3)] = s;
  if (lane == 0) sx[b] = amax / 127.0f;
}

// Block of R1_WAVES waves, RPW rows a wave, one matrix of jobs (its blocks jobs.first ..); a row's
// super-blocks over the wave's eight lane groups, J a group.
template <int DT, int KIND, bool NORM, int RPW, int J>
__device__ __forceinline__ void row1_body(const Row1In& in, const Row1Job& job, int block, int n, const Row1Conv& cv) {
  using R = RowDot<DT>;
  constexpr int NB = 8 * J;                       // super-blocks of a row at most
  constexpr int XB = NORM ? 1 : NB / R1_WAVES;    // super-blocks of x a wave quantises
  static_assert(!NORM || J == 1, "rmsnorm rows: at most GU_H_MAX");
  constexpr int ROWS = KIND == KIND_CONV ? 3 : KIND == KIND_SWIGLU ? 2 : 1;  // weight rows of one output
  constexpr int OPW = RPW / ROWS;                 // outputs of a wave
  __shared__ __align__(16) Act<NB> act;
  __shared__ __align__(16) float normed[NORM ? GU_H_MAX : 4];
  __shared__ double s_part[R1_WAVES];
  __shared__ float vals[R1_WAVES][RPW][NB];
  __shared__ uint64_t exptab[32];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 3, p = lane & 7;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nb = n / QK;
  const int o0 = (block * R1_WAVES + w) * OPW;    // the wave's first output
  const uint64_t exp_e = KIND == KIND_SWIGLU ? exp_table_entry() : 0;

  // the activation row first: its wait then leaves the weights in flight
  constexpr int NI = GU_H_MAX / 256;
  float hr[NORM ? NI : 1], yr[NORM ? NI : 1], gr[NORM ? NI : 1];
  float4 xv[XB];
  if constexpr (NORM) {
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      const int i = min(tid + 256 * it, n - 1);
      hr[it] = in.x[i];
      yr[it] = in.add ? in.add[i] : 0.0f;
      gr[it] = in.gain[i];
    }
  } else {
#pragma unroll
    for (int k = 0; k < XB; ++k)
      xv[k] = *reinterpret_cast<const float4*>(in.x + min(w + R1_WAVES * k, nb - 1) * QK + 4 * lane);
  }
  // the conv's taps and cache columns of the wave's channel (lane 3 ch + part: all three the same)
  float taps[KIND == KIND_CONV ? R1_L_MAX : 1], cols[KIND == KIND_CONV ? R1_L_MAX : 1];
  const int c_ch = KIND == KIND_CONV ? min(o0 + min(lane / 3, OPW - 1), job.n_rows - 1) : 0;
  if constexpr (KIND == KIND_CONV) {
#pragma unroll
    for (int k = 0; k < R1_L_MAX; ++k) {
      taps[k] = cv.w[(size_t)c_ch * cv.L + min(k, cv.L - 1)];
      cols[k] = cv.state[(size_t)min(k, cv.L - 2) * job.n_rows + c_ch];
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  Raw<DT> wl[RPW][J];
#pragma unroll
  for (int r = 0; r < RPW; ++r) {
    const int o = min(o0 + r / ROWS, job.n_rows - 1);  // (past the matrix: its last row again, not stored)
    const uint8_t* row = KIND == KIND_SWIGLU ? (r % 2 ? job.w2 : job.w) + (size_t)o * job.row_bytes
                                             : job.w + ((size_t)(r % ROWS) * job.n_rows + o) * job.row_bytes;
#pragma unroll
    for (int j = 0; j < J; ++j) wl[r][j].load(row + (size_t)min(g + 8 * j, nb - 1) * R::BLOCK_BYTES, p);
  }
  __builtin_amdgcn_sched_barrier(0);

  if (KIND == KIND_SWIGLU && tid < 32) exptab[tid] = exp_e;
  if constexpr (NORM) {
    double ss = 0.0;
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      const int i = tid + 256 * it;
      if (i >= n) break;
      if (in.add) {
        hr[it] = hr[it] + yr[it];
        if (block == 0 && job.first == 0) in.h_out[i] = hr[it];
      }
      ss += (double)(hr[it] * hr[it]);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) ss += __shfl_xor(ss, o);
    if (lane == 0) s_part[w] = ss;
    lds_barrier();
    const double tot = (s_part[0] + s_part[1]) + (s_part[2] + s_part[3]);
    const float mean = (float)(tot / (double)n);
    const float scale = 1.0f / sqrtf(mean + in.eps);
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      const int i = tid + 256 * it;
      if (i >= n) break;
      normed[i] = hr[it] * scale * gr[it];
    }
    lds_barrier();
    for (int b = w; b < nb; b += R1_WAVES)
      quantize_lds(*reinterpret_cast<const float4*>(normed + b * QK + 4 * lane), b, act.q, act.sx, act.sums);
  } else {
#pragma unroll
    for (int k = 0; k < XB; ++k)
      if (w + R1_WAVES * k < nb) quantize_lds(xv[k], w + R1_WAVES * k, act.q, act.sx, act.sums);
  }
  lds_barrier();
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int b = min(g + 8 * j, nb - 1);
    const typename R::X x = R::xload(act.q + b * QK, act.sums + b * 8, act.sx + b, p);
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
      const float v = R::block_value_x(wl[r][j].lane(), p, x);
      if (p == 0 && g + 8 * j < nb) vals[w][r][g + 8 * j] = v;
    }
  }
  // (a wave reads only what it wrote: its LDS accesses are performed in order)
  float acc = -0.0f;
  if (lane < RPW)
    for (int b = 0; b < nb; ++b) acc += vals[w][lane][b];
  const int o = o0 + lane / ROWS;
  const bool live = lane < RPW && o < job.n_rows;
  if constexpr (KIND == KIND_ROWS) {
    if (live) job.y[o] = acc;
  } else if constexpr (KIND == KIND_SWIGLU) {
    const float up = __shfl_down(acc, 1);
    if (live && lane % 2 == 0) job.y[o] = silu_tab(acc, exptab) * up;
  } else {
    const float c = __shfl_down(acc, 1), xg = __shfl_down(acc, 2);
    if (live && lane % 3 == 0) {
      const float bx = acc * xg;
      float sum = 0.0f;
#pragma unroll
      for (int k = 0; k < R1_L_MAX; ++k)
        if (k == cv.L - 1) sum = taps[k] * bx;
#pragma unroll
      for (int k = 0; k + 1 < R1_L_MAX; ++k)
        if (k + 1 < cv.L) sum += taps[k] * cols[k];
      job.y[o] = c * sum;
#pragma unroll
      for (int k = 0; k + 1 < R1_L_MAX; ++k)
        if (k + 1 < cv.L) cv.state[(size_t)k * job.n_rows + o] = k + 2 < cv.L ? cols[k + 1] : bx;
    }
  }
}

template <int KIND, bool NORM, int RPW, int J>
__global__ void __launch_bounds__(64 * R1_WAVES) k_row1(Row1In in, Row1Jobs jobs, int n, Row1Conv cv) {
  int k = 0;
  while (k + 1 < jobs.n && (int)blockIdx.x >= jobs.job[k + 1].first) ++k;
  const Row1Job& job = jobs.job[k];
  const int block = blockIdx.x - job.first;
  if (job.dt == DT_Q4_K) row1_body<DT_Q4_K, KIND, NORM, RPW, J>(in, job, block, n, cv);
  else row1_body<DT_Q6_K, KIND, NORM, RPW, J>(in, job, block, n, cv);
}

template <int KIND, int RPW>
hipError_t launch_kind(hipStream_t s, const Row1In& in, Row1Jobs& jobs, int n, const Row1Conv& cv) {
  constexpr int OPB = R1_WAVES * RPW / (KIND == KIND_CONV ? 3 : KIND == KIND_SWIGLU ? 2 : 1);
  int blocks = 0;
  for (int k = 0; k < jobs.n; ++k) {
    jobs.job[k].first = blocks;
    blocks += (jobs.job[k].n_rows + OPB - 1) / OPB;
  }
  const dim3 grid((unsigned)blocks), block(64 * R1_WAVES);
  if (in.gain)
    BB_LAUNCH((k_row1<KIND, true, RPW, 1>), grid, block, 0, s, in, jobs, n, cv);
  else if (n <= 8 * QK)
    BB_LAUNCH((k_row1<KIND, false, RPW, 1>), grid, block, 0, s, in, jobs, n, cv);
  else if constexpr (KIND == KIND_ROWS)
    BB_LAUNCH((k_row1<KIND, false, RPW, 4>), grid, block, 0, s, in, jobs, n, cv);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace

bool row1_applies(size_t n, bool norm) { return n % QK == 0 && n >= QK && n <= (norm ? GU_H_MAX : ROW1_N_MAX); }

hipError_t launch_row1(hipStream_t s, const Row1In& in, Row1Jobs jobs, int n) {
  if (!row1_applies(n, in.gain != nullptr) || jobs.n < 1 || jobs.n > 3) return hipErrorInvalidValue;
  return launch_kind<KIND_ROWS, 2>(s, in, jobs, n, Row1Conv{});
}

hipError_t launch_row1_conv(hipStream_t s, const Row1In& in, const uint8_t* w, int dt, size_t row_bytes, int H,
                            const Row1Conv& cv, float* y) {
  if (!row1_applies(H, true) || cv.L < 2 || cv.L > R1_L_MAX) return hipErrorInvalidValue;
  Row1Jobs jobs{1, {Row1Job{w, nullptr, row_bytes, H, dt, 0, y}}};
  return launch_kind<KIND_CONV, 6>(s, in, jobs, H, cv);
}

hipError_t launch_row1_swiglu(hipStream_t s, const Row1In& in, const uint8_t* gate, const uint8_t* up, int dt,
                              size_t row_bytes, int n, int n_out, float* y) {
  if (!row1_applies(n, true)) return hipErrorInvalidValue;
  Row1Jobs jobs{1, {Row1Job{gate, up, row_bytes, n_out, dt, 0, y}}};
  return launch_kind<KIND_SWIGLU, 4>(s, in, jobs, n, Row1Conv{});
}

}  // namespace bb
