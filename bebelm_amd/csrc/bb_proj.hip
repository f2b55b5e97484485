// bb_proj.hip — a packed weight matrix against a batch of tokens (the projections of the conv and
// attention operators and the dense FFN: matmul, kernels/matmul.rs:908-991, and dense_ffn_batch's
// gate, up and swiglu, model.rs:262-278).
//
// The matrix is one packed expert (bb_internal.h), so no grouping is needed, and the batch is
// small next to the expert GEMMs': a matrix of 2048 rows has 128 row tiles of 16, fewer than the
// chip has CUs. The work is therefore cut three ways: 16-row tiles, groups of up to M member tiles
// (16 tokens each), and the super-blocks of a row over the KS waves that share a row tile. A
// super-block's value is exact before it meets the running sum (bb_prefill.hip, Exactness), so
// those waves form their super-blocks' values side by side and hand them over in LDS, where the
// sum is taken left to right from the start value, the reference's order.
//
// Nothing else is shared. A wave streams its weight rows straight into registers, a super-block
// ahead (no other wave of the block reads them), and reads its activations from the tiled Q8
// layout below, in which a lane's MFMA operand is 16 contiguous bytes and a wave's read of it
// covers whole lines; the waves of a block read the same tiles, so most reads hit the CU's L1.
#include "bb_device.h"
#include "bb_internal.h"
#include "bb_mfma.h"
#include "bb_rowlane.h"

namespace bb {

namespace {

// A lane's weight bytes of one 16-row tile and super-block: Q4_K the header and its two qs words
// (the g-major order of q4_block), Q6_K sc, its two ql and two qh words and d.
template <int DT>
struct ProjW;
template <>
struct ProjW<DT_Q4_K> {
  uint4 h, q[2];
};
template <>
struct ProjW<DT_Q6_K> {
  uint4 sc, ql[2], qh[2];
  uint32_t d;
};

// row: the lane's row in the packed tile (0..63), sb: the super-block's byte offset.
__device__ __forceinline__ void proj_load(ProjW<DT_Q4_K>& w, __amdgpu_buffer_rsrc_t r, uint32_t row, uint32_t g,
                                          uint32_t sb) {
  w.h = buf_load16(r, 16u * row, sb);
  w.q[0] = buf_load16(r, 16u * row + 1024u * (1u + 2u * g), sb);
  w.q[1] = buf_load16(r, 16u * row + 1024u * (2u + 2u * g), sb);
}
__device__ __forceinline__ void proj_load(ProjW<DT_Q6_K>& w, __amdgpu_buffer_rsrc_t r, uint32_t row, uint32_t g,
                                          uint32_t sb) {
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    w.ql[n] = buf_load16(r, 16u * row + 1024u * g, sb + 4096u * n);
    w.qh[n] = buf_load16(r, 16u * row + 1024u * (g & 1u), sb + 1024u * (8 + 2 * n));
  }
  w.sc = buf_load16(r, 16u * row, sb + 1024u * 12);
  w.d = __builtin_amdgcn_raw_buffer_load_b16(r, (int)(1024u * 13 + 2u * row), (int)sb, 0);
}

// The MFMA weight operands of a super-block (q4_block's and q6_block's) and its f32 factors.
template <int DT>
struct ProjB {
  v4i hi[4], lo[4];
  int ms[2];  // Q4_K: the lane's two mins in every byte
  float d, dm;
};

__device__ __forceinline__ void proj_build(const ProjW<DT_Q4_K>& w, int g, ProjB<DT_Q4_K>& o) {
  const Q4Lane L = q4_lane(w.h, g);
#pragma unroll
  for (int s = 0; s < 4; ++s) q4_step_ops(w.q[s & 1], s >> 1, L, o.hi[s], o.lo[s]);
  o.ms[0] = L.ms[0];
  o.ms[1] = L.ms[1];
  o.d = L.dd;
  o.dm = L.dm;
}

__device__ __forceinline__ void proj_build(const ProjW<DT_Q6_K>& w, int g, ProjB<DT_Q6_K>& o) {
  o.d = f16_bits_to_f32(w.d & 0xffff);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    q6_step_ops(w.ql[c >> 1], w.qh[c >> 1], c == 0 ? w.sc.x : c == 1 ? w.sc.y : c == 2 ? w.sc.z : w.sc.w, c, g, o.hi[c],
                o.lo[c]);
  }
}

// A member tile's activations of one super-block in the tiled layout: [tile][super-block][16-byte
// chunk][token % 16][16 B]; step s of lane (r, g) is chunk 4g + s (Q4_K) or 4s + g (Q6_K) of
// token r.
template <int DT>
__device__ __forceinline__ uint32_t proj_xoff(int r, int g, int s) {
  return 16u * (uint32_t)r + 256u * (uint32_t)(DT == DT_Q4_K ? 4 * g + s : 4 * s + g);
}

constexpr int PROJ_WAVES = 8;

// Block = PROJ_WAVES waves: PROJ_WAVES / KS row tiles of 16, KS waves each, against the member
// tiles of group mg. Wave ks of a row tile takes super-blocks ks, ks + KS, ...; its sums of
// member tile m are kept by wave m % KS of the row tile. Gate/up: row tiles 2p and 2p + 1 of the
// block are the gate and up rows of the same 16 outputs.
template <int DT, int KIND, int M, int KS>
__global__ void __launch_bounds__(64 * PROJ_WAVES, 4) k_proj(const uint8_t* __restrict__ wpk, int nb, int n_out,
                                                             int n_rb, int T, int n_mt, int n_mg,
                                                             const int8_t* __restrict__ xq, const float* __restrict__ xs,
                                                             float* __restrict__ out) {
  constexpr int TB = GemmTraits<DT>::TB;
  constexpr int RW = PROJ_WAVES / KS;
  constexpr int MPW = (M + KS - 1) / KS;  // member tiles whose sums a wave keeps
  static_assert(KIND == GEMM_DOWN || RW % 2 == 0, "a block holds gate and up rows of the same outputs");
  constexpr int XCH = 2 * PROJ_WAVES * M;
  __shared__ __align__(16) float4 vx[XCH][64];
  __shared__ uint64_t exptab[32];
  // XCD k takes row blocks k, k + 8, ...; the member groups of one row block run one after the
  // other on it, so its weights are read from HBM once
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int mg = slot % n_mg, rb = (slot / n_mg) * 8 + xcd;
  if (rb >= n_rb) return;  // the whole block
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ks = w % KS, rw = w / KS, rt = rb * RW + rw;
  int t64, t16;
  if constexpr (KIND == GEMM_GATEUP) {
    t64 = rt >> 2;
    t16 = ((rt >> 1) & 1) + 2 * (rt & 1);
  } else {
    t64 = rt >> 2;
    t16 = rt & 3;
  }
  const uint64_t exp_e = KIND == GEMM_GATEUP ? exp_table_entry() : 0;
  // the group's member tiles: n_mt spread evenly over n_mg groups
  const int base = n_mt / n_mg, extra = n_mt % n_mg;
  const int m0 = mg * base + min(mg, extra), cnt = base + (mg < extra ? 1 : 0);
  const uint32_t tile_bytes = (uint32_t)nb * TB;
  const __amdgpu_buffer_rsrc_t rsw = buf_rsrc(wpk + (size_t)t64 * tile_bytes, tile_bytes);
  const __amdgpu_buffer_rsrc_t rsx = buf_rsrc(xq, (uint32_t)n_mt * (uint32_t)nb * 4096u);
  const __amdgpu_buffer_rsrc_t rss = buf_rsrc(xs, (uint32_t)n_mt * (uint32_t)nb * 64u);
  const uint32_t row = (uint32_t)(16 * t16 + r);
  const uint32_t xo = proj_xoff<DT>(r, g, 0);
  constexpr uint32_t XSTEP = DT == DT_Q4_K ? 256u : 1024u;

  ProjW<DT> wn;
  if (ks < nb) proj_load(wn, rsw, row, g, (uint32_t)(ks * TB));
  v4i ax[4];
  float4 sx;
  auto load_x = [&](int s, int m, int b) {
    ax[s] = __builtin_bit_cast(v4i, buf_load16(rsx, xo + XSTEP * s, (uint32_t)((m0 + m) * nb + b) * 4096u));
  };
  auto load_s = [&](int m, int b) {
    sx = __builtin_bit_cast(float4, buf_load16(rss, 16u * (uint32_t)g, (uint32_t)((m0 + m) * nb + b) * 64u));
  };
  if (ks < nb) {
#pragma unroll
    for (int s = 0; s < 4; ++s) load_x(s, 0, ks);
    load_s(0, ks);
  }
  if (KIND == GEMM_GATEUP && tid < 32) exptab[tid] = exp_e;
  float acc[MPW][4];
#pragma unroll
  for (int k = 0; k < MPW; ++k)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[k][i] = 0.0f;

  const int rounds = (nb + KS - 1) / KS;
  for (int rd = 0; rd < rounds; ++rd) {
    const int b = rd * KS + ks;
    float4(*const vr)[64] = vx + (rd & 1) * PROJ_WAVES * M;
    if (b < nb) {
      ProjB<DT> B;
      proj_build(wn, g, B);
      const int bn = b + KS;
      if (bn < nb) proj_load(wn, rsw, row, g, (uint32_t)(bn * TB));
#pragma unroll
      for (int m = 0; m < M; ++m) {
        if (m >= cnt) break;
        // the next tile's activations (or the next super-block's first) follow each step's MFMAs
        const bool last = m + 1 >= cnt;
        const int mn = last ? 0 : m + 1, bx = last ? min(bn, nb - 1) : b;
        v4i D[3] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          D[0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ax[s], B.hi[s], D[0], 0, 0, 0);
          D[1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ax[s], B.lo[s], D[1], 0, 0, 0);
          if constexpr (DT == DT_Q4_K) {
            const int mv = B.ms[s >> 1];
            D[2] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ax[s], ((v4i){mv, mv, mv, mv}), D[2], 0, 0, 0);
          }
          load_x(s, mn, bx);
        }
        const float sxv[4] = {sx.x, sx.y, sx.z, sx.w};
        load_s(mn, bx);
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (DT == DT_Q4_K) {
            const int sd = 8 * D[0][i] + D[1][i];
            v[i] = sxv[i] * ((B.d * (float)sd) - (B.dm * (float)D[2][i]));
          } else {
            const int sv = 64 * D[0][i] + D[1][i];
            v[i] = sxv[i] * (B.d * (float)sv);
          }
        }
        vr[w * M + m][lane] = make_float4(v[0], v[1], v[2], v[3]);
      }
    }
    // the round's values, then the sums of this wave's member tiles over them in order (the next
    // round writes the other half of vx, so one barrier a round is enough)
    lds_barrier();
#pragma unroll
    for (int k = 0; k < MPW; ++k) {
      const int m = ks + KS * k;
      if (m >= cnt) break;
      float4 v[KS];
#pragma unroll
      for (int j = 0; j < KS; ++j) v[j] = vr[(rw * KS + j) * M + m][lane];
#pragma unroll
      for (int j = 0; j < KS; ++j) {
        if (rd * KS + j >= nb) break;
        acc[k][0] += v[j].x;
        acc[k][1] += v[j].y;
        acc[k][2] += v[j].z;
        acc[k][3] += v[j].w;
      }
    }
  }

  if constexpr (KIND == GEMM_GATEUP) {
    // SwiGLU of a gate and an up wave of the same outputs and member tiles: the gate wave takes
    // tokens 4g, 4g + 1 of each lane group, the up wave 4g + 2, 4g + 3
    float2(*const hx)[64] = reinterpret_cast<float2(*)[64]>(vx);
    const bool up = rw & 1;
    lds_barrier();  // the last round's values have been read
#pragma unroll
    for (int k = 0; k < MPW; ++k)
      hx[(w * MPW + k)][lane] = up ? make_float2(acc[k][0], acc[k][1]) : make_float2(acc[k][2], acc[k][3]);
    lds_barrier();
    const int other = (rw ^ 1) * KS + ks;
    const int col = 32 * t64 + 16 * (t16 & 1) + r;
#pragma unroll
    for (int k = 0; k < MPW; ++k) {
      const int m = ks + KS * k;
      if (m >= cnt) break;
      const float2 o = hx[other * MPW + k][lane];
      const int t = 16 * (m0 + m) + 4 * g + (up ? 2 : 0);
      const float g0 = up ? o.x : acc[k][0], g1 = up ? o.y : acc[k][1];
      const float u0 = up ? acc[k][2] : o.x, u1 = up ? acc[k][3] : o.y;
      if (t < T) out[(size_t)t * n_out + col] = silu_tab(g0, exptab) * u0;
      if (t + 1 < T) out[(size_t)(t + 1) * n_out + col] = silu_tab(g1, exptab) * u1;
    }
  } else {
    const int col = 64 * t64 + 16 * t16 + r;
#pragma unroll
    for (int k = 0; k < MPW; ++k) {
      const int m = ks + KS * k;
      if (m >= cnt) break;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 16 * (m0 + m) + 4 * g + i;
        if (t < T) out[(size_t)t * n_out + col] = acc[k][i];
      }
    }
  }
}

// Row tiles of the matrix (16 rows; gate and up count separately).
int proj_row_tiles(int kind, int n_out) { return kind == GEMM_GATEUP ? n_out / 8 : n_out / 16; }

// (The two rules that follow count blocks and waves for 256 CUs.)
// Member tiles a block takes. Four share the operand build (about 80 VALU instructions a row tile
// and super-block, against 32 of epilogue per member tile), unless that leaves long rows with few
// blocks (2048 rows of 7168 at 64 tokens: 10.6 us with 4, 8.1 with 2; at 96 9.8 and 10.7).
int proj_group(int n_rt, int n_mt, int nb) {
  if (n_mt <= 2) return n_mt;
  return nb > 8 && n_rt * ((n_mt + 1) / 2) <= 256 ? 2 : 4;
}

// Waves a row tile's super-blocks are split over: enough for about 14 waves a CU of the (row tile,
// member group) units. 2048 rows of 7168, 130 tokens (384 units): 26.6 us with 2, 15.1 with 4,
// 13.1 with 8; 512 tokens (1024 units): 34.9, 30.4, 32.3; gate/up of 2 x 7168 rows of 2048, 512
// tokens (7168 units): 61.8 with 2, 66.9 with 4. (One wave a row tile keeps the sums of all its
// member tiles: spilled registers, 96 us there.)
int proj_split(int units, int nb, int max_ks) {
  int ks = 2;
  while (ks < max_ks && ks < nb && units * ks < 14 * 256) ks *= 2;
  return ks;
}

template <int DT, int KIND, int M, int KS>
hipError_t launch_one(hipStream_t s, const uint8_t* w, int T, int n_in, int n_out, const Q8Bufs& x, float* out) {
  constexpr int RW = PROJ_WAVES / KS;
  const int n_mt = (T + 15) / 16, n_mg = (n_mt + M - 1) / M;
  const int n_rb = proj_row_tiles(KIND, n_out) / RW;
  BB_LAUNCH((k_proj<DT, KIND, M, KS>), dim3((unsigned)((n_rb + 7) / 8 * 8 * n_mg)), dim3(64 * PROJ_WAVES), 0, s, w,
            n_in / QK, n_out, n_rb, T, n_mt, n_mg, x.q, x.scales, out);
  return hipGetLastError();
}

template <int DT, int KIND, int M>
hipError_t launch_m(hipStream_t s, int ks, const uint8_t* w, int T, int n_in, int n_out, const Q8Bufs& x, float* out) {
  if constexpr (KIND == GEMM_DOWN)
    if (ks == 8) return launch_one<DT, KIND, M, 8>(s, w, T, n_in, n_out, x, out);
  if (ks == 4) return launch_one<DT, KIND, M, 4>(s, w, T, n_in, n_out, x, out);
  return launch_one<DT, KIND, M, 2>(s, w, T, n_in, n_out, x, out);
}

template <int DT, int KIND>
hipError_t launch_dt(hipStream_t s, const uint8_t* w, int T, int n_in, int n_out, const Q8Bufs& x, float* out) {
  const int n_mt = (T + 15) / 16, n_rt = proj_row_tiles(KIND, n_out), nb = n_in / QK;
  const int m = proj_group(n_rt, n_mt, nb), n_mg = (n_mt + m - 1) / m;
  const int ks = proj_split(n_rt * n_mg, nb, KIND == GEMM_GATEUP ? 4 : 8);
  if (m == 1) return launch_m<DT, KIND, 1>(s, ks, w, T, n_in, n_out, x, out);
  if (m == 2) return launch_m<DT, KIND, 2>(s, ks, w, T, n_in, n_out, x, out);
  return launch_m<DT, KIND, 4>(s, ks, w, T, n_in, n_out, x, out);
}

}  // namespace

// (the kernel addresses the activations with 32-bit byte offsets)
bool proj_applies(const PackedW& p, size_t T, size_t n_in) {
  return p.w && T >= PROJ_MIN_T && T <= PROJ_MAX_T && (T + 15) / 16 * 16 * n_in < (size_t(1) << 31);
}

hipError_t launch_proj(hipStream_t s, const PackedW& p, bool gateup, int T, int n_in, int n_out, const Q8Bufs& x,
                       float* out) {
  if (!x.tiled || T < 1 || n_in % QK != 0 || n_out % (gateup ? 64 : 128) != 0) return hipErrorInvalidValue;
  if (p.dt == DT_Q4_K)
    return gateup ? launch_dt<DT_Q4_K, GEMM_GATEUP>(s, p.w, T, n_in, n_out, x, out)
                  : launch_dt<DT_Q4_K, GEMM_DOWN>(s, p.w, T, n_in, n_out, x, out);
  return gateup ? launch_dt<DT_Q6_K, GEMM_GATEUP>(s, p.w, T, n_in, n_out, x, out)
                : launch_dt<DT_Q6_K, GEMM_DOWN>(s, p.w, T, n_in, n_out, x, out);
}

}  // namespace bb
