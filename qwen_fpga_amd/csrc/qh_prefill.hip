// Grouped prompt kernels (gfx950): each launch runs one step of one layer for up
// to kPfGroup prompt tokens.  The decode path streams every weight byte once per
// token; here one read serves the whole group and the projections become matrix
// products on the matrix cores.
//
// Every value is the token path's, bit for bit, so that a prompt fed through
// here leaves exactly the state that feeding it token by token leaves:
//   * W8A8 products are int32 sums, exact in any order: v_mfma_i32_16x16x64_i8.
//   * W8A16 products follow the C16 order (qh_device.hpp).  The fp32 MFMAs
//     (v_mfma_f32_16x16x4_f32, v_mfma_f32_32x32x2_f32) compute, for each output,
//     the chain fma(a1,b1,fma(a0,b0,c)) in increasing k with single roundings and
//     denormals kept (compared with fmaf on 2^20 results), so a lane partial over
//     a 16-element chunk is a run of MFMAs from zero; the 64 partials are then
//     added by the same tree.
//   * Attention scores (16-lane tree over 16-element chunks) and P.V (a chain in
//     position order) have the same shape and use the same instructions.
//   * Norms, gates, conv, the delta rule and the softmax repeat the decode
//     bodies' operations in their order.
#include <type_traits>

#include "qh_prefill.hpp"
#include "qh_decode.h"
#include "qh_stages.hpp"

namespace qh {

typedef int i32x4 __attribute__((ext_vector_type(4)));

namespace {

// 16-element chunk c of token m, written to the fragments of a K-wide activation
template <int K>
__device__ __forceinline__ void put_frag_f32(float* x, int m, int c, const float (&v)[16]) {
  f32x4* p = reinterpret_cast<f32x4*>(x + pf_frag_f32(K, m, c, 0));
#pragma unroll
  for (int hb = 0; hb < 2; ++hb)
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
      *as_global_w(p + 64 * hb + 32 * kk) = f32x4{v[8 * hb + kk], v[8 * hb + 2 + kk], v[8 * hb + 4 + kk], v[8 * hb + 6 + kk]};
}
template <int K>
__device__ __forceinline__ void put_frag_i8(void* x, int m, int c, const uint32_t (&q)[4]) {
  u32x4* p = reinterpret_cast<u32x4*>(x) + ((size_t)(m >> 4) * (K / 64) + (c >> 2)) * 64 + 16 * (c & 3) + (m & 15);
  *as_global_w(p) = u32x4{q[0], q[1], q[2], q[3]};
}
__device__ __forceinline__ void quant16(const float (&v)[16], float xs, float rs, int (&q)[16], uint32_t (&pk)[4]) {
#pragma unroll
  for (int e = 0; e < 16; ++e) q[e] = quant_one_r(v[e], xs, rs);
#pragma unroll
  for (int d = 0; d < 4; ++d) pk[d] = pack4(q[4 * d], q[4 * d + 1], q[4 * d + 2], q[4 * d + 3]);
}

}  // namespace

// ---------------------------------------------------------------------------
// RMSNorm of a layer input (and, for a DeltaNet layer, its 32 gate rows): one
// token per wave, four tokens per workgroup.  The norm is gemv_body's P_NORM
// prologue.  The four normalised vectors meet in LDS and each wave forms eight
// of the 32 gate rows for all four, from gate weights it reads once (128 KiB per
// workgroup from L2 instead of per token).
// ---------------------------------------------------------------------------
template <int MODE, bool GATES>
__global__ __launch_bounds__(256) void pf_norm_kernel(const PfNorm a) {
  __shared__ __attribute__((aligned(16))) float xl[GATES ? 4 * 1024 : 4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = (int)blockIdx.x * 4, m = m0 + wave;
  const int mc = min(m, a.M - 1);
  float xv[16], nw[16];
  load16c(a.nw, lane, nw);
  float gw[8][16], al = 0.0f, db = 0.0f;   // this wave's gate rows, in flight beside the norm
  if constexpr (GATES) {
#pragma unroll
    for (int r = 0; r < 8; ++r) load16c(a.gw + (size_t)(8 * wave + r) * 1024, lane, gw[r]);
    al = as_global(a.A_log)[(8 * wave + row_of_lane<8>(lane)) & 15];
    db = as_global(a.dt_bias)[(8 * wave + row_of_lane<8>(lane)) & 15];
  }
  if (a.emb != nullptr) {
    const int tok = __builtin_amdgcn_readfirstlane(as_global(a.ids)[mc]);
    uint32_t t[4];
    load16b(a.emb + (size_t)tok * 1024 + 16 * lane, t);
    const float es = as_global(a.emb_s)[tok];
#pragma unroll
    for (int e = 0; e < 16; ++e) xv[e] = i8_at(t, e) * es;
    if (m < a.M) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        *as_global_w(reinterpret_cast<f32x4*>(a.h_out + (size_t)m * 1024 + 16 * lane + 4 * k)) =
            f32x4{xv[4 * k], xv[4 * k + 1], xv[4 * k + 2], xv[4 * k + 3]};
    }
  } else {
    load16g(a.h + (size_t)mc * 1024 + 16 * lane, xv);
  }
  float ss = dot16_f32(xv, xv, 0.0f), mu = 0.0f;
  if constexpr (MODE == M_W8A8) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      xv[e] = xv[e] * (1.0f + nw[e]);
      mu = fmaxf(mu, fabsf(xv[e]));
    }
  }
  ss = xor_sum<64>(ss);
  if constexpr (MODE == M_W8A8) mu = xor_max<64>(mu);
  const float inv = 1.0f / sqrtf(ss / 1024.0f + a.eps);
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    if constexpr (MODE == M_W8A8)
      xv[e] = xv[e] * inv;
    else
      xv[e] = (xv[e] * inv) * (1.0f + nw[e]);
  }
  if constexpr (MODE == M_W8A8) {
    const float xs = quant_scale(mu * inv);
    const float rs = 1.0f / xs;
    int q[16];
    uint32_t pk[4];
    quant16(xv, xs, rs, q, pk);
    if (m < a.M) {
      put_frag_i8<1024>(a.x, m, lane, pk);
      if (lane == 0) a.xs[m] = xs;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) xv[e] = (float)q[e] * xs;   // the gates take the dequantised activation
  } else {
    if (m < a.M) put_frag_f32<1024>(static_cast<float*>(a.x), m, lane, xv);
  }
  if constexpr (GATES) {
#pragma unroll
    for (int k = 0; k < 4; ++k)   // lane-interleaved, as load16c reads
      *as_lds_w(reinterpret_cast<f32x4*>(xl + 1024 * wave + 256 * k + 4 * lane)) =
          f32x4{xv[4 * k], xv[4 * k + 1], xv[4 * k + 2], xv[4 * k + 3]};
    lds_barrier();
    // lane l ends with row 8 wave + l / 8 of every token and finishes token l % 8 of them
    const int row = 8 * wave + row_of_lane<8>(lane);   // beta rows 0 .. 15, then g
    const int h = row & 15;
    float y = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      float x[16], p[8];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const f32x4 v = *as_lds(reinterpret_cast<const f32x4*>(xl + 1024 * t + 256 * k + 4 * lane));
#pragma unroll
        for (int e = 0; e < 4; ++e) x[4 * k + e] = v[e];
      }
#pragma unroll
      for (int r = 0; r < 8; ++r) p[r] = dot16_f32(gw[r], x, 0.0f);
      const float yt = reduce8(p, lane);
      if ((lane & 7) == t) y = yt;
    }
    const float val = row < 16 ? dev_sigmoid(y) : dev_expf(-dev_expf(al) * dev_softplus(y + db));
    const int mt = m0 + (lane & 7);
    if ((lane & 7) < 4 && mt < a.M) a.gates[((size_t)h * a.M + mt) * 2 + (row < 16 ? 1 : 0)] = val;
  }
}

// ---------------------------------------------------------------------------
// Matrix product out[m][n] = sum_k w[n][k] x[m][k].  A workgroup owns TA * 16
// weight rows, copies them whole (K bytes each) to LDS once, and multiplies them
// with its token tiles; x streams from L2 as fragments, 1 KiB per load
// instruction.  A (rows of D) = weight rows, B (columns) = tokens, so a lane ends
// with four consecutive outputs of one token.  A row's 16-byte chunk c sits at
// chunk c ^ (row & 15): the 16 rows a wave reads at once lie in 16 different bank
// groups.  The copy is global -> LDS loads, all in flight at once (through
// registers, four at a time, it took 12.6 us at K = 3584 where this takes 5).
//   W8A8   each of the four waves takes its own token tile (an MFMA step is 16
//          cycles: a tile is too short to share).
//   W8A16  the four waves split the 64 lanes of the C16 tree, 16 visits each, and
//          their subtrees meet in LDS: a token tile is 256 MFMAs of 32 cycles per
//          wave, and a short prompt still fills the chip.
// ---------------------------------------------------------------------------
template <int K, int ROWS, int THREADS, class SRC>
__device__ __forceinline__ void pf_stage_rows(int8_t* wl, SRC src) {
  constexpr int NC = K / 16;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  static_assert((ROWS * NC) % THREADS == 0, "whole passes");
#pragma unroll
  for (int i = 0; i < ROWS * NC / THREADS; ++i) {
    const int u = THREADS * i + 64 * wave, p = u + lane;   // LDS takes a wave's 64 chunks in lane order
    const int r = p / NC, c = (p % NC) ^ (r & 15);
    __builtin_amdgcn_global_load_lds(as_global(src(r) + 16 * c), as_lds_w(wl + 16 * u), 16, 0, 0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

// Outputs 16 ta + 4 g .. + 3 of token m from the scaled-by-activation sums y (PF_SWIGLU: y2 the up
// row's).  n: the output's column.
template <int MODE, int EPI>
__device__ __forceinline__ void pf_epilogue(const PfGemm& a, int si, int m, int n, const f32x4& y, const f32x4& y2) {
  f32x4 v;
  if constexpr (EPI == PF_SWIGLU) {
    const f32x4 sg = *as_global(reinterpret_cast<const f32x4*>(a.sw[0] + n));
    const f32x4 su = *as_global(reinterpret_cast<const f32x4*>(a.sw[1] + n));
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = dev_silu(y[r] * sg[r]) * (y2[r] * su[r]);
    if constexpr (MODE == M_W8A8) {
      *as_global_w(reinterpret_cast<f32x4*>(a.out + (size_t)m * a.ld + n)) = v;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) as_global_w(a.out)[pf_frag_f32(QH_INTER, m, n >> 4, (n & 15) + r)] = v[r];
    }
  } else {
    const f32x4 sw = *as_global(reinterpret_cast<const f32x4*>(a.sw[si] + (n - a.row0[si])));
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = y[r] * sw[r];
    f32x4* p = reinterpret_cast<f32x4*>(a.out + (size_t)m * a.ld + n);
    if constexpr (EPI == PF_INPROJ) {
      if (si == 1)   // z (the gated norm takes silu(z))
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = dev_silu(v[r]);
    }
    if constexpr (EPI == PF_RESID) {
      const f32x4 h = *as_global(p);
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = h[r] + v[r];
    }
    *as_global_w(p) = v;
  }
}

// the weight segment of output row n0, and the address of the row tile's row r
template <int EPI>
__device__ __forceinline__ int pf_seg(const PfGemm& a, int n0) {
  int si = 0;
  if constexpr (EPI == PF_INPROJ || EPI == PF_STORE) {
#pragma unroll
    for (int i = 1; i < 3; ++i)
      if (i < a.nseg && n0 >= a.row0[i]) si = i;
  }
  return si;
}
template <int K, int EPI>
__device__ __forceinline__ const int8_t* pf_row(const PfGemm& a, int si, int n0, int r) {
  if constexpr (EPI == PF_SWIGLU) {   // 16-row blocks alternate gate, up
    const int t = r >> 4;
    return ((t & 1) ? a.w[1] : a.w[0]) + (size_t)(n0 / 2 + (t >> 1) * 16 + (r & 15)) * K;
  } else {
    return a.w[si] + (size_t)(n0 - a.row0[si] + r) * K;
  }
}

template <int K, int TA, int EPI>
__global__ __launch_bounds__(256) void pf_gemm_i8_kernel(const PfGemm a, int tpw) {
  constexpr int ROWS = 16 * TA, NS = K / 64;
  __shared__ __attribute__((aligned(16))) int8_t wl[ROWS * K];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, j = lane & 15;
  const int n0 = (int)blockIdx.x * ROWS;   // first output (PF_SWIGLU: weight) row
  const int si = pf_seg<EPI>(a, n0);
  const int ntile = (a.M + 15) >> 4;
  const int t0 = (int)blockIdx.y * tpw, t1 = min(t0 + tpw, ntile);
  constexpr int PF = NS % 8 == 0 ? 8 : 7;   // steps of x in flight
  static_assert(NS % PF == 0, "steps");
  const i32x4* xb0 = reinterpret_cast<const i32x4*>(a.x) + lane;
  i32x4 xb[PF];
  int tt = t0 + wave;
  {   // the first tile's x is in flight beside the rows
    const i32x4* xp = xb0 + (size_t)min(tt, ntile - 1) * NS * 64;
#pragma unroll
    for (int p = 0; p < PF; ++p) xb[p] = *as_global(xp + 64 * p);
  }
  pf_stage_rows<K, ROWS, 256>(wl, [&](int r) { return pf_row<K, EPI>(a, si, n0, r); });
  for (; tt < t1; tt += 4) {
    const i32x4* xp = xb0 + (size_t)tt * NS * 64;
    const i32x4* xn = xb0 + (size_t)min(tt + 4, ntile - 1) * NS * 64;   // the next tile's
    i32x4 acc[TA];
#pragma unroll
    for (int ta = 0; ta < TA; ++ta) acc[ta] = i32x4{0, 0, 0, 0};
#pragma unroll 1
    for (int s0 = 0; s0 < NS; s0 += PF) {
      const i32x4* xq = s0 + PF < NS ? xp + 64 * (s0 + PF) : xn;
#pragma unroll
      for (int p = 0; p < PF; ++p) {
        const int s = s0 + p;
        const i32x4 b = xb[p];
        xb[p] = *as_global(xq + 64 * p);
#pragma unroll
        for (int ta = 0; ta < TA; ++ta) {
          const i32x4 wa = *as_lds(reinterpret_cast<const i32x4*>(wl + (16 * ta + j) * K + 16 * ((4 * s + g) ^ j)));
          acc[ta] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa, b, acc[ta], 0, 0, 0);
        }
      }
    }
    const int m = 16 * tt + j;
    if (m < a.M) {
      const float xs = as_global(a.xs)[m];
      f32x4 y[TA];
#pragma unroll
      for (int ta = 0; ta < TA; ++ta)
#pragma unroll
        for (int r = 0; r < 4; ++r) y[ta][r] = (float)acc[ta][r] * xs;
      if constexpr (EPI == PF_SWIGLU) {
#pragma unroll
        for (int ta = 0; ta < TA; ta += 2)
          pf_epilogue<M_W8A8, EPI>(a, si, m, n0 / 2 + (ta >> 1) * 16 + 4 * g, y[ta], y[ta + 1]);
      } else {
#pragma unroll
        for (int ta = 0; ta < TA; ++ta) pf_epilogue<M_W8A8, EPI>(a, si, m, n0 + 16 * ta + 4 * g, y[ta], y[ta]);
      }
    }
  }
}

typedef float f32x16 __attribute__((ext_vector_type(16)));

// RT row tiles of 32 rows; each is shared by KS waves, which take 64 / KS visits each.
template <int K, int RT, int KS, int EPI>
__global__ __launch_bounds__(64 * RT * KS, 2) void pf_gemm_f32_kernel(const PfGemm a, int tpw) {
  constexpr int ROWS = 32 * RT, NC = K / 16, NCH = pf_nch(K), NW = RT * KS, NV = 64 / KS;
  constexpr int LG = NV == 32 ? 5 : NV == 16 ? 4 : 3;   // tree levels inside a wave
  static_assert(NV == 1 << LG, "visits per wave");
  __shared__ __attribute__((aligned(16))) int8_t wl[ROWS * K];
  __shared__ __attribute__((aligned(16))) float red[NW * 4 * 256];   // subtree sums [wave][group of 4 rows][lane]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ks = wave % KS, rt = wave / KS;
  const int kk = lane >> 5, j = lane & 31;
  const int n0 = (int)blockIdx.x * ROWS;
  const int si = pf_seg<EPI>(a, n0);
  const int ntile = (a.M + 31) >> 5;
  const int t0 = (int)blockIdx.y * tpw, t1 = min(t0 + tpw, ntile);
  constexpr int NX = NV * NCH, PF = 4;   // steps (chunks) of a wave and tile; x of PF steps in flight
  const f32x4* xw = reinterpret_cast<const f32x4*>(a.x) + 128 * NX * ks + lane;
  f32x4 xb[PF][2];
#pragma unroll
  for (int p = 0; p < PF; ++p)
#pragma unroll
    for (int hb = 0; hb < 2; ++hb) xb[p][hb] = *as_global(xw + (size_t)t0 * pf_frags(K) * 128 + 128 * p + 64 * hb);
  pf_stage_rows<K, ROWS, 64 * NW>(wl, [&](int r) { return pf_row<K, EPI>(a, si, n0, r); });
  // lane of the tree = the visit's six bits reversed: visits NV ks + i lie at lanes (ks reversed) + KS * (i reversed)
  const int lw = pf_bitrev6(ks * NV);
  // step f = visit f / NCH, chunk f % NCH of its lane; past K (the tree's upper 32 lanes, the odd
  // visits, have one chunk less at K = 3584) there is no step
  auto live = [](int f) constexpr { return !(64 * (f % NCH) + 32 >= NC && ((f / NCH) & 1)); };
  auto next = [&](int f) constexpr {   // the next step; the last one is followed by the next tile's first
    do f = f + 1 == NX ? 0 : f + 1;
    while (!live(f));
    return f;
  };
  auto wread = [&](int f) {   // the rows' chunk of step f
    const int l = lw + pf_bitrev6(f / NCH);
    return *as_lds(reinterpret_cast<const u32x4*>(wl + (32 * rt + j) * K + 16 * ((l + 64 * (f % NCH)) ^ (j & 15))));
  };
  u32x4 wv = wread(0);
  for (int tt = t0; tt < t1; ++tt) {
    const f32x4* xp = xw + (size_t)tt * pf_frags(K) * 128;
    const f32x4* xn = xw + (size_t)min(tt + 1, t1 - 1) * pf_frags(K) * 128;   // the next tile's
    f32x16 st[LG], part;
#pragma unroll
    for (int f = 0; f < NX; ++f) {
      const int i = f / NCH;
      if (f % NCH == 0) part = f32x16{};
      f32x4 b[2];
#pragma unroll
      for (int hb = 0; hb < 2; ++hb) {
        b[hb] = xb[f % PF][hb];
        xb[f % PF][hb] = *as_global(f + PF < NX ? xp + 128 * (f + PF) + 64 * hb : xn + 128 * (f + PF - NX) + 64 * hb);
      }
      if (live(f)) {
        float wf[8];   // elements 2 e + kk
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const uint32_t t = wv[d] >> (8 * kk);
          wf[2 * d] = (float)(int)(int8_t)t;
          wf[2 * d + 1] = (float)(int)(int8_t)(t >> 16);
        }
        wv = wread(next(f));
#pragma unroll
        for (int e = 0; e < 8; ++e) part = __builtin_amdgcn_mfma_f32_32x32x2f32(wf[e], b[e >> 2][e & 3], part, 0, 0, 0);
      }
      if (f % NCH != NCH - 1) continue;
      // the tree's first LG levels (offsets 32, 16, ...): a binary counter over the visits
#pragma unroll
      for (int v = 0; v < LG; ++v) {
        const int bits = (1 << v) - 1;
        if ((i & bits) != bits) break;
        if ((i >> v) & 1)
          part = st[v] + part;
        else {
          st[v] = part;
          break;
        }
      }
    }
    // the remaining levels: the waves' subtrees of each row tile
    lds_barrier();   // the previous sums have been read
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *as_lds_w(reinterpret_cast<f32x4*>(red + (wave * 4 + q) * 256 + 4 * lane)) =
          f32x4{part[4 * q], part[4 * q + 1], part[4 * q + 2], part[4 * q + 3]};
    lds_barrier();
    auto total = [&](int r, int q) {   // rows 8 q + 4 kk .. + 3 of row tile r
      f32x4 s[KS];
#pragma unroll
      for (int w = 0; w < KS; ++w) s[w] = *as_lds(reinterpret_cast<const f32x4*>(red + ((r * KS + w) * 4 + q) * 256 + 4 * lane));
#pragma unroll
      for (int d = 1; d < KS; d *= 2)
#pragma unroll
        for (int w = 0; w < KS; w += 2 * d) s[w] = s[w] + s[w + d];
      return s[0];
    };
    const int m = 32 * tt + j;
    if constexpr (EPI == PF_SWIGLU) {   // gate rows 16 .. apart from their up rows
      for (int u = wave; u < 2 * RT; u += NW) {
        const f32x4 y = total(u >> 1, u & 1), y2 = total(u >> 1, (u & 1) + 2);
        if (m < a.M) pf_epilogue<M_W8A16, EPI>(a, si, m, n0 / 2 + 8 * u + 4 * kk, y, y2);
      }
    } else {
      for (int u = wave; u < 4 * RT; u += NW) {
        const f32x4 y = total(u >> 2, u & 3);
        if (m < a.M) pf_epilogue<M_W8A16, EPI>(a, si, m, n0 + 8 * u + 4 * kk, y, y);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Short conv + SiLU of the raw qkv rows, then the l2norm of q and k (and q's
// 1 / sqrt(128)): kConvTok tokens of kConvCh channels (four heads' q, k or v) per
// workgroup, so that 63 tokens already make 192 workgroups.  The convolution is
// elementwise: thread t takes channel quad t, so that every row load of a wave is
// consecutive memory, and the results meet in LDS, from which thread t takes chunk
// t % 32 of 16 channels of token t / 32 for the norm.  (With 16 channels per thread
// from the start each tap load touched 64 cache lines: 27 us at 512 tokens.  With
// all 6144 channels of two tokens in a workgroup, a launch of 63 tokens was 32
// workgroups whose tap loads queued behind one another: 12.3 us, where this takes 6.0.)
// q and k of (head, token) go to 256 floats in the order the scan reads them:
// elements 8 e2 + 4 qd .. + 3 of q (e2 = half of a k-group) at 64 qd + 4 e2, k 128
// further.
// ---------------------------------------------------------------------------
constexpr int kConvTok = 4, kConvCh = 512;
__global__ __launch_bounds__(128) void pf_conv_kernel(const PfConv a) {
  __shared__ __attribute__((aligned(16))) float xl[kConvTok * kConvCh];
  const int t = threadIdx.x, m0 = (int)blockIdx.x * kConvTok, ch = (int)blockIdx.y * kConvCh + 4 * t;
  f32x4 in[3 + kConvTok], tap[4];   // rows m0 - 3 ..; taps of the four channels
#pragma unroll
  for (int e = 0; e < 4; ++e) tap[e] = *as_global(reinterpret_cast<const f32x4*>(a.taps + (size_t)(ch + e) * 4));
  if (m0 == 0) {   // rows before the group: columns 1 .. 3 of the state
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const f32x4 st = *as_global(reinterpret_cast<const f32x4*>(a.state + (size_t)(ch + e) * 4));
#pragma unroll
      for (int i = 0; i < 3; ++i) in[i][e] = st[1 + i];
    }
  } else {
#pragma unroll
    for (int i = 0; i < 3; ++i) in[i] = *as_global(reinterpret_cast<const f32x4*>(a.y + (size_t)(m0 - 3 + i) * 8192 + ch));
  }
#pragma unroll
  for (int i = 0; i < kConvTok; ++i)
    in[3 + i] = *as_global(reinterpret_cast<const f32x4*>(a.y + (size_t)min(m0 + i, a.M - 1) * 8192 + ch));
#pragma unroll
  for (int k = 0; k < kConvTok; ++k) {
    f32x4 x;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float acc = 0.0f;
#pragma unroll
      for (int i = 0; i < 4; ++i) acc = acc + in[k + i][e] * tap[e][i];
      x[e] = dev_silu(acc);
    }
    *as_lds_w(reinterpret_cast<f32x4*>(xl + k * kConvCh + 4 * t)) = x;
  }
  lds_barrier();
  const int part = (int)blockIdx.y >> 2, c = 32 * ((int)blockIdx.y & 3) + (t & 31);   // q, k or v; chunk of its 128
  const int h = c >> 3, kg = c & 7, m = m0 + (t >> 5);
  float x[16];
  load16l(xl + 16 * t, x);   // (token t / 32, chunk t % 32)
  if (part < 2) {   // deltanet.hpp:134,166-169
    float ss = dot16_f32(x, x, 0.0f);
    ss = xor_sum<8>(ss);
    const float inv = 1.0f / sqrtf(ss + 1e-6f);
#pragma unroll
    for (int e = 0; e < 16; ++e) x[e] = x[e] * inv;
    if (part == 0) {
      const float sc = 1.0f / sqrtf(128.0f);
#pragma unroll
      for (int e = 0; e < 16; ++e) x[e] = x[e] * sc;
    }
    if (m >= a.M) return;
    float* p = a.qk + ((size_t)h * a.M + m) * 256 + 128 * part + 8 * kg;
#pragma unroll
    for (int d = 0; d < 4; ++d)   // half d / 2, quad d % 2
      *as_global_w(reinterpret_cast<f32x4*>(p + 64 * (d & 1) + 4 * (d >> 1))) =
          f32x4{x[4 * d], x[4 * d + 1], x[4 * d + 2], x[4 * d + 3]};
  } else if (m < a.M) {
    float* p = a.v + ((size_t)h * a.M + m) * 128 + 16 * kg;
#pragma unroll
    for (int d = 0; d < 4; ++d)
      *as_global_w(reinterpret_cast<f32x4*>(p + 4 * d)) = f32x4{x[4 * d], x[4 * d + 1], x[4 * d + 2], x[4 * d + 3]};
  }
}

// ---------------------------------------------------------------------------
// The delta rule over the group's tokens in order (deltanet_body's operations).
// It is bound by the serial chain of one token after another: p = sum_k s k over
// 16 elements in sequence and a tree of eight, delta, the update.  To shorten
// what one wave issues per token:
//   * a 16-element chain is shared by two lanes, eight elements each: the even
//     lane's partial sum passes to the odd lane, which continues it, and the
//     multiplies and updates beside the chain halve;
//   * the output q^T S runs on a second wave with its own copy of the slice, one
//     block of eight tokens behind: the first wave (A) computes delta and leaves
//     it in LDS, the second (B) repeats decay and update and forms the output.
// A workgroup holds 8 columns of one head on four waves (A and B for columns
// 0 .. 3, A and B for 4 .. 7): 256 workgroups, one wave per SIMD.  One barrier
// per eight tokens.  A token took 835 cycles with the whole column group's chain
// on one wave.
// ---------------------------------------------------------------------------
constexpr int kScanTok = 8;
struct ScanBlock {   // eight tokens of q, k (256 floats each, see pf_conv_kernel), v [token][8 columns], gates
  float qk[kScanTok * 256];
  float v[kScanTok * 8];
  float g[kScanTok * 2];
};
// a value of the even lane of each pair in both lanes / of the odd lane
__device__ __forceinline__ float pair_even(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xA0, 0xF, 0xF, false));   // quad_perm [0,0,2,2]
}
__device__ __forceinline__ float pair_odd(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xF5, 0xF, 0xF, false));   // quad_perm [1,1,3,3]
}
template <int N>   // the value N lanes away, round the row of 16
__device__ __forceinline__ float row_ror(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + N, 0xF, 0xF, false));
}
// sum over i of a[i] b[i] over the pair's 16 elements in order, then over the eight k-groups: valid in odd lanes
__device__ __forceinline__ float scan_dot(const float (&a)[8], const float (&b)[8]) {
  float t[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) t[i] = a[i] * b[i];
  float p = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) p = p + t[i];
  p = pair_even(p);
#pragma unroll
  for (int i = 0; i < 8; ++i) p = p + t[i];
  // k-groups 4, 2, 1 apart: after the sum over distance 8 the values repeat every 8 lanes of the row, so
  // that a rotation by 4 (then 2) reads the partner, in the add itself
  p = p + row_ror<8>(p);
  p = p + row_ror<4>(p);
  p = p + row_ror<2>(p);
  return p;
}
__global__ __launch_bounds__(256, 1) void pf_scan_kernel(const PfScan a) {
  __shared__ __attribute__((aligned(16))) ScanBlock blk[3];   // being filled, A's, B's
  __shared__ float dl[2][2 * 4 * kScanTok];                   // delta [A wave][token][column]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kh = lane & 15, kg = kh >> 1, vc = lane >> 4;     // half k-group, k-group, column of the wave
  const int half = wave & 1;                                  // columns 4 half ..
  const bool isA = wave < 2;
  const int h = (int)blockIdx.x >> 4, v0 = ((int)blockIdx.x & 15) * 8, v = v0 + 4 * half + vc;
  const int M = a.M, nb = (M + kScanTok - 1) / kScanTok;
  float* Sh = a.S + (size_t)h * 128 * 128;
  float s[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) s[i] = as_global(Sh)[(kh * 8 + i) * 128 + v];
  const float* qk = a.qk + (size_t)h * M * 256;
  const float* vp = a.v + (size_t)h * M * 128;
  const float* gp = a.gates + (size_t)h * M * 2;
  // a block's loads: every thread 32 bytes of q, k; wave 0 v, wave 1 the gates
  f32x4 n0, n1;
  float nx = 0.0f;
  auto fetch = [&](int b) {
    const int m0 = b * kScanTok, t = threadIdx.x;
    const float* p = qk + (size_t)min(m0 + (t >> 5), M - 1) * 256 + 8 * (t & 31);
    n0 = *as_global(reinterpret_cast<const f32x4*>(p));
    n1 = *as_global(reinterpret_cast<const f32x4*>(p + 4));
    if (wave == 0) nx = as_global(vp)[(size_t)min(m0 + (lane >> 3), M - 1) * 128 + v0 + (lane & 7)];
    if (wave == 1) nx = as_global(gp)[(size_t)min(m0 + ((lane >> 1) & 7), M - 1) * 2 + (lane & 1)];
  };
  auto put = [&](int b) {
    ScanBlock& k = blk[b % 3];
    *as_lds_w(reinterpret_cast<f32x4*>(k.qk + 8 * threadIdx.x)) = n0;
    *as_lds_w(reinterpret_cast<f32x4*>(k.qk + 8 * threadIdx.x + 4)) = n1;
    if (wave == 0) as_lds_w(k.v)[lane] = nx;
    if (wave == 1 && lane < 16) as_lds_w(k.g)[lane] = nx;
  };
  auto ld8 = [&](const float* p, float (&o)[8]) {   // this lane's 8 elements of q (k: 128 further)
    const f32x4 x = *as_lds(reinterpret_cast<const f32x4*>(p + 4 * kh));
    const f32x4 y = *as_lds(reinterpret_cast<const f32x4*>(p + 64 + 4 * kh));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[e] = x[e];
      o[4 + e] = y[e];
    }
  };
  // n tokens of block b (FULL: all eight, straight-line).  Token t + 2's vectors are read while token t
  // runs (the empty asm keeps the reads above it: next to their use, each token waited for the LDS; 768
  // tokens took 157.7 us, with the reads ahead 146.1, and with the tree's rotations 143.1).
  auto runA = [&](int b, auto full, int n) {
    const ScanBlock& B = blk[b % 3];
    float* d_out = dl[b & 1] + 32 * half;
    const float cg = as_lds(B.g)[lane & 15];
    float k[3][8], vt[3];
    auto get = [&](int t) {
      ld8(B.qk + 256 * t + 128, k[t % 3]);
      vt[t % 3] = as_lds(B.v)[8 * t + 4 * half + vc];
    };
    get(0);
    get(1);
#pragma unroll
    for (int t = 0; t < kScanTok; ++t) {
      if (!decltype(full)::value && t >= n) break;
      if (t + 2 < kScanTok) get(t + 2);
      asm volatile("" ::: "memory");
      const float (&kt)[8] = k[t % 3];
      const float gexp = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cg), 2 * t));
      const float beta = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cg), 2 * t + 1));
#pragma unroll
      for (int i = 0; i < 8; ++i) s[i] = s[i] * gexp;
      const float d = pair_odd((vt[t % 3] - scan_dot(s, kt)) * beta);
      if (kh == 0) as_lds_w(d_out)[4 * t + vc] = d;
#pragma unroll
      for (int i = 0; i < 8; ++i) s[i] = s[i] + kt[i] * d;
    }
  };
  auto runB = [&](int b, auto full, int n) {
    const ScanBlock& B = blk[b % 3];
    const float* d_in = dl[b & 1] + 32 * half;
    const float cg = as_lds(B.g)[lane & 15];
    float ov = 0.0f, k[3][8], q[3][8], d[3];
    auto get = [&](int t) {
      ld8(B.qk + 256 * t + 128, k[t % 3]);
      ld8(B.qk + 256 * t, q[t % 3]);
      d[t % 3] = as_lds(d_in)[4 * t + vc];
    };
    get(0);
    get(1);
#pragma unroll
    for (int t = 0; t < kScanTok; ++t) {
      if (!decltype(full)::value && t >= n) break;
      if (t + 2 < kScanTok) get(t + 2);
      asm volatile("" ::: "memory");
      const float gexp = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cg), 2 * t));
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        s[i] = s[i] * gexp;
        s[i] = s[i] + k[t % 3][i] * d[t % 3];
      }
      const float p = scan_dot(s, q[t % 3]);
      if (kg == t) ov = p;
    }
    if ((lane & 1) && kg < n) as_global_w(a.o)[(size_t)(b * kScanTok + kg) * 2048 + h * 128 + v] = ov;
  };
  using T = std::integral_constant<bool, true>;
  using F = std::integral_constant<bool, false>;
  fetch(0);
  put(0);
  if (nb > 1) fetch(1);
  lds_barrier();
#pragma unroll 1
  for (int b = 0; b <= nb; ++b) {   // A on block b, B on block b - 1; block b + 1 goes to LDS
    if (b + 1 < nb) {
      put(b + 1);
      if (b + 2 < nb) fetch(b + 2);
    }
    if (isA) {
      if (b < nb) {
        const int n = min(kScanTok, M - b * kScanTok);
        if (n == kScanTok) runA(b, T{}, n);
        else runA(b, F{}, n);
      }
    } else if (b > 0) {
      const int n = min(kScanTok, M - (b - 1) * kScanTok);
      if (n == kScanTok) runB(b - 1, T{}, n);
      else runB(b - 1, F{}, n);
    }
    lds_barrier();
  }
  if (isA) {
#pragma unroll
    for (int i = 0; i < 8; ++i) as_global_w(Sh)[(kh * 8 + i) * 128 + v] = s[i];
  }
}

// ---------------------------------------------------------------------------
// Gated RMSNorm (gemv_body's P_GATED prologue), one token per wave; the last
// workgroups advance the conv history by the group's tokens (the conv kernel's
// workgroups still read the old one).
// ---------------------------------------------------------------------------
template <int MODE>
__global__ __launch_bounds__(256) void pf_gated_kernel(const PfGated a) {
  const int nb = (a.M + 3) / 4;
  if ((int)blockIdx.x >= nb) {
    const int c = ((int)blockIdx.x - nb) * 256 + (int)threadIdx.x;   // channel
    f32x4* st = reinterpret_cast<f32x4*>(a.conv_state + (size_t)c * 4);
    const f32x4 old = *as_global(st);
    f32x4 nw;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = a.M - 4 + i;   // m >= -3: old column 4 + m
      nw[i] = m >= 0 ? as_global(a.y)[(size_t)m * 8192 + c] : (m == -1 ? old[3] : m == -2 ? old[2] : old[1]);
    }
    *as_global_w(st) = nw;
    return;
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = (int)blockIdx.x * 4 + wave;
  if (m >= a.M) return;
  float xv[2][16], zs[2][16], nw[16];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    load16g(a.o + (size_t)m * 2048 + 16 * (lane + 64 * j), xv[j]);
    load16g(a.y + (size_t)m * 8192 + 6144 + 16 * (lane + 64 * j), zs[j]);
  }
  load16g(a.nw + ((16 * lane) & 127), nw);   // the same gains for both chunks (64 chunks are whole heads)
  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    float ss = dot16_f32(xv[j], xv[j], 0.0f), mu = 0.0f;
    if constexpr (MODE == M_W8A8) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        xv[j][e] = (xv[j][e] * nw[e]) * zs[j][e];
        mu = fmaxf(mu, fabsf(xv[j][e]));
      }
    }
    ss = xor_sum<8>(ss);
    if constexpr (MODE == M_W8A8) mu = xor_max<8>(mu);
    const float inv = 1.0f / sqrtf(ss / 128.0f + a.eps);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      if constexpr (MODE == M_W8A8)
        xv[j][e] = xv[j][e] * inv;
      else
        xv[j][e] = ((xv[j][e] * inv) * nw[e]) * zs[j][e];
    }
    amax = fmaxf(amax, mu * inv);
  }
  if constexpr (MODE == M_W8A8) {
    const float xs = quant_scale(xor_max<64>(amax));
    const float rs = 1.0f / xs;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      int q[16];
      uint32_t pk[4];
      quant16(xv[j], xs, rs, q, pk);
      put_frag_i8<2048>(a.x, m, lane + 64 * j, pk);
    }
    if (lane == 0) a.xs[m] = xs;
  } else {
#pragma unroll
    for (int j = 0; j < 2; ++j) put_frag_f32<2048>(static_cast<float*>(a.x), m, lane + 64 * j, xv[j]);
  }
}

// ---------------------------------------------------------------------------
// Per-token activation quantisation of x [M][K] (gemv_body's P_LOAD prologue),
// one token per workgroup of K / 1024 (rounded up) waves.
// ---------------------------------------------------------------------------
template <int K>
__global__ __launch_bounds__(64 * pf_nch(K)) void pf_quant_kernel(void* xf, float* xso, const float* x) {
  constexpr int NW = pf_nch(K);
  __shared__ float sm[NW];
  const int c = threadIdx.x, lane = c & 63, wave = c >> 6, m = blockIdx.x;
  float xv[16];
  const bool in = c < K / 16;
  load16g(x + (size_t)m * K + 16 * min(c, K / 16 - 1), xv);
  float am = 0.0f;
#pragma unroll
  for (int e = 0; e < 16; ++e) am = fmaxf(am, fabsf(xv[e]));
  am = xor_max<64>(am);   // (a chunk past K repeats the last one)
  if (lane == 0) as_lds_w(sm)[wave] = am;
  lds_barrier();
  am = as_lds(sm)[0];
#pragma unroll
  for (int w = 1; w < NW; ++w) am = fmaxf(am, as_lds(sm)[w]);
  const float xs = quant_scale(am), rs = 1.0f / xs;
  int q[16];
  uint32_t pk[4];
  quant16(xv, xs, rs, q, pk);
  if (in) put_frag_i8<K>(xf, m, c, pk);
  if (c == 0) xso[m] = xs;
}

// ---------------------------------------------------------------------------
// QK-norm, RoPE and the new cache rows of the group's tokens (attn_new_pos's
// operations), one token per workgroup: waves 0, 1 the eight query heads (16
// lanes each), wave 2 the two key heads, wave 3 copies V.  Queries and keys also
// go out in fragment order.  Further workgroups bring the keys of the positions
// before the group into fragment order, one position each.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void put_qk_frag(float* base, int nh, int pos, int h, int c, const float (&v)[16]) {
  f32x4* p = reinterpret_cast<f32x4*>(base) + (((size_t)(pos >> 4) * nh + h) * 16 + c) * 64 + (pos & 15);
#pragma unroll
  for (int g = 0; g < 4; ++g) *as_global_w(p + 16 * g) = f32x4{v[g], v[4 + g], v[8 + g], v[12 + g]};
}
__global__ __launch_bounds__(256) void pf_qk_kernel(const PfAttn a) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g16 = lane & 15;
  if ((int)blockIdx.x >= a.M) {   // older keys, 8 positions per workgroup: 32 chunks of 16 each
    const int p = ((int)blockIdx.x - a.M) * 8 + (int)(threadIdx.x >> 5), c = threadIdx.x & 31;
    if (p >= a.pos0) return;
    float v[16];
    load16g(a.kc + (size_t)p * 512 + 16 * c, v);
    put_qk_frag(a.kf, 2, p, c >> 4, c & 15, v);
    return;
  }
  const int m = blockIdx.x, pos = a.pos0 + m;
  const float* row = a.qkv + (size_t)m * 5120;
  if (wave == 3) {
    const f32x4* src = reinterpret_cast<const f32x4*>(row + 4608) + lane;
    f32x4* dst = reinterpret_cast<f32x4*>(a.vc + (size_t)pos * 512) + lane;
    const f32x4 v0 = *as_global(src), v1 = *as_global(src + 64);
    *as_global_w(dst) = v0;
    *as_global_w(dst + 64) = v1;
    return;
  }
  const bool key = wave == 2;
  const int h = key ? (lane >> 4) & 1 : 4 * wave + (lane >> 4);
  float x[16], nw[16], cs[16], sn[16];
  load16g(row + (key ? 4096 + h * 256 : h * 512) + 16 * g16, x);
  load16g((key ? a.kn : a.qn) + 16 * g16, nw);
  load16g(a.rope + (size_t)pos * 64 + 16 * (g16 & 1), cs);
  load16g(a.rope + (size_t)pos * 64 + 32 + 16 * (g16 & 1), sn);
  qk_norm_rope(x, nw, a.eps, g16, cs, sn);
  if (key) {
    if (lane < 32) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        *as_global_w(reinterpret_cast<f32x4*>(a.kc + (size_t)pos * 512 + h * 256 + 16 * g16 + 4 * k)) =
            f32x4{x[4 * k], x[4 * k + 1], x[4 * k + 2], x[4 * k + 3]};
      put_qk_frag(a.kf, 2, pos, h, g16, x);
    }
  } else {
    put_qk_frag(a.qf, 8, pos - (a.pos0 & ~15), h, g16, x);
  }
}

// ---------------------------------------------------------------------------
// Attention of 16 queries (positions T0 .. T0 + 15, T0 a multiple of 16) of one
// head, contexts up to kAttnShortMax: attn_unit's 16-position splits, then the
// combine's fold in split order.  All splits below T0 are whole and shared by
// the 16 queries; query T0 + i has one more split of i positions (i > 0) and the
// split of its own position.
//   1  scores of every position into LDS (MFMA: keys are the rows of D, queries
//      the columns), wave w takes the position tiles w, w + 4, ...
//   2  16 threads per query: split maxima, p = exp(s - m), split sums, the
//      maximum over the splits, the weights exp(m - M) and L in split order
//   3  P.V: wave w takes dimensions 64 w .. + 63 (column j of tile td is
//      dimension 64 w + 4 j + td, so one 16-byte load feeds four tiles); whole
//      splits on the MFMA chain, the query's own partial split on the VALU
// The scores (16 x 2048 x 4 B) fill most of the LDS: one workgroup per CU.  The
// longest tiles start first.
// ---------------------------------------------------------------------------
template <int MODE>
__global__ __launch_bounds__(256, 1) void pf_attn_kernel(const PfAttn a) {
  extern __shared__ __attribute__((aligned(16))) float dyn[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, j = lane & 15;
  const int h = (int)blockIdx.x & 7, kvh = h >> 2;
  const int base = a.pos0 & ~15;                 // position of query tile 0
  const int qt = (int)(gridDim.x >> 3) - 1 - ((int)blockIdx.x >> 3);
  const int T0 = base + 16 * qt, na = T0 >> 4;   // whole splits below the tile
  const int last = a.pos0 + a.M - 1;             // the last position with a cache row
  const int ld = 16 * ((last >> 4) + 1) + 4;     // score row stride: 4 past a multiple of 16 (banks)
  float* sc = dyn;                               // [16][ld]
  float* sm = sc + 16 * ld;                      // [16][na + 2] split weights e
  const int lds_s = (last >> 4) + 3;
  float* sl = sm + 16 * lds_s;                   // [16][..] split sums l
  float* rL = sl + 16 * lds_s;                   // [16] 1 / L
  // ---- 1. scores
  {
    f32x4 qf[16];
    const f32x4* qp = reinterpret_cast<const f32x4*>(a.qf) + ((size_t)qt * 8 + h) * 16 * 64 + lane;
#pragma unroll
    for (int c = 0; c < 16; ++c) qf[c] = *as_global(qp + 64 * c);
    for (int t = wave; t <= na; t += 4) {
      const f32x4* kp = reinterpret_cast<const f32x4*>(a.kf) + ((size_t)t * 2 + kvh) * 16 * 64 + lane;
      f32x4 kf[16];
#pragma unroll
      for (int c = 0; c < 16; ++c) kf[c] = *as_global(kp + 64 * c);
      f32x4 st[5];
      // chunks in bit-reversed order: the 16-lane tree (offsets 8, 4, 2, 1) as a binary counter
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int c = ((i & 1) << 3) | ((i & 2) << 1) | ((i & 4) >> 1) | ((i & 8) >> 3);
        f32x4 r = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int e = 0; e < 4; ++e) r = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[c][e], qf[c][e], r, 0, 0, 0);
        if (i & 1) r = st[0] + r; else st[0] = r;
        if ((i & 3) == 3) r = st[1] + r; else if (i & 1) st[1] = r;
        if ((i & 7) == 7) r = st[2] + r; else if ((i & 3) == 3) st[2] = r;
        if (i == 15) r = st[3] + r; else if (i == 7) st[3] = r;
        st[4] = r;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) st[4][e] = st[4][e] * 0.0625f;
      *as_lds_w(reinterpret_cast<f32x4*>(sc + j * ld + 16 * t + 4 * g)) = st[4];   // query j, positions 16 t + 4 g ..
    }
  }
  __syncthreads();
  // ---- 2. softmax of query qi, by 16 threads (one 16-lane row of a wave)
  {
    const int qi = threadIdx.x >> 4, tj = threadIdx.x & 15;
    float* row = sc + qi * ld;
    const float snew = as_lds(row)[T0 + qi];   // the query's own position
    const int ns = na + (qi > 0 ? 1 : 0);      // splits before the own position's
    float M = snew;
    for (int s = tj; s < ns; s += 16) {
      const int cnt = s < na ? 16 : qi;
      float p[16], m = -__builtin_inff();
#pragma unroll
      for (int u = 0; u < 16; u += 4) {
        const f32x4 v = *as_lds(reinterpret_cast<const f32x4*>(row + 16 * s + u));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          p[u + e] = u + e < cnt ? v[e] : -__builtin_inff();
          m = fmaxf(m, p[u + e]);
        }
      }
#pragma unroll
      for (int u = 0; u < 16; ++u) p[u] = u < cnt ? dev_expf(p[u] - m) : 0.0f;
      float ap[4];
#pragma unroll
      for (int pg = 0; pg < 4; ++pg) ap[pg] = (p[pg] + p[8 + pg]) + (p[4 + pg] + p[12 + pg]);
      const float l = (ap[0] + ap[2]) + (ap[1] + ap[3]);
#pragma unroll
      for (int u = 0; u < 16; u += 4)
        *as_lds_w(reinterpret_cast<f32x4*>(row + 16 * s + u)) = f32x4{p[u], p[u + 1], p[u + 2], p[u + 3]};
      as_lds_w(sm)[qi * lds_s + s] = m;
      as_lds_w(sl)[qi * lds_s + s] = l;
      M = fmaxf(M, m);
    }
    M = xor_max<16>(M);
    for (int s = tj; s < ns; s += 16) {
      const float e = dev_expf(as_lds(sm)[qi * lds_s + s] - M);
      as_lds_w(sm)[qi * lds_s + s] = e;
      as_lds_w(sl)[qi * lds_s + s] = as_lds(sl)[qi * lds_s + s] * e;
    }
    const float en = dev_expf(snew - M);
    if (tj == 0) as_lds_w(sm)[qi * lds_s + na + 1] = en;
    lds_barrier();
    if (tj == 0) {
      float L = 0.0f;
      for (int s = 0; s < ns; ++s) L = L + as_lds(sl)[qi * lds_s + s];
      L = L + 1.0f * en;
      as_lds_w(rL)[qi] = 1.0f / L;
    }
  }
  __syncthreads();
  // ---- 3. P.V: lane (g, j) holds queries 4 g + r, dimensions d0 .. d0 + 3
  const int d0 = 64 * wave + 4 * j;
  const float* vb = a.vc + kvh * 256 + d0;
  float ctx[4][4];   // [r][td]
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int td = 0; td < 4; ++td) ctx[r][td] = 0.0f;
  f32x4 vn[4];
  auto vload = [&](int s) {
#pragma unroll
    for (int i = 0; i < 4; ++i) vn[i] = *as_global(reinterpret_cast<const f32x4*>(vb + (size_t)min(16 * s + 4 * i + g, last) * 512));
  };
  vload(0);
  for (int s = 0; s < na; ++s) {
    f32x4 vv[4];
    float p[4], e[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      vv[i] = vn[i];
      p[i] = as_lds(sc)[j * ld + 16 * s + 4 * i + g];
      e[i] = as_lds(sm)[(4 * g + i) * lds_s + s];
    }
    vload(s + 1);
    f32x4 acc[4];
#pragma unroll
    for (int td = 0; td < 4; ++td) acc[td] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int td = 0; td < 4; ++td) acc[td] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[i], vv[i][td], acc[td], 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int td = 0; td < 4; ++td) ctx[r][td] = ctx[r][td] + acc[td][r] * e[r];
  }
  // the own partial split (positions T0 .. T - 1), then the own position
  {
    float acc[4][4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int td = 0; td < 4; ++td) acc[r][td] = 0.0f;
    f32x4 own[4];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const f32x4 v = *as_global(reinterpret_cast<const f32x4*>(vb + (size_t)min(T0 + u, last) * 512));
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int qi = 4 * g + r;
        const float p = as_lds(sc)[qi * ld + T0 + u];
#pragma unroll
        for (int td = 0; td < 4; ++td) {
          const float t = __builtin_fmaf(p, v[td], acc[r][td]);
          acc[r][td] = u < qi ? t : acc[r][td];
        }
        if (u == qi) own[r] = v;
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int qi = 4 * g + r, m = T0 + qi - a.pos0;
      const float en = as_lds(sm)[qi * lds_s + na + 1], invL = as_lds(rL)[qi];
      const float ep = as_lds(sm)[qi * lds_s + na];   // read only for qi > 0
      const bool in = m >= 0 && m < a.M;
      f32x4 gate = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      if (in) gate = *as_global(reinterpret_cast<const f32x4*>(a.qkv + (size_t)m * 5120 + h * 512 + 256 + d0));
      f32x4 o;
#pragma unroll
      for (int td = 0; td < 4; ++td) {
        float x = ctx[r][td];
        if (qi > 0) x = x + acc[r][td] * ep;
        x = x + own[r][td] * en;
        o[td] = (x * invL) * dev_sigmoid(gate[td]);
      }
      if (in) {
        if constexpr (MODE == M_W8A8) {
          *as_global_w(reinterpret_cast<f32x4*>(a.og + (size_t)m * 2048 + h * 256 + d0)) = o;
        } else {   // elements 4 (j % 4) + td of chunk 16 h + 4 wave + j / 4
#pragma unroll
          for (int td = 0; td < 4; ++td)
            as_global_w(a.og)[pf_frag_f32(2048, m, 16 * h + 4 * wave + (j >> 2), 4 * (j & 3) + td)] = o[td];
        }
      }
    }
  }
}

// ===========================================================================
// Launches
// ===========================================================================
hipError_t pf_norm(const PfNorm& a, int mode, hipStream_t s) {
  const int grid = (a.M + 3) / 4;
  if (mode == M_W8A8) {
    if (a.gw != nullptr)
      pf_norm_kernel<M_W8A8, true><<<grid, 256, 0, s>>>(a);
    else
      pf_norm_kernel<M_W8A8, false><<<grid, 256, 0, s>>>(a);
  } else {
    if (a.gw != nullptr)
      pf_norm_kernel<M_W8A16, true><<<grid, 256, 0, s>>>(a);
    else
      pf_norm_kernel<M_W8A16, false><<<grid, 256, 0, s>>>(a);
  }
  return hipGetLastError();
}

namespace {
// Token tiles per workgroup: as few as keep the grid within 512 workgroups, at least `least`.  512 is one
// round of two workgroups per CU (a second, nearly empty round would cost as much as the first), which
// is what fits for every product but the fp32 one with K = 3584: its 144 KiB of LDS leave one per CU, so
// that at 768 tokens its 384 workgroups run in two rounds.
int tiles_per_wg(int row_tiles, int ntile, int least) {
  const int ny = 512 / row_tiles > 0 ? 512 / row_tiles : 1;
  int t = (ntile + ny - 1) / ny;
  t = (t + least - 1) / least * least;
  return t;
}
template <int K, int TA, int EPI>
hipError_t gemm_i8(const PfGemm& a, hipStream_t s) {
  const int ntile = (a.M + 15) / 16, rt = a.rows / (16 * TA), tpw = tiles_per_wg(rt, ntile, 4);
  pf_gemm_i8_kernel<K, TA, EPI><<<dim3(rt, (ntile + tpw - 1) / tpw), 256, 0, s>>>(a, tpw);
  return hipGetLastError();
}
template <int K, int RT, int KS, int EPI>
hipError_t gemm_f32(const PfGemm& a, hipStream_t s) {
  const int ntile = (a.M + 31) / 32, rt = a.rows / (32 * RT), tpw = tiles_per_wg(rt, ntile, 1);
  pf_gemm_f32_kernel<K, RT, KS, EPI><<<dim3(rt, (ntile + tpw - 1) / tpw), 64 * RT * KS, 0, s>>>(a, tpw);
  return hipGetLastError();
}
}  // namespace

hipError_t pf_gemm(const PfGemm& a, int K, PfEpi epi, int mode, hipStream_t s) {
  if (a.M < 1 || a.M > kPfGroup || a.rows % 64 != 0 || a.nseg < 1 || a.nseg > 3) return hipErrorInvalidValue;
  if (mode == M_W8A8) {
    if (K == 1024 && epi == PF_INPROJ) return gemm_i8<1024, 4, PF_INPROJ>(a, s);
    if (K == 1024 && epi == PF_STORE) return gemm_i8<1024, 4, PF_STORE>(a, s);
    if (K == 1024 && epi == PF_SWIGLU) return gemm_i8<1024, 4, PF_SWIGLU>(a, s);
    if (K == 2048 && epi == PF_RESID) return gemm_i8<2048, 1, PF_RESID>(a, s);
    if (K == 3584 && epi == PF_RESID) return gemm_i8<3584, 1, PF_RESID>(a, s);
  } else {
    if (K == 1024 && epi == PF_INPROJ) return gemm_f32<1024, 2, 2, PF_INPROJ>(a, s);
    if (K == 1024 && epi == PF_STORE) return gemm_f32<1024, 2, 2, PF_STORE>(a, s);
    if (K == 1024 && epi == PF_SWIGLU) return gemm_f32<1024, 2, 2, PF_SWIGLU>(a, s);
    if (K == 2048 && epi == PF_RESID) return gemm_f32<2048, 1, 4, PF_RESID>(a, s);
    if (K == 3584 && epi == PF_RESID) return gemm_f32<3584, 1, 8, PF_RESID>(a, s);
  }
  return hipErrorInvalidValue;
}

hipError_t pf_conv(const PfConv& a, hipStream_t s) {
  pf_conv_kernel<<<dim3((a.M + kConvTok - 1) / kConvTok, QH_CONV_DIM / kConvCh), 128, 0, s>>>(a);
  return hipGetLastError();
}
hipError_t pf_scan(const PfScan& a, hipStream_t s) {
  pf_scan_kernel<<<256, 256, 0, s>>>(a);
  return hipGetLastError();
}
hipError_t pf_gated(const PfGated& a, int mode, hipStream_t s) {
  const int grid = (a.M + 3) / 4 + QH_CONV_DIM / 256;
  if (mode == M_W8A8)
    pf_gated_kernel<M_W8A8><<<grid, 256, 0, s>>>(a);
  else
    pf_gated_kernel<M_W8A16><<<grid, 256, 0, s>>>(a);
  return hipGetLastError();
}
hipError_t pf_quant(void* xf, float* xs, const float* x, int K, int M, hipStream_t s) {
  if (K == 2048)
    pf_quant_kernel<2048><<<M, 64 * pf_nch(2048), 0, s>>>(xf, xs, x);
  else if (K == 3584)
    pf_quant_kernel<3584><<<M, 64 * pf_nch(3584), 0, s>>>(xf, xs, x);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}
hipError_t pf_qk(const PfAttn& a, hipStream_t s) {
  pf_qk_kernel<<<a.M + (a.pos0 + 7) / 8, 256, 0, s>>>(a);
  return hipGetLastError();
}
namespace {
constexpr int pf_attn_lds(int last) {   // bytes of a launch whose last cache row is `last` (pf_attn_kernel's dyn)
  return (int)sizeof(float) * (16 * (16 * ((last >> 4) + 1) + 4) + 2 * 16 * ((last >> 4) + 3) + 16);
}
}  // namespace
// The launches' limit is a property of the kernel, shared by every engine and thread of the process: it
// is set once, to the largest size, and never lowered between another thread's check and its launch.
hipError_t pf_attn_setup() {
  constexpr int lds = pf_attn_lds(kPfMaxPos - 1);
  static_assert(lds <= 160 * 1024, "one workgroup's LDS");
  for (const void* fn : {reinterpret_cast<const void*>(pf_attn_kernel<M_W8A8>), reinterpret_cast<const void*>(pf_attn_kernel<M_W8A16>)})
    if (const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds); e != hipSuccess) return e;
  return hipSuccess;
}
hipError_t pf_attn(const PfAttn& a, int mode, hipStream_t s) {
  const int last = a.pos0 + a.M - 1;
  if (a.M < 1 || last >= kPfMaxPos) return hipErrorInvalidValue;
  const int tiles = (last >> 4) - (a.pos0 >> 4) + 1;
  const size_t lds = pf_attn_lds(last);
  if (mode == M_W8A8)
    pf_attn_kernel<M_W8A8><<<8 * tiles, 256, lds, s>>>(a);
  else
    pf_attn_kernel<M_W8A16><<<8 * tiles, 256, lds, s>>>(a);
  return hipGetLastError();
}

}  // namespace qh
