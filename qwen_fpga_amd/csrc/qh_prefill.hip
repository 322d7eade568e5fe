// Grouped prompt kernels (gfx950): each launch runs one step of one layer for up
// to kPfGroup prompt tokens.  The decode path streams every weight byte once per
// token; here one read serves the whole group and the projections become matrix
// products on the matrix cores.
//
// Every value is the token path's, bit for bit, so that a prompt fed through
// here leaves exactly the state that feeding it token by token leaves:
//   * W8A8 products are int32 sums, exact in any order: v_mfma_i32_16x16x64_i8.
//   * W8A16 products follow the C16 order (qh_device.hpp).  v_mfma_f32_16x16x4_f32
//     computes, for each output, the chain fma(a3,b3,fma(a2,b2,fma(a1,b1,
//     fma(a0,b0,c)))) with single roundings and denormals kept (compared with
//     fmaf on 2^20 results), so a lane partial over a 16-element chunk is four
//     MFMAs from zero; the 64 partials are then added by the same tree.
//   * Attention scores (16-lane tree over 16-element chunks) and P.V (a chain in
//     position order) have the same shape and use the same instruction.
//   * Norms, gates, conv, the delta rule and the softmax repeat the decode
//     bodies' operations in their order.
#include "qh_prefill.hpp"
#include "qh_decode.h"
#include "qh_stages.hpp"

namespace qh {

typedef int i32x4 __attribute__((ext_vector_type(4)));

namespace {

// lane l's 16-element chunk c of token m, written to the fragments of a K-wide activation
template <int K>
__device__ __forceinline__ void put_frag_f32(float* x, int m, int c, const float (&v)[16]) {
  f32x4* p = reinterpret_cast<f32x4*>(x) + ((size_t)(m >> 4) * pf_frags(K) + pf_visit(K, c)) * 64 + (m & 15);
#pragma unroll
  for (int g = 0; g < 4; ++g) *as_global_w(p + 16 * g) = f32x4{v[g], v[4 + g], v[8 + g], v[12 + g]};
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
    float gw[8][16];
#pragma unroll
    for (int r = 0; r < 8; ++r) load16c(a.gw + (size_t)(8 * wave + r) * 1024, lane, gw[r]);
#pragma unroll
    for (int k = 0; k < 4; ++k)   // lane-interleaved, as load16c reads
      *as_lds_w(reinterpret_cast<f32x4*>(xl + 1024 * wave + 256 * k + 4 * lane)) =
          f32x4{xv[4 * k], xv[4 * k + 1], xv[4 * k + 2], xv[4 * k + 3]};
    lds_barrier();
    const int row = 8 * wave + row_of_lane<8>(lane);   // beta rows 0 .. 15, then g
    const int h = row & 15;
    const float al = as_global(a.A_log)[h], db = as_global(a.dt_bias)[h];
#pragma unroll 1
    for (int t = 0; t < 4; ++t) {
      if (m0 + t >= a.M) break;
      float x[16];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const f32x4 v = *as_lds(reinterpret_cast<const f32x4*>(xl + 1024 * t + 256 * k + 4 * lane));
#pragma unroll
        for (int e = 0; e < 4; ++e) x[4 * k + e] = v[e];
      }
      float p[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) p[r] = dot16_f32(gw[r], x, 0.0f);
      const float y = reduce8(p, lane);
      const float val = row < 16 ? dev_sigmoid(y) : dev_expf(-dev_expf(al) * dev_softplus(y + db));
      if ((lane & 7) == 0) a.gates[((size_t)h * a.M + m0 + t) * 2 + (row < 16 ? 1 : 0)] = val;
    }
  }
}

// ---------------------------------------------------------------------------
// Matrix product out[m][n] = sum_k w[n][k] x[m][k].  A workgroup owns TA * 16
// weight rows, copies them whole (K bytes each) to LDS once, and its four waves
// multiply them with TB token tiles each; x streams from L2 as fragments, 1 KiB
// per load instruction.  A (rows of D) = weight rows, B (columns) = tokens, so a
// lane ends with four consecutive outputs of one token.  A row's 16-byte chunk c
// sits at chunk c ^ (row & 15): the 16 rows a wave reads at once lie in 16
// different bank groups.
// Workgroups with the same rows are a multiple of 8 apart in the grid where the
// row tiles allow it, so one XCD's L2 serves them all.
// ---------------------------------------------------------------------------
template <int MODE, int K, int TA, int TB, int EPI>
__global__ __launch_bounds__(256) void pf_gemm_kernel(const PfGemm a) {
  constexpr int ROWS = 16 * TA, NC = K / 16;
  __shared__ __attribute__((aligned(16))) int8_t wl[ROWS * K];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, j = lane & 15;
  const int n0 = (int)blockIdx.x * ROWS;   // first output (PF_SWIGLU: weight) row
  // the workgroup's rows
  int si = 0;
  if constexpr (EPI != PF_SWIGLU) {
#pragma unroll
    for (int i = 1; i < 3; ++i)
      if (i < a.nseg && n0 >= a.row0[i]) si = i;
  }
  const int8_t* w0 = a.w[si];
  const int r0 = n0 - a.row0[si];
#pragma unroll 4
  for (int u = threadIdx.x; u < ROWS * NC; u += 256) {
    const int r = u / NC, c = u % NC;
    const int8_t* src;
    if constexpr (EPI == PF_SWIGLU) {   // 16-row blocks alternate gate, up
      const int t = r >> 4;
      src = ((t & 1) ? a.w[1] : a.w[0]) + (size_t)(n0 / 2 + (t >> 1) * 16 + (r & 15)) * K + 16 * c;
    } else {
      src = w0 + (size_t)(r0 + r) * K + 16 * c;
    }
    const u32x4 v = *as_global(reinterpret_cast<const u32x4*>(src));
    *as_lds_w(reinterpret_cast<u32x4*>(wl + r * K + 16 * (c ^ (r & 15)))) = v;
  }
  __syncthreads();
  const int ntile = (a.M + 15) >> 4;
  const int tt0 = ((int)blockIdx.y * 4 + wave) * TB;
  if (tt0 >= ntile) return;   // no barrier follows
  f32x4 y[TA][TB];
  if constexpr (MODE == M_W8A8) {
    i32x4 acc[TA][TB];
#pragma unroll
    for (int ta = 0; ta < TA; ++ta)
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) acc[ta][tb] = i32x4{0, 0, 0, 0};
    const i32x4* xp[TB];
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
      xp[tb] = reinterpret_cast<const i32x4*>(a.x) + (size_t)min(tt0 + tb, ntile - 1) * (K / 64) * 64 + lane;
    constexpr int PF = 4;   // steps of x in flight
    static_assert((K / 64) % PF == 0, "steps");
    i32x4 xb[PF][TB];
#pragma unroll
    for (int p = 0; p < PF; ++p)
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) xb[p][tb] = *as_global(xp[tb] + 64 * p);
#pragma unroll 1
    for (int s0 = 0; s0 < K / 64; s0 += PF) {
#pragma unroll
      for (int p = 0; p < PF; ++p) {
        const int s = s0 + p;
        i32x4 wa[TA];
#pragma unroll
        for (int ta = 0; ta < TA; ++ta)
          wa[ta] = *as_lds(reinterpret_cast<const i32x4*>(wl + (16 * ta + j) * K + 16 * ((4 * s + g) ^ j)));
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
          const i32x4 b = xb[p][tb];
          xb[p][tb] = *as_global(xp[tb] + 64 * min(s + PF, K / 64 - 1));
#pragma unroll
          for (int ta = 0; ta < TA; ++ta)
            acc[ta][tb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa[ta], b, acc[ta][tb], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
      const float xs = as_global(a.xs)[min(16 * (tt0 + tb) + j, a.M - 1)];
#pragma unroll
      for (int ta = 0; ta < TA; ++ta)
#pragma unroll
        for (int r = 0; r < 4; ++r) y[ta][tb][r] = (float)acc[ta][tb][r] * xs;
    }
  } else {
    static_assert(TB == 1, "one token tile per wave");
    constexpr int NCH = pf_nch(K);
    const f32x4* xp = reinterpret_cast<const f32x4*>(a.x) + (size_t)tt0 * pf_frags(K) * 64 + lane;
    f32x4 t0[TA], t1[TA], t2[TA];
    // Eight lanes' partials (visits 8 w8 .. 8 w8 + 7) and their three tree levels at a time; a
    // visit's x is replaced by the visit's eight later as soon as it is read.
    f32x4 xb[8 * NCH];
    auto xload = [&](int w8, int i) { return *as_global(xp + 64 * (8 * NCH * min(w8, 7) + i)); };
#pragma unroll
    for (int i = 0; i < 8 * NCH; ++i) xb[i] = xload(0, i);
#pragma unroll 1
    for (int w8 = 0; w8 < 8; ++w8) {
      // lane of the tree: bit-reversed visit; its low three bits come from w8
      const int lb = ((w8 >> 2) & 1) | (w8 & 2) | ((w8 & 1) << 2);
      f32x4 part[8][TA];   // (folded as soon as a pair is complete; at most four are live)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int l = lb + 8 * (((i >> 2) & 1) | (i & 2) | ((i & 1) << 2));
#pragma unroll
        for (int ta = 0; ta < TA; ++ta) part[i][ta] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int jj = 0; jj < NCH; ++jj) {
          if (64 * jj + 32 >= NC && (i & 1)) continue;   // chunk past K: only lanes below 32 hold it (odd visits: lanes 32 ..)
          const int c = l + 64 * jj;
          const f32x4 b = xb[i * NCH + jj];
          xb[i * NCH + jj] = xload(w8 + 1, i * NCH + jj);
#pragma unroll
          for (int ta = 0; ta < TA; ++ta) {
            const u32x4 wv = *as_lds(reinterpret_cast<const u32x4*>(wl + (16 * ta + j) * K + 16 * (c ^ j)));
            // elements g, 4 + g, 8 + g, 12 + g: byte g of the four dwords
            const float f0 = (float)(int)(int8_t)(wv[0] >> (8 * g)), f1 = (float)(int)(int8_t)(wv[1] >> (8 * g)),
                        f2 = (float)(int)(int8_t)(wv[2] >> (8 * g)), f3 = (float)(int)(int8_t)(wv[3] >> (8 * g));
            part[i][ta] = __builtin_amdgcn_mfma_f32_16x16x4f32(f0, b[0], part[i][ta], 0, 0, 0);
            part[i][ta] = __builtin_amdgcn_mfma_f32_16x16x4f32(f1, b[1], part[i][ta], 0, 0, 0);
            part[i][ta] = __builtin_amdgcn_mfma_f32_16x16x4f32(f2, b[2], part[i][ta], 0, 0, 0);
            part[i][ta] = __builtin_amdgcn_mfma_f32_16x16x4f32(f3, b[3], part[i][ta], 0, 0, 0);
          }
        }
        if (i & 1) {   // the tree's levels at offsets 32, 16, 8
#pragma unroll
          for (int ta = 0; ta < TA; ++ta) {
            part[i - 1][ta] = part[i - 1][ta] + part[i][ta];
            if ((i & 3) == 3) part[i - 3][ta] = part[i - 3][ta] + part[i - 1][ta];
            if (i == 7) part[0][ta] = part[0][ta] + part[4][ta];
          }
        }
      }
      // offsets 4, 2, 1: a binary counter over the eight groups of eight
#pragma unroll
      for (int ta = 0; ta < TA; ++ta) {
        f32x4 r = part[0][ta];
        if (w8 & 1) r = t0[ta] + r;
        else t0[ta] = r;
        if ((w8 & 3) == 3) r = t1[ta] + r;
        else if (w8 & 1) t1[ta] = r;
        if (w8 == 7) r = t2[ta] + r;
        else if (w8 == 3) t2[ta] = r;
        y[ta][0] = r;
      }
    }
  }
  // ---- epilogue: token m, outputs 16 ta + 4 g .. + 3 of the row tile
#pragma unroll
  for (int tb = 0; tb < TB; ++tb) {
    const int m = 16 * (tt0 + tb) + j;
    if (tt0 + tb >= ntile || m >= a.M) continue;
    if constexpr (EPI == PF_SWIGLU) {
#pragma unroll
      for (int ta = 0; ta < TA; ta += 2) {
        const int n = n0 / 2 + (ta >> 1) * 16 + 4 * g;
        const f32x4 sg = *as_global(reinterpret_cast<const f32x4*>(a.sw[0] + n));
        const f32x4 su = *as_global(reinterpret_cast<const f32x4*>(a.sw[1] + n));
        f32x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = dev_silu(y[ta][tb][r] * sg[r]) * (y[ta + 1][tb][r] * su[r]);
        if constexpr (MODE == M_W8A8) {
          *as_global_w(reinterpret_cast<f32x4*>(a.out + (size_t)m * a.ld + n)) = v;
        } else {   // element 4 g + r of chunk n / 16: fragment lane group r, position g
          const int c = n >> 4;
          float* p = a.out + (((size_t)(m >> 4) * pf_frags(QH_INTER) + pf_visit(QH_INTER, c)) * 64 + (m & 15)) * 4 + g;
#pragma unroll
          for (int r = 0; r < 4; ++r) as_global_w(p)[64 * r] = v[r];
        }
      }
    } else {
#pragma unroll
      for (int ta = 0; ta < TA; ++ta) {
        const int n = n0 + 16 * ta + 4 * g;
        const f32x4 sw = *as_global(reinterpret_cast<const f32x4*>(a.sw[si] + (n - a.row0[si])));
        f32x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = y[ta][tb][r] * sw[r];
        f32x4* p = reinterpret_cast<f32x4*>(a.out + (size_t)m * a.ld + n);
        if constexpr (EPI == PF_INPROJ) {
          if (si == 1)
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
  }
}

// ---------------------------------------------------------------------------
// Short conv + SiLU of the raw qkv rows, then the l2norm of q and k (and q's
// 1 / sqrt(128)): thread c takes channels 16 c .. 16 c + 15 (one k-group of a
// head) for kConvTok tokens in a row, its window in registers.  q and k of
// (head, token) go to 256 floats: element e of k-group kg of q at
// (e / 4) * 32 + 4 kg + e % 4, k 128 further (the order the scan's lanes read).
// ---------------------------------------------------------------------------
constexpr int kConvTok = 4;
__global__ __launch_bounds__(384) void pf_conv_kernel(const PfConv a) {
  const int c = threadIdx.x, ch = 16 * c;
  const int m0 = (int)blockIdx.x * kConvTok;
  float taps[16][4];
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const f32x4 t = *as_global(reinterpret_cast<const f32x4*>(a.taps + (size_t)(ch + e) * 4));
#pragma unroll
    for (int k = 0; k < 4; ++k) taps[e][k] = t[k];
  }
  float w1[16], w2[16], w3[16];   // the window's older inputs, oldest first
  auto row = [&](int m, float (&v)[16]) {   // input m of the group; before it, the state's columns 1 .. 3
    if (m >= 0) {
      load16g(a.y + (size_t)m * 8192 + ch, v);
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] = as_global(a.state)[(size_t)(ch + e) * 4 + 4 + m];
    }
  };
  row(m0 - 3, w1);
  row(m0 - 2, w2);
  row(m0 - 1, w3);
  const int part = c >> 7, h = (c & 127) >> 3, kg = c & 7;   // q, k or v; head; k-group
#pragma unroll 1
  for (int m = m0; m < min(m0 + kConvTok, a.M); ++m) {
    float y[16], x[16];
    row(m, y);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      float acc = 0.0f;
      acc = acc + w1[e] * taps[e][0];
      acc = acc + w2[e] * taps[e][1];
      acc = acc + w3[e] * taps[e][2];
      acc = acc + y[e] * taps[e][3];
      x[e] = dev_silu(acc);
      w1[e] = w2[e];
      w2[e] = w3[e];
      w3[e] = y[e];
    }
    if (part < 2) {   // deltanet.hpp:134,166-169 (whole waves: c / 128 is wave-uniform)
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
      float* p = a.qk + ((size_t)h * a.M + m) * 256 + 128 * part + 4 * kg;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        *as_global_w(reinterpret_cast<f32x4*>(p + 32 * k)) = f32x4{x[4 * k], x[4 * k + 1], x[4 * k + 2], x[4 * k + 3]};
    } else {
      float* p = a.v + ((size_t)h * a.M + m) * 128 + 16 * kg;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        *as_global_w(reinterpret_cast<f32x4*>(p + 4 * k)) = f32x4{x[4 * k], x[4 * k + 1], x[4 * k + 2], x[4 * k + 3]};
    }
  }
}

// ---------------------------------------------------------------------------
// The delta rule over the group's tokens in order (deltanet_body's operations):
// one wave per workgroup and 8 columns of one head, 256 workgroups, so every
// wave has a CU's vector memory and LDS paths to itself; the wave's 128 x 8
// slice of S stays in registers for the whole group.  Bound by its own serial
// chain of about 125 vector instructions per token; q, k, v and the gates of the
// next eight tokens are in flight while eight are computed.
// ---------------------------------------------------------------------------
constexpr int kScanTok = 8;
__global__ __launch_bounds__(64, 1) void pf_scan_kernel(const PfScan a) {
  __shared__ __attribute__((aligned(16))) float qkl[2][kScanTok * 256];
  __shared__ __attribute__((aligned(16))) float vl[2][64];
  const int lane = threadIdx.x, kg = lane & 7, vc = lane >> 3;
  const int h = (int)blockIdx.x >> 4, v = ((int)blockIdx.x & 15) * 8 + vc;
  const int M = a.M;
  float* Sh = a.S + (size_t)h * 128 * 128;
  float s[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) s[i] = as_global(Sh)[(kg * 16 + i) * 128 + v];
  const float* qk = a.qk + (size_t)h * M * 256;
  const float* vp = a.v + (size_t)h * M * 128;
  const float* gp = a.gates + (size_t)h * M * 2;
  f32x4 nq[kScanTok];
  float nv, ng;   // lane: v of token lane & 7, column lane >> 3; gate lane & 1 of token (lane >> 1) & 7
  auto fetch = [&](int m0) {
#pragma unroll
    for (int t = 0; t < kScanTok; ++t)
      nq[t] = *as_global(reinterpret_cast<const f32x4*>(qk + (size_t)min(m0 + t, M - 1) * 256 + 4 * lane));
    nv = as_global(vp)[(size_t)min(m0 + kg, M - 1) * 128 + v];
    ng = as_global(gp)[(size_t)min(m0 + ((lane >> 1) & 7), M - 1) * 2 + (lane & 1)];
  };
  fetch(0);
  int buf = 0;
#pragma unroll 1
  for (int m0 = 0; m0 < M; m0 += kScanTok, buf ^= 1) {
#pragma unroll
    for (int t = 0; t < kScanTok; ++t) *as_lds_w(reinterpret_cast<f32x4*>(&qkl[buf][256 * t + 4 * lane])) = nq[t];
    as_lds_w(vl[buf])[lane] = nv;
    const float cg = ng;
    lds_barrier();   // one wave: orders its own LDS writes and reads
    if (m0 + kScanTok < M) fetch(m0 + kScanTok);
    const int n = min(kScanTok, M - m0);
    float ov = 0.0f;
#pragma unroll
    for (int t = 0; t < kScanTok; ++t) {
      if (t < n) {
        float q[16], k[16];
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
          const f32x4 x = *as_lds(reinterpret_cast<const f32x4*>(&qkl[buf][256 * t + 32 * qd + 4 * kg]));
          const f32x4 z = *as_lds(reinterpret_cast<const f32x4*>(&qkl[buf][256 * t + 128 + 32 * qd + 4 * kg]));
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            q[4 * qd + e] = x[e];
            k[4 * qd + e] = z[e];
          }
        }
        const float vt = as_lds(vl[buf])[8 * vc + t];
        const float gexp = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cg), 2 * t));
        const float beta = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cg), 2 * t + 1));
        float p = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[i] = s[i] * gexp;
          p = p + s[i] * k[i];
        }
        p = xor_sum<8>(p);
        const float d = (vt - p) * beta;
        p = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[i] = s[i] + k[i] * d;
          p = p + s[i] * q[i];
        }
        p = xor_sum<8>(p);
        if (kg == t) ov = p;
      }
    }
    if (kg < n) as_global_w(a.o)[(size_t)(m0 + kg) * 2048 + h * 128 + v] = ov;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) as_global_w(Sh)[(kg * 16 + i) * 128 + v] = s[i];
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
          const int c = 16 * h + 4 * wave + (j >> 2);
          float* p = a.og + (((size_t)(m >> 4) * pf_frags(2048) + pf_visit(2048, c)) * 64 + (m & 15)) * 4 + (j & 3);
#pragma unroll
          for (int td = 0; td < 4; ++td) as_global_w(p)[64 * td] = o[td];
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
template <int MODE, int K, int TA, int EPI>
hipError_t gemm_launch(const PfGemm& a, hipStream_t s) {
  const int ntile = (a.M + 15) / 16;
  const dim3 grid(a.rows / (16 * TA), (ntile + 3) / 4);
  pf_gemm_kernel<MODE, K, TA, 1, EPI><<<grid, 256, 0, s>>>(a);
  return hipGetLastError();
}
template <int MODE>
hipError_t gemm_mode(const PfGemm& a, int K, PfEpi epi, hipStream_t s) {
  if (K == 1024 && epi == PF_INPROJ) return gemm_launch<MODE, 1024, 4, PF_INPROJ>(a, s);
  if (K == 1024 && epi == PF_STORE) return gemm_launch<MODE, 1024, 4, PF_STORE>(a, s);
  if (K == 1024 && epi == PF_SWIGLU) return gemm_launch<MODE, 1024, 4, PF_SWIGLU>(a, s);
  if (K == 2048 && epi == PF_RESID) return gemm_launch<MODE, 2048, 2, PF_RESID>(a, s);
  if (K == 3584 && epi == PF_RESID) return gemm_launch<MODE, 3584, 2, PF_RESID>(a, s);
  return hipErrorInvalidValue;
}
}  // namespace

hipError_t pf_gemm(const PfGemm& a, int K, PfEpi epi, int mode, hipStream_t s) {
  if (a.M < 1 || a.M > kPfGroup || a.rows % 64 != 0 || a.nseg < 1 || a.nseg > 3) return hipErrorInvalidValue;
  return mode == M_W8A8 ? gemm_mode<M_W8A8>(a, K, epi, s) : gemm_mode<M_W8A16>(a, K, epi, s);
}

hipError_t pf_conv(const PfConv& a, hipStream_t s) {
  pf_conv_kernel<<<(a.M + kConvTok - 1) / kConvTok, 384, 0, s>>>(a);
  return hipGetLastError();
}
hipError_t pf_scan(const PfScan& a, hipStream_t s) {
  pf_scan_kernel<<<256, 64, 0, s>>>(a);
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
hipError_t pf_attn(const PfAttn& a, int mode, hipStream_t s) {
  const int last = a.pos0 + a.M - 1;
  if (a.M < 1 || last >= kPfMaxPos) return hipErrorInvalidValue;
  const int tiles = (last >> 4) - (a.pos0 >> 4) + 1;
  const size_t lds = sizeof(float) * (16 * (16 * ((last >> 4) + 1) + 4) + 2 * 16 * ((last >> 4) + 3) + 16);
  const void* fn = mode == M_W8A8 ? reinterpret_cast<const void*>(pf_attn_kernel<M_W8A8>)
                                  : reinterpret_cast<const void*>(pf_attn_kernel<M_W8A16>);
  if (const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); e != hipSuccess)
    return e;
  if (mode == M_W8A8)
    pf_attn_kernel<M_W8A8><<<8 * tiles, 256, lds, s>>>(a);
  else
    pf_attn_kernel<M_W8A16><<<8 * tiles, 256, lds, s>>>(a);
  return hipGetLastError();
}

}  // namespace qh
