// Prompt path: kernels that run one layer for a group of prompt tokens at once
// (qh_prefill.hip) and the driver that runs all layers of a group.  Every value
// equals the token-by-token decode's bit for bit.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qh_kernels.hpp"

namespace qh {

constexpr int kPfTile = 16;       // tokens per MFMA tile
constexpr int kPfGroup = 1024;    // the largest group (M of every launch)
constexpr int kPfSlots = 2;       // groups in flight
constexpr int kPfMaxPos = kAttnShortMax;   // positions the grouped attention covers (16-position splits)

// Activations in MFMA fragment order: the operand of one MFMA step is consecutive memory, 16 bytes
// per lane.
//   W8A8   int8: 16-element chunk c of token m (tile tt = m / 16, j = m % 16) at byte
//          (((tt * K/64 + c/4) * 4 + c%4) * 16 + j) * 16
//   W8A16  fp32: pf_frag_f32, token tiles of 32.  The chunks stand in the order the C16 sum visits
//          them: chunk c belongs to lane l = c % 64 of the 64-lane tree, lanes are visited in
//          bit-reversed order (so that the tree needs a stack of six partial sums instead of 64),
//          and a lane's chunks l, l + 64, ... follow one another.
__host__ __device__ constexpr int pf_bitrev6(int l) {
  return ((l & 1) << 5) | ((l & 2) << 3) | ((l & 4) << 1) | ((l & 8) >> 1) | ((l & 16) >> 3) | ((l & 32) >> 5);
}
__host__ __device__ constexpr int pf_nch(int K) { return (K + 1023) / 1024; }
__host__ __device__ constexpr int pf_frags(int K) { return 64 * pf_nch(K); }
__host__ __device__ constexpr int pf_visit(int K, int c) { return pf_bitrev6(c & 63) * pf_nch(K) + (c >> 6); }
// float index of element e of chunk c of token m: lane 32 (e % 2) + m % 32, element (e / 2) % 4 of
// its 16 bytes, half e / 8 of the chunk's two steps
__host__ __device__ constexpr size_t pf_frag_f32(int K, int m, int c, int e) {
  return ((((size_t)(m >> 5) * pf_frags(K) + pf_visit(K, c)) * 2 + (e >> 3)) * 64 + 32 * (e & 1) + (m & 31)) * 4 + ((e >> 1) & 3);
}

enum PfEpi : int {
  PF_INPROJ = 0,   // qkv rows stored, z rows through SiLU
  PF_STORE = 1,    // q || gate, k, v rows stored
  PF_SWIGLU = 2,   // gate / up row pairs: act = silu(gate) * up
  PF_RESID = 3,    // added to the residual stream
};

struct PfGemm {
  const int8_t* w[3] = {};    // weight segments in output order (PF_SWIGLU: gate, up)
  const float* sw[3] = {};
  int row0[3] = {};           // first output row of each segment (multiples of 64)
  int nseg = 1;
  int rows = 0;               // output rows (PF_SWIGLU: 2 x 3584 weight rows)
  const void* x = nullptr;    // fragments
  const float* xs = nullptr;  // per-token activation scales (W8A8)
  float* out = nullptr;       // [M][ld]; W8A16 PF_SWIGLU: fragments of K = 3584
  int ld = 0;
  int M = 0;
};

struct PfNorm {
  const float* h = nullptr;       // [M][1024] residual stream
  float* h_out = nullptr;         // set with emb: receives the embedded tokens
  const int8_t* emb = nullptr;    // layer 0: the embedding row of ids[m]
  const float* emb_s = nullptr;
  const int* ids = nullptr;
  const float* nw = nullptr;      // gains, lane-interleaved (load16c)
  float eps = 1e-6f;
  const float* gw = nullptr;      // DeltaNet gate rows wb | wa (lane-interleaved) or null
  const float* A_log = nullptr;
  const float* dt_bias = nullptr;
  float* gates = nullptr;         // [16 heads][M][2]: exp(g), beta
  void* x = nullptr;              // fragments, K = 1024
  float* xs = nullptr;
  int M = 0;
};

struct PfConv {
  const float* y = nullptr;       // [M][8192]: raw qkv rows (the first 6144 columns)
  const float* taps = nullptr;    // [6144][4]
  const float* state = nullptr;   // [6144][4]
  float* qk = nullptr;            // [16][M][256]: l2-normalised q, k (quad-interleaved, see pf_conv_kernel)
  float* v = nullptr;             // [16][M][128]
  int M = 0;
};

struct PfScan {
  const float* qk = nullptr;
  const float* v = nullptr;
  const float* gates = nullptr;
  float* S = nullptr;             // [16][128][128]
  float* o = nullptr;             // [M][2048]
  int M = 0;
};

struct PfGated {
  const float* o = nullptr;       // [M][2048]
  const float* y = nullptr;       // [M][8192]: columns 6144 .. 8191 hold silu(z)
  const float* nw = nullptr;      // [128]
  float eps = 1e-6f;
  void* x = nullptr;              // fragments, K = 2048
  float* xs = nullptr;
  float* conv_state = nullptr;    // advanced by the M tokens' raw qkv
  int M = 0;
};

struct PfAttn {
  const float* qkv = nullptr;     // [M][5120]: q || gate | k | v
  const float* qn = nullptr;
  const float* kn = nullptr;
  const float* rope = nullptr;    // [max_ctx][64]
  float* kc = nullptr;            // [max_ctx][512]
  float* vc = nullptr;
  float* qf = nullptr;            // query fragments  [tile][8][16 chunks][64][4]
  float* kf = nullptr;            // key fragments    [tile][2][16 chunks][64][4]
  float* og = nullptr;            // W8A8: [M][2048]; W8A16: fragments of K = 2048
  float eps = 1e-6f;
  int pos0 = 0;                   // position of the group's first token
  int M = 0;
};

hipError_t pf_norm(const PfNorm& a, int mode, hipStream_t s);
hipError_t pf_gemm(const PfGemm& a, int K, PfEpi epi, int mode, hipStream_t s);
hipError_t pf_conv(const PfConv& a, hipStream_t s);
hipError_t pf_scan(const PfScan& a, hipStream_t s);
hipError_t pf_gated(const PfGated& a, int mode, hipStream_t s);
hipError_t pf_qk(const PfAttn& a, hipStream_t s);
// once per engine, before its first pf_attn: the kernels' dynamic LDS limit
hipError_t pf_attn_setup();
hipError_t pf_attn(const PfAttn& a, int mode, hipStream_t s);
// rows of x [M][K] quantised into fragments (W8A8), K = 2048 or 3584
hipError_t pf_quant(void* xf, float* xs, const float* x, int K, int M, hipStream_t s);

}  // namespace qh
