// gemm_chains.hip — the matmul of a few tokens, of grids too small for gemm.hip's blocks, and of bias 0, on CDNA4 i8
// MFMA with each of the four float32 lane chains on a wave of its own. The arithmetic is gemm.hip's (bias 64:
// kernels/kernel_relaxed.ts:34-67 matmul_q8r, :189-218 matmul_q6r) or the plain kernels' (bias 0: kernels/kernel.ts:
// 231-258 matmul_q8, :261-278 matmul_q6), every output to the bit:
//   bias 64: chain c adds f32(S_g) * f32(ws_g * xs_g) of the groups g = c (mod 4) below 4 * floor(G / 4), in order; the
//            chains are added ((l0 + l1) + l2) + l3, then the up to three groups past the fours one at a time.
//   bias 0:  chain k adds f32(S_gk) * f32(ws_g * xs_g) of every group in order, S_gk the sum of the group's products
//            2k, 2k + 1, 2k + 8, 2k + 9 of each half of 16; the four chains added in order.
// The chains never meet before the end, so they are the one split of K that the order allows: a row's K is read by four
// waves instead of one.
//
// Tiling: v_mfma_i32_16x16x32_i8 makes the exact group sums of 16 rows x 16 tokens. A wave makes RT x TT such tiles of
// one chain; a block is RB x 4 waves (RB row parts, 4 chains) on RB * RT * 16 rows and TT * 16 tokens. A stage is CK = 16
// or 8 groups (512 or 256 bytes of K: launch_tile) of the block's rows, tokens and scales in LDS, double buffered, and the
// loads of the stage after the next are in flight in registers: two stages' loads cover the memory's latency where a CU
// holds one block.
// For bias 0 the staging turns each half of a group's bytes so that lane sum k's 8 bytes lie side by side: the A operand
// of chain k's wave is then the group's bytes in the lanes that hold part k and zeros in the others.
#pragma clang fp contract(off)

#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace ple {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

// the accumulators' start and the float32 it stands for (gemm.hip MAGIC: f32(S) as one subtraction)
constexpr int MAGIC = 0x4B400000;
constexpr float MAGIC_F = 12582912.0f;

// what a block does with its outputs: stores them (or finishes q / k / v: a.qkv), or finishes the FFN's activation and its
// quantize_x (a.glu)
enum { EPI_STORE = 0, EPI_GLU, EPI_GELU };

// quantize_x(bias 0)'s lane sums: the 16 bytes of half a group as the four words of lane sums 0..3 (word k: bytes 2k,
// 2k + 1, 2k + 8, 2k + 9)
__device__ __forceinline__ void lane_words(uint4 v, uint32_t (&o)[4]) {
  o[0] = __builtin_amdgcn_perm(v.z, v.x, 0x05040100u);
  o[1] = __builtin_amdgcn_perm(v.z, v.x, 0x07060302u);
  o[2] = __builtin_amdgcn_perm(v.w, v.y, 0x05040100u);
  o[3] = __builtin_amdgcn_perm(v.w, v.y, 0x07060302u);
}

// four rows (row, row + 1, .. of the launch's q, k and v rows, all of one segment: every segment is whole heads) of token t
// finished as qkv_post_kernel does: + bias, RoPE's two pairs of q and k, q stored, k and v into the cache
__device__ __forceinline__ void finish_qkv(const MatArgs &a, int row, int t, const float (&s)[4]) {
  if (row >= a.total_rows) return;
  const QkvFuse &f = a.qkv;
  const int n0 = a.seg[0].rows, n1 = a.seg[1].rows;
  const int seg = row < n0 ? 0 : (row < n0 + n1 ? 1 : 2), r = row - (seg == 0 ? 0 : (seg == 1 ? n0 : n0 + n1));
  const int pos = (f.dpos ? *f.dpos : f.pos) + t;
  const float *bias = seg == 0 ? f.bq : (seg == 1 ? f.bk : f.bv);
  float v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = bias ? s[j] + bias[r + j] : s[j];
  if (seg < 2) {
#pragma unroll
    for (int j = 0; j < 4; j += 2) {
      const int at = (r + j) % f.hs;
      if (at < f.rot) {
        const float c = f.cos_t[(int64_t)pos * (f.hs / 2) + at / 2], sn = f.sin_t[(int64_t)pos * (f.hs / 2) + at / 2];
        const float v0 = v[j], v1 = v[j + 1];
        v[j] = v0 * c - v1 * sn;
        v[j + 1] = v0 * sn + v1 * c;
      }
    }
  }
  if (seg == 0) {
    float *y = a.seg[0].y + (int64_t)t * a.seg[0].y_stride + r;
#pragma unroll
    for (int j = 0; j < 4; ++j) y[j] = v[j];
    return;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t at = seg == 1 ? (int64_t)pos * f.kvdim + r + j : (int64_t)(r + j) * f.vstride + pos;
    void *cache = seg == 1 ? f.kcache : f.vcache;
    if (f.half) reinterpret_cast<uint16_t *>(cache)[at] = to_f16(v[j]);
    else reinterpret_cast<float *>(cache)[at] = v[j];
  }
}

template <bool SIX, bool PLAIN, int RT, int TT, int RB, int CK, int D, int EPI>
struct Chains {
  static constexpr int NT = 256 * RB;                    // threads
  static constexpr int PITCH = CK * 32 + 16;  // LDS bytes of a row of a stage: 16 rows' 8-byte reads fall on distinct banks
  static constexpr int ROWS = RB * RT * 16;              // rows a block
  static constexpr int TOKENS = TT * 16;                 // tokens a block
  static constexpr int WSP = ROWS + 4, XSP = TOKENS + 4;  // floats of a group's scales in LDS
  static constexpr int WUNITS = SIX ? ROWS * CK : ROWS * CK * 2;  // a thread's loads: int6 a group, int8 16 bytes
  static constexpr int XUNITS = TOKENS * CK * 2;
  static constexpr int NW = (WUNITS + NT - 1) / NT, NX = (XUNITS + NT - 1) / NT;
  static constexpr int NWS = (ROWS * CK + NT - 1) / NT, NXS = (TOKENS * CK + NT - 1) / NT;
  static constexpr int STAGE = ROWS * PITCH + TOKENS * PITCH + 4 * CK * (WSP + XSP);  // bytes
  static constexpr int XCH = 4 * 4 * 64 * 4 * RB * RT * TT;  // bytes of the chains' hand-over
  static constexpr int LDS = 2 * STAGE > XCH ? 2 * STAGE : XCH;
  struct Fetch {
    uint32_t w[NW][SIX ? 6 : 4];
    uint4 x[NX];
    float ws[NWS], xs[NXS];
  };
};

template <bool SIX, bool PLAIN, int RT, int TT, int RB, int CK, int D, int EPI>
__global__ __launch_bounds__(256 * RB) __attribute__((amdgpu_waves_per_eu(2))) void gemm_chains_kernel(const MatArgs a) {
  using P = Chains<SIX, PLAIN, RT, TT, RB, CK, D, EPI>;
  constexpr bool GLU = EPI == EPI_GLU;
  static_assert(!GLU || (RB == 2 && RT == 2), "the SwiGLU's blocks are 32 units of w1 and of w3");
  static_assert(EPI != EPI_GELU || RB * RT == 2, "the GELU's blocks are 32 units");
  constexpr int NT = P::NT, PITCH = P::PITCH;
  extern __shared__ float4 lds4[];
  uint8_t *const lds = reinterpret_cast<uint8_t *>(lds4);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int chain = wave & 3, sub = wave >> 2, l16 = lane & 15, q = lane >> 4;
  // block b runs on XCD b % 8: the (row block, token block) pairs, row-block major, dealt to the XCDs in 8 contiguous
  // ranges, so that a row block's token blocks read its weights from one XCD's L2
  const int tbn = (a.m + P::TOKENS - 1) / P::TOKENS, nblk = gridDim.x;
  const int xcd = blockIdx.x % 8, idx = xcd * (nblk / 8) + min(xcd, nblk % 8) + blockIdx.x / 8;
  const int r0 = (idx / tbn) * (GLU ? P::ROWS / 2 : P::ROWS), t0 = (idx % tbn) * P::TOKENS;
  const int G = a.k / GS;

  // the loads' places: rows and tokens past the end clamped (loaded, never stored to y); a group past the last clamped
  // in the loop (loaded, never added)
  const int n0 = a.seg[0].rows, n1 = a.seg[1].rows;
  auto row_at = [&](int br, const uint8_t **w, const float **ws) {
    int r;
    if constexpr (GLU) {
      r = min(r0 + (br >> 5) * 16 + (br & 15), n0 - 1);
      const bool second = (br & 16) != 0;
      *w = second ? a.seg[1].w : a.seg[0].w;
      *ws = second ? a.seg[1].ws : a.seg[0].ws;
    } else {
      r = min(r0 + br, a.total_rows - 1);
      const bool third = a.nseg > 2 && r >= n0 + n1, second = a.nseg > 1 && r >= n0;
      *w = third ? a.seg[2].w : (second ? a.seg[1].w : a.seg[0].w);
      *ws = third ? a.seg[2].ws : (second ? a.seg[1].ws : a.seg[0].ws);
      r -= third ? n0 + n1 : (second ? n0 : 0);
    }
    *w += (int64_t)r * (SIX ? (int64_t)G * 24 : (int64_t)a.k);
    *ws += (int64_t)r * G;
  };
  const uint8_t *wp[P::NW];
  const float *wsp[P::NWS];
  const int8_t *xp[P::NX];
  const float *xsp[P::NXS];
#pragma unroll
  for (int i = 0; i < P::NW; ++i) {
    const float *unused;
    row_at(min((tid + NT * i) / (SIX ? CK : 2 * CK), P::ROWS - 1), &wp[i], &unused);
  }
#pragma unroll
  for (int i = 0; i < P::NWS; ++i) {
    const uint8_t *unused;
    row_at(min((tid + NT * i) / CK, P::ROWS - 1), &unused, &wsp[i]);
  }
#pragma unroll
  for (int i = 0; i < P::NX; ++i)
    xp[i] = a.xq + (int64_t)min(t0 + min((tid + NT * i) / (2 * CK), P::TOKENS - 1), a.m - 1) * a.xq_stride;
#pragma unroll
  for (int i = 0; i < P::NXS; ++i) xsp[i] = a.xs + (int64_t)min(t0 + min((tid + NT * i) / CK, P::TOKENS - 1), a.m - 1) * a.xs_stride;
  // the group (of a stage) of this thread's loads: the same in each of its units
  const uint32_t gw = SIX ? tid % CK : (tid % (2 * CK)) / 2, gx = (tid % (2 * CK)) / 2, gs = tid % CK;
  const uint32_t half = (tid & 1) * 16;

  auto fetch = [&](typename P::Fetch &f, int s) {
    const uint32_t g0 = s * CK, most = G - 1;
    const uint32_t at = min(g0 + gw, most);
#pragma unroll
    for (int i = 0; i < P::NW; ++i) {
      if constexpr (SIX) {
        const uint2 *p = reinterpret_cast<const uint2 *>(wp[i] + at * 24);
        const uint2 l0 = p[0], l1 = p[1], tops = p[2];
        f.w[i][0] = l0.x; f.w[i][1] = l0.y; f.w[i][2] = l1.x; f.w[i][3] = l1.y; f.w[i][4] = tops.x; f.w[i][5] = tops.y;
      } else {
        const uint4 v = *reinterpret_cast<const uint4 *>(wp[i] + at * 32 + half);
        f.w[i][0] = v.x; f.w[i][1] = v.y; f.w[i][2] = v.z; f.w[i][3] = v.w;
      }
    }
    const uint32_t ax = min(g0 + gx, most), as = min(g0 + gs, most);
#pragma unroll
    for (int i = 0; i < P::NX; ++i) f.x[i] = *reinterpret_cast<const uint4 *>(xp[i] + ax * 32 + half);
#pragma unroll
    for (int i = 0; i < P::NWS; ++i) f.ws[i] = wsp[i][as];
#pragma unroll
    for (int i = 0; i < P::NXS; ++i) f.xs[i] = xsp[i][as];
  };
  // half a group's 16 bytes into a row of a stage (bias 0: each lane sum's word beside its other half's)
  auto put = [&](uint8_t *row, int g, int h, uint4 v) {
    if constexpr (PLAIN) {
      uint32_t o[4];
      lane_words(v, o);
      uint32_t *d = reinterpret_cast<uint32_t *>(row + g * 32 + h / 4);
#pragma unroll
      for (int k = 0; k < 4; ++k) d[2 * k] = o[k];
    } else {
      *reinterpret_cast<uint4 *>(row + g * 32 + h) = v;
    }
  };
  auto store = [&](const typename P::Fetch &f, int buf) {
    uint8_t *const wl = lds + buf * P::STAGE, *const xl = wl + P::ROWS * PITCH;
    float *const wsl = reinterpret_cast<float *>(xl + P::TOKENS * PITCH), *const xsl = wsl + CK * P::WSP;
#pragma unroll
    for (int i = 0; i < P::NW; ++i) {
      if constexpr (SIX) {
        const uint32_t L[4] = {f.w[i][0], f.w[i][1], f.w[i][2], f.w[i][3]};
        uint32_t w[8];
        six_widen(L, f.w[i][4], f.w[i][5], w);
        uint8_t *row = wl + min((tid + NT * i) / CK, P::ROWS - 1) * PITCH;
        put(row, gw, 0, make_uint4(w[0], w[1], w[2], w[3]));
        put(row, gw, 16, make_uint4(w[4], w[5], w[6], w[7]));
      } else {
        put(wl + min((tid + NT * i) / (2 * CK), P::ROWS - 1) * PITCH, gw, half,
            make_uint4(f.w[i][0], f.w[i][1], f.w[i][2], f.w[i][3]));
      }
    }
#pragma unroll
    for (int i = 0; i < P::NX; ++i) {
      uint4 v = f.x[i];
      if constexpr (!PLAIN) v = make_uint4(centre4(v.x), centre4(v.y), centre4(v.z), centre4(v.w));
      put(xl + min((tid + NT * i) / (2 * CK), P::TOKENS - 1) * PITCH, gx, half, v);
    }
#pragma unroll
    for (int i = 0; i < P::NWS; ++i) wsl[gs * P::WSP + min((tid + NT * i) / CK, P::ROWS - 1)] = f.ws[i];
#pragma unroll
    for (int i = 0; i < P::NXS; ++i) xsl[gs * P::XSP + min((tid + NT * i) / CK, P::TOKENS - 1)] = f.xs[i];
  };

  float acc[RT][TT][4], past[RT][TT][4];  // the chain's sums; the products of the group past the fours (bias 64)
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[r][t][v] = past[r][t][v] = 0.0f;
  const v4i start = {MAGIC, MAGIC, MAGIC, MAGIC};

  // a group of the stage: its products added to the chain (or, past the fours, kept)
  auto group = [&](const uint8_t *wl, const uint8_t *xl, const float *wsl, const float *xsl, int gi, auto take) {
    long A[RT], B[TT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      A[r] = *reinterpret_cast<const long *>(wl + ((sub * RT + r) * 16 + l16) * PITCH + gi * 32 + q * 8);
      if constexpr (PLAIN) A[r] = q == chain ? A[r] : 0;
    }
#pragma unroll
    for (int t = 0; t < TT; ++t) B[t] = *reinterpret_cast<const long *>(xl + (t * 16 + l16) * PITCH + gi * 32 + q * 8);
    float x[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) x[t] = xsl[gi * P::XSP + t * 16 + l16];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const float4 w4 = *reinterpret_cast<const float4 *>(wsl + gi * P::WSP + (sub * RT + r) * 16 + q * 4);
      const float w[4] = {w4.x, w4.y, w4.z, w4.w};
      v4i S[TT];
#pragma unroll
      for (int t = 0; t < TT; ++t) S[t] = __builtin_amdgcn_mfma_i32_16x16x32_i8(A[r], B[t], start, 0, 0, 0);
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) take(r, t, v, (__int_as_float(S[t][v]) - MAGIC_F) * (w[v] * x[t]));
    }
  };
  auto add = [&](int r, int t, int v, float p) { acc[r][t][v] = acc[r][t][v] + p; };
  // a whole stage: no branch, so that its groups' LDS reads, MFMAs and float32 work overlap
  auto compute = [&](int buf) {
    const uint8_t *const wl = lds + buf * P::STAGE, *const xl = wl + P::ROWS * PITCH;
    const float *const wsl = reinterpret_cast<const float *>(xl + P::TOKENS * PITCH), *const xsl = wsl + CK * P::WSP;
#pragma unroll
    for (int j = 0; j < (PLAIN ? CK : CK / 4); ++j) group(wl, xl, wsl, xsl, PLAIN ? j : 4 * j + chain, add);
  };
  // the last stage where its groups are fewer
  auto compute_part = [&](int buf, int n) {
    const uint8_t *const wl = lds + buf * P::STAGE, *const xl = wl + P::ROWS * PITCH;
    const float *const wsl = reinterpret_cast<const float *>(xl + P::TOKENS * PITCH), *const xsl = wsl + CK * P::WSP;
    if constexpr (PLAIN) {
      for (int g = 0; g < n; ++g) group(wl, xl, wsl, xsl, g, add);
    } else {
      for (int g0 = 0; g0 + 4 <= n; g0 += 4) group(wl, xl, wsl, xsl, g0 + chain, add);
      if ((n & ~3) + chain < n)
        group(wl, xl, wsl, xsl, (n & ~3) + chain, [&](int r, int t, int v, float p) { past[r][t][v] = p; });
    }
  };

  // stage s is computed from its LDS buffer while the next D stages lie in registers or fly. (Every thread loads and
  // stores each of its units, clamped to the block's last, which rewrites what is there: a load that a branch leaves
  // unused is waited for with everything after it.)
  const int full = G / CK;
  typename P::Fetch f[D];
#pragma unroll
  for (int d = 0; d < D; ++d) fetch(f[d], d);
  store(f[0], 0);
  lds_barrier();
  int s = 0;
  for (; s + D <= full; s += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      fetch(f[d], s + d + D);
      __builtin_amdgcn_sched_barrier(0);
      compute((s + d) & 1);
      // (the stores' waits and the arithmetic on what was loaded stay below the stage's work)
      __builtin_amdgcn_sched_barrier(0);
      store(f[(d + 1) % D], (s + d + 1) & 1);  // (that buffer's last readers passed the previous barrier)
      lds_barrier();
    }
  }
#pragma unroll
  for (int d = 0; d < D - 1; ++d) {  // the whole stages past the last D: their loads are on their way
    if (s + d < full) {  // uniform
      compute((s + d) & 1);
      store(f[d + 1], (s + d + 1) & 1);
      lds_barrier();
    }
  }
  if (G % CK) {  // uniform
    compute_part(full & 1, G % CK);
    lds_barrier();
  }

  // the chains meet: ((l0 + l1) + l2) + l3 by the thread that stores the four rows, then the groups past the fours
  // (chain c's wave holds group G4 + c's products)
  const int tail = PLAIN ? 0 : G & 3;
  float4 *const xch = lds4;  // [chain][sub][r][t][lane]
  constexpr int TILES = RB * RT * TT, PER = TILES * 64;
  float4 sum[(PER + NT - 1) / NT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int t = 0; t < TT; ++t)
      xch[chain * PER + ((sub * RT + r) * TT + t) * 64 + lane] =
          make_float4(acc[r][t][0], acc[r][t][1], acc[r][t][2], acc[r][t][3]);
  lds_barrier();
  // thread's output i: four consecutive rows (units) of one token, eight (RB * RT * 4) such pieces side by side a token
  constexpr int QUADS = RB * RT * 4;
  auto piece = [&](int i, int *quad, int *token) {
    const int o = tid + NT * i;
    *quad = o % QUADS;
    *token = o / QUADS;
    return ((*quad >> 2) * TT + (*token >> 4)) * 64 + (*quad & 3) * 16 + (*token & 15);
  };
#pragma unroll
  for (int i = 0; i < (PER + NT - 1) / NT; ++i) {
    int quad, token;
    const int at = piece(i, &quad, &token);
    if (PER % NT == 0 || tid + NT * i < PER) {
      const float4 c0 = xch[at], c1 = xch[PER + at], c2 = xch[2 * PER + at], c3 = xch[3 * PER + at];
      sum[i] = make_float4(((c0.x + c1.x) + c2.x) + c3.x, ((c0.y + c1.y) + c2.y) + c3.y, ((c0.z + c1.z) + c2.z) + c3.z,
                           ((c0.w + c1.w) + c2.w) + c3.w);
    }
  }
  if (tail) {  // uniform
    lds_barrier();
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int t = 0; t < TT; ++t)
        xch[chain * PER + ((sub * RT + r) * TT + t) * 64 + lane] =
            make_float4(past[r][t][0], past[r][t][1], past[r][t][2], past[r][t][3]);
    lds_barrier();
#pragma unroll
    for (int i = 0; i < (PER + NT - 1) / NT; ++i) {
      int quad, token;
      const int at = piece(i, &quad, &token);
      if (PER % NT == 0 || tid + NT * i < PER) {
        for (int c = 0; c < tail; ++c) {
          const float4 p = xch[c * PER + at];
          sum[i] = make_float4(sum[i].x + p.x, sum[i].y + p.y, sum[i].z + p.z, sum[i].w + p.w);
        }
      }
    }
  }
  if constexpr (GLU) {
    // h1 and h3 of 32 units lie in the quads of row tiles 0 (w1) and 1 (w3) of each part: through LDS once more, so that
    // a token's 8 quads of units are 8 lanes; then the SwiGLU and quantize_x of the token's group
    lds_barrier();
#pragma unroll
    for (int i = 0; i < (PER + NT - 1) / NT; ++i) {
      int quad, token;
      piece(i, &quad, &token);
      if (PER % NT == 0 || tid + NT * i < PER) xch[quad * P::TOKENS + token] = sum[i];
    }
    lds_barrier();
    for (int o = tid; o < P::TOKENS * 8; o += NT) {
      const int token = o >> 3, unit4 = o & 7, t = t0 + token;  // units 4 * unit4 ..: part unit4 / 4, quad unit4 % 4
      if (t >= a.m) break;  // (a token's 8 lanes leave together)
      const float4 h1 = xch[((unit4 >> 2) * 8 + (unit4 & 3)) * P::TOKENS + token];
      const float4 h3 = xch[((unit4 >> 2) * 8 + 4 + (unit4 & 3)) * P::TOKENS + token];
      const float4 o4 = make_float4(h1.x / (1.0f + vexp(-h1.x)) * h3.x, h1.y / (1.0f + vexp(-h1.y)) * h3.y,
                                    h1.z / (1.0f + vexp(-h1.z)) * h3.z, h1.w / (1.0f + vexp(-h1.w)) * h3.w);
      quantize_group4(o4, a.glu.q + (int64_t)t * a.glu.q_stride, a.glu.s + (int64_t)t * a.glu.s_stride, r0 + 4 * unit4,
                      r0 / 32, a.glu.bias);
    }
    return;
  }
  if constexpr (EPI == EPI_GELU) {
    // a token's 8 quads of the block's 32 units are 8 lanes already: gelu(h + b) as gelu_quant_kernel computes it, then
    // quantize_x of the token's group
#pragma unroll
    for (int i = 0; i < (PER + NT - 1) / NT; ++i) {
      int quad, token;
      piece(i, &quad, &token);
      const int t = t0 + token;
      if ((PER % NT != 0 && tid + NT * i >= PER) || t >= a.m) continue;  // (a token's 8 lanes leave together)
      const float *b = a.seg[0].bias + r0 + 4 * quad;
      const float h[4] = {sum[i].x + b[0], sum[i].y + b[1], sum[i].z + b[2], sum[i].w + b[3]};
      float o[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float inner = 0.7978845608028654f * (h[j] + ((0.044715f * h[j]) * h[j]) * h[j]);
        o[j] = h[j] / (1.0f + vexp(-2.0f * inner));
      }
      quantize_group4(make_float4(o[0], o[1], o[2], o[3]), a.glu.q + (int64_t)t * a.glu.q_stride,
                      a.glu.s + (int64_t)t * a.glu.s_stride, r0 + 4 * quad, r0 / 32, a.glu.bias);
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < (PER + NT - 1) / NT; ++i) {
    int quad, token;
    piece(i, &quad, &token);
    const int t = t0 + token, row = r0 + 4 * quad;
    if ((PER % NT != 0 && tid + NT * i >= PER) || t >= a.m) continue;
    const float v[4] = {sum[i].x, sum[i].y, sum[i].z, sum[i].w};
    if (a.qkv.on) {  // uniform
      finish_qkv(a, row, t, v);
      continue;
    }
    auto place = [&](int r, int *accumulate, const float **bias) {
      const bool third = a.nseg > 2 && r >= n0 + n1, second = a.nseg > 1 && r >= n0;
      const float *b = third ? a.seg[2].bias : (second ? a.seg[1].bias : a.seg[0].bias);
      *bias = b ? b + (r - (third ? n0 + n1 : (second ? n0 : 0))) : nullptr;
      float *y = third ? a.seg[2].y : (second ? a.seg[1].y : a.seg[0].y);
      const int stride = third ? a.seg[2].y_stride : (second ? a.seg[1].y_stride : a.seg[0].y_stride);
      *accumulate = third ? a.seg[2].accumulate : (second ? a.seg[1].accumulate : a.seg[0].accumulate);
      return y + (int64_t)t * stride + (r - (third ? n0 + n1 : (second ? n0 : 0)));
    };
    int accumulate;
    const float *bias;
    float *const dst = place(min(row, a.total_rows - 1), &accumulate, &bias);
    if (row + 3 < a.total_rows && ((n0 | n1) & 3) == 0 && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
      // the four rows lie in one segment, side by side on 16 bytes
      float4 o = make_float4(v[0], v[1], v[2], v[3]);
      if (accumulate) {
        const float4 y4 = *reinterpret_cast<const float4 *>(dst);
        o = make_float4(y4.x + v[0], y4.y + v[1], y4.z + v[2], y4.w + v[3]);
      }
      if (bias) o = make_float4(o.x + bias[0], o.y + bias[1], o.z + bias[2], o.w + bias[3]);
      *reinterpret_cast<float4 *>(dst) = o;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (row + j >= a.total_rows) break;
        float *const d = place(row + j, &accumulate, &bias);
        const float o = accumulate ? *d + v[j] : v[j];
        *d = bias ? o + *bias : o;
      }
    }
  }
}

int64_t tiles(int64_t n, int64_t size) { return (n + size - 1) / size; }

template <bool SIX, bool PLAIN, int RT, int TT, int RB, int CK, int D, int EPI>
hipError_t launch_one(const MatArgs &a, hipStream_t s) {
  using P = Chains<SIX, PLAIN, RT, TT, RB, CK, D, EPI>;
  const int64_t row_blocks = tiles(a.total_rows, P::ROWS), token_blocks = tiles(a.m, P::TOKENS), blocks = row_blocks * token_blocks;
  // a launch has fewer than 2^32 threads (more are dropped without an error): the tokens in pieces
  const int64_t most = (int64_t)(UINT32_MAX / P::NT) / row_blocks;
  if (token_blocks > most) {
    if (most < 1 || EPI != EPI_STORE || a.qkv.on) return hipErrorInvalidValue;
    for (int64_t t0 = 0; t0 < a.m; t0 += most * P::TOKENS) {
      MatArgs p = a;
      p.m = (int32_t)std::min<int64_t>(most * P::TOKENS, a.m - t0);
      p.xq = a.xq + t0 * a.xq_stride;
      p.xs = a.xs + t0 * a.xs_stride;
      for (int i = 0; i < a.nseg; ++i) p.seg[i].y = a.seg[i].y + t0 * a.seg[i].y_stride;
      const hipError_t e = launch_one<SIX, PLAIN, RT, TT, RB, CK, D, EPI>(p, s);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  if (P::LDS > 64 * 1024) {
    static bool sized = false;  // once a process: let the kernel take LDS past 64 KiB
    if (!sized) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_chains_kernel<SIX, PLAIN, RT, TT, RB, CK, D, EPI>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, P::LDS);
      if (e != hipSuccess) return e;
      sized = true;
    }
  }
  hipLaunchKernelGGL((gemm_chains_kernel<SIX, PLAIN, RT, TT, RB, CK, D, EPI>), dim3((unsigned)blocks), dim3(P::NT), P::LDS, s, a);
  return hipGetLastError();
}

// The tile of a launch (cold copies, one launch after another, us; 8 waves or fewer a CU hide a stage's latency worst):
//   16 x 16, 4 waves, 16-group stages: up to 16 tokens (any more rows or tokens would be padding: 4096 x 4096, 16
//     tokens 8.0 against 11.3 for 32 x 32), and grids of at most two such blocks a CU (4096 x 4096, 24 tokens: 10.3
//     against 11.9; 48 tokens, three a CU: 13.1 against 12.1);
//   32 x 32, 8 waves, 16-group stages: grids of at most one such block a CU (4096 x 14336, 64 tokens: 32.9 against 44
//     for 64 x 32; two a CU, 4096 x 4096, 100 tokens: 19.1 against 16.3);
//   64 x 32, 8 waves: the rest (a token's operand read once for four row tiles of the block).
constexpr int CUS = 256;

template <bool SIX, bool PLAIN>
hipError_t launch_tile(const MatArgs &a, hipStream_t s) {
  const int64_t rows = a.total_rows, m = a.m;
  if (m <= 16 || tiles(rows, 16) * tiles(m, 16) <= 2 * CUS) return launch_one<SIX, PLAIN, 1, 1, 1, 16, 2, EPI_STORE>(a, s);
  if (tiles(rows, 32) * tiles(m, 32) <= CUS) return launch_one<SIX, PLAIN, 1, 2, 2, 16, 2, EPI_STORE>(a, s);
  return launch_one<SIX, PLAIN, 2, 2, 2, 8, 2, EPI_STORE>(a, s);
}

// the SwiGLU's blocks (32 units of w1 and of w3): 16 tokens while that is at most one block a CU (4096 rows of K 512, 64
// tokens: 5.3 against 5.9 us; 128 tokens: 7.1 against 6.1); 48 for three tiles of tokens where the fullest CU would take
// twice as many blocks of 32, two of which cost more than one of 48 and less than that where it would not (40 tokens, us 48 /
// 32: 11,264 rows of K 2048, 1 or 2 a CU, 13.9 / 15.8; 16,384 of 3072, 1 or 2, 20.4 / 23.7; 28,672 of 4096, 2 or 4, 45.0 /
// 49.8; but 22,016 of 4096, 2 or 3, 44.4 / 40.1; 37,888 of 3584, 3 or 5, 60.3 / 55.6; 57,344 of 8192, 4 or 7, 171 / 165;
// int6 within 3% of these); else 32
template <bool SIX, bool PLAIN>
hipError_t launch_glu_tile(const MatArgs &a, hipStream_t s) {
  const int64_t units = tiles(a.seg[0].rows, 32), m = a.m;
  if (m <= 16 || units * tiles(m, 16) <= CUS) return launch_one<SIX, PLAIN, 2, 1, 2, 8, 2, EPI_GLU>(a, s);
  if (tiles(m, 16) == 3 && tiles(2 * units, CUS) == 2 * tiles(units, CUS))
    return launch_one<SIX, PLAIN, 2, 3, 2, 8, 2, EPI_GLU>(a, s);
  return launch_one<SIX, PLAIN, 2, 2, 2, 8, 2, EPI_GLU>(a, s);
}

// the GELU's blocks (32 units): the tiles of launch_tile that hold a whole group
template <bool SIX, bool PLAIN>
hipError_t launch_gelu_tile(const MatArgs &a, hipStream_t s) {
  const int64_t units = tiles(a.total_rows, 32), m = a.m;
  if (m <= 16) return launch_one<SIX, PLAIN, 1, 1, 2, 16, 2, EPI_GELU>(a, s);
  if (units * tiles(m, 32) <= CUS) return launch_one<SIX, PLAIN, 1, 2, 2, 16, 2, EPI_GELU>(a, s);
  return launch_one<SIX, PLAIN, 1, 2, 2, 8, 2, EPI_GELU>(a, s);
}

// gemm.hip's blocks (64 rows x 128 tokens, two a CU) take a K step of 128 in about 1.85 us while at most one lies on a
// CU, 2.3 us with two, and 2.2 us a round of 512 after that; here the time goes with the blocks of 64 x 32, 1.48 ns a
// block and K step (the SwiGLU's: 2.2). Measured on both sides of the line (us here / there): 4096 x 4096, 512 tokens
// 46.9 / 60.4, 1024 tokens 92.4 / 76.0; 6144 x 4096, 384 tokens 57.0 / 66.5, 512 tokens 69.4 / 67.4; 14336 x 4096, 100
// tokens 48.5 / 59.9, 200 tokens 78.7 / 72.7, 300 tokens (a second round there) 101.9 / 124.2; the SwiGLU at 28672 x
// 4096, 64 tokens 57.0 / 65.6, 96 tokens 73.6 / 66.9, at 4096 x 512, 300 tokens 11.3 / 12.1, 511 tokens 14.1 / 12.3.
// So a round of theirs is worth 1420 of these (int8 up to 1500, int6 from 1340), and fewer with groups past the fours, whose
// products meet in a hand-over of their own, and for short rows, where the hand-over and the stores weigh more on blocks of
// 64 x 32 (us there / here, [blocks there, here]): 18,944 x 14336, int6, 455 tokens [1184, 4440] 617 / 665; 28,460 x 3104 (97 groups), 83
// tokens [445, 1335] 57.1 / 64.0; 11,344 x 1056 (33), 505 tokens [712, 2848] 47.2 / 54.2; K of 384, 13,420 rows, 607 tokens [1050,
// 3990] 46.3 / 35.7; K of 192, 14336 rows, 100 tokens [224, 896] 11.5 / 12.0, 5105 rows, 524 tokens [400, 1360] 16.1 / 18.9,
// 6144 rows, 400 tokens [384, 1248] 16.2 / 14.0; K of 128, 12,084 rows, 175 tokens [378, 1134] 14.1 / 11.7; K of 96, 4096 rows, 256
// tokens [128, 512: two a CU] 8.8 / 7.3, 4621 rows, 242 tokens [146, 584] 8.3 / 11.1, 22,042 rows, 65 tokens [345, 1035] 10.0 / 14.5.
// Over 3200 shapes of up to 32,768 rows, K of 96-17,000 and 1024 tokens the choice costs 0.13% of the faster one's time in the mean,
// and is the 64 x 128 blocks' by more than 4% of their time for 11.
// (Past 2^27 rows the tile of 16 x 16 would have more threads than a launch takes: theirs.)
struct Grids {
  int64_t theirs, ours, rounds;
};
Grids grids(int32_t rows, int32_t m) {
  const int64_t theirs = tiles(rows, 64) * tiles(m, 128);
  return {theirs, tiles(rows, 64) * tiles(m, 32), tiles(theirs, 2 * CUS)};
}
}  // namespace

bool gemm_chains_faster(int32_t rows, int32_t m, int32_t k, bool glu) {
  if (rows > 1 << 27) return false;
  const Grids g = grids(rows, m);
  if (glu) return g.ours <= (g.theirs <= CUS ? 720 : 1000 * g.rounds);
  const bool past = k % 128 != 0;  // groups past the fours
  if (g.theirs <= CUS) {
    if (k < 128) return g.ours <= 512;
    return g.ours <= (past ? (k < 256 ? 520 : (k < 1024 ? 760 : 1250)) : (k < 256 ? 700 : (k < 384 ? 820 : 1250)));
  }
  if (k < 128) return g.ours <= 440 * g.rounds;
  return g.ours <= (past ? (k < 1024 ? 1080 : 1270) : (k <= 512 ? 1340 : 1420)) * g.rounds;
}

// (an epilogue saves a launch: 1480 a round for every K)
bool gemm_finishes(int32_t rows, int32_t m, bool relaxed) {
  if (!relaxed) return true;
  if (rows > 1 << 27) return false;
  const Grids g = grids(rows, m);
  return g.ours <= (g.theirs <= CUS ? 1250 : 1480 * g.rounds);
}

hipError_t launch_gemm_chains(const MatArgs &a, bool six, bool relaxed, hipStream_t s) {
  if (six) return relaxed ? launch_tile<true, false>(a, s) : launch_tile<true, true>(a, s);
  return relaxed ? launch_tile<false, false>(a, s) : launch_tile<false, true>(a, s);
}

hipError_t launch_gemm_chains_glu(const MatArgs &a, bool six, bool relaxed, hipStream_t s) {
  if (six) return relaxed ? launch_glu_tile<true, false>(a, s) : launch_glu_tile<true, true>(a, s);
  return relaxed ? launch_glu_tile<false, false>(a, s) : launch_glu_tile<false, true>(a, s);
}

hipError_t launch_gemm_chains_gelu(const MatArgs &a, bool six, bool relaxed, hipStream_t s) {
  if (six) return relaxed ? launch_gelu_tile<true, false>(a, s) : launch_gelu_tile<true, true>(a, s);
  return relaxed ? launch_gelu_tile<false, false>(a, s) : launch_gelu_tile<false, true>(a, s);
}

}  // namespace ple
