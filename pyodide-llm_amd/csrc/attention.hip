// attention.hip — causal grouped-query attention of m tokens (token t at position pos0 + t over the cache rows
// 0..pos0+t), to the bit of kernels/kernel.ts:448-566 attentionOf:
//   score = (l0 + l2) + (l1 + l3) of four lanes over j (q_j * k_j rounded, added in order), the tail added, times
//           isq = f32(1 / f32(sqrt(hs)));
//   softmax: the largest (order-free); e = vexp(s - max) for the positions below count & ~3, fexp past them; the sum
//           in four lanes (t % 4) in order, hsum ((l0 + l1) + l2) + l3, the tail added in order; p = e * f32(1 / sum);
//   out_j: blocks of four positions in order, out = out + ((p0 v0 + p1 v1) + (p2 v2 + p3 v3)), then the positions past
//           the fours one at a time, out = out + p v.
// The keys lie as the positions' rows ([seq_len][kv_dim]), the values as the columns' runs of positions
// ([kv_dim][vstride]). Launches: (A) the scores of 64-position tiles, every CU streaming keys once for the nh / nkv
// query heads that share them, with each tile's maxima; then for a few tokens (decode) one launch (B + C) a
// (token, head, 16 or 32 columns): the exponentials, their ordered sum, and the weighted values (short contexts: the
// scores too, attend1_kernel). A prompt block's scores, and the separate softmax and weighted values of prompt blocks
// and of contexts past these kernels' LDS, are attention_tokens.hip's.
#pragma clang fp contract(off)

#include <algorithm>

#include "attention.hpp"

namespace ple {

namespace {

// (A) grid (tiles, nkv, m)
template <int HS, bool HALF>
__global__ __launch_bounds__(256) void scores_kernel(const AttnArgs a) {
  constexpr int LD = HS + 4, C4 = HS / 4;
  __shared__ float ks[TILE * LD];
  __shared__ float qs[MAXMUL * HS];
  const int tile = blockIdx.x, kh = blockIdx.y, t = blockIdx.z;
  const int count = first_position(a) + t + 1;
  const int p0 = tile * TILE;
  if (p0 >= count) return;
  const int kvdim = a.nkv * HS, mul = a.nh / a.nkv;
  const int np = min(TILE, count - p0);
  constexpr int NL = (TILE * C4 + 255) / 256;  // float4 of keys a thread, requested together
  constexpr int NQ = (MAXMUL * C4 + 255) / 256;  // float4 of the queries a thread, requested with them
  const float *q = a.q + (int64_t)t * a.q_stride + (int64_t)kh * mul * HS;
  float4 qr[NQ];
#pragma unroll
  for (int u = 0; u < NQ; ++u) qr[u] = *reinterpret_cast<const float4 *>(q + 4 * min((int)threadIdx.x + u * 256, mul * C4 - 1));
  float4 kr4[NL];
#pragma unroll
  for (int u = 0; u < NL; ++u) {
    const int i = threadIdx.x + u * 256, p = min(i / C4, np - 1), c = i % C4;  // clamped, unconditional
    kr4[u] = cache4<HALF>(a.kcache, (int64_t)(p0 + p) * kvdim + kh * HS + 4 * c);
  }
#pragma unroll
  for (int u = 0; u < NQ; ++u) {
    const int i = threadIdx.x + u * 256;
    if (i < mul * C4) *reinterpret_cast<float4 *>(qs + 4 * i) = qr[u];
  }
#pragma unroll
  for (int u = 0; u < NL; ++u) {
    const int i = threadIdx.x + u * 256, p = i / C4, c = i % C4;
    if (p < np) *reinterpret_cast<float4 *>(ks + p * LD + 4 * c) = kr4[u];
  }
  __syncthreads();
  const float isq = 1.0f / __builtin_sqrtf((float)HS);
  float *scores = a.scores + (int64_t)t * a.nh * a.seq_len;
  for (int idx = threadIdx.x; idx < mul * TILE; idx += 256) {
    const int hl = idx / TILE, p = idx % TILE;
    float sc = -__builtin_inff();
    if (p < np) {
      const float *kr = ks + p * LD, *qr = qs + hl * HS;
      float l0 = 0.0f, l1 = 0.0f, l2 = 0.0f, l3 = 0.0f;
#pragma unroll 8
      for (int j = 0; j < HS; j += 4) {
        const float4 kv = *reinterpret_cast<const float4 *>(kr + j);
        const float4 qv = *reinterpret_cast<const float4 *>(qr + j);
        l0 = l0 + qv.x * kv.x;
        l1 = l1 + qv.y * kv.y;
        l2 = l2 + qv.z * kv.z;
        l3 = l3 + qv.w * kv.w;
      }
      sc = ((l0 + l2) + (l1 + l3)) * isq;
      scores[(int64_t)(kh * mul + hl) * a.seq_len + p0 + p] = sc;
    }
    float mx = sc;  // the tile's largest of this head (a wave is one head's 64 positions)
    for (int o = 32; o >= 1; o >>= 1) mx = wmax(mx, __shfl_xor(mx, o, 64));
    if (p == 0) a.tilemax[((int64_t)t * a.nh + kh * mul + hl) * (a.seq_len / TILE + 1) + tile] = mx;
  }
}

// (B + C) for a few tokens (decode), in one launch: one block a (token, query head, 32 of the head's columns: one
// quantization group, 16 where the head size is not a multiple of 32). The block requests everything it reads at
// once: the head's tile maxima (wave 0), its scores (every thread), the producer waves' first value chunks and the
// tail values (wave 0). Then the exponentials go into LDS (lane k's positions t % 4 == k side by side), four lanes of
// wave 0 run the ordered sums and the block has f32(1 / sum); then the producer waves each turn every NP-th item (a
// chunk of 256 positions and 16 columns, the next two requested ahead) into the four-position products ((p0 v0 + p1 v1) + (p2 v2 + p3 v3)),
// p = e * f32(1 / sum), in a ring of LDS slots, and wave 0's first lanes add them in order, a lane a column. An LDS flag
// a (slot, half) says it is filled and a counter says how many chunks wave 0 has added; every wait is on another wave
// of the block for a chunk of a lower index, so every wait ends. With a whole group, wave 0 also runs quantize_x on
// its 32 sums (the output projection's activations, no launch of their own).
// The blocks of the nh / nkv heads that share a kv head's columns are dealt to one XCD (the hardware deals blocks to
// the 8 XCDs in turn), so that the values they all read come from that XCD's L2 after the first.
constexpr int RP = 256, RB = RP / 4, RR = RB + 4;  // positions, four-position blocks, LDS row (floats) of a chunk
constexpr int ASLOTS = 8;                   // ring slots at most

template <int HS> struct Attend {
  static constexpr int AC = HS % 32 == 0 ? 32 : 16;  // columns a block
  static constexpr int H = AC / 16;                   // 16-column items a chunk
  static constexpr int NT = 512;                      // threads a block
  static constexpr int NP = NT / 64 - 1;              // producer waves
  static constexpr int SV = 16;                       // scores a thread a pass (8192 positions)
};

__device__ __forceinline__ int lds_load(const int *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
__device__ __forceinline__ void lds_store(int *p, int v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
__device__ __forceinline__ void wait_at_least(const int *p, int v) {
  while (lds_load(p) < v) __builtin_amdgcn_s_sleep(1);
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// +0.0 from the end of `rows` sums' rows of q4 values to the end of their last segment (chain16_registers), by the block's
// first 32 * rows threads
__device__ __forceinline__ void pad_rows(float *c, int rows, int rs, int q4, int tid) {
  const int row = tid >> 5, i = (q4 & ~31) + (tid & 31);
  if (row < rows && i >= q4 && (q4 & 31)) c[row * rs + chain16_at(i)] = 0.0f;
}

// 1 / the exponentials' sum: the four lanes' sums, ((l0 + l1) + l2) + l3, the tail in order; one wave, the same in each lane
__device__ __forceinline__ float inverse_sum(const float *e4, int rs, int q4, const float *tail, int rest, int lane) {
  const float part = chain16_registers<false>(e4 + (lane >> 4) * rs, q4, lane & 15);
  float sum = ((chain16_result(part, q4, 0) + chain16_result(part, q4, 1)) + chain16_result(part, q4, 2)) +
              chain16_result(part, q4, 3);
  for (int r = 0; r < rest; ++r) sum = sum + tail[r];
  return 1.0f / sum;
}

// an item's values: lane = four-position block, one float4 of positions a column of the item's 16 (clamped: never
// added past count4)
#define ATT_FETCH(item, v)                                                                                    \
  {                                                                                                           \
    const int64_t at_ = vcol + (int64_t)((item) % H * 16) * a.vstride + min((item) / H * RP + 4 * lane, count4 - 4); \
    _Pragma("unroll") for (int j_ = 0; j_ < 16; ++j_) v[j_] = cache4<HALF>(a.vcache, at_ + (int64_t)j_ * a.vstride); \
  }

template <int HS, bool HALF>
__global__ __launch_bounds__(Attend<HS>::NT) void attend_kernel(const AttnArgs a, const int nslot) {
  using P = Attend<HS>;
  constexpr int AC = P::AC, H = P::H, NT = P::NT, NP = P::NP, ASV = P::SV;
  extern __shared__ float4 lds4[];
  float *const lds = reinterpret_cast<float *>(lds4);
  __shared__ float shared_mx, shared_inv;
  __shared__ int filled[ASLOTS][H], used;
  constexpr int S = HS / AC;  // column slices a kv head
  const int mul = a.nh / a.nkv, groups = a.nkv * S;
  const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3, hl = idx % mul, g = (idx / mul) * 8 + xcd;
  if (g >= groups) return;  // the grid's rounding up: whole blocks leave
  const int kh = g / S, j0 = (g % S) * AC, h = kh * mul + hl;
  const int t = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, pw = wave - 1;
  const int count = first_position(a) + t + 1, count4 = count & ~3, q4 = count4 >> 2, rs = chain_rowstride(q4);
  float *const e4 = lds;              // [4][rs]
  float *const tail = lds + 4 * rs;   // [4]
  float *const ring = tail + 4;       // [nslot][AC][RR]
  const float *sc = a.scores + ((int64_t)t * a.nh + h) * a.seq_len;
  const int64_t vcol = (int64_t)(kh * HS + j0) * a.vstride;  // the block's first value column
  const int chunks = (count4 + RP - 1) / RP, items = chunks * H;

  if (tid < ASLOTS * H) filled[tid / H][tid % H] = 0;
  if (tid == ASLOTS * H) used = 0;
  // every load of the block, requested before anything waits: tile maxima, scores, values
  const int tiles = (count + TILE - 1) / TILE;
  const float *tm = a.tilemax + ((int64_t)t * a.nh + h) * (a.seq_len / TILE + 1);
  float tmr[2];
  if (wave == 0) {
#pragma unroll
    for (int u = 0; u < 2; ++u) tmr[u] = tm[min(lane + 64 * u, tiles - 1)];  // clamped: a repeat changes no max
  }
  float sv[ASV];
#pragma unroll
  for (int u = 0; u < ASV; ++u) sv[u] = sc[min(tid + NT * u, count - 1)];
  float4 va[16], vn[16];  // a producer's next two items
  if (wave > 0 && pw < items) ATT_FETCH(pw, va);
  if (wave > 0 && pw + NP < items) ATT_FETCH(pw + NP, vn);
  float tv[3];  // wave 0, lane j < AC: column j's values past the fours (at most 3)
  if (wave == 0) {
#pragma unroll
    for (int r = 0; r < 3; ++r)
      tv[r] = cache1<HALF>(a.vcache, vcol + (int64_t)(lane % AC) * a.vstride + min(count4 + r, count - 1));
  }
  if (wave == 0) {
    float mx = wmax(tmr[0], tmr[1]);
    for (int i = lane + 128; i < tiles; i += 64) mx = wmax(mx, tm[i]);  // past 8192 positions
    for (int o = 32; o >= 1; o >>= 1) mx = wmax(mx, __shfl_xor(mx, o, 64));
    if (lane == 0) shared_mx = mx;
  }
  __syncthreads();
  const float mx = shared_mx;
  for (int base = 0; base < count; base += NT * ASV) {
    if (base > 0) {
#pragma unroll
      for (int u = 0; u < ASV; ++u) sv[u] = sc[min(base + tid + NT * u, count - 1)];
    }
#pragma unroll
    for (int u = 0; u < ASV; ++u) {
      // the block's test first (the same for every thread: a scalar branch), so that no wave runs the exponentials
      // of positions past the count with its lanes switched off
      if (base + NT * u < count) {
        const int i = base + tid + NT * u;
        if (i < count) {
          const float d = sv[u] - mx;
          if (i < count4) e4[(i & 3) * rs + chain16_at(i >> 2)] = vexp(d);
          else tail[i - count4] = fexp(d);
        }
      }
    }
  }
  pad_rows(e4, 4, rs, q4, tid);
  __syncthreads();
  if (wave == 0) {
    const float inv = inverse_sum(e4, rs, q4, tail, count - count4, lane);
    if (lane == 0) shared_inv = inv;
  }
  __syncthreads();
  const float inv = shared_inv;
  if (wave > 0) {
    for (int it = pw; it < items; it += NP) {
      const int c = it / H, half = it % H;
      wait_at_least(&used, c - nslot + 1);  // the slot's last chunk has been added
      float *slot = ring + (c % nslot) * (AC * RR) + half * 16 * RR + lane;
      // the lane's four-position block (clamped: never added past q4)
      const int b = chain16_at(min(c * RB + lane, q4 - 1));
      const float p0 = e4[b] * inv, p1 = e4[rs + b] * inv, p2 = e4[2 * rs + b] * inv, p3 = e4[3 * rs + b] * inv;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const float4 x = va[j];
        slot[j * RR] = (p0 * x.x + p1 * x.y) + (p2 * x.z + p3 * x.w);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      if (lane == 0) lds_store(&filled[c % nslot][half], c + 1);
#pragma unroll
      for (int j = 0; j < 16; ++j) va[j] = vn[j];
      if (it + 2 * NP < items) ATT_FETCH(it + 2 * NP, vn);  // in flight while the wave waits
    }
  } else {
    // lane j < AC: column j0 + j (lanes past AC repeat column AC - 1 and store nothing). Chunks in pairs, two
    // register sets: chunk c + 1 is requested (after its flags) before chunk c's adds, which hide its latency. The
    // slot of c + 1 is free once c - 1 is released, so waiting for c + 1 before releasing c needs nslot >= 2.
    float acc = 0.0f;
    const int lr = min(lane, AC - 1);
    float4 xa[RB / 4], xb[RB / 4];
    auto ready = [&](int c) {  // every half of chunk c filled: the flags requested together, then one wait
      const int *f = filled[c % nslot];
      for (;;) {
        int least = lds_load(f);
#pragma unroll
        for (int hh = 1; hh < H; ++hh) least = min(least, lds_load(f + hh));
        if (least >= c + 1) break;
        __builtin_amdgcn_s_sleep(1);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    };
    auto fetch = [&](int c, float4 (&x)[RB / 4]) {
      const float4 *row = reinterpret_cast<const float4 *>(ring + (c % nslot) * (AC * RR) + lr * RR);
#pragma unroll
      for (int u = 0; u < RB / 4; ++u) x[u] = row[u];
    };
    auto consume = [&](int c, const float4 (&x)[RB / 4]) {
      const int nb = min(RP, count4 - c * RP) >> 2;
      if (nb == RB) {
        acc = add32(acc, x);
        acc = add32(acc, x + 8);
      } else {  // the last chunk, part full: from LDS
        acc = lds_chain(ring + (c % nslot) * (AC * RR) + lr * RR, nb, acc);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      if (lane == 0) lds_store(&used, c + 1);
    };
    if (chunks > 0) {
      ready(0);
      fetch(0, xa);
    }
    for (int c = 0; c < chunks; c += 2) {
      if (c + 1 < chunks) {
        ready(c + 1);
        fetch(c + 1, xb);
      }
      consume(c, xa);
      if (c + 1 < chunks) {
        if (c + 2 < chunks) {
          ready(c + 2);
          fetch(c + 2, xa);
        }
        consume(c + 1, xb);
      }
    }
#pragma unroll
    for (int r = 0; r < 3; ++r)
      if (r < count - count4) acc = acc + (tail[r] * inv) * tv[r];
    const int col = h * HS + j0 + lane;
    if (lane < AC) a.out[(int64_t)t * a.out_stride + col] = acc;
    if (AC == 32 && a.xq) {
      // quantize_x of the group (lanes 0-31): the largest magnitude, scale = amax / qmax, the values
      const float amax = wave_max32(__builtin_fabsf(acc));
      const float scale = amax / (a.bias == 0 ? 127.0f : 63.0f);
      const float qinv = scale > 0 ? 1.0f / scale : 0.0f;
      if (lane < 32) a.xq[(int64_t)t * a.xq_stride + col] = quant_value(acc, qinv, a.bias);
      if (lane == 0) a.xs[(int64_t)t * a.xs_stride + col / GS] = scale;
    }
  }
}
#undef ATT_FETCH

// (B + C) for a few tokens (decode) whose output the caller quantizes itself: one block of 1024 threads a (token,
// query head, 16 columns), thread b owning the four-position block b (positions 4b .. 4b+3) of the weighted values.
// The head's tile maxima and scores are requested at once, the exponentials go into LDS by lane (four rows: positions
// t % 4 == k); then every thread requests its block's 16 columns x 4 values while wave 0 runs the ordered sums, turns
// them into the columns' four-position products ((p0 v0 + p1 v1) + (p2 v2 + p3 v3)), p = e * f32(1 / sum), into LDS
// rows (one a column), and waves 0-3 add the columns' products in order, a column a row of 16 lanes, then the tail.
// (The values are requested once the exponentials are in LDS: requested at the start, their arrival slowed the scores'
// loads and the exponentials.) The sums from registers (chain16_registers) instead of four and sixteen lanes' LDS reads:
// 2060 positions, 32 / 8 heads of 128, scores included, 13.7 -> 12.8 us; 7002 positions 28.3 -> 26.1. Blocks of the query
// heads that share a kv head's columns go to one XCD, as in attend_kernel.
constexpr int A2_NT = 1024;  // threads a block
constexpr int A2_AC = 16;    // columns a block
constexpr int A2_SV = 4;     // scores a thread a pass (4096 positions)
constexpr int A2_MOST = 2 * 4 * A2_NT;  // positions: two four-position blocks a thread at most

// LDS bytes of attend2_kernel for the largest count of a launch: the exponentials' four rows, the tail, the columns'
// rows of products
size_t attend2_lds(int count) {
  const int rs = chain_rowstride((count & ~3) >> 2);
  return sizeof(float) * (size_t)((4 + A2_AC) * rs + 4);
}

template <int HS, bool HALF>
__device__ __forceinline__ void attend2(const AttnArgs &a, float *const lds) {
  constexpr int NT = A2_NT, AC = A2_AC, S = HS / AC;
  __shared__ float shared_mx, shared_inv;
  const int mul = a.nh / a.nkv, groups = a.nkv * S;
  const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3, hl = idx % mul, g = (idx / mul) * 8 + xcd;
  if (g >= groups) return;  // the grid's rounding up: whole blocks leave
  const int kh = g / S, j0 = (g % S) * AC, h = kh * mul + hl;
  const int t = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int count = first_position(a) + t + 1, count4 = count & ~3, q4 = count4 >> 2, rs = chain_rowstride(q4);
  float *const e4 = lds;             // [4][rs]
  float *const tail = lds + 4 * rs;  // [4]
  float *const blk = tail + 4;       // [AC][rs] (16-byte aligned: rs is a multiple of 16)
  const float *sc = a.scores + ((int64_t)t * a.nh + h) * a.seq_len;
  const int64_t vcol = (int64_t)(kh * HS + j0) * a.vstride;  // the block's first value column
  const int tiles = (count + TILE - 1) / TILE;
  const float *tm = a.tilemax + ((int64_t)t * a.nh + h) * (a.seq_len / TILE + 1);
  float tmr[2];
  if (wave == 0) {
#pragma unroll
    for (int u = 0; u < 2; ++u) tmr[u] = tm[min(lane + 64 * u, tiles - 1)];  // clamped: a repeat changes no max
  }
  float sv[A2_SV];
#pragma unroll
  for (int u = 0; u < A2_SV; ++u) sv[u] = sc[min(tid + NT * u, count - 1)];  // clamped, unconditional
  // waves 0-3, the 16 lanes of a row: a column's sum, and its values past the fours (at most 3)
  const int col = (wave & 3) * 4 + (lane >> 4);
  float tv[3];
  if (wave < 4) {
#pragma unroll
    for (int r = 0; r < 3; ++r)
      tv[r] = cache1<HALF>(a.vcache, vcol + (int64_t)col * a.vstride + min(count4 + r, count - 1));
  }
  if (wave == 0) {
    float mx = wmax(tmr[0], tmr[1]);
    for (int i = lane + 128; i < tiles; i += 64) mx = wmax(mx, tm[i]);  // past 8192 positions
    for (int o = 32; o >= 1; o >>= 1) mx = wmax(mx, __shfl_xor(mx, o, 64));
    if (lane == 0) shared_mx = mx;
  }
  __syncthreads();
  const float mx = shared_mx;
  for (int base = 0; base < count; base += NT * A2_SV) {
    if (base > 0) {
#pragma unroll
      for (int u = 0; u < A2_SV; ++u) sv[u] = sc[min(base + tid + NT * u, count - 1)];
    }
#pragma unroll
    for (int u = 0; u < A2_SV; ++u) {
      if (base + NT * u < count) {  // the block's test first (a scalar branch): no exponentials past the count
        const int i = base + tid + NT * u;
        if (i < count) {
          const float d = sv[u] - mx;
          if (i < count4) e4[(i & 3) * rs + chain16_at(i >> 2)] = vexp(d);
          else tail[i - count4] = fexp(d);
        }
      }
    }
  }
  pad_rows(e4, 4, rs, q4, tid);
  __syncthreads();
  // the first pass's values requested now (clamped into the column: never used past q4): they fly while wave 0 runs
  // the exponentials' ordered sum (its reads 32 values at a time, so that both fit the registers)
  float4 v0[AC];
  {
    const int bc = max(min(tid, q4 - 1), 0);
#pragma unroll
    for (int j = 0; j < AC; ++j) v0[j] = cache4<HALF>(a.vcache, vcol + (int64_t)j * a.vstride + 4 * bc);
  }
  if (wave == 0) {
    const float inv = inverse_sum(e4, rs, q4, tail, count - count4, lane);
    if (lane == 0) shared_inv = inv;
  }
  __syncthreads();
  const float inv = shared_inv;
  // block b's products: (p0 v0 + p1 v1) + (p2 v2 + p3 v3) for the 16 columns, into the columns' rows
  auto products = [&](int b, const float4 (&v)[AC]) {
    if (b < q4) {
      const int bs = chain16_at(b);
      const float p0 = e4[bs] * inv, p1 = e4[rs + bs] * inv, p2 = e4[2 * rs + bs] * inv, p3 = e4[3 * rs + bs] * inv;
#pragma unroll
      for (int j = 0; j < AC; ++j) {
        const float4 x = v[j];
        blk[j * rs + bs] = (p0 * x.x + p1 * x.y) + (p2 * x.z + p3 * x.w);
      }
    }
  };
  products(tid, v0);
  for (int b0 = NT; b0 < q4; b0 += NT) {  // (a scalar loop: every thread takes the same passes)
    const int b = b0 + tid, bc = min(b, q4 - 1);  // clamped: never stored past q4
    float4 v[AC];
#pragma unroll
    for (int j = 0; j < AC; ++j) v[j] = cache4<HALF>(a.vcache, vcol + (int64_t)j * a.vstride + 4 * bc);
    products(b, v);
  }
  pad_rows(blk, AC, rs, q4, tid);
  __syncthreads();
  if (wave < 4) {
    float acc = chain16_registers<true>(blk + col * rs, q4, lane & 15);
#pragma unroll
    for (int r = 0; r < 3; ++r)
      if (r < count - count4) acc = acc + (tail[r] * inv) * tv[r];
    if ((lane & 15) == (((q4 + 31) >> 5) & 15)) a.out[(int64_t)t * a.out_stride + h * HS + j0 + col] = acc;
  }
}

template <int HS, bool HALF>
__global__ __launch_bounds__(A2_NT) void attend2_kernel(const AttnArgs a) {
  extern __shared__ float4 lds4[];
  attend2<HS, HALF>(a, reinterpret_cast<float *>(lds4));
}

// (B + C) for a few tokens (decode) of long contexts whose output the caller quantizes itself: one block of 16 waves a
// (token, query head, 16 columns), the exponentials in LDS as attend2_kernel, the weighted values in chunks of A3_BLOCKS
// four-position blocks through two LDS buffers. Waves 4-15 make a chunk's four-position products (64 blocks and 4 columns
// a wave, the values requested three chunks ahead) while waves 0-3 read the chunk before it into registers, a column a DPP
// row of 16 lanes, and add the one before that (chain16). Bound by the two ordered sums of count / 4 steps, about 5 cycles
// a step, and the values' way from the L2 (18 TB/s: every head of a kv head reads them). With the scores, from the caches:
// 20,010 positions, 28 / 4 heads of 128, 50.4 us against 63.9 for attend_kernel, whose one wave adds 32 columns from LDS;
// 8200 positions 26.9 against 33.9; 2060 positions, 32 / 8 heads, 12.8 against 15.6. A replayed decode step's launch is fixed by
// the model's longest context: a block whose count fits attend2's LDS (up to `most2` positions) takes its steps.
constexpr int A3_NT = 1024;      // threads a block
constexpr int A3_BLOCKS = 192;   // four-position blocks a chunk: 6 segments of 32 a column (32,768 positions fit the LDS)
constexpr int A3_SV = 16;        // scores a thread a pass
constexpr int A3_AHEAD = 3;      // chunks of values a producer holds

// LDS bytes of attend3_kernel for the largest count of a launch
size_t attend3_lds(int count) {
  return sizeof(float) * (size_t)(4 * chain_rowstride((count & ~3) >> 2) + 4 + 2 * A2_AC * A3_BLOCKS);
}

// four values of the cache as they lie there, and as float32
template <bool HALF> struct Raw4 { typedef float4 T; };
template <> struct Raw4<true> { typedef uint2 T; };
__device__ __forceinline__ float4 float4_of(float4 v) { return v; }
__device__ __forceinline__ float4 float4_of(uint2 h) {
  return make_float4(from_f16((uint16_t)(h.x & 0xffff)), from_f16((uint16_t)(h.x >> 16)),
                     from_f16((uint16_t)(h.y & 0xffff)), from_f16((uint16_t)(h.y >> 16)));
}

template <int HS, bool HALF>
__global__ __launch_bounds__(A3_NT) void attend3_kernel(const AttnArgs a, const int most2) {
  constexpr int NT = A3_NT, AC = A2_AC, S = HS / AC, CB = A3_BLOCKS, PC = 4;  // PC: columns a producer
  constexpr int SEGS = CB / 32, D = A3_AHEAD;
  static_assert((NT / 64 - 4) * 64 * PC == CB * AC, "the producers make a chunk");
  typedef typename Raw4<HALF>::T Raw;
  extern __shared__ float4 lds4[];
  float *const lds = reinterpret_cast<float *>(lds4);
  if (first_position(a) + (int)blockIdx.z + 1 <= most2) {  // uniform
    attend2<HS, HALF>(a, lds);
    return;
  }
  __shared__ float wave_mx[NT / 64], shared_inv;
  const int mul = a.nh / a.nkv, groups = a.nkv * S;
  const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3, hl = idx % mul, g = (idx / mul) * 8 + xcd;
  if (g >= groups) return;  // the grid's rounding up: whole blocks leave
  const int kh = g / S, j0 = (g % S) * AC, h = kh * mul + hl;
  const int t = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int count = first_position(a) + t + 1, count4 = count & ~3, q4 = count4 >> 2, rs = chain_rowstride(q4);
  float *const e4 = lds;             // [4][rs]
  float *const tail = lds + 4 * rs;  // [4]
  float *const buffers = tail + 4;   // [2][AC][CB]
  const float *sc = a.scores + ((int64_t)t * a.nh + h) * a.seq_len;
  const int64_t vcol = (int64_t)(kh * HS + j0) * a.vstride;  // the block's first value column
  const int tiles = (count + TILE - 1) / TILE;
  const float *tm = a.tilemax + ((int64_t)t * a.nh + h) * (a.seq_len / TILE + 1);
  float mx = tm[min(tid, tiles - 1)];  // clamped: a repeat changes no max
  float sv[A3_SV];
#pragma unroll
  for (int u = 0; u < A3_SV; ++u) sv[u] = sc[min(tid + NT * u, count - 1)];  // clamped, unconditional
  const int col = (wave & 3) * 4 + (lane >> 4), l16 = lane & 15;  // waves 0-3: a column a row of 16 lanes
  float tv[3];                                                    // and its values past the fours (at most 3)
  if (wave < 4) {
#pragma unroll
    for (int r = 0; r < 3; ++r)
      tv[r] = cache1<HALF>(a.vcache, vcol + (int64_t)col * a.vstride + min(count4 + r, count - 1));
  }
  for (int i = tid + NT; i < tiles; i += NT) mx = wmax(mx, tm[i]);
  for (int o = 32; o >= 1; o >>= 1) mx = wmax(mx, __shfl_xor(mx, o, 64));
  if (lane == 0) wave_mx[wave] = mx;
  lds_barrier();
  mx = wave_mx[0];
#pragma unroll
  for (int w = 1; w < NT / 64; ++w) mx = wmax(mx, wave_mx[w]);
  // position tid + NT u of a pass lies NT / 4 floats after position tid + NT (u - 1)'s place (chain16_at keeps whole 256s)
  static_assert(NT / 4 % 256 == 0, "chain16_at's turns repeat every 256 values");
  float *const to0 = e4 + (tid & 3) * rs + chain16_at(tid >> 2);
  for (int base = 0; base < count; base += NT * A3_SV) {
    if (base > 0) {
#pragma unroll
      for (int u = 0; u < A3_SV; ++u) sv[u] = sc[min(base + tid + NT * u, count - 1)];
    }
#pragma unroll
    for (int u = 0; u < A3_SV; ++u) {
      const int i = base + tid + NT * u;
      if (base + NT * (u + 1) <= count4) {  // (scalar branches: whole passes, then the one that the fours end in)
        to0[(base + NT * u) / 4] = vexp(sv[u] - mx);
      } else if (base + NT * u < count) {
        if (i < count4) to0[(base + NT * u) / 4] = vexp(sv[u] - mx);
        else if (i < count) tail[i - count4] = fexp(sv[u] - mx);
      }
    }
  }
  pad_rows(e4, 4, rs, q4, tid);
  lds_barrier();
  // a producer's four-position block of a chunk and its 4 columns (clamped into the columns: past q4 they become 0)
  const bool producer = wave >= 4;  // uniform
  const int pw = max(wave - 4, 0), pb = pw % (CB / 64) * 64 + lane, pj = pw / (CB / 64) * PC;
  const Raw *const values = reinterpret_cast<const Raw *>(a.vcache) + (vcol + (int64_t)pj * a.vstride) / 4;
  Raw held[D][PC];
  auto fetch = [&](int c, Raw (&v)[PC]) {
    const uint32_t at = max(min(c * CB + pb, q4 - 1), 0);  // (a scalar base a column, one offset a lane)
#pragma unroll
    for (int j = 0; j < PC; ++j) v[j] = (values + (int64_t)j * (a.vstride / 4))[at];
  };
  if (wave == 0) {
    const float inv = inverse_sum(e4, rs, q4, tail, count - count4, lane);
    if (lane == 0) shared_inv = inv;
  } else if (producer) {  // (in flight meanwhile)
#pragma unroll
    for (int k = 0; k < D; ++k) fetch(k, held[k]);
  }
  lds_barrier();
  const float inv = shared_inv;
  const int chunks = (q4 + CB - 1) / CB;
  // Step c of all waves, a barrier after each: chunk c's products into buffer c % 2 (its last readers passed the barrier
  // before), chunk c - 1 from its buffer into registers, and chunk c - 2's adds
  float *const to = buffers + pj * CB + chain16_at(pb);
  auto produce = [&](int c, Raw (&v)[PC]) {
    const int b = c * CB + pb, bs = chain16_at(min(b, q4 - 1));
    const float p0 = e4[bs] * inv, p1 = e4[rs + bs] * inv, p2 = e4[2 * rs + bs] * inv, p3 = e4[3 * rs + bs] * inv;
    float *const d = to + (c & 1) * (AC * CB);
#pragma unroll
    for (int j = 0; j < PC; ++j) {
      const float4 x = float4_of(v[j]);
      const float p = (p0 * x.x + p1 * x.y) + (p2 * x.z + p3 * x.w);
      d[j * CB] = b < q4 ? p : 0.0f;
    }
    __builtin_amdgcn_sched_barrier(0);
    fetch(c + D, v);
  };
  float acc = 0.0f;
  float4 ra[8], rb[8];
  // (a chunk is 6 segments: chunk c's first starts on lane 6 c % 16 of the row)
  auto take = [&](int c, float4 (&v)[8]) {
    chain16_read(buffers + (c & 1) * (AC * CB) + col * CB, 0, SEGS, (l16 - SEGS * c) & 15, v);
  };
  auto add = [&](int c, float4 (&v)[8]) { acc = chain16_rounds<SEGS>(acc, v, (min(CB, q4 - c * CB) + 31) >> 5); };
  // (a loop a role, the same barriers in each: the roles' registers are never live together)
  const int steps = chunks ? 2 + ((chunks + 1) & ~1) : 0;
  if (producer) {
    for (int c = 0; c < steps; c += D) {
#pragma unroll
      for (int k = 0; k < D; ++k) {
        if (c + k < chunks) produce(c + k, held[k]);
        if (c + k < steps) lds_barrier();
      }
    }
  } else {
    if (chunks) {
      lds_barrier();
      take(0, ra);
      lds_barrier();
    }
    for (int c = 1; c <= chunks; c += 2) {  // steps c + 1 and c + 2 (past the last chunk: the last read again, not added)
      take(min(c, chunks - 1), rb);
      add(c - 1, ra);
      lds_barrier();
      take(min(c + 1, chunks - 1), ra);
      if (c < chunks) add(c, rb);
      lds_barrier();
    }
  }
  if (wave < 4) {
#pragma unroll
    for (int r = 0; r < 3; ++r)
      if (r < count - count4) acc = acc + (tail[r] * inv) * tv[r];
    if (l16 == (((q4 + 31) >> 5) & 15)) a.out[(int64_t)t * a.out_stride + h * HS + j0 + col] = acc;
  }
}

// The whole of a decode attention in one launch, for contexts of up to A1_MOST positions: one block of 1024 threads a
// (token, query head, 16 columns), as attend2_kernel, that makes the head's scores itself, a thread a position. The head's
// other column blocks repeat them (a1_scores bounds the keys a block reads), which costs less than the scores' launch
// where everything fits the caches. Then the maximum over the block, and attend2_kernel's steps with a thread a
// (four-position block, 4 columns), its values requested with the keys. Bound by latency: the loads, two ordered sums of
// count / 4 steps, five barriers. (With the FFN's activation in w2's GEMV: two launches a layer fewer; a sampled step of
// the 15M shape 230 -> 203 us.)
constexpr int A1_MOST = 1024;  // positions: one a thread, four threads a four-position block
// Positions * head size at most: a replayed step's launch is fixed by the model's whole context, so the line lies where a
// step's mean over the positions of the context meets that of scores_kernel + attend2_kernel. A replayed layer of 512
// dims, us here / with the two launches, at 3%, 50% and 97% of the context, and the mean over it:
//   64 Ki: 8 heads of 64, 1024 positions, float16 23.4 / 27.3, 28.8 / 28.0, 32.1 / 30.1, mean 28.1 / 28.3; float32 22.2 / 26.1,
//     29.3 / 29.0, 33.3 / 29.9, mean 28.6 / 28.4; 12 heads 28.3 / 29.7 and 29.1 / 29.4; 32 / 8 heads of 128, 512 positions,
//     float32 30.9 / 32.2; 8 / 4 heads of 256, 256 positions 29.3 / 31.7; 32 heads of 96, 680 positions, float16 31.4 / 33.0,
//     float32 (two loads of 48 dims a position) 27.2 / 31.4, 32.2 / 32.2, 38.8 / 33.3, mean 32.6 / 32.3: there 48 Ki, 31.0 / 31.8;
//   48 Ki: 6 heads of 48, 1024 positions, float16 25.7 / 27.7, float32 26.8 / 27.4; 16 Ki: 8 heads of 16 23.1 / 25.9.
constexpr int a1_scores(int hs, bool half) { return (hs == 96 && !half ? 48 : 64) * 1024; }

template <int HS> constexpr int a1_chunk() { return HS <= 64 ? HS : (HS % 64 == 0 ? 64 : 48); }  // dims in registers

template <int HS, bool HALF>
__global__ __launch_bounds__(A2_NT) void attend1_kernel(const AttnArgs a) {
  constexpr int AC = A2_AC, S = HS / AC, DC = a1_chunk<HS>();
  extern __shared__ float4 lds4[];
  float *const lds = reinterpret_cast<float *>(lds4);
  __shared__ float4 qs[HS / 4];
  __shared__ float wave_mx[16], shared_inv;
  const int mul = a.nh / a.nkv, groups = a.nkv * S;
  const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3, hl = idx % mul, g = (idx / mul) * 8 + xcd;
  if (g >= groups) return;  // the grid's rounding up: whole blocks leave
  const int kh = g / S, j0 = (g % S) * AC, h = kh * mul + hl;
  const int t = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int count = first_position(a) + t + 1, count4 = count & ~3, q4 = count4 >> 2, rs = chain_rowstride(q4);
  float *const e4 = lds;             // [4][rs]
  float *const tail = lds + 4 * rs;  // [4]
  float *const blk = tail + 4;       // [AC][rs]
  const int64_t vcol = (int64_t)(kh * HS + j0) * a.vstride;  // the block's first value column
  const int kvdim = a.nkv * HS;
  if (tid < HS / 4) qs[tid] = reinterpret_cast<const float4 *>(a.q + (int64_t)t * a.q_stride + (int64_t)h * HS)[tid];
  // this thread's position's keys and its four-position block's values of 4 columns (clamped: never used past the count)
  const int64_t krow = (int64_t)min(tid, count - 1) * kvdim + kh * HS;
  const bool scoring = wave * 64 < count;  // uniform
  float4 kr[DC / 4], v[4];
  if (scoring) {
#pragma unroll
    for (int c = 0; c < DC / 4; ++c) kr[c] = cache4<HALF>(a.kcache, krow + 4 * c);
  }
  const int b = tid & 255, cg = tid >> 8, bc = max(min(b, q4 - 1), 0);
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = cache4<HALF>(a.vcache, vcol + (int64_t)(4 * cg + j) * a.vstride + 4 * bc);
  // waves 0-3, the 16 lanes of a row: a column's sum, and its values past the fours (at most 3)
  const int col = (wave & 3) * 4 + (lane >> 4);
  float tv[3];
  if (wave < 4) {
#pragma unroll
    for (int r = 0; r < 3; ++r)
      tv[r] = cache1<HALF>(a.vcache, vcol + (int64_t)col * a.vstride + min(count4 + r, count - 1));
  }
  lds_barrier();  // (the queries; the loads stay in flight)
  float sc = -__builtin_inff();
  if (scoring) {
    float l0 = 0.0f, l1 = 0.0f, l2 = 0.0f, l3 = 0.0f;
    for (int d = 0; d < HS; d += DC) {
      if (d > 0) {
#pragma unroll
        for (int c = 0; c < DC / 4; ++c) kr[c] = cache4<HALF>(a.kcache, krow + d + 4 * c);
      }
#pragma unroll
      for (int c = 0; c < DC / 4; ++c) {
        const float4 qv = qs[d / 4 + c];
        l0 = l0 + qv.x * kr[c].x;
        l1 = l1 + qv.y * kr[c].y;
        l2 = l2 + qv.z * kr[c].z;
        l3 = l3 + qv.w * kr[c].w;
      }
    }
    if (tid < count) sc = ((l0 + l2) + (l1 + l3)) * (1.0f / __builtin_sqrtf((float)HS));
  }
  float mx = sc;
  for (int o = 32; o >= 1; o >>= 1) mx = wmax(mx, __shfl_xor(mx, o, 64));
  if (lane == 0) wave_mx[wave] = mx;
  lds_barrier();
  mx = wave_mx[0];
#pragma unroll
  for (int w = 1; w < 16; ++w) mx = wmax(mx, wave_mx[w]);
  if (tid < count) {
    const float d = sc - mx;
    if (tid < count4) e4[(tid & 3) * rs + chain16_at(tid >> 2)] = vexp(d);
    else tail[tid - count4] = fexp(d);
  }
  pad_rows(e4, 4, rs, q4, tid);
  lds_barrier();
  if (wave == 0) {
    const float inv = inverse_sum(e4, rs, q4, tail, count - count4, lane);
    if (lane == 0) shared_inv = inv;
  }
  lds_barrier();
  const float inv = shared_inv;
  if (b < q4) {
    const int bs = chain16_at(b);
    const float p0 = e4[bs] * inv, p1 = e4[rs + bs] * inv, p2 = e4[2 * rs + bs] * inv, p3 = e4[3 * rs + bs] * inv;
#pragma unroll
    for (int j = 0; j < 4; ++j) blk[(4 * cg + j) * rs + bs] = (p0 * v[j].x + p1 * v[j].y) + (p2 * v[j].z + p3 * v[j].w);
  }
  pad_rows(blk, AC, rs, q4, tid);
  lds_barrier();
  if (wave < 4) {
    float acc = chain16_registers<false>(blk + col * rs, q4, lane & 15);
#pragma unroll
    for (int r = 0; r < 3; ++r)
      if (r < count - count4) acc = acc + (tail[r] * inv) * tv[r];
    if ((lane & 15) == (((q4 + 31) >> 5) & 15)) a.out[(int64_t)t * a.out_stride + h * HS + j0 + col] = acc;
  }
}

// whether attend1_kernel takes a decode launch
bool attend1_takes(const AttnArgs &a) {
  const int count = a.pos0 + a.m;
  return a.hs % A2_AC == 0 && count <= A1_MOST && count * a.hs <= a1_scores(a.hs, a.half);
}

// LDS bytes of attend_kernel for the largest count of a launch (ring slots into *nslot), 0 where it does not fit
template <int HS>
int attend_lds(const AttnArgs &a, int *nslot) {
  const int count = a.pos0 + a.m;
  const int head = (int)sizeof(float) * (4 * chain_rowstride((count & ~3) >> 2) + 4);
  const int slot = (int)sizeof(float) * Attend<HS>::AC * RR;
  const int n = std::min(ASLOTS, (ALDS - head) / slot);
  if (n < 2) return 0;
  *nslot = n;
  return head + n * slot;
}

// whether attend2_kernel takes a decode launch: head sizes of whole 16-column slices, a context that fits its LDS
// and its two four-position blocks a thread
bool attend2_takes(const AttnArgs &a) {
  const int count = a.pos0 + a.m;
  return a.hs % A2_AC == 0 && count <= A2_MOST && attend2_lds(count) <= (size_t)ALDS;
}

// the largest count that attend2 takes in attend3_kernel's LDS for a launch of at most `count` positions
int attend3_most2(int count) {
  const int rs = (int)(attend3_lds(count) / sizeof(float) - 4) / (4 + A2_AC);  // floats a row
  return std::min(A2_MOST, std::max(0, 4 * ((rs - 16) & ~63)));
}

// whether attend3_kernel takes a decode launch: head sizes of whole 16-column slices, a context that fits its LDS
bool attend3_takes(const AttnArgs &a) {
  return a.hs % A2_AC == 0 && attend3_lds(a.pos0 + a.m) <= (size_t)ALDS;
}

template <int HS, bool HALF>
hipError_t launch_hs(const AttnArgs &a, hipStream_t s) {
  const int tiles = (a.pos0 + a.m + TILE - 1) / TILE;
  if (a.m <= DECODE_TOKENS && !a.split && !a.xq && attend1_takes(a)) {
    const int groups = a.nkv * (HS / A2_AC), g8 = (groups + 7) & ~7;
    hipLaunchKernelGGL((attend1_kernel<HS, HALF>), dim3(g8 * (a.nh / a.nkv), 1, a.m), dim3(A2_NT),
                       attend2_lds(a.pos0 + a.m), s, a);
    return hipGetLastError();
  }
  if (a.m <= DECODE_TOKENS) {
    hipLaunchKernelGGL((scores_kernel<HS, HALF>), dim3(tiles, a.nkv, a.m), dim3(256), 0, s, a);
  } else {
    const hipError_t e = launch_scores_tokens(a, s);
    if (e != hipSuccess) return e;
  }
  if (a.m <= DECODE_TOKENS && !a.split && !a.xq && attend2_takes(a)) {
    // the caller quantizes the output itself: blocks of 16 columns
    const size_t lds = attend2_lds(a.pos0 + a.m);
    if (lds > 64 * 1024) {
      static bool sized = false;  // once a process: let the kernel take LDS past 64 KiB
      if (!sized) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&attend2_kernel<HS, HALF>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, ALDS);
        if (e != hipSuccess) return e;
        sized = true;
      }
    }
    const int groups = a.nkv * (HS / A2_AC), g8 = (groups + 7) & ~7;
    hipLaunchKernelGGL((attend2_kernel<HS, HALF>), dim3(g8 * (a.nh / a.nkv), 1, a.m), dim3(A2_NT), lds, s, a);
    return hipGetLastError();
  }
  if (a.m <= DECODE_TOKENS && !a.split && !a.xq && attend3_takes(a)) {
    static bool sized = false;  // once a process: let the kernel take LDS past 64 KiB
    if (!sized) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&attend3_kernel<HS, HALF>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, ALDS);
      if (e != hipSuccess) return e;
      sized = true;
    }
    const int groups = a.nkv * (HS / A2_AC), g8 = (groups + 7) & ~7;
    hipLaunchKernelGGL((attend3_kernel<HS, HALF>), dim3(g8 * (a.nh / a.nkv), 1, a.m), dim3(A3_NT),
                       attend3_lds(a.pos0 + a.m), s, a, attend3_most2(a.pos0 + a.m));
    return hipGetLastError();
  }
  int nslot = 0;
  const int fused = a.m <= DECODE_TOKENS && !a.split ? attend_lds<HS>(a, &nslot) : 0;
  if (fused) {
    static bool sized = false;  // once a process: let the kernel take LDS past 64 KiB
    if (!sized) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&attend_kernel<HS, HALF>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, ALDS);
      if (e != hipSuccess) return e;
      sized = true;
    }
    const int groups = a.nkv * (HS / Attend<HS>::AC), g8 = (groups + 7) & ~7;
    hipLaunchKernelGGL((attend_kernel<HS, HALF>), dim3(g8 * (a.nh / a.nkv), 1, a.m), dim3(Attend<HS>::NT), fused, s,
                       a, nslot);
    return hipGetLastError();
  }
  return launch_softmax_pv(a, s);
}

template <bool HALF>
hipError_t launch_half(const AttnArgs &a, hipStream_t s) {
  switch (a.hs) {
    case 16: return launch_hs<16, HALF>(a, s);
    case 32: return launch_hs<32, HALF>(a, s);
    case 48: return launch_hs<48, HALF>(a, s);
    case 64: return launch_hs<64, HALF>(a, s);
    case 96: return launch_hs<96, HALF>(a, s);
    case 128: return launch_hs<128, HALF>(a, s);
    case 256: return launch_hs<256, HALF>(a, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

bool attention_supported(int32_t hs, int32_t nh, int32_t nkv) {
  const bool sizes = hs == 16 || hs == 32 || hs == 48 || hs == 64 || hs == 96 || hs == 128 || hs == 256;
  return sizes && nkv > 0 && nh % nkv == 0 && nh / nkv <= MAXMUL;
}

int32_t attention_most_positions() {
  int32_t n = (ALDS / 4) & ~3;
  while (n > 0 && softmax_lds(n) > (size_t)ALDS) n -= 4;
  return n;
}

bool attention_quantizes(const AttnArgs &a) {
  return attention_supported(a.hs, a.nh, a.nkv) && a.hs % 32 == 0;
}

hipError_t launch_attention(const AttnArgs &a, hipStream_t s) {
  if (!attention_supported(a.hs, a.nh, a.nkv)) return hipErrorInvalidValue;
  // pieces of equal size (each past DECODE_TOKENS when m is past ATTN_ROWS), one after another on the stream
  const int pieces = a.dpos ? 1 : (a.m + ATTN_ROWS - 1) / ATTN_ROWS, size = (a.m + pieces - 1) / pieces;
  for (int at = 0; at < a.m; at += size) {
    AttnArgs p = a;
    p.q = a.q + (int64_t)at * a.q_stride;
    p.out = a.out + (int64_t)at * a.out_stride;
    p.pos0 = a.pos0 + at;
    p.m = std::min(size, a.m - at);
    if (p.xq) {
      p.xq = a.xq + (int64_t)at * a.xq_stride;
      p.xs = a.xs + (int64_t)at * a.xs_stride;
    }
    const hipError_t e = a.half ? launch_half<true>(p, s) : launch_half<false>(p, s);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace ple
