// cis2_rows.hip — gfx950 kernels of the row-batched forward pass (several
// sequences per step, or every position of one sequence).  Each output is
// computed by one lane in the order the single-row kernels use
// (code/cis2-fp/src/main.rs:355-529), so a row's results do not depend on
// which other rows share the launch (batch invariance).
#include "cis2_chain.hpp"
#include "cis2_device_math.hpp"
#include "cis2_rows.hpp"
#include "cis2_kernels.hpp"

#include <algorithm>
#include <type_traits>
#include <cstdlib>

namespace cis2 {
namespace {

// 16-byte vector as a native vector type: local arrays of it stay in
// registers (the struct-based float4 keeps them in scratch memory).
typedef float v4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kT = 256;
// Query heads per attention workgroup at most (those of one KV head).
constexpr uint32_t kMaxHeadsPerWg = 4;
// Threads per attention workgroup.
constexpr uint32_t kAttT = 256;

#define AS_LDS __attribute__((address_space(3)))
#define AS_GLB __attribute__((address_space(1)))

// 16 bytes from global memory straight into LDS (global_load_lds_dwordx4).
// The LDS address is dst_wave + 16 * lane, with dst_wave uniform across the
// wave: lanes that take part fill consecutive slots.  The data is in LDS
// once vmcnt reaches 0, and visible to other waves after a barrier.
__device__ __forceinline__ void lds_load16(const v4* src, v4* dst_wave) {
  __builtin_amdgcn_global_load_lds((const AS_GLB void*)src, (AS_LDS void*)dst_wave, 16, 0, 0);
}
// s_waitcnt vmcnt(0) (expcnt, lgkmcnt fields at their maxima: no wait).
__device__ __forceinline__ void wait_vm0() { __builtin_amdgcn_s_waitcnt(0x0F70); }
// Lane k of this lane's 16-lane row (DPP row_newbcast:k).
template <uint32_t K>
__device__ __forceinline__ float bcast16(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + (int)K, 0xF, 0xF, false));
}
// LDS per batched-GEMM workgroup: two workgroups fit one CU; small grids
// may use one workgroup's worth of almost all of it.
constexpr uint32_t kBgemmLds = 78 * 1024;
constexpr uint32_t kBgemmLdsBig = 150 * 1024;

// ---------------------------------------------------------------------------
// Batched GEMM.  A workgroup owns one R-row block of W and TB = 256 / R batch
// rows: thread t computes output (row b0 + t / R, column blk * R + t % R).
// K runs in chunks of KC: the block's [KC/4][R] v4 slice (contiguous in
// the blocked layout) and the TB input rows' KC floats are staged in LDS,
// then each thread continues its own chain acc = acc + W[m][k] * X[b][k],
// k ascending (code/cis2-fp/src/main.rs:228-243, math.rs:40-48); in tree
// mode the chain adds one tree32 block result per 32 k (math.rs:60-125).
//
// One launch may cover up to three matrices that read the same X (q, k and
// v): the grid's x blocks run over the segments in turn.  DUAL computes two
// chains per thread over W and W2 (gate and up) and stores
// silu(gate) * up (main.rs:484-487).  NORM applies the RMSNorm of each X row
// first (main.rs:245-260): the row's squares are summed in one strict chain
// (or tree32 blocks) from 0 over the row as staged in LDS (a first pass over
// the chunks when the row spans several), inv = 1/sqrt(sum/K + eps), and
// each staged element becomes (x*inv)*w[k].
// ---------------------------------------------------------------------------
constexpr uint32_t kMaxSegs = 3;
struct BgemmArgs {
  BgemmSeg s[kMaxSegs];
  uint32_t blk0[kMaxSegs + 1];  // first x block of each segment; blk0[nseg] = grid.x
  uint32_t nseg, n, TB, KC, tree;
  const float* W2;  // DUAL
  const float* nw;  // NORM
  float eps;
};

// Sum of squares of q4 16-byte groups, continuing the strict chain acc (or
// adding one tree32 per 8 groups, the last block zero-padded), read from
// LDS or global memory.
__device__ __forceinline__ float sumsq_groups(const v4* x4, uint32_t q4, float acc, bool tree) {
  if (tree) {
    for (uint32_t q0 = 0; q0 < q4; q0 += 8) {
      float l[32];
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) {
        const v4 v = q0 + i < q4 ? x4[q0 + i] : v4{0.0f, 0.0f, 0.0f, 0.0f};
        l[4 * i] = v.x * v.x;
        l[4 * i + 1] = v.y * v.y;
        l[4 * i + 2] = v.z * v.z;
        l[4 * i + 3] = v.w * v.w;
      }
      acc = acc + tree32(l);
    }
  } else {
#pragma unroll 8
    for (uint32_t q = 0; q < q4; ++q) {
      const v4 v = x4[q];
      float sq;
      sq = v.x * v.x; acc = acc + sq;
      sq = v.y * v.y; acc = acc + sq;
      sq = v.z * v.z; acc = acc + sq;
      sq = v.w * v.w; acc = acc + sq;
    }
  }
  return acc;
}
// RMSNorm factor from a row's sum of squares over K elements.
__device__ __forceinline__ float inv_rms_of(float sumsq, uint32_t K, float eps) {
  const float mean = sumsq / (float)K;
  const float arg = mean + eps;
  return rsqrt_cr(arg);
}

template <bool DUAL, bool NORM>
__global__ __launch_bounds__(256) void k_bgemm(BgemmArgs a) {
  extern __shared__ v4 sm[];
  __shared__ float s_inv[kT];
  uint32_t si = 0;
  if (a.nseg > 1 && blockIdx.x >= a.blk0[1]) si = (a.nseg > 2 && blockIdx.x >= a.blk0[2]) ? 2 : 1;
  const BgemmSeg g = si == 0 ? a.s[0] : (si == 1 ? a.s[1] : a.s[2]);
  const uint32_t R = g.R, TB = a.TB, KC = a.KC, K = g.K;
  const uint32_t blk = blockIdx.x - a.blk0[si], b0 = blockIdx.y * TB, t = threadIdx.x;
  const uint32_t r = t % R, bb = t / R;  // the thread's row: b0 + bb
  const uint32_t wv = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
  const bool live = t < R * TB;
  const uint32_t qmax = KC / 4, xs4 = qmax + 1;  // padded X rows: no bank aliasing
  v4* Ws = sm;                                   // [q4][R] (DUAL: then W2's at Ws + qmax * R)
  v4* Xs = sm + (size_t)(DUAL ? 2 : 1) * qmax * R;
  v4* NWs = Xs + (size_t)TB * xs4;               // NORM: the chunk's norm weights
  const v4* Wg = reinterpret_cast<const v4*>(g.W + (size_t)blk * R * K);
  const v4* Wg2 = DUAL ? reinterpret_cast<const v4*>(a.W2 + (size_t)blk * R * K) : nullptr;
  float acc = 0.0f, acc2 = 0.0f;
  // the chunk's X rows (and norm weights), every load in flight at once,
  // straight into LDS; each wave instruction fills 64 consecutive 16-byte
  // slots
  auto stage_x = [&](uint32_t g0, uint32_t q4, bool with_nw) {
    const uint32_t pieces = (q4 + 63) / 64, nx = TB * pieces;
    // workgroups start at different rows: the grid's requests for the
    // shared X rows spread over the cache channels
    const uint32_t rot = (blockIdx.x * 5) % nx;
    for (uint32_t j0 = wv; j0 < nx; j0 += kT / 64) {
      const uint32_t j = j0 + rot < nx ? j0 + rot : j0 + rot - nx;
      const uint32_t bx = j / pieces, q0 = (j - bx * pieces) * 64;
      const uint32_t row = std::min(b0 + bx, a.n - 1);
      const v4* xr = reinterpret_cast<const v4*>(g.X + (size_t)row * g.ldx) + g0 + q0;
      if (q0 + lane < q4) lds_load16(xr + lane, Xs + bx * xs4 + q0);
    }
    if (NORM && with_nw) {
      const v4* nw4p = reinterpret_cast<const v4*>(a.nw) + g0;
      for (uint32_t i0 = wv * 64; i0 < q4; i0 += kT)
        if (i0 + lane < q4) lds_load16(nw4p + i0 + lane, NWs + i0);
    }
  };
  // RMSNorm of the staged rows: one lane per batch row continues its
  // sum-of-squares chain over each chunk from LDS.  Rows longer than one
  // chunk take a first pass over their chunks before the GEMM's.
  float ssq = 0.0f;
  if (NORM && K > KC) {
    for (uint32_t k0 = 0; k0 < K; k0 += KC) {
      const uint32_t q4 = std::min(KC, K - k0) / 4;
      stage_x(k0 / 4, q4, false);
      wait_vm0();
      __syncthreads();
      if (t < TB) ssq = sumsq_groups(Xs + t * xs4, q4, ssq, a.tree);
      __syncthreads();
    }
    if (t < TB) s_inv[t] = inv_rms_of(ssq, K, a.eps);
  }
  for (uint32_t k0 = 0; k0 < K; k0 += KC) {
    const uint32_t q4 = std::min(KC, K - k0) / 4, g0 = k0 / 4;
    const uint32_t nw4 = q4 * R;
    for (uint32_t i0 = wv * 64; i0 < nw4; i0 += kT)
      if (i0 + lane < nw4) lds_load16(Wg + (size_t)g0 * R + i0 + lane, Ws + i0);
    if (DUAL) {
      for (uint32_t i0 = wv * 64; i0 < nw4; i0 += kT)
        if (i0 + lane < nw4) lds_load16(Wg2 + (size_t)g0 * R + i0 + lane, Ws + qmax * R + i0);
    }
    stage_x(g0, q4, true);
    wait_vm0();
    __syncthreads();
    if (NORM) {
      if (K <= KC) {
        if (t < TB) s_inv[t] = inv_rms_of(sumsq_groups(Xs + t * xs4, q4, 0.0f, a.tree), K, a.eps);
        __syncthreads();
      }
      for (uint32_t i = t; i < TB * q4; i += kT) {
        const uint32_t bx = i / q4, q = i - bx * q4;
        const float inv = s_inv[bx];
        const v4 x = Xs[bx * xs4 + q], w = NWs[q];
        v4 y;
        float sx;
        sx = x.x * inv; y.x = sx * w.x;
        sx = x.y * inv; y.y = sx * w.y;
        sx = x.z * inv; y.z = sx * w.z;
        sx = x.w * inv; y.w = sx * w.w;
        Xs[bx * xs4 + q] = y;
      }
      __syncthreads();
    }
    if (live) {
      const v4* wp = Ws + r;
      const v4* wp2 = Ws + qmax * R + r;
      const v4* xp = Xs + bb * xs4;
      if (a.tree) {
        for (uint32_t q = 0; q < q4; q += 8) {
          float l[32], l2[32];
#pragma unroll
          for (uint32_t j = 0; j < 8; ++j) {
            v4 w = v4{0.0f, 0.0f, 0.0f, 0.0f}, x = w, w2 = w;
            if (q + j < q4) {
              w = wp[(size_t)(q + j) * R];
              x = xp[q + j];
              if (DUAL) w2 = wp2[(size_t)(q + j) * R];
            }
            asm("" : "+v"(x) : "v"(w), "v"(w2));  // W the left operand (see ChainSums)
            l[4 * j] = w.x * x.x;
            l[4 * j + 1] = w.y * x.y;
            l[4 * j + 2] = w.z * x.z;
            l[4 * j + 3] = w.w * x.w;
            if (DUAL) {
              l2[4 * j] = w2.x * x.x;
              l2[4 * j + 1] = w2.y * x.y;
              l2[4 * j + 2] = w2.z * x.z;
              l2[4 * j + 3] = w2.w * x.w;
            }
          }
          acc = acc + tree32(l);
          if (DUAL) acc2 = acc2 + tree32(l2);
        }
      } else {
        // software pipelined over two register sets: the reads of the next
        // 4 q go out before the current 4 q's products and chain steps
        // (reads past the end are clamped to the last q and unused)
        constexpr uint32_t U = 4;
        v4 aw[U], ax[U], aw2[U], bw[U], bx[U], bw2[U];
        auto load = [&](v4 (&w)[U], v4 (&x)[U], v4 (&w2)[U], uint32_t q0) {
#pragma unroll
          for (uint32_t u = 0; u < U; ++u) {
            const uint32_t qq = std::min(q0 + u, q4 - 1);
            w[u] = wp[(size_t)qq * R];
            x[u] = xp[qq];
            if (DUAL) w2[u] = wp2[(size_t)qq * R];
          }
        };
        auto step = [&](const v4 (&w)[U], const v4 (&x)[U], const v4 (&w2)[U]) {
          float p[4 * U], p2[4 * U];
#pragma unroll
          for (uint32_t u = 0; u < U; ++u) {
            p[4 * u] = w[u].x * x[u].x;
            p[4 * u + 1] = w[u].y * x[u].y;
            p[4 * u + 2] = w[u].z * x[u].z;
            p[4 * u + 3] = w[u].w * x[u].w;
            if (DUAL) {
              p2[4 * u] = w2[u].x * x[u].x;
              p2[4 * u + 1] = w2[u].y * x[u].y;
              p2[4 * u + 2] = w2[u].z * x[u].z;
              p2[4 * u + 3] = w2[u].w * x[u].w;
            }
          }
#pragma unroll
          for (uint32_t i = 0; i < 4 * U; ++i) {
            acc = acc + p[i];
            if (DUAL) acc2 = acc2 + p2[i];
          }
        };
        uint32_t q = 0;
        if (q4 >= U) {
          load(aw, ax, aw2, 0);
          for (; q + 2 * U <= q4; q += 2 * U) {
            load(bw, bx, bw2, q + U);
            step(aw, ax, aw2);
            load(aw, ax, aw2, q + 2 * U);
            step(bw, bx, bw2);
          }
          if (q + U <= q4) {  // set a holds q .. q+U-1
            step(aw, ax, aw2);
            q += U;
          }
        }
        for (; q < q4; ++q) {
          const v4 w = wp[(size_t)q * R], x = xp[q];
          const v4 w2 = DUAL ? wp2[(size_t)q * R] : w;
          float pp;
          pp = w.x * x.x; acc = acc + pp;
          pp = w.y * x.y; acc = acc + pp;
          pp = w.z * x.z; acc = acc + pp;
          pp = w.w * x.w; acc = acc + pp;
          if (DUAL) {
            pp = w2.x * x.x; acc2 = acc2 + pp;
            pp = w2.y * x.y; acc2 = acc2 + pp;
            pp = w2.z * x.z; acc2 = acc2 + pp;
            pp = w2.w * x.w; acc2 = acc2 + pp;
          }
        }
      }
    }
    __syncthreads();
  }
  const uint32_t m = blk * R + r, row = b0 + bb;
  if (live && row < a.n && m < g.M) {
    float y = acc;
    if (DUAL) {
      const float sg = silu_pinned(acc);
      y = sg * acc2;
    } else if (g.epi == kEpiBias) {
      y = acc + g.add[m];
    } else if (g.epi == kEpiResidual) {
      y = g.add[(size_t)row * g.ldadd + m] + acc;
    }
    g.Y[(size_t)row * g.ldy + m] = y;
  }
}

// ---------------------------------------------------------------------------
// Batched GEMM in tiles of 16 outputs x 16 batch rows (sequential order, W
// in blocks of R = 8 or 16 rows): a workgroup owns 16 consecutive outputs m
// (16 / R blocks of W) and 16 batch rows; lane l of wave w computes output
// (row 4w + l/16, column l%16) as one strict chain acc + W[m][k] * X[b][k],
// k ascending (code/cis2-fp/src/main.rs:228-243, math.rs:40-48), the bits
// of k_bgemm.  A 16-lane row of a wave shares one batch row: each lane
// reads 4 consecutive k of X per 16-byte LDS read (the row: 64 k), and a
// chain takes X[b][k] from lane (k/4) % 16 of its row by DPP broadcast
// (row_newbcast) inside the multiply; the chains' LDS reads are the W groups
// (a ring of D reads ahead) and one X read per 64 k, where k_bgemm's lanes
// read an X group per 4 k.  NORM: each 16-lane row computes its row's
// inverse RMS from the staged X (the squares' sum in one strict chain, the
// partial sums broadcast the same way), and the chain scales each X read,
// (x * inv) * w[k], before use.  Operands go through registers per K chunk:
// every load of the chunk in flight, then the LDS writes.
// LDS (16-byte groups): W blocks [16/R][q4max * R + 8] (the pad keeps the
// two blocks' reads in distinct banks), W2 the same (DUAL), norm weights
// [q4max], X [16][q4max + 1], then b16_slack(R) readable groups (the
// rings read up to 23 W groups, at stride R, and 31 X groups past a
// chunk's end; the values are never used).
// ---------------------------------------------------------------------------
inline uint32_t b16_slack(uint32_t R) { return 24 * R + 64; }

// Steps G .. 15 of a 16-group block starting at group q: ring slot G % D
// holds W group q + G (refilled with q + G + D), xq is this lane's X group
// q + (lane % 16); X[b][4(q + G) + j] is component j of lane G's xq.
template <bool DUAL, uint32_t D, uint32_t G = 0>
__device__ __forceinline__ void b16_block(float& acc, float& acc2, const v4& xq, v4 (&rw)[D],
                                          v4 (&rw2)[D], const v4* wp, const v4* wp2, uint32_t R,
                                          uint32_t q) {
  if constexpr (G < 16) {
    const v4 w = rw[G % D];
    const float x0 = bcast16<G>(xq.x), x1 = bcast16<G>(xq.y);
    const float x2 = bcast16<G>(xq.z), x3 = bcast16<G>(xq.w);
    float p;
    p = x0 * w.x; acc = acc + p;
    p = x1 * w.y; acc = acc + p;
    p = x2 * w.z; acc = acc + p;
    p = x3 * w.w; acc = acc + p;
    if (DUAL) {
      const v4 w2 = rw2[G % D];
      p = x0 * w2.x; acc2 = acc2 + p;
      p = x1 * w2.y; acc2 = acc2 + p;
      p = x2 * w2.z; acc2 = acc2 + p;
      p = x3 * w2.w; acc2 = acc2 + p;
    }
    rw[G % D] = wp[(size_t)(q + G + D) * R];
    if (DUAL) rw2[G % D] = wp2[(size_t)(q + G + D) * R];
    __builtin_amdgcn_sched_barrier(0);
    b16_block<DUAL, D, G + 1>(acc, acc2, xq, rw, rw2, wp, wp2, R, q);
  }
}
// The first nt (< 16) steps of b16_block.
template <bool DUAL, uint32_t D, uint32_t G = 0>
__device__ __forceinline__ void b16_tail(float& acc, float& acc2, const v4& xq, v4 (&rw)[D],
                                         v4 (&rw2)[D], const v4* wp, const v4* wp2, uint32_t R,
                                         uint32_t q, uint32_t nt) {
  if constexpr (G < 15) {
    if (G < nt) {
      const v4 w = rw[G % D];
      const float x0 = bcast16<G>(xq.x), x1 = bcast16<G>(xq.y);
      const float x2 = bcast16<G>(xq.z), x3 = bcast16<G>(xq.w);
      float p;
      p = x0 * w.x; acc = acc + p;
      p = x1 * w.y; acc = acc + p;
      p = x2 * w.z; acc = acc + p;
      p = x3 * w.w; acc = acc + p;
      if (DUAL) {
        const v4 w2 = rw2[G % D];
        p = x0 * w2.x; acc2 = acc2 + p;
        p = x1 * w2.y; acc2 = acc2 + p;
        p = x2 * w2.z; acc2 = acc2 + p;
        p = x3 * w2.w; acc2 = acc2 + p;
      }
      rw[G % D] = wp[(size_t)(q + G + D) * R];
      if (DUAL) rw2[G % D] = wp2[(size_t)(q + G + D) * R];
      __builtin_amdgcn_sched_barrier(0);
      b16_tail<DUAL, D, G + 1>(acc, acc2, xq, rw, rw2, wp, wp2, R, q, nt);
    }
  }
}
// Sum of squares of n groups x4[0 .. n-1] continuing acc, strict order:
// blocks of 8 groups, the next block's squares formed between this block's
// adds (x4 in LDS with 16 readable groups past n).
template <uint32_t U = 0>
__device__ __forceinline__ void sq_step(float& acc, float (&s)[8][4], const v4* x4, uint32_t gn) {
  if constexpr (U < 8) {
    const v4 v = x4[gn + U];
    acc = acc + s[U][0];
    s[U][0] = v.x * v.x;
    acc = acc + s[U][1];
    s[U][1] = v.y * v.y;
    acc = acc + s[U][2];
    s[U][2] = v.z * v.z;
    acc = acc + s[U][3];
    s[U][3] = v.w * v.w;
    sq_step<U + 1>(acc, s, x4, gn);
  }
}
__device__ __forceinline__ float sumsq_pipe(const v4* x4, uint32_t n, float acc) {
  float s[8][4];
#pragma unroll
  for (uint32_t u = 0; u < 8; ++u) {
    const v4 v = x4[u];
    s[u][0] = v.x * v.x;
    s[u][1] = v.y * v.y;
    s[u][2] = v.z * v.z;
    s[u][3] = v.w * v.w;
  }
  uint32_t g = 0;
  for (; g + 8 < n; g += 8) sq_step(acc, s, x4, g + 8);
#pragma unroll
  for (uint32_t u = 0; u < 8; ++u)
    if (g + u < n) {
      acc = acc + s[u][0];
      acc = acc + s[u][1];
      acc = acc + s[u][2];
      acc = acc + s[u][3];
    }
  return acc;
}

template <bool DUAL, bool NORM>
__global__ __launch_bounds__(256) void k_bgemm16(BgemmArgs a) {
  extern __shared__ v4 sm[];
  constexpr uint32_t D = 8;  // W groups read ahead (a divisor of 16: the ring slot of
                             // group q + G is G % D for every block start q)
  uint32_t si = 0;
  if (a.nseg > 1 && blockIdx.x >= a.blk0[1]) si = (a.nseg > 2 && blockIdx.x >= a.blk0[2]) ? 2 : 1;
  const BgemmSeg g = si == 0 ? a.s[0] : (si == 1 ? a.s[1] : a.s[2]);
  const uint32_t R = g.R, KC = a.KC, K = g.K, nblk = 16 / R;
  const uint32_t tile = blockIdx.x - a.blk0[si], b0 = blockIdx.y * 16, t = threadIdx.x;
  const uint32_t wv = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
  const uint32_t c = lane & 15, bb = wv * 4 + (lane >> 4);  // output column, batch row
  const uint32_t qmax = KC / 4, xs4 = qmax + 1, BS = qmax * R + 8;
  v4* Ws = sm;                                   // [nblk][BS]
  v4* W2s = Ws + (size_t)nblk * BS;              // DUAL
  v4* NWs = W2s + (DUAL ? (size_t)nblk * BS : 0);  // NORM: the chunk's norm weights
  v4* Xs = NWs + (NORM ? qmax : 0);              // [16][xs4]
  const v4* Wg = reinterpret_cast<const v4*>(g.W + (size_t)tile * 16 * K);
  const v4* Wg2 = DUAL ? reinterpret_cast<const v4*>(a.W2 + (size_t)tile * 16 * K) : nullptr;
  // A chunk's operands (groups g0 .. g0+q4-1): per round, a thread loads up
  // to 8 W (and 8 W2) groups of the tile's blocks, the X groups of 4 rows
  // (wave w: rows 4w .. 4w+3, lanes over the groups) and one norm weight
  // group, all in flight, then writes them.
  auto stage = [&](uint32_t g0, uint32_t q4, bool with_w) {
    constexpr uint32_t WB = 8, XP = 4;
    const uint32_t nwb = q4 * R, nw = with_w ? nblk * nwb : 0, pieces = (q4 + 63) / 64;
    for (uint32_t rd = 0; rd == 0 || rd * 256 * WB < nw; ++rd) {
      v4 tw[WB], tw2[WB], tx[4][XP], tn;
#pragma unroll
      for (uint32_t u = 0; u < WB; ++u) {
        const uint32_t i = (rd * WB + u) * 256 + t;
        if (i < nw) {
          const uint32_t cb = i >= nwb ? 1 : 0, j = i - cb * nwb;
          tw[u] = Wg[(size_t)cb * R * K / 4 + (size_t)g0 * R + j];
          if (DUAL) tw2[u] = Wg2[(size_t)cb * R * K / 4 + (size_t)g0 * R + j];
        }
      }
      if (rd == 0) {
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
          const uint32_t bx = wv * 4 + j, row = std::min(b0 + bx, a.n - 1);
          const v4* xr = reinterpret_cast<const v4*>(g.X + (size_t)row * g.ldx) + g0;
#pragma unroll
          for (uint32_t pc = 0; pc < XP; ++pc) {
            const uint32_t q = pc * 64 + lane;
            if (pc < pieces && q < q4) tx[j][pc] = xr[q];
          }
        }
        if (NORM && with_w && t < q4) tn = reinterpret_cast<const v4*>(a.nw)[g0 + t];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (uint32_t u = 0; u < WB; ++u) {
        const uint32_t i = (rd * WB + u) * 256 + t;
        if (i < nw) {
          const uint32_t cb = i >= nwb ? 1 : 0, j = i - cb * nwb;
          Ws[cb * BS + j] = tw[u];
          if (DUAL) W2s[cb * BS + j] = tw2[u];
        }
      }
      if (rd == 0) {
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
          const uint32_t bx = wv * 4 + j;
#pragma unroll
          for (uint32_t pc = 0; pc < XP; ++pc) {
            const uint32_t q = pc * 64 + lane;
            if (pc < pieces && q < q4) Xs[bx * xs4 + q] = tx[j][pc];
          }
        }
        if (NORM && with_w && t < q4) NWs[t] = tn;
      }
    }
  };
  // RMSNorm: the 16 lanes of a batch row chain its squares (strict order)
  // over each staged chunk (16-byte reads, the same address across the
  // row's lanes); rows longer than one chunk take a first pass over their
  // chunks before the GEMM's.
  const v4* xrow = Xs + bb * xs4;
  const v4* xr = xrow + c;
  auto sumsq_chunk = [&](uint32_t q4, float acc0) { return sumsq_pipe(xrow, q4, acc0); };
  float inv = 0.0f;
  if (NORM && K > KC) {
    float ssq = 0.0f;
    for (uint32_t k0 = 0; k0 < K; k0 += KC) {
      const uint32_t q4 = std::min(KC, K - k0) / 4;
      stage(k0 / 4, q4, false);
      __syncthreads();
      ssq = sumsq_chunk(q4, ssq);
      __syncthreads();
    }
    inv = inv_rms_of(ssq, K, a.eps);
  }
  float acc = 0.0f, acc2 = 0.0f;
  const uint32_t cb = c / R, r = c - cb * R;
  const v4* wp = Ws + cb * BS + r;
  const v4* wp2 = W2s + cb * BS + r;
  for (uint32_t k0 = 0; k0 < K; k0 += KC) {
    const uint32_t q4 = std::min(KC, K - k0) / 4;
    stage(k0 / 4, q4, true);
    __syncthreads();
    if (NORM && K <= KC) inv = inv_rms_of(sumsq_chunk(q4, 0.0f), K, a.eps);
    // this lane's X group of a block, scaled for NORM
    auto xget = [&](uint32_t q) {
      v4 x = xr[q];
      if (NORM) {
        const v4 w = NWs[q + c];
        float sx;
        sx = x.x * inv; x.x = sx * w.x;
        sx = x.y * inv; x.y = sx * w.y;
        sx = x.z * inv; x.z = sx * w.z;
        sx = x.w * inv; x.w = sx * w.w;
      }
      return x;
    };
    v4 rw[D], rw2[D];
#pragma unroll
    for (uint32_t u = 0; u < D; ++u) {
      rw[u] = wp[(size_t)u * R];
      if (DUAL) rw2[u] = wp2[(size_t)u * R];
    }
    v4 xq = xget(0);
    uint32_t q = 0;
    for (; q + 16 <= q4; q += 16) {
      const v4 xn = xget(q + 16);  // the next block's X (past the end: unused)
      b16_block<DUAL, D>(acc, acc2, xq, rw, rw2, wp, wp2, R, q);
      xq = xn;
    }
    if (q < q4) b16_tail<DUAL, D>(acc, acc2, xq, rw, rw2, wp, wp2, R, q, q4 - q);
    __syncthreads();
  }
  const uint32_t m = tile * 16 + c, row = b0 + bb;
  if (row < a.n && m < g.M) {
    float y = acc;
    if (DUAL) {
      const float sg = silu_pinned(acc);
      y = sg * acc2;
    } else if (g.epi == kEpiBias) {
      y = acc + g.add[m];
    } else if (g.epi == kEpiResidual) {
      y = g.add[(size_t)row * g.ldadd + m] + acc;
    }
    g.Y[(size_t)row * g.ldy + m] = y;
  }
}

// ---------------------------------------------------------------------------
// Batched GEMM for few rows (decode steps; sequential order): a workgroup
// owns 8 outputs x 8 batch rows, 64 chains, and splits the work of a chain
// step between its waves.  Eight product waves form p = W[m][k] * X[b][k] for
// a 16-byte group of every chain (lane l: output l % 8, row l / 8) and store
// the groups in an LDS ring of four slots of 16 groups; chain wave 0 adds
// them, k ascending, one chain per lane (k_bgemm's bits).  DUAL: chain wave 1
// runs the up projection's chains over W2, and silu(gate) * up is stored.
// NORM: wave 0 chains the rows' squares first, then the rows are scaled in
// LDS, (x * inv) * w[k].  W (and X without a norm) goes from global memory to
// the product waves' registers, D slots ahead (all of K = 576).
// What bounds it: 3.6 us of launch, prologue and end, then the chain, 9.6
// cycles per k (6.1 with nothing else on the LDS) against 16 when the chain's
// wave forms its own products (k_bgemm16).  At 8 rows, us, k_bgemm16 then
// here: 960 x 576 with the norm 12.0 8.6, 576 x 576 8.3 6.1, gate and up of
// 1536 x 576 with the norm 16.1 10.1, 576 x 1536 16.8 9.8.
// LDS (16-byte groups): ring [CW][4 slots][16][64] (first the squares), NORM:
// rows [K/4][8], then inverse RMS [8] and up sums [64].  Past K the products
// are -0, which no sum notices.
// ---------------------------------------------------------------------------
template <bool DUAL, bool NORM>
struct ChainCfg {
  static constexpr uint32_t CW = DUAL ? 2 : 1, NP = 8, T = 64 * (CW + NP);
  static constexpr uint32_t SG = 16, GPW = SG / NP;      // groups per slot, per wave of it
  static constexpr uint32_t D = DUAL ? (NORM ? 5 : 4) : (NORM ? 9 : 8);  // slots loaded ahead
  static constexpr uint32_t ring = CW * 4 * SG * 64;     // 16-byte groups
  static constexpr size_t lds(uint32_t K) {
    return ((size_t)ring + (NORM ? (size_t)K / 4 * 8 : 0)) * 16 + (8 + 64) * 4;
  }
};
// Largest dynamic LDS of a workgroup.
constexpr size_t kLdsMost = 160 * 1024 - 256;
// s_waitcnt lgkmcnt(0), then s_barrier: LDS written before it is visible
// after it; global loads in flight stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <bool DUAL, bool NORM>
__global__ __launch_bounds__((ChainCfg<DUAL, NORM>::T), 3) void k_chain_gemm(BgemmArgs a) {
  using C = ChainCfg<DUAL, NORM>;
  constexpr uint32_t CW = C::CW, NP = C::NP, GPW = C::GPW, SG = C::SG, D = C::D, T = C::T;
  // at LDS address 0, as chain_ring needs: no static __shared__ in this kernel
  extern __shared__ v4 sm[];
  uint32_t si = 0;
  if (a.nseg > 1 && blockIdx.x >= a.blk0[1]) si = (a.nseg > 2 && blockIdx.x >= a.blk0[2]) ? 2 : 1;
  const BgemmSeg g = si == 0 ? a.s[0] : (si == 1 ? a.s[1] : a.s[2]);
  const uint32_t R = g.R, K = g.K, K4 = K / 4, t = threadIdx.x;
  const uint32_t m0 = (blockIdx.x - a.blk0[si]) * 8, b0 = blockIdx.y * 8;
  const uint32_t wv = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
  const uint32_t r = lane & 7, b = lane >> 3, ns = (K4 + SG - 1) / SG;
  v4* ring = sm;
  v4* xs = sm + C::ring;                                    // [K4][8]
  float* s_inv = reinterpret_cast<float*>(xs + (NORM ? K4 * 8 : 0));  // [8]
  float* s_up = s_inv + 8;                                  // [64]
  // X rows as [group][row] (and the squares, into the ring's space): the
  // loads go out before W's, in the order they are needed
  const v4* xn = reinterpret_cast<const v4*>(g.X + (size_t)min(b0 + (t & 7), a.n - 1) * g.ldx);
  constexpr uint32_t XB = 6;  // X loads in flight (K = 1536 in one round)
  v4 x0[XB];
#pragma unroll
  for (uint32_t i = 0; i < XB; ++i)
    if (NORM && t + T * i < K4 * 8) x0[i] = xn[(t + T * i) >> 3];
  const bool chain = wv < CW;
  const size_t woff = (size_t)(m0 / R) * R * K4 + m0 % R + r;
  const v4* wp = reinterpret_cast<const v4*>(g.W) + woff;
  const v4* wp2 = DUAL ? reinterpret_cast<const v4*>(a.W2) + woff : nullptr;
  const v4* xp = reinterpret_cast<const v4*>(g.X + (size_t)min(b0 + b, a.n - 1) * g.ldx);
  v4 pw[D][GPW], pu[D][GPW], px[D][GPW];
  // the groups of slot c that this wave forms (past K: the last one again)
  auto load = [&](uint32_t c, uint32_t s) {
#pragma unroll
    for (uint32_t i = 0; i < GPW; ++i) {
      const uint32_t q = min(c * SG + i * NP + (wv - CW), K4 - 1);
      pw[s][i] = wp[q * R];
      if (DUAL) pu[s][i] = wp2[q * R];
      if (!NORM) px[s][i] = xp[q];
    }
  };
  if (!chain) {
#pragma unroll
    for (uint32_t s = 0; s < D; ++s)
      if (s < ns) load(s, s);
  }
  auto square = [](const v4& x) {
    v4 q;
    q.x = x.x * x.x;
    q.y = x.y * x.y;
    q.z = x.z * x.z;
    q.w = x.w * x.w;
    return q;
  };
  if (NORM) {
#pragma unroll
    for (uint32_t i = 0; i < XB; ++i) {
      const uint32_t e = t + T * i;
      if (e < K4 * 8) {
        xs[e] = x0[i];
        ring[e] = square(x0[i]);
      }
    }
    for (uint32_t e = t + T * XB; e < K4 * 8; e += T) {
      const v4 x = xn[e >> 3];
      xs[e] = x;
      ring[e] = square(x);
    }
    lds_barrier();
    if (wv == 0) {
      float acc = 0.0f;
      const v4* sp = ring + r;  // lane l: row l % 8
      const uint32_t np = K4 / 16;
      if (np) acc = chain_lds16_low<8>((const AS_LDS void*)sp, np, acc);
      for (uint32_t q = 16 * np; q < K4; ++q) {
        const v4 x = sp[q * 8];
        acc = acc + x.x;
        acc = acc + x.y;
        acc = acc + x.z;
        acc = acc + x.w;
      }
      const float inv = inv_rms_of(acc, K, a.eps);
      if (lane < 8) s_inv[lane] = inv;
    }
    lds_barrier();
    const float inv = s_inv[t & 7];
    for (uint32_t i = t; i < K4 * 8; i += T) {
      v4 x = xs[i];
      const v4 w = reinterpret_cast<const v4*>(a.nw)[i >> 3];
      float sx;
      sx = x.x * inv; x.x = sx * w.x;
      sx = x.y * inv; x.y = sx * w.y;
      sx = x.z * inv; x.z = sx * w.z;
      sx = x.w * inv; x.w = sx * w.w;
      xs[i] = x;
    }
  }
  // the addend's load is in flight during the chains
  const uint32_t m = m0 + r, row = b0 + b;
  const bool mine = wv == 0 && row < a.n && m < g.M;
  float addend = 0.0f;
  if (!DUAL && mine && g.epi != kEpiNone)
    addend = g.epi == kEpiBias ? g.add[m] : g.add[(size_t)row * g.ldadd + m];
  lds_barrier();
  float acc = 0.0f;
  if (chain) {
    __builtin_amdgcn_s_setprio(3);
    lds_barrier();  // slot 0
    const uint32_t base = (uint32_t)(uintptr_t)(const AS_LDS void*)(ring + wv * 4 * SG * 64);
    acc = chain_ring(base + lane * 16, base, ns, acc);
  } else {
    v4 x[GPW];
    auto xload = [&](uint32_t c) {
#pragma unroll
      for (uint32_t i = 0; i < GPW; ++i)
        if (NORM) x[i] = xs[min(c * SG + i * NP + (wv - CW), K4 - 1) * 8 + b];
    };
    xload(0);
    for (uint32_t c0 = 0; c0 < ns; c0 += D) {
#pragma unroll
      for (uint32_t s = 0; s < D; ++s) {
        const uint32_t c = c0 + s;
        if (c >= ns) break;
        v4 p[GPW], p2[GPW];
#pragma unroll
        for (uint32_t i = 0; i < GPW; ++i) {
          const v4 w = pw[s][i];
          if (!NORM) x[i] = px[s][i];
          p[i].x = w.x * x[i].x;
          p[i].y = w.y * x[i].y;
          p[i].z = w.z * x[i].z;
          p[i].w = w.w * x[i].w;
          if (DUAL) {
            const v4 w2 = pu[s][i];
            p2[i].x = w2.x * x[i].x;
            p2[i].y = w2.y * x[i].y;
            p2[i].z = w2.z * x[i].z;
            p2[i].w = w2.w * x[i].w;
          }
        }
        if ((c + 1) * SG > K4) {  // the last slot's groups past K
          const float z = __int_as_float((int)0x80000000u);
#pragma unroll
          for (uint32_t i = 0; i < GPW; ++i)
            if (c * SG + i * NP + (wv - CW) >= K4) p[i] = p2[i] = v4{z, z, z, z};
        }
        v4* slot = ring + (c & 3) * SG * 64 + lane;
#pragma unroll
        for (uint32_t i = 0; i < GPW; ++i) {
          slot[(i * NP + (wv - CW)) * 64] = p[i];
          if (DUAL) slot[(4 * SG + i * NP + (wv - CW)) * 64] = p2[i];
        }
        xload(c + 1);
        if (c + D < ns) load(c + D, s);
        lds_barrier();
      }
    }
  }
  if (DUAL) {
    if (wv == 1) s_up[lane] = acc;
    lds_barrier();
  }
  if (mine) {
    float y = acc;
    if (DUAL) {
      const float sg = silu_pinned(acc);
      y = sg * s_up[lane];
    } else if (g.epi == kEpiBias) {
      y = acc + addend;
    } else if (g.epi == kEpiResidual) {
      y = addend + acc;
    }
    g.Y[(size_t)row * g.ldy + m] = y;
  }
}

// ---------------------------------------------------------------------------
// Batched GEMM with the products formed by the matrix cores (either order,
// any block height R).  One v_mfma_f32_16x16x1_4b_f32 multiplies four
// pairs of 16-vectors; given the 16 W rows and 16 X rows of a tile at four
// consecutive k, and -0 as the addend, each of its 4 x 256 results is one
// correctly rounded product W[m][k] * X[b][k] (x + (-0) = x for every x, so
// the sign of a zero product survives; flushing and NaN bits are those of
// v_mul_f32: two million products each of subnormal operands, of results next
// to 2^-126, of NaNs of every sign and payload, of infinities and zeros differ
// in no bit).  All four blocks leave a given output in the same lane, so the
// vector units only add: acc = acc + p, k ascending, the strict chain of
// k_bgemm (code/cis2-fp/src/main.rs:228-243, math.rs:40-48).  In tree order
// they add pairs of a lane's products instead, the same number of adds.
// ---------------------------------------------------------------------------
typedef float f16v __attribute__((ext_vector_type(16)));

// The four products of a 16 x 16 tile: a holds W[row l % 16][k + l / 16] and
// b X[row l % 16][k + l / 16] of lane l; element 4u + r of the result is
// output (W row 4 (l / 16) + r, X row l % 16) at k + u.
__device__ __forceinline__ f16v products4(float a, float b, const f16v& nz) {
  return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, nz, 0, 0, 0);
}
// A 16-register operand of -0.
__device__ __forceinline__ f16v minus_zeros() {
  float z = __int_as_float((int)0x80000000u);
  asm volatile("" : "+v"(z));
  f16v v;
#pragma unroll
  for (uint32_t i = 0; i < 16; ++i) v[i] = z;
  return v;
}

// Step x of 16 k over NT tiles: its tile and its four k.  Tree order takes a
// tile's four steps in turn, so that only one tile's partial sums are open.
template <uint32_t NT, bool TREE>
constexpr __host__ __device__ uint32_t mtile_s(uint32_t x) { return TREE ? x / 4 : x % NT; }
template <uint32_t NT, bool TREE>
constexpr __host__ __device__ uint32_t mtile_k(uint32_t x) { return TREE ? x % 4 : x / NT; }

// The adds of NT tiles.  add(): products4's p, for k = 4q .. 4q + 3 of every
// 32, into tile s: k ascending, or in tree order (math.rs:60-125) the pairs'
// sums of the 32, whose total acc takes (zeros before the first step: acc is
// +0 and stays so).  In tree order the earlier sum is the left operand of
// every add, and W of every product in k_bgemm too, as in the persistent
// kernel: of two NaNs the left one is kept.  (The compiler would swap the last
// add; the empty asm makes its right operand the later value.)
template <uint32_t NT, bool TREE>
struct ChainSums {
  float t4[4] = {}, t8[4] = {}, t16[TREE ? NT : 1][4] = {};
  __device__ __forceinline__ void add(float (&acc)[NT][4], uint32_t s, uint32_t q, const f16v& p) {
    if constexpr (TREE) {
#pragma unroll
      for (uint32_t r = 0; r < 4; ++r) {
        const float lo = p[r] + p[4 + r], hi = p[8 + r] + p[12 + r];
        const float v4k = lo + hi;
        if (q % 2 == 0) {
          t4[r] = v4k;
          continue;
        }
        const float v8k = t4[r] + v4k;
        if (q % 4 == 1) {
          t8[r] = v8k;
          continue;
        }
        const float v16k = t8[r] + v8k;
        if (q == 3) {
          t16[s][r] = v16k;
          continue;
        }
        float v32k = t16[s][r] + v16k;
        asm("" : "+v"(v32k) : "v"(acc[s][r]));  // acc stays the left operand
        acc[s][r] = acc[s][r] + v32k;
      }
      float* o = q == 7 ? acc[s] : (q == 3 ? t16[s] : (q % 2 ? t8 : t4));
      asm volatile("" : "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3]));
    } else {
#pragma unroll
      for (uint32_t b = 0; b < 4; ++b)
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) acc[s][r] = acc[s][r] + p[4 * b + r];
      asm volatile("" : "+v"(acc[s][0]), "+v"(acc[s][1]), "+v"(acc[s][2]), "+v"(acc[s][3]));
    }
  }
};

struct MgemmArgs {
  BgemmSeg s[kMaxSegs];
  uint32_t tile0[kMaxSegs + 1];  // first W tile of each segment; tile0[nseg] = W tiles
  uint32_t nseg, n, tiles;       // tiles: W tiles x X tiles
  uint32_t vec;                  // 1: outputs (and addends) in 16-byte groups
  const float* W2;               // DUAL
};

// What bounds it: the vector and matrix units.  A CU forms a product on
// either in the same time and they do not overlap (a wave64 product step of
// 1024 and its 16 adds: 32 + 32 cycles per SIMD with two or more waves), so
// the least is 64 cycles per 1024 chain steps, 39 T steps/s at 2.4 GHz; 16384
// rows run at 26 .. 30 T (k_bgemm16: 10 .. 13 T: a DPP broadcast, a multiply
// and an add per 64 steps, 16 cycles).  Letting the matrix cores form the
// products saves the operand reads instead: 16 + 16 values feed 256 chains.
//
// Four waves, WM x WN of them, each SM x SN tiles of 16 outputs x 16 batch
// rows.  DUAL: the first half of a wave's SM tiles comes from W, the second
// half from W2 at the same rows, and silu(gate) * up is stored
// (main.rs:484-487).
// LDS, two buffers of one K chunk each: [chunk / 16][4][rows] 16-byte groups;
// group (g, u, row) holds k = 16 g + u + {0, 4, 8, 12} of the row, so that a
// wave's 16-byte read gives lane l (row l % 16, u = l / 16) its operands of
// four products4.  A thread stages whole (row, 16 k) pieces: four 16-byte
// loads, transposed by register naming.  Past K the pieces hold -0 for W and
// +0 for X: their products are -0, which no sum notices.  In tree order the
// block of 32 that K ends in is filled with zeros, as tree32's last block is,
// and the last chunk ends with it: a block past K would add +0, which turns a
// sum of -0 (values that cancel to a flushed subnormal) into +0.  Chunk c + PF
// is loaded into registers while chunk c is computed.
// Stores a lane's outputs m .. m + 3 of X row `row`: sums y, with y2 those of
// the second matrix (DUAL).
template <bool DUAL>
__device__ __forceinline__ void mgemm_store(const MgemmArgs& a, const BgemmSeg& g, uint32_t m,
                                            uint32_t row, const float (&acc)[4],
                                            const float (&acc2)[4]) {
  if (row >= a.n || m >= g.M) return;
  float y[4];
#pragma unroll
  for (uint32_t r = 0; r < 4; ++r) y[r] = acc[r];
  float* yp = g.Y + (size_t)row * g.ldy + m;
  if (DUAL) {
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) {
      const float sg = silu_pinned(y[r]);
      y[r] = sg * acc2[r];
    }
  }
  const float* ad = nullptr;
  if (!DUAL && g.epi == kEpiBias) ad = g.add + m;
  if (!DUAL && g.epi == kEpiResidual) ad = g.add + (size_t)row * g.ldadd + m;
  if (a.vec) {
    if (ad) {
      const v4 z = *reinterpret_cast<const v4*>(ad);
#pragma unroll
      for (uint32_t r = 0; r < 4; ++r) y[r] = g.epi == kEpiBias ? y[r] + z[r] : z[r] + y[r];
    }
    *reinterpret_cast<v4*>(yp) = v4{y[0], y[1], y[2], y[3]};
  } else {
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r)
      if (m + r < g.M) yp[r] = ad ? (g.epi == kEpiBias ? y[r] + ad[r] : ad[r] + y[r]) : y[r];
  }
}

template <bool DUAL, uint32_t SM, uint32_t SN, uint32_t WM, uint32_t WN, uint32_t KC>
struct MgemmCfg {
  static constexpr uint32_t BM = 16 * SM * WM / (DUAL ? 2 : 1);  // W rows per tile
  static constexpr uint32_t BN = 16 * SN * WN;                   // X rows per tile
  static constexpr uint32_t RA = 16 * SM * WM, RB = BN, ROWS = RA + RB;
  static constexpr uint32_t NG = KC / 16;
  static constexpr uint32_t items = ROWS * NG, NIT = (items + 255) / 256;
  static constexpr size_t buf = (size_t)4 * ROWS * NG;  // 16-byte groups of one buffer
  static_assert(WM * WN == 4 && (!DUAL || SM % 2 == 0), "four waves");
};

template <bool DUAL, bool TREE, uint32_t SM, uint32_t SN, uint32_t WM, uint32_t WN, uint32_t KC,
          uint32_t OCC, uint32_t PF>
__global__ __launch_bounds__(256, OCC) void k_mgemm(MgemmArgs a) {
  using C = MgemmCfg<DUAL, SM, SN, WM, WN, KC>;
  constexpr uint32_t ROWS = C::ROWS, RA = C::RA, NG = C::NG, NIT = C::NIT, NT = SM * SN;
  __shared__ v4 sm[2 * C::buf];
  // consecutive workgroups go to the eight XCDs in turn: give each XCD a run
  // of tiles, W tiles first, so that the tiles of one X tile share its L2
  const uint32_t per = (a.tiles + 7) / 8;
  const uint32_t tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per || tile >= a.tiles) return;
  const uint32_t wt = a.tile0[a.nseg], nt = tile / wt, ut = tile - nt * wt;
  uint32_t si = 0;
  if (a.nseg > 1 && ut >= a.tile0[1]) si = (a.nseg > 2 && ut >= a.tile0[2]) ? 2 : 1;
  const BgemmSeg g = si == 0 ? a.s[0] : (si == 1 ? a.s[1] : a.s[2]);
  const uint32_t m0 = (ut - a.tile0[si]) * C::BM, n0 = nt * C::BN;
  const uint32_t t = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
  const uint32_t K4 = g.K / 4, lastblk = (g.M - 1) / g.R;
  // staging: piece it of this thread
  const v4* src[NIT];
  uint32_t step[NIT], q0[NIT], dst[NIT];
  bool isw[NIT];
#pragma unroll
  for (uint32_t j = 0; j < NIT; ++j) {
    const uint32_t it = min(j * 256 + t, C::items - 1);
    const uint32_t row = it % ROWS, gi = it / ROWS;
    isw[j] = row < RA;
    if (isw[j]) {
      // rows past M belong to no output: any stored block serves
      const bool second = DUAL && row >= RA / 2;
      const uint32_t m = m0 + (second ? row - RA / 2 : row);
      const uint32_t blk = min(m / g.R, lastblk), r = m % g.R;
      src[j] = reinterpret_cast<const v4*>((second ? a.W2 : g.W) + (size_t)blk * g.R * g.K) + r;
      step[j] = g.R;
    } else {
      const uint32_t b = min(n0 + row - RA, a.n - 1);
      src[j] = reinterpret_cast<const v4*>(g.X + (size_t)b * g.ldx);
      step[j] = 1;
    }
    q0[j] = 4 * gi;
    dst[j] = 4 * gi * ROWS + row;
  }
  v4 stage[PF][NIT][4];
  auto load = [&](uint32_t k0, v4 (&st)[NIT][4]) {
#pragma unroll
    for (uint32_t j = 0; j < NIT; ++j)
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t q = k0 / 4 + q0[j] + i;
        if (q < K4) {
          st[j][i] = src[j][(size_t)q * step[j]];
        } else {
          const float z = isw[j] && !TREE ? __int_as_float((int)0x80000000u) : 0.0f;
          st[j][i] = v4{z, z, z, z};
        }
      }
  };
  auto store = [&](uint32_t b, const v4 (&st)[NIT][4]) {
    v4* p = sm + b * C::buf;
#pragma unroll
    for (uint32_t j = 0; j < NIT; ++j) {
      if (C::items % 256 && j * 256 + t >= C::items) break;
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u)
        p[dst[j] + u * ROWS] = v4{st[j][0][u], st[j][1][u], st[j][2][u], st[j][3][u]};
    }
  };
  // wave (wm, wn); tile i of its SM: rows 16 * (i * WM + wm) for one matrix,
  // of W then of W2 for DUAL
  const uint32_t wm = wv % WM, wn = wv / WM, u = lane >> 4, c16 = lane & 15;
  constexpr uint32_t SMH = DUAL ? SM / 2 : SM;
  auto arow = [&](uint32_t i) {  // first LDS row of A tile i
    const uint32_t h = i / SMH, ii = i - h * SMH;
    return h * (RA / 2) * (DUAL ? 1 : 0) + 16 * (wm * SMH + ii);
  };
  const f16v nz = minus_zeros();
  float acc[NT][4];
#pragma unroll
  for (uint32_t s = 0; s < NT; ++s)
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) acc[s][r] = 0.0f;
  f16v d[2];
#pragma unroll
  for (uint32_t i = 0; i < 16; ++i) d[1][i] = __int_as_float((int)0x80000000u);
  ChainSums<NT, TREE> sums;
  const uint32_t nc = (g.K + KC - 1) / KC;
  load(0, stage[0]);
  if (PF == 2 && nc > 1) load(KC, stage[1]);
  store(0, stage[0]);
  auto chunk = [&](uint32_t ci, v4 (&cur)[NIT][4], v4 (&nxt)[NIT][4]) {
    __syncthreads();
    if (ci + PF < nc) load((ci + PF) * KC, cur);
    const v4* p = sm + (ci & 1) * C::buf + u * ROWS + c16;
    v4 fa[2][SM], fb[2][SN];
    auto frags = [&](uint32_t gi, uint32_t f) {
#pragma unroll
      for (uint32_t i = 0; i < SM; ++i) fa[f][i] = p[4 * gi * ROWS + arow(i)];
#pragma unroll
      for (uint32_t j = 0; j < SN; ++j) fb[f][j] = p[4 * gi * ROWS + RA + 16 * (wn * SN + j)];
    };
    frags(0, 0);
#pragma unroll
    for (uint32_t gi = 0; gi < NG; ++gi) {
      if (TREE && gi && gi % 2 == 0 && ci * KC + 16 * gi >= g.K) break;
      if (gi + 1 < NG) frags(gi + 1, (gi + 1) & 1);
#pragma unroll
      for (uint32_t x = 0; x < 4 * NT; ++x) {
        // these products while the vector units add the ones before them
        const uint32_t m = mtile_k<NT, TREE>(x), s = mtile_s<NT, TREE>(x);
        d[x & 1] = products4(fa[gi & 1][s / SN][m], fb[gi & 1][s % SN][m], nz);
        asm volatile("" : "+v"(d[x & 1]));
        const uint32_t y = (x + 4 * NT - 1) % (4 * NT);
        sums.add(acc, mtile_s<NT, TREE>(y), 4 * ((x ? gi : gi + 1) & 1) + mtile_k<NT, TREE>(y),
                 d[(x + 1) & 1]);
      }
    }
    if (ci + 1 < nc) store((ci + 1) & 1, nxt);
  };
  // chunk ci is computed while chunk ci + PF is loaded
  for (uint32_t ci = 0; ci < nc; ci += PF) {
    chunk(ci, stage[0], stage[PF - 1]);
    if (PF == 2 && ci + 1 < nc) chunk(ci + 1, stage[1 % PF], stage[0]);
  }
  sums.add(acc, NT - 1, 7, d[1]);
  // epilogue: lane l holds outputs m .. m+3 of X row n
#pragma unroll
  for (uint32_t i = 0; i < SMH; ++i)
#pragma unroll
    for (uint32_t j = 0; j < SN; ++j)
      mgemm_store<DUAL>(a, g, m0 + 16 * (wm * SMH + i) + 4 * u, n0 + 16 * (wn * SN + j) + c16,
                        acc[i * SN + j], acc[((DUAL ? SMH : 0) + i) * SN + j]);
}

// (value, index) pick of a strict-> scan from index 0 (first maximum wins;
// a NaN wins only at index 0, handled by the caller).
struct Pick {
  float v;
  uint32_t i;  // UINT32_MAX: none
};
__device__ __forceinline__ Pick pick2(Pick a, Pick b) {
  if (b.i == UINT32_MAX) return a;
  if (a.i == UINT32_MAX) return b;
  if (b.v > a.v) return b;
  if (a.v > b.v) return a;
  return b.i < a.i ? b : a;
}
__device__ Pick pick_block(Pick x, Pick* scratch) {
  for (int off = 32; off > 0; off >>= 1) {
    Pick o;
    o.v = __shfl_xor(x.v, off, 64);
    o.i = __shfl_xor(x.i, off, 64);
    x = pick2(x, o);
  }
  const uint32_t wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if ((threadIdx.x & 63) == 0) scratch[wv] = x;
  __syncthreads();
  Pick r = scratch[0];
  for (uint32_t i = 1; i < nw; ++i) r = pick2(r, scratch[i]);
  __syncthreads();
  return r;
}

__global__ void k_embed_rows(const float* __restrict__ E, RowsDesc rows, uint32_t H,
                             uint32_t vocab, float* h, uint32_t* err) {
  const uint32_t r = blockIdx.x;
  uint32_t tok = rows.tok[r];
  if (tok >= vocab) {
    if (threadIdx.x == 0) atomicOr(err, 1u);
    tok = 0;
  }
  const float* src = E + (size_t)tok * H;
  for (uint32_t i = threadIdx.x; i < H; i += blockDim.x) h[(size_t)r * H + i] = src[i];
}

// RoPE rotate-half (main.rs:285-307): o1 = x1*c + (-x2)*s, o2 = x2*c + x1*s.
__global__ __launch_bounds__(256) void k_rope_store_rows(float* q, float* k, const float* v,
                                                         const float* __restrict__ cs,
                                                         RowsDesc rows, uint32_t nh,
                                                         uint32_t nkv, uint32_t hd,
                                                         uint32_t max_pos, float* kc, float* vc,
                                                         uint64_t seq_stride) {
  const uint32_t r = blockIdx.x, pos = rows.pos[r], half = hd / 2;
  const size_t sb = (size_t)rows.seq[r] * seq_stride;
  float* qr = q + (size_t)r * nh * hd;
  float* kr = k + (size_t)r * nkv * hd;
  const float* vr = v + (size_t)r * nkv * hd;
  const float* c = cs + (size_t)pos * half * 2;
  const uint32_t total = (nh + nkv) * half;
  for (uint32_t idx = threadIdx.x; idx < total; idx += blockDim.x) {
    const uint32_t head = idx / half, i = idx - head * half;
    float* hv = head < nh ? qr + (size_t)head * hd : kr + (size_t)(head - nh) * hd;
    const float cv = c[2 * i], sv = c[2 * i + 1];
    const float x1 = hv[i], x2 = hv[i + half];
    float t1 = x1 * cv;
    float nx2 = -x2;
    float t2 = nx2 * sv;
    float t3 = x2 * cv;
    float t4 = x1 * sv;
    const float o1 = t1 + t2, o2 = t3 + t4;
    hv[i] = o1;
    hv[i + half] = o2;
    if (head >= nh) {
      const size_t base = (size_t)(head - nh) * hd;
      kc[sb + (base + i) * max_pos + pos] = o1;
      kc[sb + (base + i + half) * max_pos + pos] = o2;
    }
  }
  for (uint32_t idx = threadIdx.x; idx < nkv * hd; idx += blockDim.x)
    vc[sb + (size_t)idx * max_pos + pos] = vr[idx];
}

// The same for a tile of up to 16 rows at consecutive positions and one KV
// head: its query heads in place, k and v through LDS so that a cache row
// takes 16 consecutive positions per store (64 bytes) where the per-row kernel
// stores 4 (4096 rows of 16 + 8 heads of 128: 32 us, 118 us with a workgroup
// per row).
// Head_dim 64 or 128.
__global__ __launch_bounds__(256) void k_rope_store_tiles(
    float* q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ cs, const AttTile* __restrict__ tiles, uint32_t nh, uint32_t nkv,
    uint32_t hd, uint32_t max_pos, float* kc, float* vc, uint64_t seq_stride) {
  __shared__ float kt[128 * 17], vt[128 * 17];
  const AttTile tl = tiles[blockIdx.x];
  const uint32_t kvh = blockIdx.y, group = nh / nkv, half = hd / 2, h4 = half / 4, t = threadIdx.x;
  const v4* cs4 = reinterpret_cast<const v4*>(cs + (size_t)tl.p0 * hd);
  for (uint32_t i = t; i < tl.nr * (group + 1) * h4; i += 256) {
    const uint32_t ri = i / ((group + 1) * h4), x = i - ri * (group + 1) * h4;
    const uint32_t h = x / h4, i4 = x - h * h4;
    const size_t row = tl.row0 + ri;
    float* qr = q + (row * nh + kvh * group + h) * hd;
    const float* src = h < group ? qr : k + (row * nkv + kvh) * hd;
    const v4 x1 = reinterpret_cast<const v4*>(src)[i4];
    const v4 x2 = reinterpret_cast<const v4*>(src + half)[i4];
    const v4 ca = cs4[(size_t)ri * (half / 2) + 2 * i4], cb = cs4[(size_t)ri * (half / 2) + 2 * i4 + 1];
    const float c[4] = {ca.x, ca.z, cb.x, cb.z}, sn[4] = {ca.y, ca.w, cb.y, cb.w};
    v4 o1, o2;
#pragma unroll
    for (uint32_t e = 0; e < 4; ++e) {
      const float t1 = x1[e] * c[e];
      const float nx2 = -x2[e];
      const float t2 = nx2 * sn[e];
      const float t3 = x2[e] * c[e];
      const float t4 = x1[e] * sn[e];
      o1[e] = t1 + t2;
      o2[e] = t3 + t4;
    }
    if (h < group) {
      reinterpret_cast<v4*>(qr)[i4] = o1;
      reinterpret_cast<v4*>(qr + half)[i4] = o2;
    } else {
#pragma unroll
      for (uint32_t e = 0; e < 4; ++e) {
        kt[(4 * i4 + e) * 17 + ri] = o1[e];
        kt[(half + 4 * i4 + e) * 17 + ri] = o2[e];
      }
    }
  }
  for (uint32_t i = t; i < tl.nr * hd; i += 256) {
    const uint32_t ri = i / hd, d = i - ri * hd;
    vt[d * 17 + ri] = v[((size_t)(tl.row0 + ri) * nkv + kvh) * hd + d];
  }
  __syncthreads();
  const size_t base = (size_t)tl.seq * seq_stride + (size_t)kvh * hd * max_pos + tl.p0;
  const uint32_t ri = t & 15;
  if (ri < tl.nr)
    for (uint32_t d = t >> 4; d < hd; d += 16) {
      kc[base + (size_t)d * max_pos + ri] = kt[d * 17 + ri];
      vc[base + (size_t)d * max_pos + ri] = vt[d * 17 + ri];
    }
}

// One workgroup per (row, HPW query heads that share one KV head): per head
// scores_j = dot(q, k_j) * scale (dot_seq, or dot_tree), softmax (first-wins
// max, pinned exp, strict or tree denominator, true divide), then
// out_d = fold_j (p_j * v_j[d]) in position order
// (code/cis2-fp/src/main.rs:429-467; math.rs:425-465).  The heads of a
// workgroup read each K and V element once: a column's K values are loaded
// once for all HPW score chains, and the V rows of the HPW * hd output
// chains come from the same addresses.
// LDS: q [HPW][hd4], scores [HPW][ls], tree partials [HPW][nbs], with
// hd4 = hd rounded up to 4 and ls = max_len rounded up to 4.
template <uint32_t HPW>
__global__ __launch_bounds__(kAttT) void k_attention_rows(const float* __restrict__ q,
                                                        const float* __restrict__ kc,
                                                        const float* __restrict__ vc,
                                                        RowsDesc rows, uint32_t nh, uint32_t nkv,
                                                        uint32_t hd, uint32_t max_pos,
                                                        uint64_t seq_stride, float scale,
                                                        float* out, uint32_t tree, uint32_t ls) {
  extern __shared__ v4 sh4[];  // 16-byte aligned: q and scores are read 16 bytes at a time
  float* sh = reinterpret_cast<float*>(sh4);
  __shared__ Pick red[kAttT / 64];
  __shared__ float s_den[HPW];
  const uint32_t r = blockIdx.x, qh0 = blockIdx.y * HPW;  // rows on x: up to 2^31 of them
  const uint32_t group = nh / nkv, kvh = qh0 / group, pos = rows.pos[r], len = pos + 1;
  const uint32_t hd4 = (hd + 3) & ~3u, nbs = (ls + 31) / 32, t = threadIdx.x;
  const size_t sb = (size_t)rows.seq[r] * seq_stride;
  float* sq = sh;
  float* ssb = sh + HPW * hd4;
  float* partb = ssb + HPW * ls;
  const float* qv = q + (size_t)r * nh * hd + (size_t)qh0 * hd;
  for (uint32_t i = t; i < HPW * hd; i += blockDim.x) {
    const uint32_t h = i / hd, d = i - h * hd;
    sq[h * hd4 + d] = qv[i];
  }
  __syncthreads();
  const float* kb = kc + sb + (size_t)kvh * hd * max_pos;
  for (uint32_t j = t; j < len; j += blockDim.x) {
    float acc[HPW];
#pragma unroll
    for (uint32_t h = 0; h < HPW; ++h) acc[h] = 0.0f;
    if (tree) {
      for (uint32_t d0 = 0; d0 < hd; d0 += 32) {
        float kv[32];
#pragma unroll
        for (uint32_t i = 0; i < 32; ++i) kv[i] = d0 + i < hd ? kb[(size_t)(d0 + i) * max_pos + j] : 0.0f;
#pragma unroll
        for (uint32_t h = 0; h < HPW; ++h) {
          float l[32];
#pragma unroll
          for (uint32_t i = 0; i < 32; ++i) l[i] = d0 + i < hd ? sq[h * hd4 + d0 + i] * kv[i] : 0.0f;
          acc[h] = acc[h] + tree32(l);
        }
      }
    } else {
      // the column's loads go out 64 at a time, then the heads' chain steps
      // over them, interleaved
      uint32_t d0 = 0;
      for (; d0 + 64 <= hd; d0 += 64) {
        float kv[64];
#pragma unroll
        for (uint32_t i = 0; i < 64; ++i) kv[i] = kb[(size_t)(d0 + i) * max_pos + j];
#pragma unroll
        for (uint32_t i = 0; i < 64; ++i) {
#pragma unroll
          for (uint32_t h = 0; h < HPW; ++h) {
            const float p = sq[h * hd4 + d0 + i] * kv[i];
            acc[h] = acc[h] + p;
          }
        }
      }
      for (; d0 < hd; ++d0) {
        const float kv = kb[(size_t)d0 * max_pos + j];
#pragma unroll
        for (uint32_t h = 0; h < HPW; ++h) {
          const float p = sq[h * hd4 + d0] * kv;
          acc[h] = acc[h] + p;
        }
      }
    }
#pragma unroll
    for (uint32_t h = 0; h < HPW; ++h) ssb[h * ls + j] = acc[h] * scale;
  }
  __syncthreads();
  // per head: first-wins maximum (NaN at 0 wins), then exp(s - max)
  for (uint32_t h = 0; h < HPW; ++h) {
    float* ss = ssb + h * ls;
    Pick best = {0.0f, UINT32_MAX};
    for (uint32_t j = t; j < len; j += blockDim.x) {
      const float v = ss[j];
      if (v == v) best = pick2(best, Pick{v, j});
    }
    best = pick_block(best, red);
    const float mx = (ss[0] != ss[0]) ? ss[0] : best.v;
    for (uint32_t j = t; j < len; j += blockDim.x) {
      const float dlt = ss[j] - mx;
      ss[j] = exp_pinned(dlt);
    }
  }
  __syncthreads();
  const uint32_t nb = (len + 31) / 32;
  if (tree) {
    for (uint32_t i = t; i < HPW * nb; i += blockDim.x) {
      const uint32_t h = i / nb, tb = i - h * nb;
      const float* ss = ssb + h * ls;
      float l[32];
#pragma unroll
      for (uint32_t k = 0; k < 32; ++k) l[k] = 32 * tb + k < len ? ss[32 * tb + k] : 0.0f;
      partb[h * nbs + tb] = tree32(l);
    }
    __syncthreads();
  }
  // denominators: wave w sums heads w, w + 4, ...; every lane of the wave
  // runs the same chain
  for (uint32_t h = t >> 6; h < HPW; h += blockDim.x >> 6) {
    float acc = 0.0f;
    if (tree) {
      for (uint32_t tb = 0; tb < nb; ++tb) acc = acc + partb[h * nbs + tb];
    } else {
      // 16-byte reads (every lane the same address), 8 of them per batch
      const float* ss = ssb + h * ls;
      const v4* s4p = reinterpret_cast<const v4*>(ss);
      uint32_t j = 0;
      for (; j + 32 <= len; j += 32) {
        v4 e[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) e[u] = s4p[j / 4 + u];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) {
          acc = acc + e[u].x;
          acc = acc + e[u].y;
          acc = acc + e[u].z;
          acc = acc + e[u].w;
        }
      }
      for (; j < len; ++j) acc = acc + ss[j];
    }
    if ((t & 63) == 0) s_den[h] = acc;
  }
  __syncthreads();
  for (uint32_t i = t; i < HPW * len; i += blockDim.x) {
    const uint32_t h = i / len, j = i - h * len;
    const float pj = ssb[h * ls + j] / s_den[h];
    ssb[h * ls + j] = pj;
  }
  __syncthreads();
  const float* vb = vc + sb + (size_t)kvh * hd * max_pos;
  for (uint32_t i = t; i < HPW * hd; i += blockDim.x) {
    const uint32_t h = i / hd, d = i - h * hd;
    float* o = out + (size_t)r * nh * hd + (size_t)(qh0 + h) * hd;
    const float* ss = ssb + h * ls;
    // row d of V is contiguous: 16-byte loads, a batch of 64 positions in
    // flight while the previous batch's chain steps run
    const v4* vr4 = reinterpret_cast<const v4*>(vb + (size_t)d * max_pos);
    const v4* p4 = reinterpret_cast<const v4*>(ss);
    float acc = 0.0f;
    uint32_t j = 0;
    constexpr uint32_t VB = 16;
    v4 cur[VB], nxt[VB];
    const uint32_t full = len / (4 * VB);
    if (full > 0) {
#pragma unroll
      for (uint32_t u = 0; u < VB; ++u) cur[u] = vr4[u];
    }
    for (uint32_t bt = 0; bt < full; ++bt, j += 4 * VB) {
      if (bt + 1 < full) {
#pragma unroll
        for (uint32_t u = 0; u < VB; ++u) nxt[u] = vr4[(j + 4 * VB) / 4 + u];
      }
#pragma unroll
      for (uint32_t u = 0; u < VB; ++u) {
        const v4 pp = p4[j / 4 + u];
        float p;
        p = pp.x * cur[u].x; acc = acc + p;
        p = pp.y * cur[u].y; acc = acc + p;
        p = pp.z * cur[u].z; acc = acc + p;
        p = pp.w * cur[u].w; acc = acc + p;
      }
#pragma unroll
      for (uint32_t u = 0; u < VB; ++u) cur[u] = nxt[u];
    }
    const float* vr = vb + (size_t)d * max_pos;
    for (; j < len; ++j) {
      const float p = ss[j] * vr[j];
      acc = acc + p;
    }
    o[d] = acc;
  }
}

// Strict sums over LDS with a ring of 16-byte reads in flight; the caller
// keeps D groups of readable LDS after the last one, so the ring is refilled
// unconditionally at fixed offsets (the extra reads are never used) and the
// last partial round adds its groups under uniform tests.  n wave-uniform.
//   chain_lds_s:  acc + x[0] + x[1] + ... + x[n-1]
//   mix_lds_s:    acc + p[0]*v[0] + ... + p[n-1]*v[n-1]
// x, p and v 16-byte aligned.
template <uint32_t D>
__device__ __forceinline__ float chain_lds_s(const float* x, uint32_t n, float acc) {
  const v4* x4 = reinterpret_cast<const v4*>(x);
  const uint32_t ng = n / 4;
  v4 ring[D];
#pragma unroll
  for (uint32_t u = 0; u < D; ++u) ring[u] = x4[u];
  uint32_t g = 0;
  for (; g + D <= ng; g += D) {
#pragma unroll
    for (uint32_t u = 0; u < D; ++u) {
      const v4 r = ring[u];
      acc = acc + r.x;
      acc = acc + r.y;
      acc = acc + r.z;
      acc = acc + r.w;
      ring[u] = x4[g + u + D];
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (uint32_t u = 0; u + 1 < D; ++u) {
    if (g + u < ng) {
      const v4 r = ring[u];
      acc = acc + r.x;
      acc = acc + r.y;
      acc = acc + r.z;
      acc = acc + r.w;
    }
  }
  for (uint32_t j = 4 * ng; j < n; ++j) acc = acc + x[j];
  return acc;
}
template <uint32_t D>
__device__ __forceinline__ float mix_lds_s(const float* p, const float* v, uint32_t n, float acc) {
  const v4* p4 = reinterpret_cast<const v4*>(p);
  const v4* v4p = reinterpret_cast<const v4*>(v);
  const uint32_t ng = n / 4;
  v4 rp[D], rv[D];
#pragma unroll
  for (uint32_t u = 0; u < D; ++u) {
    rp[u] = p4[u];
    rv[u] = v4p[u];
  }
  auto step = [&](const v4& a, const v4& b) {
    float pr;
    pr = a.x * b.x; acc = acc + pr;
    pr = a.y * b.y; acc = acc + pr;
    pr = a.z * b.z; acc = acc + pr;
    pr = a.w * b.w; acc = acc + pr;
  };
  uint32_t g = 0;
  for (; g + D <= ng; g += D) {
#pragma unroll
    for (uint32_t u = 0; u < D; ++u) {
      step(rp[u], rv[u]);
      rp[u] = p4[g + u + D];
      rv[u] = v4p[g + u + D];
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (uint32_t u = 0; u + 1 < D; ++u)
    if (g + u < ng) step(rp[u], rv[u]);
  for (uint32_t j = 4 * ng; j < n; ++j) {
    const float pr = p[j] * v[j];
    acc = acc + pr;
  }
  return acc;
}
// The same strict sum from two register sets of 8 groups: the next set's
// reads go out before the current set's 32 adds (one wait per set); no read
// past the end.  Faster than the ring on chains of 100+ groups.
__device__ __forceinline__ float chain_lds_pp(const float* x, uint32_t n, float acc) {
  constexpr uint32_t U = 8;
  const v4* x4 = reinterpret_cast<const v4*>(x);
  const uint32_t ng = n / 4;
  auto add1 = [&](const v4 v) {
    acc = acc + v.x;
    acc = acc + v.y;
    acc = acc + v.z;
    acc = acc + v.w;
  };
  uint32_t g = 0;
  if (ng >= U) {
    v4 a[U], b[U];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) a[u] = x4[u];
    for (; g + 3 * U <= ng; g += 2 * U) {
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) b[u] = x4[g + U + u];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) add1(a[u]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) a[u] = x4[g + 2 * U + u];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) add1(b[u]);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (uint32_t u = 0; u < U; ++u)
      if (g + U + u < ng) b[u] = x4[g + U + u];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) add1(a[u]);
    g += U;
#pragma unroll
    for (uint32_t u = 0; u < U; ++u)
      if (g + u < ng) add1(b[u]);
    g = g + U < ng ? g + U : ng;
  }
  for (; g < ng; ++g) add1(x4[g]);
  for (uint32_t j = 4 * ng; j < n; ++j) acc = acc + x[j];
  return acc;
}
// Readable floats the decode-rows attention keeps after its LDS regions.
constexpr uint32_t kKvSlack = 64;

// acc + p[0] + ... + p[n-1], strictly left to right (16-byte LDS reads,
// eight of them per batch).
__device__ __forceinline__ float chain_lds(const float* p, uint32_t n, float acc) {
  const v4* p4 = reinterpret_cast<const v4*>(p);
  uint32_t j = 0;
  for (; j + 32 <= n; j += 32) {
    v4 e[8];
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u) e[u] = p4[j / 4 + u];
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u) {
      acc = acc + e[u].x;
      acc = acc + e[u].y;
      acc = acc + e[u].z;
      acc = acc + e[u].w;
    }
  }
  for (; j < n; ++j) acc = acc + p[j];
  return acc;
}

// ---------------------------------------------------------------------------
// Attention of decode rows (few rows, one per sequence): one workgroup of
// kKvT threads per (row, KV head) takes the HPW = nh / nkv query heads of
// that KV head, with the per-row kernel's arithmetic in the same order
// (scores d ascending, dot_seq or tree32 blocks, first-wins maximum, pinned
// exp, strict or tree denominator, true divide, V-mix j ascending;
// code/cis2-fp/src/main.rs:429-467, math.rs:425-465), so every output has
// the per-row kernel's bits.
//   scores:  a thread takes two adjacent positions per round (8-byte K
//            loads, 64 d per batch in flight), one chain per (position,
//            head);
//   V rows:  then copied into LDS with global_load_lds by every wave, in
//            chunks of C <= 256 positions over two buffers (row stride
//            C + 4 floats: lane d's 16-byte reads fall in distinct banks);
//            the softmax's barriers wait for LDS only, so the copies land
//            meanwhile; a buffer is refilled two chunks ahead while the
//            V-mix runs over the other;
//   softmax: the maximum with DPP, exp, the HPW denominators on HPW waves
//            at once (a ring of LDS reads), the divide;
//   V-mix:   HPW * HD / 64 waves, lane = d, each product formed with p_j
//            taken by DPP broadcast (row_newbcast) from a register holding
//            16 consecutive probabilities in every 16-lane row, the next 16
//            positions' reads in flight.
// LDS (floats): q [HPW][HD], scores [HPW][ls], tree partials [HPW][nbs]
// (rounded up to 4), V [2][HD][C + 4], kKvSlack readable floats (the read
// rings run up to 56 floats past a row's end).
// ---------------------------------------------------------------------------
constexpr uint32_t kKvT = 512;
typedef float v2 __attribute__((ext_vector_type(2)));
// RoPE inputs of the fused form: the rows' raw k and v ([n][nkv][hd]) and
// the cos/sin table ([max_pos][hd/2][2]).
struct KvFuse {
  const float* k;
  const float* v;
  const float* rope_cs;
  uint32_t nkv;
};

// acc + P_0 * v[0].x + P_1 * v[0].y + ... + P_15 * v[3].w in order (P_k:
// lane k of this lane's 16-lane row), each product rounded, then the add.
template <uint32_t K = 0>
__device__ __forceinline__ void mix16(float& acc, float P, const v4 (&v)[4]) {
  if constexpr (K < 16) {
    const v4 w = v[K / 4];
    const float x = K % 4 == 0 ? w.x : K % 4 == 1 ? w.y : K % 4 == 2 ? w.z : w.w;
    const float t = bcast16<K>(P) * x;
    acc = acc + t;
    mix16<K + 1>(acc, P, v);
  }
}
// The first rem (< 16) steps of mix16.
template <uint32_t K = 0>
__device__ __forceinline__ void mix16_part(float& acc, float P, const v4 (&v)[4], uint32_t rem) {
  if constexpr (K < 15) {
    if (K < rem) {
      const v4 w = v[K / 4];
      const float x = K % 4 == 0 ? w.x : K % 4 == 1 ? w.y : K % 4 == 2 ? w.z : w.w;
      const float t = bcast16<K>(P) * x;
      acc = acc + t;
      mix16_part<K + 1>(acc, P, v, rem);
    }
  }
}
// acc + p[0]*v[0] + ... + p[n-1]*v[n-1] in order; p and v in LDS, 16-byte
// aligned, 16 readable floats past n; two register sets, each block of 16
// positions read one block ahead.  n wave-uniform.
__device__ __forceinline__ float mix_dpp(const float* p, const float* v, uint32_t n, float acc) {
  const uint32_t k = threadIdx.x & 15, nb = n >> 4;
  const v4* v4p = reinterpret_cast<const v4*>(v);
  float PA = p[k], PB;
  v4 vA[4], vB[4];
#pragma unroll
  for (uint32_t u = 0; u < 4; ++u) vA[u] = v4p[u];
  uint32_t m = 0;
  for (; m + 2 <= nb; m += 2) {
    PB = p[16 * (m + 1) + k];
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) vB[u] = v4p[4 * (m + 1) + u];
    mix16(acc, PA, vA);
    PA = p[16 * (m + 2) + k];
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) vA[u] = v4p[4 * (m + 2) + u];
    mix16(acc, PB, vB);
  }
  if (m < nb) {  // one whole block left
    PB = p[16 * (m + 1) + k];
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) vB[u] = v4p[4 * (m + 1) + u];
    mix16(acc, PA, vA);
    PA = PB;
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) vA[u] = vB[u];
  }
  mix16_part(acc, PA, vA, n - 16 * nb);
  return acc;
}

template <uint32_t HPW, uint32_t HD, bool FUSE>
__global__ __launch_bounds__(kKvT) void k_attention_kv(const float* __restrict__ q,
                                                     float* kc, float* vc, RowsDesc rows,
                                                     uint32_t nh, uint32_t max_pos,
                                                     uint64_t seq_stride, float scale,
                                                     float* out, uint32_t tree, uint32_t ls,
                                                     uint32_t C, KvFuse fz) {
  constexpr uint32_t NW = kKvT / 64, WPH = HD / 64, CW = HPW * WPH;
  static_assert(HD % 64 == 0 && CW <= NW, "chain waves");
  extern __shared__ v4 sh4[];
  float* sh = reinterpret_cast<float*>(sh4);
  __shared__ float s_red[NW][HPW];
  __shared__ float s_den[HPW];
  const uint32_t r = blockIdx.x, kvh = blockIdx.y, qh0 = kvh * HPW, t = threadIdx.x;
  const uint32_t wv = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
  const uint32_t pos = rows.pos[r], len = pos + 1, S = C + 4;
  // FUSE: position pos comes from this launch (its K and V from LDS), the
  // caches serve positions 0 .. pos-1
  const uint32_t lc = FUSE ? pos : len;
  const uint32_t nbs = (ls + 31) / 32, len4 = (lc + 3) & ~3u;
  const size_t sb = (size_t)rows.seq[r] * seq_stride;
  float* kb = kc + sb + (size_t)kvh * HD * max_pos;
  float* vb = vc + sb + (size_t)kvh * HD * max_pos;
  float* sq = sh;
  float* kself = sq + HPW * HD;  // FUSE: this position's rotated k and its v
  float* vself = kself + HD;
  float* ssb = vself + HD;
  float* partb = ssb + HPW * ls;
  float* VL = partb + ((HPW * nbs + 3) & ~3u);
  const uint32_t nch = (lc + C - 1) / C;
  // chunk ch of V row d into buffer ch % 2: one wave instruction (C <= 256
  // positions), lanes past the chunk or the row's end idle
  auto stage_row = [&](uint32_t ch, uint32_t d) {
    const uint32_t o = lane * 4, j = ch * C + o;
    if (o < C && j < len4)
      lds_load16(reinterpret_cast<const v4*>(vb + (size_t)d * max_pos + j),
                 reinterpret_cast<v4*>(VL + (size_t)(ch & 1) * HD * S + (size_t)d * S));
  };
  const float* qv = q + (size_t)r * nh * HD + (size_t)qh0 * HD;
  if constexpr (FUSE) {
    // RoPE at pos of the HPW query heads and of KV head kvh, in
    // k_rope_store_rows's order (o1 = x1*c + (-x2)*s, o2 = x2*c + x1*s); the
    // rotated k and the raw v also into the caches at pos
    constexpr uint32_t half = HD / 2;
    const float* cs = fz.rope_cs + (size_t)pos * half * 2;
    const float* kin = fz.k + (size_t)r * fz.nkv * HD + (size_t)kvh * HD;
    const float* vin = fz.v + (size_t)r * fz.nkv * HD + (size_t)kvh * HD;
    for (uint32_t i = t; i < (HPW + 1) * half; i += kKvT) {
      const uint32_t h = i / half, ii = i - h * half;
      const float* src = h < HPW ? qv + (size_t)h * HD : kin;
      const float cv = cs[2 * ii], sv = cs[2 * ii + 1];
      const float x1 = src[ii], x2 = src[ii + half];
      const float t1 = x1 * cv;
      const float nx2 = -x2;
      const float t2 = nx2 * sv;
      const float t3 = x2 * cv;
      const float t4 = x1 * sv;
      const float o1 = t1 + t2, o2 = t3 + t4;
      if (h < HPW) {
        sq[h * HD + ii] = o1;
        sq[h * HD + ii + half] = o2;
      } else {
        kself[ii] = o1;
        kself[ii + half] = o2;
        kb[(size_t)ii * max_pos + pos] = o1;
        kb[(size_t)(ii + half) * max_pos + pos] = o2;
      }
    }
    for (uint32_t d = t; d < HD; d += kKvT) {
      const float vv = vin[d];
      vself[d] = vv;
      vb[(size_t)d * max_pos + pos] = vv;
    }
  } else {
    for (uint32_t i = t; i < HPW * HD; i += kKvT) sq[i] = qv[i];
  }
  lds_barrier();
  // FUSE: position pos's scores from the rotated k in LDS, one lane per head
  if (FUSE && t < HPW) {
    float acc = 0.0f;
    if (tree) {
#pragma unroll
      for (uint32_t d0 = 0; d0 < HD; d0 += 32) {
        float l[32];
#pragma unroll
        for (uint32_t i = 0; i < 32; ++i) l[i] = sq[t * HD + d0 + i] * kself[d0 + i];
        acc = acc + tree32(l);
      }
    } else {
      for (uint32_t d = 0; d < HD; ++d) {
        const float pr = sq[t * HD + d] * kself[d];
        acc = acc + pr;
      }
    }
    ssb[t * ls + pos] = acc * scale;
  }
  // scores: thread t takes positions jp, jp + 1 (jp = 2 * (t + k * kKvT);
  // len4 <= max_pos, so a pair below len4 stays in the row; a pair's
  // second position past the cached ones is computed and dropped)
  for (uint32_t jp = 2 * t; jp < lc; jp += 2 * kKvT) {
    float acc[2][HPW];
#pragma unroll
    for (uint32_t p = 0; p < 2; ++p)
#pragma unroll
      for (uint32_t h = 0; h < HPW; ++h) acc[p][h] = 0.0f;
#pragma unroll
    for (uint32_t d0 = 0; d0 < HD; d0 += 64) {
      v2 kv[64];
#pragma unroll
      for (uint32_t i = 0; i < 64; ++i)
        kv[i] = *reinterpret_cast<const v2*>(kb + (size_t)(d0 + i) * max_pos + jp);
      if (tree) {
#pragma unroll
        for (uint32_t b0 = 0; b0 < 64; b0 += 32)
#pragma unroll
          for (uint32_t p = 0; p < 2; ++p)
#pragma unroll
            for (uint32_t h = 0; h < HPW; ++h) {
              float l[32];
#pragma unroll
              for (uint32_t i = 0; i < 32; ++i)
                l[i] = sq[h * HD + d0 + b0 + i] * (p ? kv[b0 + i].y : kv[b0 + i].x);
              acc[p][h] = acc[p][h] + tree32(l);
            }
      } else {
#pragma unroll
        for (uint32_t i = 0; i < 64; ++i)
#pragma unroll
          for (uint32_t h = 0; h < HPW; ++h) {
            const float qd = sq[h * HD + d0 + i];
            float pr;
            pr = qd * kv[i].x; acc[0][h] = acc[0][h] + pr;
            pr = qd * kv[i].y; acc[1][h] = acc[1][h] + pr;
          }
      }
    }
#pragma unroll
    for (uint32_t p = 0; p < 2; ++p)
      if (jp + p < lc)
#pragma unroll
        for (uint32_t h = 0; h < HPW; ++h) ssb[h * ls + jp + p] = acc[p][h] * scale;
  }
  // the V copies of chunks 0 and 1, spread over the waves
  for (uint32_t d = wv; d < HD; d += NW) {
    stage_row(0, d);
    if (nch > 1) stage_row(1, d);
  }
  lds_barrier();
  // maximum per head: the largest non-NaN score (its value does not depend
  // on which of equal scores is first: exp(s - (+0)) = exp(s - (-0))), a NaN
  // score at 0 wins
  {
    float m[HPW];
#pragma unroll
    for (uint32_t h = 0; h < HPW; ++h) m[h] = -__builtin_huge_valf();
    for (uint32_t j = t; j < len; j += kKvT)
#pragma unroll
      for (uint32_t h = 0; h < HPW; ++h) {
        const float v = ssb[h * ls + j];
        m[h] = v > m[h] ? v : m[h];
      }
#pragma unroll
    for (uint32_t h = 0; h < HPW; ++h) {
      m[h] = wave_max(m[h]);
      if (lane == 0) s_red[wv][h] = m[h];
    }
    lds_barrier();
#pragma unroll
    for (uint32_t h = 0; h < HPW; ++h) {
      float mx = s_red[0][h];
#pragma unroll
      for (uint32_t w = 1; w < NW; ++w) mx = s_red[w][h] > mx ? s_red[w][h] : mx;
      const float s0 = ssb[h * ls];
      m[h] = s0 != s0 ? s0 : mx;
    }
    for (uint32_t j = t; j < len; j += kKvT)
#pragma unroll
      for (uint32_t h = 0; h < HPW; ++h) {
        const float dlt = ssb[h * ls + j] - m[h];
        ssb[h * ls + j] = exp_pinned(dlt);
      }
  }
  lds_barrier();
  const uint32_t nb = (len + 31) / 32;
  if (tree) {
    for (uint32_t i = t; i < HPW * nb; i += kKvT) {
      const uint32_t h = i / nb, tb = i - h * nb;
      const float* ss = ssb + h * ls;
      float l[32];
#pragma unroll
      for (uint32_t k = 0; k < 32; ++k) l[k] = 32 * tb + k < len ? ss[32 * tb + k] : 0.0f;
      partb[h * nbs + tb] = tree32(l);
    }
    lds_barrier();
  }
  // denominators: wave h sums head h (every lane the same chain)
  if (wv < HPW) {
    const float acc = tree ? chain_lds_s<14>(partb + wv * nbs, nb, 0.0f)
                           : chain_lds_pp(ssb + wv * ls, len, 0.0f);
    if (lane == 0) s_den[wv] = acc;
  }
  lds_barrier();
#pragma unroll
  for (uint32_t h = 0; h < HPW; ++h) {
    const float den = s_den[h];
    for (uint32_t j = t; j < len; j += kKvT) {
      const float pj = ssb[h * ls + j] / den;
      ssb[h * ls + j] = pj;
    }
  }
  // V-mix over the staged chunks
  const uint32_t h = wv / WPH, d = (wv - h * WPH) * 64 + lane;
  const float* ps = ssb + (size_t)(wv < CW ? h : 0) * ls;
  float acc = 0.0f;
  for (uint32_t ch = 0; ch < nch; ++ch) {
    // chunk ch's copies (issued after the scores or two chunks back) have
    // landed and every wave is done with chunk ch - 1, whose buffer takes
    // chunk ch + 1 (copied by the waves without a chain)
    wait_vm0();
    __syncthreads();
    if (wv >= CW && ch > 0 && ch + 1 < nch)
      for (uint32_t dd = wv - CW; dd < HD; dd += NW - CW) stage_row(ch + 1, dd);
    if (wv < CW) {
      const uint32_t jc = ch * C;
      acc = mix_dpp(ps + jc, VL + (size_t)(ch & 1) * HD * S + (size_t)d * S,
                    std::min(C, lc - jc), acc);
    }
  }
  wait_vm0();  // no copy still in flight when the workgroup ends (lc = 0)
  if (FUSE && nch == 0) __syncthreads();  // the divide's p_pos, with no chunk loop
  if (FUSE && wv < CW) {
    const float pr = ps[pos] * vself[d];
    acc = acc + pr;
  }
  if (wv < CW) out[(size_t)r * nh * HD + (size_t)(qh0 + h) * HD + d] = acc;
}

// ---------------------------------------------------------------------------
// Attention of many decode rows (sequential order): one wave per (row, query
// head), no barrier, with the per-row kernel's arithmetic in the same order.
// Lane j takes position j of every 64 (the column's 64 K loads in flight, q
// by LDS broadcast); maximum by shuffles; every lane runs the denominator
// chain; lane d mixes output dim d from its contiguous V row.  FUSE: RoPE of
// the row's q head and k head, whose first query head stores k and v at pos,
// as in k_attention_kv.
// What bounds it: the cache lines of short K and V rows (and one 4-byte store
// per row of either); thousands of waves hide each other's chains and load
// latency, where a workgroup per pair spent its time in barriers with most
// threads idle.
// LDS per wave (floats): q [HD], k [HD], v [HD], scores [ls].
// ---------------------------------------------------------------------------
// LDS written by other lanes of this wave is readable after it.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_s_waitcnt(0xC07F);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
}

template <uint32_t HD, bool FUSE>
__global__ __launch_bounds__(256) void k_attention_wave(
    const float* __restrict__ q, float* kc, float* vc, RowsDesc rows, uint32_t nh, uint32_t group,
    uint32_t max_pos, uint64_t seq_stride, float scale, float* out, uint32_t ls, KvFuse fz) {
  extern __shared__ v4 sh4[];
  constexpr uint32_t half = HD / 2;
  const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const uint32_t item = blockIdx.x * 4 + wv;
  if (item >= rows.n * nh) return;
  const uint32_t r = item / nh, h = item - r * nh, kvh = h / group;
  const uint32_t pos = rows.pos[r], len = pos + 1, lc = FUSE ? pos : len;
  float* sq = reinterpret_cast<float*>(sh4) + wv * (3 * HD + ls);
  float *kself = sq + HD, *vself = kself + HD, *ss = vself + HD;
  const size_t sb = (size_t)rows.seq[r] * seq_stride + (size_t)kvh * HD * max_pos;
  float* kb = kc + sb;
  float* vb = vc + sb;
  const float* qv = q + ((size_t)r * nh + h) * HD;
  if constexpr (FUSE) {
    const float* cs = fz.rope_cs + (size_t)pos * half * 2;
    const float* kin = fz.k + ((size_t)r * fz.nkv + kvh) * HD;
    const float* vin = fz.v + ((size_t)r * fz.nkv + kvh) * HD;
    const bool first = h == kvh * group;
    if (lane < half) {
      const float cv = cs[2 * lane], sv = cs[2 * lane + 1];
      auto rotate = [&](const float* src, float& o1, float& o2) {
        const float x1 = src[lane], x2 = src[lane + half];
        const float t1 = x1 * cv;
        const float nx2 = -x2;
        const float t2 = nx2 * sv;
        const float t3 = x2 * cv;
        const float t4 = x1 * sv;
        o1 = t1 + t2;
        o2 = t3 + t4;
      };
      float o1, o2;
      rotate(qv, o1, o2);
      sq[lane] = o1;
      sq[lane + half] = o2;
      rotate(kin, o1, o2);
      kself[lane] = o1;
      kself[lane + half] = o2;
      if (first) {
        kb[(size_t)lane * max_pos + pos] = o1;
        kb[(size_t)(lane + half) * max_pos + pos] = o2;
      }
    }
#pragma unroll
    for (uint32_t d = 0; d < HD; d += 64) {
      const float vv = vin[d + lane];
      vself[d + lane] = vv;
      if (first) vb[(size_t)(d + lane) * max_pos + pos] = vv;
    }
  } else {
#pragma unroll
    for (uint32_t d = 0; d < HD; d += 64) sq[d + lane] = qv[d + lane];
  }
  wave_lds_sync();
  float m = -__builtin_inff();
  for (uint32_t j0 = 0; j0 < len; j0 += 64) {
    const uint32_t j = j0 + lane, jl = j < lc ? j : 0;
    const bool self = FUSE && pos < j0 + 64;  // the round that holds pos
    float acc = 0.0f;
#pragma unroll
    for (uint32_t d0 = 0; d0 < HD; d0 += 64) {
      float kv[64];
#pragma unroll
      for (uint32_t i = 0; i < 64; ++i) kv[i] = kb[(size_t)(d0 + i) * max_pos + jl];
      if (self) {
#pragma unroll
        for (uint32_t i = 0; i < 64; i += 4) {
          const v4 k4 = *reinterpret_cast<const v4*>(kself + d0 + i);
#pragma unroll
          for (uint32_t e = 0; e < 4; ++e) kv[i + e] = j == pos ? k4[e] : kv[i + e];
        }
      }
#pragma unroll
      for (uint32_t i = 0; i < 64; i += 4) {
        const v4 q4 = *reinterpret_cast<const v4*>(sq + d0 + i);
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e) {
          const float p = q4[e] * kv[i + e];
          acc = acc + p;
        }
      }
    }
    const float sc = acc * scale;
    if (j < len) {
      ss[j] = sc;
      m = sc > m ? sc : m;
    }
  }
#pragma unroll
  for (uint32_t off = 32; off > 0; off >>= 1) {
    const float o = __shfl_xor(m, off, 64);
    m = o > m ? o : m;
  }
  wave_lds_sync();
  // the largest non-NaN score; a NaN at position 0 wins with its own bits
  const float s0 = ss[0];
  const float mx = s0 != s0 ? s0 : m;
  wave_lds_sync();
  for (uint32_t j = lane; j < len; j += 64) {
    const float dlt = ss[j] - mx;
    ss[j] = exp_pinned(dlt);
  }
  wave_lds_sync();
  const float den = chain_lds(ss, len, 0.0f);
  wave_lds_sync();
  for (uint32_t j = lane; j < len; j += 64) {
    const float pj = ss[j] / den;
    ss[j] = pj;
  }
  wave_lds_sync();
#pragma unroll
  for (uint32_t x = 0; x < HD / 64; ++x) {
    const uint32_t d = 64 * x + lane;
    const float* vr = vb + (size_t)d * max_pos;
    float acc = 0.0f;
    uint32_t j = 0;
    for (; j + 16 <= lc; j += 16) {
      v4 v[4], p4[4];
#pragma unroll
      for (uint32_t e = 0; e < 4; ++e) v[e] = *reinterpret_cast<const v4*>(vr + j + 4 * e);
#pragma unroll
      for (uint32_t e = 0; e < 4; ++e) p4[e] = *reinterpret_cast<const v4*>(ss + j + 4 * e);
#pragma unroll
      for (uint32_t e = 0; e < 4; ++e)
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) {
          const float p = p4[e][c] * v[e][c];
          acc = acc + p;
        }
    }
    for (; j < lc; j += 4) {  // up to 3 positions past lc are read, not added
      const v4 v = *reinterpret_cast<const v4*>(vr + j);
#pragma unroll
      for (uint32_t c = 0; c < 4; ++c)
        if (j + c < lc) {
          const float p = ss[j + c] * v[c];
          acc = acc + p;
        }
    }
    if (FUSE) {
      const float p = ss[pos] * vself[d];
      acc = acc + p;
    }
    out[((size_t)r * nh + h) * HD + d] = acc;
  }
}

// ---------------------------------------------------------------------------
// Attention of prefill rows in tiles.  A tile is up to kAttQT rows of one
// sequence at consecutive positions p0 .. p0+nr-1 (built on the host); a work
// item is one tile and HPT query heads of one KV head, P = kAttQT * HPT
// (row, head) pairs (pair a = head h * 16 + row i).  Each pair's arithmetic
// is the per-row kernel's, in the same order, with the products of both
// contractions formed by the matrix cores (products4, above) and the chains'
// adds by the vector units:
//   scores  s_j = dot_seq(q, k_j) * scale, d ascending: A is 16 pairs of one
//           head, B 16 positions; a wave takes 64 positions at a time, and a
//           16-byte load per lane of 4 rows of K is the B operand of four
//           position tiles, straight from global memory, used by all HPT
//           heads; the scores go to a scratch row per pair, the maximum (NaN
//           at position 0 wins) is kept on the way;
//   softmax the denominator as one strict chain per pair: waves 1..3 copy
//           stages of TE scores into LDS one stage ahead and turn them into
//           exp(s - max) in place (written back for the V-mix) while lanes
//           a < P of wave 0 continue their chains;
//   V-mix   out_d = fold_j (p_j * v_j[d]), j ascending, p_j = e_j / den: A is
//           16 pairs, B 16 dims; the p tiles of TP positions are divided one
//           tile ahead into LDS in operand order, V goes from global memory
//           to registers (four groups of 16 positions ahead) and is
//           transposed between lanes there (permlane swaps).  In the groups
//           that reach past the tile's first row's length every add is
//           selected by j < the row's length.
// TREE: the scores' products are added in blocks of 32 d and the denominators
// in blocks of 32 positions (tree32); the V-mix is the same fold.
// What bounds it: the vector and matrix units, at the GEMM's 64 cycles per
// 1024 chain steps, and the exps (about a fifth of a head_dim-64 step).
// 4096 rows of 16 heads of 128: 1.89 ms per layer (18 T chain steps/s),
// 4.32 ms with operands read from LDS and multiplied by the vector units;
// 64 ragged prompts of 16 .. 512 rows, 9 heads of 64: 0.31 ms against 1.37.
// Tree order, us per layer with k_attention_rows | with this: one prompt of 544
// rows 290 | 213 (9 heads of 64), 948 | 662 (16 of 128); 200 rows 143 | 135,
// 404 | 331.
// Workgroups walk the items with a fixed stride, the longest tiles first and
// every other round in reverse order, each with one scratch slot, so the
// scratch stays a few hundred MB whatever the row count; the stride is a
// multiple of 8 and the heads of a tile are neighbours, so the XCD that a
// workgroup runs on meets one KV head of eight and keeps it in its L2.
// LDS: q in operand order, then the phase regions (e stages 2 x [P][TE+4]; p
// tiles 2 x [P][TP]), the wave maxima, the pairs' maximum and denominator.
// ---------------------------------------------------------------------------
constexpr uint32_t kAttQT = kAttTileRows;  // rows per attention tile
constexpr uint32_t kAttTE = 64;            // positions per softmax stage
static_assert(kAttQT == 16, "a tile's rows are one operand's rows");

template <uint32_t HPT>
struct AttTileCfg {
  static constexpr uint32_t P = kAttQT * HPT;
  static constexpr uint32_t ES = kAttTE + 4;                             // e stage row stride
  static constexpr uint32_t TP = HPT >= 3 ? 64 : (HPT == 2 ? 128 : 256);  // positions per p tile
  static constexpr size_t region1 = 2 * (size_t)P * ES, region2 = 2 * (size_t)P * TP;
  static constexpr size_t region = region1 > region2 ? region1 : region2;
  static constexpr size_t floats(uint32_t hd) { return (size_t)P * hd + region + 6 * P; }
  static_assert(P * TP / 16 <= 256, "one p piece per thread");
  static_assert(P <= 64, "one denominator lane per pair in wave 0");
};

// Lane l's four values x = M[l / 16 row][4 (l / 16) + c] become
// M[row][4 c + l / 16]: a 4 x 4 transpose between the 16-lane groups.
__device__ __forceinline__ void transpose4(v4& x) {
  typedef uint32_t u2 __attribute__((ext_vector_type(2)));
  uint32_t r[4];
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) r[i] = __float_as_uint(x[i]);
  u2 a = __builtin_amdgcn_permlane16_swap(r[0], r[1], false, false);
  u2 b = __builtin_amdgcn_permlane16_swap(r[2], r[3], false, false);
  u2 c = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false);
  u2 d = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
  x = v4{__uint_as_float(c[0]), __uint_as_float(d[0]), __uint_as_float(c[1]),
         __uint_as_float(d[1])};
}

template <uint32_t HPT, uint32_t HD, bool TREE>
__global__ __launch_bounds__(256, 2) void k_attention_tiles(
    const float* __restrict__ q, const float* __restrict__ kc, const float* __restrict__ vc,
    const AttTile* __restrict__ tiles, uint32_t nitem, uint32_t nh, uint32_t group,
    uint32_t max_pos, uint64_t seq_stride, float scale, float* out, float* scratch, uint32_t ls) {
  using C = AttTileCfg<HPT>;
  constexpr uint32_t P = C::P, ES = C::ES, TP = C::TP, DG = HD / 16, NB = HD / 64;
  constexpr uint32_t NT1 = 4 * HPT, NT3 = HPT * NB;
  extern __shared__ v4 sh4[];
  v4* qf = sh4;                                    // [DG][4][P]
  float* reg = reinterpret_cast<float*>(qf + (size_t)DG * 4 * P);
  float* wmx = reg + C::region;                    // [4][P] wave maxima
  float* smx = wmx + 4 * P;                        // [P] maxima
  float* sden = smx + P;                           // [P] denominators
  const uint32_t nhb = nh / HPT, G = gridDim.x;
  float* S = scratch + (size_t)blockIdx.x * P * ls;  // [P][ls] scores, then exps
  for (uint32_t round = 0; (uint64_t)round * G < nitem; ++round) {
    // the thread id through an opaque copy: its many derived values are
    // formed where they are used, not kept in registers across the items
    uint32_t t = threadIdx.x;
    asm volatile("" : "+v"(t));
    const uint32_t wv = __builtin_amdgcn_readfirstlane(t >> 6);
    uint32_t lane = t & 63, u = lane >> 4, c16 = lane & 15;
    const f16v nz = minus_zeros();
    // odd rounds in reverse, by runs of 8 (a workgroup keeps its head's XCD)
    const uint32_t b = round & 1 ? G - 8 - (blockIdx.x & ~7u) + (blockIdx.x & 7) : blockIdx.x;
    const uint64_t w64 = (uint64_t)round * G + b;
    if (w64 >= nitem) continue;  // the same for the whole workgroup
    const uint32_t w = (uint32_t)w64, ti = w / nhb, qh0 = (w - ti * nhb) * HPT;
    const AttTile tl = tiles[ti];
    const uint32_t kvh = qh0 / group, len_max = tl.p0 + tl.nr, len_min = tl.p0 + 1;
    const size_t sb = (size_t)tl.seq * seq_stride + (size_t)kvh * HD * max_pos;
    const float* kb = kc + sb;
    const float* vb = vc + sb;
    const float* q0 = q + ((size_t)tl.row0 * nh + qh0) * HD;
    auto pair_len = [=](uint32_t a) { return tl.p0 + a % kAttQT + 1; };
    auto live = [=](uint32_t a) { return a % kAttQT < tl.nr; };
    __syncthreads();  // the item before this one is done with the LDS
    // q of every pair in operand order (rows past nr: zero, never stored)
    for (uint32_t i = t; i < P * DG; i += 256) {
      const uint32_t a = i % P, g = i / P;
      const v4* src = reinterpret_cast<const v4*>(
          q0 + (a % kAttQT * nh + a / kAttQT) * HD + 16 * g);
      v4 x[4];
#pragma unroll
      for (uint32_t m = 0; m < 4; ++m) x[m] = live(a) ? src[m] : v4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (uint32_t e = 0; e < 4; ++e)
        qf[(4 * g + e) * P + a] = v4{x[0][e], x[1][e], x[2][e], x[3][e]};
    }
    __syncthreads();
    // ---- scores ------------------------------------------------------------
    float best[HPT][4];
#pragma unroll
    for (uint32_t h = 0; h < HPT; ++h)
#pragma unroll
      for (uint32_t r = 0; r < 4; ++r) best[h][r] = -__builtin_inff();
#pragma unroll 1
    for (uint32_t j0 = 64 * wv; j0 < len_max; j0 += 256) {
      // columns past the cache's end are clamped; scores past a row's length
      // are never used
      const uint32_t ko = u * max_pos + min(j0 + 4 * c16, max_pos - 4);
      auto kload = [&](uint32_t d4) {  // rows 4 d4 .. 4 d4 + 3 of K
        return *reinterpret_cast<const v4*>(kb + (size_t)(4 * d4) * max_pos + ko);
      };
      float acc[NT1][4];
#pragma unroll
      for (uint32_t s = 0; s < NT1; ++s)
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) acc[s][r] = 0.0f;
      ChainSums<NT1, TREE> sums;
      f16v d[2];
      d[1] = nz;
      v4 kf[2][4];
#pragma unroll
      for (uint32_t m = 0; m < 4; ++m) kf[0][m] = kload(m);
      auto dgroup = [&](uint32_t g, uint32_t odd, const v4 (&cur)[4], v4 (&nxt)[4]) {
        if (g + 1 < DG) {
#pragma unroll
          for (uint32_t m = 0; m < 4; ++m) nxt[m] = kload(4 * (g + 1) + m);
        }
        v4 fa[HPT];
#pragma unroll
        for (uint32_t h = 0; h < HPT; ++h) fa[h] = qf[(4 * g + u) * P + 16 * h + c16];
#pragma unroll
        for (uint32_t x = 0; x < 4 * NT1; ++x) {
          const uint32_t m = mtile_k<NT1, TREE>(x), s = mtile_s<NT1, TREE>(x);
          d[x & 1] = products4(fa[s / 4][m], cur[m][s % 4], nz);
          asm volatile("" : "+v"(d[x & 1]));
          const uint32_t y = (x + 4 * NT1 - 1) % (4 * NT1);  // the products before these
          sums.add(acc, mtile_s<NT1, TREE>(y), 4 * ((x ? odd : odd + 1) & 1) + mtile_k<NT1, TREE>(y),
                   d[(x + 1) & 1]);
        }
      };
#pragma unroll 1
      for (uint32_t g = 0; g < DG; g += 2) {
        dgroup(g, 0, kf[0], kf[1]);
        dgroup(g + 1, 1, kf[1], kf[0]);
      }
      sums.add(acc, NT1 - 1, 7, d[1]);
      const uint32_t j = j0 + 4 * c16;
#pragma unroll
      for (uint32_t h = 0; h < HPT; ++h)
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) {
          const uint32_t i = 4 * u + r, len = len_min + i;
          v4 sv;
#pragma unroll
          for (uint32_t c = 0; c < 4; ++c) {
            sv[c] = acc[4 * h + c][r] * scale;
            best[h][r] = (j + c < len && sv[c] > best[h][r]) ? sv[c] : best[h][r];
          }
          if (i < tl.nr && j < ls)
            *reinterpret_cast<v4*>(S + (size_t)(16 * h + r) * ls + (4 * u * ls + j)) = sv;
        }
    }
#pragma unroll
    for (uint32_t h = 0; h < HPT; ++h)
#pragma unroll
      for (uint32_t r = 0; r < 4; ++r) {
        float m = best[h][r];
#pragma unroll
        for (uint32_t off = 1; off < 16; off <<= 1) {
          const float o = __shfl_xor(m, off, 64);
          m = o > m ? o : m;
        }
        if (c16 == 0) wmx[wv * P + 16 * h + 4 * u + r] = m;
      }
    // ---- softmax denominators ---------------------------------------------
    asm volatile("" : "+v"(t));
    lane = t & 63, u = lane >> 4, c16 = lane & 15;
    // the scores are stored before they are read back; writer and reader
    // waves share the CU and its cache, so the workgroup's scope is enough
    // (an agent-scope fence writes the XCD's L2 back: 5 x the time of a
    // short tile)
    __threadfence_block();
    __syncthreads();
    // the largest non-NaN score; a NaN at position 0 wins with its own bits
    if (t < P && live(t)) {
      float m = wmx[t];
#pragma unroll
      for (uint32_t w4 = 1; w4 < 4; ++w4) m = wmx[w4 * P + t] > m ? wmx[w4 * P + t] : m;
      const float s0 = S[t * ls];
      smx[t] = s0 != s0 ? s0 : m;
    }
    const uint32_t nst = (len_max + kAttTE - 1) / kAttTE;
    auto es = [=](uint32_t i) { return reg + (i & 1) * P * ES; };
    // waves 1..3: copy stage i of the pairs' scores and exponentiate it in
    // place, four pair rows per wave instruction, each wave on the rows it
    // copied
    auto stage = [=](uint32_t i) {
      const uint32_t j0 = i * kAttTE, j = j0 + 4 * c16;
      float* st = es(i);
      for (uint32_t a = 4 * (wv - 1) + u; a < P; a += 12) {
        const uint32_t len = pair_len(a);
        if (!live(a) || j >= len) continue;
        v4* sp = reinterpret_cast<v4*>(S + (a * ls + j));
        const float mx = smx[a];
        v4 e = *sp;
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) {
          const float dlt = e[c] - mx;
          e[c] = exp_pinned(dlt);
        }
        *reinterpret_cast<v4*>(st + (a * ES + 4 * c16)) = e;
        *sp = e;
      }
    };
    __syncthreads();
    if (wv >= 1) stage(0);
    __syncthreads();
    float den = 0.0f;
    for (uint32_t i = 0; i < nst; ++i) {
      // lanes a < P of wave 0 chain stage i; waves 1..3 prepare stage i+1 in
      // the other buffer (its stage i-1 was chained before this barrier)
      if (wv == 0) {
        if (lane < P && live(lane)) {
          const uint32_t j0 = i * kAttTE, len = pair_len(lane);
          const float* ep = es(i) + lane * ES;
          if constexpr (TREE) {
#pragma unroll
            for (uint32_t b = 0; b < kAttTE; b += 32)
              if (j0 + b < len) {
                float l[32];
#pragma unroll
                for (uint32_t k = 0; k < 32; ++k) l[k] = j0 + b + k < len ? ep[b + k] : 0.0f;
                den = den + tree32(l);
              }
          } else if (j0 < len) {
            den = chain_lds(ep, min(kAttTE, len - j0), den);
          }
        }
      } else if (i + 1 < nst) {
        stage(i + 1);
      }
      __syncthreads();
    }
    if (wv == 0 && lane < P) sden[lane] = den;
    __threadfence_block();  // the exps are stored before they are read back
    __syncthreads();
    // ---- V-mix --------------------------------------------------------------
    asm volatile("" : "+v"(t));
    lane = t & 63, u = lane >> 4, c16 = lane & 15;
    // p tile T of TP positions: this thread's piece is 16 positions of a pair
    const uint32_t pa = t % P, pg = t / P;
    const bool mine = t < P * TP / 16;
    v4* pf0 = reinterpret_cast<v4*>(reg);  // 2 x [TP / 16][4][P]
    v4 ev[4];
    auto load_e = [&](uint32_t T) {
      if (mine) {
#pragma unroll
        for (uint32_t m = 0; m < 4; ++m)
          ev[m] = *reinterpret_cast<const v4*>(S + (pa * ls + min(T * TP + 16 * pg + 4 * m, ls - 4)));
      }
    };
    auto store_p = [&](uint32_t T) {
      if (mine) {
        const float dn = sden[pa];
#pragma unroll
        for (uint32_t m = 0; m < 4; ++m)
#pragma unroll
          for (uint32_t e = 0; e < 4; ++e) ev[m][e] = ev[m][e] / dn;
        v4* pf = pf0 + (T & 1) * (P * TP / 4);
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e)
          pf[(4 * pg + e) * P + pa] = v4{ev[0][e], ev[1][e], ev[2][e], ev[3][e]};
      }
    };
    float acc[NT3][4];
#pragma unroll
    for (uint32_t s = 0; s < NT3; ++s)
#pragma unroll
      for (uint32_t r = 0; r < 4; ++r) acc[s][r] = 0.0f;
    auto add = [&](uint32_t s, const f16v& p) {
#pragma unroll
      for (uint32_t e = 0; e < 4; ++e)
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) acc[s][r] = acc[s][r] + p[4 * e + r];
      asm volatile("" : "+v"(acc[s][0]), "+v"(acc[s][1]), "+v"(acc[s][2]), "+v"(acc[s][3]));
    };
    // V of 16-position group gi: lane (dim c16 of a 16-dim tile, u) loads
    // positions 4u .. 4u+3
    v4 vr[4][NB];
    auto load_v = [&](uint32_t gi, v4 (&v)[NB]) {
      const uint32_t col = min(16 * gi + 4 * u, max_pos - 4);
#pragma unroll
      for (uint32_t x = 0; x < NB; ++x)
        v[x] = *reinterpret_cast<const v4*>(vb + (size_t)(16 * (wv * NB + x)) * max_pos +
                                            (c16 * max_pos + col));
    };
    const uint32_t ngr = (len_max + 15) / 16, ntile = (len_max + TP - 1) / TP;
#pragma unroll
    for (uint32_t g = 0; g < 4; ++g)
      if (g < ngr) load_v(g, vr[g]);
    f16v d[2];
    d[1] = nz;
    load_e(0);
    store_p(0);
#pragma unroll 1
    for (uint32_t T = 0; T < ntile; ++T) {
      __syncthreads();
      if (T + 1 < ntile) load_e(T + 1);
      const v4* pf = pf0 + (T & 1) * (P * TP / 4);
#pragma unroll 1
      for (uint32_t g4 = 0; g4 < TP / 16; g4 += 4) {
#pragma unroll
        for (uint32_t gg = 0; gg < 4; ++gg) {
          const uint32_t gl = g4 + gg, gi = T * (TP / 16) + gl;
          if (gi >= ngr) break;
          v4 fb[NB], fa[HPT];
#pragma unroll
          for (uint32_t x = 0; x < NB; ++x) {
            fb[x] = vr[gg][x];
            transpose4(fb[x]);
          }
          if (gi + 4 < ngr) load_v(gi + 4, vr[gg]);
#pragma unroll
          for (uint32_t h = 0; h < HPT; ++h) fa[h] = pf[(4 * gl + u) * P + 16 * h + c16];
          if (16 * gi + 16 <= len_min) {
#pragma unroll
            for (uint32_t m = 0; m < 4; ++m)
#pragma unroll
              for (uint32_t s = 0; s < NT3; ++s) {
                const uint32_t x = m * NT3 + s;
                d[x & 1] = products4(fa[s / NB][m], fb[s % NB][m], nz);
                asm volatile("" : "+v"(d[x & 1]));
                add((s + NT3 - 1) % NT3, d[(x + 1) & 1]);
              }
          } else {
            // the pending tile's adds, then adds of j < the row's length only
            add(NT3 - 1, d[1]);
            d[1] = nz;
#pragma unroll
            for (uint32_t m = 0; m < 4; ++m)
#pragma unroll
              for (uint32_t s = 0; s < NT3; ++s) {
                f16v p = products4(fa[s / NB][m], fb[s % NB][m], nz);
                asm volatile("" : "+v"(p));
#pragma unroll
                for (uint32_t e = 0; e < 4; ++e)
#pragma unroll
                  for (uint32_t r = 0; r < 4; ++r) {
                    const float y = acc[s][r] + p[4 * e + r];
                    acc[s][r] = 16 * gi + 4 * m + e < len_min + 4 * u + r ? y : acc[s][r];
                  }
                asm volatile("" : "+v"(acc[s][0]), "+v"(acc[s][1]), "+v"(acc[s][2]), "+v"(acc[s][3]));
              }
          }
        }
      }
      if (T + 1 < ntile) store_p(T + 1);
    }
    add(NT3 - 1, d[1]);
    float* o0 = out + ((size_t)tl.row0 * nh + qh0) * HD;
#pragma unroll
    for (uint32_t s = 0; s < NT3; ++s)
#pragma unroll
      for (uint32_t r = 0; r < 4; ++r) {
        const uint32_t i = 4 * u + r, h = s / NB, dd = 16 * (wv * NB + s % NB) + c16;
        if (i < tl.nr) o0[(i * nh + h) * HD + dd] = acc[s][r];
      }
  }
}

__global__ void k_gather_rows(const float* __restrict__ src, const uint32_t* __restrict__ idx,
                              uint32_t width, float* dst) {
  const uint32_t r = blockIdx.x;
  const float* s = src + (size_t)idx[r] * width;
  for (uint32_t i = threadIdx.x; i < width; i += blockDim.x) dst[(size_t)r * width + i] = s[i];
}

__global__ void k_advance_rows(uint32_t* pos, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) pos[i] = pos[i] + 1u;
}

__global__ __launch_bounds__(1024) void k_argmax_rows(const float* __restrict__ v,
                                                      uint32_t width, uint32_t* out) {
  __shared__ Pick red[16];
  const float* row = v + (size_t)blockIdx.x * width;
  Pick best = {0.0f, UINT32_MAX};
  for (uint32_t i = threadIdx.x; i < width; i += blockDim.x) {
    const float x = row[i];
    if (x == x) best = pick2(best, Pick{x, i});
  }
  best = pick_block(best, red);
  if (threadIdx.x == 0) {
    const float v0 = row[0];
    out[blockIdx.x] = (v0 != v0 || best.i == UINT32_MAX) ? 0u : best.i;
  }
}

}  // namespace

template <bool DUAL, bool NORM>
hipError_t launch_bgemm_t(const BgemmArgs& a, dim3 grid, size_t lds, hipStream_t st) {
  hipLaunchKernelGGL((k_bgemm<DUAL, NORM>), grid, dim3(kT), lds, st, a);
  return hipGetLastError();
}

// The LDS limit of every k_bgemm and k_attention_kv variant, set at the
// first launch of any (a forward launches a GEMM before its first
// attention), so that no attribute call happens later, e.g. inside a graph
// capture.
hipError_t rows_configure() {
  const void* fns[18] = {reinterpret_cast<const void*>(&k_bgemm<false, false>),
                         reinterpret_cast<const void*>(&k_bgemm16<false, false>),
                         reinterpret_cast<const void*>(&k_bgemm16<false, true>),
                         reinterpret_cast<const void*>(&k_bgemm16<true, false>),
                         reinterpret_cast<const void*>(&k_bgemm16<true, true>),
                         reinterpret_cast<const void*>(&k_bgemm<false, true>),
                         reinterpret_cast<const void*>(&k_bgemm<true, false>),
                         reinterpret_cast<const void*>(&k_bgemm<true, true>),
                         reinterpret_cast<const void*>(&k_attention_kv<1, 64, false>),
                         reinterpret_cast<const void*>(&k_attention_kv<2, 64, false>),
                         reinterpret_cast<const void*>(&k_attention_kv<3, 64, false>),
                         reinterpret_cast<const void*>(&k_attention_kv<1, 128, false>),
                         reinterpret_cast<const void*>(&k_attention_kv<2, 128, false>),
                         reinterpret_cast<const void*>(&k_attention_kv<1, 64, true>),
                         reinterpret_cast<const void*>(&k_attention_kv<2, 64, true>),
                         reinterpret_cast<const void*>(&k_attention_kv<3, 64, true>),
                         reinterpret_cast<const void*>(&k_attention_kv<1, 128, true>),
                         reinterpret_cast<const void*>(&k_attention_kv<2, 128, true>)};
  for (const void* f : fns) {
    hipError_t e = ensure_dynamic_lds(f, kBgemmLdsBig);
    if (e != hipSuccess) return e;
  }
  for (const void* f : {reinterpret_cast<const void*>(&k_chain_gemm<false, false>),
                        reinterpret_cast<const void*>(&k_chain_gemm<false, true>),
                        reinterpret_cast<const void*>(&k_chain_gemm<true, false>),
                        reinterpret_cast<const void*>(&k_chain_gemm<true, true>)}) {
    hipError_t e = ensure_dynamic_lds(f, kLdsMost);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// CIS2_BGEMM16=0 keeps every batched GEMM on k_bgemm (for A/B timing and
// tests; the results are the same bits either way).
static bool bgemm16_allowed() {
  const char* e = std::getenv("CIS2_BGEMM16");
  return !(e && e[0] == '0' && e[1] == 0);
}

// k_bgemm16 for sequential-order GEMMs whose W blocks have 8 or 16 rows and
// whose segments are whole 16-output tiles.
static hipError_t launch_bgemm16(const BgemmSeg* segs, uint32_t nseg, uint32_t n,
                                 const BgemmOpts& o, int ncu, hipStream_t st) {
  const BgemmSeg& s0 = segs[0];
  BgemmArgs a = {};
  a.blk0[0] = 0;
  for (uint32_t i = 0; i < nseg; ++i) {
    a.s[i] = segs[i];
    a.blk0[i + 1] = a.blk0[i] + segs[i].M / 16;
  }
  for (uint32_t i = nseg; i < kMaxSegs; ++i) {
    a.s[i] = s0;
    a.blk0[i + 1] = a.blk0[nseg];
  }
  a.nseg = nseg;
  a.n = n;
  a.TB = 16;
  a.tree = 0;
  a.W2 = o.W2;
  a.nw = o.norm_w;
  a.eps = o.eps;
  const uint32_t S = o.W2 ? 2 : 1, NW = o.norm_w ? 1 : 0, nblk = 16 / s0.R;
  const uint64_t wgs = (uint64_t)a.blk0[nseg] * ((n + 15) / 16);
  const uint32_t budget = wgs <= (uint64_t)ncu ? kBgemmLdsBig : kBgemmLds;
  // LDS groups: S * nblk * (q * R + 8) + NW * q + 16 * (q + 1) + slack
  const uint32_t fixed = 8 * S * nblk + 16 + b16_slack(s0.R);
  const uint32_t q_fit = (budget / 16 - fixed) / (16 * S + NW + 16);
  uint32_t KC = std::min((q_fit * 4) & ~31u, 1024u);
  if (KC == 0) return hipErrorInvalidValue;
  const uint32_t K32 = (s0.K + 31) & ~31u;
  if (KC > K32) KC = K32;
  a.KC = KC;
  const size_t q = KC / 4;
  const size_t lds =
      ((size_t)S * nblk * (q * s0.R + 8) + NW * q + 16 * (q + 1) + b16_slack(s0.R)) * 16;
  const dim3 grid(a.blk0[nseg], (n + 15) / 16);
  if (o.W2)
    hipLaunchKernelGGL((o.norm_w ? k_bgemm16<true, true> : k_bgemm16<true, false>), grid,
                       dim3(kT), lds, st, a);
  else
    hipLaunchKernelGGL((o.norm_w ? k_bgemm16<false, true> : k_bgemm16<false, false>), grid,
                       dim3(kT), lds, st, a);
  return hipGetLastError();
}

// Arguments of a grid of bm x bn tiles.
static bool mgemm_args(const BgemmSeg* segs, uint32_t nseg, uint32_t n, const float* W2,
                       uint32_t bm, uint32_t bn, MgemmArgs* out) {
  MgemmArgs a = {};
  a.nseg = nseg;
  a.n = n;
  a.W2 = W2;
  a.vec = 1;
  for (uint32_t i = 0; i < kMaxSegs; ++i) {
    a.s[i] = segs[i < nseg ? i : 0];
    if (i < nseg) {
      a.tile0[i + 1] = a.tile0[i] + (segs[i].M + bm - 1) / bm;
      if (segs[i].M % 4 || segs[i].ldy % 4 || segs[i].ldadd % 4) a.vec = 0;
    } else {
      a.tile0[i + 1] = a.tile0[nseg];
    }
  }
  const uint64_t tiles = (uint64_t)a.tile0[nseg] * ((n + bn - 1) / bn);
  if (tiles > 0x7fffffffu - 8) return false;
  a.tiles = (uint32_t)tiles;
  *out = a;
  return true;
}

template <bool DUAL, bool TREE, uint32_t SM, uint32_t SN, uint32_t WM, uint32_t WN, uint32_t KC,
          uint32_t OCC, uint32_t PF>
static hipError_t launch_mgemm(const BgemmSeg* segs, uint32_t nseg, uint32_t n,
                                 const float* W2, hipStream_t st) {
  using C = MgemmCfg<DUAL, SM, SN, WM, WN, KC>;
  MgemmArgs a;
  if (!mgemm_args(segs, nseg, n, W2, C::BM, C::BN, &a)) return hipErrorInvalidValue;
  hipLaunchKernelGGL((k_mgemm<DUAL, TREE, SM, SN, WM, WN, KC, OCC, PF>), dim3((a.tiles + 7) / 8 * 8),
                     dim3(256), 0, st, a);
  return hipGetLastError();
}

template <bool DUAL, bool NORM>
static hipError_t launch_chain_gemm(const BgemmSeg* segs, uint32_t nseg, uint32_t n,
                                    const BgemmOpts& o, hipStream_t st) {
  BgemmArgs a = {};
  for (uint32_t i = 0; i < kMaxSegs; ++i) {
    a.s[i] = segs[i < nseg ? i : 0];
    a.blk0[i + 1] = i < nseg ? a.blk0[i] + (segs[i].M + 7) / 8 : a.blk0[nseg];
  }
  a.nseg = nseg;
  a.n = n;
  a.W2 = o.W2;
  a.nw = o.norm_w;
  a.eps = o.eps;
  hipLaunchKernelGGL((k_chain_gemm<DUAL, NORM>), dim3(a.blk0[nseg], (n + 7) / 8), dim3(ChainCfg<DUAL, NORM>::T),
                     (ChainCfg<DUAL, NORM>::lds(segs[0].K)), st, a);
  return hipGetLastError();
}
// k_chain_gemm takes segments whose blocks are whole groups of 8 rows, rows
// that fit the LDS beside the ring (fused norm), and grids that the CUs hold
// at once, one workgroup per CU: a second round costs more than k_bgemm16's
// one (n = 8 | 16 | 24, us, k_bgemm16 then k_chain_gemm: 576 x 1536 16.7
// 9.8 | 16.7 10.0 | 16.8 10.1, 768 x 3072 30.4 16.0 | 30.3 16.4 | 30.5 28.5).
// Below 256 k its two prologue round trips are not won back (K = 52: 4.6
// against 5.5).
static bool chain_gemm_fits(const BgemmSeg* segs, uint32_t nseg, uint32_t n, const BgemmOpts& o,
                            uint32_t ncu) {
  const uint32_t K = segs[0].K;
  if (segs[0].R % 8 || K < 256) return false;
  if (o.norm_w) {
    if ((o.W2 ? ChainCfg<true, true>::lds(K) : ChainCfg<false, true>::lds(K)) > kLdsMost ||
        (size_t)K / 4 * 8 > (o.W2 ? ChainCfg<true, true>::ring : ChainCfg<false, true>::ring))
      return false;
  }
  uint64_t wgs = 0;
  for (uint32_t i = 0; i < nseg; ++i) wgs += (segs[i].M + 7) / 8;
  return wgs * ((n + 7) / 8) <= ncu;
}

// Which kernel a GEMM without a fused norm takes.  Every
// form costs a time per k that depends on how many workgroups the fullest CU
// gets; measured on the layer shapes of the three models at n = 7 .. 16384,
// in ns per k (two figures: one matrix, gate and up):
//   k_bgemm16 / k_bgemm  256 chains per workgroup     11 | 21 at one per CU,
//                                                     7.7 | 14.5 each beyond
//   k_bgemm, tree order                               18 | 36, 10.8 | 21.6
//   k_mgemm, 32 x 32     1024 chains (2048 for two)   19 | 39, then 11 | 21 each
//   k_mgemm, 64 x 64     4096 chains                  57, then 37.5 each
// A small grid is bound by one wave's latency and wants many short
// workgroups, a large one by the vector units and wants operands reused: the
// least of the three estimates is taken.  (o projection of 576 x 576, us:
// n = 64 8.6 | 12.8 | 35.4, n = 544 23.3 | 16.8 | 35.7, n = 16384 518 | 254 |
// 188; gate and up of 3072 x 1024 at n = 16384 8254 | 3635 | 3293.  Tree order,
// us per layer, k_bgemm | 32 x 32 | 64 x 64: 30-layer shape of 576, 64 rows
// 104 | 105 | 234, 124 rows 141 | 114 | 244, 2000 rows 1298 | 476 | 520; that
// of 1024, 16 rows 195 | 219 | 498, 2000 rows 5908 | 2281 | 2096.)
// The constants are fits, so they were tried on eleven shapes that they were
// not fitted to: hidden sizes 100 .. 4096, inner sizes 260 .. 11008, groups of
// 1 .. 8 heads of 20 .. 128, 2 .. 256 decode rows, runs of 2 .. 8 rows, prompts
// of 2 .. 599 rows.  Layer times without the matrix cores (and without
// k_chain_gemm and the norm's placement) over those with them: sequential
// 0.97 .. 6.7, tree 0.97 .. 5.9, under 1 only by what two runs differ.
enum class MgemmTile { none, small, large };
struct MgemmPlan {
  MgemmTile tile;
  double none_ns, best_ns;  // per k, without and with the matrix cores
};
static MgemmPlan mgemm_plan(const BgemmSeg* segs, uint32_t nseg, uint32_t n, const BgemmOpts& o,
                            uint32_t ncu) {
  const bool dual = o.W2 != nullptr;
  uint64_t t16 = 0, t32 = 0, t64 = 0;  // W tiles of 16, 32 (16 x 64 rows) and 64 rows
  const uint32_t sm = n <= 16 && !dual ? 64 : 32, sn = n <= 16 && !dual ? 16 : 32;
  for (uint32_t i = 0; i < nseg; ++i) {
    t16 += (segs[i].M + 15) / 16;
    t32 += (segs[i].M + sm - 1) / sm;
    t64 += (segs[i].M + (dual ? 31 : 63)) / (dual ? 32 : 64);
  }
  auto per_cu = [&](uint64_t wt, uint32_t bn) {
    return (double)((wt * ((n + bn - 1) / bn) + ncu - 1) / ncu);
  };
  const double two = dual ? 2.0 : 1.0;
  const double t0 = (o.tree ? std::max(18.0, 10.8 * per_cu(t16, 16))
                            : std::max(10.5, 7.5 * per_cu(t16, 16))) * two;
  const double ts = std::max(19.0, 10.5 * per_cu(t32, sn) + 2.0) * two;
  const double tl = std::max(57.0, 37.5 * per_cu(t64, 64));
  if (t0 <= ts && t0 <= tl) return {MgemmTile::none, t0, t0};
  return {ts <= tl ? MgemmTile::small : MgemmTile::large, t0, std::min(ts, tl)};
}

template <bool TREE>
static hipError_t launch_mgemm_tile(MgemmTile tile, const BgemmSeg* segs, uint32_t nseg,
                                    uint32_t n, const float* W2, hipStream_t st) {
  if (tile == MgemmTile::large)
    return W2 ? launch_mgemm<true, TREE, 2, 2, 2, 2, 32, 3, 1>(segs, nseg, n, W2, st)
              : launch_mgemm<false, TREE, 2, 2, 2, 2, 32, 3, 1>(segs, nseg, n, W2, st);
  if (W2) return launch_mgemm<true, TREE, 2, 1, 2, 2, 32, 2, 2>(segs, nseg, n, W2, st);
  // up to 16 rows: 64 x 16 tiles (the LM head at n = 16: 26 against 41 us)
  return n <= 16 ? launch_mgemm<false, TREE, 1, 1, 4, 1, 64, 2, 1>(segs, nseg, n, W2, st)
                 : launch_mgemm<false, TREE, 1, 1, 2, 2, 64, 3, 2>(segs, nseg, n, W2, st);
}

bool bgemm_norm_apart(const BgemmSeg* segs, uint32_t nseg, uint32_t n, const BgemmOpts& o) {
  if (n == 0 || nseg == 0 || nseg > kMaxSegs) return false;
  const uint32_t ncu = (uint32_t)device_cu_count();
  if (!bgemm16_allowed()) return n > kFuseNormRows;
  if (!o.tree && chain_gemm_fits(segs, nseg, n, o, ncu)) return false;
  // the fused norm costs a chain of the row inside the launch (about 6 ns per
  // k), the separate one a launch of 7 us: 960 x 576, us, fused | apart:
  // 64 rows 12.2 | 19.8, 130 rows 19 | 20, 256 rows 22 | 20.5; in tree order
  // 20 ns per k (us per layer, 2 rows: 105 | 96, 146 | 134, 199 | 180)
  const MgemmPlan p = mgemm_plan(segs, nseg, n, o, ncu);
  return (p.none_ns + (o.tree ? 20.0 : 6.0)) * segs[0].K > p.best_ns * segs[0].K + 7000.0;
}

hipError_t launch_bgemm_multi(const BgemmSeg* segs, uint32_t nseg, uint32_t n,
                              const BgemmOpts& o, hipStream_t st) {
  if (n == 0) return hipSuccess;
  if (nseg == 0 || nseg > kMaxSegs || (o.W2 && nseg != 1)) return hipErrorInvalidValue;
  {
    hipError_t e = rows_configure();
    if (e != hipSuccess) return e;
  }
  const BgemmSeg& s0 = segs[0];
  if (s0.K % 4 || s0.ldx % 4 || s0.R == 0 || s0.R > kT) return hipErrorInvalidValue;
  for (uint32_t i = 0; i < nseg; ++i)
    if (segs[i].M == 0 || segs[i].K != s0.K || segs[i].R != s0.R || segs[i].X != s0.X ||
        segs[i].ldx != s0.ldx)
      return hipErrorInvalidValue;
  const int ncu = device_cu_count();
  if (o.tree && !o.norm_w && bgemm16_allowed()) {
    const MgemmTile tile = mgemm_plan(segs, nseg, n, o, (uint32_t)ncu).tile;
    if (tile != MgemmTile::none) return launch_mgemm_tile<true>(tile, segs, nseg, n, o.W2, st);
  }
  if (!o.tree && bgemm16_allowed()) {
    if (chain_gemm_fits(segs, nseg, n, o, (uint32_t)ncu)) {
      if (o.W2) return o.norm_w ? launch_chain_gemm<true, true>(segs, nseg, n, o, st)
                                : launch_chain_gemm<true, false>(segs, nseg, n, o, st);
      return o.norm_w ? launch_chain_gemm<false, true>(segs, nseg, n, o, st)
                      : launch_chain_gemm<false, false>(segs, nseg, n, o, st);
    }
    if (!o.norm_w) {
      const MgemmTile tile = mgemm_plan(segs, nseg, n, o, (uint32_t)ncu).tile;
      if (tile != MgemmTile::none) return launch_mgemm_tile<false>(tile, segs, nseg, n, o.W2, st);
    }
    bool tiles = s0.R == 8 || s0.R == 16;
    for (uint32_t i = 0; i < nseg && tiles; ++i) tiles = segs[i].M % 16 == 0;
    if (tiles) return launch_bgemm16(segs, nseg, n, o, ncu, st);
  }
  BgemmArgs a = {};
  a.blk0[0] = 0;
  for (uint32_t i = 0; i < nseg; ++i) {
    a.s[i] = segs[i];
    a.blk0[i + 1] = a.blk0[i] + (segs[i].M + segs[i].R - 1) / segs[i].R;
  }
  for (uint32_t i = nseg; i < kMaxSegs; ++i) {
    a.s[i] = s0;
    a.blk0[i + 1] = a.blk0[nseg];
  }
  a.nseg = nseg;
  a.n = n;
  a.TB = kT / s0.R;
  a.tree = o.tree ? 1u : 0u;
  a.W2 = o.W2;
  a.nw = o.norm_w;
  a.eps = o.eps;
  const uint32_t S = o.W2 ? 2 : 1;
  const uint64_t wgs = (uint64_t)a.blk0[nseg] * ((n + a.TB - 1) / a.TB);
  // a grid of at most one workgroup per CU may take most of a CU's LDS
  // (fewer K chunks, each a full round trip); larger grids keep two
  // workgroups per CU, so that up to two per CU all run at once
  const uint32_t budget = wgs <= (uint64_t)ncu ? kBgemmLdsBig : kBgemmLds;
  // largest chunk (a multiple of 32 k) whose W slices, X rows and norm
  // weights fit
  const uint32_t NW = o.norm_w ? 1 : 0;
  const uint32_t q_fit = (budget / 16 - a.TB) / (S * s0.R + a.TB + NW);
  uint32_t KC = (q_fit * 4) & ~31u;
  if (KC == 0) return hipErrorInvalidValue;
  const uint32_t K32 = (s0.K + 31) & ~31u;
  if (KC > K32) KC = K32;
  a.KC = KC;
  const size_t lds = ((size_t)(KC / 4) * (s0.R * S + NW) + (size_t)a.TB * (KC / 4 + 1)) * 16;
  const dim3 grid(a.blk0[nseg], (n + a.TB - 1) / a.TB);
  if (o.W2) return o.norm_w ? launch_bgemm_t<true, true>(a, grid, lds, st)
                            : launch_bgemm_t<true, false>(a, grid, lds, st);
  return o.norm_w ? launch_bgemm_t<false, true>(a, grid, lds, st)
                  : launch_bgemm_t<false, false>(a, grid, lds, st);
}

hipError_t launch_bgemm(const BgemmSeg& s, uint32_t n, bool tree, hipStream_t st) {
  BgemmOpts o;
  o.tree = tree;
  return launch_bgemm_multi(&s, 1, n, o, st);
}

hipError_t launch_embed_rows(const float* E, RowsDesc rows, uint32_t H, uint32_t vocab,
                             float* h, uint32_t* err, hipStream_t st) {
  if (rows.n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_embed_rows, dim3(rows.n), dim3(kT), 0, st, E, rows, H, vocab, h, err);
  return hipGetLastError();
}

hipError_t launch_rope_store_rows(float* q, float* k, const float* v, const float* rope_cs,
                                  RowsDesc rows, uint32_t nh, uint32_t nkv, uint32_t hd,
                                  uint32_t max_pos, float* kc, float* vc, uint64_t seq_stride,
                                  hipStream_t st) {
  if (rows.n == 0) return hipSuccess;
  if (hd % 2) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_rope_store_rows, dim3(rows.n), dim3(kT), 0, st, q, k, v, rope_cs, rows,
                     nh, nkv, hd, max_pos, kc, vc, seq_stride);
  return hipGetLastError();
}

hipError_t launch_rope_store_tiles(float* q, const float* k, const float* v, const float* rope_cs,
                                   const AttTile* tiles, uint32_t ntiles, uint32_t nh,
                                   uint32_t nkv, uint32_t hd, uint32_t max_pos, float* kc,
                                   float* vc, uint64_t seq_stride, hipStream_t st) {
  if (ntiles == 0) return hipSuccess;
  if (!attention_tiles_supported(nh, nkv, hd)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_rope_store_tiles, dim3(ntiles, nkv), dim3(kT), 0, st, q, k, v, rope_cs,
                     tiles, nh, nkv, hd, max_pos, kc, vc, seq_stride);
  return hipGetLastError();
}

// CIS2_ATT_KV=0 keeps decode rows on the one-head-per-workgroup kernel;
// CIS2_ATT_KV=<n> caps the V chunk at n positions (rounded down to a
// multiple of 64), so that short rows run through the chunk ring too.  For
// A/B timing and tests: the results are the same bits either way.
static size_t kv_attention_cap() {
  const char* e = std::getenv("CIS2_ATT_KV");
  if (!e || !*e) return SIZE_MAX;
  return (size_t)std::strtoul(e, nullptr, 10) / 64 * 64;
}

// Decode rows (rows x kv heads < 4 x CUs), head_dim 64 or 128: one
// workgroup per (row, KV head) with the V rows staged in LDS, in chunks of C
// positions (two buffers: the longest row in one pass of each when they
// fit).  A grid of at most one workgroup per CU may take most of the LDS,
// larger ones half.  C = 0: another kernel.
struct KvPlan {
  size_t C = 0, shmem = 0;
  uint32_t group = 0, ls = 0;
};
static hipError_t kv_plan(uint32_t n, uint32_t nh, uint32_t nkv, uint32_t hd, uint32_t max_len,
                          KvPlan* p) {
  *p = KvPlan{};
  if (nkv == 0 || nh % nkv) return hipErrorInvalidValue;
  const uint32_t group = nh / nkv;
  const int ncu = device_cu_count();
  const uint64_t wgs_kv = (uint64_t)n * nkv;
  // instances for groups of up to 3 heads at head_dim 64 and 2 at 128 (a
  // group of 4 at head_dim 64 needed more registers than a wave has and
  // spilled to scratch; such models take the per-row kernel)
  if (!(wgs_kv < 4 * (uint64_t)ncu && ((hd == 64 && group <= 3) || (hd == 128 && group <= 2))))
    return hipSuccess;
  hipError_t e = rows_configure();
  if (e != hipSuccess) return e;
  const size_t ls = ((size_t)max_len + 3) / 4 * 4, nbs = (ls + 31) / 32;
  const size_t fixed =
      (group * hd + 2 * hd + group * ls + ((group * nbs + 3) & ~(size_t)3)) * 4;
  const size_t budget = wgs_kv <= (uint64_t)ncu ? kBgemmLdsBig : kBgemmLds;
  const size_t c_need =
      std::min<size_t>((((size_t)max_len + 1) / 2 + 63) & ~(size_t)63, 256);
  size_t c_fit = 0;
  if (budget > fixed + kKvSlack * 4 + 8 * hd * 68)
    c_fit = ((budget - fixed - kKvSlack * 4) / (8 * hd) - 4) & ~(size_t)63;
  const size_t C = std::min(std::min(c_need, c_fit), kv_attention_cap());
  if (C < 64) return hipSuccess;
  p->C = C;
  p->shmem = fixed + 2 * hd * (C + 4) * 4 + kKvSlack * 4;
  p->group = group;
  p->ls = (uint32_t)ls;
  return hipSuccess;
}
static hipError_t launch_kv(const KvPlan& kp, bool fuse, const float* q, float* kc, float* vc,
                            RowsDesc rows, uint32_t nh, uint32_t hd, uint32_t max_pos,
                            uint64_t seq_stride, float scale, float* out, bool tree,
                            const KvFuse& fz, hipStream_t st) {
  const dim3 grid(rows.n, nh / kp.group);
  const uint32_t tr = tree ? 1u : 0u, c32 = (uint32_t)kp.C;
#define CIS2_ATT_KV(H, D)                                                                     \
  do {                                                                                        \
    if (fuse)                                                                                 \
      hipLaunchKernelGGL((k_attention_kv<H, D, true>), grid, dim3(kKvT), kp.shmem, st, q, kc, \
                         vc, rows, nh, max_pos, seq_stride, scale, out, tr, kp.ls, c32, fz);  \
    else                                                                                      \
      hipLaunchKernelGGL((k_attention_kv<H, D, false>), grid, dim3(kKvT), kp.shmem, st, q,    \
                         kc, vc, rows, nh, max_pos, seq_stride, scale, out, tr, kp.ls, c32,   \
                         fz);                                                                 \
  } while (0)
  if (hd == 64) {
    switch (kp.group) {
      case 1: CIS2_ATT_KV(1, 64); break;
      case 2: CIS2_ATT_KV(2, 64); break;
      default: CIS2_ATT_KV(3, 64);
    }
  } else {
    if (kp.group == 1) CIS2_ATT_KV(1, 128);
    else CIS2_ATT_KV(2, 128);
  }
#undef CIS2_ATT_KV
  return hipGetLastError();
}

// k_attention_wave where the (row, head) pairs give every SIMD two waves or
// more and no row is long (us per layer with k_attention_rows and k_rope_store
// | here; 300 rows of 12 heads of 64: 40 positions 299 | 269, 200 349 | 341,
// 500 477 | 462, 1500 793 | 833; 256 rows of 16 heads of 128: 637 | 582, 683 |
// 674, 882 | 833, 1236 | 1373); false for another kernel.  Larger groups, whose
// heads read K and V again here, gain as much, and so do short runs of one
// sequence (without FUSE; 256 rows at 100 | 400 positions, then 256 runs of 3
// rows at 100 | 400): groups of 4, 16 heads of 64: 286 | 249, 315 | 309, 560 |
// 494, 642 | 625; of 7, 14 of 64: 323 | 296, 380 | 349, 705 | 595, 920 | 723; of
// 8, 32 of 64: 675 | 622, 733 | 716, 1612 | 1479, 1765 | 1712; of 4, 32 of 128:
// 2088 | 1979, 2256 | 2196, 5586 | 5281, 5971 | 5899.
constexpr uint32_t kWaveLen = 512;
static bool wave_attention(uint32_t n, uint32_t nh, uint32_t nkv, uint32_t hd, uint32_t max_len,
                           bool tree, size_t* lds) {
  const size_t ls = ((size_t)max_len + 3) / 4 * 4;
  *lds = 4 * (3 * (size_t)hd + ls) * sizeof(float);
  return !tree && (hd == 64 || hd == 128) && nkv != 0 && nh % nkv == 0 &&
         (uint64_t)n * nh >= 8 * (uint64_t)device_cu_count() &&
         (uint64_t)n * nh <= 0x7fffffffu && max_len <= kWaveLen && kv_attention_cap() != 0;
}
static hipError_t launch_wave(bool fuse, const float* q, float* kc, float* vc, RowsDesc rows,
                              uint32_t max_len, uint32_t nh, uint32_t nkv, uint32_t hd,
                              uint32_t max_pos, uint64_t seq_stride, float scale, float* out,
                              size_t lds, const KvFuse& fz, hipStream_t st) {
  const uint32_t ls = (max_len + 3) / 4 * 4, g = nh / nkv;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((rows.n * nh + 3) / 4), dim3(256), lds, st, q, kc, vc, rows,
                       nh, g, max_pos, seq_stride, scale, out, ls, fz);
    return hipGetLastError();
  };
  if (hd == 64) return fuse ? go(k_attention_wave<64, true>) : go(k_attention_wave<64, false>);
  return fuse ? go(k_attention_wave<128, true>) : go(k_attention_wave<128, false>);
}

hipError_t launch_rope_attention_rows(const float* q, const float* k, const float* v,
                                      const float* rope_cs, RowsDesc rows, uint32_t max_len,
                                      uint32_t nh, uint32_t nkv, uint32_t hd, uint32_t max_pos,
                                      float* kc, float* vc, uint64_t seq_stride, float scale,
                                      float* out, bool tree, hipStream_t st) {
  if (rows.n == 0) return hipSuccess;
  if (max_len == 0 || max_len > max_pos || max_pos % 4 || hd % 2) return hipErrorInvalidValue;
  KvPlan kp;
  hipError_t e = kv_plan(rows.n, nh, nkv, hd, max_len, &kp);
  if (e != hipSuccess) return e;
  const KvFuse fz{k, v, rope_cs, nkv};
  if (!kp.C) {
    size_t lds;
    if (!wave_attention(rows.n, nh, nkv, hd, max_len, tree, &lds)) return hipErrorNotSupported;
    return launch_wave(true, q, kc, vc, rows, max_len, nh, nkv, hd, max_pos, seq_stride, scale,
                       out, lds, fz, st);
  }
  return launch_kv(kp, true, q, kc, vc, rows, nh, hd, max_pos, seq_stride, scale, out, tree, fz,
                   st);
}

// LDS of k_attention_rows with hpw heads per workgroup, and its limit.
static size_t attention_rows_lds(uint32_t hpw, uint32_t hd, uint32_t max_len) {
  const size_t hd4 = ((size_t)hd + 3) / 4 * 4, ls = ((size_t)max_len + 3) / 4 * 4;
  return hpw * (hd4 + ls + (ls + 31) / 32) * sizeof(float);
}
constexpr size_t kAttRowsLds = 60 * 1024;
bool attention_rows_fit(uint32_t hd, uint32_t max_len) {
  return attention_rows_lds(1, hd, max_len) <= kAttRowsLds;
}

hipError_t launch_attention_rows(const float* q, const float* kc, const float* vc,
                                 RowsDesc rows, uint32_t max_len, uint32_t nh, uint32_t nkv,
                                 uint32_t hd, uint32_t max_pos, uint64_t seq_stride, float scale,
                                 float* out, bool tree, hipStream_t st) {
  if (rows.n == 0) return hipSuccess;
  if (nkv == 0 || nh % nkv || max_len == 0 || max_len > max_pos || max_pos % 4)
    return hipErrorInvalidValue;
  const uint32_t group = nh / nkv;
  const int ncu = device_cu_count();
  const uint64_t wgs_kv = (uint64_t)rows.n * nkv;
  const uint32_t tr = tree ? 1u : 0u, ls = (max_len + 3) / 4 * 4;
  {
    KvPlan kp;
    hipError_t e = kv_plan(rows.n, nh, nkv, hd, max_len, &kp);
    if (e != hipSuccess) return e;
    if (kp.C) return launch_kv(kp, false, q, const_cast<float*>(kc), const_cast<float*>(vc),
                               rows, nh, hd, max_pos, seq_stride, scale, out, tree, KvFuse{}, st);
    size_t lds;
    if (wave_attention(rows.n, nh, nkv, hd, max_len, tree, &lds))
      return launch_wave(false, q, const_cast<float*>(kc), const_cast<float*>(vc), rows, max_len,
                         nh, nkv, hd, max_pos, seq_stride, scale, out, lds, KvFuse{}, st);
  }
  // Otherwise, few rows: one head per workgroup, for the most workgroups.
  // Many rows: the most heads of one KV head (a divisor of the group) whose
  // LDS fits, so K and V are read once per group.
  uint32_t hpw = 1;
  if (wgs_kv >= 4 * (uint64_t)ncu) {
    for (uint32_t h = std::min(group, kMaxHeadsPerWg); h > 1; --h)
      if (group % h == 0 && attention_rows_lds(h, hd, max_len) <= kAttRowsLds) {
        hpw = h;
        break;
      }
  }
  const size_t shmem = attention_rows_lds(hpw, hd, max_len);
  if (shmem > kAttRowsLds) return hipErrorInvalidValue;
  const dim3 grid(rows.n, nh / hpw);
  switch (hpw) {
    case 4:
      hipLaunchKernelGGL(k_attention_rows<4>, grid, dim3(kAttT), shmem, st, q, kc, vc, rows, nh,
                         nkv, hd, max_pos, seq_stride, scale, out, tr, ls);
      break;
    case 3:
      hipLaunchKernelGGL(k_attention_rows<3>, grid, dim3(kAttT), shmem, st, q, kc, vc, rows, nh,
                         nkv, hd, max_pos, seq_stride, scale, out, tr, ls);
      break;
    case 2:
      hipLaunchKernelGGL(k_attention_rows<2>, grid, dim3(kAttT), shmem, st, q, kc, vc, rows, nh,
                         nkv, hd, max_pos, seq_stride, scale, out, tr, ls);
      break;
    default:
      hipLaunchKernelGGL(k_attention_rows<1>, grid, dim3(kAttT), shmem, st, q, kc, vc, rows, nh,
                         nkv, hd, max_pos, seq_stride, scale, out, tr, ls);
  }
  return hipGetLastError();
}

hipError_t launch_gather_rows(const float* src, const uint32_t* idx, uint32_t n, uint32_t width,
                              float* dst, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_gather_rows, dim3(n), dim3(kT), 0, st, src, idx, width, dst);
  return hipGetLastError();
}

hipError_t launch_advance_rows(uint32_t* pos, uint32_t n, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_advance_rows, dim3((n + kT - 1) / kT), dim3(kT), 0, st, pos, n);
  return hipGetLastError();
}

hipError_t launch_argmax_rows(const float* v, uint32_t n, uint32_t width, uint32_t* out,
                              hipStream_t st) {
  if (n == 0) return hipSuccess;
  if (width == 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_argmax_rows, dim3(n), dim3(1024), 0, st, v, width, out);
  return hipGetLastError();
}


// Workgroups of k_attention_tiles: two per CU (its registers), a multiple of
// eight, no more than the items need.
static uint32_t att_tiles_grid(uint64_t nitem) {
  const uint64_t most = (2 * (uint64_t)device_cu_count() + 7) / 8 * 8;
  return (uint32_t)std::min<uint64_t>(most, (nitem + 7) / 8 * 8);
}
// Query heads per item: those of one KV head share its K and V loads where
// that leaves enough items for two workgroups per CU, else one.  At head_dim
// 128 up to three (four spilled registers), in tree order up to two (three).
static uint32_t att_tiles_heads(uint32_t ntiles, uint32_t nh, uint32_t nkv, uint32_t hd,
                                bool tree) {
  const uint32_t group = nh / nkv, ncu = (uint32_t)device_cu_count();
  for (uint32_t h = std::min(group, tree ? 2u : (hd == 64 ? 4u : 3u)); h > 1; --h)
    if (group % h == 0 && (uint64_t)ntiles * (nh / h) >= 2 * (uint64_t)ncu) return h;
  return 1;
}

template <uint32_t HPT, uint32_t HD, bool TREE>
static hipError_t launch_att_tiles_t(const float* q, const float* kc, const float* vc,
                                     const AttTile* tiles, uint32_t ntiles, uint32_t nh,
                                     uint32_t group, uint32_t max_pos, uint64_t seq_stride,
                                     float scale, float* out, float* scratch, uint32_t ls,
                                     hipStream_t st) {
  const size_t lds = AttTileCfg<HPT>::floats(HD) * sizeof(float);
  hipError_t e = ensure_dynamic_lds(reinterpret_cast<const void*>(&k_attention_tiles<HPT, HD, TREE>), lds);
  if (e != hipSuccess) return e;
  const uint64_t nitem = (uint64_t)ntiles * (nh / HPT);
  if (nitem > 0x7fffffffu) return hipErrorInvalidValue;
  hipLaunchKernelGGL((k_attention_tiles<HPT, HD, TREE>), dim3(att_tiles_grid(nitem)), dim3(256), lds, st,
                     q, kc, vc, tiles, (uint32_t)nitem, nh, group, max_pos, seq_stride, scale, out,
                     scratch, ls);
  return hipGetLastError();
}

bool attention_tiles_supported(uint32_t nh, uint32_t nkv, uint32_t hd) {
  return nkv != 0 && nh % nkv == 0 && (hd == 64 || hd == 128);
}

size_t attention_tiles_scratch_floats(uint32_t ntiles, uint32_t nh, uint32_t nkv, uint32_t hd,
                                      uint32_t max_len, bool tree) {
  const size_t ls = ((size_t)max_len + 3) / 4 * 4;
  const uint32_t h = att_tiles_heads(ntiles, nh, nkv, hd, tree);
  return (size_t)att_tiles_grid((uint64_t)ntiles * (nh / h)) * kAttQT * h * ls;
}

hipError_t launch_attention_tiles(const float* q, const float* kc, const float* vc,
                                  const AttTile* tiles, uint32_t ntiles, uint32_t max_len,
                                  uint32_t nh, uint32_t nkv, uint32_t hd, uint32_t max_pos,
                                  uint64_t seq_stride, float scale, float* out, float* scratch,
                                  hipStream_t st, bool tree) {
  if (ntiles == 0) return hipSuccess;
  if (!attention_tiles_supported(nh, nkv, hd) || max_len == 0 || max_len > max_pos ||
      max_pos % 4)
    return hipErrorInvalidValue;
  const uint32_t g = nh / nkv, ls = (max_len + 3) / 4 * 4;
#define CIS2_ATT_TILES(H, D, TREE)                                                               \
  return launch_att_tiles_t<H, D, TREE>(q, kc, vc, tiles, ntiles, nh, g, max_pos, seq_stride,    \
                                        scale, out, scratch, ls, st)
  switch ((tree ? 10000 : 0) + att_tiles_heads(ntiles, nh, nkv, hd, tree) * 1000 + hd) {
    case 1064: CIS2_ATT_TILES(1, 64, false);
    case 2064: CIS2_ATT_TILES(2, 64, false);
    case 3064: CIS2_ATT_TILES(3, 64, false);
    case 4064: CIS2_ATT_TILES(4, 64, false);
    case 1128: CIS2_ATT_TILES(1, 128, false);
    case 2128: CIS2_ATT_TILES(2, 128, false);
    case 3128: CIS2_ATT_TILES(3, 128, false);
    case 11064: CIS2_ATT_TILES(1, 64, true);
    case 12064: CIS2_ATT_TILES(2, 64, true);
    case 11128: CIS2_ATT_TILES(1, 128, true);
    case 12128: CIS2_ATT_TILES(2, 128, true);
    default: return hipErrorInvalidValue;
  }
#undef CIS2_ATT_TILES
}

}  // namespace cis2
