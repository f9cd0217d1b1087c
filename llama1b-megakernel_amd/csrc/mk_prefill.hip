// mk_prefill.hip — context encoding (prefill) of one sequence, layer by layer,
// on the matrix cores of MI355X (gfx950).
//
// The reference encodes a prompt with its baseline decoder layers before the
// megakernel takes over token generation (llama_with_megakernel.py:194-204;
// the layer is llama.py:1039-1139). With T prompt tokens the step is T rows
// of GEMMs against every layer's weights, so it runs layer-major: each layer's
// weights stream once per chunk of up to `cap` tokens (the decode megakernel
// would stream them once per token, and its batched prefill once per 32).
//
// Per layer (all launches on the caller's stream, in order):
//   pf_norm   x -> xn = bf16(x * rsqrt(mean(x^2) + eps))      (layer 0: x = embed[token])
//   pf_gemm   QKV: xn W_qkv^T, bf16, RoPE on (d, d+32) pairs -> q; K/V rows -> the caches
//   pf_attn   causal GQA attention of every token over cache rows [0, pos] -> att
//   pf_gemm   O:    att W_o^T  + x  -> h1                       (bf16 residual add)
//   pf_norm   h1 -> xn
//   pf_gemm   GU:   xn W_gu^T, bf16(silu(g) * u) -> act
//   pf_gemm   DOWN: act W_d^T + h1 -> x (the next layer's input)
// The rounding points are those of the decode kernels (the reference's
// attention.py / mlp.py). The last layer runs only its QKV GEMM (its K/V
// rows are the prefill's output) unless the caller asks for the hidden state.
//
// GEMMs (pf_gemm): bf16 v_mfma_f32_16x16x32_bf16 with fp32 accumulation. The
// activations are kept in A-tile order (the producing kernel writes them so)
// and the weights are the MFMA-tiled copies, so each k-step's operands of an
// output tile are blocks of 1 KiB that go from memory straight into LDS. The
// tile (64x64 to 256x256) and, for short prompts, a split of K into fp32
// partials are chosen per projection by estimated time (gemm_plan); the
// partials are summed in a fixed order by pf_reduce_norm (O and down) and
// pf_qkv_finish (QKV, with RoPE and the scatter).
//
// Attention: per (kv head, block of 16 tokens) one workgroup; S^T = K Q^T on
// the matrix cores (keys on M, the 16 tokens x 4 q heads on N), an online
// softmax per (token, head) column, and O^T = V^T P^T on the matrix cores with
// p rounded to bf16 as the reference rounds it (relative to the running
// maximum). K and V tiles of 32 keys go through LDS (V transposed there).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include "mk.h"
#include "mk_common.h"
#include "mk_prefill.h"

namespace {

using namespace mk;

constexpr int PF_TB = 16;                 // tokens per attention workgroup

enum : int { EPI_QKV = 0, EPI_RES = 1, EPI_SWIGLU = 2, EPI_PART = 3 };

struct GemmArgs {
  const uint16_t* a;     // activations, A-tile order [M16][K]
  const uint16_t* b;     // weights [N][K]: MFMA tile order (tiled) or row-major
  int tiled;
  int M, N, K;
  int mt;                // row tiles
  int splits;            // EPI_PART: the K range is cut into `splits` parts (blockIdx.y)
  const uint16_t* res;   // EPI_RES: residual, row-major [M][N]
  uint16_t* out;         // EPI_RES: row-major [M][N]; EPI_SWIGLU: A-tile order [M16][N/2]; EPI_QKV: q [M][2048]
  float* part;           // EPI_PART: fp32 [splits][M][N]
  uint16_t* kc;          // EPI_QKV: the layer's caches, bf16 [8][s_max][64]
  uint16_t* vc;
  const uint16_t* rope;  // bf16 [rows][128]
  int s_max, p0;
};

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// This wave's copies up to the last N have landed and its LDS reads up to the
// last R have returned, and so have every wave's.
template <int N, int R>
__device__ __forceinline__ void wait_copies() {
  static_assert(N < 64 && R < 16, "wait counts");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(%1)\n\ts_barrier" ::"n"(N), "n"(R) : "memory");
}

// C = A B^T, one (16 MI WM) x (16 NI WN) output tile per workgroup of WM x WN
// waves, 16 MI x 16 NI of it per wave.
//
// What bounds it: a k-step of 32 columns costs the tile's MFMAs (16 cycles
// each), the copies of its operands into the CU (64 B/cycle) and their traffic
// through LDS (128 B/cycle, written once and read by every wave that uses them).
// A 128x128 tile of 64x64 per wave (the only one before) takes 256 cycles of
// each at one wave per SIMD and got 770-850 TFLOP/s; 256x256 on eight waves of
// 128x64 halves the copies per MFMA and puts two waves on a SIMD, so that one
// multiplies while the other waits: 16384 x 2048 weights at 3000 tokens 208 ->
// 147 us (1370 TFLOP/s). Smaller tiles serve the shapes that would leave the
// device idle (gemm_plan).
//
// Operands are 1 KiB blocks (16 rows x 32 columns) copied from memory straight
// into a ring of NS k-steps in LDS, NS - 1 ahead; each wave reads the next
// k-step's operands into registers while it multiplies the current one
// (interleaved one read per few MFMAs; without that 1180 instead of 1370).
// Copies past the operands (k-steps >= ke, rows past the matrix) write zeros
// from out-of-range offsets: the count in flight stays fixed, so waits count.
//
// The weights are the MFMA's first operand and the tokens the second, so a lane
// holds four consecutive columns of one token: pairs (gate, up) and (d, d + 32)
// meet in a lane, and rows leave through the wave's LDS as 16-byte pieces. The
// 2-byte stores of the transposed form took 14 us per round of 256x256 tiles.
template <int EPI, int MI, int NI, int WM, int WN, int NS>
__global__ void __launch_bounds__(64 * WM * WN, 2) pf_gemm(GemmArgs g) {
  constexpr int NW = WM * WN, AB = MI * WM, BB = NI * WN, NB = AB + BB;   // waves; A, B and all blocks of a k-step
  constexpr int CPW = (NB + NW - 1) / NW;                                // copies per wave and k-step
  constexpr bool SPARE = NB % NW != 0;                                   // the last wave's surplus copies
  constexpr int EROW = 16 * NI * 2 + 16;                                 // bytes of a staged output row (padded)
  static_assert(NS >= 3 && 16 * EROW * NW <= NS * NB * 1024, "operand ring; staged outputs fit in it");
  __shared__ u32x4 L[(NS * NB + (SPARE ? 1 : 0)) * 64];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;   // (uniform: LDS copy bases)
  // Workgroup w runs on XCD w % 8: each XCD gets a contiguous range of tiles,
  // rows first, so the workgroups that share weight columns share its L2.
  const int nt = g.N / (16 * BB), total = g.mt * nt;
  const int xcd = blockIdx.x & 7, q8 = total >> 3, r8 = total & 7;
  const int tile = xcd * q8 + min(xcd, r8) + ((int)blockIdx.x >> 3);
  const int tm = tile % g.mt, tn = tile / g.mt;
  const int m16 = (g.M + 15) / 16, kb = g.K / 32;
  const rsrc_t ra = make_rsrc(g.a, (size_t)m16 * 16 * g.K * 2);
  const rsrc_t rb = make_rsrc(g.b, (size_t)g.N * g.K * 2);
  // the k-steps of this workgroup: all of K, or part blockIdx.y of `splits` (an even number)
  const int kn = EPI == EPI_PART ? kb / g.splits : kb;
  const int k0 = EPI == EPI_PART ? (int)blockIdx.y * kn : 0, ke = k0 + kn;
  // this wave's blocks of a k-step: wave * CPW + u of the A blocks, then the B blocks
  const uint32_t bstep = g.tiled ? 1024u : 64u;
  const uint32_t arow = (uint32_t)(lane * 16);
  const uint32_t brow = g.tiled ? arow : (uint32_t)((lane & 15) * g.K * 2 + (lane >> 4) * 16);
  uint32_t off[CPW];
#pragma unroll
  for (int u = 0; u < CPW; ++u) {
    const int c = wave * CPW + u;
    off[u] = c < AB ? arow + (uint32_t)(tm * AB + c) * (uint32_t)kb * 1024u
                    : brow + (uint32_t)(tn * BB + c - AB) * (uint32_t)kb * 1024u;
    if (SPARE && c >= NB) off[u] = OOB;
  }
  auto issue = [&](int ks, int stg) {
    const bool in = ks < ke;
    const uint32_t sa = in ? (uint32_t)ks * 1024u : 0u, sb = in ? (uint32_t)ks * bstep : 0u;
#pragma unroll
    for (int u = 0; u < CPW; ++u) {
      const int c = wave * CPW + u;
      const lds_ptr_t dst = (lds_ptr_t)&L[(SPARE && c >= NB ? NS * NB : stg * NB + c) * 64];
      const uint32_t vo = in ? off[u] : OOB;
      if (c < AB) __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, dst, 16, vo, sa, 0, 0);
      else __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, dst, 16, vo, sb, 0, 0);
    }
  };
  // wave (wm, wn) computes rows 16 MI wm .. and columns 16 NI wn .. of the tile
  const int wm = wave % WM, wn = wave / WM;
  f32x4 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 av[2][MI], bv[2][NI];
  auto read = [&](int stg, u32x4(&a)[MI], u32x4(&b)[NI]) {
    const u32x4* S = &L[stg * NB * 64 + lane];
#pragma unroll
    for (int i = 0; i < MI; ++i) a[i] = S[(MI * wm + i) * 64];
#pragma unroll
    for (int j = 0; j < NI; ++j) b[j] = S[(AB + NI * wn + j) * 64];
  };
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) issue(k0 + s, s);
  int stg = 0, fill = NS - 1;
  wait_copies<(NS - 2) * CPW, 0>();
  read(0, av[0], bv[0]);
  for (int ks = k0; ks < ke; ks += 2) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      // k-step ks + s + 1 is in LDS, and every wave has read the stage refilled
      // next (k-step ks + s - 1's; the MI + NI reads since are ks + s's)
      wait_copies<(NS - 3) * CPW, MI + NI>();
      issue(ks + s + NS - 1, fill);
      fill = stg;
      stg = stg + 1 == NS ? 0 : stg + 1;
      read(stg, av[s ^ 1], bv[s ^ 1]);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = mfma16(bv[s][j], av[s][i], acc[i][j]);
      // one LDS read, then its share of the MFMAs
      constexpr int R = MI + NI, MM = MI * NI, Q = MM / R, X = MM % R;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        if (i < X) __builtin_amdgcn_sched_group_barrier(0x008, Q + 1, 0);
        else if (Q) __builtin_amdgcn_sched_group_barrier(0x008, Q, 0);
      }
    }
  }

  // the ring is free once every wave has read its last operands and its trailing
  // copies have landed; each wave then stages its rows in a part of its own
  wait_copies<0, 0>();

  // epilogue: acc[i][j][r] is (row m0(i) + lane%16, column n0 + 16j + 4*(lane/16) + r)
  const int n0 = 16 * (tn * BB + NI * wn), mw = 16 * (tm * AB + MI * wm);
  const int lm = lane & 15, lq = lane >> 4;
  if constexpr (EPI == EPI_PART) {
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int m = mw + 16 * i + lm;
      if (m < g.M)
#pragma unroll
        for (int j = 0; j < NI; ++j)
          *reinterpret_cast<f32x4*>(g.part + ((size_t)blockIdx.y * g.M + m) * g.N + n0 + 16 * j + 4 * lq) = acc[i][j];
    }
    return;
  }
  // (a wave's LDS accesses complete in order; lds_order keeps the compiler's order)
  auto lds_order = [] { asm volatile("" ::: "memory"); };
  char* my = reinterpret_cast<char*>(L) + wave * 16 * EROW;
  if constexpr (EPI == EPI_SWIGLU) {
    // columns (gate_i, up_i) interleaved: 8 outputs of a token per 16 columns, a
    // 16-byte slot of the A-tile block (16 tokens x 32 outputs) that 64 columns fill
    const int kbo = g.N / 64;   // blocks per row of tiles of the output
    char* out = reinterpret_cast<char*>(g.out) + (size_t)(n0 / 64) * 1024 + (size_t)(n0 % 64) * 16;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const f32x4 v = acc[i][j];
        *reinterpret_cast<uint32_t*>(my + (j * 16 + lm) * 16 + lq * 4) =
            pack_bf2(v[0] / (1.0f + __expf(-v[0])) * v[1], v[2] / (1.0f + __expf(-v[2])) * v[3]);
      }
      lds_order();
      const int m0 = mw + 16 * i;
      if (m0 < g.M && lane < 16 * NI)   // (rows past M of the last block: padding of the buffer)
        *reinterpret_cast<u32x4*>(out + (size_t)(m0 >> 4) * kbo * 1024 + lane * 16) =
            *reinterpret_cast<const u32x4*>(my + lane * 16);
      lds_order();
    }
  } else {
    constexpr int PR = 2 * NI, RP = 64 / PR, NP = 16 / RP;   // 16-byte pieces per row, rows per pass, passes
    const int pc = lane % PR, pr = lane / PR;
    // QKV: the wave's columns belong to one head (64 columns, RoPE pairs (d, d + 32))
    const int head = n0 >> 6, d = (n0 & 63) / 2 + 4 * pc;
    const bool rot = head < NQ + NKV;
    // the epilogue's side input of up to CI row blocks in flight at once
    constexpr int CI = MI < 4 ? MI : 4;
    u32x4 side[EPI == EPI_RES ? CI * NP : 1];
    uint2 rp[EPI == EPI_QKV ? CI * NP : 1][4];
    auto load_side = [&](int i0) {
#pragma unroll
      for (int i = i0; i < i0 + CI && i < MI; ++i)
#pragma unroll
        for (int k = 0; k < NP; ++k) {
          const int m = mw + 16 * i + k * RP + pr, at = (i - i0) * NP + k;
          if constexpr (EPI == EPI_RES) {
            side[at] = u32x4{0u, 0u, 0u, 0u};
            if (m < g.M) side[at] = *reinterpret_cast<const u32x4*>(g.res + (size_t)m * g.N + n0 + 8 * pc);
          } else if (rot && m < g.M) {
            const uint16_t* rrow = g.rope + (size_t)(g.p0 + m) * (2 * HD) + d;   // cos[d], cos[d+32], sin[d], sin[d+32]
#pragma unroll
            for (int e = 0; e < 4; ++e) rp[at][e] = *reinterpret_cast<const uint2*>(rrow + 32 * e);
          }
        }
    };
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      if (i % CI == 0) load_side(i);
#pragma unroll
      for (int j = 0; j < NI; ++j)
        *reinterpret_cast<uint2*>(my + lm * EROW + j * 32 + lq * 8) =
            uint2{pack_bf2(acc[i][j][0], acc[i][j][1]), pack_bf2(acc[i][j][2], acc[i][j][3])};
      lds_order();
#pragma unroll
      for (int k = 0; k < NP; ++k) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(my + (k * RP + pr) * EROW + pc * 16);
        const int m = mw + 16 * i + k * RP + pr;
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        if constexpr (EPI == EPI_RES) {
          const u32x4 r = side[i % CI * NP + k];
          const uint32_t rw[4] = {r.x, r.y, r.z, r.w};
          uint32_t o[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = pack_bf2(bf_lo(rw[e]) + bf_lo(w[e]), bf_hi(rw[e]) + bf_hi(w[e]));
          if (m < g.M) *reinterpret_cast<u32x4*>(g.out + (size_t)m * g.N + n0 + 8 * pc) = u32x4{o[0], o[1], o[2], o[3]};
        } else if (m < g.M) {
          float lo[4], hi[4];   // dims d .. d + 3 and d + 32 .. d + 35
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            lo[e] = bf_lo(w[e]);
            hi[e] = bf_hi(w[e]);
          }
          if (rot) {
            const uint2* R = rp[i % CI * NP + k];
            const uint32_t c0[2] = {R[0].x, R[0].y}, c1[2] = {R[1].x, R[1].y};
            const uint32_t s0[2] = {R[2].x, R[2].y}, s1[2] = {R[3].x, R[3].y};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float a = lo[e], b = hi[e];
              const float ca = e & 1 ? bf_hi(c0[e >> 1]) : bf_lo(c0[e >> 1]), sa = e & 1 ? bf_hi(s0[e >> 1]) : bf_lo(s0[e >> 1]);
              const float cb = e & 1 ? bf_hi(c1[e >> 1]) : bf_lo(c1[e >> 1]), sb = e & 1 ? bf_hi(s1[e >> 1]) : bf_lo(s1[e >> 1]);
              lo[e] = rbf(rbf(a * ca) + rbf(-b * sa));
              hi[e] = rbf(rbf(b * cb) + rbf(a * sb));
            }
          }
          uint16_t* dst;
          if (head < NQ) dst = g.out + (size_t)m * H + head * HD;
          else if (rot) dst = g.kc + ((size_t)(head - NQ) * g.s_max + g.p0 + m) * HD;
          else dst = g.vc + ((size_t)(head - NQ - NKV) * g.s_max + g.p0 + m) * HD;
          *reinterpret_cast<uint2*>(dst + d) = uint2{pack_bf2(lo[0], lo[1]), pack_bf2(lo[2], lo[3])};
          *reinterpret_cast<uint2*>(dst + d + 32) = uint2{pack_bf2(hi[0], hi[1]), pack_bf2(hi[2], hi[3])};
        }
      }
      lds_order();
    }
  }
}

// The split-K tail of the O and down projections (N = 2048), one workgroup per
// token row t, 8 columns per thread: v = the sum of the SPLITS fp32 partials in
// split order, out = bf16(res + bf16(v)) (row-major), and, if xn is given, the
// next RMSNorm of out into xn (A-tile order), as pf_norm computes it. Latency
// bounds it: every load of the row is in flight at once (33 tokens of 16 splits
// on one wave per row, four rounds of loads: 9.4 us).
template <int SPLITS>
__global__ void __launch_bounds__(NT) pf_reduce_norm(const float* part, const uint16_t* res, uint16_t* out,
                                                     uint16_t* xn, int T) {
  static_assert(H == 8 * NT, "8 columns per thread");
  __shared__ float sums[NWAVE];
  const int t = blockIdx.x, c = (int)threadIdx.x * 8;
  float4 pv[SPLITS][2];
#pragma unroll
  for (int sp = 0; sp < SPLITS; ++sp) {
    const float4* pp = reinterpret_cast<const float4*>(part + ((size_t)sp * T + t) * H + c);
    pv[sp][0] = pp[0];
    pv[sp][1] = pp[1];
  }
  const u32x4 rv = *reinterpret_cast<const u32x4*>(res + (size_t)t * H + c);
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int sp = 0; sp < SPLITS; ++sp) {
    const float4 p0 = pv[sp][0], p1 = pv[sp][1];
    v[0] += p0.x; v[1] += p0.y; v[2] += p0.z; v[3] += p0.w;
    v[4] += p1.x; v[5] += p1.y; v[6] += p1.z; v[7] += p1.w;
  }
  const uint32_t rw[4] = {rv.x, rv.y, rv.z, rv.w};
  uint32_t o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = pack_bf2(bf_lo(rw[e]) + rbf(v[2 * e]), bf_hi(rw[e]) + rbf(v[2 * e + 1]));
  *reinterpret_cast<u32x4*>(out + (size_t)t * H + c) = u32x4{o[0], o[1], o[2], o[3]};
  if (!xn) return;
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) ss = fmaf(bf_hi(o[e]), bf_hi(o[e]), fmaf(bf_lo(o[e]), bf_lo(o[e]), ss));
  ss = wave_sum(ss);
  if (lane_id() == 0) sums[wave_id()] = ss;
  __syncthreads();
  const float inv = rsqrtf(((sums[0] + sums[1]) + (sums[2] + sums[3])) * (1.0f / H) + EPS);
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = cvt_bf2(bf_lo(o[e]) * inv, bf_hi(o[e]) * inv);
  *reinterpret_cast<u32x4*>(xn + a_tile_off(t, c, H / 32)) = u32x4{o[0], o[1], o[2], o[3]};
}

// The split-K tail of the QKV projection of short prompts (N = 3072): thread
// (t, j) takes RoPE pairs 2j and 2j + 1 of token row t, i.e. columns 4j .. 4j + 3
// (dims d, d + 32, d + 1, d + 33 of one head, d = 2j mod 32), in one 16-byte
// load per split: each column summed over the SPLITS fp32 partials in split
// order and rounded to bf16, RoPE on the q and k pairs as the QKV GEMM's
// epilogue does it, q to the q buffer and k and v to the caches at row
// p0 + t, two bf16 per 4-byte store. Grid (T, QKV_PAIRS / 2 / NT).
template <int SPLITS>
__global__ void __launch_bounds__(NT) pf_qkv_finish(const float* part, const uint16_t* rope, uint16_t* q,
                                                    uint16_t* kc, uint16_t* vc, int T, int p0, int s_max) {
  const int t = blockIdx.x, j = blockIdx.y * NT + (int)threadIdx.x;
  if (t >= T || j >= QKV_PAIRS / 2) return;
  const int pos = p0 + t, pr = 2 * j, hp = pr & 31;
  float4 pv[SPLITS];
#pragma unroll
  for (int sp = 0; sp < SPLITS; ++sp)
    pv[sp] = *reinterpret_cast<const float4*>(part + ((size_t)sp * T + t) * QKV_ROWS + 4 * j);
  float v0 = 0.f, v1 = 0.f, v2 = 0.f, v3 = 0.f;
#pragma unroll
  for (int sp = 0; sp < SPLITS; ++sp) {
    v0 += pv[sp].x;
    v1 += pv[sp].y;
    v2 += pv[sp].z;
    v3 += pv[sp].w;
  }
  // pair 2j: (x[d], x[d + 32]) = (a0, b0); pair 2j + 1: (x[d + 1], x[d + 33]) = (a1, b1)
  const float a0 = rbf(v0), b0 = rbf(v1), a1 = rbf(v2), b1 = rbf(v3);
  float o00 = a0, o01 = b0, o10 = a1, o11 = b1;
  if (pr < Q_PAIRS + K_PAIRS) {
    const uint16_t* rrow = rope + (size_t)pos * (2 * HD);
    const uint32_t c0 = *reinterpret_cast<const uint32_t*>(rrow + hp);            // cos[d], cos[d + 1]
    const uint32_t s0 = *reinterpret_cast<const uint32_t*>(rrow + HD + hp);       // sin[d], sin[d + 1]
    const uint32_t c1 = *reinterpret_cast<const uint32_t*>(rrow + hp + 32);       // cos[d + 32], ...
    const uint32_t s1 = *reinterpret_cast<const uint32_t*>(rrow + HD + hp + 32);  // sin[d + 32], ...
    o00 = rbf(rbf(a0 * bf_lo(c0)) + rbf(-b0 * bf_lo(s0)));
    o01 = rbf(rbf(b0 * bf_lo(c1)) + rbf(a0 * bf_lo(s1)));
    o10 = rbf(rbf(a1 * bf_hi(c0)) + rbf(-b1 * bf_hi(s0)));
    o11 = rbf(rbf(b1 * bf_hi(c1)) + rbf(a1 * bf_hi(s1)));
  }
  uint16_t* dst;
  if (pr < Q_PAIRS) dst = q + (size_t)t * H + (pr >> 5) * HD;
  else if (pr < Q_PAIRS + K_PAIRS) dst = kc + ((size_t)((pr - Q_PAIRS) >> 5) * s_max + pos) * HD;
  else dst = vc + ((size_t)((pr - Q_PAIRS - K_PAIRS) >> 5) * s_max + pos) * HD;
  *reinterpret_cast<uint32_t*>(dst + hp) = pack_bf2(o00, o10);
  *reinterpret_cast<uint32_t*>(dst + hp + 32) = pack_bf2(o01, o11);
}

// xn (A-tile order [T16][2048]) = bf16(x * rsqrt(mean(x^2) + eps)) per token
// row, one wave per token; with `tokens`, x is the embedding row of the token
// and is also copied to x_out (row-major) as the first residual.
__global__ void __launch_bounds__(NT) pf_norm(const uint16_t* x, const int32_t* tokens, const uint16_t* embed,
                                              uint16_t* x_out, uint16_t* xn, int T) {
  const int t = blockIdx.x * NWAVE + wave_id(), lane = lane_id();
  if (t >= T) return;
  const uint16_t* src = x + (size_t)t * H;
  if (tokens) {
    int tok = tokens[t];
    tok = tok < 0 ? 0 : (tok >= VOCAB ? VOCAB - 1 : tok);
    src = embed + (size_t)tok * H;
  }
  u32x4 xs[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) xs[i] = *reinterpret_cast<const u32x4*>(src + i * 512 + lane * 8);
  if (tokens) {
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4*>(x_out + (size_t)t * H + i * 512 + lane * 8) = xs[i];
  }
  rmsnorm2048(xs, nullptr);
#pragma unroll
  for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4*>(xn + a_tile_off(t, i * 512 + lane * 8, H / 32)) = xs[i];
}

struct AttnArgs {
  const uint16_t* q;     // [T][2048] row-major, after RoPE
  const uint16_t* kc;    // the layer's caches bf16 [8][s_max][64]
  const uint16_t* vc;
  uint16_t* att;         // A-tile order [T16][2048]
  int T, p0, s_max;
};

constexpr int KS_STRIDE = HD + 8;   // K tile row in LDS (bf16): 144 bytes, rows on distinct banks
constexpr int VT_STRIDE = 32 + 4;   // transposed V tile row (one dim, 32 keys): 72 bytes

struct AttnLds {
  uint16_t k[2][32][KS_STRIDE];
  uint16_t vt[2][HD][VT_STRIDE];
};

// Token t of the sequence (position p0 + t) attends to cache rows [0, p0 + t],
// its own row included (written by the QKV GEMM before this launch).
__global__ void __launch_bounds__(NT) pf_attn(AttnArgs a) {
  __shared__ AttnLds L;
  const int tid = threadIdx.x, wave = wave_id(), lane = lane_id();
  const int nblk = (a.T + PF_TB - 1) / PF_TB;
  const int tb = nblk - 1 - (int)blockIdx.x;   // the longest blocks first
  const int g = blockIdx.y;                    // kv head
  const int t0 = tb * PF_TB;
  const int n_keys = a.p0 + min(t0 + PF_TB, a.T);
  // this lane's column: token t0 + 4*wave + (lane%16)/4, q head 4g + lane%4
  const int col = lane & 15, q4 = lane >> 4;
  const int tq = t0 + 4 * wave + (col >> 2);
  const int hq = GQA * g + (col & 3);
  const int lim = a.p0 + min(tq, a.T - 1);     // last key of the column (padding tokens: any finite row)
  const rsrc_t rq = make_rsrc(a.q, (size_t)a.T * H * 2);
  u32x4 qv[2];
#pragma unroll
  for (int s = 0; s < 2; ++s)
    qv[s] = ld16(rq, tq < a.T ? (uint32_t)(((size_t)tq * H + hq * HD + 32 * s + q4 * 8) * 2) : OOB);
  const rsrc_t rk = make_rsrc(a.kc + (size_t)g * a.s_max * HD, (size_t)a.s_max * HD * 2);
  const rsrc_t rv = make_rsrc(a.vc + (size_t)g * a.s_max * HD, (size_t)a.s_max * HD * 2);
  // staging of a 32-key block: thread t loads key row t/8, dims (t%8)*8 .. +7 of K and of V
  const int sr = tid >> 3, sc = tid & 7;
  auto load_blk = [&](int kb, u32x4& kk, u32x4& vv) {
    const int key = kb * 32 + sr;
    const uint32_t off = key < n_keys ? (uint32_t)((key * HD + sc * 8) * 2) : OOB;
    kk = ld16(rk, off);
    vv = ld16(rv, off);
  };
  auto store_blk = [&](int buf, const u32x4& kk, const u32x4& vv) {
    *reinterpret_cast<u32x4*>(&L.k[buf][sr][sc * 8]) = kk;
    const uint32_t w[4] = {vv.x, vv.y, vv.z, vv.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      L.vt[buf][sc * 8 + 2 * e][sr] = (uint16_t)(w[e] & 0xffffu);
      L.vt[buf][sc * 8 + 2 * e + 1][sr] = (uint16_t)(w[e] >> 16);
    }
  };
  const int nb = (n_keys + 31) / 32;
  {
    u32x4 kk, vv;
    load_blk(0, kk, vv);
    store_blk(0, kk, vv);
  }
  __syncthreads();
  f32x4 acc[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;
  for (int kb = 0; kb < nb; ++kb) {
    const int buf = kb & 1;
    u32x4 kk, vv;
    const bool more = kb + 1 < nb;
    if (more) load_blk(kb + 1, kk, vv);
    // S^T: keys 16*ks + 4*q4 + i of the block, this lane's column
    float sc4[2][4];
    float mb = -INFINITY;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int sd = 0; sd < 2; ++sd) {
        const u32x4 ko = *reinterpret_cast<const u32x4*>(&L.k[buf][16 * ks + col][32 * sd + q4 * 8]);
        s = mfma16(ko, qv[sd], s);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = kb * 32 + 16 * ks + 4 * q4 + i;
        const float v = key <= lim ? s[i] * SM_SCALE : -INFINITY;
        sc4[ks][i] = v;
        mb = fmaxf(mb, v);
      }
    }
    mb = max_xor32(max_xor16(mb));          // the column's maximum over the 32 keys
    const float m_new = fmaxf(m_run, mb);   // finite: key 0 is in every column's range
    const float alpha = __expf(m_run - m_new);
    m_run = m_new;
    float ps = 0.f;
    float p[2][4];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[ks][i] = __expf(sc4[ks][i] - m_new);
        ps += p[ks][i];
      }
    l_run = l_run * alpha + ps;
    // P^T as the B operand: k-slots 8*q4 .. +7 of lane (q4, col) are the keys
    // 4*q4 + i and 16 + 4*q4 + i it holds (the V^T operand uses the same key order)
    const u32x4 pb = {cvt_bf2(p[0][0], p[0][1]), cvt_bf2(p[0][2], p[0][3]), cvt_bf2(p[1][0], p[1][1]),
                      cvt_bf2(p[1][2], p[1][3])};
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const uint16_t* vrow = &L.vt[buf][16 * d + col][0];
      const uint2 lo = *reinterpret_cast<const uint2*>(vrow + 4 * q4);
      const uint2 hi = *reinterpret_cast<const uint2*>(vrow + 16 + 4 * q4);
      const u32x4 vo = {lo.x, lo.y, hi.x, hi.y};
      f32x4 c = acc[d];
#pragma unroll
      for (int i = 0; i < 4; ++i) c[i] *= alpha;
      acc[d] = mfma16(vo, pb, c);
    }
    if (more) store_blk(buf ^ 1, kk, vv);
    __syncthreads();
  }
  // the column's sum over its four lanes; o = acc / l, dims 16d + 4*q4 + i
  const float l_tot = add_xor32(add_xor16(l_run));
  const float inv = 1.0f / l_tot;
  if (tq < a.T) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int dim = 16 * d + 4 * q4;
      uint2 w;
      w.x = pack_bf2(acc[d][0] * inv, acc[d][1] * inv);
      w.y = pack_bf2(acc[d][2] * inv, acc[d][3] * inv);
      *reinterpret_cast<uint2*>(a.att + a_tile_off(tq, hq * HD + dim, H / 32)) = w;
    }
  }
}

size_t ws_per_token() { return (size_t)H * 2 * 5 + (size_t)INTER * 2; }
// fp32 partials of a split-K projection: splits * M * N floats in all
constexpr size_t PART_BYTES = (size_t)2048 * H * 4;

// The output tiles pf_gemm is built for: rows, columns, and the time of a
// launch, fixed + rounds * (round + kstep * k-steps) in us, with one round per
// 256 workgroups (in fractions above one for the 64x64 tile, three of which
// share a CU): fitted to launches with weights not in cache over 26 row counts
// from 16 to 4096 by the four projections' shapes by 1-16 splits (rms error
// 5-13%). Choosing by it gives up 2% on average against the fastest of nine
// tiles. (The fixed and round parts are fits, not durations.)
struct GemmTile {
  int tm, tn;
  float fixed, round, kstep;
};
constexpr GemmTile TILES[] = {{64, 64, 2.73f, 0.50f, 0.13f},    {128, 128, 0.34f, 5.07f, 0.24f},
                              {192, 128, -1.88f, 8.42f, 0.32f}, {256, 128, -0.94f, 10.66f, 0.37f},
                              {192, 128, 8.99f, -0.77f, 0.33f}, {160, 256, 0.30f, 10.96f, 0.45f},
                              {256, 256, -2.26f, 19.51f, 0.54f}};
// (built with every epilogue up to here: the others hardly ever win for N = 2048, or with K split)
constexpr int TILES_RES = 4, TILES_PART = 3, TILES_ALL = sizeof(TILES) / sizeof(TILES[0]);

template <int EPI, int MI, int NI, int WM, int WN, int NS>
void gemm_launch(const GemmArgs& g, const GemmTile& t, hipStream_t st) {
  hipLaunchKernelGGL((pf_gemm<EPI, MI, NI, WM, WN, NS>), dim3(g.mt * (g.N / t.tn), g.splits), dim3(64 * WM * WN), 0, st,
                     g);
}
template <int EPI>
void gemm_run(GemmArgs g, int tile, hipStream_t st) {
  const GemmTile& t = TILES[tile];
  g.mt = (g.M + t.tm - 1) / t.tm;
  switch (tile) {
    case 0: return gemm_launch<EPI, 2, 2, 2, 2, 6>(g, t, st);
    case 1: return gemm_launch<EPI, 2, 4, 4, 2, 6>(g, t, st);
    case 2: return gemm_launch<EPI, 3, 4, 4, 2, 5>(g, t, st);
  }
  if constexpr (EPI != EPI_PART) {
    if (tile == 3) return gemm_launch<EPI, 4, 4, 4, 2, 4>(g, t, st);
    if constexpr (EPI != EPI_RES) {
      if (tile == 4) return gemm_launch<EPI, 6, 4, 2, 2, 4>(g, t, st);
      if (tile == 5) return gemm_launch<EPI, 5, 4, 2, 4, 4>(g, t, st);
      if (tile == 6) return gemm_launch<EPI, 8, 4, 2, 4, 4>(g, t, st);
    }
  }
}

// Tile and K splits of a projection of M tokens: the least estimated time, a
// split's partials and tail included (tail: us of a tail kernel that only a
// split needs; the partials are written and read once at 3-4 TB/s). An output
// is the same whatever the tile (its k-steps are summed in order) but not
// whatever the split, so the splits are those of M rounded up to 128 tokens
// (of 64 for the first 128, where short turns lie): a prompt of up to 128
// tokens gives the same bits in any chunks.
struct GemmPlan {
  int tile, splits;
};
float gemm_us(const GemmTile& t, int M, int N, int K, int splits, float tail) {
  const int wg = (M + t.tm - 1) / t.tm * (N / t.tn) * splits;
  const float rounds = t.tm == 64 ? fmaxf(1.f, (float)wg / 256.f) : (float)((wg + 255) / 256);
  const float us = t.fixed + rounds * (t.round + t.kstep * (float)(K / 32 / splits));
  return splits == 1 ? us : us + tail + (float)splits * (float)M * (float)N * 4.f / 7e6f;
}
GemmPlan gemm_plan(int M, int N, int K, int tiles, bool split, float tail) {
  GemmPlan best = {0, 1};
  const int most = (M + 127) / 128 * 128, Ms = most <= 128 ? 64 : most;
  for (int sp = 2; split && sp <= 16 && (size_t)sp * most * N * 4 <= PART_BYTES; sp *= 2) {
    auto least = [&](int s) {
      const int n = s > 1 ? TILES_PART : tiles;
      float us = gemm_us(TILES[0], Ms, N, K, s, tail);
      for (int i = 1; i < n; ++i) us = fminf(us, gemm_us(TILES[i], Ms, N, K, s, tail));
      return us;
    };
    if (least(sp) < least(best.splits)) best.splits = sp;
  }
  const int n = best.splits > 1 ? TILES_PART : tiles;
  for (int i = 1; i < n; ++i)
    if (gemm_us(TILES[i], M, N, K, best.splits, tail) < gemm_us(TILES[best.tile], M, N, K, best.splits, tail)) best.tile = i;
  return best;
}

}  // namespace

namespace mk {

size_t prefill_ws_bytes(int tokens) {
  const size_t t16 = (size_t)(tokens + 15) / 16 * 16;
  return t16 * ws_per_token() + PART_BYTES + 256;
}

int prefill_chunk_cap(size_t bytes) {
  if (bytes < prefill_ws_bytes(16)) return 0;
  const size_t t = (bytes - 256 - PART_BYTES) / ws_per_token() / 16 * 16;
  return t > (size_t)PREFILL_MAX_CHUNK ? PREFILL_MAX_CHUNK : (int)t;
}

hipError_t prefill_launch(const mk_weights* w, const mk_prefill_args* a, int cap) {
  hipStream_t st = static_cast<hipStream_t>(a->stream);
  const bool tiled = w->t_qkv && w->t_o && w->t_gu && w->t_down;
  const uint16_t* Wqkv = static_cast<const uint16_t*>(tiled ? w->t_qkv : w->w_qkv);
  const uint16_t* Wo = static_cast<const uint16_t*>(tiled ? w->t_o : w->w_o);
  const uint16_t* Wgu = static_cast<const uint16_t*>(tiled ? w->t_gu : w->w_gu);
  const uint16_t* Wd = static_cast<const uint16_t*>(tiled ? w->t_down : w->w_down);
  const size_t c16 = (size_t)(cap + 15) / 16 * 16;
  uint8_t* base = static_cast<uint8_t*>(a->workspace);
  uint16_t* x = reinterpret_cast<uint16_t*>(base);
  uint16_t* h1 = x + c16 * H;
  uint16_t* q = h1 + c16 * H;
  uint16_t* xn = q + c16 * H;
  uint16_t* att = xn + c16 * H;
  uint16_t* act = att + c16 * H;
  float* part = reinterpret_cast<float*>(act + c16 * INTER);
  const int L = a->n_layers, l0 = a->first_layer;
  // An N = 2048 projection (O: K = 2048, down: K = 8192) of T tokens with the
  // residual add, followed by the RMSNorm of its output into xn if `norm`:
  // as one GEMM with the add in its epilogue plus pf_norm, or, where few tiles
  // would leave the device idle, split over K into fp32 partials that
  // pf_reduce_norm sums (in split order), adds and normalises.
  auto res_gemm = [&](GemmArgs g, const uint16_t* res, uint16_t* out, bool norm, int T) {
    const GemmPlan pl = gemm_plan(T, g.N, g.K, TILES_RES, true, -0.5f);
    g.splits = pl.splits;
    if (pl.splits == 1) {
      g.res = res;
      g.out = out;
      gemm_run<EPI_RES>(g, pl.tile, st);
      if (norm)
        hipLaunchKernelGGL(pf_norm, dim3((unsigned)((T + NWAVE - 1) / NWAVE)), dim3(NT), 0, st, (const uint16_t*)out,
                           (const int32_t*)nullptr, (const uint16_t*)nullptr, (uint16_t*)nullptr, xn, T);
    } else {
      g.part = part;
      gemm_run<EPI_PART>(g, pl.tile, st);
      uint16_t* xn_out = norm ? xn : nullptr;
      switch (pl.splits) {   // gemm_plan gives 2, 4, 8 or 16
        case 2: hipLaunchKernelGGL(pf_reduce_norm<2>, dim3(T), dim3(NT), 0, st, (const float*)part, res, out, xn_out, T); break;
        case 4: hipLaunchKernelGGL(pf_reduce_norm<4>, dim3(T), dim3(NT), 0, st, (const float*)part, res, out, xn_out, T); break;
        case 8: hipLaunchKernelGGL(pf_reduce_norm<8>, dim3(T), dim3(NT), 0, st, (const float*)part, res, out, xn_out, T); break;
        default: hipLaunchKernelGGL(pf_reduce_norm<16>, dim3(T), dim3(NT), 0, st, (const float*)part, res, out, xn_out, T); break;
      }
    }
  };
  // Every chunk starts again from the embeddings of its own tokens; the rows
  // of earlier chunks are in the caches by then. A chunk's last layer needs
  // only its QKV GEMM unless the hidden state is asked for.
  for (int c0 = 0; c0 < a->n_tokens; c0 += cap) {
    const int T = min(cap, a->n_tokens - c0), p0 = a->start_pos + c0;
    hipLaunchKernelGGL(pf_norm, dim3((T + NWAVE - 1) / NWAVE), dim3(NT), 0, st, (const uint16_t*)nullptr,
                       a->tokens + c0, static_cast<const uint16_t*>(w->embed), x, xn, T);
    for (int li = 0; li < L; ++li) {
      const int l = l0 + li;
      const bool tail = li == L - 1 && !a->hidden_out;
      GemmArgs g;
      memset(&g, 0, sizeof(g));
      g.tiled = tiled;
      g.M = T;
      g.splits = 1;
      g.rope = static_cast<const uint16_t*>(w->rope);
      g.s_max = a->s_max;
      g.p0 = p0;
      uint16_t* kc = static_cast<uint16_t*>(a->k_cache[li]);
      uint16_t* vc = static_cast<uint16_t*>(a->v_cache[li]);
      // QKV + RoPE; K/V rows into the caches
      g.a = xn;
      g.b = Wqkv + (size_t)l * QKV_ROWS * H;
      g.N = QKV_ROWS;
      g.K = H;
      g.out = q;
      g.kc = kc;
      g.vc = vc;
      const GemmPlan qp = gemm_plan(T, QKV_ROWS, H, TILES_ALL, true, 4.5f);
      g.splits = qp.splits;
      if (qp.splits == 1) {
        gemm_run<EPI_QKV>(g, qp.tile, st);
      } else {   // short prompts: split over K, RoPE and the scatter in the tail
        g.part = part;
        gemm_run<EPI_PART>(g, qp.tile, st);
        const uint16_t* rope = static_cast<const uint16_t*>(w->rope);
        const dim3 fg(T, QKV_PAIRS / 2 / NT);
        switch (qp.splits) {   // gemm_plan gives 2, 4, 8 or 16
          case 2: hipLaunchKernelGGL(pf_qkv_finish<2>, fg, dim3(NT), 0, st, (const float*)part, rope, q, kc, vc, T, p0, a->s_max); break;
          case 4: hipLaunchKernelGGL(pf_qkv_finish<4>, fg, dim3(NT), 0, st, (const float*)part, rope, q, kc, vc, T, p0, a->s_max); break;
          case 8: hipLaunchKernelGGL(pf_qkv_finish<8>, fg, dim3(NT), 0, st, (const float*)part, rope, q, kc, vc, T, p0, a->s_max); break;
          default: hipLaunchKernelGGL(pf_qkv_finish<16>, fg, dim3(NT), 0, st, (const float*)part, rope, q, kc, vc, T, p0, a->s_max); break;
        }
        g.splits = 1;
      }
      if (tail) break;   // the last layer's K/V rows are all the caller needs
      AttnArgs aa;
      aa.q = q;
      aa.kc = kc;
      aa.vc = vc;
      aa.att = att;
      aa.T = T;
      aa.p0 = p0;
      aa.s_max = a->s_max;
      hipLaunchKernelGGL(pf_attn, dim3((T + PF_TB - 1) / PF_TB, NKV), dim3(NT), 0, st, aa);
      // O projection + residual -> h1, its RMSNorm -> xn
      g.a = att;
      g.b = Wo + (size_t)l * H * H;
      g.N = H;
      g.K = H;
      g.kc = g.vc = nullptr;
      res_gemm(g, x, h1, true, T);
      // gate/up + SwiGLU -> act
      g.a = xn;
      g.b = Wgu + (size_t)l * 2 * INTER * H;
      g.N = 2 * INTER;
      g.K = H;
      g.out = act;
      g.splits = 1;
      gemm_run<EPI_SWIGLU>(g, gemm_plan(T, g.N, g.K, TILES_ALL, false, 0.f).tile, st);
      // down projection + residual -> x (the next layer's input) and its RMSNorm -> xn,
      // or the caller's hidden state after the last layer
      g.a = act;
      g.b = Wd + (size_t)l * H * INTER;
      g.N = H;
      g.K = INTER;
      if (li + 1 < L) res_gemm(g, h1, x, true, T);
      else res_gemm(g, h1, static_cast<uint16_t*>(a->hidden_out) + (size_t)c0 * H, false, T);
    }
  }
  return hipGetLastError();
}

}  // namespace mk
