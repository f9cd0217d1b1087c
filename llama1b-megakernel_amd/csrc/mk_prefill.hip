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
// tile (64x64 to 256x256) and, for few tokens, a split of K into fp32 partials are
// chosen per projection by estimated time (gemm_tile, gemm_splits; calls of up to
// 128 tokens have splits of their own, gemm_short); the partials are summed in a
// fixed order by pf_reduce_norm (O and down) and pf_qkv_finish (QKV, with RoPE and
// the scatter).
//
// Attention: per (kv head, block of 16 or 32 tokens, range of keys) one
// workgroup, a q head per wave; S^T = K Q^T on the matrix cores (keys on M, 16
// tokens on N), an online softmax per column, and O^T = V^T P^T on the matrix
// cores with p rounded to bf16 as the reference rounds it (relative to the
// running maximum). K and V go through LDS in steps of 64 keys (V transposed
// there); where the keys are split, pf_attn_merge combines the parts.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include <type_traits>

#include "mk.h"
#include "mk_common.h"
#include "mk_prefill.h"

namespace {

using namespace mk;

// fp32 partials: a projection's (splits * M * N floats) or the attention's key splits
constexpr size_t PART_BYTES = (size_t)2048 * H * 4;

// Short calls, of up to SHORT_TOKENS tokens, give every token the same bits however
// a prompt is cut into them, at any row: the order of all its sums follows from its
// row in the cache alone. The first EARLY_ROWS rows keep the order that short
// prompts have always had, so their outputs have not changed: K in SHORT_QKV or
// SHORT_RES parts, the attention's maximum over 32 keys. Later rows take a faster
// one: half as many parts, each the sum of two, maxima over 64 keys, and the keys
// split (gemm_short, pf_attn, short_split).
constexpr int SHORT_TOKENS = 128, EARLY_ROWS = 128;

enum : int { EPI_QKV = 0, EPI_RES = 1, EPI_SWIGLU = 2, EPI_PART = 3, EPI_PAIR = 4 };

struct GemmArgs {
  const uint16_t* a;     // activations, A-tile order [M16][K]
  const uint16_t* b;     // weights [N][K]: MFMA tile order (tiled) or row-major
  int tiled;
  int M, N, K;
  int mt;                // row tiles
  int splits;            // EPI_PART, EPI_PAIR: the K range is cut into `splits` parts
  const uint16_t* res;   // EPI_RES: residual, row-major [M][N]
  uint16_t* out;         // EPI_RES: row-major [M][N]; EPI_SWIGLU: A-tile order [M16][N/2]; EPI_QKV: q [M][2048]
  float* part;           // EPI_PART, EPI_PAIR: fp32 [splits][M][N]
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
// 147 us timed alone (1370 TFLOP/s; 163 in a layer). Smaller tiles serve the shapes
// that would leave the device idle (gemm_tile).
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
  constexpr bool SPLIT_K = EPI == EPI_PART || EPI == EPI_PAIR;
  constexpr int NW = WM * WN, AB = MI * WM, BB = NI * WN, NB = AB + BB;   // waves; A, B and all blocks of a k-step
  constexpr int CPW = (NB + NW - 1) / NW;                                // copies per wave and k-step
  constexpr bool SPARE = NB % NW != 0;                                   // the last wave's surplus copies
  constexpr int EROW = 16 * NI * 2 + 16;                                 // bytes of a staged output row (padded)
  static_assert(NS >= 3 && 16 * EROW * NW <= NS * NB * 1024, "operand ring; staged outputs fit in it");
  __shared__ u32x4 L[(NS * NB + (SPARE ? 1 : 0)) * 64];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;   // (uniform: LDS copy bases)
  // Workgroup w runs on XCD w % 8: each XCD gets a contiguous range of tiles,
  // rows first, so the workgroups that share weight columns share its L2.
  const int nt = g.N / (16 * BB), tiles = g.mt * nt, total = SPLIT_K ? tiles * g.splits : tiles;
  const int xcd = blockIdx.x & 7, q8 = total >> 3, r8 = total & 7;
  const int item = xcd * q8 + min(xcd, r8) + ((int)blockIdx.x >> 3);
  const int split = SPLIT_K ? item / tiles : 0, tile = SPLIT_K ? item - split * tiles : item;
  const int tm = tile % g.mt, tn = tile / g.mt;
  const int m16 = (g.M + 15) / 16, kb = g.K / 32;
  const rsrc_t ra = make_rsrc(g.a, (size_t)m16 * 16 * g.K * 2);
  const rsrc_t rb = make_rsrc(g.b, (size_t)g.N * g.K * 2);
  // the k-steps of this workgroup: all of K, or one of `splits` parts (even numbers, as equal as they can be)
  const int k0 = SPLIT_K ? kb / 2 * split / g.splits * 2 : 0;
  const int ke = SPLIT_K ? kb / 2 * (split + 1) / g.splits * 2 : kb;
  const int kmid = (k0 + ke) / 4 * 2;   // EPI_PAIR: the second half, summed from zero, begins here
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
  f32x4 first[EPI == EPI_PAIR ? MI : 1][EPI == EPI_PAIR ? NI : 1];
  for (int ks = k0; ks < ke; ks += 2) {
    if constexpr (EPI == EPI_PAIR)
      if (ks == kmid) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) {
            first[i][j] = acc[i][j];
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
      }
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
  if constexpr (SPLIT_K) {
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int m = mw + 16 * i + lm;
      if constexpr (EPI == EPI_PAIR)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = first[i][j] + acc[i][j];
      if (m < g.M)
#pragma unroll
        for (int j = 0; j < NI; ++j)
          *reinterpret_cast<f32x4*>(g.part + ((size_t)split * g.M + m) * g.N + n0 + 16 * j + 4 * lq) = acc[i][j];
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

__device__ __forceinline__ float4 sum4(const float4& a, const float4& b) {
  return float4{a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w};
}

// The split-K tail of the O and down projections (N = 2048), one workgroup per
// token row t, 8 columns per thread: v = the sum of the SPLITS fp32 partials in
// split order (MIXED, a short call across EARLY_ROWS: of their pairs' sums from that
// row on), out = bf16(res + bf16(v)) (row-major), and, if xn is given, the
// next RMSNorm of out into xn (A-tile order), with pf_norm's bits. Latency
// bounds it: every load of the row is in flight at once (33 tokens of 16 splits
// on one wave per row, four rounds of loads: 9.4 us).
template <int SPLITS, bool MIXED>
__global__ void __launch_bounds__(NT) pf_reduce_norm(const float* part, const uint16_t* res, uint16_t* out,
                                                     uint16_t* xn, int T, int p0) {
  static_assert(H == 8 * NT, "8 columns per thread");
  __shared__ u32x4 row[NT];
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
  auto add = [&](const float4& a, const float4& b) {
    v[0] += a.x; v[1] += a.y; v[2] += a.z; v[3] += a.w;
    v[4] += b.x; v[5] += b.y; v[6] += b.z; v[7] += b.w;
  };
  if (MIXED && p0 + t >= EARLY_ROWS) {
#pragma unroll
    for (int sp = 0; sp + 1 < SPLITS; sp += 2) add(sum4(pv[sp][0], pv[sp + 1][0]), sum4(pv[sp][1], pv[sp + 1][1]));
  } else {
#pragma unroll
    for (int sp = 0; sp < SPLITS; ++sp) add(pv[sp][0], pv[sp][1]);
  }
  const uint32_t rw[4] = {rv.x, rv.y, rv.z, rv.w};
  uint32_t o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = pack_bf2(bf_lo(rw[e]) + rbf(v[2 * e]), bf_hi(rw[e]) + rbf(v[2 * e + 1]));
  *reinterpret_cast<u32x4*>(out + (size_t)t * H + c) = u32x4{o[0], o[1], o[2], o[3]};
  if (!xn) return;
  // every wave sums the whole row's squares, in rmsnorm2048's order
  row[threadIdx.x] = u32x4{o[0], o[1], o[2], o[3]};
  __syncthreads();
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < H / 512; ++i) {
    const u32x4 x = row[64 * i + lane_id()];
    const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) ss = fmaf(bf_hi(w[e]), bf_hi(w[e]), fmaf(bf_lo(w[e]), bf_lo(w[e]), ss));
  }
  const float inv = rsqrtf(wave_sum(ss) * (1.0f / H) + EPS);
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = cvt_bf2(bf_lo(o[e]) * inv, bf_hi(o[e]) * inv);
  *reinterpret_cast<u32x4*>(xn + a_tile_off(t, c, H / 32)) = u32x4{o[0], o[1], o[2], o[3]};
}

// The split-K tail of the QKV projection of short calls (N = 3072): thread
// (t, j) takes RoPE pairs 2j and 2j + 1 of token row t, i.e. columns 4j .. 4j + 3
// (dims d, d + 32, d + 1, d + 33 of one head, d = 2j mod 32), in one 16-byte
// load per split: each column summed over the SPLITS fp32 partials in split
// order (MIXED: as in pf_reduce_norm) and rounded to bf16, RoPE on the q and k pairs as the QKV GEMM's
// epilogue does it, q to the q buffer and k and v to the caches at row
// p0 + t, two bf16 per 4-byte store. Grid (T, QKV_PAIRS / 2 / NT).
template <int SPLITS, bool MIXED>
__global__ void __launch_bounds__(NT) pf_qkv_finish(const float* part, const uint16_t* rope, uint16_t* q,
                                                    uint16_t* kc, uint16_t* vc, int T, int p0, int s_max) {
  const int t = blockIdx.x, j = blockIdx.y * NT + (int)threadIdx.x;
  if (t >= T || j >= QKV_PAIRS / 2) return;
  const int pos = p0 + t, pr = 2 * j, hp = pr & 31;
  float4 pv[SPLITS];
#pragma unroll
  for (int sp = 0; sp < SPLITS; ++sp)
    pv[sp] = *reinterpret_cast<const float4*>(part + ((size_t)sp * T + t) * QKV_ROWS + 4 * j);
  float4 v = {0.f, 0.f, 0.f, 0.f};
  if (MIXED && pos >= EARLY_ROWS) {
#pragma unroll
    for (int sp = 0; sp + 1 < SPLITS; sp += 2) v = sum4(v, sum4(pv[sp], pv[sp + 1]));
  } else {
#pragma unroll
    for (int sp = 0; sp < SPLITS; ++sp) v = sum4(v, pv[sp]);
  }
  // pair 2j: (x[d], x[d + 32]) = (a0, b0); pair 2j + 1: (x[d + 1], x[d + 33]) = (a1, b1)
  const float a0 = rbf(v.x), b0 = rbf(v.y), a1 = rbf(v.z), b1 = rbf(v.w);
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
  float* part;           // key splits: o of (split, token, q head) [64], then (max, sum) of each
  int T, p0, s_max;
  int nb;                // blocks of tokens
  int split;             // keys per split (a multiple of KB); short calls: short_split instead
  int nsplit;
};
// The rows a launch of pf_attn is for: any, or a short call's (early: before EARLY_ROWS).
enum : int { ANY = 0, SHORT_EARLY = 1, SHORT_LATE = 2, SHORT_BOTH = 3 };

constexpr int KB = 64;                // keys per step
constexpr int VT_LD = KB + 8;         // bf16 per row (one dim) of the transposed V tile: 144 bytes
constexpr int ANS = 3;                // steps of K and V in LDS
constexpr float QK_LOG2 = SM_SCALE * 1.4426950408889634f;   // scores in units of log2: p = 2^(s - max)

// K and V of one step in LDS: K as 8 blocks of 1 KiB, (16 keys x 32 dims) in
// the MFMA's operand order (a_tile_off's), block 2 * (key / 16) + dim / 32; V
// transposed, the keys of a 32-key half in the order of the MFMA's k-slots (the
// 8 slots of lane group q4 are keys 4 q4 + i and 16 + 4 q4 + i, as p is held).
struct AttnTile {
  u32x4 k[8][64];
  uint16_t vt[HD][VT_LD];
};

// Short calls: keys per split for the token at `row` of the cache, the same for the
// 16 rows of an aligned block: all of them up to SHORT_WHOLE, else an eighth in
// steps of KB (it grows every 512 rows, between blocks).
constexpr int SHORT_WHOLE = 640;
__host__ __device__ inline int short_split(int row) {
  const int n = (row | 15) + 1;   // keys the block's last token sees
  return n <= SHORT_WHOLE ? SHORT_WHOLE : max(4 * KB, (n + 8 * KB - 1) / (8 * KB) * KB);
}
static_assert((size_t)8 * SHORT_TOKENS * NQ * (HD + 2) * 4 <= PART_BYTES, "eight parts of each token fit");

// Causal attention. Token t of the sequence (position p0 + t) attends to cache
// rows [0, p0 + t], its own row included (written by the QKV projection before
// this launch). A workgroup takes 16 NTL tokens of one kv head, wave h the
// group's q head h, NTL tiles of 16 tokens; SPLIT: one range of keys of them,
// its unnormalised output to `part` for pf_attn_merge.
//
// What bounds it: with many workgroups the exponentials (16 cycles each for a
// wave) and the operations around them, 28 cycles per 64 scores against 16 of
// MFMA; so the scale and the maximum go into one fma, masks are applied only on
// the diagonal, the accumulators are rescaled only when a maximum moved, and a
// step is 64 keys. With few, memory latency and what one CU can read: K goes
// from memory straight into LDS two steps ahead, V is loaded two steps ahead and
// transposed into LDS one step ahead, four keys by four dims at a time (one
// 8-byte store per dim). Workgroup w runs on XCD w % 8, which is its kv head: a
// head's K and V are read into one L2. Within a head the longest come first.
// Measured against 16-token workgroups with 32-key steps, one step ahead, and V
// transposed by 2-byte stores: 3001 tokens 112 -> 69 us, 1100 tokens 28.8 -> 23.
// Three and four tiles per wave are slower than two (84 and 94 us at 3001).
//
// Short calls: a workgroup's tokens are those of 16 rows of the cache from a
// multiple of 16 on, and their key split is those rows' (short_split). For the rows
// before EARLY_ROWS the running maximum moves every 32 keys, scores exponentiated
// as they are.
template <int NTL, bool SPLIT, int ROWS>
__global__ void __launch_bounds__(NT, NTL > 2 ? 2 : 3) pf_attn(AttnArgs a) {
  __shared__ AttnTile L[ANS];
  const int h = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), tid_ = threadIdx.x, lane = tid_ & 63;
  const int skew = ROWS == ANY ? 0 : a.p0 & 15;   // rows of the call's first block before its first token
  const int g = blockIdx.x & 7;                // kv head
  static_assert(NKV == 8, "a kv head per XCD");
  const int tb = a.nb - 1 - ((int)blockIdx.x >> 3) % a.nb, sp = ((int)blockIdx.x >> 3) / a.nb;
  const int t0 = tb * 16 * NTL - skew;
  const int k_end = a.p0 + min(t0 + 16 * NTL, a.T);
  const int split = ROWS == ANY ? a.split : short_split(a.p0 + t0);
  const int key0 = SPLIT ? sp * split : 0, n_keys = SPLIT ? min(k_end, key0 + split) : k_end;
  if (SPLIT && key0 >= k_end) return;          // (the merge knows)
  const int col = lane & 15, q4 = lane >> 4, hq = GQA * g + h;
  const rsrc_t rq = make_rsrc(a.q, (size_t)a.T * H * 2);
  u32x4 qv[NTL][2];   // this lane's token: t0 + 16 j + col
#pragma unroll
  for (int j = 0; j < NTL; ++j)
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int tq = t0 + 16 * j + col;
      qv[j][s] = ld16(rq, (uint32_t)tq < (uint32_t)a.T ? (uint32_t)(((size_t)tq * H + hq * HD + 32 * s + q4 * 8) * 2) : OOB);
    }
  const rsrc_t rk = make_rsrc(a.kc + (size_t)g * a.s_max * HD, (size_t)a.s_max * HD * 2);
  const rsrc_t rv = make_rsrc(a.vc + (size_t)g * a.s_max * HD, (size_t)a.s_max * HD * 2);
  // Staging: wave h copies K blocks 2h and 2h + 1 (keys 16 h + lane%16); thread
  // t loads V rows 4 (t/16) .. + 3, dims 4 (t%16) .. + 3. Keys past the range
  // read zero (no memory access), so the number in flight is fixed.
  const int vk = (tid_ >> 4) * 4, vd = (tid_ & 15) * 4;
  auto stage_k = [&](int k0, AttnTile& t) {
    const int key = k0 + 16 * h + col;
    const uint32_t off = key < n_keys ? (uint32_t)((key * HD + q4 * 8) * 2) : OOB;
#pragma unroll
    for (int s = 0; s < 2; ++s)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (lds_ptr_t)&t.k[2 * h + s][0], 16, off + 64u * s, 0, 0, 0);
  };
  auto load_v = [&](int k0, uint2 (&v)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = k0 + vk + i;
      const auto w = __builtin_amdgcn_raw_buffer_load_b64(rv, key < n_keys ? (int)((key * HD + vd) * 2) : (int)OOB, 0, 0);
      v[i] = uint2{(uint32_t)w[0], (uint32_t)w[1]};
    }
  };
  auto store_v = [&](const uint2 (&v)[4], AttnTile& t) {
    // keys vk .. + 3 of dim vd + e, at the k-slots of keys vk % 32 .. + 3
    const int slot = (vk & 32) + ((vk & 15) >> 2) * 8 + ((vk >> 4) & 1) * 4;
    const uint32_t lo[4] = {v[0].x, v[1].x, v[2].x, v[3].x}, hi[4] = {v[0].y, v[1].y, v[2].y, v[3].y};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t* w = e < 2 ? lo : hi;
      const uint32_t sel = e & 1 ? 0x07060302u : 0x05040100u;   // the upper or the lower halves of two words
      *reinterpret_cast<uint2*>(&t.vt[vd + e][slot]) =
          uint2{__builtin_amdgcn_perm(w[1], w[0], sel), __builtin_amdgcn_perm(w[3], w[2], sel)};
    }
  };
  f32x4 acc[NTL][4];
  float m_run[NTL], l_run[NTL];
#pragma unroll
  for (int j = 0; j < NTL; ++j) {
    m_run[j] = -INFINITY;
    l_run[j] = 0.f;
#pragma unroll
    for (int d = 0; d < 4; ++d) acc[j][d] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // the 32 keys hf of a step at a time
  auto compute_half = [&](int k0, int hf, const AttnTile& cur) {
    const int lim = a.p0 + min(t0 + col, a.T - 1);   // (padding tokens: any finite row)
    float s[2][4], mb = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      const u32x4 ka = cur.k[4 * hf + 2 * kt][lane], kb = cur.k[4 * hf + 2 * kt + 1][lane];
      const f32x4 v = mfma16(kb, qv[0][1], mfma16(ka, qv[0][0], f32x4{0.f, 0.f, 0.f, 0.f}));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[kt][i] = k0 + 32 * hf + 16 * kt + 4 * q4 + i <= lim ? v[i] * SM_SCALE : -INFINITY;
        mb = fmaxf(mb, s[kt][i]);
      }
    }
    const float m_new = fmaxf(m_run[0], max_xor32(max_xor16(mb)));   // finite: every token sees key 0
    const float alpha = __expf(m_run[0] - m_new);
    m_run[0] = m_new;
    float p[2][4], ps = 0.f;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[kt][i] = __expf(s[kt][i] - m_new);
        ps += p[kt][i];
      }
    l_run[0] = l_run[0] * alpha + ps;
    const u32x4 pb = {cvt_bf2(p[0][0], p[0][1]), cvt_bf2(p[0][2], p[0][3]), cvt_bf2(p[1][0], p[1][1]),
                      cvt_bf2(p[1][2], p[1][3])};
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const u32x4 vo = *reinterpret_cast<const u32x4*>(&cur.vt[16 * d + col][32 * hf + 8 * q4]);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[0][d][i] *= alpha;
      acc[0][d] = mfma16(vo, pb, acc[0][d]);
    }
  };
  auto compute = [&](int k0, const AttnTile& cur) {
    // S^T: keys 16 kt + 4 q4 + i of the step, this lane's token of each tile
    f32x4 s[NTL][4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      const u32x4 ka = cur.k[2 * kt][lane], kb = cur.k[2 * kt + 1][lane];
#pragma unroll
      for (int j = 0; j < NTL; ++j)
        s[j][kt] = mfma16(kb, qv[j][1], mfma16(ka, qv[j][0], f32x4{0.f, 0.f, 0.f, 0.f}));
    }
    u32x4 pb[NTL][2];
#pragma unroll
    for (int j = 0; j < NTL; ++j) {
      if (k0 + KB - 1 > a.p0 + t0 + 16 * j) {   // keys past some token of the tile
        const int lim = a.p0 + min(t0 + 16 * j + col, a.T - 1);   // (padding tokens: any finite row)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (k0 + 16 * kt + 4 * q4 + i > lim) s[j][kt][i] = -INFINITY;
      }
      float mb = fmaxf(fmaxf(s[j][0][0], s[j][0][1]), fmaxf(s[j][0][2], s[j][0][3]));
#pragma unroll
      for (int kt = 1; kt < 4; ++kt)
        mb = fmaxf(mb, fmaxf(fmaxf(s[j][kt][0], s[j][kt][1]), fmaxf(s[j][kt][2], s[j][kt][3])));
      mb = max_xor32(max_xor16(mb)) * QK_LOG2;   // the token's maximum over the step
      const float m_new = fmaxf(m_run[j], mb);
      const float m_use = SPLIT && m_new == -INFINITY ? 0.f : m_new;   // (a split's keys may all be masked)
      if (__any(m_new != m_run[j])) {
        const float alpha = __builtin_amdgcn_exp2f(m_run[j] - m_use);
        l_run[j] *= alpha;
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[j][d][i] *= alpha;
        m_run[j] = m_new;
      }
      float p[4][4];
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) p[kt][i] = __builtin_amdgcn_exp2f(fmaf(s[j][kt][i], QK_LOG2, -m_use));
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) l_run[j] += (p[kt][0] + p[kt][1]) + (p[kt][2] + p[kt][3]);
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
        pb[j][hf] = u32x4{cvt_bf2(p[2 * hf][0], p[2 * hf][1]), cvt_bf2(p[2 * hf][2], p[2 * hf][3]),
                          cvt_bf2(p[2 * hf + 1][0], p[2 * hf + 1][1]), cvt_bf2(p[2 * hf + 1][2], p[2 * hf + 1][3])};
    }
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const u32x4 vo = *reinterpret_cast<const u32x4*>(&cur.vt[16 * d + col][32 * hf + 8 * q4]);
#pragma unroll
        for (int j = 0; j < NTL; ++j) acc[j][d] = mfma16(vo, pb[j][hf], acc[j][d]);
      }
  };
  // Step i: its K copies and V loads are issued two steps before, V goes to LDS
  // one step before. Every wait leaves the 6 loads of the latest step in flight.
  constexpr int FLY = 6;
  uint2 v[2][4];
  load_v(key0, v[0]);
  stage_k(key0, L[0]);
  load_v(key0 + KB, v[1]);
  stage_k(key0 + KB, L[1]);
  store_v(v[0], L[0]);
  wait_copies<FLY, 0>();
  const int steps = (n_keys - key0 + KB - 1) / KB;
  auto run_steps = [&](auto early) {
    int slot = 0;
    for (int it = 0; it < steps; it += 2) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (it + u < steps) {
          const int k0 = key0 + (it + u) * KB, s1 = slot == ANS - 1 ? 0 : slot + 1, s2 = s1 == ANS - 1 ? 0 : s1 + 1;
          load_v(k0 + 2 * KB, v[u]);
          stage_k(k0 + 2 * KB, L[s2]);
          if constexpr (early.value) {
            static_assert(NTL == 1 && !SPLIT && EARLY_ROWS <= SHORT_WHOLE, "one tile, all keys");
            compute_half(k0, 0, L[slot]);
            compute_half(k0, 1, L[slot]);
          } else {
            compute(k0, L[slot]);
          }
          store_v(v[u ^ 1], L[s1]);
          wait_copies<FLY, 0>();
          slot = s1;
        }
      }
    }
  };
  if constexpr (ROWS == SHORT_BOTH) {
    if (a.p0 + t0 < EARLY_ROWS) run_steps(std::true_type{});
    else run_steps(std::false_type{});
  } else {
    run_steps(std::bool_constant<ROWS == SHORT_EARLY>{});
  }
  // the token's sum over its four lanes; o = acc / l, dims 16 d + 4 q4 + i
#pragma unroll
  for (int j = 0; j < NTL; ++j) {
    const int tq = t0 + 16 * j + col;
    const float l_tot = add_xor32(add_xor16(l_run[j]));
    if ((uint32_t)tq >= (uint32_t)a.T) continue;
    if constexpr (SPLIT) {
      const size_t at = ((size_t)sp * a.T + tq) * NQ + hq, n = (size_t)a.nsplit * a.T * NQ;
#pragma unroll
      for (int d = 0; d < 4; ++d) *reinterpret_cast<f32x4*>(a.part + at * HD + 16 * d + 4 * q4) = acc[j][d];
      if (q4 == 0) *reinterpret_cast<float2*>(a.part + n * HD + at * 2) = float2{m_run[j], l_tot};
    } else {
      const float inv = 1.0f / l_tot;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        uint2 w;
        w.x = pack_bf2(acc[j][d][0] * inv, acc[j][d][1] * inv);
        w.y = pack_bf2(acc[j][d][2] * inv, acc[j][d][3] * inv);
        *reinterpret_cast<uint2*>(a.att + a_tile_off(tq, hq * HD + 16 * d + 4 * q4, H / 32)) = w;
      }
    }
  }
}

// The attention output from the splits' parts: 16 lanes per (token, q head),
// four dims each; the splits that hold keys of the token's workgroup (SHORT: of
// the token), in order.
template <bool SHORT>
__global__ void __launch_bounds__(NT) pf_attn_merge(AttnArgs a) {
  const int i = (int)blockIdx.x * (NT / 16) + ((int)threadIdx.x >> 4), t = i / NQ, hq = i % NQ;
  const int d = ((int)threadIdx.x & 15) * 4;
  if (t >= a.T) return;
  const int k_end = SHORT ? a.p0 + t + 1 : a.p0 + min((t / 16 + 1) * 16, a.T);
  const int split = SHORT ? short_split(a.p0 + t) : a.split;
  const int ns = min((k_end + split - 1) / split, a.nsplit);
  const float2* ml = reinterpret_cast<const float2*>(a.part + (size_t)a.nsplit * a.T * NQ * HD);
  float M = -INFINITY;
  for (int s = 0; s < ns; ++s) M = fmaxf(M, ml[((size_t)s * a.T + t) * NQ + hq].x);
  float l = 0.f;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < ns; ++s) {
    const size_t at = ((size_t)s * a.T + t) * NQ + hq;
    const float2 x = ml[at];
    const float f = __builtin_amdgcn_exp2f(x.x - M);
    l = fmaf(x.y, f, l);
    o += *reinterpret_cast<const f32x4*>(a.part + at * HD + d) * f;
  }
  const float inv = 1.0f / l;
  *reinterpret_cast<uint2*>(a.att + a_tile_off(t, hq * HD + d, H / 32)) =
      uint2{pack_bf2(o[0] * inv, o[1] * inv), pack_bf2(o[2] * inv, o[3] * inv)};
}

template <int NTL, bool SPLIT, int ROWS = ANY>
void attn_launch(const AttnArgs& a, hipStream_t st) {
  static_assert(NTL == 1 || (!SPLIT && ROWS == ANY), "pf_attn_merge and short calls count 16 tokens per workgroup");
  hipLaunchKernelGGL((pf_attn<NTL, SPLIT, ROWS>), dim3(a.nb * NKV * (SPLIT ? a.nsplit : 1)), dim3(NT), 0, st, a);
  if (SPLIT)
    hipLaunchKernelGGL(pf_attn_merge<ROWS != ANY>, dim3((a.T * NQ + NT / 16 - 1) / (NT / 16)), dim3(NT), 0, st, a);
}
// Tiles of 16 tokens up to 2048 tokens, of 32 above (one 16-token tile per wave
// against two: 2048 tokens 44 against 47 us, 3001 tokens 92 against 71). Few
// workgroups over many keys split them, up to 8 ways, as far as the device has
// room for (three workgroups per CU) and the partials fit: a step of 64 keys
// takes one workgroup 0.85 us, the parts and the merge 5 us and what they move
// (33 tokens at 4000 rows: 55 us whole, 17.5 in 8 parts; at 700 rows 13.6 and
// 11.0). Splits begin at multiples of 64 keys of the cache.
//
// Short calls split a token's keys by its row alone (short_split). One across
// EARLY_ROWS takes a kernel with both forms of a step: 33 tokens at row 100 49.7 us,
// with a launch for either side 54.9. The other calls would lose 0.7 us by it.
void attn_run(AttnArgs a, hipStream_t st) {
  if (a.T <= SHORT_TOKENS) {
    const int base = a.p0 & ~15;
    a.nb = (a.p0 + a.T - base + 15) / 16;
    a.nsplit = 1;
    for (int row = base; row < a.p0 + a.T; row += 16)
      a.nsplit = max(a.nsplit, (min(row + 16, a.p0 + a.T) + short_split(row) - 1) / short_split(row));
    if (a.p0 + a.T <= EARLY_ROWS) return attn_launch<1, false, SHORT_EARLY>(a, st);
    if (a.p0 < EARLY_ROWS) return attn_launch<1, false, SHORT_BOTH>(a, st);
    if (a.nsplit == 1) return attn_launch<1, false, SHORT_LATE>(a, st);
    return attn_launch<1, true, SHORT_LATE>(a, st);
  }
  static_assert(EARLY_ROWS % 16 == 0 && EARLY_ROWS + SHORT_TOKENS <= SHORT_WHOLE, "early and split rows in no one call");
  a.nb = (a.T + 15) / 16;
  const int n_keys = a.p0 + a.T, wgs = a.nb * NKV;
  const int most = (int)(PART_BYTES / ((size_t)NQ * (HD + 2) * 4)) / a.T;   // splits whose parts fit
  const int ns = min(min(8, 3 * 256 / wgs), most);
  if (ns >= 2) {
    const int split = max(4 * KB, (n_keys + ns * KB - 1) / (ns * KB) * KB);
    const float saved = (float)(n_keys - split) / KB * 0.85f;
    if (saved > 5.f + (float)(ns * a.T) * (NQ * (HD + 2) * 4) * 2.f / 4e6f) {
      a.split = split;
      a.nsplit = (n_keys + split - 1) / split;
      return attn_launch<1, true>(a, st);
    }
  }
  if (a.T <= 2048) return attn_launch<1, false>(a, st);
  a.nb = (a.T + 31) / 32;
  attn_launch<2, false>(a, st);
}

size_t ws_per_token() { return (size_t)H * 2 * 5 + (size_t)INTER * 2; }
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
// The tiles each epilogue is built on: [first, end) of TILES. Unsplit, N = 2048
// never takes 64x64 (K is split wherever it would) and hardly ever one above 256x128;
// with K split those above 192x128 hardly ever win; short calls are the fastest on
// 64x64 in pairs.
struct TileRange {
  int first, end;
};
constexpr TileRange tiles_of(int epi) {
  return epi == EPI_RES ? TileRange{1, 4} : epi == EPI_PART ? TileRange{0, 3} : epi == EPI_PAIR ? TileRange{0, 1}
                                                                                               : TileRange{0, 7};
}

template <int EPI, int TILE, int MI, int NI, int WM, int WN, int NS>
void gemm_launch(const GemmArgs& g, hipStream_t st) {
  constexpr GemmTile t = TILES[TILE];
  static_assert(t.tm == 16 * MI * WM && t.tn == 16 * NI * WN, "the tile of TILES");
  if constexpr (TILE >= tiles_of(EPI).first && TILE < tiles_of(EPI).end)
    hipLaunchKernelGGL((pf_gemm<EPI, MI, NI, WM, WN, NS>), dim3(g.mt * (g.N / t.tn) * g.splits), dim3(64 * WM * WN), 0,
                       st, g);
}
template <int EPI>
void gemm_run(GemmArgs g, int tile, hipStream_t st) {
  g.mt = (g.M + TILES[tile].tm - 1) / TILES[tile].tm;
  switch (tile) {
    case 0: return gemm_launch<EPI, 0, 2, 2, 2, 2, 6>(g, st);
    case 1: return gemm_launch<EPI, 1, 2, 4, 4, 2, 6>(g, st);
    case 2: return gemm_launch<EPI, 2, 3, 4, 4, 2, 5>(g, st);
    case 3: return gemm_launch<EPI, 3, 4, 4, 4, 2, 4>(g, st);
    case 4: return gemm_launch<EPI, 4, 6, 4, 2, 2, 4>(g, st);
    case 5: return gemm_launch<EPI, 5, 5, 4, 2, 4, 4>(g, st);
    case 6: return gemm_launch<EPI, 6, 8, 4, 2, 4, 4>(g, st);
  }
}

// The estimated time of a projection of M tokens. A split adds what it moves (its
// partials' bytes at 7 TB/s: a weight, not a bandwidth, since the fitted times hold
// the GEMM's own stores) less 0.5 us, as its tail takes the place of pf_norm. Four
// times that weight chooses fewer parts: a layer of 200 tokens then takes 72 us
// instead of 69, one of 512 102.6 instead of 104.3, of 900 157 instead of 156.
float gemm_us(const GemmTile& t, int M, int N, int K, int splits) {
  const int wg = (M + t.tm - 1) / t.tm * (N / t.tn) * splits;
  const float rounds = t.tm == 64 ? fmaxf(1.f, (float)wg / 256.f) : (float)((wg + 255) / 256);
  const float us = t.fixed + rounds * (t.round + t.kstep * (float)((K / 64 + splits - 1) / splits * 2));
  return splits == 1 ? us : us - 0.5f + (float)splits * (float)M * (float)N * 4.f / 7e6f;
}
// The tile for it among an epilogue's: the least estimated time.
int gemm_tile(int epi, int M, int N, int K, int splits) {
  const TileRange r = tiles_of(epi);
  int best = r.first;
  for (int i = r.first + 1; i < r.end; ++i)
    if (gemm_us(TILES[i], M, N, K, splits) < gemm_us(TILES[best], M, N, K, splits)) best = i;
  return best;
}
// The K splits of an N = 2048 projection of M > SHORT_TOKENS tokens whose partials
// fit in part_bytes: the least estimated time. An output is the same whatever the
// tile (its k-steps are summed in order) but not whatever the split, so it is that of
// M rounded up to 128 tokens. (3 and 5 fill the device where 2 and 4 leave a
// quarter of it idle and the partials of 8 do not fit: the down projection of 383
// tokens on 240 workgroups instead of 192 takes 20.4 us instead of 23.1, its tail
// 6.0 instead of 5.8; the parts of K then differ by one pair of k-steps.)
int gemm_splits(int M, int N, int K, size_t part_bytes) {
  const int most = (M + 127) / 128 * 128;
  auto least = [&](int s) {
    const int epi = s == 1 ? EPI_RES : EPI_PART;
    return gemm_us(TILES[gemm_tile(epi, most, N, K, s)], most, N, K, s);
  };
  int best = 1;
  for (int sp : {2, 3, 4, 5, 8})
    if ((size_t)sp * most * N * 4 <= part_bytes && least(sp) < least(best)) best = sp;
  return best;
}
// Short calls cut K into SHORT_QKV or SHORT_RES parts. From row EARLY_ROWS on a
// workgroup takes two of them, each summed from zero, and stores the sum (EPI_PAIR:
// half the partials); an earlier call stores each part, and where it reaches past
// EARLY_ROWS its tails add the pairs there (MIXED). A row's sums are the same.
// One layer, 33 tokens at row 700: 51 us as with the splits of least estimated
// time (5, 8 and 8), 128 tokens at row 200: 61 us; every part stored and every
// maximum over 32 keys there: 55 and 71 us.
constexpr int SHORT_QKV = 8, SHORT_RES = 16;
static_assert((size_t)SHORT_TOKENS * 4 * SHORT_QKV * QKV_ROWS <= PART_BYTES &&
                  (size_t)SHORT_TOKENS * 4 * SHORT_RES * H <= PART_BYTES,
              "a short call's partials fit");
void gemm_short(GemmArgs g, int parts, hipStream_t st) {
  const bool pairs = g.p0 >= EARLY_ROWS;
  g.splits = pairs ? parts / 2 : parts;
  if (pairs) gemm_run<EPI_PAIR>(g, 0, st);
  else gemm_run<EPI_PART>(g, gemm_tile(EPI_PART, g.M, g.N, g.K, parts), st);
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
  uint16_t* xn = h1 + c16 * H;
  uint16_t* act = xn + c16 * H;
  uint16_t* att = act + c16 * INTER;
  uint16_t* q = att + c16 * H;
  float* part = reinterpret_cast<float*>(q + c16 * H);
  const int L = a->n_layers, l0 = a->first_layer;
  // A short call's parts of K: f(number of partials, whether the tail adds pairs).
  auto with_parts = [](auto parts, const GemmArgs& g, auto&& f) {
    if (g.p0 >= EARLY_ROWS) return f(std::integral_constant<int, parts.value / 2>{}, std::false_type{});
    if (g.p0 + g.M <= EARLY_ROWS) return f(parts, std::false_type{});
    return f(parts, std::true_type{});
  };
  // The split-K tail of an N = 2048 projection: SPLITS partials, summed as pf_reduce_norm says.
  auto reduce = [&](auto splits, auto mixed, const GemmArgs& g, const uint16_t* res, uint16_t* out, bool norm) {
    hipLaunchKernelGGL((pf_reduce_norm<splits.value, mixed.value>), dim3(g.M), dim3(NT), 0, st, (const float*)g.part, res,
                       out, norm ? xn : (uint16_t*)nullptr, g.M, g.p0);
  };
  // An N = 2048 projection (O: K = 2048, down: K = 8192) of T tokens with the
  // residual add, followed by the RMSNorm of its output into xn if `norm`:
  // as one GEMM with the add in its epilogue plus pf_norm, or, where few tiles
  // would leave the device idle, split over K into fp32 partials that
  // pf_reduce_norm sums (in split order), adds and normalises.
  auto res_gemm = [&](GemmArgs g, const uint16_t* res, uint16_t* out, bool norm, float* parts, size_t part_bytes) {
    const auto plain = std::false_type{};
    g.part = parts;
    if (g.M <= SHORT_TOKENS) {
      gemm_short(g, SHORT_RES, st);
      return with_parts(std::integral_constant<int, SHORT_RES>{}, g,
                        [&](auto n, auto mixed) { reduce(n, mixed, g, res, out, norm); });
    }
    g.splits = gemm_splits(g.M, g.N, g.K, part_bytes);
    const int tile = gemm_tile(g.splits == 1 ? EPI_RES : EPI_PART, g.M, g.N, g.K, g.splits);
    if (g.splits == 1) {
      g.res = res;
      g.out = out;
      gemm_run<EPI_RES>(g, tile, st);
      if (norm)
        hipLaunchKernelGGL(pf_norm, dim3((unsigned)((g.M + NWAVE - 1) / NWAVE)), dim3(NT), 0, st, (const uint16_t*)out,
                           (const int32_t*)nullptr, (const uint16_t*)nullptr, (uint16_t*)nullptr, xn, g.M);
      return;
    }
    gemm_run<EPI_PART>(g, tile, st);
    switch (g.splits) {
      case 2: return reduce(std::integral_constant<int, 2>{}, plain, g, res, out, norm);
      case 3: return reduce(std::integral_constant<int, 3>{}, plain, g, res, out, norm);
      case 4: return reduce(std::integral_constant<int, 4>{}, plain, g, res, out, norm);
      case 5: return reduce(std::integral_constant<int, 5>{}, plain, g, res, out, norm);
      case 8: return reduce(std::integral_constant<int, 8>{}, plain, g, res, out, norm);
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
      if (T > SHORT_TOKENS) {
        gemm_run<EPI_QKV>(g, gemm_tile(EPI_QKV, T, QKV_ROWS, H, 1), st);
      } else {   // split over K, RoPE and the scatter in the tail
        g.part = part;
        gemm_short(g, SHORT_QKV, st);
        const uint16_t* rope = static_cast<const uint16_t*>(w->rope);
        with_parts(std::integral_constant<int, SHORT_QKV>{}, g, [&](auto n, auto mixed) {
          hipLaunchKernelGGL((pf_qkv_finish<n.value, mixed.value>), dim3(T, QKV_PAIRS / 2 / NT), dim3(NT), 0, st,
                             (const float*)part, rope, q, kc, vc, T, p0, a->s_max);
        });
      }
      if (tail) break;   // the last layer's K/V rows are all the caller needs
      AttnArgs aa;
      aa.q = q;
      aa.kc = kc;
      aa.vc = vc;
      aa.att = att;
      aa.part = part;
      aa.T = T;
      aa.p0 = p0;
      aa.s_max = a->s_max;
      attn_run(aa, st);
      // O projection + residual -> h1, its RMSNorm -> xn
      g.a = att;
      g.b = Wo + (size_t)l * H * H;
      g.N = H;
      g.K = H;
      g.kc = g.vc = nullptr;
      res_gemm(g, x, h1, true, part, PART_BYTES);
      // gate/up + SwiGLU -> act
      g.a = xn;
      g.b = Wgu + (size_t)l * 2 * INTER * H;
      g.N = 2 * INTER;
      g.K = H;
      g.out = act;
      gemm_run<EPI_SWIGLU>(g, gemm_tile(EPI_SWIGLU, T, g.N, g.K, 1), st);
      // down projection + residual -> x (the next layer's input) and its RMSNorm -> xn,
      // or the caller's hidden state after the last layer
      g.a = act;
      g.b = Wd + (size_t)l * H * INTER;
      g.N = H;
      g.K = INTER;
      // (att and q hold nothing any more and lie before `part`)
      float* down_part = reinterpret_cast<float*>(att);
      const size_t down_bytes = PART_BYTES + (size_t)T * H * 2 * 2;
      if (li + 1 < L) res_gemm(g, h1, x, true, down_part, down_bytes);
      else res_gemm(g, h1, static_cast<uint16_t*>(a->hidden_out) + (size_t)c0 * H, false, down_part, down_bytes);
    }
  }
  return hipGetLastError();
}

}  // namespace mk
