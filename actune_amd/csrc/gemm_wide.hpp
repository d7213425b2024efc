#pragma once
// Wide-tile packed group-64 GEMM for gfx950 on 32x32x32 int8 MFMAs, with an
// exact split of K over the waves of a workgroup.
//
// Restates actune/kernels/grouped.py:74-94 / grouped_native.cu:42-88 with the
// canonical chunked fp32 order (common.hpp), bit-identical to every other
// kernel of the library.
//
// Layout. A wave owns 32 weight rows and TM tiles of 32 tokens (WN x WM waves
// side by side: BN = 32 WN rows by BM = 32 TM WM tokens per workgroup). Lane
// (i, h) of an MFMA operand holds row / token i = lane % 32 and, of a group's
// 64 codes, 32 h .. 32 h + 31: both halves of a row's group are consecutive
// packed bytes, so a lane's weight load needs no exchange between lanes
// before its unpack. A lane's 16 results of a 32x32 tile share one token, so
// one scale register serves 16 rescales.
//  * Weights are staged packed, once per workgroup and quad (4 groups), with
//    loads of whole row runs, and unpacked by the waves that read them.
//  * Activations are staged once per workgroup and quad in LDS as 16-byte
//    slots in the weight width's element order, with their group scales
//    (2^-T folded in), one quad ahead, double-buffered: one barrier per quad.
//  * The MFMAs of a tile are issued beside the rescale of the tile before.
//
// K split (KS > 1): KS sets of waves work on the same output tile, set kg on
// the chunks kg, kg + KS, ... of the canonical order, each with its own
// staging buffers. After each round of KS chunks the sets exchange their
// partials through LDS: set d owns the d-th part of a wave's outputs and adds
// the round's partials of that part in chunk order, so the sum is the
// canonical one bit for bit and each set adds as much as an unsplit wave
// would per chunk. A set without a chunk in a round (or with a shorter one)
// multiplies scales of 0, whose products add nothing.
//
// Bound by the vector pipe: the rescale is one cvt and one fma per output and
// group beside 64 int8 MACs, half of the int8 MFMA issue rate at best. Counters
// (profiles/gemm_wide_m512_pmc.md): 2 x 11008x4096 W4A8 at M = 512 vector pipe
// 65% busy, 16 of its 26 instructions per MFMA the rescale, matrix pipe 20%,
// waves waiting 20% of the time; 4096x4096 W8A8, one workgroup per CU, 48%, 16%
// and 38%. Measured on MI355X with
// the 16x16x64 kernel that it replaced, or the prefill kernel, before:
// quantizer included, W4A8 11008x4096 at M = 2000 246 -> 182 us, W8A8 4096 x
// 4096 at M = 512 31.7 -> 28.2; GEMM alone, W8A8 22016x4096 at M = 64 83.8 ->
// 28.4. 32-row tiles rather than 16: one scale register per 16 results, and
// half the LDS reads per product.
#include "common.hpp"
#include "launch.hpp"
#include "operands.hpp"

namespace actune {

typedef int v16i __attribute__((ext_vector_type(16)));

__device__ __forceinline__ v16i mfma32x32x32(const uint32_t a[4], const uint32_t b[4], v16i c) {
  v4i av = {(int)a[0], (int)a[1], (int)a[2], (int)a[3]};
  v4i bv = {(int)b[0], (int)b[1], (int)b[2], (int)b[3]};
  return __builtin_amdgcn_mfma_i32_32x32x32_i8(av, bv, c, 0, 0, 0);
}

// LDS byte offset of 16-byte slot `slot` (0..15 of the quad) of token row
// `row`: XORed by the row so that both the 32 rows of a read and the slots a
// row's lanes write fall on distinct bank groups.
__device__ __forceinline__ int wide_slot_addr(int row, int slot) { return (row * 16 + (slot ^ (row & 15))) * 16; }

template <int W, int WN, int WM, int TM, int KS>
struct WideShape {
  static constexpr int BN = 32 * WN, BM = 32 * TM * WM;
  static constexpr int NT = 64 * WN * WM;                // threads of one K set
  static constexpr int R = 16 * TM, PR = R / KS;         // outputs per lane; of those, owned after the split
  static constexpr int ABYTES = BM * 256, SBYTES = BM * 16, WROW = 32 * W, WBYTES = BN * WROW;
  static constexpr int STAGE = ABYTES + SBYTES + WBYTES;
  static constexpr int XO = KS * 2 * STAGE;              // exchanged partials
  static constexpr int XB = KS > 1 ? WN * WM * KS * (KS - 1) * 64 * PR * 4 : 0;
  static constexpr int CO = XO + XB, LDS = CO + 2 * BN * 4;  // weight scales and biases
  static_assert(PR % 4 == 0, "an owner keeps whole row quads");
};

template <int W, int A, int WN, int WM, int TM, int KS, bool CPS>
__global__ __launch_bounds__(64 * WN * WM * KS, 2) void gemm_wide(const LinearArgs args, int tiles_m) {
  // sibling problems on grid y; grid x holds the tiles of the widest one
  const Problem prob = args.prob[blockIdx.y];
  using S = WideShape<W, WN, WM, TM, KS>;
  constexpr int T = shift_of(W) + shift_of(A);
  constexpr int NT = S::NT, BN = S::BN, BM = S::BM, PR = S::PR;
  constexpr int AROW = 32 * A;  // packed activation bytes per token and quad
  constexpr int ACH = BM * AROW / 16, APT = (ACH + NT - 1) / NT;
  constexpr int SPT = (BM * 4 + NT - 1) / NT;
  extern __shared__ __align__(16) uint8_t wide_lds[];

  const float fold = __builtin_ldexpf(1.0f, -T);
  const int M = args.M, K = args.K, N = prob.N, G = K / kGroup, Q = (G + 3) / 4;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int kg = wave / (WN * WM), tid = (int)threadIdx.x - kg * NT;  // K set; thread in it
  const int wg = wave % (WN * WM), wn = wg % WN, wm = wg / WN;
  const int l32 = lane & 31, h = lane >> 5;
  uint8_t* const stage = wide_lds + kg * 2 * S::STAGE;
  float* const wsl = reinterpret_cast<float*>(wide_lds + S::CO);
  float* const bsl = wsl + BN;

  // XCD-aware tile order: XCD x = id % 8 takes a contiguous range of tiles in
  // groups of 8 token blocks, row blocks before token blocks inside a group:
  // the tiles an XCD works on at a time share both operands in its L2.
  const int id = (int)blockIdx.x, tiles_n = (N + BN - 1) / BN, ntiles = tiles_n * tiles_m;
  if (id >= ntiles) return;
  const int xcd = id % 8, per = ntiles / 8, rem = ntiles % 8;
  const int idx = xcd * per + (xcd < rem ? xcd : rem) + id / 8;
  const int mg = idx / (8 * tiles_n), gm = min(8, tiles_m - 8 * mg), in_g = idx - mg * 8 * tiles_n;
  const int n_blk = in_g / gm * BN, m_blk = (8 * mg + in_g % gm) * BM;
  const int n_wave = n_blk + 32 * wn, t_wave = 32 * TM * wm;  // first row; first token of the block

  const uint32_t wrow_bytes = (uint32_t)K * W / 8, arow_bytes = (uint32_t)K * A / 8;
  const Rsrc wres = make_rsrc(prob.w, (uint32_t)N * wrow_bytes);
  const Rsrc ares = make_rsrc(args.a, (uint32_t)M * arow_bytes);
  const Rsrc sres = make_rsrc(args.as, (uint32_t)M * G * 4);

  // ------------------------------------------------ this set's quads, in order
  // CPS (Q <= kChunks): a chunk is one quad, a round one step. Otherwise a
  // round is as many steps as its longest chunk has quads. Step s of chunk c
  // reads quad qbeg(c) + s, or Q (past K: scales 0) where the chunk is over.
  const int nC = CPS ? Q : kChunks, rounds = (nC + KS - 1) / KS;
  auto qbeg = [&](int c) { return CPS ? min(c, Q) : min(c, kChunks) * Q / kChunks; };
  auto round_len = [&](int r) {
    if constexpr (CPS) return 1;
    int l = 0;
#pragma unroll
    for (int k = 0; k < KS; ++k) l = max(l, qbeg(r * KS + k + 1) - qbeg(r * KS + k));
    return l;
  };
  struct Step {
    int round, s;
  };
  auto next = [&](Step t) {
    if (CPS || t.s + 1 >= round_len(t.round)) return Step{t.round + 1, 0};
    return Step{t.round, t.s + 1};
  };
  auto quad_of = [&](Step t) {
    const int c = t.round * KS + kg, q = qbeg(c) + t.s;
    return q < qbeg(c + 1) ? q : Q;
  };

  // ------------------------------------------------ operand movers
  constexpr int WCH = S::WBYTES / 16, WPT = (WCH + NT - 1) / NT, WRC = S::WROW / 16;  // weight chunks
  uint32_t wbase[WPT], wraw[WPT][4];
#pragma unroll
  for (int t = 0; t < WPT; ++t) {
    const int ch = tid + t * NT, row = ch / WRC, cc = ch % WRC;
    wbase[t] = ch < WCH && n_blk + row < N ? (uint32_t)(n_blk + row) * wrow_bytes + cc * 16 : kOff;
  }
  auto load_weights = [&](int q) {
#pragma unroll
    for (int t = 0; t < WPT; ++t) buffer_slot<8>(wres, wbase[t] + (uint32_t)(q * S::WROW), wraw[t]);
  };
  // chunk c of staged weight row r sits at c ^ wswz(r)
  auto wpos = [&](int r, int byte) {
    constexpr int RP = 256 / S::WROW > 0 ? 256 / S::WROW : 1;  // rows per 256 bytes
    return r * S::WROW + 16 * ((byte >> 4) ^ ((r / RP) % WRC)) + (byte & 15);
  };
  auto store_weights = [&](uint8_t* buf) {
#pragma unroll
    for (int t = 0; t < WPT; ++t) {
      const int ch = tid + t * NT;
      if (WCH % NT && ch >= WCH) break;
      *reinterpret_cast<v4u*>(buf + S::ABYTES + S::SBYTES + wpos(ch / WRC, ch % WRC * 16)) =
          v4u{wraw[t][0], wraw[t][1], wraw[t][2], wraw[t][3]};
    }
  };
  uint32_t abase[APT];
#pragma unroll
  for (int t = 0; t < APT; ++t) {
    const int ch = tid + t * NT, row = ch / (AROW / 16), cc = ch % (AROW / 16);
    abase[t] = ch < ACH && m_blk + row < M ? (uint32_t)(m_blk + row) * arow_bytes + cc * 16 : kOff;
  }
  uint32_t araw[APT][4];
  float sraw[SPT];
  auto load_acts = [&](int q) {
#pragma unroll
    for (int t = 0; t < APT; ++t) buffer_slot<8>(ares, abase[t] + (uint32_t)(q * AROW), araw[t]);
#pragma unroll
    for (int t = 0; t < SPT; ++t) {
      const int e = tid + t * NT, m = m_blk + e / 4, g = q * 4 + e % 4;
      sraw[t] = buffer_f32(sres, e < BM * 4 && m < M && g < G ? ((uint32_t)m * G + g) * 4u : kOff);
    }

  };
  auto store_acts = [&](uint8_t* buf) {
#pragma unroll
    for (int t = 0; t < APT; ++t) {
      const int ch = tid + t * NT;
      if (ACH % NT && ch >= ACH) break;
      const int row = ch / (AROW / 16), cc = ch % (AROW / 16);
      constexpr int SPC = 8 / A;
#pragma unroll
      for (int u = 0; u < SPC; ++u) {
        uint32_t d[4];
        unpack_slot<A>(&araw[t][u * A / 2], d);
        reorder_slot<A, W>(d);
        *reinterpret_cast<v4u*>(buf + wide_slot_addr(row, cc * SPC + u)) = v4u{d[0], d[1], d[2], d[3]};
      }
    }
    float* sl = reinterpret_cast<float*>(buf + S::ABYTES);
#pragma unroll
    for (int t = 0; t < SPT; ++t) {
      const int e = tid + t * NT;
      if (BM * 4 % NT == 0 || e < BM * 4) sl[e] = sraw[t] * fold;
    }

  };

  // ------------------------------------------------ accumulators
  // MFMA results of tile t of a quad live in D[t & 1] until the next tile's
  // block rescales them (t of a quad's last tile is odd).
  v16i D[2];
  float acc[PR], p[TM][16];
#pragma unroll
  for (int r = 0; r < PR; ++r) acc[r] = 0.f;
#pragma unroll
  for (int y = 0; y < TM; ++y)
#pragma unroll
    for (int r = 0; r < 16; ++r) p[y][r] = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) D[0][r] = D[1][r] = 0;
  float slast = 0.f;  // scale of the previous step's last group, last token tile

  auto rescale = [&](int par, int y, float s, bool first) {
#pragma unroll
    for (int r = 0; r < 16; ++r)
      p[y][r] = first ? (float)D[par][r] * s : __builtin_fmaf((float)D[par][r], s, p[y][r]);
  };
  // KS = 1: token tile y's chunk partial joins the sum
  auto close_tile = [&](int y) {
    if constexpr (KS == 1) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[16 * y + r] = acc[16 * y + r] + p[y][r];
        if constexpr (!CPS) p[y][r] = 0.f;
      }
    }
  };
  // KS > 1: the round's chunk partials join the sums of their owners
  auto close_round = [&]() {
    if constexpr (KS > 1) {
      float* const xb = reinterpret_cast<float*>(wide_lds + S::XO);
      auto xat = [&](int src, int dst) {
        return xb + (((wg * KS + src) * (KS - 1) + (dst < src ? dst : dst - 1)) * 64 + lane) * PR;
      };
#pragma unroll
      for (int d = 0; d < KS; ++d) {
        if (d == kg) continue;  // uniform
        float* const to = xat(kg, d);
#pragma unroll
        for (int r = 0; r < PR; r += 4) {
          const float* v = &p[(d * PR + r) / 16][(d * PR + r) % 16];
          *reinterpret_cast<v4f*>(to + r) = v4f{v[0], v[1], v[2], v[3]};
        }
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        if (k == kg) {  // uniform
#pragma unroll
          for (int d = 0; d < KS; ++d)
            if (d == kg) {
#pragma unroll
              for (int r = 0; r < PR; ++r) acc[r] = acc[r] + p[(d * PR + r) / 16][(d * PR + r) % 16];
            }
        } else {
          const float* const from = xat(k, kg);
#pragma unroll
          for (int r = 0; r < PR; r += 4) {
            const v4f v = *reinterpret_cast<const v4f*>(from + r);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[r + e] = acc[r + e] + v[e];
          }
        }
      }
      if constexpr (!CPS) {
#pragma unroll
        for (int y = 0; y < TM; ++y)
#pragma unroll
          for (int r = 0; r < 16; ++r) p[y][r] = 0.f;
      }
    }
  };

  // ------------------------------------------------ prologue
  Step t0{0, 0}, t1 = next(t0), t2 = next(t1);  // this step and the two after it
  {
    load_acts(quad_of(t0));
    load_weights(quad_of(t0));
    store_acts(stage);
    store_weights(stage);
    load_acts(quad_of(t1));
    load_weights(quad_of(t1));
    for (int t = threadIdx.x; t < BN; t += NT * KS) {
      const ChannelConst cc = fetch_channel(prob.ws, prob.bias, args.bias_dt, N, n_blk + t, true);
      wsl[t] = cc.ws;
      bsl[t] = bias_from_bits(cc.bias_bits, args.bias_dt);
    }

  }
  __syncthreads();

  // ------------------------------------------------ main loop, two steps per trip
  bool closing = false;  // KS = 1, !CPS: the previous step ended a chunk
  while (t0.round < rounds) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (t0.round < rounds) {  // uniform: false only in the last trip
        const uint8_t* buf = stage + u * S::STAGE;
        const float* sl = reinterpret_cast<const float*>(buf + S::ABYTES);
        const int q2 = quad_of(t2);
        const bool ends = t1.round != t0.round;  // this step ends its round
        float sq[TM][4];
#pragma unroll
        for (int y = 0; y < TM; ++y) {
          const v4f s4 = *reinterpret_cast<const v4f*>(sl + (t_wave + 32 * y + l32) * 4);
#pragma unroll
          for (int gl = 0; gl < 4; ++gl) sq[y][gl] = s4[gl];
        }

        uint32_t bf[2][2][4];
        auto read_b = [&](int gl, int y, uint32_t (&dst)[2][4]) {
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const v4u b = *reinterpret_cast<const v4u*>(buf + wide_slot_addr(t_wave + 32 * y + l32, gl * 4 + 2 * h + j));
#pragma unroll
            for (int e = 0; e < 4; ++e) dst[j][e] = b[e];
          }
        };
        uint32_t wf[2][W];  // lane (row l32, half h): 32 codes of a group
        auto read_w = [&](int gl, uint32_t (&dst)[W]) {
          const uint8_t* wb = buf + S::ABYTES + S::SBYTES;
          if constexpr (W == 2) {
            const v2u v = *reinterpret_cast<const v2u*>(wb + wpos(32 * wn + l32, gl * 16 + 8 * h));
            dst[0] = v[0]; dst[1] = v[1];
          } else {
#pragma unroll
            for (int s = 0; s < W / 4; ++s) {
              const v4u v = *reinterpret_cast<const v4u*>(wb + wpos(32 * wn + l32, gl * 8 * W + 4 * W * h + 16 * s));
#pragma unroll
              for (int e = 0; e < 4; ++e) dst[4 * s + e] = v[e];
            }
          }
        };
        read_w(0, wf[0]);
        read_b(0, 0, bf[0]);
#pragma unroll
        for (int gl = 0; gl < 4; ++gl) {
          uint32_t wd[2][4];
#pragma unroll
          for (int j = 0; j < 2; ++j) unpack_slot<W>(&wf[gl & 1][j * W / 2], wd[j]);
          if (gl + 1 < 4) read_w(gl + 1, wf[(gl + 1) & 1]);
#pragma unroll
          for (int y = 0; y < TM; ++y) {
            const int t = gl * TM + y, par = t & 1;
            if (t + 1 < 4 * TM) read_b((t + 1) / TM, (t + 1) % TM, bf[(t + 1) & 1]);
            v16i z;
#pragma unroll
            for (int r = 0; r < 16; ++r) z[r] = 0;
            D[par] = mfma32x32x32(wd[0], bf[t & 1][0], z);
            D[par] = mfma32x32x32(wd[1], bf[t & 1][1], D[par]);
            // the previous tile's rescale runs beside this tile's MFMAs
            const int py = t == 0 ? TM - 1 : (t - 1) % TM, pg = t == 0 ? 3 : (t - 1) / TM;
            rescale(1 - par, py, t == 0 ? slast : sq[py][pg], CPS && t != 0 && pg == 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 16, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 16, 0);
            if (KS == 1 && pg == 3) {
              if constexpr (CPS) close_tile(py);
              else if (t == 0 ? closing : ends) close_tile(py);
            }
            // keep the rescale and the close in this block
#pragma unroll
            for (int r = 0; r < 16; ++r) asm volatile("" ::"v"(p[py][r]));
            if constexpr (KS == 1) {
#pragma unroll
              for (int r = 0; r < 16; ++r) asm volatile("" ::"v"(acc[16 * py + r]));
            }

            __builtin_amdgcn_sched_barrier(0);
          }
        }
        slast = sq[TM - 1][3];
        closing = ends;
        store_acts(stage + (1 - u) * S::STAGE);
        store_weights(stage + (1 - u) * S::STAGE);
        load_acts(q2);
        load_weights(q2);
        if (KS > 1 && ends) {
          rescale(1, TM - 1, slast, false);
          slast = 0.f;  // the next step's rescale of these results adds nothing
          close_round();
        }
        t0 = t1;
        t1 = t2;
        t2 = next(t2);
        __syncthreads();
      }
    }
  }
  if constexpr (KS == 1) {
    rescale(1, TM - 1, slast, false);
    close_tile(TM - 1);
  }

  // ------------------------------------------------ epilogue
  // a lane's 4 consecutive rows are 4 consecutive outputs of one token: one
  // vector store when N and the output pointer keep them aligned
  const bool has_bias = prob.bias != nullptr;
  const int ebytes = args.out_dt == kF32 ? 4 : 2;
  void* const out = prob.out;
  const bool vec_out = N % 4 == 0 && ((uintptr_t)out % (4 * ebytes)) == 0;
#pragma unroll
  for (int o = 0; o < PR; o += 4) {
    const int ro = kg * PR + o;  // of the wave's R outputs per lane
    const int m = m_blk + t_wave + 32 * (ro / 16) + l32;
    if (m >= M) continue;
    const int nl = 32 * wn + 8 * (ro % 16 / 4) + 4 * h, n0 = n_blk + nl;
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      v[r] = has_bias ? __builtin_fmaf(acc[o + r], wsl[nl + r], bsl[nl + r]) : acc[o + r] * wsl[nl + r];
    const long at = (long)m * N + n0;
    if (vec_out && n0 + 3 < N) {
      if (args.out_dt == kF32) {
        *reinterpret_cast<v4f*>((float*)out + at) = v4f{v[0], v[1], v[2], v[3]};
      } else {
        uint32_t e[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) e[r] = args.out_dt == kBF16 ? f32_to_bf16(v[r]) : f32_to_f16(v[r]);
        *reinterpret_cast<v2u*>((uint16_t*)out + at) = v2u{e[0] | (e[1] << 16), e[2] | (e[3] << 16)};
      }
      continue;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (n0 + r >= N) break;
      if (args.out_dt == kBF16) store_out<kBF16>(out, at + r, v[r]);
      else if (args.out_dt == kF16) store_out<kF16>(out, at + r, v[r]);
      else store_out<kF32>(out, at + r, v[r]);
    }
  }
}

constexpr int kWideLdsMax = 160 * 1024;  // a gfx950 CU's LDS

// One launch over the problems of g (grid y) with geometry (WN, WM, TM, KS).
template <int W, int A, int WN, int WM, int TM, int KS>
inline void launch_wide_t(const LinearArgs& g, hipStream_t st) {
  using S = WideShape<W, WN, WM, TM, KS>;
  static_assert(S::LDS <= kWideLdsMax, "LDS budget");
  int n_max = 0;
  for (int p = 0; p < g.nprob; ++p) n_max = g.prob[p].N > n_max ? g.prob[p].N : n_max;
  const int tm = (g.M + S::BM - 1) / S::BM;
  const dim3 grid((unsigned)((n_max + S::BN - 1) / S::BN * tm), (unsigned)g.nprob);
  if ((g.K / kGroup + 3) / 4 <= kChunks) {
    if constexpr (S::LDS > 64 * 1024) allow_dynamic_lds<gemm_wide<W, A, WN, WM, TM, KS, true>>(S::LDS);
    gemm_wide<W, A, WN, WM, TM, KS, true><<<grid, S::NT * KS, S::LDS, st>>>(g, tm);
  } else {
    if constexpr (S::LDS > 64 * 1024) allow_dynamic_lds<gemm_wide<W, A, WN, WM, TM, KS, false>>(S::LDS);
    gemm_wide<W, A, WN, WM, TM, KS, false><<<grid, S::NT * KS, S::LDS, st>>>(g, tm);
  }
}

// Shapes: 0 = 128x64 (W8: 128x128, whose 8 waves share one weight stage), 1 =
// 64x64, 2 = 128x32 with K split in two (W8: 64x128, 8 waves), 3 = 64x32 with
// K split in four (W8: in two, its weight stages being twice as large).
template <int W, int A>
inline void launch_wide_shape(int shape, const LinearArgs& g, hipStream_t st) {
  switch (shape) {
    case 0:
      if constexpr (W == 8) launch_wide_t<W, A, 4, 2, 2, 1>(g, st);
      else launch_wide_t<W, A, 4, 1, 2, 1>(g, st);
      break;
    case 1: launch_wide_t<W, A, 2, 2, 1, 1>(g, st); break;
    case 2:
      if constexpr (W == 8) launch_wide_t<W, A, 2, 4, 1, 1>(g, st);
      else launch_wide_t<W, A, 4, 1, 1, 2>(g, st);
      break;
    default: launch_wide_t<W, A, 2, 1, 1, (W == 8 ? 2 : 4)>(g, st); break;
  }
}

template <int W>
inline void launch_wide_width(int A, int shape, const LinearArgs& g, hipStream_t st) {
  if (A == 8) launch_wide_shape<W, 8>(shape, g, st);
  else if (A == 4) launch_wide_shape<W, 4>(shape, g, st);
  else launch_wide_shape<W, 2>(shape, g, st);
}

}  // namespace actune
