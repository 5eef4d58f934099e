// The latent block's projections (kimi.py:317, 325-328) for more than 64
// tokens, as bf16 GEMMs:
//
//   k_lgemm<0>  latent   = bf16(x @ latent_down.T)
//               shared_h = bf16(act(bf16(x @ shared_gate.T), bf16(x @ shared_up.T)))
//   k_lnorm     en       = bf16(bf16(rms_normalize(bf16(expert_sum))) * latent_norm)
//   k_lgemm<1>  out      = bf16(bf16(en @ latent_up.T) + bf16(shared_h @ shared_down.T))
//
// (up to 64 tokens the skinny kernels of k3moe_latent.hpp stream the weights
// once; run 64 rows at a time they reread the 136 MB of a TP8 rank per 64
// tokens, 13 x 31 and 13 x 32 us at 777 tokens.)
//
// Tile = (32 RW weight rows, up to 32 TW tokens) of one workgroup: waves 0-7
// multiply, 4 x 2, RW / 2 x TW 16x16x32 MFMA tiles each, two waves per SIMD (one's LDS
// reads beside the other's MFMAs); waves 8-11 load. The
// operands move 64 k at a time through Ring LDS slots filled by direct-to-LDS
// loads Ring - 1 steps ahead, one barrier per step: rows of 128 bytes, the
// 16-byte chunk c of row r at position c ^ ((r >> 1) & 7), so that the reads of
// 16 rows cover all banks. An MFMA wave reads the next 32 k's operands (after
// the next step's barrier, at a step's second half) before it multiplies the
// ones it holds. The loaders run over tile boundaries.
//
// <0>'s rows are the latent_down rows, then 16-row tiles of 8 shared_gate rows
// and the same 8 shared_up rows (the activation meets them with one exchange
// between lanes). <1> is two reductions, rounded apart: a tile's shared part is
// multiplied first and stored as bf16, and the same lanes add it to the routed
// part when that is done.
//
//   k_lgemm<2>  the general path's router logits, x @ router.T as fp32 partials
//               per k split, which the top-k kernel sums (kimi.py:308)
//
// Work is (row block, k split, token group); RW, TW and the number of splits
// are chosen by lgemm_plan from the rounds of the grid and a step's cost. With
// splits, fp32 partials go to the workspace and k_lreduce sums them in split
// order: results do not depend on timing. The latent entry points' workspace is the
// 64-token kernels' for every batch; inside the block the MoE step's, free before
// and after it, takes the partials and the normalised rows.
//
// Measured on a Kimi K3 TP8 rank (h 7168, lh 3584, S 768): <0> 21 + 6 us at 65
// tokens (62 in two skinny launches), 98 at 777 (407), 208 at 2048 (988); <1> with
// its norm 20 + 5 + 5, 75 + 7 (416), 169 + 10 us (1024). With four MFMA waves <0> took 26,
// 109 and 213 us, <1> 24, 73 and 165; timing builds of that <0> at 777: without the
// loads 83 us, without the MFMAs 80, without either 36, and the loads about 50 KB/us a
// CU also with every line in L2.
#pragma once

#include "k3moe_device.hpp"
#include "k3moe_latent.hpp"
#include "k3moe_plan.hpp"
#include "k3moe_sgemm.hpp"

namespace k3moe {

constexpr int kLgMfma = 8;  // MFMA waves, 4 x 2 over a tile's rows and tokens
constexpr int kLgThreads = (kLgMfma + 4) * 64;

template <int RW, int TW>
struct LgGeom {
  static constexpr int slot = 4096 * (RW + TW);
  static constexpr int fit = kDecMaxLds / slot;
  static constexpr int ring = fit < 6 ? fit : 6;
  static constexpr int lds = ring * slot;
  static_assert(ring >= 3);
};

// x: <0> x [B, h], <1> en [B, lh]; x2: <1> shared_h [B, S]; wa: latent_down / latent_up;
// wb: shared_gate / shared_down; wc: shared_up; ya: latent / out; yb: shared_h. <2>: x,
// wa = router, part = the logits' partials [split][B][N].
template <int OUT, int RW, int TW>
__global__ __launch_bounds__(kLgThreads, 1) void k_lgemm(LgPlan pl, const uint16_t *__restrict__ x,
                                                        const uint16_t *__restrict__ x2,
                                                        const uint16_t *__restrict__ wa,
                                                        const uint16_t *__restrict__ wb,
                                                        const uint16_t *__restrict__ wc, uint16_t *ya, uint16_t *yb,
                                                        float *part) {
  typedef LgGeom<RW, TW> Geo;
  constexpr int Ring = Geo::ring, Ahead = Ring - 1, Slot = Geo::slot, OffB = 4096 * RW;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, l = tid & 63, i = l & 15, q = l >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int w = wv & (kLgMfma - 1);  // the MFMA wave, or the loader 0 .. 3
  const int xcds = gridDim.x < 8 ? (int)gridDim.x : 8;
  const int xcd = blockIdx.x % xcds, nslot = gridDim.x / xcds, slot = blockIdx.x / xcds;
  const int j0 = (int)((long)pl.items * xcd / xcds), j1 = (int)((long)pl.items * (xcd + 1) / xcds);
  const int spi = OUT != 1 || pl.splits > 1 ? 1 : pl.segs;  // segments a workgroup runs one after the other per item
  const int nu = j1 - j0 > slot ? ((j1 - j0 - slot + nslot - 1) / nslot) * spi : 0;
  if (nu == 0) return;

  // Segment u of this workgroup: row block, token group, k segment and its steps [k0, k1).
  struct UnitP {
    int rb, tg, seg, k0, k1;
  };
  auto unit_at = [&](int u) {
    UnitP U;
    unsigned v = (unsigned)(j0 + slot + (u / spi) * nslot);  // ((row block, segment), token group)
    U.tg = (int)(v % (unsigned)pl.NTG);
    v /= (unsigned)pl.NTG;
    if (spi == 1 && pl.segs > 1) {
      U.seg = (int)(v % (unsigned)pl.segs);
      U.rb = (int)(v / (unsigned)pl.segs);
    } else {
      U.seg = u % spi;
      U.rb = (int)v;
    }
    const int KS = (OUT == 1 ? pl.lh : pl.h) / kLgStepK;
    if (OUT == 1 && U.seg == 0) {
      U.k0 = 0;
      U.k1 = pl.S / kLgStepK;
    } else {
      const int s = OUT == 1 ? U.seg - 1 : U.seg;
      U.k0 = (int)((long)KS * s / pl.splits);
      U.k1 = (int)((long)KS * (s + 1) / pl.splits);
    }
    return U;
  };

  if (wv >= kLgMfma) {  // ------------------------------------------ loader
    // Loader w fills the 8-row blocks w + 4u of the weight rows (wave-uniform bases, to
    // which a load adds the lane's offset itself) and of the token rows: lane L covers row
    // L / 8 of the block at position L % 8. <0>, <1>: a block lies in one matrix, and
    // blocks past the weights repeat the last one; <2>: any number of experts, so rows
    // past the last repeat it, also inside a block. Rows past the tokens repeat the last
    // (none of these results are used).
    struct LoadP {
      const uint16_t *a[RW], *b[TW];
      uint32_t al[OUT == 2 ? RW : 1];  // the lane's byte offset in a weight block
    };
    // position L % 8 of row r holds chunk (L % 8) ^ ((r >> 1) & 7); blocks are 8 rows: r >> 1 is 4 (block) + (L >> 4)
    const uint32_t c0 = (uint32_t)((l & 7) ^ ((4 * (w & 1) + (l >> 4)) & 7)) * 16;
    auto load_params = [&](const UnitP &U) {
      LoadP P;
      const bool shared = OUT == 1 && U.seg == 0;
      const int pitch = shared ? pl.S : OUT == 1 ? pl.lh : pl.h;  // elements of a weight row, and of a token row
      const int rows = OUT == 2 ? pl.lh : pl.N;
      if (OUT != 2) P.al[0] = (uint32_t)(l >> 3) * (uint32_t)pitch * 2u + c0;
#pragma unroll
      for (int u = 0; u < RW; ++u) {
        const int row = U.rb * 32 * RW + 8 * (w + 4 * u);
        const uint16_t *base;
        if (OUT == 0 && row < pl.N && row >= pl.lh) {  // pair tile sr / 16: 8 gate rows, then the same 8 up rows
          const int sr = row - pl.lh;
          base = ((sr & 8) ? wc : wb) + (size_t)(8 * (sr >> 4)) * pl.h;
        } else if (OUT == 2) {
          const int first = min(row, rows - 1);
          base = wa + (size_t)first * pitch;
          P.al[OUT == 2 ? u : 0] = (uint32_t)min(l >> 3, rows - 1 - first) * (uint32_t)pitch * 2u + c0;
        } else {
          base = (shared ? wb : wa) + (size_t)min(row, (OUT == 0 ? pl.lh : rows) - 8) * pitch;
        }
        P.a[u] = base + U.k0 * kLgStepK;
      }
#pragma unroll
      for (int u = 0; u < TW; ++u) {
        const int t = min(U.tg * pl.TG + 8 * (w + 4 * u) + (l >> 3), pl.B - 1);
        P.b[u] = (shared ? x2 : x) + (size_t)t * pitch + c0 / 2 + U.k0 * kLgStepK;
      }
      return P;
    };
    int iu = 0, iks = 0, isl = 0;
    UnitP Ui = unit_at(0);
    LoadP P = load_params(Ui);
    constexpr int kLoads = RW + TW;
    auto issue_next = [&]() -> int {
      if (iu >= nu) return 0;
      char *base = lds + isl * Slot;
#pragma unroll
      for (int u = 0; u < RW; ++u) load_lds<16>(reinterpret_cast<const char *>(P.a[u] + iks * kLgStepK) + P.al[OUT == 2 ? u : 0], base + (w + 4 * u) * 1024);
#pragma unroll
      for (int u = 0; u < TW; ++u) load_lds<16>(P.b[u] + iks * kLgStepK, base + OffB + (w + 4 * u) * 1024);
      if (++isl == Ring) isl = 0;
      if (++iks == Ui.k1 - Ui.k0) {
        iks = 0;
        if (++iu < nu) {
          Ui = unit_at(iu);
          P = load_params(Ui);
        }
      }
      return kLoads;
    };
    int later = 0;  // loads issued after the awaited step's
    issue_next();
#pragma unroll
    for (int k = 0; k < Ahead - 1; ++k) later += issue_next();
    for (int u = 0; u < nu; ++u) {
      const UnitP U = unit_at(u);
      for (int ks = U.k0; ks < U.k1; ++ks) {
        wait_vm_upto(later);  // this step's loads have landed
        ring_barrier();       // and the MFMA waves have read the step before it
        later += issue_next() - kLoads;  // (steps hold equal numbers: the next awaited one's go out of the count)
        if (later < 0) later = 0;
      }
    }
    ring_barrier();  // the MFMA waves' barrier at the end of the last step
    return;
  }

  // ---------------------------------------------------------- MFMA wave
  constexpr int RV = RW / 2;  // the wave's row tiles
  const int wr = w >> 1, wt = w & 1;
  u32x4 fa[2][RV], fb[2][TW];  // operands of the step's two 32-k halves
  int la[2], lb[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    la[kk] = i * 128 + (((4 * kk + q) ^ ((i >> 1) & 7)) * 16);
    lb[kk] = la[kk] + OffB + wt * TW * 2048;
    la[kk] += wr * RV * 2048;
  }
  asm("" : "+v"(la[0]), "+v"(la[1]), "+v"(lb[0]), "+v"(lb[1]));
  auto read = [&](int sl, int kk) {
    const char *pa = lds + (sl * Slot + la[kk]), *pb = lds + (sl * Slot + lb[kk]);
#pragma unroll
    for (int t = 0; t < TW; ++t) fb[kk][t] = *reinterpret_cast<const u32x4 *>(pb + t * 2048);
#pragma unroll
    for (int r = 0; r < RV; ++r) fa[kk][r] = *reinterpret_cast<const u32x4 *>(pa + r * 2048);
  };
  f32x4 acc[RV][TW];
  // The MFMAs of half kk, with the other half's operand reads spread between them:
  // a wave gets 16 bytes a lane from LDS in about 31 cycles (two MFMAs' time), and
  // reads issued in a row hold up its MFMAs.
  auto multiply = [&](int kk) {
#pragma unroll
    for (int r = 0; r < RV; ++r)
#pragma unroll
      for (int t = 0; t < TW; ++t) acc[r][t] = mfma16(as_bf16x8(fa[kk][r]), as_bf16x8(fb[kk][t]), acc[r][t]);
#pragma unroll
    for (int n = 0; n < RV + TW; ++n) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                            // an LDS read
      __builtin_amdgcn_sched_group_barrier(0x8, (RV * TW) / (RV + TW), 0);          // MFMAs
    }
    __builtin_amdgcn_sched_group_barrier(0x8, RV * TW, 0);
  };
  int g = 0;
  ring_barrier();
  read(0, 0);
  for (int u = 0; u < nu; ++u) {
    const UnitP U = unit_at(u);
#pragma unroll
    for (int r = 0; r < RV; ++r)
#pragma unroll
      for (int t = 0; t < TW; ++t) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int ks = U.k0; ks < U.k1; ++ks) {
      read(g, 1);
      multiply(0);
      __builtin_amdgcn_sched_barrier(0);
      ring_barrier();  // (waits for the reads of the second half too: the slot is free after it)
      g = g + 1 == Ring ? 0 : g + 1;
      read(g, 0);      // (after the last segment: a stale slot, unused)
      multiply(1);
      __builtin_amdgcn_sched_barrier(0);
    }
    // lane (token column i, q) holds rows 4q .. 4q + 3 of each tile
    const int row0 = U.rb * 32 * RW + wr * RV * 16;
    const int tend = min(pl.B, (U.tg + 1) * pl.TG);
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      const int tok = U.tg * pl.TG + (wt * TW + t) * 16 + i;
      const bool ok = tok < tend;
#pragma unroll
      for (int r = 0; r < RV; ++r) {
        const int row = row0 + 16 * r;
        if (row >= pl.N) break;  // wave-uniform (N: whole tiles)
        const f32x4 c = acc[r][t];
        if (OUT == 2 || pl.splits > 1) {
          if (ok) *reinterpret_cast<f32x4 *>(part + ((size_t)U.seg * pl.B + tok) * pl.N + row + 4 * q) = c;
        } else if constexpr (OUT == 1) {
          u32x2 *dst = reinterpret_cast<u32x2 *>(ya + (size_t)(ok ? tok : 0) * pl.h + row + 4 * q);
          if (U.seg == 0) {
            if (ok) *dst = pack_bf16x4(c[0], c[1], c[2], c[3]);
          } else if (ok) {
            const u32x2 s = *dst;  // the shared part
            *dst = pack_bf16x4(round_bf16(c[0]) + bf16_bits_to_f32(s[0] & 0xFFFFu), round_bf16(c[1]) + bf16_bits_to_f32(s[0] >> 16),
                               round_bf16(c[2]) + bf16_bits_to_f32(s[1] & 0xFFFFu), round_bf16(c[3]) + bf16_bits_to_f32(s[1] >> 16));
          }
        } else if (row < pl.lh) {
          if (ok) *reinterpret_cast<u32x2 *>(ya + (size_t)tok * pl.lh + row + 4 * q) = pack_bf16x4(c[0], c[1], c[2], c[3]);
        } else {  // lanes q < 2 hold gate rows, lanes q + 2 the same up rows
          float hv[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const float up = shfl_xor(c[v], 32);
            hv[v] = apply_act(pl.act, round_bf16(c[v]), round_bf16(up));
          }
          if (ok && q < 2)
            *reinterpret_cast<u32x2 *>(yb + (size_t)tok * pl.S + (row - pl.lh) / 2 + 4 * q) = pack_bf16x4(hv[0], hv[1], hv[2], hv[3]);
        }
      }
    }
  }
}

// Sums the k splits' partials of k_lgemm<OUT> in split order and writes its
// outputs: one thread per token and 4 rows (<0>'s pair tiles: 4 gate rows and their up rows).
template <int OUT>
__global__ __launch_bounds__(256) void k_lreduce(LgPlan pl, const float *__restrict__ part, uint16_t *__restrict__ ya,
                                                uint16_t *__restrict__ yb) {
  const int N4 = pl.N / 4;
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (long)pl.B * N4) return;
  const int t = (int)(idx / N4), row = (int)(idx % N4) * 4;
  const size_t seg = (size_t)pl.B * pl.N;
  auto sum = [&](int r, int s0) {
    const float *src = part + (size_t)t * pl.N + r + s0 * seg;
    f32x4 v = *reinterpret_cast<const f32x4 *>(src);
    for (int s = s0 + 1; s < pl.segs; ++s) {
      src += seg;
      const f32x4 o = *reinterpret_cast<const f32x4 *>(src);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = __fadd_rn(v[j], o[j]);
    }
    return v;
  };
  if (OUT) {
    const f32x4 c = sum(row, 1), s = *reinterpret_cast<const f32x4 *>(part + (size_t)t * pl.N + row);
    *reinterpret_cast<u32x2 *>(ya + (size_t)t * pl.h + row) =
        pack_bf16x4(round_bf16(c[0]) + round_bf16(s[0]), round_bf16(c[1]) + round_bf16(s[1]),
                    round_bf16(c[2]) + round_bf16(s[2]), round_bf16(c[3]) + round_bf16(s[3]));
  } else if (row < pl.lh) {
    const f32x4 c = sum(row, 0);
    *reinterpret_cast<u32x2 *>(ya + (size_t)t * pl.lh + row) = pack_bf16x4(c[0], c[1], c[2], c[3]);
  } else if (!(row & 8)) {
    const f32x4 gt = sum(row, 0), up = sum(row + 8, 0);
    float hv[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) hv[v] = apply_act(pl.act, round_bf16(gt[v]), round_bf16(up[v]));
    const int sr = row - pl.lh;
    *reinterpret_cast<u32x2 *>(yb + (size_t)t * pl.S + 8 * (sr >> 4) + (sr & 7)) = pack_bf16x4(hv[0], hv[1], hv[2], hv[3]);
  }
}

// en[t] = bf16(bf16(e r) w), e = bf16(expert_sum[t]), r = 1 / sqrt(mean(e^2) + eps)
// (kimi.py:325, common.py:13-21): one workgroup per token, the row read once (it
// stays in registers up to a width of 4096).
__global__ __launch_bounds__(256) void k_lnorm(int lh, const float *__restrict__ esum,
                                              const uint16_t *__restrict__ norm, uint16_t *__restrict__ en) {
  constexpr int kHeld = 4;
  __shared__ float s_sum[4];
  const int tid = threadIdx.x;
  const float *row = esum + (size_t)blockIdx.x * lh;
  f32x4 v[kHeld];
  float ss = 0.f;
  auto square = [&](const f32x4 &c) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float e = round_bf16(c[j]);
      ss += e * e;
    }
  };
#pragma unroll
  for (int m = 0; m < kHeld; ++m) {
    const int k = 4 * (tid + 256 * m);
    v[m] = k < lh ? *reinterpret_cast<const f32x4 *>(row + k) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int m = 0; m < kHeld; ++m) square(v[m]);
  for (int k = 4 * (tid + 256 * kHeld); k < lh; k += 1024) square(*reinterpret_cast<const f32x4 *>(row + k));
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) ss += shfl_xor(ss, m);
  if ((tid & 63) == 0) s_sum[tid >> 6] = ss;
  __syncthreads();
  const float tot = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
  const float r = 1.0f / __fsqrt_rn(tot / (float)lh + kLatRmsEps);
  auto put = [&](int k, const f32x4 &c) {
    const u32x2 wp = *reinterpret_cast<const u32x2 *>(norm + k);
    float o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t wbits = j & 1 ? wp[j >> 1] >> 16 : wp[j >> 1] & 0xFFFFu;
      o[j] = round_bf16(round_bf16(c[j]) * r) * bf16_bits_to_f32(wbits);
    }
    *reinterpret_cast<u32x2 *>(en + (size_t)blockIdx.x * lh + k) = pack_bf16x4(o[0], o[1], o[2], o[3]);
  };
#pragma unroll
  for (int m = 0; m < kHeld; ++m) {
    const int k = 4 * (tid + 256 * m);
    if (k < lh) put(k, v[m]);
  }
  for (int k = 4 * (tid + 256 * kHeld); k < lh; k += 1024) put(k, *reinterpret_cast<const f32x4 *>(row + k));
}

}  // namespace k3moe
