// Grouped expert GEMMs of the general path (batches past the decode kernel's):
// gate/up and down projections of kimi.py:321-322 as one GEMM per active expert, on
// the bf16 MFMA with the MXFP4 weights decoded in registers, or (FP4) on the scaled
// FP4 MFMA with the weights as stored and two-term activations (k3moe_fgemm.hpp).
//
// Unit = (group j, row block nb). A group is up to SM = 32, 64 or 96 of one active
// expert's token-expert pairs, an expert's groups of equal size (the group table of
// k_group_scan); a row block is gate/up: 128 rows of I and the same up rows, down:
// 256 rows of the hidden dimension. Twelve waves, three per SIMD: waves 8-11 issue
// loads and nothing else, waves 0-7 multiply. Loader 8 + w feeds row group w's four
// 16-row weight tiles (gate/up: gate rows 32w + 16r, r < 2, and the same up rows, so
// the activation is applied in registers; down: rows 64w + 16r). Operands move one
// 128-k step at a time through Ring LDS slots filled by direct-to-LDS loads Ring - 1
// steps ahead, one barrier per step: at SM = 32, 64 KiB of weights in flight per CU.
// The loaders run over unit boundaries, so the stream goes on through the MFMA
// waves' epilogues; their waits allow exactly the loads issued after the awaited
// step's.
//
// LDS slot: the activation rows (bf16: SM x 256 bytes, the 16-byte chunk c of row r at
// position c ^ s_swizzle(r); FP4: the hi rows, then the lo rows, SM x 128 bytes each,
// chunk c at c ^ ((r >> 1) & 7), then their scale dwords), then the 16 weight tiles
// (block q of row i at position 4 i + (q ^ a_swizzle(i)), one MXFP4 block each). Only
// the row blocks that hold tokens are loaded; columns without a token multiply
// whatever the slot held and are never stored (an MFMA's columns are independent).
// Weight scales: rows of whole 16-byte words (KB % 16 == 0) go through two buffers in
// chunks of ScSteps steps (4 ScSteps bytes of a row at a time: read 4 bytes per step,
// each line was fetched about ten times), other rows 4 bytes per step.
//
// Schedule: a persistent grid; XCD x takes the groups [J x / 8, J (x + 1) / 8) and its
// workgroups the XCD's units in turn, so that the row blocks of a group, and an
// expert's groups, run on one XCD at about the same time.
//
// Measured (gate/up + down us; per-16-token streams and the former FP4 GEMMs, whose
// loads ran two steps ahead of four MFMA waves, in brackets): a TP8 rank's shard at 203
// tokens 140 + 80 (286 + 100), at 700 199 + 101 (620 + 154), at 2999 304 + 200 (314 + 303); the
// unsharded experts at 4096 2283 + 1199 (2678 + 1209), at 700 1299 + 653 (3658 + 1489); the
// Kimi rank at 777 319 + 178 (754 + 245; 282 + 161 before the clock falls). At 203 tokens HBM
// bounds it (740 MB of gate/up weights at 5.3 TB/s). At 85 tokens per expert timing builds of the
// bf16 form took 1604 us with neither loads nor decode (the matrix cores' rate of a
// large library product), 1951 without the loads, 1777 without the MFMAs.
#pragma once

#include "k3moe_device.hpp"
#include "k3moe_fgemm.hpp"
#include "k3moe_plan.hpp"

namespace k3moe {

constexpr int kSMfma = 8;                        // MFMA waves: 4 row groups x 2 halves of the token tiles
constexpr int kSThreads = (kSMfma + 4) * 64;     // and 4 loaders

// LDS layout of a variant: operand form, SM pairs per unit, Ring slots, ScSteps k-steps per weight-scale chunk.
template <bool FP4, int SM, int Ring, int ScSteps>
struct SGeom {
  static constexpr int ahead = Ring - 1;          // k-steps of loads in flight ahead of the current one
  static constexpr int off_xs = SM * 256;         // FP4: the rows' scale dwords, hi then lo
  static constexpr int off_w = off_xs + (FP4 ? 1024 : 0);  // weight tiles of a slot
  static constexpr int slot = off_w + 16 * 1024;
  static constexpr int sc_buf = 256 * 4 * ScSteps;   // one chunk of the unit's 256 weight rows
  static constexpr int off_sc = Ring * slot;         // two chunk buffers, or Ring pieces of 1 KiB
  static constexpr int row_words = SM > 64 ? 128 : 64;
  static constexpr int off_row = off_sc + 2 * sc_buf;  // gate/up: each loader's token rows, two units
  static constexpr int lds = off_row + 4 * 2 * row_words * 4;
  static constexpr int row_loads = FP4 ? SM / 32 : SM / 16;  // a loader's blocks of activation rows (FP4: 8 rows of each term; 4 rows)
  static_assert(!FP4 || SM % 32 == 0);
  static_assert(!FP4 || SM <= 128, "the scale dwords' KiB");
  static_assert(SM % 16 == 0 && SM <= 128 && (ScSteps == 16 || ScSteps == 8));
  static_assert(Ring * 1024 <= 2 * sc_buf, "the per-step scale pieces fit the chunk buffers");
  static_assert(lds <= kDecMaxLds);
};

// Entry j of the group table: {expert, first pair, pairs}, read by scalar loads
// (written by k_group_scan, an earlier launch).
struct GroupEntry {
  int e, p0, m;
};
__device__ __forceinline__ GroupEntry group_entry(const char *tab, int j) {
  typedef const int __attribute__((address_space(4))) cint;
  const cint *src = reinterpret_cast<const cint *>(reinterpret_cast<uint64_t>(tab) + (uint64_t)(uint32_t)j * 16u);
  return GroupEntry{src[0], src[1], src[2]};
}

// Position of a 256-byte activation row's 16-byte chunk c: c ^ s_swizzle(row). A
// b128 LDS read takes its lanes sixteen at a time (0-3, 12-15, 20-23, 24-27 and the
// complements), four rows of one k quarter with four others' of the next: those
// fall on distinct banks this way (with c ^ row they meet two by two).
__device__ __forceinline__ int s_swizzle(int row) {
  const int r = row & 15;
  return r ^ ((((r >> 3) ^ (r >> 2)) & 1) << 2);
}

// A weight tile's 1 KiB in LDS: block q of row i at position 4 i + (q ^
// a_swizzle(i)). A direct-to-LDS load puts lane L's 16 bytes at position L, so four
// lanes in a row read a row's 64 contiguous bytes: with the A operand's lane order
// (16 rows, then the next block) as the order of the load, every 16 lanes touch 16
// lines, which the address unit takes at 16 bytes a cycle instead of over 60. The
// swizzle keeps the operand's LDS reads, in that order, on distinct banks.
__device__ __forceinline__ int a_swizzle(int row) { return (0 - (row >> 2)) & 3; }

// Waits until at most n (wave-uniform, 0 .. 40) of this wave's loads are in flight.
__device__ __forceinline__ void wait_vm_upto(int n) {
  switch (n) {
#define K3_W(k) case k: wait_vm<k>(); break;
    K3_W(1) K3_W(2) K3_W(3) K3_W(4) K3_W(5) K3_W(6) K3_W(7) K3_W(8) K3_W(9) K3_W(10)
    K3_W(11) K3_W(12) K3_W(13) K3_W(14) K3_W(15) K3_W(16) K3_W(17) K3_W(18) K3_W(19) K3_W(20)
    K3_W(21) K3_W(22) K3_W(23) K3_W(24) K3_W(25) K3_W(26) K3_W(27) K3_W(28) K3_W(29) K3_W(30)
    K3_W(31) K3_W(32) K3_W(33) K3_W(34) K3_W(35) K3_W(36) K3_W(37) K3_W(38) K3_W(39) K3_W(40)
#undef K3_W
    default: wait_vm<0>(); break;
  }
}

// Two row tiles' packed bf16 quads of a token column (lane q: rows 4q .. 4q+3 of
// tile 0 in a, of tile 1 in b) -> eight consecutive rows per lane: lane q holds
// rows 8 (q / 2) .. + 7 of tile q & 1.
__device__ __forceinline__ u32x4 join_rows(u32x2 a, u32x2 b) {
  u32x4 o;
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const auto s = __builtin_amdgcn_permlane16_swap(a[d], b[d], false, false);
    o[d] = s[0];
    o[2 + d] = s[1];
  }
  return o;
}

__device__ __forceinline__ u32x2 pack_bf16x4(float a, float b, float c, float d) {
  return u32x2{(uint32_t)f32_to_bf16_bits(a) | ((uint32_t)f32_to_bf16_bits(b) << 16),
               (uint32_t)f32_to_bf16_bits(c) | ((uint32_t)f32_to_bf16_bits(d) << 16)};
}

// GU: gate/up of the gathered rows of act [B, K] -> h (pl.act applied); otherwise
// down of the pair rows of act = h [P, I] -> y. FP4: activations and h as two E4M3
// terms, otherwise bf16.
template <bool GU, bool FP4, int SM, int Ring, int ScSteps>
__global__ __launch_bounds__(kSThreads, 1) void k_sgemm(Plan pl, MxAct act,
                                                       const uint8_t *__restrict__ blk0,
                                                       const uint8_t *__restrict__ scl0,
                                                       const uint8_t *__restrict__ blk1,
                                                       const uint8_t *__restrict__ scl1, char *ws) {
  typedef SGeom<FP4, SM, Ring, ScSteps> Geo;
  constexpr int kSAhead = Geo::ahead, kSSlot = Geo::slot, kSOffW = Geo::off_w, kSOffSc = Geo::off_sc,
                kSScBuf = Geo::sc_buf, kSRowLoads = Geo::row_loads, kRowWords = Geo::row_words;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, l = tid & 63, i = l & 15, q = l >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int w = wv & 3;
  const char *gtab = ws + pl.o_gtab;
  const uint8_t *zero = reinterpret_cast<const uint8_t *>(ws + pl.o_zero);
  const int J = group_entry(ws + pl.o_nact, 0).p0;  // {active experts, groups}
  const int Kd = GU ? pl.K : pl.I;                  // reduction length, a multiple of 128
  const int KB = Kd / kBlockK, KS = Kd / 128;
  const int Nout = GU ? pl.I : pl.K;
  const int RPB = GU ? 128 : 256;                   // output rows per unit
  const int NB = (Nout + RPB - 1) / RPB;
  const int xcds = gridDim.x < 8 ? (int)gridDim.x : 8;
  const int xcd = blockIdx.x % xcds, nslot = gridDim.x / xcds, slot = blockIdx.x / xcds;
  if (slot >= nslot) return;  // (a grid that is not a multiple of the XCD count)
  const int j0 = (int)((long)J * xcd / xcds), j1 = (int)((long)J * (xcd + 1) / xcds);
  const int units = (j1 - j0) * NB;
  // round u of the XCD's units: this workgroup takes position slot + 17 u (mod nslot) of the
  // round, so that no workgroup meets an expert's larger or smaller group every time
  const int full = units / nslot;
  const int nu = full + ((slot + 17 * full) % nslot < units - full * nslot ? 1 : 0);  // this workgroup's units
  if (nu == 0) return;
  const bool wide = KB % 16 == 0;
  const int NSC = (KS + ScSteps - 1) / ScSteps;

  struct UnitP {
    int e, p0, m, nb;
  };
  auto unit_at = [&](int u) {
    const unsigned v = (unsigned)(u * nslot + (slot + 17 * u) % nslot);
    const unsigned jj = v / (unsigned)NB;
    const GroupEntry g = group_entry(gtab, j0 + (int)jj);
    return UnitP{g.e, g.p0, g.m, (int)(v - jj * (unsigned)NB)};
  };

  if (wv >= kSMfma) {  // ------------------------------------------- loader
    const int *ptok = reinterpret_cast<const int *>(ws + pl.o_ptok);
    int *rows = reinterpret_cast<int *>(lds + Geo::off_row) + w * 2 * kRowWords;  // [2][kRowWords]
    // the token rows of unit U into buffer buf (lanes past its pairs repeat the last one's)
    auto gather = [&](const UnitP &U, int buf) {
#pragma unroll
      for (int u = 0; u < kRowWords / 64; ++u)
        load_lds<4>(ptok + U.p0 + min(64 * u + l, U.m - 1), reinterpret_cast<char *>(rows + buf * kRowWords + 64 * u));
    };
    struct LoadP {  // one unit's load addresses for this lane
      const uint8_t *w[4], *s[4];  // weight tile rows (the lane's block of its row), scale rows
      const uint8_t *sn;           // scale row of the lane's row (tile q, row i), for rows of no whole words
      const uint8_t *x[kSRowLoads];  // bf16 rows; FP4: the hi rows
      const uint8_t *xs;             // FP4: the lane's row of scales
      int nx;                        // blocks of activation rows of this loader that hold tokens
    };
    auto load_params = [&](const UnitP &U, int buf) {
      LoadP P;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int orow = min(U.nb * RPB + (GU ? 32 * w + 16 * (r & 1) : 64 * w + 16 * r), Nout - 16);
        const size_t row = (size_t)U.e * Nout + orow;
        P.w[r] = (GU && r >= 2 ? blk1 : blk0) + (row + (l >> 2)) * KB * 16 + ((l & 3) ^ a_swizzle(l >> 2)) * 16;
        P.s[r] = (GU && r >= 2 ? scl1 : scl0) + row * KB;
      }
      {
        const int orow = min(U.nb * RPB + (GU ? 32 * w + 16 * (q & 1) : 64 * w + 16 * q), Nout - 16);
        P.sn = (GU && q >= 2 ? scl1 : scl0) + ((size_t)U.e * Nout + orow + i) * KB;
      }
      P.nx = 0;
#pragma unroll
      for (int u = 0; u < kSRowLoads; ++u) {
        const int r0 = (FP4 ? 8 : 4) * (w + 4 * u), r = r0 + (FP4 ? l >> 3 : q);
        P.nx += r0 < U.m ? 1 : 0;
        const int rc = min(r, U.m - 1);
        const size_t arow = GU ? (size_t)rows[buf * kRowWords + rc] : (size_t)(U.p0 + rc);
        if constexpr (FP4) P.x[u] = act.hi + arow * Kd + ((l & 7) ^ ((r >> 1) & 7)) * 16;
        else P.x[u] = act.hi + (arow * Kd + (i ^ s_swizzle(r)) * 8) * 2;
      }
      if constexpr (FP4) {  // loader w: the scale dwords 64 w + L, the rows' hi ones, then their lo ones
        const int d = 64 * w + l, r = d < SM ? d : d - SM;
        const int rc = min(min(r, SM - 1), U.m - 1);
        const size_t arow = GU ? (size_t)rows[buf * kRowWords + rc] : (size_t)(U.p0 + rc);
        P.xs = (d < SM ? act.shi : act.slo) + arow * KB;
      }
      return P;
    };
    auto chunk_at = [&](int s) {
      return s == 0 || (s >= kSAhead && (s - kSAhead) % ScSteps == 0 && (s - kSAhead) / ScSteps + 1 < NSC);
    };
    // the loads of step ks of unit P into ring slot sl; cb0: the unit's first chunk number.
    // Returns their number.
    auto issue = [&](const LoadP &P, int ks, int sl, int cb0) -> int {
      char *base = lds + sl * kSSlot;
      int n = 4 + (FP4 ? 2 : 1) * P.nx;
      if constexpr (FP4) {
        if (64 * w < 2 * SM) {  // wave-uniform
          load_lds<4>(P.xs + 4 * ks, base + Geo::off_xs + w * 256);
          n += 1;
        }
      }
      if (!wide) {  // lane L: step ks's 4 scale bytes of row L of the 64
        load_lds<4>(P.sn + 4 * ks, lds + kSOffSc + sl * 1024 + w * 256);
        n += 1;
      } else if (chunk_at(ks)) {
        // lane L: 16 bytes of one row's chunk (zero area past the row). ScSteps 16: row L / 4,
        // one tile a load; 8: row L / 2 of 32, two tiles a load; a row's words rotated by its
        // number, so that 16 rows' bytes of one step lie in distinct banks. The chunk
        // replaces chunk c - 2, whose last step's reads are done at this step's issue.
        const int c = ks == 0 ? 0 : (ks - kSAhead) / ScSteps + 1;
        char *const dst = lds + kSOffSc + ((cb0 + c) & 1) * kSScBuf + 4 * w * (64 * ScSteps);
        if constexpr (ScSteps == 16) {
          const int at = 64 * c + 16 * ((l & 3) ^ ((l >> 4) & 3));
#pragma unroll
          for (int r = 0; r < 4; ++r) load_lds<16>(at < KB ? P.s[r] + (size_t)(l >> 2) * KB + at : zero, dst + r * 1024);
          n += 4;
        } else {
          const int at = 32 * c + 16 * ((l & 1) ^ ((l >> 4) & 1));
#pragma unroll
          for (int r = 0; r < 4; r += 2) {
            const uint8_t *row = (l < 32 ? P.s[r] : P.s[r + 1]) + (size_t)((l >> 1) & 15) * KB;
            load_lds<16>(at < KB ? row + at : zero, dst + r * 512);
          }
          n += 2;
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) load_lds<16>(P.w[r] + ks * 64, base + kSOffW + (4 * w + r) * 1024);
#pragma unroll
      for (int u = 0; u < kSRowLoads; ++u)
        if (u < P.nx) {
          if constexpr (FP4) {
            load_lds<16>(P.x[u] + ks * 128, base + 8 * (w + 4 * u) * 128);
            load_lds<16>(P.x[u] + (act.lo - act.hi) + ks * 128, base + SM * 128 + 8 * (w + 4 * u) * 128);
          } else {
            load_lds<16>(P.x[u] + ks * 256, base + 4 * (w + 4 * u) * 256);
          }
        }
      return n;
    };
    // the stream: step iks of unit iu is the next to go out
    int iu = 0, iks = 0, isl = 0, cbi = 0;
    UnitP Ui = unit_at(0), Un = nu > 1 ? unit_at(1) : Ui;
    if (GU) {
      gather(Ui, 0);
      wait_vm<0>();
    }
    LoadP P = load_params(Ui, 0);
    auto issue_next = [&]() -> int {
      if (iu >= nu) return 0;
      int n = 0;
      if (iks == 0) {
        if (iu > 0) {  // its rows (gate/up) landed with step 0 of the previous unit
          P = load_params(Un, iu & 1);
          if (iu + 1 < nu) Un = unit_at(iu + 1);
        }
        if (GU && iu + 1 < nu) {
          gather(Un, (iu + 1) & 1);
          n = kRowWords / 64;
        }
      }
      n += issue(P, iks, isl, cbi);
      if (++isl == Ring) isl = 0;
      if (++iks == KS) {
        iks = 0;
        ++iu;
        cbi += NSC;
      }
      return n;
    };
    issue_next();
    int cn[kSAhead - 1], later = 0;  // loads of the steps after the current one, and their sum
#pragma unroll
    for (int k = 0; k < kSAhead - 1; ++k) later += cn[k] = issue_next();
    for (int u = 0; u < nu; ++u)
      for (int ks = 0; ks < KS; ++ks) {
        wait_vm_upto(later);  // this step's loads have landed
        ring_barrier();       // and the MFMA waves have read the step before it
        later -= cn[0];
#pragma unroll
        for (int k = 0; k + 1 < kSAhead - 1; ++k) cn[k] = cn[k + 1];
        later += cn[kSAhead - 2] = issue_next();
      }
    ring_barrier();  // the MFMA waves' barrier at the end of the last step
    return;
  }

  // ---------------------------------------------------------- MFMA wave
  // Wave w + 4 half takes the row group w's four tiles for the token tiles t = 2 j +
  // half: two waves per SIMD, so that one's LDS reads and decodes run beside the
  // other's MFMAs. A step is 2 NT items of 8 MFMAs, (half of the step's 128 k, token
  // tile), tiles inside halves: a half's decoded weights are 32 registers, a whole
  // step's would be 64. The B operands are read an item ahead and the weights
  // decoded between the MFMAs of the half before. The barrier of the next step falls
  // two items before the end of a step, when every read of the step's slot has been
  // made; at a unit's end the next step is the next unit's first, read before the
  // epilogue (after the last unit the same reads find stale slots and go unused: the
  // loop keeps no branch).
  const int half = wv >> 2;
  uint16_t *out = reinterpret_cast<uint16_t *>(ws + (GU ? pl.o_h : pl.o_y));
  u32x4 wa[4];         // a step's weights as stored, and their scale bytes
  uint32_t sa[4];
  u32x4 wn[4];         // FP4: the next step's
  uint32_t sn[4];
  bf16x8 av[4][2];     // bf16: the decoded half
  u32x4 bb[2][2];      // B operands of item n in slot n & 1
  uint32_t sb[2];      // FP4: and their scale bytes
  int g = 0;           // ring slot of the step read last
  // LDS offsets of this lane, as values the compiler keeps whole (it would
  // otherwise hoist one address per tile and spill them): everything else of an
  // address is wave-uniform or an immediate
  int la = kSOffW + 4 * w * 1024 + (4 * i + (q ^ a_swizzle(i))) * 16;
  int ls = wide ? kSOffSc + (4 * w * 16 + i) * (4 * ScSteps) + q : kSOffSc + w * 256 + i * 4 + q;
  const int tile_scales = wide ? 64 * ScSteps : 64;  // bytes from one tile's scales to the next's
  const int lx = !wide ? 0 : ScSteps == 16 ? 16 * (i >> 2) : 16 * (i >> 3);  // the row's rotation
  // bf16: chunk 4q of the row (chunk 4q + kk: ^ 16 kk); FP4: chunk q (chunk 4 + q: ^ 64)
  int lb = FP4 ? half * 2048 + i * 128 + ((q ^ ((i >> 1) & 7)) * 16)
               : half * 4096 + i * 256 + (((4 * q) ^ s_swizzle(i)) * 16);
  asm("" : "+v"(la), "+v"(ls), "+v"(lb));
  auto read_a = [&](int sl, int c, int ks, u32x4 (&wa)[4], uint32_t (&sa)[4]) {
    const char *base = lds + (sl * kSSlot + la);
#pragma unroll
    for (int r = 0; r < 4; ++r) wa[r] = *reinterpret_cast<const u32x4 *>(base + r * 1024);
    const int so = wide ? (c & 1) * kSScBuf : sl * 1024, word = wide ? 4 * (ks % ScSteps) : 0;
    const int at = (word ^ lx) + ls;  // (words of 16 bytes: the xor leaves the byte in the word)
#pragma unroll
    for (int r = 0; r < 4; ++r) sa[r] = *reinterpret_cast<const uint8_t *>(lds + (so + r * tile_scales + at));
  };
  auto decode = [&](int r, int kh) {
    const float sc = e8m0_to_f32(sa[r]);
    av[r][0] = fp4x8_to_bf16(wa[r][2 * kh], sc);
    av[r][1] = fp4x8_to_bf16(wa[r][2 * kh + 1], sc);
  };
  // Item n of a step over NT tiles: bf16 (k half, tile), FP4 (tile, term). Operands of
  // the wave's j-th token tile (2 j + half), k half or term h.
  auto read_b = [&](int sl, int h, int j, int n) {
    u32x4(&b)[2] = bb[n & 1];
    if constexpr (FP4) {
      const int base = sl * kSSlot + h * SM * 128 + j * 4096;
      b[0] = *reinterpret_cast<const u32x4 *>(lds + (base + lb));
      b[1] = *reinterpret_cast<const u32x4 *>(lds + (base + (lb ^ 64)));
      sb[n & 1] = *reinterpret_cast<const uint8_t *>(lds + (sl * kSSlot + Geo::off_xs + h * SM * 4 + (2 * j + half) * 64) + (4 * i + q));
    } else {
#pragma unroll
      for (int k = 0; k < 2; ++k)
        b[k] = *reinterpret_cast<const u32x4 *>(lds + (sl * kSSlot + (lb ^ (16 * (2 * h + k)))) + j * 8192);
    }
  };
  auto tiles_of = [&](const UnitP &U) { return (((U.m + 15) >> 4) + 1 - half) >> 1; };  // the wave's token tiles of a unit

  UnitP U = unit_at(0);
  int cb0 = 0;
  ring_barrier();
  read_a(0, 0, 0, wa, sa);
  read_b(0, 0, 0, 0);
  if constexpr (!FP4) {
#pragma unroll
    for (int r = 0; r < 4; ++r) decode(r, 0);
  }
  for (int u = 0; u < nu; ++u) {
    const bool last = u + 1 == nu;
    const UnitP Un = unit_at(last ? u : u + 1);
    // the k-loop and the epilogue for NT token tiles
    auto run = [&](auto nt) {
      constexpr int NT = decltype(nt)::value, N2 = 2 * NT;
      f32x4 acc[4][NT];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int ks = 0; ks < KS; ++ks) {
        const bool inner = ks + 1 < KS;
#pragma unroll
        for (int n = 0; n < N2; ++n) {
          const int h = FP4 ? n & 1 : n / NT, t = FP4 ? n >> 1 : n % NT;  // term, or k half
          if (n + 1 < N2) read_b(g, FP4 ? (n + 1) & 1 : (n + 1) / NT, FP4 ? (n + 1) >> 1 : (n + 1) % NT, n + 1);
          if (n == N2 - 2) {
            ring_barrier();
            g = g + 1 == Ring ? 0 : g + 1;
          }
          if (n == (NT > 1 || FP4 ? N2 - 2 : 1)) {
            const int c = inner ? cb0 + (ks + 1) / ScSteps : cb0 + NSC, k1 = inner ? ks + 1 : 0;
            if constexpr (FP4) read_a(g, c, k1, wn, sn);
            else read_a(g, c, k1, wa, sa);
          }
          if (n + 1 == N2) read_b(g, 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          u32x4(&b)[2] = bb[n & 1];
          if constexpr (FP4) {
            const i32x8 b8 = {(int)b[0][0], (int)b[0][1], (int)b[0][2], (int)b[0][3],
                              (int)b[1][0], (int)b[1][1], (int)b[1][2], (int)b[1][3]};
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[r][t] = mfma_fp4x8(wa[r], b8, sa[r], sb[n & 1], acc[r][t]);
          } else if (t + 1 < NT) {
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[r][t] = mfma16(av[r][k], as_bf16x8(b[k]), acc[r][t]);
          } else {  // the half's last tile: two row tiles at a time, then their next half's weights
#pragma unroll
            for (int r0 = 0; r0 < 4; r0 += 2) {
#pragma unroll
              for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int r = r0; r < r0 + 2; ++r) acc[r][t] = mfma16(av[r][k], as_bf16x8(b[k]), acc[r][t]);
#pragma unroll
              for (int r = r0; r < r0 + 2; ++r) decode(r, h ^ 1);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (FP4) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            wa[r] = wn[r];
            sa[r] = sn[r];
          }
        }
      }

      // epilogue: lane (token column i, q) holds rows 4q .. 4q + 3 of each tile
      const int orow0 = U.nb * RPB + (GU ? 32 : 64) * w;  // first output row of the wave's tiles
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int jrow = 16 * (2 * t + half) + i;
        const bool ok = jrow < U.m;
        uint16_t *dst = out + (size_t)(U.p0 + (ok ? jrow : 0)) * Nout + orow0 + 16 * (q & 1) + 8 * (q >> 1);
        if constexpr (GU && FP4) {
          // one 32-column block of I per token: gate tiles 0, 1 with up tiles 2, 3
          float h[2][4];
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
            for (int v = 0; v < 4; ++v)
              h[s2][v] = round_bf16(fast_act(pl.act, round_bf16(acc[s2][t][v]), round_bf16(acc[2 + s2][t][v])));
          uint32_t hw[2], lw[2], sh, sl;
          mx8_split8(h, hw, lw, sh, sl);
          // eight consecutive columns per lane: of tile q & 1, from 8 (q / 2)
          const auto hs = __builtin_amdgcn_permlane16_swap(hw[0], hw[1], false, false);
          const auto ls2 = __builtin_amdgcn_permlane16_swap(lw[0], lw[1], false, false);
          if (ok) {
            const size_t p = (size_t)(U.p0 + jrow), nh = (size_t)pl.P * pl.I;
            uint8_t *const hq = reinterpret_cast<uint8_t *>(ws + pl.o_hq);
            uint8_t *const dh = hq + p * pl.I + orow0 + 16 * (q & 1) + 8 * (q >> 1);
            *reinterpret_cast<u32x2 *>(dh) = u32x2{hs[0], hs[1]};
            *reinterpret_cast<u32x2 *>(dh + nh) = u32x2{ls2[0], ls2[1]};
            if (q == 0) {
              uint8_t *const ds = hq + 2 * nh + p * (pl.I / kBlockK) + orow0 / kBlockK;
              ds[0] = (uint8_t)sh;
              ds[(size_t)pl.P * (pl.I / kBlockK)] = (uint8_t)sl;
            }
          }
        } else if constexpr (GU) {
          u32x2 hp[2];
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2) {
            float h[4];
#pragma unroll
            for (int v = 0; v < 4; ++v)
              h[v] = apply_act(pl.act, round_bf16(acc[s2][t][v]), round_bf16(acc[2 + s2][t][v]));
            hp[s2] = pack_bf16x4(h[0], h[1], h[2], h[3]);
          }
          const u32x4 o = join_rows(hp[0], hp[1]);
          if (ok) *reinterpret_cast<u32x4 *>(dst) = o;
        } else {
#pragma unroll
          for (int r = 0; r < 4; r += 2) {
            const f32x4 a0 = acc[r][t], a1 = acc[r + 1][t];
            const u32x4 o = join_rows(pack_bf16x4(a0[0], a0[1], a0[2], a0[3]), pack_bf16x4(a1[0], a1[1], a1[2], a1[3]));
            if (ok && orow0 + 16 * r < Nout) *reinterpret_cast<u32x4 *>(dst + 16 * r) = o;  // (Nout: a multiple of 32)
          }
        }
      }
    };
    const int nt = tiles_of(U);
    if (nt == 0) {  // one tile, the other half's: the steps' barriers, then the next unit's first reads
      for (int ks = 0; ks < KS; ++ks) {
        ring_barrier();
        g = g + 1 == Ring ? 0 : g + 1;
      }
      read_a(g, cb0 + NSC, 0, wa, sa);
      read_b(g, 0, 0, 0);
      if constexpr (!FP4) {
#pragma unroll
        for (int r = 0; r < 4; ++r) decode(r, 0);
      }
    } else if (SM == 32 || nt == 1) {
      run(IntC<1>{});
    } else if (SM == 64 || nt == 2) {
      run(IntC<SM >= 64 ? 2 : 1>{});
    } else {
      run(IntC<SM >= 96 ? 3 : 1>{});
    }
    U = Un;
    cb0 += NSC;
  }
}

}  // namespace k3moe
