// dedisperse.hip -- brute-force dedispersion kernels for gfx950.
//
// out[d][t] = sum_{c=0}^{C-1} in[c][t + D[c][d]]   (FP32 accumulation, channel order)
//
// Design (MI355X), tiles that read a word per add.  A workgroup of 4 wave64s owns a tile of TD = 4*MW DM
// trials x TT time samples; every wave owns MW consecutive trials and every
// lane a few samples spaced 64 (FP32) or 128 (packed pairs) apart.  Channels
// are processed in blocks: each block's input windows [t0 + D[c][d0],
// t0 + TT + D[c][d_last]) are staged into one of two LDS buffers while the
// waves add the previous block, so HBM/L2 latency overlaps the adds.  Each
// staged sample is reused by TD trials.  The per-trial offsets inside a
// window are wave-uniform and independent of the time tile: they are
// tabulated once per plan, a block's offsets sit 16 per VGPR, and one trial
// costs one DPP-broadcast address add for K LDS reads (issued in pairs as
// ds_read2st64).  These adds are bound by LDS reads, not by HBM, so the
// storage formats trade LDS bytes per add.  The register-window tiles (the
// defaults of every storage type) read a word once per wave instead of once
// per trial and are bound by instruction issue; calls of few outputs use no
// tiles at all (direct kernel).  The word-per-add formats:
//   F32  4 B per add: one float per LDS word, staged by direct buffer->LDS
//        loads (buffer_load_dword ... lds) that use no data VGPRs.
//   F16  2 B per add: LDS words hold pairs of consecutive samples in two
//        copies (even and odd alignment), so any wave-uniform offset reads
//        an aligned word; v_fma_mix_f32 (half operand selected by op_sel,
//        times 1.0, plus the FP32 accumulator) adds one half with one IEEE
//        round-to-nearest-even.  (v_dot2_f32_f16 would add two halves per
//        instruction but is not correctly rounded: it drops low bits of
//        the exact sum in cancellation and wide-exponent cases.)
//   F16_PAIRS  the F16 layout; for each trial the words of channels 2k and
//        2k+1 are added with one v_pk_add_f16 (two samples, each one IEEE
//        FP16 rounding) and the pair sum goes into the FP32 accumulators
//        with v_fma_mix_f32: three VALU instructions per four adds instead
//        of four, at about 1.7x the rounding error of F16 against FP64.
//        The pair-sum tiles build those sums once per delay difference of
//        the two channels instead and read one word per trial (one LDS word
//        and two v_fma_mix_f32 per four adds), where the survey allows.
//   U8   2 B per add: bytes widened to pairs of u16 in the same two-copy
//        layout, summed exactly with v_pk_add_u16 (two adds per
//        instruction); every <= 256 channels their high bytes move into a
//        second u16 pair accumulator (sum = 256 * high + low, exact).
// Results are bit-identical to a sequential FP32 sum in channel order (F32,
// F16 storage), to the FP32 sum of FP16 channel-pair sums (F16_PAIRS) or to
// the exact integer sum (U8).  MFMA is not used: the
// operation is shift-and-add, not a contraction.
//
// Reference counterpart: shared_dedispersion
// (src/mdsm-multibeam/multibeam_dedispersion_kernel.cu:44-95) and its
// launcher shared_brute_force (multibeam_dedispersion_thread.cu:204-221),
// which stages one channel per two barriers for a 128 x 32 tile.
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "internal.h"

namespace mdsm {
namespace {

typedef __attribute__((address_space(3))) void lds_void;
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef unsigned short ushort2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// s_waitcnt vmcnt(0) with expcnt and lgkmcnt left at their maxima (GFX9 encoding).
__device__ __forceinline__ void wait_vmem() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// One 64-dword chunk from global memory straight into LDS: lane l copies the
// dword at src + 4 l to lds_dst + 4 l (rows are shorter than 2 GiB).  The copy goes through a raw buffer
// resource whose base is src and whose size is `avail` bytes, so lanes at
// or past `avail` read 0 instead of touching memory (the hardware range
// check replaces a per-lane compare), and the only per-lane operand is the
// constant 4*lane (no 64-bit address arithmetic in VGPRs).  Dword 3 of the
// resource (0x00020000: 32-bit data format, raw addressing) is the GFX9
// family value.
__device__ __forceinline__ void chunk_to_lds(const void *src, uint32_t avail, void *lds_dst,
                                             uint32_t lane4) {
  // the operands are wave-uniform; readfirstlane keeps the resource in SGPRs
  const uint64_t a = reinterpret_cast<uint64_t>(src);
  const uint64_t au = ((uint64_t)uniform((uint32_t)(a >> 32)) << 32) | (uint64_t)uniform((uint32_t)a);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      reinterpret_cast<void *>(au), (short)0, (int)uniform(avail), 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void *)lds_dst, 4, (int)lane4, 0, 0, 0);
}

// LDS byte offsets of the wave's trials inside the windows of one channel
// block, relative to the block buffer plus the lane's own word.  Lane l of
// register n holds the offset of (r, i) = divmod(16 n + l % 16, MW) (the 16
// values repeat in each row of 16 lanes), i.e. channel cb+r and trial dw+i
// (both clamped into range), from rel = D[c][d] - D[c][d0]:
//   PACK 0 (one sample per word):  word = r*rw + rel
//   PACK 1 (pairs, window starts at element D[c][d0] of an even word
//           origin): q = rel + (D[c][d0] & 1), word = r*rw + q/2 + (q&1)*rw/2
//   PACK 2 (pairs, origin on a 4-sample boundary): as 1 with D[c][d0] & 3
// (copy P is the first half of a row, copy Q the second).  Computed once per
// block; a trial's address is then one v_add_u32 whose offset operand is
// broadcast from lane i of each row by DPP row_newbcast (no v_readlane).
template <int MW, int PACK>
__device__ __forceinline__ int32_t rel_entry(const int32_t *__restrict__ table, uint32_t ndms,
                                             uint32_t nchans, uint32_t cb, uint32_t d0,
                                             uint32_t dw, uint32_t idx, uint32_t rw) {
  const uint32_t r = idx / MW;
  const uint32_t c = min(cb + r, nchans - 1u);
  const uint32_t d = min(dw + idx % MW, ndms - 1u);
  const int32_t *row = table + (uint64_t)c * ndms;
  const int32_t base = row[d0];
  const uint32_t rel = (uint32_t)(row[d] - base);
  uint32_t w;
  if (PACK == 0) {
    w = r * rw + rel;
  } else {
    const uint32_t q = rel + ((uint32_t)base & (PACK == 1 ? 1u : 3u));
    w = r * rw + (q >> 1) + (q & 1u) * (rw >> 1);
  }
  return (int32_t)(4u * w);
}

// The offsets do not depend on the time tile, so they are tabulated once per
// plan and tile shape (trial_offset_kernel) as [DM tile][channel block][wave]
// [register][16] and each block's registers are one load per register from a
// wave-uniform base plus the lane's constant (lane % 16) word.
template <int MW, int CB, int PACK>
struct RelOffsets {
  static constexpr int N = (CB * MW + 15) / 16;
  static constexpr int WORDS = 16 * N;  // table words per (DM tile, block, wave)
  int32_t v[N];
  __device__ __forceinline__ void load(const int32_t *__restrict__ p, uint32_t lane) {
#pragma unroll
    for (int n = 0; n < N; ++n) v[n] = p[16u * n + (lane & 15u)];
  }
  // offset of (r, i) in every lane: DPP row_newbcast of lane idx % 16 (the
  // callers' loops are unrolled, so the switch folds to one case)
  __device__ __forceinline__ int32_t get(int r, int i) const {
    const int idx = r * MW + i;
    const int32_t x = v[idx >> 4];
#define MDSM_BCAST(j) \
  case j: return __builtin_amdgcn_update_dpp(0, x, 0x150 + j, 0xF, 0xF, false);
    switch (idx & 15) {
      MDSM_BCAST(0) MDSM_BCAST(1) MDSM_BCAST(2) MDSM_BCAST(3) MDSM_BCAST(4) MDSM_BCAST(5)
      MDSM_BCAST(6) MDSM_BCAST(7) MDSM_BCAST(8) MDSM_BCAST(9) MDSM_BCAST(10) MDSM_BCAST(11)
      MDSM_BCAST(12) MDSM_BCAST(13) MDSM_BCAST(14) default: return __builtin_amdgcn_update_dpp(0, x, 0x15F, 0xF, 0xF, false);
    }
#undef MDSM_BCAST
  }
};

template <typename T>
__device__ __forceinline__ const T *at_bytes(const T *p, int32_t bytes) {
  return reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + bytes);
}

// ======================================================================= F32
// BURST > 0: the LDS reads of BURST trials are issued together ahead of
// their adds (a scheduling fence keeps them grouped), so more reads are in
// flight per wave at the cost of BURST*K registers; 0 leaves the order to
// the compiler.
template <int MW, int K, int CB_, int BURST = 0>
struct F32Tile {
  static constexpr bool PAIRS = false;
  static constexpr int TT = 64 * K;
  static constexpr int TD = 4 * MW;
  static constexpr int CB = CB_;
  static constexpr int ALIGN = 1;  // ld multiple, in elements
  using T = float;

  static uint32_t row_words(uint32_t spread) { return ((uint32_t)TT + spread + 63u) & ~63u; }
  static uint32_t lds_words_per_row(uint32_t rw) { return 2u * rw; }
  static bool fits(uint32_t) { return true; }

  static constexpr int PACK = 0;
  using Rel = RelOffsets<MW, CB_, PACK>;
  __device__ __forceinline__ static void run(const float *__restrict__ in, uint64_t ld,
                             const int32_t *__restrict__ table, const int32_t *__restrict__ reltab,
                             uint32_t nchans, uint32_t nsamp, uint32_t ndms, uint32_t rw,
                             uint32_t cbr, float *__restrict__ out, uint32_t tt, uint32_t dt,
                             float *lds) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = uniform(threadIdx.x >> 6);
    const uint32_t t0 = tt * TT, d0 = dt * TD;
    const uint32_t dlast = min(d0 + TD, ndms) - 1u;
    const uint32_t dw = d0 + wave * MW;
    const uint32_t bufw = cbr * rw;  // words per LDS buffer (offsets keep the LDS address space)

    // wave w copies 64-word chunks w, w+4, ... of each row from global
    // memory straight into LDS; words past the end of the row read as 0
    // (they only feed outputs beyond nsamp)
    const uint32_t lane4 = 4u * lane;
    auto stage = [&](uint32_t cb, float *b) {
      const uint32_t nc = min(cbr, nchans - cb);
      for (uint32_t r = 0; r < nc; ++r) {
        const int32_t *trow = table + (uint64_t)(cb + r) * ndms;
        const int32_t base = trow[d0];
        const uint32_t len = (uint32_t)TT + (uint32_t)(trow[dlast] - base);
        const uint64_t g0 = (uint64_t)t0 + (uint32_t)base;
        const float *src = in + (uint64_t)(cb + r) * ld + g0;
        // bytes to the row end (rows are shorter than 2 GiB, so signed 32-bit
        // offsets hold them and the clamps stay scalar)
        const int32_t ld32 = (int32_t)ld;
        const int32_t avail = 4 * (ld32 - min((int32_t)g0, ld32));
        const uint32_t nq = (len + 63u) >> 6;
        for (uint32_t q = wave; q < nq; q += 4u) {
          const int32_t rest = max(avail - 256 * (int32_t)q, 0);
          chunk_to_lds(src + 64u * q, (uint32_t)rest, b + r * rw + 64u * q, lane4);
        }
      }
    };

    float acc[MW][K];
#pragma unroll
    for (int i = 0; i < MW; ++i)
#pragma unroll
      for (int j = 0; j < K; ++j) acc[i][j] = 0.0f;

    Rel rel, rel_next;
    const uint32_t nblocks = (nchans + cbr - 1u) / cbr;
    const int32_t *rt = reltab + ((uint64_t)dt * nblocks * 4u + wave) * Rel::WORDS;
    stage(0, lds);
    rel.load(rt, lane);
    wait_vmem();
    __syncthreads();
    uint32_t k = 0;
    for (uint32_t cb = 0; cb < nchans; cb += cbr, ++k) {
      const float *cur = lds + (k & 1u) * bufw + lane;
      const bool more = cb + cbr < nchans;
      if (more) {
        stage(cb + cbr, lds + ((k + 1u) & 1u) * bufw);
        rel_next.load(rt + (uint64_t)(k + 1u) * 4u * Rel::WORDS, lane);
      }
      const uint32_t nc = min(cbr, nchans - cb);
#pragma unroll
      for (int r = 0; r < CB; ++r) {
        if ((uint32_t)r < nc) {
          if constexpr (BURST > 0) {
#pragma unroll
            for (int i0 = 0; i0 < MW; i0 += BURST) {
              float w[BURST][K];
#pragma unroll
              for (int g = 0; g < BURST; ++g) {
                const float *p = at_bytes(cur, rel.get(r, i0 + g));
#pragma unroll
                for (int j = 0; j < K; ++j) w[g][j] = p[64 * j];
              }
              __builtin_amdgcn_sched_barrier(0);
#pragma unroll
              for (int g = 0; g < BURST; ++g)
#pragma unroll
                for (int j = 0; j < K; ++j) acc[i0 + g][j] += w[g][j];
            }
          } else {
#pragma unroll
            for (int i = 0; i < MW; ++i) {
              const float *p = at_bytes(cur, rel.get(r, i));
#pragma unroll
              for (int j = 0; j < K; ++j) acc[i][j] += p[64 * j];
            }
          }
        }
      }
      wait_vmem();
      __syncthreads();
      if (more) rel = rel_next;
    }

#pragma unroll
    for (int i = 0; i < MW; ++i) {
      const uint32_t d = dw + (uint32_t)i;
      if (d < ndms) {
        float *o = out + (uint64_t)d * nsamp;
#pragma unroll
        for (int j = 0; j < K; ++j) {
          const uint32_t t = t0 + lane + 64u * j;
          if (t < nsamp) o[t] = acc[i][j];
        }
      }
    }
  }
};

// ================================================== register-window tiles
// Tiles that read each LDS word once per wave and channel instead of once
// per trial.  A lane owns K = 20 CONSECUTIVE samples, so the words that the
// wave's MW = 4 trials need of one channel are one window of
// K + (D[last] - D[first]) FP32 words per lane.  It is read with
// ds_read_b128 (80-byte lane stride: the 8 lanes of a group cover all 32
// banks once) into fixed VGPRs, and a trial adds its K words with K plain
// v_add_f32, which this GPU issues at about 64 T lane-adds/s where
// v_fma_mix_f32, the packed 16-bit adds and any add in VGPR index mode reach
// 33-37 T (measured).  Registers cannot be indexed at that rate, so the adds
// exist once per trial and word offset (4 x 17 blocks of 20 adds, 6.4 KB of
// code) and the wave jumps from block to block: the plan's table holds, per
// channel and trial, the offset of the trial's block inside that code.
//
// Table entry of a channel and wave, 8 words: d[i] is the code offset of
// trial i's block, or of a reading stub when trial i needs another window (i
// = 0 always); e[i] then holds the block's code offset (low half) and the
// window's LDS byte offset / 16 (high half).  The stubs differ in how many
// 16-byte reads they make.
//
// Bound: instruction issue.  1024 channels x 4096 trials x 2^17 samples, F32:
// 40.5 T adds/s (18.5 with one LDS read per add), the VALU at two thirds of the
// 64 T it issues, LDS reads under half of their rate; one wave issues at most
// one instruction per about 5 clocks, so 4 waves per SIMD (128 VGPRs) set
// MW * K + WIN, and K = 20 at MW = 4 the fewest jumps (49 T without staging
// and tables; MW = 8, K = 12 at 3 waves 41 T).
//
// F16 and U8 rows are widened to FP32 in LDS by one pass per channel block
// (exact; all trials of the tile share it), so all storage types run the same adds: F16
// in FP32 channel order, U8 as exact integers (at most 65536 * 255 < 2^24).
struct WindowCode {
  static constexpr int MW = 4, K = 20;
  static constexpr int WIN = 36;                  // window words, VGPRs 92..127
  static constexpr int NV = WIN - K + 1;          // word offsets of a trial
  static constexpr int BLOCK = 96;                // code bytes per block, per stub
  static constexpr int STUB = 128, MINREADS = 6, STUBS = 4;
  static constexpr int STUB0 = MW * NV * BLOCK;   // stubs follow the blocks
  static constexpr int BYTES = STUB0 + MW * STUBS * STUB;
  static_assert(STUB0 % STUB == 0 && BYTES < 65536, "code offsets are 16 bits");
  static_assert(4 * (MINREADS + STUBS - 1) == WIN && 4 * MINREADS >= K + 3, "reads of a window");
  static_assert(MW == 4 && NV == 17 && BLOCK == 96 && STUBS == 4 && STUB == 128, "add_channel's text");
  typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));
  typedef __attribute__((address_space(4))) const u32x8 const_u32x8;

  // The entry of a channel whose trials read from LDS byte offsets
  // o[0] <= o[1] <= o[2] <= o[3] (a trial stays in the open window while its
  // words lie inside WIN).
  __device__ static void entry(const uint32_t o[MW], uint32_t *out) {
    uint32_t base = 0, rd[MW], idx[MW];
    int open = -1;
    for (int i = 0; i < MW; ++i) {
      rd[i] = 0;
      if (open < 0 || (o[i] - base) / 4u > (uint32_t)(NV - 1)) {
        base = o[i] & ~15u;
        open = i;
      }
      idx[i] = (o[i] - base) / 4u;
      rd[open] = max((uint32_t)MINREADS, (idx[i] + K + 3u) / 4u);
    }
    for (int i = 0; i < MW; ++i) {
      const uint32_t blk = ((uint32_t)i * NV + idx[i]) * BLOCK;
      out[i] = rd[i] ? (uint32_t)STUB0 + ((uint32_t)i * STUBS + rd[i] - MINREADS) * STUB : blk;
      out[MW + i] = rd[i] ? blk | ((o[i] & ~15u) >> 4 << 16) : 0u;
    }
  }

  // The adds of one channel: window reads, blocks and the jumps between them;
  // returns the entry at `next`, loaded while the adds run (the scalar loads
  // share the LDS reads' wait counter, so it is asked for after those came)
  // (s[96:97]: address of the code, s[98:99]: jump target).  The .org
  // directives place every block and stub (and fail to assemble where one is
  // too long).
#define MDSM_WIN_ADD(i, j) "v_add_f32 %[x" #i "_" #j "], v[92+" #j "+\\v], %[x" #i "_" #j "]\n\t"
#define MDSM_WIN_ADDS(i)                                                                        \
  MDSM_WIN_ADD(i, 0) MDSM_WIN_ADD(i, 1) MDSM_WIN_ADD(i, 2) MDSM_WIN_ADD(i, 3) MDSM_WIN_ADD(i, 4) \
  MDSM_WIN_ADD(i, 5) MDSM_WIN_ADD(i, 6) MDSM_WIN_ADD(i, 7) MDSM_WIN_ADD(i, 8) MDSM_WIN_ADD(i, 9) \
  MDSM_WIN_ADD(i, 10) MDSM_WIN_ADD(i, 11) MDSM_WIN_ADD(i, 12) MDSM_WIN_ADD(i, 13)               \
  MDSM_WIN_ADD(i, 14) MDSM_WIN_ADD(i, 15) MDSM_WIN_ADD(i, 16) MDSM_WIN_ADD(i, 17)               \
  MDSM_WIN_ADD(i, 18) MDSM_WIN_ADD(i, 19)
#define MDSM_WIN_JUMP(d) \
  "s_add_u32 s98, s96, " d "\n\ts_addc_u32 s99, s97, 0\n\ts_setpc_b64 s[98:99]\n\t"
#define MDSM_WIN_BLOCKS(i, next)                                                                \
  ".irp v,0,1,2,3,4,5,6,7,8,9,10,11,12,13,14,15,16\n\t" MDSM_WIN_ADDS(i) next                   \
  ".org .Lmdsm_code%=+(" #i "*17+\\v+1)*96\n\t.endr\n\t"
#define MDSM_WIN_STUB(i, n, reads, more)                                                                 \
  "s_lshr_b32 s98, %[e" #i "], 16\n\tv_lshl_add_u32 %[av], s98, 4, %[cur]\n\t"                   \
  ".irp q," reads "\n\tds_read_b128 v[92+4*\\q:95+4*\\q], %[av] offset:16*\\q\n\t.endr\n\t"      \
  "s_and_b32 s98, %[e" #i "], 0xffff\n\ts_add_u32 s98, s96, s98\n\ts_addc_u32 s99, s97, 0\n\t"   \
  "s_waitcnt lgkmcnt(0)\n\t" more "s_setpc_b64 s[98:99]\n\t"                                    \
  ".org .Lmdsm_code%=+4*17*96+(" #i "*4+" #n "+1)*128\n\t"
#define MDSM_WIN_STUBS(i, more)                                                                 \
  MDSM_WIN_STUB(i, 0, "0,1,2,3,4,5", more) MDSM_WIN_STUB(i, 1, "0,1,2,3,4,5,6", more)           \
  MDSM_WIN_STUB(i, 2, "0,1,2,3,4,5,6,7", more) MDSM_WIN_STUB(i, 3, "0,1,2,3,4,5,6,7,8", more)
#define MDSM_WIN_ACC(i)                                                                         \
  [x##i##_0] "+v"(acc[i][0]), [x##i##_1] "+v"(acc[i][1]), [x##i##_2] "+v"(acc[i][2]),            \
      [x##i##_3] "+v"(acc[i][3]), [x##i##_4] "+v"(acc[i][4]), [x##i##_5] "+v"(acc[i][5]),        \
      [x##i##_6] "+v"(acc[i][6]), [x##i##_7] "+v"(acc[i][7]), [x##i##_8] "+v"(acc[i][8]),        \
      [x##i##_9] "+v"(acc[i][9]), [x##i##_10] "+v"(acc[i][10]), [x##i##_11] "+v"(acc[i][11]),    \
      [x##i##_12] "+v"(acc[i][12]), [x##i##_13] "+v"(acc[i][13]), [x##i##_14] "+v"(acc[i][14]),  \
      [x##i##_15] "+v"(acc[i][15]), [x##i##_16] "+v"(acc[i][16]), [x##i##_17] "+v"(acc[i][17]),  \
      [x##i##_18] "+v"(acc[i][18]), [x##i##_19] "+v"(acc[i][19])
  __device__ __forceinline__ static u32x8 add_channel(float (&acc)[MW][K], uint32_t cur, u32x8 t,
                                                      const_u32x8 *next) {
    uint32_t av;
    u32x8 tn;
    asm volatile(
        "s_getpc_b64 s[96:97]\n.Lmdsm_pc%=:\n\t"
        "s_add_u32 s96, s96, .Lmdsm_code%=-.Lmdsm_pc%=\n\ts_addc_u32 s97, s97, 0\n\t"
        MDSM_WIN_JUMP("%[d0]")
        ".p2align 7\n.Lmdsm_code%=:\n\t"
        MDSM_WIN_BLOCKS(0, MDSM_WIN_JUMP("%[d1]"))
        MDSM_WIN_BLOCKS(1, MDSM_WIN_JUMP("%[d2]"))
        MDSM_WIN_BLOCKS(2, MDSM_WIN_JUMP("%[d3]"))
        MDSM_WIN_BLOCKS(3, "s_branch .Lmdsm_end%=\n\t")
        MDSM_WIN_STUBS(0, "s_load_dwordx8 %[tn], %[next], 0x0\n\t")
        MDSM_WIN_STUBS(1, "") MDSM_WIN_STUBS(2, "") MDSM_WIN_STUBS(3, "")
        ".Lmdsm_end%=:\n\ts_waitcnt lgkmcnt(0)"
        : MDSM_WIN_ACC(0), MDSM_WIN_ACC(1), MDSM_WIN_ACC(2), MDSM_WIN_ACC(3), [av] "=&v"(av),
          [tn] "=&s"(tn)
        : [cur] "v"(cur), [next] "s"(next), [d0] "s"(t[0]), [d1] "s"(t[1]), [d2] "s"(t[2]), [d3] "s"(t[3]),
          [e0] "s"(t[4]), [e1] "s"(t[5]), [e2] "s"(t[6]), [e3] "s"(t[7])
        : "v92", "v93", "v94", "v95", "v96", "v97", "v98", "v99", "v100", "v101", "v102", "v103",
          "v104", "v105", "v106", "v107", "v108", "v109", "v110", "v111", "v112", "v113", "v114",
          "v115", "v116", "v117", "v118", "v119", "v120", "v121", "v122", "v123", "v124", "v125",
          "v126", "v127", "s96", "s97", "s98", "s99", "scc", "memory");
    return tn;
  }
#undef MDSM_WIN_ACC
#undef MDSM_WIN_STUBS
#undef MDSM_WIN_STUB
#undef MDSM_WIN_BLOCKS
#undef MDSM_WIN_JUMP
#undef MDSM_WIN_ADDS
#undef MDSM_WIN_ADD

  // The wave's sums to out: a lane's 20 consecutive samples become 64-sample
  // rows through the wave's own 640 words of LDS, half of the lanes at a time.
  template <bool IS_U8>
  __device__ __forceinline__ static void store(const float (&acc)[MW][K], float *lds, uint32_t wave,
                                               uint32_t lane, float *__restrict__ out, uint32_t nsamp,
                                               uint32_t ndms, uint32_t dw, uint32_t t0, uint32_t nchans) {
    float *mine = lds + wave * 640u;
    const double base = (double)nchans * -4.0;
#pragma unroll
    for (int i = 0; i < MW; ++i) {
      const uint32_t d = dw + (uint32_t)i;
      if (d >= ndms) break;
      float *orow = out + (uint64_t)d * nsamp;
#pragma unroll
      for (uint32_t h = 0; h < 2u; ++h) {
        if ((lane >> 5) == h) {
#pragma unroll
          for (int j = 0; j < K; j += 4)
            *reinterpret_cast<float4 *>(mine + K * (lane & 31u) + j) =
                make_float4(acc[i][j], acc[i][j + 1], acc[i][j + 2], acc[i][j + 3]);
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (uint32_t j = 0; j < 10u; ++j) {
          const uint32_t t = t0 + 640u * h + lane + 64u * j;
          float v = mine[lane + 64u * j];
          if constexpr (IS_U8) v = (float)((double)(uint32_t)v * (8.0 / 255.0) + base);
          if (t < nsamp) orow[t] = v;
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
  }
};

// A workgroup is NW waves: 16 (64 trials, all 160 KB of a CU's LDS) stage and
// widen a row for twice the trials and meet at half the barriers per add of 8
// (32 trials, 80 KB): F32 40.5 against 34.6 T adds/s, F16 37.7 against 36.5,
// U8 38.3 against 37.5.  8 pads surveys of few trials less.
template <int MODE, int NW>
struct WindowTile {
  using W = WindowCode;
  static constexpr bool PAIRS = false;
  static constexpr bool IS_F32 = MODE == MDSM_F32, IS_U8 = MODE == MDSM_U8;
  static constexpr int MW = W::MW, K = W::K, WAVES = NW, THREADS = 64 * NW;
  static constexpr int TT = 64 * K, TD = NW * MW;
  static constexpr int CB = NW == 8 ? (IS_F32 ? 6 : 8) : (IS_F32 ? 12 : 16);
  // staging (and widening): WPR waves share a row of a block, every wave has
  // up to RPW rows
  static constexpr uint32_t WPR = NW == 8 && IS_F32 ? 4 : 1, RSTEP = NW / WPR, RPW = (CB + RSTEP - 1) / RSTEP;
  using T = std::conditional_t<IS_F32, float, std::conditional_t<IS_U8, uint8_t, __half>>;
  static constexpr uint32_t PER = 4u / sizeof(T);  // samples per source dword
  static uint64_t table_words(uint32_t nchans, uint32_t ndms) {
    return (uint64_t)((ndms + TD - 1u) / TD) * NW * (nchans + 1u) * 8u;
  }
  static bool fits(uint32_t) { return true; }
  // FP32 row words: the window of TT + spread samples from an origin that is
  // a multiple of PER samples; reads end up to 3 words past it
  static uint32_t row_words(uint32_t spread) { return ((uint32_t)TT + spread + 8u + 63u) & ~63u; }
  // raw source dwords per row (F16, U8)
  static __host__ __device__ uint32_t raw_words(uint32_t rw) { return IS_F32 ? rw : (rw / PER + 63u) & ~63u; }
  // F32: two buffers of rows; F16, U8: raw dwords and widened rows
  static uint32_t lds_words_per_row(uint32_t rw) { return rw + raw_words(rw); }

  __device__ __forceinline__ static void run(const T *__restrict__ in, uint64_t ld,
                                             const int32_t *__restrict__ table,
                                             const int32_t *__restrict__ reltab, uint32_t nchans,
                                             uint32_t nsamp, uint32_t ndms, uint32_t rw,
                                             uint32_t cbr, float *__restrict__ out, uint32_t tt,
                                             uint32_t dt, float *lds) {
    typedef W::u32x8 u32x8;
    typedef W::const_u32x8 const_u32x8;
    typedef __attribute__((address_space(3))) float lds_float;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = uniform(threadIdx.x >> 6);
    const uint32_t t0 = tt * TT, d0 = dt * TD;
    const uint32_t dlast = min(d0 + TD, ndms) - 1u;
    const uint32_t dw = d0 + wave * MW;
    const uint32_t rawn = raw_words(rw);
    // F32: row buffers A and B; F16, U8: widened rows and raw dwords
    float *const second = lds + cbr * rw;
    // this wave's first row of a block and its part of the row's 64-dword chunks
    const uint32_t srow = wave / WPR, part = wave % WPR;
    const uint32_t voff = 4u * lane + 256u * part;
    int32_t spos[RPW], slen[RPW];  // first delay and last of the rows the next stage() takes
    auto prefetch = [&](uint32_t cb) {
#pragma unroll
      for (uint32_t i = 0; i < RPW; ++i) {
        const int32_t *trow = table + (uint64_t)min(cb + srow + RSTEP * i, nchans - 1u) * ndms;
        spos[i] = trow[d0];
        slen[i] = trow[dlast];
      }
    };
    auto stage = [&](uint32_t cb, float *b) {
#pragma unroll
      for (uint32_t i = 0; i < RPW; ++i) {
        const uint32_t r = srow + RSTEP * i;
        if (r >= min(cbr, nchans - cb)) break;
        const uint32_t g0 = t0 + (uint32_t)spos[i];
        const uint32_t len = (uint32_t)TT + (uint32_t)(slen[i] - spos[i]) + (g0 & (PER - 1u));
        const uint32_t w0 = g0 / PER, ldw = (uint32_t)(ld / PER);  // rows < 2 GiB
        const uint32_t *src = reinterpret_cast<const uint32_t *>(in) + (uint64_t)(cb + r) * ldw + w0;
        // rows end at the resource's size: dwords past it read as 0 (they only
        // feed outputs beyond nsamp)
        const uint32_t avail = 4u * (ldw - min(w0, ldw));
        const uint64_t a = reinterpret_cast<uint64_t>(src);
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            reinterpret_cast<void *>(((uint64_t)uniform((uint32_t)(a >> 32)) << 32) | uniform((uint32_t)a)),
            (short)0, (int)uniform(avail), 0x00020000);
        const uint32_t nq = (len + 64u * PER - 1u) / (64u * PER);
        float *dst = b + r * (IS_F32 ? rw : rawn) + 64u * part;
        // (the immediate offset applies to the LDS address too)
        uint32_t q = part, vo = voff;
        for (; q + 3u * WPR < nq; q += 4u * WPR, vo += 1024u * WPR, dst += 256u * WPR) {
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void *)dst, 4, (int)vo, 0, 0, 0);
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void *)dst, 4, (int)vo, 0, 256 * (int)WPR, 0);
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void *)dst, 4, (int)vo, 0, 512 * (int)WPR, 0);
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void *)dst, 4, (int)vo, 0, 768 * (int)WPR, 0);
        }
        for (; q < nq; q += WPR, vo += 256u * WPR, dst += 64u * WPR)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void *)dst, 4, (int)vo, 0, 0, 0);
      }
    };
    // FP32 rows from the raw dwords
    auto widen = [&](uint32_t cb) {
#pragma unroll
      for (uint32_t i = 0; i < RPW; ++i) {
        const uint32_t r = srow + RSTEP * i;
        if (r >= min(cbr, nchans - cb)) break;
        const uint32_t *R = reinterpret_cast<const uint32_t *>(second) + r * rawn;
        float *P = lds + r * rw;
        for (uint32_t n = 4u * (lane + 64u * part); n < rw; n += 256u * WPR) {
          float4 v;
          if constexpr (IS_U8) {
            const uint32_t x = R[n / 4u];
            v = make_float4((float)(x & 0xFFu), (float)((x >> 8) & 0xFFu), (float)((x >> 16) & 0xFFu),
                            (float)(x >> 24));
          } else {
            const uint2 x = *reinterpret_cast<const uint2 *>(R + n / 2u);
            const half2_t a = __builtin_bit_cast(half2_t, x.x), c = __builtin_bit_cast(half2_t, x.y);
            v = make_float4((float)a.x, (float)a.y, (float)c.x, (float)c.y);
          }
          *reinterpret_cast<float4 *>(P + n) = v;
        }
      }
    };

    float acc[MW][K];
#pragma unroll
    for (int i = 0; i < MW; ++i)
#pragma unroll
      for (int j = 0; j < K; ++j) acc[i][j] = 0.0f;

    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_float *)lds + (uint32_t)(4 * K) * lane;
    // the wave's table entries, one per channel (scalar loads)
    const const_u32x8 *rt =
        (const const_u32x8 *)(uintptr_t)reltab + ((uint64_t)dt * NW + wave) * (nchans + 1u);
    prefetch(0);
    stage(0, IS_F32 ? lds : second);
    if (cbr < nchans) prefetch(cbr);
    u32x8 o = *rt;
    wait_vmem();
    __syncthreads();
    if constexpr (!IS_F32) {
      widen(0);
      __syncthreads();
    }
    uint32_t k = 0;
    for (uint32_t cb = 0; cb < nchans; cb += cbr, ++k) {
      const bool more = cb + cbr < nchans;
      if (more) {
        stage(cb + cbr, IS_F32 ? ((k & 1u) ? lds : second) : second);
        if (cb + 2u * cbr < nchans) prefetch(cb + 2u * cbr);
      }
      const uint32_t nc = min(cbr, nchans - cb);
      const uint32_t cur = lds0 + (IS_F32 ? 4u * ((k & 1u) * cbr * rw) : 0u);
      for (uint32_t r = 0; r < nc; ++r) {
        // (with the next channel's entry; one follows the last channel's)
        ++rt;
        o = W::add_channel(acc, cur, o, rt);
      }
      wait_vmem();
      __syncthreads();
      if constexpr (!IS_F32) {
        if (more) widen(cb + cbr);
        __syncthreads();
      }
    }

    W::store<IS_U8>(acc, lds, wave, lane, out, nsamp, ndms, dw, t0, nchans);
  }
};

template <typename T>
struct IsWindow : std::false_type {};
template <int MODE, int NW>
struct IsWindow<WindowTile<MODE, NW>> : std::true_type {};
// Threads per workgroup: four waves, or the window tiles' 16 or eight.
template <typename T>
constexpr int tile_threads() {
  if constexpr (IsWindow<T>::value) return T::THREADS;
  else return 256;
}

// Table of a window tile: entry ((dt * WAVES + wave) * (nchans + 1) + c) for
// channel c and trials 4 wave .. 4 wave + 3 of DM tile dt, at their samples'
// byte offsets in the block's FP32 rows (row c % cbr starts at a multiple of
// PER samples at or below the tile's first delay); entry nchans, which is
// loaded and not used, repeats the last channel's.
template <typename Tile>
__global__ __launch_bounds__(256) void window_table_kernel(const int32_t *__restrict__ table,
                                                           uint32_t nchans, uint32_t ndms,
                                                           uint32_t rw, uint32_t cbr,
                                                           uint64_t entries,
                                                           int32_t *__restrict__ reltab) {
  const uint64_t e = (uint64_t)blockIdx.x * 256u + threadIdx.x;
  if (e >= entries) return;
  const uint32_t c = min((uint32_t)(e % (nchans + 1u)), nchans - 1u);
  const uint64_t g = e / (nchans + 1u);
  const uint32_t wave = (uint32_t)(g % Tile::WAVES), dt = (uint32_t)(g / Tile::WAVES);
  const uint32_t d0 = dt * Tile::TD;
  const int32_t *row = table + (uint64_t)c * ndms;
  const uint32_t base = (uint32_t)row[d0], skew = base & (Tile::PER - 1u);
  uint32_t o[WindowCode::MW], w[2 * WindowCode::MW];
  for (uint32_t i = 0; i < (uint32_t)WindowCode::MW; ++i) {
    const uint32_t d = min(d0 + wave * WindowCode::MW + i, ndms - 1u);
    o[i] = 4u * (c % cbr * rw + skew + ((uint32_t)row[d] - base));
  }
  WindowCode::entry(o, w);
  for (int i = 0; i < 2 * WindowCode::MW; ++i) reltab[e * 8u + i] = (int32_t)w[i];
}

// ============================================================ packed (F16, U8)
// LDS row of a channel: copy P (words 0..wp-1) then copy Q (words wp..2wp-1).
// With f the even word origin of the row window (elements 2f, 2f+1, ... of
// the global row), P[w] = (e[2(f+w)], e[2(f+w)+1]) and Q[w] = (e[2(f+w)+1],
// e[2(f+w)+2]) as two 16-bit halves.  For the window start a = g0 + rel of a
// trial (wave-uniform), the lane's pair (a + 2 lane + 128 j, +1) is word
// (a>>1) - f + lane + 64 j of copy (a & 1).
template <int MW, int K2, int CB_>
struct PackedGeom {
  static constexpr int TT = 128 * K2;
  static constexpr int TD = 4 * MW;
  static constexpr int CB = CB_;
  static uint32_t copy_words(uint32_t spread) {
    return ((uint32_t)(64 * K2) + (spread + 4u) / 2u + 2u + 63u) & ~63u;
  }
  static uint32_t row_words(uint32_t spread) { return 2u * copy_words(spread); }
};

// Packed tiles (F16 and U8 storage, rows 4-byte aligned).  Per channel block
// the raw dwords of each window are copied into LDS by direct global->LDS
// loads while the previous block is added; after the barrier one LDS->LDS
// pass builds the pair copies (F16: P is the copy itself and Q its 16-bit
// funnel shift; U8: bytes widened to u16 pairs with v_perm into P and Q).
template <int MODE, int MW, int K2, int CB_, int BURST = 0>
struct PackedTile : PackedGeom<MW, K2, CB_> {
  using G = PackedGeom<MW, K2, CB_>;
  static constexpr int TT = G::TT, TD = G::TD, CB = CB_;
  static constexpr bool IS_U8 = MODE == MDSM_U8;
  // F16_PAIRS: channel blocks hold an even number of rows (stage_channels)
  static constexpr bool PAIRS = MODE == MDSM_F16_PAIRS;
  static_assert(!PAIRS || CB_ % 2 == 0, "F16_PAIRS tiles stage whole channel pairs");
  using T = std::conditional_t<IS_U8, uint8_t, __half>;
  static bool fits(uint32_t) { return true; }
  // raw staging dwords per row (U8): wp/2 + 2 source dwords, padded to 64
  static __host__ __device__ uint32_t raw_words(uint32_t rw) {
    return IS_U8 ? ((rw / 4u + 2u + 63u) & ~63u) : 0u;
  }
  static uint32_t row_words(uint32_t spread) { return G::row_words(spread); }
  static uint32_t lds_words_per_row(uint32_t rw) { return 2u * rw + raw_words(rw); }

  static constexpr int PACK = IS_U8 ? 2 : 1;
  using Rel = RelOffsets<MW, CB_, PACK>;
  __device__ __forceinline__ static void run(const T *__restrict__ in, uint64_t ld,
                                             const int32_t *__restrict__ table,
                                             const int32_t *__restrict__ reltab, uint32_t nchans,
                                             uint32_t nsamp, uint32_t ndms, uint32_t rw,
                                             uint32_t cbr, float *__restrict__ out, uint32_t tt,
                                             uint32_t dt, float *ldsf) {
    uint32_t *lds = reinterpret_cast<uint32_t *>(ldsf);
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u;
    const uint32_t wave = uniform(tid >> 6);
    const uint32_t t0 = tt * TT, d0 = dt * TD;
    const uint32_t dw = d0 + wave * MW;
    const uint32_t wp = rw / 2u;
    const uint32_t rawn = raw_words(rw);
    const uint64_t ldw = IS_U8 ? ld / 4u : ld / 2u;  // source dwords per row
    const uint32_t *src32 = reinterpret_cast<const uint32_t *>(in);
    const uint32_t bufw = cbr * rw;  // words per LDS buffer (offsets keep the LDS address space)
    uint32_t *raw = lds + 2u * cbr * rw;

    auto g0_of = [&](uint32_t c) { return t0 + (uint32_t)table[(uint64_t)c * ndms + d0]; };
    // copy the window dwords of rows [cb, cb+nc) into P of buffer b (F16) or
    // into the raw area (U8); wave w takes 64-dword chunks w, w+4, ...;
    // dwords past the end of the row read as 0
    const uint32_t lane4 = 4u * lane;
    // the window starts of the rows the next stage() takes, loaded one block
    // ahead so that their scalar loads do not delay the copies
    uint32_t g0pre[CB_];
    auto prefetch = [&](uint32_t cb) {
#pragma unroll
      for (int r = 0; r < CB_; ++r)
        if ((uint32_t)r < cbr && cb + (uint32_t)r < nchans) g0pre[r] = g0_of(cb + (uint32_t)r);
    };
    auto stage = [&](uint32_t cb, uint32_t *b) {
      const uint32_t nc = min(cbr, nchans - cb);
#pragma unroll
      for (int rr = 0; rr < CB_; ++rr) {
        if ((uint32_t)rr >= nc) break;
        const uint32_t r = (uint32_t)rr;
        const uint32_t g0 = g0pre[rr];
        const uint64_t w0 = IS_U8 ? (g0 >> 2) : (g0 >> 1);
        const uint32_t *src = src32 + (uint64_t)(cb + r) * ldw + w0;
        const int32_t ldw32 = (int32_t)ldw;  // rows < 2 GiB
        const int32_t avail = 4 * (ldw32 - min((int32_t)w0, ldw32));
        uint32_t *dst = IS_U8 ? raw + r * rawn : b + r * rw;
        const uint32_t n = IS_U8 ? rawn : wp;
        for (uint32_t q = wave; 64u * q < n; q += 4u) {
          const int32_t rest = max(avail - 256 * (int32_t)q, 0);
          chunk_to_lds(src + 64u * q, (uint32_t)rest, dst + 64u * q, lane4);
        }
      }
    };
    // build the pair copies of rows [cb, cb+nc) in buffer b
    // (F16: wave w builds rows w, w+4, ..., four Q words per lane from one
    // 16-byte and one 4-byte LDS read; Q[wp-1], which no trial reads, may
    // take the stale word past P.  U8: also one wave per row.)
    auto build = [&](uint32_t cb, uint32_t *b) {
      const uint32_t nc = min(cbr, nchans - cb);
      if (IS_U8) {
        // wave w widens rows w, w+4, ...: raw dwords n, n+1 (and n+2 for
        // the last Q word) become P words 2n..2n+3 and Q words 2n..2n+3
        // (two 16-byte writes)
        for (uint32_t r = wave; r < nc; r += 4u) {
          uint32_t *P = b + r * rw;
          uint32_t *Q = P + wp;
          const uint32_t *R = raw + r * rawn;
          // two raw dwords per lane (wp is a multiple of 64, so the four
          // P and Q words of a lane are whole 16-byte groups)
          for (uint32_t n = 2u * lane; 2u * n < wp; n += 128u) {
            const uint2 xy = *reinterpret_cast<const uint2 *>(R + n);
            const uint32_t x = xy.x, y = xy.y, z = R[n + 2];
            *reinterpret_cast<uint4 *>(P + 2 * n) =
                make_uint4(__builtin_amdgcn_perm(y, x, 0x0C010C00u), __builtin_amdgcn_perm(y, x, 0x0C030C02u),
                           __builtin_amdgcn_perm(z, y, 0x0C010C00u), __builtin_amdgcn_perm(z, y, 0x0C030C02u));
            *reinterpret_cast<uint4 *>(Q + 2 * n) =
                make_uint4(__builtin_amdgcn_perm(y, x, 0x0C020C01u), __builtin_amdgcn_perm(y, x, 0x0C040C03u),
                           __builtin_amdgcn_perm(z, y, 0x0C020C01u), __builtin_amdgcn_perm(z, y, 0x0C040C03u));
          }
        }
      } else {
        for (uint32_t r = wave; r < nc; r += 4u) {
          uint32_t *P = b + r * rw;
          uint32_t *Q = P + wp;
          // four Q words per lane (wp is a multiple of 64, rows 16-byte aligned)
          for (uint32_t w = 4u * lane; w + 3u < wp; w += 256u) {
            const uint4 a = *reinterpret_cast<const uint4 *>(P + w);
            const uint32_t c = P[w + 4];
            *reinterpret_cast<uint4 *>(Q + w) = make_uint4(__builtin_amdgcn_alignbit(a.y, a.x, 16),
                                                           __builtin_amdgcn_alignbit(a.z, a.y, 16),
                                                           __builtin_amdgcn_alignbit(a.w, a.z, 16),
                                                           __builtin_amdgcn_alignbit(c, a.w, 16));
          }
        }
        // F16_PAIRS, odd block (the last of an odd channel count): row nc,
        // inside the buffer since cbr is even, becomes the zero partner
        if (PAIRS && (nc & 1u)) {
          uint32_t *Z = b + nc * rw;
          for (uint32_t w = 4u * tid; w < rw; w += 1024u)
            *reinterpret_cast<uint4 *>(Z + w) = make_uint4(0u, 0u, 0u, 0u);
        }
      }
    };

    // F16: FP32 accumulators.  U8: two u16 pair accumulators per output
    // pair, the running sum S = 256*uhi + uacc held exactly: a fold moves
    // uacc's high bytes into uhi (three packed instructions per pair) and
    // leaves uacc <= 255, so 256 more channels of bytes fit in 16 bits, and
    // uhi <= S/256 < nchans fits while nchans <= 65536.
    float facc[IS_U8 ? 1 : MW][IS_U8 ? 1 : K2][2];
    ushort2_t uacc[IS_U8 ? MW : 1][IS_U8 ? K2 : 1];
    ushort2_t uhi[IS_U8 ? MW : 1][IS_U8 ? K2 : 1];
#pragma unroll
    for (int i = 0; i < MW; ++i)
#pragma unroll
      for (int j = 0; j < K2; ++j) {
        if (IS_U8) {
          uacc[i][j] = ushort2_t{0, 0};
          uhi[i][j] = ushort2_t{0, 0};
        } else {
          facc[i][j][0] = facc[i][j][1] = 0.0f;
        }
      }
    auto fold = [&]() {
      if (IS_U8) {
#pragma unroll
        for (int i = 0; i < MW; ++i)
#pragma unroll
          for (int j = 0; j < K2; ++j) {
            uhi[i][j] += uacc[i][j] >> (ushort)8;
            uacc[i][j] &= (ushort)0xFF;
          }
      }
    };
    // 1.0 from an opaque scalar move: fma(fpext(h), one, acc) then selects
    // v_fma_mix_f32 instead of being folded into a convert plus an add
    uint32_t one_bits;
    asm("s_mov_b32 %0, 0x3f800000" : "=s"(one_bits));
    const float one = __builtin_bit_cast(float, one_bits);

    Rel rel, rel_next;
    const uint32_t nblocks = (nchans + cbr - 1u) / cbr;
    const int32_t *rt = reltab + ((uint64_t)dt * nblocks * 4u + wave) * Rel::WORDS;
    prefetch(0);
    stage(0, lds);
    if (cbr < nchans) prefetch(cbr);
    rel.load(rt, lane);
    wait_vmem();
    __syncthreads();
    build(0, lds);
    __syncthreads();
    uint32_t k = 0, since_fold = 0;
    for (uint32_t cb = 0; cb < nchans; cb += cbr, ++k) {
      const uint32_t *cur = lds + (k & 1u) * bufw + lane;
      const bool more = cb + cbr < nchans;
      if (more) {
        stage(cb + cbr, lds + ((k + 1u) & 1u) * bufw);
        if (cb + 2u * cbr < nchans) prefetch(cb + 2u * cbr);
        rel_next.load(rt + (uint64_t)(k + 1u) * 4u * Rel::WORDS, lane);
      }
      const uint32_t nc = min(cbr, nchans - cb);
      if (IS_U8) {
        if (since_fold + nc > 256u) {  // 255 + 256 * 255 = 65535 still fits in 16 bits
          fold();
          since_fold = 0;
        }
        since_fold += nc;
      }
      auto add_word = [&](int i, int j, uint32_t word) {
        if (IS_U8) {
          uacc[i][j] += __builtin_bit_cast(ushort2_t, word);
        } else {
          const half2_t h = __builtin_bit_cast(half2_t, word);
          facc[i][j][0] = __builtin_fmaf((float)h.x, one, facc[i][j][0]);
          facc[i][j][1] = __builtin_fmaf((float)h.y, one, facc[i][j][1]);
        }
      };
      if constexpr (PAIRS) {
        // rows r, r+1 of the block are channels 2k, 2k+1 (blocks start at
        // even channels); the pair sum rounds once to FP16, then to FP32.
        // An odd last channel pairs with the zero row build() leaves after
        // it: h + 0 = h exactly, and the accumulators, which start at +0,
        // are never -0, so adding +0 for -0 changes no result.
        auto add_pair = [&](int i, int j, uint32_t a, uint32_t b2) {
          const half2_t s = __builtin_bit_cast(half2_t, a) + __builtin_bit_cast(half2_t, b2);
          add_word(i, j, __builtin_bit_cast(uint32_t, s));
        };
#pragma unroll
        for (int r = 0; r < CB; r += 2) {
          if ((uint32_t)r < nc) {
            if constexpr (BURST > 0) {
#pragma unroll
              for (int i0 = 0; i0 < MW; i0 += BURST) {
                uint32_t w0[BURST][K2], w1[BURST][K2];
#pragma unroll
                for (int g = 0; g < BURST; ++g) {
                  const uint32_t *p0 = at_bytes(cur, rel.get(r, i0 + g));
                  const uint32_t *p1 = at_bytes(cur, rel.get(r + 1, i0 + g));
#pragma unroll
                  for (int j = 0; j < K2; ++j) {
                    w0[g][j] = p0[64 * j];
                    w1[g][j] = p1[64 * j];
                  }
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int g = 0; g < BURST; ++g)
#pragma unroll
                  for (int j = 0; j < K2; ++j) add_pair(i0 + g, j, w0[g][j], w1[g][j]);
              }
            } else {
#pragma unroll
              for (int i = 0; i < MW; ++i) {
                const uint32_t *p0 = at_bytes(cur, rel.get(r, i));
                const uint32_t *p1 = at_bytes(cur, rel.get(r + 1, i));
#pragma unroll
                for (int j = 0; j < K2; ++j) add_pair(i, j, p0[64 * j], p1[64 * j]);
              }
            }
          }
        }
      } else {
#pragma unroll
        for (int r = 0; r < CB; ++r) {
          if ((uint32_t)r < nc) {
            if constexpr (BURST > 0) {
#pragma unroll
              for (int i0 = 0; i0 < MW; i0 += BURST) {
                uint32_t w[BURST][K2];
#pragma unroll
                for (int g = 0; g < BURST; ++g) {
                  const uint32_t *p = at_bytes(cur, rel.get(r, i0 + g));
#pragma unroll
                  for (int j = 0; j < K2; ++j) w[g][j] = p[64 * j];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int g = 0; g < BURST; ++g)
#pragma unroll
                  for (int j = 0; j < K2; ++j) add_word(i0 + g, j, w[g][j]);
              }
            } else {
#pragma unroll
              for (int i = 0; i < MW; ++i) {
                const uint32_t *p = at_bytes(cur, rel.get(r, i));
#pragma unroll
                for (int j = 0; j < K2; ++j) add_word(i, j, p[64 * j]);
              }
            }
          }
        }
      }
      wait_vmem();
      __syncthreads();
      if (more) {
        build(cb + cbr, lds + ((k + 1u) & 1u) * bufw);
        __syncthreads();
        rel = rel_next;
      }
    }

    const double base = (double)nchans * -4.0;
#pragma unroll
    for (int i = 0; i < MW; ++i) {
      const uint32_t d = dw + (uint32_t)i;
      if (d < ndms) {
        float *o = out + (uint64_t)d * nsamp;
#pragma unroll
        for (int j = 0; j < K2; ++j) {
          const uint32_t t = t0 + 2u * lane + 128u * j;
          float v0, v1;
          if (IS_U8) {
            const uint32_t s0 = 256u * (uint32_t)uhi[i][j].x + (uint32_t)uacc[i][j].x;
            const uint32_t s1 = 256u * (uint32_t)uhi[i][j].y + (uint32_t)uacc[i][j].y;
            v0 = (float)((double)s0 * (8.0 / 255.0) + base);
            v1 = (float)((double)s1 * (8.0 / 255.0) + base);
          } else {
            v0 = facc[i][j][0];
            v1 = facc[i][j][1];
          }
          if (t < nsamp) o[t] = v0;
          if (t + 1u < nsamp) o[t + 1] = v1;
        }
      }
    }
  }
};

template <int MW, int K2, int CB, int BURST = 0>
using F16Tile = PackedTile<MDSM_F16, MW, K2, CB, BURST>;
template <int MW, int K2, int CB, int BURST = 0>
using U8Tile = PackedTile<MDSM_U8, MW, K2, CB, BURST>;
// The F16_PAIRS tile of an F16 tile shape; grouped reads take half as many
// trials, since each reads two channels.
template <typename F16T>
struct PairsOf;
template <int MW, int K2, int CB, int BURST>
struct PairsOf<PackedTile<MDSM_F16, MW, K2, CB, BURST>> {
  using type = PackedTile<MDSM_F16_PAIRS, MW, K2, CB, BURST / 2>;
};
template <int NW>
struct PairsOf<WindowTile<MDSM_F16, NW>> {
  using type = PackedTile<MDSM_F16_PAIRS, 12, 4, 4>;
};

// ================================================ pair-sum rows (F16, U8)
// F16_PAIRS and U8 tiles that add each channel pair once per distinct delay
// difference instead of once per trial.  For channels c0 = 2k, c1 = 2k+1
// and trial d, the pair sum x0[t + D0(d)] + x1[t + D1(d)] (F16_PAIRS: one
// FP16 rounding; U8: exact in 16 bits) depends on d only through D0(d) and
// delta(d) = D1(d) - D0(d), and inside one DM tile delta takes a few
// consecutive values dmin .. dmin+n-1.  After a channel block is staged (one
// raw window per channel), the build pass adds the pair's windows once per
// value into sum rows S_j[s] = x0[s] + x1[s + dmin + j] (a P and a Q copy,
// as in the F16 layout), and each trial reads one word of S_{delta(d)-dmin}
// at D0(d): one LDS word per four channel adds, then two v_fma_mix_f32
// (F16_PAIRS) or one v_pk_add_u16 (U8), where the packed layouts above read
// two words per trial.  The sums are the same operations on the same
// operands, so the results are identical to those layouts'.  A shape takes
// a survey when n <= NS and delta >= 0 for every DM tile and pair
// (pairsum_accepts); the packed shapes take every survey.
//
// LDS: the raw windows of the block's cbr channels (wp words each, one
// buffer: the build has consumed them before the next block is staged),
// then NS sum rows of 2 wp words (P, Q) per pair.  The trial loop reads only
// the sum rows, so the next block's windows can arrive while it runs.
// Table: the trial offsets (one per pair and trial, relative to the sum
// rows), then per (DM tile, block, pair) the words {dmin, n}.
template <int MODE, int MW, int K2, int CBP, int NS, int BURST = 0>
struct PairSumTile {
  static constexpr int TT = 128 * K2;
  static constexpr int TD = 4 * MW;
  static constexpr int CB = 2 * CBP;
  static constexpr bool PAIRS = true;
  static constexpr bool IS_U8 = MODE == MDSM_U8;
  static constexpr int NSUM = NS;
  // window origins on even samples (F16: one dword = 2 samples) or on
  // multiples of 4 (U8: one dword = 4 samples)
  static constexpr uint32_t ORIGIN = IS_U8 ? 4u : 2u;
  static constexpr int PACK = 1;
  using T = std::conditional_t<IS_U8, uint8_t, __half>;
  using Rel = RelOffsets<MW, CBP, PACK>;
  static_assert(MODE == MDSM_F16_PAIRS || MODE == MDSM_U8, "pair sums of F16 or U8 rows");
  static_assert(NS >= 1 && NS <= 4, "sum rows per pair (shifts up to 4 samples)");
  static_assert(CBP == 1 || CBP == 2 || CBP == 4, "waves per pair in the build: 4 / CBP");
  static bool fits(uint32_t) { return true; }
  // rw: words of one copy (window of TT + spread samples from an even origin)
  static uint32_t row_words(uint32_t spread) { return PackedGeom<MW, K2, CB>::copy_words(spread); }
  // raw window dwords per channel: F16 one copy; U8 the bytes of 2 rw + 8
  // samples, padded to 64
  static __host__ __device__ uint32_t raw_words(uint32_t rw) {
    return IS_U8 ? ((rw / 2u + 2u + 63u) & ~63u) : rw;
  }
  // per staged channel: its raw window and half of its pair's sum rows
  static uint32_t lds_words_per_row(uint32_t rw) { return raw_words(rw) + (uint32_t)NS * rw; }

  // U8: the n sum rows of one pair, exact u16 pairs: row j is P_j[k] =
  // (x0[2k] + x1[2k + SH], x0[2k + 1] + x1[2k + 1 + SH]) with SH = j + F,
  // F = dmin & 3, samples counted from the 4-aligned origins of the two raw
  // windows (bytes widened by v_perm_b32, added by v_pk_add_u16; sums <=
  // 510), and its Q copy.  Lane l builds words k0 + 4 l .. + 3 of every
  // `step` from 3 dwords of R0 and 4 of R1 (reads end at most 2 dwords past
  // word wp / 2 of a row, inside the row's padding).
  template <int F>
  __device__ __forceinline__ static void build_pair_u8(const uint32_t *R0, const uint32_t *R1,
                                                       uint32_t *S, uint32_t wp, uint32_t n,
                                                       bool solo, uint32_t k0, uint32_t step) {
    for (uint32_t k = k0; k < wp; k += step) {
      const uint2 a01 = *reinterpret_cast<const uint2 *>(R0 + k / 2u);
      const uint32_t a2 = R0[k / 2u + 2u];
      // x0 samples 2i, 2i + 1 as a u16 pair, i = 0..4
      const uint32_t av[5] = {__builtin_amdgcn_perm(0u, a01.x, 0x0C010C00u),
                              __builtin_amdgcn_perm(0u, a01.x, 0x0C030C02u),
                              __builtin_amdgcn_perm(0u, a01.y, 0x0C010C00u),
                              __builtin_amdgcn_perm(0u, a01.y, 0x0C030C02u),
                              __builtin_amdgcn_perm(0u, a2, 0x0C010C00u)};
      uint32_t z[4] = {0u, 0u, 0u, 0u};
      if (!solo) {
        const uint2 z01 = *reinterpret_cast<const uint2 *>(R1 + k / 2u);
        const uint2 z23 = *reinterpret_cast<const uint2 *>(R1 + k / 2u + 2u);
        z[0] = z01.x, z[1] = z01.y, z[2] = z23.x, z[3] = z23.y;
      }
#pragma unroll
      for (int j = 0; j < NS; ++j) {
        if ((uint32_t)j >= n) break;
        const int sh = j + F;
        uint32_t sv[5];
#pragma unroll
        for (int i = 0; i < 5; ++i) {
          // x1 bytes b = 2i + sh and b + 1: dword b / 4 (and the next one
          // when b % 4 == 3), selected into the low bytes of the two halves
          const int bb = 2 * i + sh, w = bb >> 2, o = bb & 3;
          const uint32_t lo = z[w], hi = o == 3 ? z[w + 1] : z[w];
          const uint32_t bv = __builtin_amdgcn_perm(hi, lo, 0x0C000C00u | (uint32_t)o | ((uint32_t)(o + 1) << 16));
          const ushort2_t sum = __builtin_bit_cast(ushort2_t, av[i]) + __builtin_bit_cast(ushort2_t, bv);
          sv[i] = __builtin_bit_cast(uint32_t, sum);
        }
        uint32_t *P = S + (uint32_t)j * 2u * wp;
        *reinterpret_cast<uint4 *>(P + k) = make_uint4(sv[0], sv[1], sv[2], sv[3]);
        *reinterpret_cast<uint4 *>(P + wp + k) = make_uint4(
            __builtin_amdgcn_alignbit(sv[1], sv[0], 16), __builtin_amdgcn_alignbit(sv[2], sv[1], 16),
            __builtin_amdgcn_alignbit(sv[3], sv[2], 16), __builtin_amdgcn_alignbit(sv[4], sv[3], 16));
      }
    }
  }

  // F16: the n sum rows of one pair over part of the window: row j is
  // P_j[k] = fl16(R0[k] + R1 shifted by SH = j + F samples) (two halves per
  // word, one v_pk_add_f16) and its Q copy, F = dmin & 1.  Lane l builds
  // words k0 + 4 l .. + 3 of every `step`; R0 and R1 are read once for all
  // rows.  R0 reads run one word past the row and R1 reads up to four (into
  // the next staged row or the sum rows, inside the allocation); those words
  // only reach P and Q words that no trial reads.
  template <int F>
  __device__ __forceinline__ static void build_pair(const uint32_t *R0, const uint32_t *R1, uint32_t *S,
                                                    uint32_t wp, uint32_t n, bool solo, uint32_t k0,
                                                    uint32_t step) {
    for (uint32_t k = k0; k < wp; k += step) {
      const uint4 a = *reinterpret_cast<const uint4 *>(R0 + k);
      const uint32_t av[5] = {a.x, a.y, a.z, a.w, R0[k + 4]};
      uint32_t z[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
      if (!solo) {
        const uint4 z0 = *reinterpret_cast<const uint4 *>(R1 + k);
        const uint4 z1 = *reinterpret_cast<const uint4 *>(R1 + k + 4);
        z[0] = z0.x, z[1] = z0.y, z[2] = z0.z, z[3] = z0.w;
        z[4] = z1.x, z[5] = z1.y, z[6] = z1.z, z[7] = z1.w;
      }
#pragma unroll
      for (int j = 0; j < NS; ++j) {
        if ((uint32_t)j >= n) break;
        const int sh = j + F, m = sh >> 1;
        const bool e = (sh & 1) != 0;
        uint32_t sv[5];
#pragma unroll
        for (int i = 0; i < 5; ++i) {
          const uint32_t b = e ? __builtin_amdgcn_alignbit(z[m + i + 1], z[m + i], 16) : z[m + i];
          const half2_t h = __builtin_bit_cast(half2_t, av[i]) + __builtin_bit_cast(half2_t, b);
          sv[i] = __builtin_bit_cast(uint32_t, h);
        }
        uint32_t *P = S + (uint32_t)j * 2u * wp;
        *reinterpret_cast<uint4 *>(P + k) = make_uint4(sv[0], sv[1], sv[2], sv[3]);
        *reinterpret_cast<uint4 *>(P + wp + k) = make_uint4(
            __builtin_amdgcn_alignbit(sv[1], sv[0], 16), __builtin_amdgcn_alignbit(sv[2], sv[1], 16),
            __builtin_amdgcn_alignbit(sv[3], sv[2], 16), __builtin_amdgcn_alignbit(sv[4], sv[3], 16));
      }
    }
  }

  __device__ __forceinline__ static void run(const T *__restrict__ in, uint64_t ld,
                                             const int32_t *__restrict__ table,
                                             const int32_t *__restrict__ reltab, uint32_t nchans,
                                             uint32_t nsamp, uint32_t ndms, uint32_t wp,
                                             uint32_t cbr, float *__restrict__ out, uint32_t tt,
                                             uint32_t dt, float *ldsf) {
    uint32_t *lds = reinterpret_cast<uint32_t *>(ldsf);
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u;
    const uint32_t wave = uniform(tid >> 6);
    const uint32_t t0 = tt * TT, d0 = dt * TD;
    const uint32_t dw = d0 + wave * MW;
    const uint64_t ldw = IS_U8 ? ld / 4u : ld / 2u;  // source dwords per row
    const uint32_t *src32 = reinterpret_cast<const uint32_t *>(in);
    const uint32_t rawn = raw_words(wp);
    uint32_t *raw = lds;                 // cbr windows of rawn dwords
    uint32_t *sums = lds + cbr * rawn;   // (cbr / 2) * NS * 2 wp words
    const uint32_t nblocks = (nchans + cbr - 1u) / cbr;
    const uint32_t n_dtiles = (ndms + TD - 1u) / TD;
    const int32_t *dtab =
        reltab + (uint64_t)n_dtiles * nblocks * 4u * Rel::WORDS + (uint64_t)dt * nblocks * CBP * 2u;
    const uint32_t lane4 = 4u * lane;

    // window starts of the next block to stage, and its pairs' {dmin, n}
    uint32_t g0pre[CB];
    int32_t dminpre[CBP];
    uint32_t npre[CBP];
    auto prefetch = [&](uint32_t cb, uint32_t k) {
#pragma unroll
      for (int p = 0; p < CBP; ++p) {
        const uint32_t c0 = cb + 2u * (uint32_t)p;
        if (2u * (uint32_t)p < cbr && c0 < nchans) {
          const uint32_t g = t0 + (uint32_t)table[(uint64_t)c0 * ndms + d0];
          dminpre[p] = dtab[((uint64_t)k * CBP + p) * 2u];
          npre[p] = (uint32_t)dtab[((uint64_t)k * CBP + p) * 2u + 1u];
          g0pre[2 * p] = g;
          g0pre[2 * p + 1] = (g & ~(ORIGIN - 1u)) + (uint32_t)dminpre[p];
        }
      }
    };
    auto stage = [&](uint32_t cb) {
      const uint32_t nc = min(cbr, nchans - cb);
#pragma unroll
      for (int rr = 0; rr < CB; ++rr) {
        if ((uint32_t)rr >= nc) break;
        const uint32_t r = (uint32_t)rr;
        const uint64_t w0 = IS_U8 ? g0pre[rr] >> 2 : g0pre[rr] >> 1;
        const uint32_t *src = src32 + (uint64_t)(cb + r) * ldw + w0;
        const int32_t ldw32 = (int32_t)ldw;  // rows < 2 GiB
        const int32_t avail = 4 * (ldw32 - min((int32_t)w0, ldw32));
        uint32_t *dst = raw + r * rawn;
        for (uint32_t q = wave; 64u * q < rawn; q += 4u) {
          const int32_t rest = max(avail - 256 * (int32_t)q, 0);
          chunk_to_lds(src + 64u * q, (uint32_t)rest, dst + 64u * q, lane4);
        }
      }
    };
    int32_t dmin[CBP];
    uint32_t nrow[CBP];
    auto take = [&]() {
#pragma unroll
      for (int p = 0; p < CBP; ++p) {
        dmin[p] = dminpre[p];
        nrow[p] = npre[p];
      }
    };
    // pair p is built by waves p W .. p W + W - 1 (W = 4 / CBP), wave p W + h
    // taking the 256-word parts h, h + W, ... of the window; all of a pair's
    // sum rows come from one read of its two windows
    auto build = [&](uint32_t cb) {
      const uint32_t nc = min(cbr, nchans - cb);
      constexpr uint32_t W = 4u / CBP;
      const uint32_t p = wave / W, h = wave % W;
      if (2u * p >= nc) return;
      const bool solo = 2u * p + 1u >= nc;
      const uint32_t *R0 = raw + 2u * p * rawn;
      uint32_t *S = sums + p * (uint32_t)NS * 2u * wp;
      const uint32_t k0 = 256u * h + 4u * lane, step = 256u * W;
      // dmin and nrow of pair p, selected with compile-time indices
      int32_t dm = dmin[0];
      uint32_t nr = nrow[0];
#pragma unroll
      for (int q = 1; q < CBP; ++q)
        if (p == (uint32_t)q) dm = dmin[q], nr = nrow[q];
      if constexpr (IS_U8) {
        switch ((uint32_t)dm & 3u) {
          case 0: build_pair_u8<0>(R0, R0 + rawn, S, wp, nr, solo, k0, step); break;
          case 1: build_pair_u8<1>(R0, R0 + rawn, S, wp, nr, solo, k0, step); break;
          case 2: build_pair_u8<2>(R0, R0 + rawn, S, wp, nr, solo, k0, step); break;
          default: build_pair_u8<3>(R0, R0 + rawn, S, wp, nr, solo, k0, step); break;
        }
      } else {
        if ((uint32_t)dm & 1u) build_pair<1>(R0, R0 + rawn, S, wp, nr, solo, k0, step);
        else build_pair<0>(R0, R0 + rawn, S, wp, nr, solo, k0, step);
      }
    };

    // F16: FP32 accumulators.  U8: u16 pair accumulators with the running
    // sum S = 256 * uhi + uacc held exactly, as in the U8 tile: a fold moves
    // uacc's high bytes into uhi and leaves uacc <= 255, so 256 more channels
    // (128 pair sums <= 510) fit in 16 bits.
    float facc[IS_U8 ? 1 : MW][IS_U8 ? 1 : K2][2];
    ushort2_t uacc[IS_U8 ? MW : 1][IS_U8 ? K2 : 1];
    ushort2_t uhi[IS_U8 ? MW : 1][IS_U8 ? K2 : 1];
#pragma unroll
    for (int i = 0; i < MW; ++i)
#pragma unroll
      for (int j = 0; j < K2; ++j) {
        if constexpr (IS_U8) {
          uacc[i][j] = ushort2_t{0, 0};
          uhi[i][j] = ushort2_t{0, 0};
        } else {
          facc[i][j][0] = facc[i][j][1] = 0.0f;
        }
      }
    // 1.0 from an opaque scalar move: fma(fpext(h), one, acc) then selects
    // v_fma_mix_f32 instead of a convert plus an add
    uint32_t one_bits;
    asm("s_mov_b32 %0, 0x3f800000" : "=s"(one_bits));
    const float one = __builtin_bit_cast(float, one_bits);

    Rel rel, rel_next;
    const int32_t *rt = reltab + ((uint64_t)dt * nblocks * 4u + wave) * Rel::WORDS;
    prefetch(0, 0);
    stage(0);
    take();
    if (cbr < nchans) prefetch(cbr, 1);
    rel.load(rt, lane);
    wait_vmem();
    __syncthreads();
    build(0);
    __syncthreads();
    const uint32_t *cur = sums + lane;
    uint32_t k = 0, since_fold = 0;
    for (uint32_t cb = 0; cb < nchans; cb += cbr, ++k) {
      const bool more = cb + cbr < nchans;
      if (more) {
        stage(cb + cbr);
        take();
        if (cb + 2u * cbr < nchans) prefetch(cb + 2u * cbr, k + 2u);
        rel_next.load(rt + (uint64_t)(k + 1u) * 4u * Rel::WORDS, lane);
      }
      const uint32_t nc = min(cbr, nchans - cb);
      if constexpr (IS_U8) {
        if (since_fold + nc > 256u) {  // 255 + 128 * 510 = 65535 still fits in 16 bits
#pragma unroll
          for (int i = 0; i < MW; ++i)
#pragma unroll
            for (int j = 0; j < K2; ++j) {
              uhi[i][j] += uacc[i][j] >> (ushort)8;
              uacc[i][j] &= (ushort)0xFF;
            }
          since_fold = 0;
        }
        since_fold += nc;
      }
      auto add_word = [&](int i, int j, uint32_t w) {
        if constexpr (IS_U8) {
          uacc[i][j] += __builtin_bit_cast(ushort2_t, w);
        } else {
          const half2_t h = __builtin_bit_cast(half2_t, w);
          facc[i][j][0] = __builtin_fmaf((float)h.x, one, facc[i][j][0]);
          facc[i][j][1] = __builtin_fmaf((float)h.y, one, facc[i][j][1]);
        }
      };
#pragma unroll
      for (int p = 0; p < CBP; ++p) {
        if (2u * (uint32_t)p < nc) {
          if constexpr (BURST > 0) {
            // the reads of BURST trials are issued together ahead of their
            // adds (a scheduling fence keeps them grouped)
#pragma unroll
            for (int i0 = 0; i0 < MW; i0 += BURST) {
              uint32_t w[BURST][K2];
#pragma unroll
              for (int g = 0; g < BURST; ++g) {
                const uint32_t *q = at_bytes(cur, rel.get(p, i0 + g));
#pragma unroll
                for (int j = 0; j < K2; ++j) w[g][j] = q[64 * j];
              }
              __builtin_amdgcn_sched_barrier(0);
#pragma unroll
              for (int g = 0; g < BURST; ++g)
#pragma unroll
                for (int j = 0; j < K2; ++j) add_word(i0 + g, j, w[g][j]);
            }
          } else {
#pragma unroll
            for (int i = 0; i < MW; ++i) {
              const uint32_t *q = at_bytes(cur, rel.get(p, i));
#pragma unroll
              for (int j = 0; j < K2; ++j) add_word(i, j, q[64 * j]);
            }
          }
        }
      }
      wait_vmem();
      __syncthreads();
      if (more) {
        build(cb + cbr);
        __syncthreads();
        rel = rel_next;
      }
    }

    const double base = (double)nchans * -4.0;
#pragma unroll
    for (int i = 0; i < MW; ++i) {
      const uint32_t d = dw + (uint32_t)i;
      if (d < ndms) {
        float *o = out + (uint64_t)d * nsamp;
#pragma unroll
        for (int j = 0; j < K2; ++j) {
          const uint32_t t = t0 + 2u * lane + 128u * j;
          float v0, v1;
          if constexpr (IS_U8) {
            const uint32_t s0 = 256u * (uint32_t)uhi[i][j].x + (uint32_t)uacc[i][j].x;
            const uint32_t s1 = 256u * (uint32_t)uhi[i][j].y + (uint32_t)uacc[i][j].y;
            v0 = (float)((double)s0 * (8.0 / 255.0) + base);
            v1 = (float)((double)s1 * (8.0 / 255.0) + base);
          } else {
            v0 = facc[i][j][0];
            v1 = facc[i][j][1];
          }
          if (t < nsamp) o[t] = v0;
          if (t + 1u < nsamp) o[t + 1] = v1;
        }
      }
    }
  }
};

template <typename T>
struct IsPairSum : std::false_type {};
template <int MODE, int MW, int K2, int CBP, int NS, int BURST>
struct IsPairSum<PairSumTile<MODE, MW, K2, CBP, NS, BURST>> : std::true_type {};

// Register windows over pair-sum rows: the sum rows S_j of each channel pair,
// built in LDS as FP32 (F16_PAIRS: the FP16-rounded pair sums widened, U8: the
// exact sums), are read by WindowCode's adds, so one v_add_f32 adds two
// channels.  Trials of one wave that differ in j or run out of a window read
// another one (1.9 windows and 12 reads per wave and pair at 1024 channels
// and a DM step of 0.2, against one and 7 for single channels).  Results are
// those of the other pair-sum shapes.  1024 channels x 4096 trials x 2^17
// samples: U8 12.1 ms (45.6 T adds/s; 14.9 with shape 20), F16_PAIRS 12.4
// (44.5; 14.1).  With eight waves the twelve barriers per LDS fill are shared
// by half the trials: 33 T.
template <int MODE, int NW>
struct WindowPairTile {
  using W = WindowCode;
  static constexpr bool PAIRS = true;
  static constexpr bool IS_U8 = MODE == MDSM_U8;
  static constexpr int MW = W::MW, K = W::K, WAVES = NW, THREADS = 64 * NW;
  static constexpr int TT = 64 * K, TD = NW * MW, CB = NW == 8 ? 6 : 12, CBP = CB / 2, NSUM = 3;
  using T = std::conditional_t<IS_U8, uint8_t, __half>;
  static constexpr uint32_t PER = 4u / sizeof(T);  // samples per source dword, origin of a window
  // staging: WPR waves share a row of a block, every wave has up to RPW rows;
  // building: 512 threads take a pair (four samples each), every 512 of the
  // workgroup every NG-th pair
  static constexpr uint32_t WPR = NW == 8 ? 4 : 1, RSTEP = NW / WPR, RPW = (CB + RSTEP - 1) / RSTEP;
  static constexpr uint32_t NG = THREADS / 512, PPG = CBP / NG;
  static bool fits(uint32_t) { return true; }
  static uint32_t row_words(uint32_t spread) { return ((uint32_t)TT + spread + 16u + 63u) & ~63u; }
  // raw dwords per channel: the samples of a sum row and 8 more (shifts)
  static __host__ __device__ uint32_t raw_words(uint32_t rw) { return (rw / PER + 4u + 63u) & ~63u; }
  static uint32_t lds_words_per_row(uint32_t rw) { return raw_words(rw) + (uint32_t)NSUM * rw / 2u; }
  static uint64_t table_entries(uint32_t nchans, uint32_t ndms) {
    return (uint64_t)((ndms + TD - 1u) / TD) * NW * ((nchans + 1u) / 2u + 1u);
  }
  // 8 words per entry, then {dmin, n} per DM tile and pair
  static uint64_t table_words(uint32_t nchans, uint32_t ndms) {
    return 8u * table_entries(nchans, ndms) +
           2u * (uint64_t)((ndms + TD - 1u) / TD) * ((nchans + 1u) / 2u);
  }

  __device__ __forceinline__ static void run(const T *__restrict__ in, uint64_t ld,
                                             const int32_t *__restrict__ table,
                                             const int32_t *__restrict__ reltab, uint32_t nchans,
                                             uint32_t nsamp, uint32_t ndms, uint32_t rw,
                                             uint32_t cbr, float *__restrict__ out, uint32_t tt,
                                             uint32_t dt, float *lds) {
    typedef W::u32x8 u32x8;
    typedef W::const_u32x8 const_u32x8;
    typedef __attribute__((address_space(3))) float lds_float;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = uniform(threadIdx.x >> 6);
    const uint32_t t0 = tt * TT, d0 = dt * TD;
    const uint32_t dw = d0 + wave * MW;
    const uint32_t rawn = raw_words(rw);
    const uint32_t npairs = (nchans + 1u) / 2u, n_dtiles = (ndms + TD - 1u) / TD;
    typedef __attribute__((address_space(4))) const int32_t const_i32;  // scalar loads
    const const_i32 *dtab = (const const_i32 *)(uintptr_t)reltab +
                            8u * ((uint64_t)n_dtiles * NW * (npairs + 1u)) + 2u * (uint64_t)dt * npairs;
    const const_i32 *ctable = (const const_i32 *)(uintptr_t)table;
    // LDS: cbr / 2 pairs of NSUM sum rows, then cbr raw windows
    uint32_t *const raw = reinterpret_cast<uint32_t *>(lds) + (cbr / 2u) * (uint32_t)NSUM * rw;
    const uint32_t srow = wave / WPR, part = wave % WPR;
    // window starts of the rows the next stage() takes
    uint32_t gpre[RPW];
    auto prefetch = [&](uint32_t cb) {
#pragma unroll
      for (uint32_t i = 0; i < RPW; ++i) {
        const uint32_t c = min(cb + srow + RSTEP * i, nchans - 1u), c0 = c & ~1u;
        const uint32_t g = t0 + (uint32_t)ctable[(uint64_t)c0 * ndms + d0];
        gpre[i] = (c & 1u) ? (g & ~(PER - 1u)) + (uint32_t)dtab[c0] : g;
      }
    };
    auto stage = [&](uint32_t cb) {
#pragma unroll
      for (uint32_t i = 0; i < RPW; ++i) {
        const uint32_t r = srow + RSTEP * i;
        if (r >= min(cbr, nchans - cb)) break;
        const uint32_t w0 = gpre[i] / PER, ldw = (uint32_t)(ld / PER);  // rows < 2 GiB
        const uint32_t *src = reinterpret_cast<const uint32_t *>(in) + (uint64_t)(cb + r) * ldw + w0;
        const uint32_t avail = 4u * (ldw - min(w0, ldw));  // dwords past the row read as 0
        const uint64_t a = reinterpret_cast<uint64_t>(src);
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            reinterpret_cast<void *>(((uint64_t)uniform((uint32_t)(a >> 32)) << 32) | uniform((uint32_t)a)),
            (short)0, (int)uniform(avail), 0x00020000);
        uint32_t *dst = raw + r * rawn + 64u * part;
        uint32_t vo = 4u * (threadIdx.x & 63u) + 256u * part;
        asm volatile("" : "+v"(vo));
        for (uint32_t q = part; 64u * q < rawn; q += WPR, vo += 256u * WPR, dst += 64u * WPR)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void *)dst, 4, (int)vo, 0, 0, 0);
      }
    };
    // the block's pairs: dmin's part below the window origin's grid, and the
    // number of sum rows (0: no such pair)
    const uint32_t grp = wave / 8u;
    uint32_t frac[PPG], nrow[PPG];
    auto pairs_of = [&](uint32_t cb) {
      const uint32_t np = (min(cbr, nchans - cb) + 1u) / 2u;
#pragma unroll
      for (uint32_t i = 0; i < PPG; ++i) {
        const uint32_t p = grp + NG * i, q = min(cb / 2u + p, npairs - 1u);
        frac[i] = (uint32_t)dtab[2u * q] & (PER - 1u);
        nrow[i] = p < np ? (uint32_t)dtab[2u * q + 1u] : 0u;
      }
    };
    // S_j[n .. n+3] = x0[n ..] + x1[n + SH ..], SH = j + frac; a pair without
    // its second channel adds 0.  The reads of all pairs are issued together.
    // (n0 is opaque, so that no address is kept in registers over the adds)
    auto build = [&](uint32_t cb) {
      const bool odd = cb + cbr >= nchans && (nchans & 1u);  // the block's last pair is one channel
      const uint32_t last = (min(cbr, nchans - cb) - 1u) / 2u;
      uint32_t n0 = 4u * (threadIdx.x & 511u);
      asm volatile("" : "+v"(n0));
      for (uint32_t n = n0; n < rw; n += 2048u) {
        uint32_t x[PPG][2], z[PPG][4];
#pragma unroll
        for (uint32_t i = 0; i < PPG; ++i) {
          const uint32_t *R0 = raw + 2u * min(grp + NG * i, last) * rawn, *R1 = R0 + rawn;
          if constexpr (IS_U8) {
            x[i][0] = R0[n / 4u];
            z[i][0] = R1[n / 4u], z[i][1] = R1[n / 4u + 1u], z[i][2] = R1[n / 4u + 2u];
          } else {
            const uint2 a = *reinterpret_cast<const uint2 *>(R0 + n / 2u);
            const uint2 c = *reinterpret_cast<const uint2 *>(R1 + n / 2u);
            const uint2 e = *reinterpret_cast<const uint2 *>(R1 + n / 2u + 2u);
            x[i][0] = a.x, x[i][1] = a.y;
            z[i][0] = c.x, z[i][1] = c.y, z[i][2] = e.x, z[i][3] = e.y;
          }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t i = 0; i < PPG; ++i) {
          float *S = lds + (grp + NG * i) * NSUM * rw;
          if (odd && grp + NG * i == last) z[i][0] = z[i][1] = z[i][2] = z[i][3] = 0u;
          uint32_t y[3];  // U8: bytes n + frac .., F16: halves n + frac ..
          if constexpr (IS_U8) {
            y[0] = __builtin_amdgcn_alignbyte(z[i][1], z[i][0], frac[i]);
            y[1] = __builtin_amdgcn_alignbyte(z[i][2], z[i][1], frac[i]);
          } else {
            y[0] = __builtin_amdgcn_alignbit(z[i][1], z[i][0], 16u * frac[i]);
            y[1] = __builtin_amdgcn_alignbit(z[i][2], z[i][1], 16u * frac[i]);
            y[2] = __builtin_amdgcn_alignbit(z[i][3], z[i][2], 16u * frac[i]);
          }
#pragma unroll
          for (int j = 0; j < NSUM; ++j) {
            if ((uint32_t)j >= nrow[i]) break;
            float4 v;
            if constexpr (IS_U8) {
              const uint32_t a = x[i][0], c = __builtin_amdgcn_alignbyte(y[1], y[0], (uint32_t)j);
              v = make_float4((float)((a & 0xFFu) + (c & 0xFFu)), (float)(((a >> 8) & 0xFFu) + ((c >> 8) & 0xFFu)),
                              (float)(((a >> 16) & 0xFFu) + ((c >> 16) & 0xFFu)), (float)((a >> 24) + (c >> 24)));
            } else {
              const uint32_t a = j == 1 ? __builtin_amdgcn_alignbit(y[1], y[0], 16) : y[j / 2];
              const uint32_t c = j == 1 ? __builtin_amdgcn_alignbit(y[2], y[1], 16) : y[j / 2 + 1];
              const half2_t s0 = __builtin_bit_cast(half2_t, x[i][0]) + __builtin_bit_cast(half2_t, a);
              const half2_t s1 = __builtin_bit_cast(half2_t, x[i][1]) + __builtin_bit_cast(half2_t, c);
              v = make_float4((float)s0.x, (float)s0.y, (float)s1.x, (float)s1.y);
            }
            *reinterpret_cast<float4 *>(S + j * rw + n) = v;
          }
        }
      }
    };

    float acc[MW][K];
#pragma unroll
    for (int i = 0; i < MW; ++i)
#pragma unroll
      for (int j = 0; j < K; ++j) acc[i][j] = 0.0f;

    const uint32_t cur = (uint32_t)(uintptr_t)(lds_float *)lds + (uint32_t)(4 * K) * lane;
    const const_u32x8 *rt =
        (const const_u32x8 *)(uintptr_t)reltab + ((uint64_t)dt * NW + wave) * (npairs + 1u);
    prefetch(0);
    stage(0);
    pairs_of(0);
    if (cbr < nchans) prefetch(cbr);
    u32x8 o = *rt;
    wait_vmem();
    __syncthreads();
    build(0);
    __syncthreads();
    for (uint32_t cb = 0; cb < nchans; cb += cbr) {
      const bool more = cb + cbr < nchans;
      if (more) {
        stage(cb + cbr);
        pairs_of(cb + cbr);
        if (cb + 2u * cbr < nchans) prefetch(cb + 2u * cbr);
      }
      const uint32_t np = (min(cbr, nchans - cb) + 1u) / 2u;
      for (uint32_t p = 0; p < np; ++p) {
        ++rt;
        o = W::add_channel(acc, cur, o, rt);
      }
      wait_vmem();
      __syncthreads();
      if (more) build(cb + cbr);
      __syncthreads();
    }
    W::store<IS_U8>(acc, lds, wave, lane, out, nsamp, ndms, dw, t0, nchans);
  }
};

template <typename T>
struct IsWindowPair : std::false_type {};
template <int MODE, int NW>
struct IsWindowPair<WindowPairTile<MODE, NW>> : std::true_type {};
template <int MODE, int NW>
struct IsWindow<WindowPairTile<MODE, NW>> : std::true_type {};

// Table of a window pair-sum tile (layout at table_words): entry ((dt * WAVES +
// wave) * (npairs + 1) + p), and {dmin, n} of pair p in DM tile dt.  A pair
// without its second channel sums with zero: dmin 0, n 1.
template <typename Tile>
__global__ __launch_bounds__(256) void window_pair_table_kernel(const int32_t *__restrict__ table,
                                                                uint32_t nchans, uint32_t ndms,
                                                                uint32_t rw, uint32_t cbr,
                                                                uint64_t entries,
                                                                int32_t *__restrict__ reltab) {
  const uint64_t e = (uint64_t)blockIdx.x * 256u + threadIdx.x;
  if (e >= entries) return;
  const uint32_t npairs = (nchans + 1u) / 2u;
  const uint32_t p = min((uint32_t)(e % (npairs + 1u)), npairs - 1u);
  const uint64_t g = e / (npairs + 1u);
  const uint32_t wave = (uint32_t)(g % Tile::WAVES), dt = (uint32_t)(g / Tile::WAVES);
  const uint32_t d0 = dt * Tile::TD, dl = min(d0 + (uint32_t)Tile::TD, ndms) - 1u;
  const uint32_t c0 = 2u * p;
  const bool solo = c0 + 1u >= nchans;
  const int32_t *r0 = table + (uint64_t)c0 * ndms, *r1 = solo ? r0 : r0 + ndms;
  int32_t dmin = r1[d0] - r0[d0], dmax = dmin;
  for (uint32_t d = d0 + 1u; d <= dl; ++d) {
    const int32_t v = r1[d] - r0[d];
    dmin = min(dmin, v);
    dmax = max(dmax, v);
  }
  const uint32_t base = (uint32_t)r0[d0], skew = base & (Tile::PER - 1u);
  uint32_t o[WindowCode::MW], w[2 * WindowCode::MW];
  for (uint32_t i = 0; i < (uint32_t)WindowCode::MW; ++i) {
    const uint32_t d = min(d0 + wave * WindowCode::MW + i, ndms - 1u);
    const uint32_t j = min((uint32_t)(r1[d] - r0[d] - dmin), (uint32_t)Tile::NSUM - 1u);
    o[i] = 4u * ((p % (cbr / 2u) * Tile::NSUM + j) * rw + skew + ((uint32_t)r0[d] - base));
  }
  WindowCode::entry(o, w);
  for (int i = 0; i < 2 * WindowCode::MW; ++i) reltab[e * 8u + i] = (int32_t)w[i];
  if (wave == 0) {
    int32_t *t = reltab + entries * 8u + 2u * ((uint64_t)dt * npairs + p);
    t[0] = dmin;
    t[1] = dmax - dmin + 1;
  }
}

// Trial offsets and {dmin, n} of a pair-sum tile (layout above): entry e <
// nrel is ((dt * nblocks + k) * 4 + w) * WORDS + idx with (p, i) =
// divmod(idx, MW); the byte offset of trial dw + i of pair p inside the sum
// rows, from q0 = D0(d) - D0(d0) + (D0(d0) & 1) (sample position from the
// even window origin) and j = delta(d) - dmin: word ((p NS + j) 2 + (q0 & 1))
// wp + q0 / 2.  Entries past nrel hold {dmin, n} per (dt, k, p).  A pair
// without its second channel (odd nchans) sums with zero: dmin 0, n 1.
template <typename Tile>
__global__ __launch_bounds__(256) void pairsum_offset_kernel(const int32_t *__restrict__ table,
                                                             uint32_t nchans, uint32_t ndms,
                                                             uint32_t wp, uint32_t cbr,
                                                             uint32_t nblocks, uint64_t nrel,
                                                             uint64_t total,
                                                             int32_t *__restrict__ reltab) {
  using Rel = typename Tile::Rel;
  constexpr uint32_t MW = Tile::TD / 4, CBP = Tile::CB / 2, NS = Tile::NSUM;
  const uint64_t e = (uint64_t)blockIdx.x * 256u + threadIdx.x;
  if (e >= total) return;
  uint32_t k, dt, p, i = 0, w = 0, field = 0;
  const bool is_rel = e < nrel;
  if (is_rel) {
    const uint32_t idx = (uint32_t)(e % Rel::WORDS);
    const uint64_t g = e / Rel::WORDS;
    w = (uint32_t)(g & 3u);
    const uint64_t blk = g >> 2;
    k = (uint32_t)(blk % nblocks);
    dt = (uint32_t)(blk / nblocks);
    p = min(idx / MW, CBP - 1u);  // padding words repeat the last pair
    i = idx % MW;
  } else {
    const uint64_t q = e - nrel;
    field = (uint32_t)(q & 1u);
    const uint64_t pq = q >> 1;
    p = (uint32_t)(pq % CBP);
    const uint64_t blk = pq / CBP;
    k = (uint32_t)(blk % nblocks);
    dt = (uint32_t)(blk / nblocks);
  }
  const uint32_t d0 = dt * Tile::TD, dl = min(d0 + (uint32_t)Tile::TD, ndms) - 1u;
  const uint32_t c0 = min(k * cbr + 2u * p, nchans - 1u);
  const bool solo = c0 + 1u >= nchans;
  const int32_t *r0 = table + (uint64_t)c0 * ndms;
  const int32_t *r1 = table + (uint64_t)(solo ? c0 : c0 + 1u) * ndms;
  int32_t dmin = 0, dmax = 0;
  if (!solo) {
    dmin = dmax = r1[d0] - r0[d0];
    for (uint32_t d = d0 + 1u; d <= dl; ++d) {
      const int32_t v = r1[d] - r0[d];
      dmin = min(dmin, v);
      dmax = max(dmax, v);
    }
  }
  if (!is_rel) {
    reltab[e] = field ? dmax - dmin + 1 : dmin;
    return;
  }
  const uint32_t d = min(d0 + w * MW + i, ndms - 1u);
  const int32_t base = r0[d0];
  const uint32_t q0 = (uint32_t)(r0[d] - base) + ((uint32_t)base & (Tile::ORIGIN - 1u));
  const uint32_t j = solo ? 0u : (uint32_t)(r1[d] - r0[d] - dmin);
  const uint32_t word = ((p * NS + min(j, NS - 1u)) * 2u + (q0 & 1u)) * wp + (q0 >> 1);
  reltab[e] = (int32_t)(4u * word);
}

// XCD-aware workgroup order for the single-beam launch: off unless
// MDSM_XCD_REMAP=1 (measured at 1024 channels x 4096 trials x 2^20 samples it
// was level for FP32 and 2-6% slower for FP16/U8 than the plain order)
bool xcd_remap_enabled() {
  static const bool on = [] {
    const char *e = getenv("MDSM_XCD_REMAP");
    return e && e[0] == '1';
  }();
  return on;
}

// Waves per SIMD the persistent kernel is compiled for: its item loop costs
// a few VGPRs over the flat kernel, which drops the 12 x 4 and 10 x 4
// pair-sum tiles from 4 to 3 waves (above 128 VGPRs).  Held at 4 they spill
// a few dwords and still run faster (32-beam batch, persistent launch: FP16
// pair sums 1160 against 1240-1266 ms, U8 1076 against 1270-1285 ms); for
// the 8 x 4 FP16 tile the same hold (6 waves) was slower (1795 against
// 1705-1725 ms), so the other tiles are left to the compiler.
template <typename Tile>
struct PersistWaves {
  static constexpr int value = 1;
};
// Every launch shape of the register-window tiles: their fixed window
// registers end at v127, which leaves 4 waves per SIMD if nothing is placed
// above them.
template <typename Tile>
struct FlatWaves {
  static constexpr int value = 1;
};
template <int MODE, int NW>
struct FlatWaves<WindowTile<MODE, NW>> {
  static constexpr int value = 4;
};
template <int MODE, int NW>
struct PersistWaves<WindowTile<MODE, NW>> {
  static constexpr int value = 4;
};
template <int MODE, int NW>
struct FlatWaves<WindowPairTile<MODE, NW>> {
  static constexpr int value = 4;
};
template <int MODE, int NW>
struct PersistWaves<WindowPairTile<MODE, NW>> {
  static constexpr int value = 4;
};
template <int MODE, int MW, int K2, int CBP, int NS, int BURST>
struct PersistWaves<PairSumTile<MODE, MW, K2, CBP, NS, BURST>> {
  static constexpr int value = 4;
};

// ================================================================= kernels
template <typename Tile>
__global__ __launch_bounds__(tile_threads<Tile>()) __attribute__((amdgpu_waves_per_eu(FlatWaves<Tile>::value)))
void dedisp_kernel(const typename Tile::T *__restrict__ in,
                                                     uint64_t ld,
                                                     const int32_t *__restrict__ table,
                                                     const int32_t *__restrict__ reltab,
                                                     uint32_t nchans, uint32_t nsamp,
                                                     uint32_t ndms, uint32_t rw, uint32_t cbr,
                                                     uint32_t n_dtiles, uint32_t n_ttiles,
                                                     uint32_t xcd_remap, float *__restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  // DM tiles vary fastest: the workgroups resident at one time then share a
  // narrow time range of the input.  Workgroup IDs are dealt round-robin over
  // the 8 XCDs, each with its own L2; with xcd_remap, XCD x takes the time
  // tiles tt = x (mod 8), so all DM tiles re-reading one time window run
  // behind one L2 (grid: 8 * ceil(n_ttiles / 8) * n_dtiles).
  const uint32_t b = blockIdx.x;
  uint32_t tt, dt;
  if (xcd_remap) {
    const uint32_t x = b & 7u, k = b >> 3;
    tt = ((k / n_dtiles) << 3) + x;
    dt = k % n_dtiles;
    if (tt >= n_ttiles) return;  // whole workgroup, before any barrier
  } else {
    tt = b / n_dtiles;
    dt = b % n_dtiles;
  }
  Tile::run(in, ld, table, reltab, nchans, nsamp, ndms, rw, cbr, out, tt, dt, lds);
}

// Trial-offset table of one tile shape: entry ((dt * nblocks + k) * 4 + w)
// * WORDS + 16 n + l holds the byte offset of (r, i) = divmod(16 n + l, MW)
// for channel block k (cbr channels) and wave w of DM tile dt.
template <typename Tile>
__global__ __launch_bounds__(256) void trial_offset_kernel(const int32_t *__restrict__ table,
                                                           uint32_t nchans, uint32_t ndms,
                                                           uint32_t rw, uint32_t cbr,
                                                           uint32_t nblocks, uint64_t total,
                                                           int32_t *__restrict__ reltab) {
  using Rel = typename Tile::Rel;
  constexpr uint32_t MW = Tile::TD / 4;
  const uint64_t e = (uint64_t)blockIdx.x * 256u + threadIdx.x;
  if (e >= total) return;
  const uint32_t idx = (uint32_t)(e % Rel::WORDS);
  const uint64_t g = e / Rel::WORDS;  // (dt * nblocks + k) * 4 + w
  const uint32_t w = (uint32_t)(g & 3u);
  const uint64_t blk = g >> 2;
  const uint32_t k = (uint32_t)(blk % nblocks), dt = (uint32_t)(blk / nblocks);
  const uint32_t d0 = dt * Tile::TD;
  reltab[e] = rel_entry<MW, Tile::PACK>(table, ndms, nchans, k * cbr, d0, d0 + w * MW, idx, rw);
}

// Multi-beam item numbering (both launch shapes): a beam's items are
// XCD-major, 8 A * ceil(n_ttiles / (8 A)) * n_dtiles of them starting at a
// multiple of 8, A = tgroup; item g belongs to XCD g % 8, and with slot s =
// (g + rot) % 8, k = (g - begin) / 8, j = k / (A n_dtiles), r = k % (A
// n_dtiles) it is DM tile r / A of time tile 8 A j + A s + r % A: each XCD takes groups of A
// adjacent time tiles and runs a DM tile for all A of them back to back, so
// their shifted windows overlap in its L2 (A = 1: time tile 8 j + s, DM
// tile r).  Padding items with a time tile past the beam's end do nothing.
struct BeamItem {
  const BeamDesc *bd;
  uint32_t tt, dt;
  bool valid;
};

__device__ __forceinline__ BeamItem decode_item(const BeamDesc *__restrict__ beams, uint32_t nbeams,
                                                uint32_t g) {
  uint32_t lo = 0, hi = nbeams - 1u;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1u) >> 1;
    if (beams[mid].item_begin <= g) lo = mid;
    else hi = mid - 1u;
  }
  const BeamDesc *bd = beams + lo;
  const uint32_t local = g - bd->item_begin;
  const uint32_t k = local >> 3, A = bd->tgroup;
  const uint32_t per = A * bd->n_dtiles;
  const uint32_t j = k / per, r = k - j * per;
  BeamItem it;
  it.bd = bd;
  it.dt = r / A;
  it.tt = 8u * A * j + A * ((local + bd->rot) & 7u) + (r - it.dt * A);
  it.valid = it.tt < bd->n_ttiles;
  return it;
}

// (The dynamic LDS array is declared 16-byte aligned: it follows any static
// LDS of the kernel, and the packed tiles access it with 8-byte operations.)
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
  return ((uint64_t)uniform((uint32_t)(v >> 32)) << 32) | (uint64_t)uniform((uint32_t)v);
}

// Every tile parameter goes through readfirstlane: inside the persistent
// kernel's item loop the compiler cannot prove the descriptor fields
// wave-uniform and would otherwise keep the per-block address arithmetic in
// VALU registers.
template <typename Tile>
__device__ __forceinline__ void run_item(const BeamDesc *__restrict__ beams, const BeamItem &it,
                                         uint32_t cbr, float *lds) {
  const BeamDesc &bd = *it.bd;
  char *base = reinterpret_cast<char *>(const_cast<BeamDesc *>(beams));
  Tile::run(reinterpret_cast<const typename Tile::T *>(base + (int64_t)uniform64((uint64_t)bd.in_off)),
            uniform64(bd.ld), reinterpret_cast<const int32_t *>(base + (int64_t)uniform64((uint64_t)bd.table_off)),
            reinterpret_cast<const int32_t *>(base + (int64_t)uniform64((uint64_t)bd.rel_off)),
            uniform(bd.nchans), uniform(bd.nsamp), uniform(bd.ndms), uniform(bd.row_words), cbr,
            reinterpret_cast<float *>(base + (int64_t)uniform64((uint64_t)bd.out_off)), uniform(it.tt),
            uniform(it.dt), lds);
}

// Persistent multi-beam kernel: resident workgroups pull items from eight
// queues, one per XCD slot (workgroup b drains queue b % 8, the XCD the
// dispatcher puts it on), until the queue passes total_items; every wave
// of every workgroup reaches the exit.  Beams are ordered by the host,
// largest first.
template <typename Tile>
__global__ __launch_bounds__(tile_threads<Tile>()) __attribute__((amdgpu_waves_per_eu(PersistWaves<Tile>::value)))
void batch_kernel(const BeamDesc *__restrict__ beams,
                                                    uint32_t nbeams, uint32_t total_items,
                                                    uint32_t cbr, uint32_t *__restrict__ counter) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  // the item goes through the tile's first word: a tile may take all of a
  // CU's LDS, and any word beside it would make that launch fail
  uint32_t *const item_s = reinterpret_cast<uint32_t *>(lds);
  const uint32_t slot = blockIdx.x & 7u;
  while (true) {
    if (threadIdx.x == 0) *item_s = atomicAdd(counter + slot, 1u) * 8u + slot;
    __syncthreads();
    // wave-uniform: the descriptor lookup and every tile parameter stay scalar
    const uint32_t item = uniform(*item_s);
    __syncthreads();
    if (item >= total_items) break;
    const BeamItem it = decode_item(beams, nbeams, item);
    if (it.valid) run_item<Tile>(beams, it, cbr, lds);
    __syncthreads();
  }
}

// Flat multi-beam kernel: one workgroup per item (workgroup ID = item, so
// the dispatcher's round-robin puts item g on XCD g % 8).
template <typename Tile>
__global__ __launch_bounds__(tile_threads<Tile>()) __attribute__((amdgpu_waves_per_eu(FlatWaves<Tile>::value)))
void batch_flat_kernel(const BeamDesc *__restrict__ beams,
                                                         uint32_t nbeams, uint32_t cbr) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const BeamItem it = decode_item(beams, nbeams, blockIdx.x);
  if (!it.valid) return;  // whole workgroup, before any barrier
  run_item<Tile>(beams, it, cbr, lds);
}

// ------------------------------------------------------------ direct kernel
// Few outputs (launch_dedisperse's shape 0): tiles would leave most of the
// chip idle while each of them walks all channels behind barriers.  A wave
// takes 256 samples of one trial, four consecutive ones per lane, straight
// from the rows: 16 channels' loads in flight (one access per lane and
// channel, at any alignment), summed in channel order.  The four waves of a
// workgroup take four consecutive trials, whose rows overlap in L1.  The table
// is the delay table transposed, [trial][channel], 16 channels per scalar
// load.  Lanes past the row's last whole group repeat that group (they store
// the same values again).
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
typedef _Float16 half4u __attribute__((ext_vector_type(4), aligned(2)));
struct __attribute__((packed)) byte4u {
  uint32_t v;
};

template <int MODE>
__global__ __launch_bounds__(256) void dedisp_direct_kernel(const void *__restrict__ in, uint64_t ld,
                                                            const int32_t *__restrict__ dtab,
                                                            uint32_t nchans, uint32_t cpad, uint32_t nsamp,
                                                            uint32_t ndms, float *__restrict__ out) {
  typedef int32_t i32x16 __attribute__((ext_vector_type(16)));
  typedef __attribute__((address_space(4))) const i32x16 const_i32x16;
  const uint32_t lane = threadIdx.x & 63u;
  // An eighth (give or take one) of the time blocks to each XCD (workgroup IDs
  // are dealt round-robin), which runs through all their trials one after the
  // other, so that their rows stay in its L2; of the pairs (time block, four
  // trials) in that order where an XCD's blocks are more than it can hold at a
  // time (256 workgroups), so that few time blocks of many trials leave no XCD
  // idle (15 trials x 5 blocks split: 78 us instead of 57; 8000 x 1 not split: 2.2
  // ms instead of 0.3).
  const uint32_t ndg = (ndms + 3u) / 4u, ntb = (nsamp + 255u) / 256u, x = blockIdx.x & 7u;
  const uint32_t unit = (ntb + 7u) / 8u * ndg <= 256u ? ndg : 1u, units = unit > 1u ? ntb : ntb * ndg;
  const uint32_t first = (units / 8u * x + units % 8u * x / 8u) * unit;
  const uint32_t past = (units / 8u * (x + 1u) + units % 8u * (x + 1u) / 8u) * unit;
  const uint32_t item = first + (blockIdx.x >> 3);
  if (item >= past) return;
  const uint32_t tb = item / ndg;
  const uint32_t d = uniform((item - tb * ndg) * 4u + (threadIdx.x >> 6));
  if (d >= ndms) return;
  const uint32_t t = min((tb * 64u + lane) * 4u, nsamp - 4u);
  constexpr uint32_t SZ = MODE == MDSM_F32 ? 4u : (MODE == MDSM_U8 ? 1u : 2u);
  const const_i32x16 *tab = (const const_i32x16 *)(uintptr_t)(dtab + (uint64_t)d * cpad);
  const char *row = reinterpret_cast<const char *>(in);  // of the channel
  const uint64_t step = ld * SZ;
  const uint32_t off = t * SZ;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  uint32_t sum[4] = {0u, 0u, 0u, 0u};
  auto run16 = [&](uint32_t n, i32x16 o) {
    float4u f[16];
    half4u h[16];
    uint32_t u[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      // (channels past the last one repeat it and are not added)
      const char *q = row + (uint64_t)(uint32_t)o[c] * SZ + off;
      if constexpr (MODE == MDSM_F32) f[c] = *reinterpret_cast<const float4u *>(q);
      else if constexpr (MODE == MDSM_U8) u[c] = reinterpret_cast<const byte4u *>(q)->v;
      else h[c] = *reinterpret_cast<const half4u *>(q);
      if ((uint32_t)c + 1u < n) row += step;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      if ((uint32_t)c < n) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (MODE == MDSM_F32) {
            acc[e] += f[c][e];
          } else if constexpr (MODE == MDSM_F16) {
            acc[e] += (float)h[c][e];
          } else if constexpr (MODE == MDSM_U8) {
            sum[e] += (u[c] >> (8 * e)) & 0xFFu;
          } else if (c % 2 == 0) {  // channel pairs: one FP16 rounding (a last channel alone adds 0)
            const _Float16 z = (uint32_t)c + 1u < n ? h[c + 1][e] : (_Float16)0.0f;
            acc[e] += (float)(_Float16)(h[c][e] + z);
          }
        }
      }
    }
  };
  uint32_t c = 0;
  for (; c + 16u <= nchans; c += 16u) {
    const i32x16 o = *tab++;
    run16(16u, o);
    if (c + 16u < nchans) row += step;
  }
  if (c < nchans) {
    const i32x16 o = *tab;
    run16(nchans - c, o);
  }
  float4u v;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    v[e] = MODE == MDSM_U8 ? (float)((double)sum[e] * (8.0 / 255.0) + (double)nchans * -4.0) : acc[e];
  *reinterpret_cast<float4u *>(out + (uint64_t)d * nsamp + t) = v;
}

// [trial][cpad] from [channel][trial]; entries past the last channel repeat it
__global__ __launch_bounds__(256) void direct_table_kernel(const int32_t *__restrict__ table,
                                                           uint32_t nchans, uint32_t cpad, uint32_t ndms,
                                                           uint64_t total, int32_t *__restrict__ dtab) {
  const uint64_t e = (uint64_t)blockIdx.x * 256u + threadIdx.x;
  if (e >= total) return;
  const uint32_t d = (uint32_t)(e % ndms), c = (uint32_t)(e / ndms);
  dtab[(uint64_t)d * cpad + c] = table[(uint64_t)min(c, nchans - 1u) * ndms + d];
}
inline uint32_t direct_pad(uint32_t nchans) { return (nchans + 15u) & ~15u; }
// Workgroups (256 samples of four trials each), as many to each XCD as its
// share can be.
inline uint64_t direct_grid(uint32_t ndms, uint32_t nsamp) {
  const uint64_t ntb = ((uint64_t)nsamp + 255u) / 256u, ndg = ((uint64_t)ndms + 3u) / 4u;
  const uint64_t whole = (ntb + 7u) / 8u * ndg;
  return 8u * (whole <= 256u ? whole : (ntb * ndg + 7u) / 8u);
}
// Rows of four samples or more (a lane's), whose grid IDs have 31 bits.
inline bool direct_takes(uint32_t ndms, uint32_t nsamp) { return nsamp >= 4u && direct_grid(ndms, nsamp) < (1ull << 31); }

// ------------------------------------------------------------ variant table
// Variant v: F32 tile (MW, K, CB) and packed tiles (MW, K2, CB) with the same
// TD = 4*MW and similar time extent.
template <int V>
struct VariantDef;
template <> struct VariantDef<1> { using F32 = F32Tile<8, 4, 8>;   using F16 = F16Tile<8, 2, 8>;   using U8 = U8Tile<8, 2, 8>; };
template <> struct VariantDef<2> { using F32 = F32Tile<16, 4, 4>;  using F16 = F16Tile<16, 2, 4>;  using U8 = WindowTile<MDSM_U8, 16>; };
template <> struct VariantDef<3> { using F32 = F32Tile<8, 8, 8>;   using F16 = F16Tile<8, 4, 8>;   using U8 = U8Tile<8, 4, 8>; };
template <> struct VariantDef<4> { using F32 = F32Tile<16, 8, 4>;  using F16 = F16Tile<16, 4, 4>;  using U8 = U8Tile<16, 4, 4>; };
template <> struct VariantDef<5> { using F32 = F32Tile<32, 2, 2>;  using F16 = F16Tile<32, 1, 2>;  using U8 = U8Tile<32, 1, 2>; };
// grouped-read forms of 2 and 1
template <> struct VariantDef<6> { using F32 = F32Tile<16, 4, 4, 8>; using F16 = F16Tile<16, 2, 4, 16>; using U8 = U8Tile<16, 2, 4, 16>; };
template <> struct VariantDef<7> { using F32 = F32Tile<8, 4, 8, 8>;  using F16 = F16Tile<8, 2, 8, 8>;   using U8 = U8Tile<8, 2, 8, 8>; };
template <> struct VariantDef<8> { using F32 = F32Tile<16, 4, 4, 4>; using F16 = F16Tile<16, 2, 4, 8>;  using U8 = U8Tile<16, 2, 4, 8>; };
// few trials per wave, many samples per lane: one address add per 8 (F32)
// or 16 (packed) adds, a smaller delay spread per tile, larger windows
template <> struct VariantDef<9> { using F32 = F32Tile<8, 8, 4>;    using F16 = F16Tile<8, 4, 4>;   using U8 = U8Tile<8, 4, 4>; };
template <> struct VariantDef<10> { using F32 = F32Tile<4, 16, 8>;  using F16 = F16Tile<4, 8, 8>;   using U8 = U8Tile<4, 8, 8>; };
template <> struct VariantDef<11> { using F32 = F32Tile<4, 16, 4>;  using F16 = F16Tile<4, 8, 4>;   using U8 = U8Tile<4, 8, 4>; };
// register windows (F32 and F16 here, U8 in 2); 12 or 16 trials per wave
// with more samples per lane: one address add per 8 or 6 packed adds
template <> struct VariantDef<12> { using F32 = WindowTile<MDSM_F32, 16>; using F16 = WindowTile<MDSM_F16, 16>; using U8 = U8Tile<12, 4, 4>; };
template <> struct VariantDef<13> { using F32 = F32Tile<16, 6, 4>;  using F16 = F16Tile<16, 3, 4>;  using U8 = U8Tile<16, 3, 4>; };
// 16 trials per wave over 8-channel blocks: half the barriers per add
template <> struct VariantDef<14> { using F32 = F32Tile<16, 4, 8>;  using F16 = F16Tile<16, 2, 8>;  using U8 = U8Tile<16, 2, 8>; };
// 12 trials per wave, 2 pairs per lane: fewer accumulators, 7 waves per
// SIMD for the packed tiles (68-72 VGPRs)
template <> struct VariantDef<15> { using F32 = F32Tile<12, 4, 4>;  using F16 = F16Tile<12, 2, 4>;  using U8 = U8Tile<12, 2, 4>; };
constexpr int kNumVariants = 15;
// F16_PAIRS and U8 only: pair-sum tiles (MW, K2, pairs per block, sum rows per pair)
template <int V>
struct PairSumDef;
template <> struct PairSumDef<16> { template <int M> using type = PairSumTile<M, 8, 4, 2, 3>; };
template <> struct PairSumDef<17> { template <int M> using type = PairSumTile<M, 12, 4, 2, 3>; };
template <> struct PairSumDef<18> { template <int M> using type = PairSumTile<M, 12, 2, 2, 3>; };
template <> struct PairSumDef<19> { template <int M> using type = PairSumTile<M, 16, 3, 2, 4>; };
// 17, and 10 trials per wave, with the reads of 2 trials issued ahead of their adds
template <> struct PairSumDef<20> { template <int M> using type = PairSumTile<M, 12, 4, 2, 3, 2>; };
template <> struct PairSumDef<21> { template <int M> using type = PairSumTile<M, 10, 4, 2, 3, 2>; };
// register windows over FP32 sum rows
template <> struct PairSumDef<22> { template <int M> using type = WindowPairTile<M, 16>; };
constexpr int kNumPairSumVariants = 7;
// Eight-wave forms of the register-window shapes (narrow_variant), numbered
// after the public ones: 16 for F32 and F16; 23 (pair sums) and 24 for U8, 23
// for F16_PAIRS.
constexpr int narrow_shapes(int dtype) { return dtype == MDSM_U8 ? 2 : 1; }

template <typename V, typename Fn>
int pick_dtype(int dtype, Fn &&fn) {
  switch (dtype) {
    case MDSM_F32: return fn((typename V::F32 *)nullptr);
    case MDSM_F16: return fn((typename V::F16 *)nullptr);
    case MDSM_U8: return fn((typename V::U8 *)nullptr);
    case MDSM_F16_PAIRS: return fn((typename PairsOf<typename V::F16>::type *)nullptr);
  }
  set_error("unknown input dtype %d", dtype);
  return MDSM_ERR_ARG;
}

template <typename Fn>
int with_tile(int dtype, int variant, Fn &&fn) {
  switch (variant) {
    case 1: return pick_dtype<VariantDef<1>>(dtype, fn);
    case 2: return pick_dtype<VariantDef<2>>(dtype, fn);
    case 3: return pick_dtype<VariantDef<3>>(dtype, fn);
    case 4: return pick_dtype<VariantDef<4>>(dtype, fn);
    case 5: return pick_dtype<VariantDef<5>>(dtype, fn);
    case 6: return pick_dtype<VariantDef<6>>(dtype, fn);
    case 7: return pick_dtype<VariantDef<7>>(dtype, fn);
    case 8: return pick_dtype<VariantDef<8>>(dtype, fn);
    case 9: return pick_dtype<VariantDef<9>>(dtype, fn);
    case 10: return pick_dtype<VariantDef<10>>(dtype, fn);
    case 11: return pick_dtype<VariantDef<11>>(dtype, fn);
    case 12: return pick_dtype<VariantDef<12>>(dtype, fn);
    case 13: return pick_dtype<VariantDef<13>>(dtype, fn);
    case 14: return pick_dtype<VariantDef<14>>(dtype, fn);
    case 15: return pick_dtype<VariantDef<15>>(dtype, fn);
  }
  if (dtype == MDSM_F16_PAIRS) {
    switch (variant) {
      case 16: return fn((PairSumDef<16>::type<MDSM_F16_PAIRS> *)nullptr);
      case 17: return fn((PairSumDef<17>::type<MDSM_F16_PAIRS> *)nullptr);
      case 18: return fn((PairSumDef<18>::type<MDSM_F16_PAIRS> *)nullptr);
      case 19: return fn((PairSumDef<19>::type<MDSM_F16_PAIRS> *)nullptr);
      case 20: return fn((PairSumDef<20>::type<MDSM_F16_PAIRS> *)nullptr);
      case 21: return fn((PairSumDef<21>::type<MDSM_F16_PAIRS> *)nullptr);
      case 22: return fn((PairSumDef<22>::type<MDSM_F16_PAIRS> *)nullptr);
    }
  }
  if (dtype == MDSM_U8) {
    switch (variant) {
      case 16: return fn((PairSumDef<16>::type<MDSM_U8> *)nullptr);
      case 17: return fn((PairSumDef<17>::type<MDSM_U8> *)nullptr);
      case 18: return fn((PairSumDef<18>::type<MDSM_U8> *)nullptr);
      case 19: return fn((PairSumDef<19>::type<MDSM_U8> *)nullptr);
      case 20: return fn((PairSumDef<20>::type<MDSM_U8> *)nullptr);
      case 21: return fn((PairSumDef<21>::type<MDSM_U8> *)nullptr);
      case 22: return fn((PairSumDef<22>::type<MDSM_U8> *)nullptr);
    }
  }
  if (variant == num_variants(dtype) + 1) {
    if (dtype == MDSM_F32) return fn((WindowTile<MDSM_F32, 8> *)nullptr);
    if (dtype == MDSM_F16) return fn((WindowTile<MDSM_F16, 8> *)nullptr);
    if (dtype == MDSM_U8) return fn((WindowPairTile<MDSM_U8, 8> *)nullptr);
    if (dtype == MDSM_F16_PAIRS) return fn((WindowPairTile<MDSM_F16_PAIRS, 8> *)nullptr);
  }
  if (variant == num_variants(dtype) + 2 && dtype == MDSM_U8) return fn((WindowTile<MDSM_U8, 8> *)nullptr);
  set_error("unknown dedispersion variant %d", variant);
  return MDSM_ERR_ARG;
}

// LDS of a workgroup: 64 KB; window tiles, whose registers leave 16 waves per
// CU, take its 160 KB in one workgroup of 16 waves or two of eight.
template <typename Tile>
constexpr uint64_t tile_lds() {
  if constexpr (IsWindow<Tile>::value) return (Tile::WAVES == 8 ? 80 : 160) * 1024;
  else return 64 * 1024;
}

// Channels staged per block: the tile's CB, reduced while the block's LDS
// (two buffers, plus raw staging for U8) exceeds tile_lds (160 KB per CU); even
// for F16_PAIRS, whose channel pairs must not straddle two blocks.
template <typename Tile>
uint32_t stage_channels(uint32_t rw) {
  const uint64_t per = Tile::lds_words_per_row(rw) * sizeof(float);
  const uint64_t step = Tile::PAIRS ? 2 : 1;
  uint64_t n = (uint64_t)Tile::CB;
  while (n > step && n * per > tile_lds<Tile>()) n -= step;
  if (n * per > 160 * 1024) return 0;
  return (uint32_t)n;
}

}  // namespace

int num_variants(int dtype) {
  return (dtype == MDSM_F16_PAIRS || dtype == MDSM_U8) ? kNumVariants + kNumPairSumVariants
                                                       : kNumVariants;
}

// Untuned defaults.  F32 and F16 take the register-window tile, which was
// the fastest shape of every survey tried: 1024 channels x 4096 trials x 2^17
// samples 13.5 ms against 29.7 (F32, shape 8) and 14.6 against 21.9 (F16,
// shape 15); delay slopes from 0.1 to 24 samples per trial 1.5 to 2.5 times;
// 64 channels 1.6 times.  F16_PAIRS and U8 prefer the register windows over
// pair sums (12.4 ms against 14.1, 12.1 against 14.9 of the other pair-sum
// shapes), which take only surveys with few delay differences per channel pair
// and DM tile, and fall back to shapes that take more of them, the last one
// every survey whose delay spread it can stage.
int preferred_variant(int dtype) {
  switch (dtype) {
    case MDSM_F32: return 12;
    case MDSM_F16: return 12;
    default: return 22;
  }
}

// Surveys whose delay differences suit DM tiles of fewer trials than 64 take
// the pair-sum shapes of 40 (U8: 36 against 33 T adds/s of shape 2) or 48, 40
// and 32 trials (F16_PAIRS: 36, 33 and 31 against 25 of shape 15; 256 channels
// x 1920 trials x 81920 samples).
int fallback_variant(int dtype, int n) {
  switch (dtype) {
    case MDSM_F32: return n == 0 ? 8 : 0;
    case MDSM_F16: return n == 0 ? 15 : 0;
    case MDSM_U8: return n == 0 ? 21 : (n == 1 ? 2 : 0);
    default: return n == 0 ? 20 : (n == 1 ? 21 : (n == 2 ? 16 : (n == 3 ? 15 : 0)));
  }
}

int num_shapes(int dtype) { return num_variants(dtype) + narrow_shapes(dtype); }

int narrow_variant(int dtype, int variant) {
  const int nv = num_variants(dtype);
  switch (dtype) {
    case MDSM_F32:
    case MDSM_F16: return variant == 12 ? nv + 1 : 0;
    case MDSM_U8: return variant == 22 ? nv + 1 : (variant == 2 ? nv + 2 : 0);
    default: return variant == 22 ? nv + 1 : 0;
  }
}

// What took a number's surveys before the register windows had it: a survey that
// neither of their forms takes runs there (F32: shape 1's smaller tiles; 22: 40
// trials, 21: 48 trials of pair sums).
static int stand_in(int dtype, int variant) {
  if (dtype == MDSM_F32) return variant == 12 ? 1 : 0;
  if (dtype == MDSM_U8 || dtype == MDSM_F16_PAIRS) return variant == 22 ? 21 : (variant == 21 ? 20 : 0);
  return 0;
}

int numbered_shape(int dtype, int variant, const std::vector<bool> &fits, const std::function<double(int)> &cost,
                   bool *own) {
  const int narrow = narrow_variant(dtype, variant), other = stand_in(dtype, variant);
  *own = true;
  if (narrow && fits[narrow] && (!fits[variant] || cost(narrow) < kBetter * cost(variant))) return narrow;
  if (fits[variant]) return variant;
  *own = false;
  return other && fits[other] ? other : variant;
}

// The shapes that may replace a default one where its tiles pad too much or
// its workgroups wait for their stores (n = 0, 1, ..; 0: no more).
int other_shape(int dtype, int nominal, int n) {
  const int nv = num_variants(dtype);
  if (dtype == MDSM_U8) {
    static const int after22[] = {23, 21, 0}, after21[] = {2, 24, 0}, after2[] = {24, 0};
    return nominal == 22 ? after22[n] : (nominal == 21 ? after21[n] : (nominal == 2 ? after2[n] : 0));
  }
  if (dtype == MDSM_F16_PAIRS) {
    static const int after22[] = {23, 20, 0}, after20[] = {21, 16, 15, 0};
    if (nominal == 22) return after22[n];
    return nominal == 20 ? after20[n] : (nominal == 21 ? after20[n + 1] : (nominal == 16 ? after20[n + 2] : 0));
  }
  return n == 0 && nominal == 12 ? nv + 1 : 0;
}

double tile_count(int dtype, int shape, uint32_t ndms, uint32_t nsamp) {
  const TileShape sh = variant_shape(dtype, shape);
  return (double)((ndms + sh.td() - 1) / sh.td()) * ((nsamp + sh.tt() - 1) / sh.tt());
}

// Estimated time (us) of a launch of `tiles` tiles over nchans channels (in the
// mean of the tiles, `most` in the beam that has most), for the shapes that untuned launches choose between: the rounds of adds, and what
// goes on beside them.
//   Adds: every CU runs one (16 waves) or two workgroups of a shape at a time,
//   so tiles take whole rounds of 256 or 512, each at the shape's full rate; a
//   last round of up to 256 of two per CU, three quarters of one (F32 nine
//   tenths: 256 tiles of 32 trials 204 us, of 64 187, 320 channels).  Tiles of
//   several beams (not equal) end at different times: half a round over the
//   mean instead, and no less than the beam of most channels alone.  T adds/s
//   of the windows measured at 512 to 1024 channels, 1920 trials x 81920 samples,
//   and 0.87 of their time where rows come from the caches (32 to 320 channels);
//   eight waves per workgroup 1.04 to 1.5 times as long per add; 0.4 us per
//   channel at least however few tiles there are.  The word-per-add shapes fit no
//   rounds: 16 (F32) or 25 T adds/s, 0.6 or 0.5 us at least.
//   Beside them: a window tile's workgroups fill their CUs alone, so nothing
//   adds while they store: 0.8 us per million outputs, 7 to 9 at least, 0.7 (F32
//   0.85) and 4 to 7.5 of two eight-wave ones per CU, 0.35 (4) of the pair-sum
//   shapes, 0.5 (3.5) of the word-per-add ones.  At few
//   channels that decides: 64 channels x 4000 trials x 50000 samples 388 us in
//   shape 20 against 427 in 22 (F16_PAIRS), 393 in 21 against 426 (U8); 32 x 160
//   x 256000 F16 60 us in eight waves against 81.
double launch_estimate(int dtype, int shape, double tiles, bool equal, double nchans, double most, double outputs) {
  const int nv = num_variants(dtype);
  const TileShape sh = variant_shape(dtype, shape);
  const double work = (double)sh.td() * sh.tt();
  const bool word = (dtype == MDSM_F32 && shape == 8) || (dtype == MDSM_F16 && shape == 15) ||
                    (dtype == MDSM_F16_PAIRS && shape == 15);
  const bool pair_sums = (dtype == MDSM_U8 || dtype == MDSM_F16_PAIRS) && shape >= 16 && shape <= 21;
  // time of one round's adds and of all of them, and beside them
  double round, adds, start = 3.5, store = 0.5;
  if (word) {
    round = dtype == MDSM_F32 ? 0.6 : 0.5;
    adds = std::max(round * most, 1e-6 * tiles * work / (dtype == MDSM_F32 ? 16.0 : 25.0) * nchans);
  } else {
    const bool pair_windows = shape == 22 || (shape == nv + 1 && (dtype == MDSM_U8 || dtype == MDSM_F16_PAIRS));
    const double wide = dtype == MDSM_F32 ? 39.0 : (pair_windows ? 42.0 : (dtype == MDSM_U8 ? 34.5 : 36.5));
    double rate = wide / 0.87, slots = 256.0;
    start = pair_windows ? 9.0 : (dtype == MDSM_F32 ? 7.0 : 8.5), store = 0.8;
    if (shape > nv) {
      rate /= pair_windows ? 1.5 : (dtype == MDSM_F32 ? 1.17 : 1.04);
      slots = 512.0;
      start -= dtype == MDSM_F32 ? 3.0 : (pair_windows ? 1.5 : 2.0);
      if (!pair_windows) store = dtype == MDSM_F32 ? 0.85 : 0.7;
    } else if (pair_sums) {
      rate = dtype == MDSM_U8 ? 40.5 : (shape == 20 ? 39.5 : (shape == 21 ? 34.5 : 32.5));
      slots = 512.0;
      start = 4.0, store = 0.35;
    }
    // one workgroup alone on its CU, of two that share it
    const double lone = slots > 256.0 ? (dtype == MDSM_F32 ? 0.9 : 0.75) : 1.0;
    double rounds = ceil(tiles / slots);
    if (tiles <= slots * rounds - 256.0) rounds -= 1.0 - lone;
    round = 1e-6 * slots * work / rate;
    if (!equal) {
      const double mean = tiles / slots + 0.5;
      adds = round * std::max(lone * most, (rounds > 1.0 ? mean : std::min(mean, rounds)) * nchans);
    } else {
      adds = std::max(0.4, rounds * round) * nchans;
    }
  }
  return 3.0 + std::max(start, store * 1e-6 * outputs) + adds;
}

// The shape an untuned plan launches for its tile variant `nominal`: the least
// estimate.
//   Eight waves instead of 16, or a shape that pads the trials less (46 trials x
//   218486 samples x 295 channels F16_PAIRS, delay differences for 40 trials:
//   264 us in two such tiles, 205 in one of 48; 32 trials x 600000 samples x 512
//   channels F32: 399 against 598 us; 856 channels x 1222 trials x 15994
//   samples U8, 260 tiles of 16 waves: 540 against 766 us).
//   (by 1 % at least: 514 channels x 700 trials x 19652 samples U8, 234 against
//   236 us by the estimate, 260 against 222 in truth).
//   The word-per-add shapes for F16 rows of fewer than 4 samples, and where few
//   channels (13 of F32, 40 of F16) meet fewer than 128 window tiles, which leave
//   half of the CUs idle (16 channels x 200 trials x 20000 samples F16: 13 us
//   against 16); with more tiles their short rows store slower (3 channels x 6820
//   trials x 311399 samples F32: 3.0 ms against 2.2).
//   Direct kernel, up to 5.3 million outputs of rows padded to 256 samples (2.3
//   to 4.3 of less than 32 trials): 8.5 (F32), 6.6 (F16), 12 (U8) or 6.4 T adds/s
//   (pair sums), 4 us to start and 0.8 us per million outputs stored (256 channels
//   x 64 trials x 8192 samples F32: 18 against 132 us; 512 x 256 x 12000: 205
//   against 257; 646 x 890 x 22 F16: 31 against 300).  More outputs of few trials
//   read their rows from HBM for every four of them (421 channels x 6 trials x
//   10^6 samples F16_PAIRS: 621 us against 540).
// `fits` holds the shapes that take the survey.
int untuned_shape(int dtype, int nominal, const std::vector<bool> &fits, uint32_t nchans, uint32_t ndms,
                  uint32_t nsamp) {
  const double outputs = (double)ndms * nsamp;
  auto tiles = [&](int shape) { return tile_count(dtype, shape, ndms, nsamp); };
  auto cost = [&](int shape) { return launch_estimate(dtype, shape, tiles(shape), true, nchans, nchans, outputs); };
  int best = nominal;
  for (int n = 0, shape; (shape = other_shape(dtype, nominal, n)) != 0; ++n)
    if (fits[shape] && cost(shape) < kBetter * cost(best)) best = shape;
  if ((dtype == MDSM_F32 || dtype == MDSM_F16) && nominal == 12) {
    const int word = dtype == MDSM_F32 ? 8 : 15;
    const bool few = tiles(nominal) < 128.0 && nchans < (dtype == MDSM_F32 ? 13u : 40u);
    if (fits[word] && (few || (dtype == MDSM_F16 && nsamp < 4u))) best = word;
  }
  const double rate = dtype == MDSM_F32 ? 8.5 : dtype == MDSM_F16 ? 6.6 : dtype == MDSM_U8 ? 12.0 : 6.4;
  const double padded = (double)ndms * ((nsamp + 255u) / 256u * 256u);
  const double direct = 4.0 + 0.8e-6 * outputs + 1e-6 * nchans * padded / rate;
  const double limit = ndms >= 32u ? 5.3e6 : 0.36e6 * rate;
  if (direct_takes(ndms, nsamp) && padded <= limit && direct < cost(best)) return kDirectShape;
  return best;
}

TileShape variant_shape(int dtype, int variant) {
  TileShape sh{0, 0, 0};
  with_tile(dtype, variant, [&](auto *tp) {
    using Tile = std::remove_pointer_t<decltype(tp)>;
    sh.mw = Tile::TD / 4;
    sh.k = Tile::TT / 64;
    sh.cb = Tile::CB;
    return MDSM_OK;
  });
  return sh;
}

// Pair-sum tiles: every channel pair's delay difference is >= 0 and takes
// at most ns values inside each DM tile of td trials.
static bool pairsum_accepts(const int32_t *table, uint32_t nchans, uint32_t ndms, uint32_t td,
                            uint32_t ns) {
  for (uint32_t c0 = 0; c0 + 1u < nchans; c0 += 2u) {
    const int32_t *r0 = table + (uint64_t)c0 * ndms, *r1 = r0 + ndms;
    for (uint32_t d0 = 0; d0 < ndms; d0 += td) {
      const uint32_t dl = std::min(d0 + td, ndms);
      int32_t lo = r1[d0] - r0[d0], hi = lo;
      for (uint32_t d = d0 + 1u; d < dl; ++d) {
        const int32_t v = r1[d] - r0[d];
        lo = std::min(lo, v);
        hi = std::max(hi, v);
      }
      if (lo < 0 || (int64_t)hi - lo + 1 > (int64_t)ns) return false;
    }
  }
  return true;
}

uint32_t lds_row_words(int dtype, int variant, uint32_t spread, const int32_t *table,
                       uint32_t nchans, uint32_t ndms) {
  uint32_t rw = 0;
  with_tile(dtype, variant, [&](auto *tp) {
    using Tile = std::remove_pointer_t<decltype(tp)>;
    rw = Tile::fits(spread) ? Tile::row_words(spread) : 0u;
    if constexpr (IsPairSum<Tile>::value || IsWindowPair<Tile>::value) {
      if (!pairsum_accepts(table, nchans, ndms, Tile::TD, Tile::NSUM)) rw = 0;
    }
    return MDSM_OK;
  });
  return rw;
}

uint32_t input_alignment(int dtype) {
  return dtype == MDSM_F32 ? 1u : (storage_dtype(dtype) == MDSM_F16 ? 2u : 4u);
}

uint32_t stage_channels(int dtype, int variant, uint32_t rw) {
  uint32_t cbr = 0;
  with_tile(dtype, variant, [&](auto *tp) {
    using Tile = std::remove_pointer_t<decltype(tp)>;
    cbr = rw ? stage_channels<Tile>(rw) : 0u;
    return MDSM_OK;
  });
  return cbr;
}

uint64_t trial_offset_words(int dtype, int variant, uint32_t nchans, uint32_t ndms, uint32_t cbr) {
  if (variant == kDirectShape) return (uint64_t)ndms * direct_pad(nchans);
  uint64_t n = 0;
  with_tile(dtype, variant, [&](auto *tp) {
    using Tile = std::remove_pointer_t<decltype(tp)>;
    if constexpr (IsWindow<Tile>::value) {
      n = Tile::table_words(nchans, ndms);
      return MDSM_OK;
    } else {
    const uint64_t n_dtiles = (ndms + Tile::TD - 1) / Tile::TD;
    const uint64_t nblocks = cbr ? (nchans + cbr - 1) / cbr : 0;
    n = n_dtiles * nblocks * 4u * Tile::Rel::WORDS;
    if constexpr (IsPairSum<Tile>::value) n += n_dtiles * nblocks * (uint64_t)(Tile::CB / 2) * 2u;
    return MDSM_OK;
    }
  });
  return n;
}

int launch_trial_offsets(int dtype, int variant, const int32_t *table, uint32_t nchans,
                         uint32_t ndms, uint32_t rw, uint32_t cbr, int32_t *reltab, hipStream_t s) {
  if (variant == kDirectShape) {
    const uint64_t total = (uint64_t)ndms * direct_pad(nchans);
    hipLaunchKernelGGL(direct_table_kernel, dim3((uint32_t)((total + 255u) / 256u)), dim3(256), 0, s, table,
                       nchans, direct_pad(nchans), ndms, total, reltab);
    MDSM_HIP(hipGetLastError());
    return MDSM_OK;
  }
  MDSM_REQUIRE(rw > 0 && cbr > 0, MDSM_ERR_ARG, "tile variant %d cannot stage this survey", variant);
  return with_tile(dtype, variant, [&](auto *tp) -> int {
    using Tile = std::remove_pointer_t<decltype(tp)>;
    const uint32_t nblocks = (nchans + cbr - 1) / cbr;
    const uint64_t total = trial_offset_words(dtype, variant, nchans, ndms, cbr);
    const uint64_t grid = (total + 255u) / 256u;
    MDSM_REQUIRE(grid < (1ull << 31), MDSM_ERR_ARG, "trial offset table too large");
    if constexpr (IsPairSum<Tile>::value) {
      MDSM_REQUIRE(cbr % 2u == 0u, MDSM_ERR_ARG, "pair-sum tiles stage whole channel pairs");
      const uint64_t nrel = (uint64_t)((ndms + Tile::TD - 1) / Tile::TD) * nblocks * 4u * Tile::Rel::WORDS;
      hipLaunchKernelGGL(pairsum_offset_kernel<Tile>, dim3((uint32_t)grid), dim3(256), 0, s, table,
                         nchans, ndms, rw, cbr, nblocks, nrel, total, reltab);
    } else if constexpr (IsWindowPair<Tile>::value) {
      MDSM_REQUIRE(cbr % 2u == 0u, MDSM_ERR_ARG, "pair-sum tiles stage whole channel pairs");
      const uint64_t entries = Tile::table_entries(nchans, ndms);
      hipLaunchKernelGGL(window_pair_table_kernel<Tile>, dim3((uint32_t)((entries + 255u) / 256u)),
                         dim3(256), 0, s, table, nchans, ndms, rw, cbr, entries, reltab);
    } else if constexpr (IsWindow<Tile>::value) {
      const uint64_t entries = total / 8u;
      hipLaunchKernelGGL(window_table_kernel<Tile>, dim3((uint32_t)((entries + 255u) / 256u)), dim3(256),
                         0, s, table, nchans, ndms, rw, cbr, entries, reltab);
    } else {
      hipLaunchKernelGGL(trial_offset_kernel<Tile>, dim3((uint32_t)grid), dim3(256), 0, s, table,
                         nchans, ndms, rw, cbr, nblocks, total, reltab);
    }
    MDSM_HIP(hipGetLastError());
    return MDSM_OK;
  });
}

int launch_dedisperse(int dtype, int variant, const void *in, uint64_t ld, const int32_t *table,
                      const int32_t *reltab, uint32_t nchans, uint32_t nsamp, uint32_t ndms,
                      uint32_t rw, float *out, hipStream_t s) {
  if (variant == kDirectShape) {
    MDSM_REQUIRE(reltab, MDSM_ERR_STATE, "delay table missing");
    MDSM_REQUIRE(direct_takes(ndms, nsamp), MDSM_ERR_ARG, "rows too short or too many for the kernel without tiles");
    const dim3 grid((uint32_t)direct_grid(ndms, nsamp));
    const uint32_t cpad = direct_pad(nchans);
    switch (dtype) {
      case MDSM_F32: hipLaunchKernelGGL(dedisp_direct_kernel<MDSM_F32>, grid, dim3(256), 0, s, in, ld, reltab, nchans, cpad, nsamp, ndms, out); break;
      case MDSM_F16: hipLaunchKernelGGL(dedisp_direct_kernel<MDSM_F16>, grid, dim3(256), 0, s, in, ld, reltab, nchans, cpad, nsamp, ndms, out); break;
      case MDSM_U8: hipLaunchKernelGGL(dedisp_direct_kernel<MDSM_U8>, grid, dim3(256), 0, s, in, ld, reltab, nchans, cpad, nsamp, ndms, out); break;
      default: hipLaunchKernelGGL(dedisp_direct_kernel<MDSM_F16_PAIRS>, grid, dim3(256), 0, s, in, ld, reltab, nchans, cpad, nsamp, ndms, out); break;
    }
    MDSM_HIP(hipGetLastError());
    return MDSM_OK;
  }
  MDSM_REQUIRE(rw > 0, MDSM_ERR_ARG,
               "delay spread too large for tile variant %d (choose another variant)", variant);
  MDSM_REQUIRE(reltab, MDSM_ERR_STATE, "trial offset table missing for tile variant %d", variant);
  return with_tile(dtype, variant, [&](auto *tp) -> int {
    using Tile = std::remove_pointer_t<decltype(tp)>;
    const uint32_t n_ttiles = (nsamp + Tile::TT - 1) / Tile::TT;
    const uint32_t n_dtiles = (ndms + Tile::TD - 1) / Tile::TD;
    const uint32_t remap = xcd_remap_enabled() ? 1u : 0u;
    const uint64_t blocks =
        (uint64_t)(remap ? (n_ttiles + 7u) / 8u * 8u : n_ttiles) * n_dtiles;
    MDSM_REQUIRE(blocks < (1ull << 31), MDSM_ERR_ARG, "dedispersion grid too large");
    const uint32_t cbr = stage_channels<Tile>(rw);
    MDSM_REQUIRE(cbr >= 1, MDSM_ERR_ARG, "delay spread too large for LDS staging (%u words)", rw);
    const size_t lds = (size_t)cbr * Tile::lds_words_per_row(rw) * sizeof(float);
    hipLaunchKernelGGL(dedisp_kernel<Tile>, dim3((uint32_t)blocks), dim3(tile_threads<Tile>()), lds, s,
                       reinterpret_cast<const typename Tile::T *>(in), ld, table, reltab, nchans,
                       nsamp, ndms, rw, cbr, n_dtiles, n_ttiles, remap, out);
    MDSM_HIP(hipGetLastError());
    return MDSM_OK;
  });
}

size_t batch_lds_bytes(int dtype, int variant, uint32_t max_rw) {
  size_t bytes = 0;
  with_tile(dtype, variant, [&](auto *tp) {
    using Tile = std::remove_pointer_t<decltype(tp)>;
    bytes = (size_t)stage_channels<Tile>(max_rw) * Tile::lds_words_per_row(max_rw) * sizeof(float);
    return MDSM_OK;
  });
  return bytes;
}

int launch_batch_flat(int dtype, int variant, const BeamDesc *d_beams, uint32_t nbeams,
                      uint32_t total_items, uint32_t max_rw, hipStream_t s) {
  MDSM_REQUIRE(max_rw > 0, MDSM_ERR_ARG, "delay spread too large for tile variant %d", variant);
  return with_tile(dtype, variant, [&](auto *tp) -> int {
    using Tile = std::remove_pointer_t<decltype(tp)>;
    const uint32_t cbr = stage_channels<Tile>(max_rw);
    MDSM_REQUIRE(cbr >= 1, MDSM_ERR_ARG, "delay spread too large for LDS staging");
    const size_t lds = (size_t)cbr * Tile::lds_words_per_row(max_rw) * sizeof(float);
    hipLaunchKernelGGL(batch_flat_kernel<Tile>, dim3(total_items), dim3(tile_threads<Tile>()), lds, s, d_beams,
                       nbeams, cbr);
    MDSM_HIP(hipGetLastError());
    return MDSM_OK;
  });
}

int launch_batch_dedisperse(int dtype, int variant, const BeamDesc *d_beams, uint32_t nbeams,
                            const uint32_t *, uint32_t total_items, uint32_t *d_counter,
                            uint32_t max_rw, int grid, hipStream_t s) {
  MDSM_REQUIRE(max_rw > 0, MDSM_ERR_ARG, "delay spread too large for tile variant %d", variant);
  return with_tile(dtype, variant, [&](auto *tp) -> int {
    using Tile = std::remove_pointer_t<decltype(tp)>;
    const uint32_t cbr = stage_channels<Tile>(max_rw);
    MDSM_REQUIRE(cbr >= 1, MDSM_ERR_ARG, "delay spread too large for LDS staging");
    const size_t lds = (size_t)cbr * Tile::lds_words_per_row(max_rw) * sizeof(float);
    if (grid <= 0) {
      // persistent: as many workgroups as can be resident at once
      int per_cu = 0, dev = 0, cus = 0;
      MDSM_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, batch_kernel<Tile>, tile_threads<Tile>(), lds));
      MDSM_HIP(hipGetDevice(&dev));
      MDSM_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
      grid = std::max(1, per_cu) * std::max(1, cus);
    }
    // every one of the eight queues needs workers: a multiple of 8, at least 8
    grid = std::max(8, (grid + 7) / 8 * 8);
    hipLaunchKernelGGL(batch_kernel<Tile>, dim3(grid), dim3(tile_threads<Tile>()), lds, s, d_beams, nbeams,
                       total_items, cbr, d_counter);
    MDSM_HIP(hipGetLastError());
    return MDSM_OK;
  });
}

}  // namespace mdsm
