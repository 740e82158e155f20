// ingest.hip -- SIGPROC sample unpack fused with the corner turn.
//
// The reference unpacks each spectrum on the host (read_block,
// src/mdsm-multibeam/file_handler.cpp:193-287) and scatters it into
// [beam][chan][t] float rows one value at a time (readBinaryData,
// src/MDSM.cpp:71-104).  Here the packed bytes are copied to the device
// as they are (1/8 of the float volume for 4-bit data) and one kernel
// decodes and transposes them:
//
//   tile = 64 spectra x 64 channels, 256 threads (4 waves);
//   read:  each wave reads one spectrum's 64 channels (consecutive bytes,
//          shorts or floats) and decodes them into LDS row t;
//   write: each wave writes 64 consecutive samples (256 B) of one channel
//          row from LDS column c (row pitch 65 words: no bank conflicts).
//
// The kernel moves nbits/8 bytes in and 4 bytes out per sample: it is
// bound by HBM writes, and in a streaming reader by the PCIe copy before it.
#include <hip/hip_runtime.h>

#include "internal.h"

namespace mdsm {
namespace {

constexpr int CT_T = 64;   // spectra per tile
constexpr int CT_C = 64;   // channels per tile
constexpr int CT_NT = 256;

template <int NBITS>
__device__ __forceinline__ float decode(const uint8_t *__restrict__ row, uint32_t g) {
  if constexpr (NBITS < 8) {
    const uint32_t bit = g * NBITS;
    return (float)((row[bit >> 3] >> (bit & 7)) & ((1u << NBITS) - 1u));
  } else if constexpr (NBITS == 8) {
    return (float)row[g];
  } else if constexpr (NBITS == 16) {
    return (float)reinterpret_cast<const uint16_t *>(row)[g];
  } else {
    return reinterpret_cast<const float *>(row)[g];
  }
}

template <int NBITS>
__global__ __launch_bounds__(CT_NT) void unpack_ct_kernel(const uint8_t *__restrict__ in,
                                                          uint64_t spec_bytes, uint32_t nspec,
                                                          uint32_t ctot, uint32_t nchans,
                                                          float *__restrict__ out, uint64_t ld,
                                                          uint64_t beam_stride, uint64_t col0) {
  __shared__ float tile[CT_T][CT_C + 1];
  const uint32_t lx = threadIdx.x & 63, ly = threadIdx.x >> 6;
  const uint64_t t0 = (uint64_t)blockIdx.x * CT_T;
  const uint32_t g0 = blockIdx.y * CT_C;
  const uint32_t g = g0 + lx;
  for (uint32_t r = ly; r < CT_T; r += CT_NT / 64) {
    const uint64_t t = t0 + r;
    if (t < nspec && g < ctot) tile[r][lx] = decode<NBITS>(in + t * spec_bytes, g);
  }
  __syncthreads();
  const uint64_t t = t0 + lx;
  if (t >= nspec) return;
  for (uint32_t r = ly; r < CT_C; r += CT_NT / 64) {
    const uint32_t gg = g0 + r;
    if (gg >= ctot) break;
    const uint32_t b = gg / nchans, c = gg - b * nchans;
    out[b * beam_stride + (uint64_t)c * ld + col0 + t] = tile[lx][r];
  }
}

// Register corner turn: a lane reads CH channels of four consecutive spectra
// (accesses of up to 16 bytes) and writes four consecutive samples of CH
// channel rows, one 16-byte store each, so a wave writes 1 KB of a row at a
// time and nothing goes through LDS.  The four waves of a workgroup take
// neighbouring groups of channels, so the cache lines of their 256 spectra
// are used up while they are near.  Bound by HBM writes and by the partial
// lines at the ends of each 1 KB: 1024 channels x 65536 8-bit spectra into
// rows off the line grid 74 us (4.5 TB/s in and out; 159 us through the LDS
// tile, whose loads and stores are of one value per lane), 4 bits 56 us, 1
// bit 46 us, 32 bits with cache-bypassing stores 87 us (139 us without; 8
// bits 84 us with them).
constexpr int CT8_T = 256;  // spectra per workgroup (4 per lane)
// groups of CH channels per wave, and whether stores bypass the caches: with
// more input per output the L2 is better left to the input
constexpr int ct8_groups(int nbits) { return nbits >= 16 ? 2 : 1; }

template <int NBITS, int CH>
__global__ __launch_bounds__(CT_NT) void unpack_ct8_kernel(const uint8_t *__restrict__ in,
                                                           uint64_t spec_bytes, uint32_t nspec,
                                                           uint32_t ntb, uint32_t ctot, uint32_t nchans,
                                                           float *__restrict__ out, uint64_t ld,
                                                           uint64_t beam_stride, uint64_t col0) {
  typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
  constexpr uint32_t BYTES = CH * NBITS / 8;  // of one spectrum
  constexpr uint32_t G = ct8_groups(NBITS);
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  // workgroups are dealt round-robin over the 8 XCDs: XCD x takes a run of
  // adjacent time blocks, so that the cache lines shared by two of them meet
  // in one L2
  const uint32_t per = (ntb + 7u) / 8u, k = blockIdx.x >> 3;
  const uint32_t tb = (blockIdx.x & 7u) * per + k % per, cblk = k / per;
  const uint64_t t = (uint64_t)tb * CT8_T + 4u * lane;
  if (tb >= ntb || t >= nspec) return;
  const uint32_t have = (uint32_t)(nspec - t < 4u ? nspec - t : 4u);
  for (uint32_t g = 0; g < G; ++g) {
    const uint32_t c0 = (uint32_t)CH * ((cblk * G + g) * (CT_NT / 64) + wave);
    if (c0 >= ctot) return;
    uint32_t w[4][(BYTES + 3) / 4];
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
      // (spectra past the last one repeat it; they are not stored)
      const uint8_t *p = in + (t + (k < have ? k : have - 1u)) * spec_bytes + (uint64_t)c0 * NBITS / 8u;
      if constexpr (BYTES == 1) w[k][0] = *p;
      else if constexpr (BYTES == 2) w[k][0] = *reinterpret_cast<const uint16_t *>(p);
      else if constexpr (BYTES == 4) w[k][0] = *reinterpret_cast<const uint32_t *>(p);
      else if constexpr (BYTES == 8) {
        const uint2 q = *reinterpret_cast<const uint2 *>(p);
        w[k][0] = q.x, w[k][1] = q.y;
      } else {
#pragma unroll
        for (uint32_t i = 0; i < BYTES / 16u; ++i) {
          const uint4 q = reinterpret_cast<const uint4 *>(p)[i];
          w[k][4 * i] = q.x, w[k][4 * i + 1] = q.y, w[k][4 * i + 2] = q.z, w[k][4 * i + 3] = q.w;
        }
      }
    }
    auto value = [&](uint32_t k, uint32_t e) {
      const uint32_t word = w[k][e * NBITS / 32];
      if constexpr (NBITS == 32) return __uint_as_float(word);
      else return (float)((word >> (e * NBITS % 32)) & ((1u << NBITS) - 1u));
    };
#pragma unroll
    for (uint32_t e = 0; e < (uint32_t)CH; ++e) {
      const uint32_t gg = c0 + e, b = gg / nchans, c = gg - b * nchans;
      float *o = out + b * beam_stride + (uint64_t)c * ld + col0 + t;
      if (have == 4u) {
        const float4u v = {value(0, e), value(1, e), value(2, e), value(3, e)};
        if constexpr (NBITS >= 16) __builtin_nontemporal_store(v, reinterpret_cast<float4u *>(o));
        else *reinterpret_cast<float4u *>(o) = v;
      } else {
        for (uint32_t k = 0; k < have; ++k) o[k] = k == 0 ? value(0, e) : k == 1 ? value(1, e) : value(2, e);
      }
    }
  }
}

// The register form takes whole groups of 8 channels (16 in up to 8 bits where
// the count allows) whose bytes start on a multiple of their access size.
template <int NBITS, int CH>
bool launch_ct8(const uint8_t *in, uint64_t spec_bytes, uint32_t nspec, uint32_t ctot, uint32_t nchans,
                float *out, uint64_t ld, uint64_t beam_stride, uint64_t col0, hipStream_t s) {
  constexpr uint64_t A = CH * NBITS / 8 < 16 ? CH * NBITS / 8 : 16;
  if (ctot % CH != 0 || (reinterpret_cast<uintptr_t>(in) | spec_bytes) % A != 0) return false;
  constexpr uint32_t per = CH * ct8_groups(NBITS) * (CT_NT / 64);
  const uint32_t ntb = (nspec + CT8_T - 1) / CT8_T;
  const uint64_t blocks = (uint64_t)((ntb + 7u) / 8u * 8u) * ((ctot + per - 1) / per);
  if (blocks >= (1ull << 31)) return false;
  hipLaunchKernelGGL((unpack_ct8_kernel<NBITS, CH>), dim3((uint32_t)blocks), dim3(CT_NT), 0, s, in, spec_bytes,
                     nspec, ntb, ctot, nchans, out, ld, beam_stride, col0);
  return true;
}

template <int NBITS>
void launch_ct(const uint8_t *in, uint64_t spec_bytes, uint32_t nspec, uint32_t ctot, uint32_t nchans,
               float *out, uint64_t ld, uint64_t beam_stride, uint64_t col0, hipStream_t s) {
  if (NBITS <= 8 &&
      launch_ct8<NBITS, (NBITS <= 8 ? 16 : 8)>(in, spec_bytes, nspec, ctot, nchans, out, ld, beam_stride, col0, s))
    return;
  if (launch_ct8<NBITS, 8>(in, spec_bytes, nspec, ctot, nchans, out, ld, beam_stride, col0, s)) return;
  hipLaunchKernelGGL(unpack_ct_kernel<NBITS>, dim3((nspec + CT_T - 1) / CT_T, (ctot + CT_C - 1) / CT_C),
                     dim3(CT_NT), 0, s, in, spec_bytes, nspec, ctot, nchans, out, ld, beam_stride, col0);
}

}  // namespace

int launch_unpack_corner_turn(const void *in, int nbits, uint32_t nspec, uint32_t nchans,
                              uint32_t nbeams, float *out, uint64_t ld, uint64_t beam_stride,
                              uint64_t col0, hipStream_t s) {
  const uint32_t ctot = nchans * nbeams;
  const uint64_t spec_bytes = (uint64_t)ctot * nbits / 8;
  if (nspec == 0) return MDSM_OK;
  const auto *p = static_cast<const uint8_t *>(in);
  switch (nbits) {
    case 1: launch_ct<1>(p, spec_bytes, nspec, ctot, nchans, out, ld, beam_stride, col0, s); break;
    case 2: launch_ct<2>(p, spec_bytes, nspec, ctot, nchans, out, ld, beam_stride, col0, s); break;
    case 4: launch_ct<4>(p, spec_bytes, nspec, ctot, nchans, out, ld, beam_stride, col0, s); break;
    case 8: launch_ct<8>(p, spec_bytes, nspec, ctot, nchans, out, ld, beam_stride, col0, s); break;
    case 16: launch_ct<16>(p, spec_bytes, nspec, ctot, nchans, out, ld, beam_stride, col0, s); break;
    case 32: launch_ct<32>(p, spec_bytes, nspec, ctot, nchans, out, ld, beam_stride, col0, s); break;
    default: set_error("nbits must be 1, 2, 4, 8, 16 or 32 (got %d)", nbits); return MDSM_ERR_ARG;
  }
  MDSM_HIP(hipGetLastError());
  return MDSM_OK;
}

}  // namespace mdsm
