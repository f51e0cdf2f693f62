// Packed export of the quantized weight: integer codes as an nbits-wide bitstream per row
// plus a [ngroups, R] scale table and a per-column group index.
//
// The reference keeps its export as two full fp32 [R, C] tensors (int_weight and scale,
// gptq_utils/gptq_plus_utils.py:1866-1871); this format carries the same information in
// nbits/32 + a fraction of the space.  Codes are what fasterquant produced
// (clamp(rint(w/s), -(maxq+1), maxq)); they are stored offset by 2^(nbits-1), so nbits is
// `bits` for sym and `bits + 1` for asym (the asym fake_quantize clamps to the signed range
// [-(maxq+1), maxq], quant_utils.py:477, which needs one more bit).
//
// Row r is a little-endian bitstream: code c occupies bits [c*nbits, (c+1)*nbits) of the
// row, bit b of the row is bit (b & 31) of 32-bit word (b >> 5).  Words past the last code
// are zero-padded.  Dequantisation: Q[r, c] = scales[g_idx[c]][r] * (field(r, c) - 2^(nbits-1)).
//
// k_pack_words (HBM-bound: 2·R·C + R·C·nbits/8 bytes): a workgroup stages whole rows of codes in
// LDS with 16-byte loads; a thread builds word w of each of them, the <= 32/nbits + 2 codes that
// overlap it taken from LDS through invperm (codes still in act_order's permuted order), whose
// entries it reads once for all the rows.  k_pack_rows is the same one word at a time, for rows
// wider than the LDS a workgroup may have.
// k_unpack_dequant (HBM-bound as well): a thread takes 8 columns, nbits whole bytes of the
// bitstream, reads the words they span once and stores 16 bytes of weights or codes.
// 14336 x 4096 codes of 5 bits, permuted, fp16: packing 282 -> 106 us, unpacking 95 -> 45 us (one
// thread per word / per weight before).
#include <type_traits>

#include "rq_common.h"

namespace {

__global__ __launch_bounds__(256) void k_pack_rows(const int16_t* __restrict__ codes, int R, int C,
                                                   int64_t ldc, const int64_t* __restrict__ invperm,
                                                   int nbits, uint32_t* __restrict__ out,
                                                   int64_t ldo, int words, int* __restrict__ range_flag) {
  const int w = blockIdx.x * 256 + threadIdx.x;
  if (w >= words) return;
  const int half = 1 << (nbits - 1);
  const uint32_t mask = (1u << nbits) - 1u;
  const int64_t bit0 = (int64_t)w * 32;
  const int c0 = (int)(bit0 / nbits);
  const int c1 = min(C - 1, (int)((bit0 + 31) / nbits));
  int bad = 0;
  for (int r = blockIdx.y; r < R; r += gridDim.y) {
    const int16_t* crow = codes + (int64_t)r * ldc;
    uint32_t word = 0;
    for (int c = c0; c <= c1; ++c) {
      const int64_t j = invperm ? invperm[c] : c;
      const int v = (int)crow[j] + half;
      bad |= (v < 0) | (v > (int)mask);
      const uint32_t u = (uint32_t)v & mask;
      const int shift = (int)((int64_t)c * nbits - bit0);   // in (-nbits, 32)
      word |= shift >= 0 ? (u << shift) : (u >> (-shift));
    }
    out[(int64_t)r * ldo + w] = word;
  }
  if (bad && range_flag) atomicOr(range_flag, 1);
}

// Rows [r0, r0 + nr) of codes in LDS (row stride cpad elements, a whole number of 16 bytes).
__device__ __forceinline__ void stage_codes(const int16_t* __restrict__ codes, int64_t ldc, int r0, int nr, int C,
                                            int cpad, bool vec, int16_t* buf) {
  if (vec) {
    const int n16 = C / 8, tot = nr * n16;
    for (int q0 = threadIdx.x; q0 < tot; q0 += 256 * 4) {
      uint4 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int q = q0 + 256 * u;
        if (q < tot) v[u] = reinterpret_cast<const uint4*>(codes + (int64_t)(r0 + q / n16) * ldc)[q % n16];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int q = q0 + 256 * u;
        if (q < tot) reinterpret_cast<uint4*>(buf + (q / n16) * cpad)[q % n16] = v[u];
      }
    }
  } else {
    for (int rr = 0; rr < nr; ++rr)
      for (int q = threadIdx.x; q < C; q += 256) buf[rr * cpad + q] = codes[(int64_t)(r0 + rr) * ldc + q];
  }
}

template <int NB>
__global__ __launch_bounds__(256) void k_pack_words(const int16_t* __restrict__ codes, int R, int C, int64_t ldc,
                                                    const int64_t* __restrict__ invperm, uint32_t* __restrict__ out,
                                                    int64_t ldo, int words, int rpw, bool vec,
                                                    int* __restrict__ range_flag) {
  extern __shared__ __attribute__((aligned(16))) int16_t buf[];
  constexpr int NC = (31 + NB - 1) / NB + 1;     // most codes that overlap one word
  constexpr int half = 1 << (NB - 1);
  constexpr uint32_t mask = (1u << NB) - 1u;
  const int r0 = blockIdx.x * rpw, nr = min(rpw, R - r0);
  const int cpad = (C + 7) / 8 * 8;
  stage_codes(codes, ldc, r0, nr, C, cpad, vec, buf);
  __syncthreads();
  uint32_t bad = 0;
  for (int w = threadIdx.x; w < words; w += 256) {
    const int64_t bit0 = (int64_t)w * 32;
    const int c0 = (int)(bit0 / NB);
    const int sh0 = (int)((int64_t)c0 * NB - bit0);       // in (-NB, 0]
    int j[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int c = c0 + k;
      j[k] = (c < C && sh0 + k * NB < 32) ? (invperm ? (int)invperm[c] : c) : -1;
    }
    for (int rr = 0; rr < nr; ++rr) {
      uint32_t word = 0;
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        const uint32_t u = j[k] < 0 ? 0u : (uint32_t)((int)buf[rr * cpad + j[k]] + half);
        bad |= u & ~mask;                                 // a negative field has its high bits set
        const int sh = sh0 + k * NB;
        // sh >= 32 only for a code that is not there (j < 0, u = 0)
        word |= k == 0 ? ((u & mask) >> (-sh)) : ((u & mask) << (sh & 31));
      }
      out[(int64_t)(r0 + rr) * ldo + w] = word;
    }
  }
  if (bad && range_flag) atomicOr(range_flag, 1);
}

template <typename T>
struct alignas(16) Out8 {
  T v[8];
};

template <typename TQ, int NB>
__global__ __launch_bounds__(256) void k_unpack_dequant(const uint32_t* __restrict__ packed, int R,
                                                        int C, int64_t ldp, const float* __restrict__ scales,
                                                        int64_t lds, const int32_t* __restrict__ g_idx,
                                                        TQ* __restrict__ q_out, int64_t ldq,
                                                        int16_t* __restrict__ codes_out, bool vec_q, bool vec_c) {
  const int c = (blockIdx.x * 256 + threadIdx.x) * 8;
  if (c >= C) return;
  const int nc = min(8, C - c);
  constexpr int half = 1 << (NB - 1);
  constexpr uint32_t mask = (1u << NB) - 1u;
  constexpr int NW = (24 + 8 * NB + 31) / 32;            // words that 8 fields may span
  const int64_t bit = (int64_t)c * NB;
  const int64_t wi = bit >> 5;
  const int off = (int)(bit & 31);                       // 0, 8, 16 or 24
  const int nw = (off + nc * NB + 31) >> 5;              // words that these fields span
  int g[8];
  bool one = true;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    g[k] = (q_out && g_idx) ? g_idx[c + (k < nc ? k : 0)] : 0;
    one = one && g[k] == g[0];
  }
  for (int r = blockIdx.y; r < R; r += gridDim.y) {
    const uint32_t* prow = packed + (int64_t)r * ldp + wi;
    uint32_t w[NW + 1];
#pragma unroll
    for (int k = 0; k < NW; ++k) w[k] = k < nw ? prow[k] : 0u;
    w[NW] = 0u;
    // shift the fields down to bit 0
#pragma unroll
    for (int k = 0; k < NW; ++k) w[k] = (uint32_t)((((uint64_t)w[k + 1] << 32) | w[k]) >> off);
    int code[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      constexpr int last = NW;
      const int b = k * NB, i = b >> 5, o = b & 31;
      const uint32_t hi = i + 1 < last ? w[i + 1] : 0u;
      code[k] = (int)((uint32_t)((((uint64_t)hi << 32) | w[i]) >> o) & mask) - half;
    }
    if (codes_out) {
      int16_t* dst = codes_out + (int64_t)r * C + c;
      if (vec_c && nc == 8) {
        Out8<int16_t> v;
#pragma unroll
        for (int k = 0; k < 8; ++k) v.v[k] = (int16_t)code[k];
        *reinterpret_cast<Out8<int16_t>*>(dst) = v;
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (k < nc) dst[k] = (int16_t)code[k];
      }
    }
    if (q_out) {
      const float s0 = scales[(int64_t)g[0] * lds + r];
      Out8<TQ> v;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        float qf = (one ? s0 : scales[(int64_t)g[k] * lds + r]) * (float)code[k];
        // keep fl32(s * code) and the cast to the output type as two roundings (the
        // compiler would otherwise fuse them into one v_fma_mix), as in the write-back
        asm volatile("" : "+v"(qf));
        v.v[k] = rq_cast<TQ>(qf);
      }
      TQ* dst = q_out + (int64_t)r * ldq + c;
      if (vec_q && nc == 8) {
        *reinterpret_cast<Out8<TQ>*>(dst) = v;
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (k < nc) dst[k] = v.v[k];
      }
    }
  }
}

inline int rows_grid(int rows) { return rows < 1024 ? rows : 1024; }

// kernel<NB> for the run-time nbits in [2, 16].
template <typename F>
inline void with_nbits(int nbits, F&& f) {
  switch (nbits) {
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 7: f(std::integral_constant<int, 7>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 9: f(std::integral_constant<int, 9>{}); break;
    case 10: f(std::integral_constant<int, 10>{}); break;
    case 11: f(std::integral_constant<int, 11>{}); break;
    case 12: f(std::integral_constant<int, 12>{}); break;
    case 13: f(std::integral_constant<int, 13>{}); break;
    case 14: f(std::integral_constant<int, 14>{}); break;
    case 15: f(std::integral_constant<int, 15>{}); break;
    default: f(std::integral_constant<int, 16>{}); break;
  }
}

inline bool aligned16(const void* p, int64_t ld_bytes) { return ((uintptr_t)p & 15) == 0 && ld_bytes % 16 == 0; }

}  // namespace

extern "C" int64_t rq_packed_words_per_row(int C, int nbits) {
  if (C <= 0 || nbits < 2 || nbits > 16) return RQ_EINVAL;
  return ((int64_t)C * nbits + 31) / 32;
}

extern "C" int rq_pack_codes(const int16_t* codes, int R, int C, int64_t ldc, const int64_t* invperm,
                             int nbits, uint32_t* out, int64_t ldo, int* range_flag, void* stream) {
  if (!codes || !out || R <= 0 || C <= 0 || ldc < C || nbits < 2 || nbits > 16) return RQ_EINVAL;
  const int64_t words = rq_packed_words_per_row(C, nbits);
  if (ldo < words || words > INT32_MAX) return RQ_EINVAL;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  // Rows staged per workgroup: as many as keep 1024 workgroups (invperm is read once per workgroup),
  // at most 8 and 64 KB of LDS (two workgroups per CU at least); a row of over 64 KB is packed
  // from memory.
  const int64_t rb = (int64_t)(C + 7) / 8 * 16;
  if (rb <= 64 * 1024) {
    int rpw = R / 1024;
    rpw = rpw < 1 ? 1 : (rpw > 8 ? 8 : rpw);
    while (rpw > 1 && rpw * rb > 64 * 1024) --rpw;
    const bool vec = C % 8 == 0 && aligned16(codes, ldc * 2);
    with_nbits(nbits, [&](auto nb) {
      hipLaunchKernelGGL(k_pack_words<decltype(nb)::value>, dim3((R + rpw - 1) / rpw), dim3(256), (size_t)(rpw * rb), s,
                         codes, R, C, ldc, invperm, out, ldo, (int)words, rpw, vec, range_flag);
    });
  } else {
    dim3 grid((unsigned)((words + 255) / 256), rows_grid(R)), block(256);
    hipLaunchKernelGGL(k_pack_rows, grid, block, 0, s, codes, R, C, ldc, invperm, nbits, out, ldo,
                       (int)words, range_flag);
  }
  RQ_CHECK_LAUNCH();
  return RQ_OK;
}

extern "C" int rq_unpack_dequant(const uint32_t* packed, int R, int C, int64_t ldp, int nbits,
                                 const float* scales, int64_t lds, const int32_t* g_idx, void* q_out,
                                 int q_dtype, int64_t ldq, int16_t* codes_out, void* stream) {
  if (!packed || R <= 0 || C <= 0 || nbits < 2 || nbits > 16) return RQ_EINVAL;
  if (ldp < rq_packed_words_per_row(C, nbits)) return RQ_EINVAL;
  if (!q_out && !codes_out) return RQ_EINVAL;
  if (q_out && (!scales || lds < R || ldq < C)) return RQ_EINVAL;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int units = (C + 7) / 8;
  dim3 grid((units + 255) / 256, rows_grid(R)), block(256);
  const bool vec_c = codes_out && aligned16(codes_out, (int64_t)C * 2);
  auto run = [&](auto* q) {
    typedef typename std::remove_pointer<decltype(q)>::type TQ;
    const bool vec_q = q && aligned16(q, ldq * (int64_t)sizeof(TQ));
    with_nbits(nbits, [&](auto nb) {
      hipLaunchKernelGGL((k_unpack_dequant<TQ, decltype(nb)::value>), grid, block, 0, s, packed, R, C, ldp, scales,
                         lds, g_idx, q, ldq, codes_out, vec_q, vec_c);
    });
  };
  if (!q_out || q_dtype == RQ_F16)
    run((__half*)q_out);
  else if (q_dtype == RQ_BF16)
    run((__hip_bfloat16*)q_out);
  else if (q_dtype == RQ_F32)
    run((float*)q_out);
  else
    return RQ_EINVAL;
  RQ_CHECK_LAUNCH();
  return RQ_OK;
}
