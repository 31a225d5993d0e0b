// Launchers of the flash-attention forward kernel for the padded and the
// packed bidirectional / causal geometries; attention_kernel.h has the
// kernel and its design notes.
#include "attention_kernel.h"

#define ATTN_ARGS                                                            \
  (const unsigned short*)Q, (const unsigned short*)K,                        \
      (const unsigned short*)V, mask, (unsigned short*)O

extern "C" void launch_attn_fwd(const void* Q, const void* K, const void* V,
                                const float* mask, void* O, int B, int SQ,
                                int SKV, int H, int HKV, int D, bool causal,
                                float scale, long bstr_q, long tstr_q,
                                long bstr_k, long tstr_k,
                                hipStream_t stream) {
  const int nqb = (SQ + 4 * QWAVE - 1) / (4 * QWAVE);
  const bool hm = mask != nullptr;
#define ATTN(DD, CC, MM)                                                     \
  hipLaunchKernelGGL((attn_fwd_kernel<DD, CC, MM>), dim3(B * H * nqb),       \
                     dim3(256), attn_lds(DD, DD, 0, MM), stream, ATTN_ARGS,  \
                     B, SQ, SKV, H, HKV, scale, bstr_q, tstr_q, bstr_k,      \
                     tstr_k)
#define ATTN_D(DD)                                                           \
  do {                                                                       \
    if (causal && hm) ATTN(DD, true, true);                                  \
    else if (causal) ATTN(DD, true, false);                                  \
    else if (hm) ATTN(DD, false, true);                                      \
    else ATTN(DD, false, false);                                             \
  } while (0)
  if (D == 64) ATTN_D(64);
  else if (D == 128) ATTN_D(128);
#undef ATTN_D
#undef ATTN
}

extern "C" void launch_attn_varlen(const void* Q, const void* K,
                                   const void* V, void* O, const int* cu,
                                   const int* blk_seq, const int* blk_qb,
                                   int nblocks, int B, int T, int H, int HKV,
                                   int D, long tstr_q, long tstr_k,
                                   float scale, hipStream_t stream) {
  const float* mask = nullptr;
  const int zero = 8;  // workgroups for the rows past the last sequence
#define AVL(DD)                                                              \
  hipLaunchKernelGGL((attn_fwd_kernel<DD, false, false, true>),              \
                     dim3(nblocks * H + zero), dim3(256),                    \
                     attn_lds(DD, DD, 0, false), stream, ATTN_ARGS, B,       \
                     nblocks, T, H, HKV, scale, 0L, tstr_q, 0L, tstr_k, cu,  \
                     blk_seq, blk_qb)
  if (D == 64) AVL(64);
  else if (D == 128) AVL(128);
#undef AVL
}
