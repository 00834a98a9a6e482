// One translation unit per (head dim, element type) of the attention kernels: hbsattn_amd/build.py compiles this file
// once for each value of HBSA_D (32, 64, 128, 256), HBSA_E (ElemBF16, ElemF16) and HBSA_PART:
//   1  forward with 16-bit output (both forms)     2  forward with fp32 output (fp32 tensors staged as fp16)
//   3  backward                                    4  forward on fp32 operands
//   5  forward, head dims up to HBSA_D (also 96, 160 and 192)
//   6  forward, few queries per item                 7  forward that counts the blocks itself
//   8, 9  forms 1 (one launch) and 5 cut over key blocks
//   10, 11  forms 1 and 7, and 5, with two teams for the tiles of an item
//   12  form 1 on a prepared mask, packed slots, cut over key blocks
//   13  the one-launch form of 1, packed slots, eight wavefronts
#if HBSA_PART == 1
#include "hbsa_fwd_kernel.h"
template int hbsa::launch_fwd<HBSA_D, hbsa::HBSA_E, false>(const FwdParams &, long long, hipStream_t);
template int hbsa::launch_fwd_fused<HBSA_D, hbsa::HBSA_E>(const FwdParams &, long long, hipStream_t);
#elif HBSA_PART == 2
#include "hbsa_fwd_kernel.h"
template int hbsa::launch_fwd<HBSA_D, hbsa::HBSA_E, true>(const FwdParams &, long long, hipStream_t);
#elif HBSA_PART == 3
#include "hbsa_bwd.h"
template int hbsa::launch_bwd<HBSA_D, hbsa::HBSA_E>(const BwdParams &, int, int, hipStream_t);
#elif HBSA_PART == 4
#include "hbsa_fwd_f32.h"
template int hbsa::launch_fwd_f32<HBSA_D>(const FwdParams &, float, long long, hipStream_t);
#elif HBSA_PART == 5
#include "hbsa_fwd_kernel.h"
template int hbsa::launch_fwd_cols<HBSA_D, hbsa::HBSA_E, false, 1>(const FwdParams &, long long, hipStream_t);
#elif HBSA_PART == 6
#include "hbsa_fwd_decode.h"
template int hbsa::launch_fwd_decode<HBSA_D, hbsa::HBSA_E>(const FwdParams &, int, long long, hipStream_t);
#elif HBSA_PART == 7
#include "hbsa_fwd_kernel.h"
template int hbsa::launch_fwd_counted<HBSA_D, hbsa::HBSA_E>(const FwdParams &, long long, hipStream_t);
#elif HBSA_PART == 8
#include "hbsa_fwd_kernel.h"
template int hbsa::launch_fwd_parts<HBSA_D, hbsa::HBSA_E>(const FwdParams &, long long, hipStream_t);
#elif HBSA_PART == 9
#include "hbsa_fwd_kernel.h"
template int hbsa::launch_fwd_cols<HBSA_D, hbsa::HBSA_E, true, 1>(const FwdParams &, long long, hipStream_t);
#elif HBSA_PART == 10
#include "hbsa_fwd_kernel.h"
template int hbsa::launch_fwd_teams<HBSA_D, hbsa::HBSA_E>(const FwdParams &, long long, hipStream_t);
#elif HBSA_PART == 11
#include "hbsa_fwd_kernel.h"
template int hbsa::launch_fwd_cols<HBSA_D, hbsa::HBSA_E, false, 2>(const FwdParams &, long long, hipStream_t);
#elif HBSA_PART == 12
#include "hbsa_fwd_kernel.h"
template int hbsa::launch_fwd_prepared_parts<HBSA_D, hbsa::HBSA_E>(const FwdParams &, long long, hipStream_t);
#elif HBSA_PART == 13
#include "hbsa_fwd_kernel.h"
template int hbsa::launch_packed_eights<HBSA_D, hbsa::HBSA_E>(const FwdParams &, long long, hipStream_t);
#else
#error "HBSA_PART is 1 to 13"
#endif
