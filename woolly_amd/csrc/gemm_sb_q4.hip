// gemm_sb_q4.hip -- gemm_sb.hpp for Q4_K (a translation unit per type: they compile side by side).
#include "gemm_sb.hpp"

int wh::launch_gemm_sb_q4(const SbGemm& a, hipStream_t s) { return sb_launch_type<kGemmQ4S>(a, s); }
