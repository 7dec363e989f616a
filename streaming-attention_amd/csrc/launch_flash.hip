// Launches of the pair attention kernel (flash_attn_kernel) for one configuration.  The build compiles
// this unit once per padded key width DP (16, 32, 64, 128), value-column tile count DVT (1, 2, 4, 8, 16) and
// element size ES (4: fp32, 2: bf16 / fp16), given as -DSTA_FLASH_DP=, -DSTA_FLASH_DVT= and -DSTA_FLASH_ES=, so
// the forty units compile in parallel; each holds the three weights (softmax, exp, Taylor) of its input types.
#include "api_common.hpp"
#include "flash_attn.hip"

#if !defined(STA_FLASH_DP) || !defined(STA_FLASH_DVT) || !defined(STA_FLASH_ES)
#error "launch_flash.hip is compiled with -DSTA_FLASH_DP= -DSTA_FLASH_DVT= -DSTA_FLASH_ES="
#endif

namespace sta_api {

template <int DP, int DVT, int IN>
static void launch_weight(const sta::FlashArgs& a, int weight, unsigned grid, hipStream_t s) {
  if (weight == sta::FLASH_EXP)
    hipLaunchKernelGGL((sta::flash_attn_kernel<DP, DVT, IN, sta::FLASH_EXP>), dim3(grid), dim3(256), 0, s, a);
  else if (weight == sta::FLASH_TAYLOR)
    hipLaunchKernelGGL((sta::flash_attn_kernel<DP, DVT, IN, sta::FLASH_TAYLOR>), dim3(grid), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((sta::flash_attn_kernel<DP, DVT, IN, sta::FLASH_SOFTMAX>), dim3(grid), dim3(256), 0, s, a);
}

template <int DP, int DVT, int ES>
int launch_flash(const sta::FlashArgs& a, int weight, int64_t bh, hipStream_t s) {
  const int64_t grid = bh * a.n_tiles * a.nsplit;
  if (grid <= 0 || grid > 0x7fffffff) return STA_ERR_SHAPE;
  const unsigned g = static_cast<unsigned>(grid);
  if constexpr (ES == 4)
    launch_weight<DP, DVT, sta::F32>(a, weight, g, s);
  else if (a.dtype == STA_F16)
    launch_weight<DP, DVT, sta::F16>(a, weight, g, s);
  else
    launch_weight<DP, DVT, sta::BF16>(a, weight, g, s);
  return check_launch();
}

template int launch_flash<STA_FLASH_DP, STA_FLASH_DVT, STA_FLASH_ES>(const sta::FlashArgs&, int, int64_t, hipStream_t);

}  // namespace sta_api
