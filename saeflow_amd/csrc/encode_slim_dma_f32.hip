// Small-tile encode kernels, W by LDS DMA, f32 inputs (encode_slim.h).
#define SF_SLIM_DEFINE
#include "encode_slim.h"
namespace sfenc {
template hipError_t launch_slim<SF_F32, S_NMAJOR>(const GemmArgs&, int, int, hipStream_t);
template hipError_t launch_slim<SF_F32, S_KMAJOR>(const GemmArgs&, int, int, hipStream_t);
}  // namespace sfenc
