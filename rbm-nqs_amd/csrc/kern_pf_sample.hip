// The samplers with the Pfaffian factor (kern_launch.hpp: why a unit of their own).
#include "kern_launch.hpp"
namespace rbmgpu {
template hipError_t launch_sample_pf<float>(const SampArgs<float>&, Shape, int, hipStream_t);
template hipError_t launch_sample_pf<double>(const SampArgs<double>&, Shape, int, hipStream_t);
}
