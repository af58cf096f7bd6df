// Given states with the Pfaffian factor (kern_launch.hpp: why a unit of their own).
#include "kern_launch.hpp"
namespace rbmgpu {
template hipError_t launch_eval_pf<float>(const EvalArgs<float>&, Shape, int, hipStream_t);
template hipError_t launch_eval_pf<double>(const EvalArgs<double>&, Shape, int, hipStream_t);
}
