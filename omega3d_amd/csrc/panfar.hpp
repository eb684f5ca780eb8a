// panfar.hpp -- panel sums with their separated pairs on the matrix cores (panfar.hip)
#pragma once
#include "pan_kernels.hpp"

namespace o3d {

struct PtPanArgs;

// the recursive rule and the 7-point rule of panels acting on points, and particles
// acting on panels
enum { PANFAR_POINTS = 0, PANFAR_POINTS7 = 1, PANFAR_PARTICLES = 2 };

// whether a call of `units` sources (panels or particles) on nt targets is better off there
bool panfar_pays(int rule, int64_t units, int64_t nt, int method, int tile, int prec);
// the stream's workspace of at least `bytes`, when it can be had: no allocation while the
// stream is captured, and the direct kernels need far less when memory is short (hold
// stream_ws_mutex())
bool panfar_scratch(size_t bytes, hipStream_t st, void** ws);
// scratch of a call, and the call on it: FP32 or compensated, outputs accumulated
size_t panfar_bytes(int rule, int64_t units, int64_t nt, bool grad);
int panfar_points(const PanArgs& p, int rule, bool grad, int prec, void* ws, hipStream_t st);
int panfar_particles(const PtPanArgs& t, int prec, void* ws, hipStream_t st);

}  // namespace o3d
