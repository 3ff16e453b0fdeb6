// tdbp_api_internal.h -- host helpers shared by the API, batch and drop-in
// translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "tdbp_internal.h"

namespace tdbp {

int set_error(int code, const char* fmt, ...);
int hip_check(hipError_t e, const char* what);
int ensure_device(int device);
int current_device_ready();
int cu_count();
bool stream_captures(hipStream_t s);   // whether a graph is being captured from it
int validate_geom(const tdbp_geom* g);
void fill_burst(const tdbp_geom* g, BurstDev* b);
int set_tiles(BurstDev* b, int variant, bool named);
std::vector<double> pack_orbit(const tdbp_geom* g);
void point_orbit(BurstDev* b, const double* d_orbit, int n);
int check_samples(const tdbp_samples* s, int precision);
// The variant of a launch that names none, and the same without regard to
// tdbp_set_variant.  named: set by that or in the environment, not built in.
int automatic_variant(int precision, bool* named);
int default_variant(int precision, bool* named);
int fit_on_stream(BurstDev& b, const tdbp_geom* g, double* d_coef,
                  hipStream_t s);
int run_backproject(const tdbp_geom* g, const tdbp_samples* smp,
                    const double* d_satloc, const int16_t* d_dem,
                    const double* d_coef, void* d_out, int precision,
                    int variant, hipStream_t s);

}  // namespace tdbp
