// Host <-> device copies in the caller's layouts (hostio.hip); every call
// returns after its copies have completed.
#pragma once

#include <vector>

#include "common.h"

namespace epic {

constexpr int IO_MAX_GROUPS = 8, IO_MAX_COMP = 8;

// one array of the caller, [parcel][ncomp] FP64, and the device arrays of its
// components (FP64 when wide, else FP32)
struct IoGroup {
    int ncomp;
    bool wide;
    void *dev[IO_MAX_COMP];
    double *host;   // may be null: not copied (download), zeros (upload)
};

// parcel caller index o is slot inv[o], the inverse of orig, which is formed
// in inv (n ints); orig null: slots are caller indices
hipError_t download_parcels(int64_t n, const int *orig, int *inv, const std::vector<IoGroup> &groups, hipStream_t s);
hipError_t upload_parcels(int64_t n, const int *orig, int *inv, const std::vector<IoGroup> &groups, hipStream_t s);
hipError_t launch_iota(int64_t n, int *p, hipStream_t s);

// gives the idle staging buffers back, all of them or all but one set
void release_staging(bool all);
// hipMalloc, tried again without them when memory is short
hipError_t device_malloc(void **p, size_t bytes);

// ncomp components of 32-bit words to out, (-1:nz+1, -1:ny+1, -1:nx+1[, ncomp])
template <class In, class Out> hipError_t download_field(const Grid &g, const In *fld, int ncomp, Out *out, hipStream_t s);
// the interior columns of in (its x and y halos are not read), planes -1..nz+1
hipError_t upload_field(const Grid &g, float *fld, int ncomp, const double *in, hipStream_t s);

}  // namespace epic
