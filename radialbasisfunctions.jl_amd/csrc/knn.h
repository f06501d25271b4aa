// Internal interface of the grid-hashed k-NN.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rbfx {

// Grow-only device scratch for binning (owned by the library, one per device).
struct KnnWorkspace {
    int32_t *count = nullptr, *start = nullptr, *qcount = nullptr, *qstart = nullptr;
    int32_t *cell = nullptr, *sidx = nullptr, *qcell = nullptr, *qorder = nullptr;
    double *sx = nullptr, *bbox = nullptr;
    double* hbox = nullptr;  // pinned host memory the bounding box is written to
    void *scan_tmp = nullptr, *grid = nullptr;
    size_t cap_count = 0, cap_start = 0, cap_qcount = 0, cap_qstart = 0;
    size_t cap_cell = 0, cap_sidx = 0, cap_qcell = 0, cap_qorder = 0, cap_sx = 0;
    size_t scan_tmp_bytes = 0;
    hipError_t reserve_points(int64_t n_data, int64_t n_query, int dim, bool self, hipStream_t st);
    hipError_t reserve_cells(int64_t ncell, bool self);
};

// out_order (optional, n_query): a processing order of the queries in which neighbours in the
// list are neighbours in space (a Z-curve of the grid's cells).
hipError_t run_knn(KnnWorkspace& ws, const double* data, int64_t n_data, const double* query, int64_t n_query,
                   int dim, int k, const int64_t* q_ptr, int32_t* out, int32_t* out_order, hipStream_t st);

}  // namespace rbfx
