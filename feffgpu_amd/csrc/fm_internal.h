// Calls between the library's sources (not part of the C ABI).
#pragma once
#include "fm_path.h"

namespace fm {

// The multiple-scattering paths of 3-6 legs of one bucket (all of one edge and leg count) and what their adjoint reads
// and writes; field meanings as in fm_cchi_backward and fm_chi_paths_backward.
struct MsAdjoint {
    fm_edge ed;
    int npath, first, edge_id, nleg;
    const int32_t *order;
    PathSrc src;
    const void *gcchi;        // mode 0: [npath][E] complex
    const double *greff;      // mode 0: [npath] or NULL
    fm_grid G;                // mode 1
    const int32_t *segment;   // mode 1
    const double *gseg;       // mode 1: [nseg][nk]
    const void *gpath;        // mode 1: [npath][nk] or NULL
    double *gcoord;           // [npath][nslot][3]
    int nslot, nk;
    unsigned char *work;
    size_t work_bytes;
    const void *keep;         // the bucket's kept matrices, or NULL: rebuilt in the workspace
};
hipError_t ms_adjoint(int precision, const MsAdjoint &a, const fm_launch &pol, hipStream_t st);
// Bytes ms_adjoint needs for 16 paths of nleg legs with nothing kept, at the largest E.
size_t ms_adjoint_bytes16(int precision, int nleg);

// The scattering matrices of a launch's paths into keep (the layout of fm_launch.keep).
hipError_t forward_matrices(int precision, const fm_edge &ed, const PathSrc &src, const int32_t *order, int first,
                            int npath, int nleg, void *keep, const fm_launch &pol, hipStream_t st);

}  // namespace fm
