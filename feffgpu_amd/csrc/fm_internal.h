// Calls between the library's sources (not part of the C ABI).
#pragma once
#include <vector>

#include "fm_path.h"

constexpr int FM_SIDE = 2;      // side streams of a set: with the call's own, three lanes
struct fm_overlap {
    int dev = -1;
    hipStream_t side[FM_SIDE] = {};
    hipEvent_t fork = nullptr, join[FM_SIDE] = {};
};

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

// Bytes ms_adjoint runs cnt paths in without chunks.
size_t ms_adjoint_bytes(int precision, const fm_edge &ed, int nleg, int cnt, bool keep);

// The lanes of one call: up to `want` of the stream st and o's side streams, which wait for what st holds so far; join
// (also at the end of its life) makes st wait for them. One lane without o, on another device than o's, or where a
// side stream takes part in a capture that st does not.
struct Lanes {
    fm_overlap *o;
    hipStream_t st;
    int n = 1;
    hipError_t err = hipSuccess;
    Lanes(fm_overlap *o, hipStream_t st, int want);
    ~Lanes() { (void)join(); }
    Lanes(const Lanes &) = delete;
    hipStream_t at(int lane) const { return lane == 0 || lane >= n ? st : o->side[lane - 1]; }
    hipError_t join();
};
// The lane of every bucket: the costliest (paths times legs) first, each to the lane with the least so far.
std::vector<int> lanes_of(int nbucket, const int32_t *offset, const int32_t *nleg, int nlane);

}  // namespace fm
