// dc_fold_fp16x3.hip -- FP16X3 instances of the mirrored-pair phase GEMM (dc_fold.h).
#include "dc_fold.h"

namespace dc {

hipError_t launch_fold_fp16x3(int t, const AtomRec *rec, const int *slice_beg, float2 *partial, const float *sq,
                            const int *slice_sq, const GemmGeom &g, const FoldGeom &fg, int slice0, int nslice, int nwg,
                            hipStream_t st) {
    return fold_dispatch<SCH_FP16X3>(t, rec, slice_beg, partial, sq, slice_sq, g, fg, slice0, nslice, nwg, st);
}

}  // namespace dc
