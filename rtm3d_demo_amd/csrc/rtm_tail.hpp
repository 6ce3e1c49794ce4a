// rtm_tail.hpp -- the small operators after a step of one grid, in one launch
// (kernels in rtm_ops.hip).
#pragma once
#include "rtm_internal.hpp"

namespace rtmhip {

// Receivers (extended coordinates; record [rnx][rny][ntstep], time lt).  mode
// 1: sample the field, 2: set it, 3: set it and image the receiver cells.
struct TailReceivers {
    float *rec;
    int rx0, ry0, rz, rdx, rdy, rnx, rny, ntstep, lt, mode;
};
// PP[off] += table[it]
struct TailSource {
    const float *table;
    long long off;
    int it;
};
// After a step with taper3D on its output: the cells with x or y within R of a
// face tapered `taps` times, the front-right edge from the stored (b, y, z),
// the source and the receivers (mode 1 or 2) of PP; taps 0: the source and the
// receivers only.  With tapers the source and
// the receivers must lie off the borders.
template <typename T>
hipError_t launch_tail_all(T *PP, const float *taper, const Grid &g, int b, int R, int taps,
                           const TailReceivers *receivers, const TailSource *source,
                           hipStream_t s);

// After an HBC step: the upper taper of PP's frame (taps times; 0: none), the
// upper-border layer [nx][ny][R] of PP into save or of `field` from restore
// (at most one), the receivers, with img the imaging condition img += ps * PP
// off the step's cells, the source (z >= b).  hold: the step left the layer
// untapered; it is saved with its frame cells tapered taps - 1 times, then
// tapered once.
template <typename T>
struct TailLayer {
    int taps, hold;
    T *save;
    T *field;
    const T *restore;
};
template <typename T>
hipError_t launch_tail_upper(T *PP, const float *taper, const Grid &g, int b, int R,
                             const TailLayer<T> &layer, const TailReceivers *receivers,
                             const TailSource *source, float *img, const T *ps, hipStream_t s);

}  // namespace rtmhip
