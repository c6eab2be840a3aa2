// Host-side helpers shared by the C-ABI launchers (argument checks and
// launch-status capture). Not part of the public header.
#pragma once

#include <cstdint>
#include <cstdio>
#include <hip/hip_runtime.h>

#include "../../include/flashcqt.h"

namespace fcqt {

// grid.x = workgroups per slice * batch must stay below 2^31; the band
// kernel has the most workgroups per slice (< 256), so this is generous.
constexpr int64_t kMaxBatch = 1 << 22;

// fcqt_sliced_analysis runs calls of kAnalysisChunkMinBatch slices and more
// in chunks of about kAnalysisChunk (the header's buffer contract)
constexpr int64_t kAnalysisChunk = FCQT_ANALYSIS_CHUNK;
constexpr int64_t kAnalysisChunkMinBatch = FCQT_ANALYSIS_CHUNK_MIN_BATCH;
static_assert(kAnalysisChunk == 128 && kAnalysisChunkMinBatch == 256, "chunk constants of the header");

// From these sizes on a buffer is written or read past the caches
// (Store::kStream, load_in<true>). Per slice a round trip touches x, W, X,
// the coefficients, F and y: 2.7 MB in the headline layout, so about 96 slices
// fill the 256 MB memory-side cache, and past that a buffer without a nearby
// reader only pushes W, X and F out to HBM. Limits that depend on the
// coefficients' size are in bytes. Measured on one set of buffers over three
// inputs in turn, kept in the caches / streamed, us; A the headline layout
// (132,992 coefficients), B the layout (4, 3) x (12, 48) (99,072); rt a round
// trip, fwd and bwd one direction alone:
//
//   x, 124 slices
//     A rt   96 106.2 / 99.3   112 118.5 / 113.4   128 138.6 / 131.8   144 156.0 / 156.2
//     A fwd  112 53.6 / 54.5   120 58.5 / 58.7     128 62.2 / 61.0     160 79.5 / 75.8
//     B rt   96 91.6 / 89.5    112 104.9 / 102.2   128 120.4 / 114.6   160 159.4 / 160.0
//     B fwd  112 47.4 / 48.5   120 50.0 / 52.0     128 52.8 / 54.4     136 59.7 / 59.2
//     Inputs never seen before (24 in turn) are no slower streamed at any size from
//     96 on (A fwd 112 54.6 / 54.2, B fwd 128 55.2 / 54.0); the losses above are of
//     analyses that repeat an input which the cache still holds.
//   y, 105 slices (its reader, if any, is the caller)
//     A rt   105 116.0 / 112.6  120 132.2 / 128.1  136 150.9 / 150.8   200 203.6 / 200.1
//     A bwd  105 65.1 / 63.9    120 70.8 / 70.6    144 83.9 / 83.9
//     B rt   105 102.8 / 99.9   120 116.7 / 111.8  136 130.7 / 125.9   200 180.5 / 176.8
//     B bwd  105 58.9 / 57.6    120 64.0 / 64.2    144 77.6 / 77.7
//     TrainableCQT's y is a new buffer on each call, which a loss reads at once; steps take
//     -1.4 to +2.7% by it (loops that keep their last result), round trips without gradients
//     gain 2-4% where the last result is dropped and lose up to 5% where it is kept:
//     A step 105 313.7 / 311.6  120 345.2 / 351.5  128 351.8 / 355.7   136 391.2 / 401.7
//     B step 105 289.5 / 285.3  120 315.8 / 319.7  128 324.3 / 331.6   136 350.7 / 355.7
//     A rt, kept 112 125.7 / 129.9   128 137.5 / 142.1   136 154.5 / 163.5   144 153.8 / 153.5
//     A rt, dropped  122.5 / 117.9       131.8 / 129.3       147.4 / 143.1       153.6 / 153.2
//   coefficient planes read by the scatter, x + W + X + planes of 259 MB: the planes
//   just written no longer outlive the rest of the analysis (A 140 slices, B 165)
//     A rt   132 146.2 / 144.5  144 159.5 / 155.0  152 170.6 / 164.1   160 188.2 / 169.8
//     A bwd  132 77.6 / 78.0    144 82.2 / 83.1    164 93.7 / 93.9     172 97.7 / 96.9
//     B rt   144 137.3 / 143.4  160 158.4 / 160.6  164 162.0 / 161.1   172 177.5 / 165.5
//     B bwd  144 76.3 / 77.5    164 83.9 / 85.1    168 88.7 / 87.0     172 88.4 / 87.6
//   coefficient planes written by the route, the same buffers of 354 MB (A and C 192, B 224):
//   round trips gain from about there on; analyses alone rewrite planes of which the
//   cache still holds a part and gain later (C the layout (2, 5, 2) x (4, 8, 64), 131,968)
//     A rt   192 197.7 / 197.7  216 217.1 / 217.6  229 246.4 / 234.8   272 312.4 / 271.2
//     A fwd  192 88.7 / 89.2    216 99.0 / 100.0   229 107.7 / 108.0   280 148.9 / 124.4
//     C rt   200 211.7 / 202.6  229 239.0 / 228.0      C fwd 200 92.5 / 92.0   229 107.5 / 104.1
//     B rt   200 182.4 / 185.4  216 192.7 / 196.8  229 207.4 / 207.5   260 247.6 / 238.9
//     B fwd  200 80.3 / 84.5    216 83.8 / 90.1    229 91.0 / 93.9     280 111.5 / 111.7
//   TrainableCQT's coefficients (interleaved, a new buffer on each call, so that the
//   cache holds nothing of it), 140 slices, written
//     A step 136 402.3 / 387.7  144 407.2 / 393.5  160 433.0 / 428.5   192 504.3 / 493.1
//     A rt   128 132.8 / 140.0  136 151.0 / 150.8  144 154.9 / 154.9   160 169.8 / 167.7
//     B step 136 361.3 / 348.8  144 368.4 / 359.9  160 404.1 / 387.5   192 452.6 / 445.8
//     B rt   128 114.9 / 123.2  136 128.6 / 132.5  144 139.7 / 138.5   160 150.5 / 148.7
//   and read, with the gradients, which are read as coefficients too
//     A step 132 385.4 / 368.0  140 389.0 / 378.9  160 429.5 / 421.3   172 453.3 / 450.2
//     A rt   132 142.5 / 143.3  140 149.9 / 148.8  160 170.6 / 164.9   172 182.8 / 175.7
//     B step 132 340.5 / 335.8  140 353.8 / 346.6  160 386.9 / 382.2   172 415.8 / 413.8
//     B rt   132 121.1 / 123.9  140 133.4 / 133.5  160 149.4 / 146.7   172 162.0 / 157.7
//   (loops that drop each result; one that keeps its last gains at every size from 105 on)
//   W read by the row pass, 192 slices of a whole call (in the 128-slice chunks of
//   fcqt_sliced_analysis, whose W was written just before, either form is within 1%:
//   A fwd 384 188.9 / 190.7, 512 263.9 / 262.2, rt 320 364.0 / 360.3, 512 566.0 / 567.4)
//     A rt   192 196.6 / 196.2  224 227.4 / 227.3  256 268.6 / 262.8   320 333.6 / 319.6
//     B rt   192 183.8 / 183.6  224 205.1 / 204.0  256 235.8 / 233.4   320 299.7 / 286.3
//   SlicedCQT's coefficients (a new buffer on each call), written and read, 105 slices;
//   in a loop that keeps its last result, and, dropping it before the next call, so that
//   the allocator hands the same block out again
//     A rt   104 136.5 / 124.2  120 147.8 / 136.7  136 167.8 / 157.2   144 181.2 / 163.8
//       dropped: 118.2 / 124.1      133.8 / 136.8      160.3 / 157.0       180.0 / 163.7
//     A fwd  104 60.8 / 54.5    120 66.0 / 59.9    136 77.4 / 72.5     144 81.1 / 74.0
//       dropped: 52.6 / 55.0        59.5 / 60.1        74.3 / 72.7         78.3 / 74.4
//     B rt   104 122.1 / 110.5  120 128.2 / 122.0  136 149.3 / 142.3   144 160.8 / 147.8
//       dropped: 104.5 / 111.2      116.3 / 122.2      138.5 / 141.6       151.7 / 148.1
//   SlicedCQT's output, kStreamYMinBatch: rt 120 137.6 / 135.7, 160 184.3 / 178.3, 224 246.4 /
//   239.2, bwd 512 304.4 / 292.1. Its signals are read twice (the overlap) and not streamed.
constexpr int64_t kStreamXMinBatch = 124;
constexpr int64_t kStreamYMinBatch = 105;
constexpr int64_t kStreamPlanesInBytes = 259000000;
constexpr int64_t kStreamPlanesOutBytes = 353600000;
constexpr int64_t kStreamInterleavedMinBatch = 140;
constexpr int64_t kStreamWMinBatch = 192;
constexpr int64_t kStreamSlicedCoefMinBatch = 105;

// Bytes of x, W, X and the coefficients of a call of `batch` slices.
inline int64_t analysis_bytes(int64_t batch, int64_t ncoef) { return batch * (4 * FCQT_N + 16 * FCQT_L + 8 * ncoef); }
inline bool stream_planes_in(int64_t batch, int64_t ncoef) {
    return analysis_bytes(batch, ncoef) >= kStreamPlanesInBytes;
}
inline bool stream_planes_out(int64_t batch, int64_t ncoef) {
    return analysis_bytes(batch, ncoef) >= kStreamPlanesOutBytes;
}

inline bool aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

// Checks shared by the band launchers (FCQT_OK, FCQT_EARG or FCQT_EALIGN):
// record and task tables, the descriptor's coefficient span against ncoef,
// layout, alignment; defined in bands.hip.
int check_band_args(const fcqt_tables* tab, const int32_t* rec, const float* cre, const float* cim, int layout,
                    int64_t batch);

// fcqt_packed_fft_inv; last = true when nothing reads y soon after the call
// (large batches then store it without keeping it in the caches); defined
// in packed_fft.hip.
int packed_fft_inv(const fcqt_tables* tab, const int32_t* ovf, const float* f, float* y, float* work, int64_t batch,
                   bool last, hipStream_t stream);

// fcqt_slice_fft_fwd of one chunk of a call of `total` slices (which sets
// the cache choices); defined in packed_fft.hip.
int slice_fft_fwd(const fcqt_tables* tab, const float* sig, int64_t sig_len, const float* window, int64_t nsig,
                  int64_t nslices, int64_t first, int64_t origin, float* xs, float* work, int64_t total,
                  hipStream_t stream);

// The inverse passes of one streamed slice per signal with the half-slice
// overlap-add in the row pass's store (arguments checked by the caller);
// defined in packed_fft.hip.
int stream_inv_passes(const fcqt_tables* tab, const int32_t* ovf, const float* f, float* work, float* tail, float* out,
                      int64_t nsig, int64_t slice, hipStream_t stream);

// Text of the last failed launch on this host thread.
inline char* last_error_buf() {
    static thread_local char buf[256] = {0};
    return buf;
}

// Status of the launch just issued: FCQT_OK, or FCQT_ELAUNCH with the HIP
// error text recorded for fcqt_last_hip_error().
inline int launch_status() {
    const hipError_t e = hipGetLastError();
    if (e == hipSuccess) return FCQT_OK;
    std::snprintf(last_error_buf(), 256, "%s (%d)", hipGetErrorString(e), (int)e);
    return FCQT_ELAUNCH;
}

}  // namespace fcqt
