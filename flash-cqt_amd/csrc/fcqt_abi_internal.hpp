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

// From these batch sizes on a buffer is written or read past the caches
// (Store::kStream, load_in<true>). Per slice a round trip touches x, W, X,
// the coefficients, F and y: 2.7 MB, so about 96 slices fill the 256 MB
// memory-side cache, and past that a buffer without a nearby reader only
// pushes W, X and F out to HBM. Measured as loops over three inputs, kept in
// the caches against streamed (us, headline layout; round trip, or the
// direction that is named):
//   x:      B = 96 104.4 / 96.7, 127 140.8 / 133.3, but the analysis alone
//           112 53.5 / 56.2, 120 58.2 / 59.3, 127 62.2 / 62.4, 160 80.1 / 75.0
//   y:      B = 105 116.2 / 113.5, 127 140.8 / 137.8, 144 165.6 / 162.9 (with x)
//   coefficients read by the scatter (with x, y): B = 127 130.5 / 138.9,
//           136 147.9 / 149.6, 144 162.9 / 153.7, 160 189.5 / 166.8
//   coefficients written by the route (with those): B = 160 166.8 / 167.2,
//           176 183.9 / 182.8, 200 210.3 / 206.4, 512 592 / 550; the analysis
//           alone 256 134.7 / 117.4, 512 271.8 / 221.2
//   W read by the row pass (with those): B = 192 194.7 / 194.9,
//           256 266.1 / 257.7, 512 550 / 518; not in the 128-slice chunks of
//           fcqt_sliced_analysis, whose W is in the caches (256 slices 125.5 / 125.8,
//           320 166.5 / 167.9, 512 263 / 263; layout (4, 3) x (12, 48) 109.1 / 110.5, 146.5 / 148.1, 231 / 229)
// TrainableCQT's coefficients (interleaved) go to a new buffer each call, so
// nothing in the caches is there for them: written past the caches from 140
// slices on, training steps at 144 / 160 / 176 slices 404 / 436 / 469 -> 386 / 418 /
// 460 us and round trips without gradients 153.5 / 167.7 / 183.1 -> 151.8 / 163.9 /
// 177.7 (from 105 on steps gain as much, but round trips lose 4 us up to 127).
// So do SlicedCQT's, and streaming both their ends pays earlier: 120 slices 144.4 / 139.2, 128 153.6 / 145.1, 160
// 212.9 / 188.9, 224 296.4 / 262.3 (its analysis alone 57.6 / 58.6 at 120,
// 116.2 / 100.9 at 224), and so does its output from kStreamYMinBatch on:
// 120 slices 137.6 / 135.7, 160 184.3 / 178.3, 224 246.4 / 239.2, its inverse
// alone at 512 304.4 / 292.1. Its signals are read twice (the overlap), so those
// are not streamed.
constexpr int64_t kStreamXMinBatch = 124;
constexpr int64_t kStreamYMinBatch = 105;
constexpr int64_t kStreamCoefInMinBatch = 140;
constexpr int64_t kStreamCoefOutMinBatch = 192;
constexpr int64_t kStreamNewCoefOutMinBatch = 140;
constexpr int64_t kStreamWMinBatch = 192;
constexpr int64_t kStreamSlicedCoefMinBatch = 105;

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
