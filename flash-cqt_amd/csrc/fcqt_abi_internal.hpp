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
// the coefficients, F and y: 2.7 MB, so about 96 slices fill the 256 MB
// memory-side cache, and past that a buffer without a nearby reader only
// pushes W, X and F out to HBM. Measured as loops over three inputs, kept in
// the caches against streamed (us, headline layout; round trip, or the
// direction that is named):
//   x:      B = 96 104.4 / 96.7, 127 140.8 / 133.3, but the analysis alone
//           112 53.5 / 56.2, 120 58.2 / 59.3, 127 62.2 / 62.4, 160 80.1 / 75.0
//   y:      B = 105 116.2 / 113.5, 127 140.8 / 137.8, 144 165.6 / 162.9 (with x)
//   coefficient planes read by the scatter (with x, y): once an analysis's buffers
//           (x, W, X, planes) hold 259 MB, a little more than the cache, which the planes do
//           not outlive: 140 slices; 165 in the layout of 99,072 coefficients. B = 132
//           146.2 / 144.5, 136 147.4 / 145.5, 144 159.5 / 155.0, 160 188.2 / 169.8; that layout 144 137.3 / 143.4,
//           160 158.4 / 160.6, 164 162.0 / 161.1, 172 177.5 / 165.5 (the synthesis alone
//           144 82.2 / 83.1, 164 93.7 / 93.9, 172 97.7 / 96.9; 144 76.3 / 77.5, 168 88.7 / 87.0)
//   interleaved coefficients read: from 140 slices on in both layouts (training steps, which also
//           read their gradients so, 140 389.0 / 378.9, 160 429.5 / 421.3; 353.8 / 346.6, 386.9 /
//           382.2; round trips without gradients 140 149.9 / 148.8, 160 170.6 / 164.9; 133.4 / 133.5, 149.4 / 146.7)
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
// So do SlicedCQT's, and streaming both their ends pays earlier, from where a
// round trip's buffers hold 340 MB (126 slices; 140 in the layout (4, 3) x (12, 48) of
// 99,072 coefficients against 132,992): round trips at 105 / 112 / 120 / 128 / 136 /
// 144 / 160 slices 120.5 / 125.1 / 132.7 / 142.6 / 162.0 / 181.3 / 205.3 kept, 126.7 /
// 130.5 / 137.1 / 142.9 / 160.9 / 165.0 / 176.6 streamed; in that layout 108.2 / 112.5 /
// 116.8 / 123.5 / 142.4 / 150.8 / 177.4 against 113.3 / 117.5 / 123.3 / 128.6 / 144.9 /
// 148.9 / 163.8 (two signals of half as many slices alike). So does its output from kStreamYMinBatch on:
// 120 slices 137.6 / 135.7, 160 184.3 / 178.3, 224 246.4 / 239.2, its inverse
// alone at 512 304.4 / 292.1. Its signals are read twice (the overlap), so those
// are not streamed.
constexpr int64_t kStreamXMinBatch = 124;
constexpr int64_t kStreamYMinBatch = 105;
constexpr int64_t kStreamPlanesInBytes = 259000000;
constexpr int64_t kStreamCoefInMinBatch = 140;
constexpr int64_t kStreamCoefOutMinBatch = 192;
constexpr int64_t kStreamNewCoefOutMinBatch = 140;
constexpr int64_t kStreamWMinBatch = 192;
constexpr int64_t kStreamSlicedCoefBytes = 340000000;

// Bytes of x, W, X and the coefficients, and of a round trip's buffers (F and y
// too), for a call of `batch` slices.
inline int64_t analysis_bytes(int64_t batch, int64_t ncoef) { return batch * (4 * FCQT_N + 16 * FCQT_L + 8 * ncoef); }
inline int64_t round_trip_bytes(int64_t batch, int64_t ncoef) {
    return analysis_bytes(batch, ncoef) + batch * (8 * FCQT_FROW + 4 * FCQT_N);
}
inline bool stream_planes_in(int64_t batch, int64_t ncoef) {
    return analysis_bytes(batch, ncoef) >= kStreamPlanesInBytes;
}
inline bool stream_sliced_coef(int64_t batch, int64_t ncoef) {
    return round_trip_bytes(batch, ncoef) >= kStreamSlicedCoefBytes;
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
