// Integral images on the device (RGBDImage::calculateIntegral,
// image.cpp:236-277 and :531-556).
//
// 8-bit colour and integer depth: the reference integrates in double with a
// Kahan term; for integer input every partial sum is an exact integer below
// 2^53, so its result is the exact sum rounded once to float (colour) or the
// exact integer (depth, valid).  Here the sums are exact 32-bit integer prefix
// sums (wrapping for depth, see boxDepth), built in two passes:
//   pass A: column prefix sums, 16 row segments per column (coalesced along x);
//   pass B: one wave per row scans 64-pixel segments with DPP/shuffle scans.
// Float colour (non-integer values, CIELab): the reference's sequential
// recurrence is replayed exactly, one lane per channel.
#include <algorithm>

#include "cf_internal.h"

namespace cf {

// pass A: column prefix of 5 channels (r, g, b, depth mm, valid) into tmp[5][H][W].
// A workgroup takes 16 columns; its 16 x 16 lanes split the rows into 16
// segments: each lane sums its segment, the segment totals meet in LDS, and
// each lane writes its segment's prefix sums starting from the totals of the
// segments above (integer sums, so the order of additions does not matter).
// Workgroups of 256 lanes: the serving loop integrates frames while the
// classification of others fills the CUs, and a workgroup of 1024 lanes (16
// waves) got a CU only when a classification launch drained, so the next
// launch, which waits for the frame, started late.
constexpr int kColChunk = 16, kRowSegs = 16;

__global__ void __launch_bounds__(kColChunk * kRowSegs) k_integral_cols_u8(const uint8_t* __restrict__ rgb,
        const uint16_t* __restrict__ depth, int W, int H, uint32_t* __restrict__ tmp) {
    __shared__ uint32_t total[kRowSegs][5][kColChunk];
    const int cx = threadIdx.x % kColChunk, seg = threadIdx.x / kColChunk;
    const int x = blockIdx.x * kColChunk + cx;
    const int rowsPer = (H + kRowSegs - 1) / kRowSegs;
    const int y0 = min(H, seg * rowsPer), y1 = min(H, y0 + rowsPer);
    const bool col = x < W;
    uint32_t sum[5] = {0u, 0u, 0u, 0u, 0u};
    if (col) {
#pragma unroll 4
        for (int y = y0; y < y1; y++) {
            const size_t p = static_cast<size_t>(y) * W + x;
            const uint32_t mm = depth[p];
            sum[0] += rgb[3 * p + 0];
            sum[1] += rgb[3 * p + 1];
            sum[2] += rgb[3 * p + 2];
            sum[3] += mm;
            sum[4] += (mm > 0) ? 1u : 0u;
        }
    }
#pragma unroll
    for (int c = 0; c < 5; c++) total[seg][c][cx] = sum[c];
    __syncthreads();
    uint32_t run[5] = {0u, 0u, 0u, 0u, 0u};
    for (int k = 0; k < seg; k++) {
#pragma unroll
        for (int c = 0; c < 5; c++) run[c] += total[k][c][cx];
    }
    if (!col) return;
    const size_t plane = static_cast<size_t>(W) * H;
#pragma unroll 4
    for (int y = y0; y < y1; y++) {
        const size_t p = static_cast<size_t>(y) * W + x;
        const uint32_t mm = depth[p];
        run[0] += rgb[3 * p + 0];
        run[1] += rgb[3 * p + 1];
        run[2] += rgb[3 * p + 2];
        run[3] += mm;
        run[4] += (mm > 0) ? 1u : 0u;
        tmp[p] = run[0];
        tmp[plane + p] = run[1];
        tmp[2 * plane + p] = run[2];
        tmp[3 * plane + p] = run[3];
        tmp[4 * plane + p] = run[4];
    }
}

// The same for int32 depth (float-colour path: colour handled by the Kahan kernel): channels 3 and 4, rows in
// 16 segments per column (640x480: 199 us with one lane per column walking all rows).
__global__ void __launch_bounds__(kColChunk * kRowSegs) k_integral_cols_depth_i32(const int32_t* __restrict__ depth,
        int W, int H, uint32_t* __restrict__ tmp) {
    __shared__ uint32_t total[kRowSegs][2][kColChunk];
    const int cx = threadIdx.x % kColChunk, seg = threadIdx.x / kColChunk;
    const int x = blockIdx.x * kColChunk + cx;
    const int rowsPer = (H + kRowSegs - 1) / kRowSegs;
    const int y0 = min(H, seg * rowsPer), y1 = min(H, y0 + rowsPer);
    const bool col = x < W;
    uint32_t d = 0, v = 0;
    if (col) {
#pragma unroll 4
        for (int y = y0; y < y1; y++) {
            const int32_t mm = depth[static_cast<size_t>(y) * W + x];
            d += static_cast<uint32_t>(mm > 0 ? mm : 0);
            v += (mm > 0) ? 1u : 0u;
        }
    }
    total[seg][0][cx] = d;
    total[seg][1][cx] = v;
    __syncthreads();
    d = v = 0;
    for (int k = 0; k < seg; k++) {
        d += total[k][0][cx];
        v += total[k][1][cx];
    }
    if (!col) return;
    const size_t plane = static_cast<size_t>(W) * H;
#pragma unroll 4
    for (int y = y0; y < y1; y++) {
        const size_t p = static_cast<size_t>(y) * W + x;
        const int32_t mm = depth[p];
        d += static_cast<uint32_t>(mm > 0 ? mm : 0);
        v += (mm > 0) ? 1u : 0u;
        tmp[3 * plane + p] = d;
        tmp[4 * plane + p] = v;
    }
}

__device__ __forceinline__ uint32_t waveInclusiveScan(uint32_t v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t n = __shfl_up(v, o, 64);
        if (lane >= o) v += n;
    }
    return v;
}

// pass B: row prefix.  blockDim = 256 (4 waves), one wave per (row, channel)
// job; channels 0..2 -> float colour, channel 3+4 -> int2 depth.
__global__ void __launch_bounds__(256) k_integral_rows(const uint32_t* __restrict__ tmp, int W, int H,
        int firstChannel, float* __restrict__ col, int2* __restrict__ dep) {
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    const int numCh = 4 - firstChannel;  // jobs: colour channels [firstChannel,3) + one depth job
    if (wave >= H * numCh) return;
    const int y = wave / numCh;
    const int ch = firstChannel + wave % numCh;
    const size_t plane = static_cast<size_t>(W) * H;
    const size_t row = static_cast<size_t>(y) * W;
    if (ch < 3) {
        uint32_t carry = 0;
        for (int x0 = 0; x0 < W; x0 += 64) {
            const int x = x0 + lane;
            const uint32_t v = (x < W) ? tmp[ch * plane + row + x] : 0u;
            const uint32_t s = waveInclusiveScan(v) + carry;
            if (x < W) col[ch * plane + row + x] = __uint2float_rn(s);
            carry = __shfl(s, 63, 64);
        }
    } else {
        uint32_t cd = 0, cv = 0;
        for (int x0 = 0; x0 < W; x0 += 64) {
            const int x = x0 + lane;
            const uint32_t d = (x < W) ? tmp[3 * plane + row + x] : 0u;
            const uint32_t v = (x < W) ? tmp[4 * plane + row + x] : 0u;
            const uint32_t sd = waveInclusiveScan(d) + cd;
            const uint32_t sv = waveInclusiveScan(v) + cv;
            if (x < W) dep[row + x] = make_int2(static_cast<int>(sd), static_cast<int>(sv));
            cd = __shfl(sd, 63, 64);
            cv = __shfl(sv, 63, 64);
        }
    }
}

// Sequential double Kahan integration of one float channel per thread,
// operation by operation as image.cpp:250-277 with T = double.
__global__ void k_integral_kahan_f32(const float* __restrict__ color, int W, int H, double* __restrict__ work,
        float* __restrict__ col) {
    const int ch = threadIdx.x;
    if (ch >= 3) return;
    const size_t plane = static_cast<size_t>(W) * H;
    const float* in = color + ch * plane;
    double* d = work + ch * plane;
    float* out = col + ch * plane;
    double c = 0.0;
    for (int y = 0; y < H; ++y) {
        for (int x = 0; x < W; ++x) {
            const double above = (y > 0) ? d[(y - 1) * W + x] : 0.0;
            const double left = (x > 0) ? d[y * W + x - 1] : 0.0;
            const double aboveLeft = (x > 0 && y > 0) ? d[(y - 1) * W + x - 1] : 0.0;
            const double cur = static_cast<double>(in[y * W + x]);
            const double dy = __dsub_rn(__dadd_rn(left, above), aboveLeft) - c;
            const double t = __dadd_rn(cur, dy);
            c = __dsub_rn(__dsub_rn(t, cur), dy);
            d[y * W + x] = t;
            out[y * W + x] = __double2float_rn(t);
        }
    }
}

// The same recurrence with everything but its chain of additions taken off the lanes that run it.  A row is
// cut into chunks; while wave 0 (lanes 0..2: the channels) runs chunk n from LDS, the other three waves, one
// per channel, bring chunk n + 1 of the image into LDS as doubles and convert and store the sums of chunk
// n - 1.  The row of partial sums is overwritten in place, the left and above-left terms stay in registers
// (the values are the ones the recurrence stored, so results are identical), and the operands of the next
// kAhead pixels are read while the current ones are summed.  Bound by the four dependent double additions of a
// pixel (about 18 cycles each).  640x480: 9.4 ms; 42.7 ms with loads, conversions and stores in the same lanes.
constexpr int kKahanChunk = 256;
constexpr int kAhead = 8;

__global__ void __launch_bounds__(256) k_integral_kahan_f32_lds(const float* __restrict__ color, int W, int H, int chunk,
        float* __restrict__ col) {
    extern __shared__ double lds[];
    double* rows = lds;                                        // [3][W]
    double* in = lds + static_cast<size_t>(3) * W;             // [2][3][chunk]
    const size_t plane = static_cast<size_t>(W) * H;
    const int perRow = (W + chunk - 1) / chunk;                // at least 2
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int numChunks = perRow * H;
    for (int i = threadIdx.x; i < 3 * W; i += 256) rows[i] = 0.0;
    // chunk n of channel ch into LDS; its sums from the row to memory (waves 1..3)
    auto load = [&](int n, int ch) {
        const int y = n / perRow, x0 = (n - y * perRow) * chunk, len = min(chunk, W - x0);
        const float* src = color + ch * plane + static_cast<size_t>(y) * W + x0;
        double* dst = in + (static_cast<size_t>(n & 1) * 3 + ch) * chunk;
        for (int i = lane; i < len; i += 64) dst[i] = static_cast<double>(src[i]);
    };
    auto store = [&](int n, int ch) {
        const int y = n / perRow, x0 = (n - y * perRow) * chunk, len = min(chunk, W - x0);
        float* dst = col + ch * plane + static_cast<size_t>(y) * W + x0;
        const double* src = rows + static_cast<size_t>(ch) * W + x0;
        for (int i = lane; i < len; i += 64) dst[i] = __double2float_rn(src[i]);
    };
    if (wave > 0) load(0, wave - 1);
    double c = 0.0, left = 0.0, aboveLeft = 0.0;
    for (int n = 0; n < numChunks; n++) {
        __syncthreads();
        if (wave > 0) {
            if (n + 1 < numChunks) load(n + 1, wave - 1);
            if (n > 0) store(n - 1, wave - 1);
        } else if (lane < 3) {
            const int k = n % perRow, x0 = k * chunk, len = min(chunk, W - x0);
            if (k == 0) left = aboveLeft = 0.0;
            double* row = rows + static_cast<size_t>(lane) * W + x0;
            const double* cur = in + (static_cast<size_t>(n & 1) * 3 + lane) * chunk;
            auto step = [&](double above, double v) {
                const double dy = __dsub_rn(__dsub_rn(__dadd_rn(left, above), aboveLeft), c);
                const double t = __dadd_rn(v, dy);
                c = __dsub_rn(__dsub_rn(t, v), dy);
                left = t;
                aboveLeft = above;
                return t;
            };
            int x = 0;
            if (len >= kAhead) {
                double a[kAhead], v[kAhead];
#pragma unroll
                for (int i = 0; i < kAhead; i++) {
                    a[i] = row[i];
                    v[i] = cur[i];
                }
                for (; x + kAhead <= len; x += kAhead) {
                    double na[kAhead], nv[kAhead];
                    const int xn = x + 2 * kAhead <= len ? x + kAhead : x;   // past the last whole block: reread, unused
#pragma unroll
                    for (int i = 0; i < kAhead; i++) {
                        na[i] = row[xn + i];
                        nv[i] = cur[xn + i];
                    }
#pragma unroll
                    for (int i = 0; i < kAhead; i++) row[x + i] = step(a[i], v[i]);
#pragma unroll
                    for (int i = 0; i < kAhead; i++) {
                        a[i] = na[i];
                        v[i] = nv[i];
                    }
                }
            }
            for (; x < len; x++) row[x] = step(row[x], cur[x]);
        }
    }
    __syncthreads();
    if (wave > 0) store(numChunks - 1, wave - 1);
}

void launchIntegralU8(hipStream_t s, const uint8_t* rgb, const uint16_t* depth, int W, int H, uint32_t* tmp,
        float* col, int2* dep) {
    hipLaunchKernelGGL(k_integral_cols_u8, dim3((W + kColChunk - 1) / kColChunk), dim3(kColChunk * kRowSegs), 0, s,
            rgb, depth, W, H, tmp);
    const int jobs = H * 4;
    hipLaunchKernelGGL(k_integral_rows, dim3((jobs * 64 + 255) / 256), dim3(256), 0, s, tmp, W, H, 0, col, dep);
}

void launchIntegralF32(hipStream_t s, const float* color, const int32_t* depth, int W, int H, uint32_t* tmp,
        double* work, float* col, int2* dep) {
    // chunks of at most half a row, so that a chunk's sums are stored before the next row overwrites them
    const int chunk = std::min(kKahanChunk, (W + 1) / 2);
    const size_t lds = (static_cast<size_t>(3) * W + static_cast<size_t>(6) * chunk) * sizeof(double);
    if (W > 1 && lds <= deviceLdsLimit()) {
        allowLds(reinterpret_cast<const void*>(&k_integral_kahan_f32_lds), lds);
        hipLaunchKernelGGL(k_integral_kahan_f32_lds, dim3(1), dim3(256), lds, s, color, W, H, chunk, col);
    } else {
        hipLaunchKernelGGL(k_integral_kahan_f32, dim3(1), dim3(64), 0, s, color, W, H, work, col);
    }
    hipLaunchKernelGGL(k_integral_cols_depth_i32, dim3((W + kColChunk - 1) / kColChunk), dim3(kColChunk * kRowSegs), 0, s,
            depth, W, H, tmp);
    const int jobs = H;  // depth job only
    hipLaunchKernelGGL(k_integral_rows, dim3((jobs * 64 + 255) / 256), dim3(256), 0, s, tmp, W, H, 3, col, dep);
}

// An image smaller than its set's slot, integrated at its own size and then
// padded the way loadImages pads integrated images (RGBDImage::resizeImage,
// image.cpp:449-475): colour NaN and depth sums / valid counts 0 outside it.
__global__ void __launch_bounds__(256) k_integral_pad(const float* __restrict__ srcCol,
        const int2* __restrict__ srcDep, int w, int h, int W, int H, float* __restrict__ col, int2* __restrict__ dep) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y;
    if (x >= W || y >= H) return;
    const bool inside = x < w && y < h;
    const size_t plane = static_cast<size_t>(W) * H, src = static_cast<size_t>(y) * w + x;
    const size_t dst = static_cast<size_t>(y) * W + x;
    const float nan = __int_as_float(0x7fc00000);
#pragma unroll
    for (int c = 0; c < 3; c++) col[c * plane + dst] = inside ? srcCol[c * static_cast<size_t>(w) * h + src] : nan;
    dep[dst] = inside ? srcDep[src] : make_int2(0, 0);
}

void launchIntegralPad(hipStream_t s, const float* srcCol, const int2* srcDep, int w, int h, int W, int H, float* col,
        int2* dep) {
    hipLaunchKernelGGL(k_integral_pad, dim3((W + 255) / 256, H), dim3(256), 0, s, srcCol, srcDep, w, h, W, H, col, dep);
}

}  // namespace cf
