// fp32 activations for the fp16 MFMA kernels: the power-of-two prescale that brings a tensor into fp16's
// range, and the split of (prescaled) values into fp16 terms.
//
// The ternary kernels multiply fp16 operands. fp32 activations are carried as hi = fp16(x), lo = fp16(x - hi)
// (22 significant bits), which only works while x sits inside fp16's exponent range: above 65504 hi
// overflows, below ~6e-5 the terms are subnormal and lose their bits. The reference multiplies in fp32
// (tmq/tmq_cuda.cu:242-427) and has no such limit. So a caller first scales the tensor by the power of two s
// that puts max|x| into [1024, 2048) -- exact, whatever the magnitude -- and folds 1/s into the
// per-channel scale of the epilogue; elements more than 2^14 below the maximum keep an absolute
// precision of 2^-35 of that maximum, which is below the rounding of the fp32 accumulation.
#include "common.h"
#include "mfma.h"
#include "range.h"

namespace tmq {
namespace {

constexpr int kPartials = 1024;           // partial maxima of the multi-block scan
constexpr int64_t kSingleMax = 1 << 16;   // up to here one workgroup does everything in one launch

// The partial maxima of a scan, reduced by every workgroup of 256 of the reordering launch behind it: the (at most 1024)
// values are asked for at once and ahead of the workgroup's own data -- four trips to memory one after the other
// otherwise --, and after the one barrier every thread takes the largest of the four wavefronts' maxima itself (with the
// scan: [32, 128, 28, 28] 10.3 -> 9.7 us, [64, 64, 56, 56] 31.0 -> 27.5, [1, 16, 512, 512] 13.6 -> 10.5).
struct PartialMaxima {
    float v[kPartials / 256];
    __device__ __forceinline__ PartialMaxima(const float *__restrict__ partials, int count) {
#pragma unroll
        for (int i = 0; i < kPartials / 256; i++) {
            const int at = i * 256 + (int)threadIdx.x;
            v[i] = 0.f;
            if (at < count) v[i] = partials[at];
        }
    }
    __device__ __forceinline__ float reduce(float *lds /* 4 floats, used once */) const {
        float m = 0.f;
#pragma unroll
        for (int i = 0; i < kPartials / 256; i++) m = fmaxf(m, v[i]);
        m = wave_max(m);
        if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = m;
        __syncthreads();
        return fmaxf(fmaxf(lds[0], lds[1]), fmaxf(lds[2], lds[3]));
    }
};

// maximum over the workgroup, valid in every thread
__device__ __forceinline__ float block_max(float v, float *lds /* >= 17 floats */) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    v = wave_max(v);
    if (lane == 0) lds[wv] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        float t = 0.f;
        for (int i = 0; i < nw; i++) t = fmaxf(t, lds[i]);
        lds[16] = t;
    }
    __syncthreads();
    return lds[16];
}

__device__ __forceinline__ float scan_abs_max(const float *__restrict__ x, int64_t n, int64_t first, int64_t stride, bool vec) {
    float m = 0.f;
    if (vec) {
        const int64_t n4 = n / 4;
        for (int64_t i = first; i < n4; i += stride) {
            const floatx4 v = *reinterpret_cast<const floatx4 *>(x + 4 * i);
            m = fmaxf(fmaxf(m, fmaxf(finite_abs(v[0]), finite_abs(v[1]))), fmaxf(finite_abs(v[2]), finite_abs(v[3])));
        }
        for (int64_t i = 4 * n4 + first; i < n; i += stride) m = fmaxf(m, finite_abs(x[i]));
    } else {
        for (int64_t i = first; i < n; i += stride) m = fmaxf(m, finite_abs(x[i]));
    }
    return m;
}

__device__ __forceinline__ void write_scale(const float *scale_in, float *scale_out, int64_t channels, float inv) {
    if (!scale_out) return;
    for (int64_t c = threadIdx.x; c < channels; c += blockDim.x) scale_out[c] = (scale_in ? scale_in[c] : 1.f) * inv;
}

// Small tensors: one workgroup scans, derives the prescale, writes the scaled copy and the adjusted
// per-channel scale -- one launch in front of a GEMV.
__global__ __launch_bounds__(1024) void prescale_single_kernel(const float *__restrict__ x, int64_t n, float *prescale,
                                                               float *__restrict__ xs, const float *scale_in,
                                                               float *scale_out, int64_t channels, int vec) {
    __shared__ float lds[17];
    const float amax = block_max(scan_abs_max(x, n, threadIdx.x, blockDim.x, vec != 0), lds);
    float s, inv;
    make_prescale(amax, s, inv);
    if (threadIdx.x == 0) {
        prescale[0] = s;
        prescale[1] = inv;
    }
    if (xs) {
        if (vec) {
            const int64_t n4 = n / 4;
            for (int64_t i = threadIdx.x; i < n4; i += blockDim.x)
                *reinterpret_cast<floatx4 *>(xs + 4 * i) = *reinterpret_cast<const floatx4 *>(x + 4 * i) * s;
            for (int64_t i = 4 * n4 + threadIdx.x; i < n; i += blockDim.x) xs[i] = x[i] * s;
        } else {
            for (int64_t i = threadIdx.x; i < n; i += blockDim.x) xs[i] = x[i] * s;
        }
    }
    write_scale(scale_in, scale_out, channels, inv);
}

__global__ __launch_bounds__(256) void absmax_partial_kernel(const float *__restrict__ x, int64_t n, float *partials, int vec) {
    __shared__ float lds[17];
    const float m = block_max(scan_abs_max(x, n, (int64_t)blockIdx.x * 256 + threadIdx.x, (int64_t)gridDim.x * 256, vec != 0), lds);
    if (threadIdx.x == 0) partials[blockIdx.x] = m;
}

__global__ __launch_bounds__(1024) void prescale_finalize_kernel(const float *partials, int count, float *prescale,
                                                                 const float *scale_in, float *scale_out, int64_t channels) {
    __shared__ float lds[17];
    const float amax = block_max((int)threadIdx.x < count ? partials[threadIdx.x] : 0.f, lds);
    float s, inv;
    make_prescale(amax, s, inv);
    if (threadIdx.x == 0) {
        prescale[0] = s;
        prescale[1] = inv;
    }
    write_scale(scale_in, scale_out, channels, inv);
}

__global__ __launch_bounds__(256) void scale_copy_kernel(const float *__restrict__ x, const float *prescale,
                                                         float *__restrict__ xs, int64_t n, int vec) {
    const float s = prescale[0];
    const int64_t i0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i0 >= n) return;
    if (vec && i0 + 4 <= n) {
        *reinterpret_cast<floatx4 *>(xs + i0) = __builtin_nontemporal_load(reinterpret_cast<const floatx4 *>(x + i0)) * s;
    } else {
        for (int64_t i = i0; i < n && i < i0 + 4; i++) xs[i] = x[i] * s;
    }
}

// x s = hi + lo with hi = fp16(x s), lo = fp16(x s - hi): 22 significant bits in two fp16 values (s = 1 without
// a prescale; lo may be left out). 8 elements per thread (two 16-byte loads, a 16-byte store per term) when
// the pointers allow it.
template <bool LO, bool SCALED>
__global__ __launch_bounds__(256) void split_terms_kernel(const float *__restrict__ x, const float *prescale,
                                                          _Float16 *__restrict__ hi, _Float16 *__restrict__ lo, int64_t n,
                                                          int vec) {
    float s = 1.f;
    if constexpr (SCALED) s = prescale[0];
    const int64_t i0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (i0 >= n) return;
    if (vec && i0 + 8 <= n) {
        floatx4 a = __builtin_nontemporal_load(reinterpret_cast<const floatx4 *>(x + i0));
        floatx4 b = __builtin_nontemporal_load(reinterpret_cast<const floatx4 *>(x + i0 + 4));
        if constexpr (SCALED) {
            a *= s;
            b *= s;
        }
        half8 h, l;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            h[e] = (_Float16)a[e];
            h[4 + e] = (_Float16)b[e];
            l[e] = (_Float16)(a[e] - (float)h[e]);
            l[4 + e] = (_Float16)(b[e] - (float)h[4 + e]);
        }
        *reinterpret_cast<half8 *>(hi + i0) = h;
        if constexpr (LO) *reinterpret_cast<half8 *>(lo + i0) = l;
    } else {
        for (int64_t i = i0; i < n && i < i0 + 8; i++) {
            const float v = SCALED ? x[i] * s : x[i];
            const _Float16 h = (_Float16)v;
            hi[i] = h;
            if constexpr (LO) lo[i] = (_Float16)(v - (float)h);
        }
    }
}

// A few fp32 rows as fp16 row pairs, each row with a prescale of its own: one workgroup per row finds the row's
// largest finite |x|, scales by the power of two s that brings it into [1024, 2048) and writes hi = fp16(s x) and
// lo = fp16(s x - hi) to x16, 1 / s to row_scale[m]. The rows go in groups of `group` (the last may be shorter):
// group g occupies x16 rows 2 g group onwards, its hi rows first, then its lo rows. The fp16 rows have Kp >= K values
// (a multiple of 8), zeros behind the K-th. vec: K a multiple of 4 and x 16-byte aligned (whole float4s).
__global__ __launch_bounds__(1024) void split_rows_kernel(const float *__restrict__ x, int64_t K, int64_t Kp, int rows, int group,
                                                          _Float16 *__restrict__ x16, float *__restrict__ row_scale, int vec) {
    __shared__ float lds[17];
    const int m = blockIdx.x;
    const int g = m / group, w = m - g * group, in_group = rows - g * group < group ? rows - g * group : group;
    const float *row = x + (int64_t)m * K;
    const float amax = block_max(scan_abs_max(row, K, threadIdx.x, 1024, vec != 0), lds);
    float s, inv;
    make_prescale(amax, s, inv);
    if (threadIdx.x == 0) row_scale[m] = inv;
    _Float16 *hi = x16 + (int64_t)(2 * g * group + w) * Kp, *lo = hi + (int64_t)in_group * Kp;
    for (int64_t i0 = (int64_t)threadIdx.x * 8; i0 < Kp; i0 += 8192) {
        floatx4 a = {0.f, 0.f, 0.f, 0.f}, b = {0.f, 0.f, 0.f, 0.f};
        if (vec) {
            if (i0 < K) a = *reinterpret_cast<const floatx4 *>(row + i0) * s;
            if (i0 + 4 < K) b = *reinterpret_cast<const floatx4 *>(row + i0 + 4) * s;
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (i0 + e < K) a[e] = row[i0 + e] * s;
                if (i0 + 4 + e < K) b[e] = row[i0 + 4 + e] * s;
            }
        }
        half8 h, l;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            h[e] = (_Float16)a[e];
            h[4 + e] = (_Float16)b[e];
            l[e] = (_Float16)(a[e] - (float)h[e]);
            l[4 + e] = (_Float16)(b[e] - (float)h[4 + e]);
        }
        *reinterpret_cast<half8 *>(hi + i0) = h;
        *reinterpret_cast<half8 *>(lo + i0) = l;
    }
}

// Largest finite |x| of 4096 values per workgroup and round (four 16-byte loads per thread in flight), one partial
// per workgroup. x 16-byte aligned; the n % 4 values at the end go to workgroup 0.
__global__ __launch_bounds__(256) void absmax_wide_kernel(const float *__restrict__ x, int64_t n, float *partials) {
    __shared__ float lds[17];
    const int64_t n4 = n / 4;
    float m = 0.f;
    for (int64_t base = (int64_t)blockIdx.x * 1024; base < n4; base += (int64_t)gridDim.x * 1024) {
        floatx4 v[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int64_t at = base + i * 256 + threadIdx.x;
            v[i] = at < n4 ? __builtin_nontemporal_load(reinterpret_cast<const floatx4 *>(x) + at) : floatx4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
            m = fmaxf(fmaxf(m, fmaxf(finite_abs(v[i][0]), finite_abs(v[i][1]))), fmaxf(finite_abs(v[i][2]), finite_abs(v[i][3])));
    }
    if (blockIdx.x == 0 && threadIdx.x < (n & 3)) m = fmaxf(m, finite_abs(x[4 * n4 + threadIdx.x]));
    m = block_max(m, lds);
    if (threadIdx.x == 0) partials[blockIdx.x] = m;
}

// hi = fp16(s x) for the whole tensor in the launch after absmax_wide_kernel: every workgroup asks for its 8192 values
// first, reduces the partial maxima itself while they are on their way (at most 1024 floats), derives s, converts, and
// writes its slice of the per-channel scale divided by s; workgroup 0 also writes the prescale.
__global__ __launch_bounds__(256) void convert_prescaled_kernel(const float *__restrict__ x, int64_t n,
                                                                const float *__restrict__ partials, int count,
                                                                _Float16 *__restrict__ hi, float *prescale,
                                                                const float *scale_in, float *scale_out, int64_t channels,
                                                                int vec) {
    __shared__ float lds[17];
    constexpr int kQuads = 8;                                      // float4s per thread
    const int64_t n4 = n / 4, base = (int64_t)blockIdx.x * (256 * kQuads);
    floatx4 v[kQuads];
    if (vec) {
#pragma unroll
        for (int i = 0; i < kQuads; i++) {
            const int64_t at = base + i * 256 + threadIdx.x;
            v[i] = at < n4 ? __builtin_nontemporal_load(reinterpret_cast<const floatx4 *>(x) + at) : floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
    float pm = 0.f;
    for (int i = threadIdx.x; i < count; i += 256) pm = fmaxf(pm, partials[i]);      // (PartialMaxima: 51 MB 23.0 -> 24.4 us)
    float s, inv;
    make_prescale(block_max(pm, lds), s, inv);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        prescale[0] = s;
        prescale[1] = inv;
    }
    if (scale_out)
        for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < channels; c += (int64_t)gridDim.x * 256)
            scale_out[c] = (scale_in ? scale_in[c] : 1.f) * inv;
    if (vec) {
#pragma unroll
        for (int i = 0; i < kQuads; i++) {
            const int64_t at = base + i * 256 + threadIdx.x;
            if (at >= n4) continue;
            const floatx4 a = v[i] * s;
            *reinterpret_cast<half4 *>(hi + 4 * at) = half4{(_Float16)a[0], (_Float16)a[1], (_Float16)a[2], (_Float16)a[3]};
        }
        if (blockIdx.x == 0 && threadIdx.x < (n & 3)) hi[4 * n4 + threadIdx.x] = (_Float16)(x[4 * n4 + threadIdx.x] * s);
    } else {
        for (int64_t i = base * 4 + threadIdx.x; i < n && i < (base + 256 * kQuads) * 4; i += 256) hi[i] = (_Float16)(x[i] * s);
    }
}

// The same conversion for a planar tensor [B][C][HW] into channels-last order [B][HW][C] (what the convolution kernels
// read): a workgroup takes CT channels x PT = 4096 / CT pixels, a thread 4 channels x 4 pixels of it -- four 16-byte loads
// along the planes, all on their way while the partial maxima are reduced -- turns its block in registers, and the tile
// goes out through LDS in pieces of 8 channels, 128-byte runs per pixel at CT = 64. Bound by memory: 4 bytes in, 2 out a
// value. Converted in place and left to a strided copy before: [32, 128, 28, 28] 7.8 + 13.6 us in two launches; the layer (128 -> 128, 3 x 3) 38.3 -> 29.4 us.
// (Where tiles are mostly empty the two launches are faster: planar_tiles_pay.)
// vec: HW a multiple of 4 and x 16-byte aligned (a quad of pixels is one load); out_piece 8 / 4: C a multiple of 8 / 4 and
// hi 16- / 8-byte aligned (pieces of 8 / 4 channels are one store); everything else element by element.
template <int CT>
__global__ __launch_bounds__(256) void convert_prescaled_nhwc_kernel(const float *__restrict__ x, int64_t C, int64_t HW,
                                                                     int tiles_p, int tiles_c, int64_t tiles,
                                                                     const float *__restrict__ partials,
                                                                     int count, _Float16 *__restrict__ hi, float *prescale,
                                                                     const float *scale_in, float *scale_out, int64_t channels,
                                                                     int vec, int out_piece) {
    constexpr int PT = 4096 / CT, QP = PT / 4, kRow = CT + 4;      // (rows of CT + 4 halfs: the 8-byte accesses spread over the banks)
    __shared__ float lds[4];
    __shared__ __attribute__((aligned(16))) _Float16 tile[PT * kRow];
    const int tid = threadIdx.x, pq = tid % QP, cq = tid / QP;
    float s = 1.f, inv;
    const PartialMaxima maxima(partials, count);
    for (int64_t t = blockIdx.x; t < tiles; t += gridDim.x) {
        int tp, tc;
        const int64_t bt = div_rem(t, tiles_p, tp), b = div_rem(bt, tiles_c, tc);
        const int64_t c0 = (int64_t)tc * CT, p0 = (int64_t)tp * PT;
        const int64_t c = c0 + cq * 4, p = p0 + pq * 4;
        const float *src = x + (b * C + c) * HW + p;
        floatx4 v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            v[k] = floatx4{0.f, 0.f, 0.f, 0.f};
            if (c + k < C) {
                if (vec) {
                    if (p < HW) v[k] = __builtin_nontemporal_load(reinterpret_cast<const floatx4 *>(src + k * HW));
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (p + e < HW) v[k][e] = src[k * HW + e];
                }
            }
        }
        if (t == blockIdx.x) {                                     // once per workgroup
            make_prescale(maxima.reduce(lds), s, inv);
            if (blockIdx.x == 0 && tid == 0) {
                prescale[0] = s;
                prescale[1] = inv;
            }
            if (scale_out)
                for (int64_t i = (int64_t)blockIdx.x * 256 + tid; i < channels; i += (int64_t)gridDim.x * 256)
                    scale_out[i] = (scale_in ? scale_in[i] : 1.f) * inv;
        } else {
            __syncthreads();                                       // the last tile has been read out
        }
#pragma unroll
        for (int e = 0; e < 4; e++)
            *reinterpret_cast<half4 *>(&tile[(pq * 4 + e) * kRow + cq * 4]) =
                half4{(_Float16)(v[0][e] * s), (_Float16)(v[1][e] * s), (_Float16)(v[2][e] * s), (_Float16)(v[3][e] * s)};
        __syncthreads();
        _Float16 *dst = hi + (b * HW + p0) * C + c0;
        const int live_p = HW - p0 < PT ? (int)(HW - p0) : PT, live_c = C - c0 < CT ? (int)(C - c0) : CT;
        if (out_piece == 8) {
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int at = i * 256 + tid, row = at / (CT / 8), c8 = (at % (CT / 8)) * 8;
                if (row >= live_p || c8 >= live_c) continue;
                const half4 lo = *reinterpret_cast<const half4 *>(&tile[row * kRow + c8]), up = *reinterpret_cast<const half4 *>(&tile[row * kRow + c8 + 4]);
                *reinterpret_cast<half8 *>(dst + row * C + c8) = half8{lo[0], lo[1], lo[2], lo[3], up[0], up[1], up[2], up[3]};
            }
        } else if (out_piece == 4) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int at = i * 256 + tid, row = at / (CT / 4), c4 = (at % (CT / 4)) * 4;
                if (row >= live_p || c4 >= live_c) continue;
                *reinterpret_cast<half4 *>(dst + row * C + c4) = *reinterpret_cast<const half4 *>(&tile[row * kRow + c4]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int at = i * 256 + tid, row = at / CT, ch = at % CT;
                if (row < live_p && ch < live_c) dst[row * C + ch] = tile[row * kRow + ch];
            }
        }
    }
}

// channels per tile: no more than there are, so that few channels don't leave most of a tile empty
inline int planar_tile_channels(int64_t C) { return C <= 16 ? 16 : C <= 32 ? 32 : 64; }
inline int64_t planar_tiles(int64_t B, int64_t C, int64_t HW) {
    const int64_t CT = planar_tile_channels(C), PT = 4096 / CT;
    return B * ((C + CT - 1) / CT) * ((HW + PT - 1) / PT);
}
inline bool planar_vec(const void *x, int64_t HW) { return HW % 4 == 0 && aligned16(x); }

// Whether the reordering launch beats the conversion in place followed by a strided copy. Every tile costs a workgroup
// that reduces the partial maxima again, however little of it exists (4.5 ns each beyond the first round, 5.6 without quad
// loads), where the two launches cost 5 us more at rest and 2.7 ns per 4096 values. 618 shapes of 3e4, 1e6 and 1.2e7 values,
// 2 .. 2048 channels, planes of 2 .. 111222 pixels, copy = 1: up to 1.00 where this says yes, 0.78 and more where it says no --
// [64, 3, 224, 224] 1.94, [20000, 8, 3, 3] 5.8, [125000, 2, 2, 2] 38; against 0.38 for [32, 128, 28, 28], 0.42 for [64, 512, 7, 7].
inline bool planar_tiles_pay(const void *x, int64_t B, int64_t C, int64_t HW) {
    const int64_t n = B * C * HW, tiles = planar_tiles(B, C, HW);
    return tiles <= 1024 + n / (planar_vec(x, HW) ? 2048 : 4096) || 8192 * tiles <= 3 * n;
}

// Many fp32 rows as fp16 row pairs in groups of eight, every group under a power of two s of its own: a workgroup
// of 1024 takes the group's 8 K values -- float4 number 1024 i + t to thread t, up to NQ of them in
// registers and all asked for at once (a single trip to memory; longer rows are read a second time) -- finds the
// largest finite |x|, and writes hi = fp16(s x) of row m to x16 row 16 (m / 8) + m % 8, lo = fp16(s x - hi) eight rows
// further on (rows past M of the last group: zeros) and 1 / s to group_scale[m / 8]. K a multiple of 4.
template <int NQ>
__global__ __launch_bounds__(1024) void split_groups_kernel(const float *__restrict__ x, int64_t M, int64_t K,
                                                            _Float16 *__restrict__ x16, float *__restrict__ group_scale) {
    __shared__ float lds[17];
    const int64_t g = blockIdx.x, q_row = K / 4, quads = 8 * q_row;              // float4s per row / per group
    const float *src = x + g * 8 * K;
    int64_t live = (M - g * 8) * q_row;                                            // float4s that exist
    if (live > quads) live = quads;
    const bool held = quads <= (int64_t)NQ * 1024;
    floatx4 q[NQ];
    float amax = 0.f;
    if (held) {
#pragma unroll
        for (int i = 0; i < NQ; i++) {
            const int64_t at = (int64_t)i * 1024 + threadIdx.x;
            q[i] = at < live ? __builtin_nontemporal_load(reinterpret_cast<const floatx4 *>(src) + at) : floatx4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int i = 0; i < NQ; i++)
            amax = fmaxf(fmaxf(amax, fmaxf(finite_abs(q[i][0]), finite_abs(q[i][1]))), fmaxf(finite_abs(q[i][2]), finite_abs(q[i][3])));
    } else {
        for (int64_t at = threadIdx.x; at < live; at += 1024) {
            const floatx4 v = *(reinterpret_cast<const floatx4 *>(src) + at);
            amax = fmaxf(fmaxf(amax, fmaxf(finite_abs(v[0]), finite_abs(v[1]))), fmaxf(finite_abs(v[2]), finite_abs(v[3])));
        }
    }
    amax = block_max(amax, lds);
    float s, inv;
    make_prescale(amax, s, inv);
    if (threadIdx.x == 0 && blockIdx.y == 0) group_scale[g] = inv;
    // gridDim.y workgroups (a power of two) share a group: each takes the whole group for the maximum -- one CU pulls
    // ~40 GB/s, and the idle CUs are free -- and converts every gridDim.y-th run of 1024 float4s
    const int share = gridDim.y - 1, mine = blockIdx.y;
    _Float16 *dst = x16 + g * 16 * K;                                              // the group's hi rows, then its lo rows
    auto emit = [&](int64_t at, floatx4 v) {
        v *= s;
        half4 h, l;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            h[e] = (_Float16)v[e];
            l[e] = (_Float16)(v[e] - (float)h[e]);
        }
        *reinterpret_cast<half4 *>(dst + 4 * at) = h;                              // row at / q_row of the group, same position
        *reinterpret_cast<half4 *>(dst + 8 * K + 4 * at) = l;
    };
    if (held) {
#pragma unroll
        for (int i = 0; i < NQ; i++) {
            const int64_t at = (int64_t)i * 1024 + threadIdx.x;
            if ((i & share) == mine && at < quads) emit(at, q[i]);
        }
    } else {
        for (int64_t at = (int64_t)mine * 1024 + threadIdx.x; at < quads; at += (int64_t)(share + 1) * 1024)
            emit(at, at < live ? *(reinterpret_cast<const floatx4 *>(src) + at) : floatx4{0.f, 0.f, 0.f, 0.f});
    }
}

}  // namespace

int launch_absmax(const float *x, int64_t n, float *partials, int vec, void *stream) {
    const int64_t per = vec ? 4096 : 8192;                 // 16 or 32 values per thread and round
    int64_t blocks = (n + per - 1) / per;
    if (blocks > kPartials) blocks = kPartials;
    if (vec)
        hipLaunchKernelGGL(absmax_wide_kernel, dim3((uint32_t)blocks), dim3(256), 0, as_stream(stream), x, n, partials);
    else
        hipLaunchKernelGGL(absmax_partial_kernel, dim3((uint32_t)blocks), dim3(256), 0, as_stream(stream), x, n, partials, 0);
    return (int)blocks;
}

// The same split for rows of any length and alignment, written as rows of Kp >= K values (Kp a multiple of 8) with
// zeros behind the K-th: one workgroup per group of eight rows, element-wise reads, one 16-byte piece of a hi row and
// of its lo row per thread and step. The second pass over the group's 32 K bytes comes from L2. With few groups,
// gridDim.y workgroups share one: each finds the group's maximum itself and writes every gridDim.y-th run of pieces.
// VEC: K is a multiple of 4 and x 16-byte aligned -- whole float4s, two per piece (K a multiple of 8: never across the end).
template <bool VEC>
__global__ __launch_bounds__(1024) void split_groups_padded_kernel(const float *__restrict__ x, int64_t M, int K, int Kp,
                                                                   FastDiv by_row, _Float16 *__restrict__ x16,
                                                                   float *__restrict__ group_scale) {
    __shared__ float lds[17];
    const int64_t g = blockIdx.x;
    const float *src = x + g * 8 * (int64_t)K;
    const int rows = M - g * 8 < 8 ? (int)(M - g * 8) : 8;
    float amax = 0.f;
    if constexpr (VEC) {
        for (int at = threadIdx.x; at < rows * (K / 4); at += 1024) {
            const floatx4 v = *(reinterpret_cast<const floatx4 *>(src) + at);
            amax = fmaxf(fmaxf(amax, fmaxf(finite_abs(v[0]), finite_abs(v[1]))), fmaxf(finite_abs(v[2]), finite_abs(v[3])));
        }
    } else {
        for (int at = threadIdx.x; at < rows * K; at += 1024) amax = fmaxf(amax, finite_abs(src[at]));
    }
    amax = block_max(amax, lds);
    float s, inv;
    make_prescale(amax, s, inv);
    if (threadIdx.x == 0 && blockIdx.y == 0) group_scale[g] = inv;
    _Float16 *dst = x16 + g * 16 * (int64_t)Kp;                    // the group's hi rows, then its lo rows
    const uint32_t pieces = 8u * (uint32_t)(Kp / 8);
    for (uint32_t p = blockIdx.y * 1024u + threadIdx.x; p < pieces; p += 1024u * gridDim.y) {
        int c;
        const int r = (int)by_row.divmod(p, c);
        const int k0 = c * 8;
        half8 h = {0, 0, 0, 0, 0, 0, 0, 0}, l = {0, 0, 0, 0, 0, 0, 0, 0};
        if (r < rows) {
            if constexpr (VEC) {
#pragma unroll
                for (int q = 0; q < 2; q++)
                    if (k0 + 4 * q < K) {
                        const floatx4 f = *reinterpret_cast<const floatx4 *>(src + (int64_t)r * K + k0 + 4 * q);
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const float v = s * f[e];
                            h[4 * q + e] = (_Float16)v;
                            l[4 * q + e] = (_Float16)(v - (float)h[4 * q + e]);
                        }
                    }
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (k0 + e < K) {
                        const float v = s * src[(int64_t)r * K + k0 + e];
                        h[e] = (_Float16)v;
                        l[e] = (_Float16)(v - (float)h[e]);
                    }
            }
        }
        *reinterpret_cast<half8 *>(dst + (int64_t)r * Kp + k0) = h;
        *reinterpret_cast<half8 *>(dst + (int64_t)(8 + r) * Kp + k0) = l;
    }
}

// x16: 16 ceil(M / 8) rows of Kp fp16 values (Kp >= K, a multiple of 8; zeros behind the K-th), 16-byte aligned;
// group_scale: ceil(M / 8) floats. Whole float4s of 16-byte aligned rows and Kp == K take the kernel above.
int launch_split_groups(const float *x, int64_t M, int64_t K, int64_t Kp, void *x16, float *group_scale, void *stream) {
    const int64_t groups = (M + 7) / 8, quads = 8 * (K / 4);
    if (groups > 0x7FFFFFFF) return TMQ_ERR_TOO_LARGE;
    if (Kp != K || K % 4 != 0 || !aligned16(x)) {
        if (8 * Kp > 0x7FFFFFFF) return TMQ_ERR_TOO_LARGE;
        // few groups: up to eight workgroups each (M = 17, K = 4000: 3 workgroups -> 12)
        const int64_t runs = (Kp + 1023) / 1024;
        const uint32_t share = groups > 64 ? 1 : (uint32_t)(runs < 1 ? 1 : runs > 8 ? 8 : runs);
        auto padded = K % 4 == 0 && aligned16(x) ? split_groups_padded_kernel<true> : split_groups_padded_kernel<false>;
        hipLaunchKernelGGL(padded, dim3((uint32_t)groups, share), dim3(1024), 0, as_stream(stream), x, M, (int)K,
                           (int)Kp, FastDiv((uint32_t)(Kp / 8)), static_cast<_Float16 *>(x16), group_scale);
        return check_launch();
    }
    auto kernel = quads <= 2 * 1024 ? split_groups_kernel<2> : quads <= 4 * 1024 ? split_groups_kernel<4>
                : quads <= 8 * 1024 ? split_groups_kernel<8> : split_groups_kernel<16>;
    // up to 64 groups share a group among up to four workgroups (M = 32 at K = 4096: 14.5 -> 13.4 us in all, M = 512
    // 42.4 -> 40.8; M = 1024, where the CUs are busy anyway, 62.0 -> 63.1)
    const uint32_t share = groups > 64 || quads <= 1024 ? 1 : quads <= 2048 ? 2 : 4;
    hipLaunchKernelGGL(kernel, dim3((uint32_t)groups, share), dim3(1024), 0, as_stream(stream), x, M, K,
                       static_cast<_Float16 *>(x16), group_scale);
    return check_launch();
}

// Rows of K fp16 values copied to rows of Kp >= K values (Kp a multiple of 8), zeros behind the K-th: a thread moves
// one 16-byte piece of the destination (vec: K % 8 == 0 and x 16-byte aligned, so the piece is one load as well).
__global__ __launch_bounds__(256) void pad_rows_kernel(const _Float16 *__restrict__ x, uint32_t pieces, int K, FastDiv by_row,
                                                       _Float16 *__restrict__ out, int vec) {
    const uint32_t id = blockIdx.x * 256u + threadIdx.x;
    if (id >= pieces) return;
    int c;
    const uint32_t m = by_row.divmod(id, c);
    const int k0 = c * 8;
    const _Float16 *src = x + (int64_t)m * K + k0;
    half8 v = {0, 0, 0, 0, 0, 0, 0, 0};
    if (vec) {
        if (k0 < K) v = *reinterpret_cast<const half8 *>(src);
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++)
            if (k0 + e < K) v[e] = src[e];
    }
    *reinterpret_cast<half8 *>(out + (int64_t)id * 8) = v;
}

// out: M rows of Kp fp16 values, 16-byte aligned; Kp % 8 == 0, M Kp < 2^31.
int launch_pad_rows(const void *x, int64_t M, int64_t K, int64_t Kp, void *out, void *stream) {
    const int64_t pieces = M * (Kp / 8);
    if (pieces <= 0 || pieces > 0x7FFFFFFF) return TMQ_ERR_TOO_LARGE;
    hipLaunchKernelGGL(pad_rows_kernel, dim3((uint32_t)((pieces + 255) / 256)), dim3(256), 0, as_stream(stream),
                       static_cast<const _Float16 *>(x), (uint32_t)pieces, (int)K, FastDiv((uint32_t)(Kp / 8)),
                       static_cast<_Float16 *>(out), (K % 8 == 0 && aligned16(x)) ? 1 : 0);
    return check_launch();
}

// x16: 2 M rows of Kp >= K fp16 values (Kp % 8 == 0, zeros behind the K-th), 16-byte aligned; row_scale: M floats.
int launch_split_rows(const float *x, int64_t M, int64_t K, int64_t Kp, int64_t group, void *x16, float *row_scale, void *stream) {
    hipLaunchKernelGGL(split_rows_kernel, dim3((uint32_t)M), dim3(1024), 0, as_stream(stream), x, K, Kp, (int)M, (int)group,
                       static_cast<_Float16 *>(x16), row_scale, (K % 4 == 0 && aligned16(x)) ? 1 : 0);
    return check_launch();
}

}  // namespace tmq

using namespace tmq;

extern "C" {

size_t tmq_f32_prescale_workspace_bytes(int64_t n) { return n > kSingleMax ? kPartials * sizeof(float) : 0; }

int tmq_f32_prescale(const float *x, int64_t n, float *prescale, float *xs, const float *scale_in, float *scale_out,
                     int64_t channels, void *workspace, void *stream) {
    if (n <= 0 || !x || !prescale || channels < 0 || (scale_out && channels == 0)) return TMQ_ERR_INVALID_ARG;
    const int vec = aligned16(x) && (!xs || aligned16(xs));
    if (n <= kSingleMax) {
        hipLaunchKernelGGL(prescale_single_kernel, dim3(1), dim3(1024), 0, as_stream(stream), x, n, prescale, xs, scale_in,
                           scale_out, channels, vec);
        return check_launch();
    }
    if (!workspace) return TMQ_ERR_INVALID_ARG;
    float *partials = static_cast<float *>(workspace);
    int64_t blocks = (n + 8191) / 8192;                    // 32 values per thread and more
    if (blocks > kPartials) blocks = kPartials;
    hipLaunchKernelGGL(absmax_partial_kernel, dim3((uint32_t)blocks), dim3(256), 0, as_stream(stream), x, n, partials,
                       (int)aligned16(x));
    int rc = check_launch();
    if (rc != TMQ_OK) return rc;
    hipLaunchKernelGGL(prescale_finalize_kernel, dim3(1), dim3(1024), 0, as_stream(stream), partials, (int)blocks, prescale,
                       scale_in, scale_out, channels);
    rc = check_launch();
    if (rc != TMQ_OK || !xs) return rc;
    const int64_t cblocks = (n + 1023) / 1024;
    if (cblocks > 0x7FFFFFFF) return TMQ_ERR_TOO_LARGE;
    hipLaunchKernelGGL(scale_copy_kernel, dim3((uint32_t)cblocks), dim3(256), 0, as_stream(stream), x, prescale, xs, n, vec);
    return check_launch();
}

int tmq_split_f32_scaled(const float *x, const float *prescale, void *hi, void *lo, int64_t n, void *stream) {
    if (n < 0 || (n > 0 && (!x || !hi))) return TMQ_ERR_INVALID_ARG;
    if (n == 0) return TMQ_OK;
    const int64_t blocks = (n + 2047) / 2048;
    if (blocks > 0x7FFFFFFF) return TMQ_ERR_TOO_LARGE;
    const int vec = aligned16(x) && aligned16(hi) && aligned16(lo);
    auto kernel = lo ? (prescale ? split_terms_kernel<true, true> : split_terms_kernel<true, false>)
                     : (prescale ? split_terms_kernel<false, true> : split_terms_kernel<false, false>);
    hipLaunchKernelGGL(kernel, dim3((uint32_t)blocks), dim3(256), 0, as_stream(stream), x, prescale,
                       static_cast<_Float16 *>(hi), static_cast<_Float16 *>(lo), n, vec);
    return check_launch();
}

size_t tmq_f32_to_f16_prescaled_workspace_bytes(int64_t n) { return n > 0 ? kPartials * sizeof(float) : 0; }

int tmq_f32_to_f16_prescaled(const float *x, int64_t n, float *prescale, void *hi, const float *scale_in, float *scale_out,
                             int64_t channels, void *workspace, void *stream) {
    if (n <= 0 || !x || !prescale || !hi || !workspace || channels < 0 || (scale_out && channels == 0)) return TMQ_ERR_INVALID_ARG;
    float *partials = static_cast<float *>(workspace);
    const int vec = aligned16(x) && (reinterpret_cast<uintptr_t>(hi) & 7u) == 0;
    const int blocks = launch_absmax(x, n, partials, vec, stream);
    if (int rc = check_launch()) return rc;
    const int64_t groups = (n + 8191) / 8192;
    if (groups > 0x7FFFFFFF) return TMQ_ERR_TOO_LARGE;
    hipLaunchKernelGGL(convert_prescaled_kernel, dim3((uint32_t)groups), dim3(256), 0, as_stream(stream), x, n, partials, blocks,
                       static_cast<_Float16 *>(hi), prescale, scale_in, scale_out, channels, vec);
    return check_launch();
}

int tmq_f32_nchw_to_f16_nhwc_pays(const float *x, int64_t B, int64_t C, int64_t HW) {
    return B > 0 && C > 0 && HW > 0 && planar_tiles_pay(x, B, C, HW) ? 1 : 0;
}

int tmq_f32_nchw_to_f16_nhwc_prescaled(const float *x, int64_t B, int64_t C, int64_t HW, float *prescale, void *hi,
                                       const float *scale_in, float *scale_out, int64_t channels, void *workspace, void *stream) {
    if (B <= 0 || C <= 0 || HW <= 0 || !x || !prescale || !hi || !workspace || channels < 0 || (scale_out && channels == 0))
        return TMQ_ERR_INVALID_ARG;
    float *partials = static_cast<float *>(workspace);
    const int CT = planar_tile_channels(C);
    const int64_t tiles_p = (HW + 4096 / CT - 1) / (4096 / CT), tiles_c = (C + CT - 1) / CT;
    if (tiles_p > 0x7FFFFFFF || tiles_c > 0x7FFFFFFF) return TMQ_ERR_TOO_LARGE;
    const int64_t tiles = planar_tiles(B, C, HW), groups = tiles < (1 << 20) ? tiles : (1 << 20);
    const int blocks = launch_absmax(x, B * C * HW, partials, (int)aligned16(x), stream);
    if (int rc = check_launch()) return rc;
    const int vec = planar_vec(x, HW);
    const uintptr_t at = reinterpret_cast<uintptr_t>(hi);
    const int piece = C % 8 == 0 && (at & 15u) == 0 ? 8 : C % 4 == 0 && (at & 7u) == 0 ? 4 : 1;
    auto kernel = CT == 16 ? convert_prescaled_nhwc_kernel<16> : CT == 32 ? convert_prescaled_nhwc_kernel<32> : convert_prescaled_nhwc_kernel<64>;
    hipLaunchKernelGGL(kernel, dim3((uint32_t)groups), dim3(256), 0, as_stream(stream), x, C, HW, (int)tiles_p,
                       (int)tiles_c, tiles, partials, blocks, static_cast<_Float16 *>(hi), prescale, scale_in, scale_out, channels, vec, piece);
    return check_launch();
}

int tmq_split_f32(const float *x, void *hi, void *lo, int64_t n, void *stream) {
    if (n > 0 && !lo) return TMQ_ERR_INVALID_ARG;
    return tmq_split_f32_scaled(x, nullptr, hi, lo, n, stream);
}

}  // extern "C"
