// Up to sixteen fp32 rows against a layer, split into fp16 terms inside the workgroup that multiplies them: one launch.
//
// fp32 rows travel through the fp16 matrix pipe as hi = fp16(s x), lo = fp16(s x - hi), s a power of two of the row's own
// (prescale.hip). Made by a launch of its own, in a workspace, the split costs more than the product it serves: a handful
// of short rows is a few thousand values, and a launch that does nothing takes 1.6 us. Here every workgroup of eight
// wavefronts asks for the rows and for all its weights at once, finds each row's largest finite |x|, writes both terms to
// LDS in operand order and multiplies; the reduction is dealt to the wavefronts in 64-index pairs and summed in their order.
//   * Rows: 8 / rows wavefronts a row (one for five to eight rows; two rows each beyond), eight consecutive values a lane.
//   * LDS: 16-byte chunk c of column j (hi of row j, lo of row j - 8; two sets of sixteen columns from nine rows on) sits at
//     position (j + c) % 16 of 256 bytes: both the writers, on neighbouring chunks, and the readers, on neighbouring
//     columns, meet every bank.
//   * Bound by the chain argument fetch -> rows -> maximum -> LDS -> product -> sum, about 2 us behind a launch's 1.6;
//     neither memory nor the matrix pipe is busy. 5 rows, 1000 -> 3000: 6.1 us in two launches
//     before, 3.7 so; 16 rows 9.6 in three, 4.8.
#include "common.h"
#include "mfma.h"
#include "range.h"

namespace tmq {
namespace {

typedef floatx4 floatx4_any __attribute__((aligned(4)));   // four floats at any float's address

struct Rows32 {
    const float *x;
    const uint32_t *native;
    const float *scale, *bias;
    const void *residual;
    void *y;
    int32_t M, K, N, Nb, Kb, pairs;
    int32_t relu, y_f16, vec;            // vec: whole quads of results and constants
};

// v_max with a lane `ctrl` (a DPP control) away, in rows of sixteen lanes
template <int ctrl>
__device__ __forceinline__ float max_dpp(float v) {
    return fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xF, 0xF, false)));
}
// maximum over the wavefront, uniform
__device__ __forceinline__ float wave_max_uniform(float v) {
    v = max_dpp<0xB1>(v);                  // quad_perm [1,0,3,2]
    v = max_dpp<0x4E>(v);                  // quad_perm [2,3,0,1]
    v = max_dpp<0x141>(v);                 // row_half_mirror
    v = max_dpp<0x140>(v);                 // row_mirror
    const int i = __builtin_bit_cast(int, v);
    return fmaxf(fmaxf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(i, 0)), __builtin_bit_cast(float, __builtin_amdgcn_readlane(i, 16))),
                 fmaxf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(i, 32)), __builtin_bit_cast(float, __builtin_amdgcn_readlane(i, 48))));
}

// SETS: sets of sixteen columns (1: up to 8 rows, 2: up to 16). WN: 16-channel blocks per workgroup. NP: pairs per
// wavefront at most. NC: chunks of eight values a lane holds of a row.
template <int SETS, int WN, int NP, int NC>
__global__ __launch_bounds__(512) void rows32_kernel(const Rows32 a) {
    constexpr int kChunk = SETS * 256;     // bytes of a chunk's columns
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    __shared__ float row_max[16], row_inv[16];
    // every kernel argument is asked for here, in one go
    asm volatile("" ::"s"(a.x), "s"(a.native), "s"(a.scale), "s"(a.bias), "s"(a.residual), "s"(a.y), "s"(a.M), "s"(a.K), "s"(a.N), "s"(a.Nb),
                 "s"(a.Kb), "s"(a.pairs), "s"(a.relu), "s"(a.y_f16), "s"(a.vec));
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, g = lane >> 4, n0 = blockIdx.x * (16 * WN);

    // the rows: `share` wavefronts a row, chunk part * 64 + lane + i * 64 * share
    const int shift = a.M <= 1 ? 3 : a.M <= 2 ? 2 : a.M <= 4 ? 1 : 0, share = 1 << shift, part = wv & (share - 1);
    const int chunks = a.pairs * 8;
    floatx4 v[SETS][NC][2];
#pragma unroll
    for (int r = 0; r < SETS; r++) {
        const int row = (wv >> shift) + 8 * r;
        if (row >= a.M) continue;
        const float *src = a.x + (int64_t)row * a.K;
#pragma unroll
        for (int i = 0; i < NC; i++) {
            const int k = ((i * share + part) * 64 + lane) * 8;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                floatx4 q = {0.f, 0.f, 0.f, 0.f};
                const int left = a.K - k - 4 * h;
                if (left >= 4) {
                    q = *reinterpret_cast<const floatx4_any *>(src + k + 4 * h);
                } else if (left > 0) {
#pragma unroll
                    for (int e = 0; e < 3; e++)
                        if (e < left) q[e] = src[k + 4 * h + e];
                }
                v[r][i][h] = q;
            }
        }
    }
    // the weights: pairs wv, wv + 8, ...; past the last one it again, never multiplied
    uint32_t w[NP][WN];
#pragma unroll
    for (int nj = 0; nj < WN; nj++) {
        int nb = n0 / 16 + nj;
        if (nb >= a.Nb) nb = a.Nb - 1;                              // finite bits, never stored
        const uint32_t *block = a.native + (int64_t)nb * a.Kb * 256 + lane * 4;
#pragma unroll
        for (int p = 0; p < NP; p++) {
            int pi = wv + 8 * p;
            if (pi >= a.pairs) pi = a.pairs - 1;
            w[p][nj] = block[(pi >> 2) * 256 + (pi & 3)];
        }
    }

    float amax[SETS];
#pragma unroll
    for (int r = 0; r < SETS; r++) {
        float m = 0.f;
        if ((wv >> shift) + 8 * r < a.M) {
#pragma unroll
            for (int i = 0; i < NC; i++)
#pragma unroll
                for (int h = 0; h < 2; h++)
#pragma unroll
                    for (int e = 0; e < 4; e++) m = fmaxf(m, finite_abs(v[r][i][h][e]));
        }
        amax[r] = wave_max_uniform(m);
    }
    if (share > 1) {                                                // (uniform; rows shared by wavefronts are at most four, SETS is 1)
        if (lane == 0) row_max[wv] = amax[0];
        __syncthreads();
        for (int q = 0; q < share; q++) amax[0] = fmaxf(amax[0], row_max[wv - part + q]);
    }
#pragma unroll
    for (int r = 0; r < SETS; r++) {
        const int row = (wv >> shift) + 8 * r;
        if (row >= a.M) continue;
        float s, inv;
        make_prescale(amax[r], s, inv);
        if (lane == 0 && part == 0) row_inv[row] = inv;
#pragma unroll
        for (int i = 0; i < NC; i++) {
            const int c = (i * share + part) * 64 + lane;
            half8 hi, lo;
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float f = v[r][i][h][e] * s;
                    hi[4 * h + e] = (_Float16)f;
                    lo[4 * h + e] = (_Float16)(f - (float)hi[4 * h + e]);
                }
            if (c < chunks) {
                unsigned char *at = lds + c * kChunk;
                // one set: lo in columns 8 .. 15; two: in the second set
                *reinterpret_cast<half8 *>(at + ((row + c) & 15) * 16) = hi;
                *reinterpret_cast<half8 *>(at + (SETS - 1) * 256 + ((row + (SETS == 1 ? 8 : 0) + c) & 15) * 16) = lo;
            }
        }
    }
    __syncthreads();

    floatx4 acc[WN][SETS];
#pragma unroll
    for (int nj = 0; nj < WN; nj++)
#pragma unroll
        for (int t = 0; t < SETS; t++) acc[nj][t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const int pi = wv + 8 * p;
        if (pi >= a.pairs) break;
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const int c = pi * 8 + 4 * s + g;
            half8 b[SETS];
#pragma unroll
            for (int t = 0; t < SETS; t++) b[t] = *reinterpret_cast<const half8 *>(lds + c * kChunk + t * 256 + ((j + c) & 15) * 16);
#pragma unroll
            for (int nj = 0; nj < WN; nj++) {
                const half8 wd = decode_step(w[p][nj], s);
#pragma unroll
                for (int t = 0; t < SETS; t++) acc[nj][t] = mfma16(wd, b[t], acc[nj][t]);
            }
        }
    }

    // sums over the wavefronts: a lane's accumulators are channels 16 nj + 4 g .. + 3 of column j
    __syncthreads();                                                // the operands have been read out
    floatx4 *const park = reinterpret_cast<floatx4 *>(lds);
#pragma unroll
    for (int nj = 0; nj < WN; nj++)
#pragma unroll
        for (int t = 0; t < SETS; t++) park[((wv * WN + nj) * SETS + t) * 64 + lane] = acc[nj][t];
    __syncthreads();
    for (int q = tid; q < a.M * 4 * WN; q += 512) {
        const int c4 = q % (4 * WN), row = q / (4 * WN), nj = c4 >> 2, from = (c4 & 3) * 16;
        const int n = n0 + c4 * 4;
        if (n >= a.N) continue;
        auto sums = [&](int t, int col) {
            floatx4 f = park[(nj * SETS + t) * 64 + from + col];
#pragma unroll
            for (int k = 1; k < 8; k++) f += park[((k * WN + nj) * SETS + t) * 64 + from + col];
            return f;
        };
        floatx4 f = (sums(0, row) + (SETS == 1 ? sums(0, row + 8) : sums(SETS - 1, row))) * (row_inv[row] * (1.0f / kWeightUnit));
        const int64_t o = (int64_t)row * a.N + n;
        if (a.vec) {
            if (a.scale) f *= *reinterpret_cast<const floatx4 *>(a.scale + n);
            if (a.bias) f += *reinterpret_cast<const floatx4 *>(a.bias + n);
            if (a.residual) {
                if (a.y_f16) {
                    const half4 r = *reinterpret_cast<const half4 *>(static_cast<const _Float16 *>(a.residual) + o);
#pragma unroll
                    for (int e = 0; e < 4; e++) f[e] += (float)r[e];
                } else {
                    f += *reinterpret_cast<const floatx4 *>(static_cast<const float *>(a.residual) + o);
                }
            }
            if (a.relu) {
#pragma unroll
                for (int e = 0; e < 4; e++) f[e] = f[e] < 0.f ? 0.f : f[e];
            }
            if (a.y_f16) *reinterpret_cast<half4 *>(static_cast<_Float16 *>(a.y) + o) = half4{(_Float16)f[0], (_Float16)f[1], (_Float16)f[2], (_Float16)f[3]};
            else *reinterpret_cast<floatx4 *>(static_cast<float *>(a.y) + o) = f;
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (n + e >= a.N) break;
                float t = f[e];
                if (a.scale) t *= a.scale[n + e];
                if (a.bias) t += a.bias[n + e];
                if (a.residual) t += a.y_f16 ? (float)static_cast<const _Float16 *>(a.residual)[o + e] : static_cast<const float *>(a.residual)[o + e];
                if (a.relu) t = t < 0.f ? 0.f : t;
                if (a.y_f16) static_cast<_Float16 *>(a.y)[o + e] = (_Float16)t;
                else static_cast<float *>(a.y)[o + e] = t;
            }
        }
    }
}

template <int SETS, int WN, int NP, int NC>
int launch(const Rows32 &a, void *stream) {
    const size_t rows = (size_t)a.pairs * 8 * SETS * 256, park = (size_t)8 * WN * SETS * 1024, bytes = rows > park ? rows : park;
    auto kernel = rows32_kernel<SETS, WN, NP, NC>;
    if (bytes > 48 * 1024) {
        if (int st = allow_dynamic_lds(reinterpret_cast<const void *>(kernel), bytes)) return st;
    }
    hipLaunchKernelGGL(kernel, dim3((uint32_t)((a.N + 16 * WN - 1) / (16 * WN))), dim3(512), bytes, as_stream(stream), a);
    return check_launch();
}

template <int SETS, int WN>
int by_pairs(const Rows32 &a, void *stream) {
    if (a.pairs <= 8) return launch<SETS, WN, 1, 1>(a, stream);
    if (a.pairs <= 16) return launch<SETS, WN, 2, 2>(a, stream);
    if constexpr (SETS == 1 && WN == 1)                        // (rows32_ok: more than 2048 values, at most 4096 channels)
        if (a.pairs > 32) return launch<SETS, WN, 8, 8>(a, stream);
    return launch<SETS, WN, 4, 4>(a, stream);
}

// One pass of workgroups over the CUs where that can be had: every workgroup prepares all the rows, whatever it multiplies.
// 600 shapes of up to 32768 columns: within 2 % of the best width on average.
template <int SETS>
int by_width(const Rows32 &a, void *stream) {
    const int blocks = a.Nb;
    if (blocks <= 256) return by_pairs<SETS, 1>(a, stream);
    if (blocks <= 512) return by_pairs<SETS, 2>(a, stream);
    if (blocks <= 1024) return by_pairs<SETS, 4>(a, stream);
    return by_pairs<SETS, 8>(a, stream);
}

}  // namespace

// Which rows the launch that multiplies them can split. The terms of the rows have to fit LDS (32 bytes an index, 64 from
// nine rows on), and every workgroup prepares them again, which wide layers over long rows pay for: against the split in a
// launch of its own, 600 shapes, 0.85 of its time at the median of 1 .. 8 rows and 0.5 of 9 .. 16 inside these lines, 1.08 .. 1.65
// beyond (2304 x 25768, 6 rows 10.6 -> 14.0 us). 16 rows x 512 -> 512: 9.2 -> 3.5 us; 8 rows x 2048 -> 2048 6.5 -> 4.6; 3 rows x
// 4096 -> 4096 7.2 -> 6.3.
bool rows32_ok(const void *x, int64_t M, int64_t K, int64_t N) {
    if (M < 1 || M > 16 || K < 1 || N < 1 || !aligned16(x)) return false;
    if (M > 8) return K <= 2048 && K * N <= (int64_t)1 << 25;
    return K <= 2048 ? K * N <= (int64_t)3 << 23 : K <= 4096 && N <= 4096;
}

// Where that is also the faster way for a caller with a workspace. The widest layers pay for the repeated preparation with rows
// of any length, from the second round of workgroups on (their sums leave room for one a CU). Against the split of its own, 360
// shapes of 12000 columns and more: up to 32768 columns 0.42 .. 0.90 for 9 .. 16 rows, beyond 0.81 .. 0.95 for up to 12 short ones
// to 65536 and 0.93 .. 1.36 for the others (16 rows x 40 -> 338116 65.6 -> 84.4 us); 5 .. 8 rows 0.50 .. 0.99 to 131072 columns and
// to 32768 for more than 512 values, 0.79 .. 1.05 from there on; fewer rows 0.40 .. 0.85 at any width. More than 1024 values
// against more than 16384 columns 1.04 .. 1.12 from three rows on. (Inside all lines 1.03 at most.)
bool rows32_pays(const void *x, int64_t M, int64_t K, int64_t N) {
    if (!rows32_ok(x, M, K, N)) return false;
    if (M > 8) return N <= 32768 || (M <= 12 && N <= 65536 && K <= 512);
    return !((M > 4 && N > (K > 512 ? 32768 : 131072)) || (M > 2 && K > 1024 && N > 16384));
}

int launch_rows32(const void *x, int64_t M, int64_t K, const void *native, int64_t N, const float *scale, const float *bias,
                  const void *residual, int relu, void *y, int y_f16, void *stream) {
    Rows32 a{};
    a.x = static_cast<const float *>(x);
    a.native = static_cast<const uint32_t *>(native);
    a.scale = scale;
    a.bias = bias;
    a.residual = residual;
    a.y = y;
    a.M = (int32_t)M;
    a.K = (int32_t)K;
    a.N = (int32_t)N;
    a.Nb = (int32_t)native_blocks_n(N);
    a.Kb = (int32_t)native_blocks_k(K);
    a.pairs = (int32_t)((K + 63) / 64);
    a.relu = relu;
    a.y_f16 = y_f16;
    a.vec = N % 4 == 0 && aligned16(scale) && aligned16(bias) && aligned16(residual) && aligned16(y) ? 1 : 0;
    return M > 8 ? by_width<2>(a, stream) : by_width<1>(a, stream);
}

}  // namespace tmq
