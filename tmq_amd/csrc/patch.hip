// Stride-1 ternary convolutions over 256 or 512 channels out of input patches in LDS, one round of workgroups, for gfx950.
//
// The im2col kernels (gemm.hip, mid.hip) fetch an input pixel once per filter tap and column tile through L1, and a wavefront
// of theirs expands every weight for 64 rows. Here a workgroup fetches the input its output pixels' windows cover once, and a
// wavefront multiplies a unit of 112 pixels (7 fragments of 16) x 64 channels over ONE 64-channel slab of the input, all taps:
// the workgroup's wavefronts split the slabs (four or eight) and sum through LDS.
//   * Patch: the padded images as one run of positions (one row / column of padding serves the end of a row and the start of
//     the next), so consecutive outputs' windows are one contiguous piece and a tap is a constant distance in it. A pixel's slab
//     is 128 bytes in a pitch of 144: linear addresses that still spread sixteen pixels over all banks. Pixels go global ->
//     LDS directly, seven an instruction; padding is written as zeros.
//   * Per 56 MFMAs: 14 operand reads (seven ahead), 60 vector instructions of weight expansion, 14 of addresses -- 1.5 an
//     MFMA where a SIMD hides 2.4 (the 64 x 64 tiles issue 4 to 8).
//   * Weights are the MFMA's first operand: a lane's accumulators are channels of one pixel and go to memory without a
//     transpose, in 64-byte runs per pixel.
//   * Everybody fetches, multiplies and stores at the same time, so a second round would add both ends again: worth it for one
//     round that fills the chip. Clock stamps for 256 -> 256 on 14 x 14, batch 64, us: patch in LDS at 3.3, products 11.0 (1.87
//     GHz, MFMAs 80 % of the time), sums and stores 3.4.
// Batch 64, 3 x 3, us: 256 -> 256 on 14 x 14 20.1 -> 17.8; 512 -> 512 on 7 x 7 23.1 -> 18.6 (25.0 -> 19.8 on another machine).
#include "common.h"
#include "mfma.h"
#include "tile_epilogue.h"
#include <utility>

namespace tmq {
namespace {

constexpr int kSlab = 64;                 // channels per slab
constexpr int kPixelBytes = 144;          // a patch pixel in LDS: 64 fp16 channels and 16 bytes of pitch
constexpr int kFragments = 7;             // fragments of 16 pixels a wavefront multiplies
constexpr int kJobPixels = 7;             // pixels a wavefront fetches with one instruction (7 x 9 chunks of 16 bytes <= 64 lanes)

struct PatchConv {
    const _Float16 *x;
    const uint32_t *native;
    int32_t Kb, Nb, M, N, C, H, W, B;
    int32_t py, px, Hp, Wp;                // the padded image
    int32_t ky, kx, dy, dx, reach;         // reach: largest distance of a tap
    int32_t pixels;                        // pixels of a patch, an upper bound over all workgroups
    int32_t rows;                          // output pixels of a workgroup, at most 112
    uint32_t x_bytes;
    int32_t du, dv;                        // sixteen results further on: rows and columns of the grid
    FastDiv by_tiles_n, by_w, by_h, by_wp, by_hp;   // the grid of results, the padded image
    int32_t jobs;                          // per image row
};

template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N_, class F>
__device__ __forceinline__ void static_for(F &&f) {
    static_for_impl(f, std::make_integer_sequence<int, N_>{});
}

typedef float float2v __attribute__((ext_vector_type(2)));

// Eight channels of a lane, half h of its sixteen: n0 + 32 h + 8 g .. + 7 for fp16 results (one 16-byte piece), n0 + 32 h +
// 4 g .. + 3 and 16 further for fp32 ones; the four lanes of a pixel write 64 contiguous bytes either way.
template <bool F16>
struct LaneChannels {
    static constexpr int kElt = F16 ? 2 : 4, kGap = F16 ? 4 : 16;   // bytes a value; channels from the first four to the other four
    int c;                                 // the first of them
    floatx4 sc[2], bi[2];
    __device__ __forceinline__ void init(const Epilogue &ep, int N, int n0, int g, int h) {
        c = n0 + 32 * h + (F16 ? 8 : 4) * g;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            sc[q] = floatx4{1.f, 1.f, 1.f, 1.f};
            bi[q] = floatx4{0.f, 0.f, 0.f, 0.f};
            if (c + q * kGap < N) {
                if (ep.scale) sc[q] = *reinterpret_cast<const floatx4 *>(ep.scale + c + q * kGap);
                if (ep.bias) bi[q] = *reinterpret_cast<const floatx4 *>(ep.bias + c + q * kGap);
            }
            sc[q] *= 1.0f / kWeightUnit;
        }
    }
};

// Where a pixel's results start, in bytes of y; kNone: the lane stores none.
constexpr uint32_t kNone = 0xFFFFFFFFu;

// The residual of those channels of one pixel.
struct Residual {
    u32x4 r[2];
    template <bool F16>
    __device__ __forceinline__ void request(const Epilogue &ep, const LaneChannels<F16> &ch, int N, uint32_t o) {
        if (o == kNone) return;
        const unsigned char *base = static_cast<const unsigned char *>(ep.residual);
#pragma unroll
        for (int q = 0; q < (F16 ? 1 : 2); q++)
            if (ch.c + q * ch.kGap < N) r[q] = *reinterpret_cast<const u32x4 *>(base + (o + (uint32_t)(ch.c + q * ch.kGap) * ch.kElt));
    }
};

template <bool F16>
__device__ __forceinline__ void store_channels(const float (&acc)[8], const LaneChannels<F16> &ch, const Residual &rs, const Epilogue &ep, int N,
                                               uint32_t o) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = __builtin_fmaf(acc[e], ch.sc[e >> 2][e & 3], ch.bi[e >> 2][e & 3]);
    if (ep.residual) {
        [[maybe_unused]] const floatx4 f[2] = {__builtin_bit_cast(floatx4, rs.r[0]), __builtin_bit_cast(floatx4, rs.r[1])};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if constexpr (F16) {
                v[2 * e] = add_half_lo(rs.r[0][e], v[2 * e]);
                v[2 * e + 1] = add_half_hi(rs.r[0][e], v[2 * e + 1]);
            } else {
                v[e] += f[0][e];
                v[4 + e] += f[1][e];
            }
        }
    }
    if (ep.relu) {
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = v[e] < 0.f ? 0.f : v[e];
    }
    unsigned char *base = static_cast<unsigned char *>(ep.y);
    if constexpr (F16) {
        half8 out;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const half2v p = __builtin_convertvector(float2v{v[2 * e], v[2 * e + 1]}, half2v);
            out[2 * e] = p[0];
            out[2 * e + 1] = p[1];
        }
        if (o != kNone && ch.c < N) *reinterpret_cast<half8 *>(base + (o + (uint32_t)ch.c * 2)) = out;
    } else {
#pragma unroll
        for (int q = 0; q < 2; q++)
            if (o != kNone && ch.c + q * ch.kGap < N)
                __builtin_nontemporal_store(floatx4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]},
                                            reinterpret_cast<floatx4 *>(base + (o + (uint32_t)(ch.c + q * ch.kGap) * 4)));
    }
}

template <int CG, int SG, bool F16>
__global__ __launch_bounds__(64 * CG * SG, 2) void patch_conv_kernel(PatchConv cv, Epilogue ep) {
    constexpr int WM = kFragments, WN = 4, WG = CG * SG, T = 64 * WG, NQ = 2 * WM, kAhead = WM;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int id = xcd_contiguous(blockIdx.x, gridDim.x);
    int tn;
    const int tm = (int)cv.by_tiles_n.divmod((uint32_t)id, tn);
    const int m0 = tm * cv.rows, m1 = m0 + cv.rows < cv.M ? m0 + cv.rows : cv.M;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int sg = wv % SG, n0 = (tn * CG + wv / SG) * 64;
    const int r16 = lane & 15, g = lane >> 4;
    constexpr int slabs = SG;               // a wavefront's unit is one slab
    const int taps = cv.ky * cv.kx, patch_bytes = cv.pixels * kPixelBytes;

    struct Place { int b, u, v; };          // image, row and column of a result in the grid
    auto place = [&](int m) {
        Place p;
        const uint32_t t = cv.by_w.divmod((uint32_t)m, p.v);
        p.b = (int)cv.by_h.divmod(t, p.u);
        return p;
    };
    auto padded = [&](const Place &p) { return (p.b * cv.Hp + p.u) * cv.Wp + p.v; };   // its position in the padded image
    const int start = __builtin_amdgcn_readfirstlane(padded(place(m0)));
    const int end = __builtin_amdgcn_readfirstlane(padded(place(m1 - 1))) + cv.reach + 1;

    // the patch: rows pr0 .. of the padded image stack, the columns in front of `start` and from `end` on left out
    {
        const BufferResource xr = make_buffer_resource(cv.x, cv.x_bytes);
        int c_first, c_last, ph0;
        const int pr0 = (int)cv.by_wp.divmod((uint32_t)start, c_first), pr1 = (int)cv.by_wp.divmod((uint32_t)(end - 1), c_last);
        int b = (int)cv.by_hp.divmod((uint32_t)pr0, ph0);
        const int lane_px = (lane * 57) >> 9, lane_part = lane - lane_px * 9;        // lane / 9, lane % 9
        const uint32_t lane_off = (uint32_t)(lane_px * cv.C * 2 + lane_part * 16);
        const bool lane_on = lane_part < 8 && lane < 63;
        int row = pr0, ih = ph0 - cv.py, jj = wv;
        for (;;) {
            while (jj >= cv.jobs) {                               // this wavefront's next job is in the next row
                jj -= cv.jobs;
                row++;
                if (++ih == cv.Hp - cv.py) {
                    ih = -cv.py;
                    b++;
                }
            }
            if (row > pr1 || b >= cv.B) break;
            // real columns of this row inside the patch, from this job's seven on
            int a = (row == pr0 ? c_first : 0) - cv.px, e = (row == pr1 ? c_last + 1 : cv.Wp) - cv.px;
            a = (a < 0 ? 0 : a) + jj * kJobPixels;
            e = e > cv.W ? cv.W : e;
            if ((unsigned)ih < (unsigned)cv.H && a < e) {
                const uint32_t base = (uint32_t)((b * cv.H + ih) * cv.W + a) * (uint32_t)cv.C * 2u + lane_off;
                unsigned char *dst = lds + (row * cv.Wp + a + cv.px - start) * kPixelBytes;
                if (lane_on && lane_px < e - a)
                    for (int s = 0; s < slabs; s++) buffer_to_lds(xr, base + (uint32_t)(s * 2 * kSlab), dst + s * patch_bytes);
            }
            jj += WG;
        }
    }

    // weights: a lane's dword of (tap, slab) for its row of fragment j
    uint32_t woff[WN];
#pragma unroll
    for (int j = 0; j < WN; j++) {
        const int c = F16 ? (r16 & 2) * 16 + (r16 >> 2) * 8 + (r16 & 1) * 4 + j : j * 16 + r16;   // channel of the wavefront's 64
        int nb = n0 / 16 + (c >> 4);
        if (nb >= cv.Nb) nb = cv.Nb - 1;                          // finite bits, never stored
        woff[j] = (uint32_t)(nb * cv.Kb) * 1024u + (uint32_t)((c & 15) + 16 * g) * 16u;
    }
    const unsigned char *native = reinterpret_cast<const unsigned char *>(cv.native);
    auto load_w = [&](u32x4 &w, int kt) {
        const unsigned char *at = native + ((uint32_t)(kt >> 2) * 1024u + (uint32_t)(kt & 3) * 4u);
#pragma unroll
        for (int j = 0; j < WN; j++) w[j] = *reinterpret_cast<const uint32_t *>(at + woff[j]);
    };
    u32x4 w, wnext;
    load_w(w, sg);

    // padding of the patch: zeros
    for (int p = tid; p < end - start; p += T) {
        int pw, phr;
        const uint32_t row = cv.by_wp.divmod((uint32_t)(start + p), pw);
        const int b = (int)cv.by_hp.divmod(row, phr);
        const bool in = (b < cv.B) & ((unsigned)(phr - cv.py) < (unsigned)cv.H) & ((unsigned)(pw - cv.px) < (unsigned)cv.W);
        if (!in)
            for (int s = 0; s < slabs; s++)
#pragma unroll
                for (int c = 0; c < 8; c++) *reinterpret_cast<u32x4 *>(lds + s * patch_bytes + p * kPixelBytes + c * 16) = u32x4{0u, 0u, 0u, 0u};
    }

    floatx4 acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; i++)
#pragma unroll
        for (int j = 0; j < WN; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    const int alive = m1 - m0 - r16;          // row fragment i has a result for this lane if 16 i < alive
    auto sixteen_on = [&](Place &p) {
        p.v += cv.dv;
        p.u += cv.du;
        const bool row = p.v >= (int)cv.by_w.d;
        p.v -= row ? (int)cv.by_w.d : 0;
        p.u += row ? 1 : 0;
        const bool image = p.u >= (int)cv.by_h.d;
        p.u -= image ? (int)cv.by_h.d : 0;
        p.b += image ? 1 : 0;
    };
    uint32_t arow[WM];                     // LDS offset of the lane's operand bytes, tap (0, 0), slab 0
    const int first = m0 + r16 < cv.M ? m0 + r16 : cv.M - 1;
    {
        Place p = place(first);
#pragma unroll
        for (int i = 0; i < WM; i++) {
            const int at = 16 * i < alive ? padded(p) - start : 0;
            arow[i] = (uint32_t)((at) * kPixelBytes + g * 16);
            sixteen_on(p);
        }
    }
    auto load_a = [&](int q, uint32_t off) { return *reinterpret_cast<const half8 *>(lds + arow[q % WM] + off + (q / WM) * 64); };

    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);

    {
        half8 a[kAhead], b0[WN], b1[WN];
        // a step is one tap of the wavefront's slab; `at` walks them one ahead of the multiplication
        struct Step { int ti, tj; } at{0, 0};
        auto advance = [&](int step) {                            // to the step behind `step`; the last one stays
            if (step + 1 >= taps) return;
            if (++at.tj == cv.kx) {
                at.tj = 0;
                ++at.ti;
            }
        };
        auto distance = [&] { return (uint32_t)(sg * patch_bytes + (at.ti * cv.dy * cv.Wp + at.tj * cv.dx) * kPixelBytes); };
        uint32_t off = distance(), noff;
        advance(0);
        noff = distance();
#pragma unroll
        for (int q = 0; q < kAhead; q++) a[q] = load_a(q, off);
#pragma unroll
        for (int j = 0; j < WN; j++) b0[j] = decode_step(w[j], 0);
        for (int step = 0; step < taps; step++) {
            load_w(wnext, (at.ti * cv.kx + at.tj) * slabs + sg);
            advance(step + 1);
            const uint32_t noff2 = distance();
            __builtin_amdgcn_sched_barrier(0);
            static_for<NQ>([&](auto qc) {
                constexpr int Q = decltype(qc)::value, fi = Q % WM, fs = Q / WM;
#pragma unroll
                for (int j = 0; j < WN; j++) acc[fi][j] = mfma16(fs == 0 ? b0[j] : b1[j], a[Q % kAhead], acc[fi][j]);
                constexpr int R = (Q + kAhead) % NQ;
                a[Q % kAhead] = load_a(R, Q + kAhead < NQ ? off : noff);
                if constexpr (fs == 0 && fi < WN) b1[fi] = decode_step(w[fi], 1);
                if constexpr (fs == 1 && fi >= WM - WN) b0[fi - (WM - WN)] = decode_step(wnext[fi - (WM - WN)], 0);
#pragma unroll
                for (int j = 0; j < WN; j++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);       // MFMA
                    __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);       // VALU
                }
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);           // DS read
                __builtin_amdgcn_sched_barrier(0);
            });
            w = wnext;
            off = noff;
            noff = noff2;
        }
    }

    uint32_t out[WM];                       // byte of y where the pixel of row fragment i starts
    {
        const uint32_t pixel = (uint32_t)cv.N * (F16 ? 2u : 4u);
#pragma unroll
        for (int i = 0; i < WM; i++) out[i] = 16 * i < alive ? (uint32_t)(first + 16 * i) * pixel : kNone;
    }
    // channels of half h of a lane's accumulators (LaneChannels)
    auto half_of = [&](const floatx4 (&a)[WN], int h, float (&v)[8]) {
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = F16 ? a[e & 3][2 * h + (e >> 2)] : a[2 * h + (e >> 2)][e & 3];
    };
    {
        // Partial tiles through LDS, up to four row fragments of every wavefront at a time; fragment i is added up, in slab
        // order, by the wavefront of slab group i % SG.
        constexpr int kFrags = 4, kOwn = (WM + SG - 1) / SG;
        LaneChannels<F16> ch[2];
        Residual rs[kOwn][2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            ch[h].init(ep, cv.N, n0, g, h);
            if (ep.residual) {
#pragma unroll
                for (int i = 0; i < WM; i++)
                    if (i % SG == sg) rs[i / SG][h].request(ep, ch[h], cv.N, out[i]);
            }
        }
        floatx4 *const park = reinterpret_cast<floatx4 *>(lds);
        auto slot = [&](int wave, int i, int j) { return ((wave * kFrags + i) * WN + j) * 64 + lane; };
        static_for<(WM + kFrags - 1) / kFrags>([&](auto pc) {
            constexpr int I0 = decltype(pc)::value * kFrags, I1 = I0 + kFrags < WM ? I0 + kFrags : WM;
            lds_barrier();
#pragma unroll
            for (int i = I0; i < I1; i++)
                if (i % SG != sg) {
#pragma unroll
                    for (int j = 0; j < WN; j++) park[slot(wv, i - I0, j)] = acc[i][j];
                }
            lds_barrier();
#pragma unroll
            for (int i = I0; i < I1; i++)
                if (i % SG == sg) {
                    floatx4 sum[WN];
#pragma unroll
                    for (int j = 0; j < WN; j++) sum[j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
                    for (int s = 0; s < SG; s++) {
                        if (s == sg) {
#pragma unroll
                            for (int j = 0; j < WN; j++) sum[j] += acc[i][j];
                        } else {
#pragma unroll
                            for (int j = 0; j < WN; j++) sum[j] += park[slot(wv - sg + s, i - I0, j)];
                        }
                    }
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        float v[8];
                        half_of(sum, h, v);
                        store_channels(v, ch[h], rs[i / SG][h], ep, cv.N, out[i]);
                    }
                }
        });
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);
}

int64_t gcd(int64_t a, int64_t b) { return b ? gcd(b, a % b) : a; }

// Positions of the padded image that `rows` consecutive outputs of an h x w grid can span, from any multiple of `rows` on:
// each crossing of a row of the grid adds Wp - w, each crossing of an image (Hp - h) Wp; and a tap's reach.
int64_t patch_pixels(int64_t rows, int64_t h, int64_t w, int64_t Hp, int64_t Wp, int64_t reach) {
    auto crossings = [&](int64_t n) { return (n - gcd(rows, n) + rows - 1) / n; };
    return rows + crossings(w) * (Wp - w) + crossings(h * w) * (Hp - h) * Wp + reach;
}

template <int CG, int SG, bool F16>
int launch(PatchConv cv, const Epilogue &ep, int64_t bytes, int64_t groups, void *stream) {
    auto kernel = patch_conv_kernel<CG, SG, F16>;
    if (int st = allow_dynamic_lds(reinterpret_cast<const void *>(kernel), (size_t)bytes)) return st;
    hipLaunchKernelGGL(kernel, dim3((uint32_t)groups), dim3(64 * CG * SG), (uint32_t)bytes, as_stream(stream), cv, ep);
    return check_launch();
}

struct PatchPlan {
    int slabs, columns;                    // 64-channel slabs; column groups of 64 in a workgroup
    int64_t Hp, Wp, reach;                 // the padded image and the largest distance of a tap: any padding and dilation comes here
    int64_t rows, groups, pixels, bytes;   // output pixels and LDS of a workgroup, workgroups
};

// Whether the convolution is one well-filled round of units, and how it is cut. Workgroups of eight wavefronts, one a CU (256
// channels to at most 64 outputs: four wavefronts, two a CU). Against the im2col kernels, 4 .. 640 outputs: at 256 channels with
// 0.6 of the chip's units taken 0.68 .. 1.05 of their time (268 shapes, 0.89 on average); at 512, where a round of theirs is 256
// tiles of 64 x 64, 0.70 .. 0.88 beyond one round (130 shapes, 0.79) and 0.92 .. 1.09 up to there (512 -> 576 on 23 x 3, batch 25:
// 243 tiles, 17.4 us and 19.1; on 7 x 6, batch 44: 261, 23.1 and 18.0); with less filled, or over several rounds, up to 1.6;
// windows of fewer than nine taps don't pay for their ends. Nor do 128 channels: a wavefront's share of the reduction is half
// as long, and 190 shapes that fill 0.8 of a round took 0.83 .. 1.33 (0.98 on average; to at most 64 outputs 0.95 .. 1.52, half
// of whose workgroups do not fit beside each other); 128 -> 128 on 28 x 28, batch 64, as part of ResNet-18's second stage 81.0 us
// against 81.4 without.
bool patch_plan(const tmq_conv_shape *s, int ho, int wo, PatchPlan &p) {
    if (s->sy != 1 || s->sx != 1 || !(s->C == 256 || s->C == 512) || s->ky * s->kx < 9) return false;
    const int64_t down = (int64_t)(s->ky - 1) * s->dy, across = (int64_t)(s->kx - 1) * s->dx;
    const int64_t top = s->py, left = s->px, bottom = ho - 1 - top + down - (s->H - 1), right = wo - 1 - left + across - (s->W - 1);
    // one row / column of padding serves the end of a row and the start of the next
    p.Hp = s->H + (top > bottom ? top : bottom);
    p.Wp = s->W + (left > right ? left : right);
    if (p.Hp < ho || p.Wp < wo || 16 / wo + 1 > ho) return false;      // more padding than window; planes of a few pixels
    p.slabs = s->C / kSlab;
    p.columns = p.slabs == 8 || s->N <= 64 ? 1 : 2;
    const int waves = p.slabs * p.columns;
    const int64_t M = (int64_t)s->B * ho * wo, tn = (s->N + 64 * p.columns - 1) / (64 * p.columns), slots = 1024 * 2 / waves;
    const int64_t units = (M + 16 * kFragments - 1) / (16 * kFragments) * tn;
    if (units > slots || tn > slots || M >= (int64_t)1 << 30 || M * s->N * 4 >= (int64_t)kNone) return false;
    const double filled = (double)units / slots * s->N / (64.0 * p.columns * tn);
    if (filled < (p.slabs == 8 ? 0.55 : 0.6) || (p.slabs == 8 && (M + 63) / 64 * ((s->N + 63) / 64) <= 256)) return false;
    // the pixels spread evenly over the round
    p.rows = (M + slots / tn - 1) / (slots / tn);
    p.groups = (M + p.rows - 1) / p.rows * tn;
    p.reach = down * p.Wp + across;
    if (s->B * p.Hp * p.Wp + p.reach >= (int64_t)1 << 31) return false;     // places in the padded images are 32 bits
    p.pixels = patch_pixels(p.rows, ho, wo, p.Hp, p.Wp, p.reach);
    p.bytes = p.slabs * p.pixels * kPixelBytes;
    const int64_t sums = (int64_t)waves * 4096 * 4;
    if (p.bytes < sums) p.bytes = sums;
    return p.bytes <= (waves > 4 ? 160 : 80) * 1024;
}

bool patch_conv_ok(const tmq_conv_shape *s, int ho, int wo, int y_f16, PatchPlan &p) {
    return s->N % (y_f16 ? 8 : 4) == 0 && (int64_t)s->B * s->H * s->W * s->C < (int64_t)0x7FFFFFF0 &&
           native_blocks_n(s->N) * native_blocks_k((int64_t)s->C * s->ky * s->kx) < (1 << 21) && patch_plan(s, ho, wo, p);
}

}  // namespace

bool patch_conv_ok(const tmq_conv_shape *s, int ho, int wo, int y_f16) {
    PatchPlan p;
    return patch_conv_ok(s, ho, wo, y_f16, p);
}

bool launch_patch_conv(const void *x, const tmq_conv_shape *s, int ho, int wo, const void *native, const float *scale, const float *bias,
                       const void *residual, int relu, void *y, int y_f16, void *stream, int *status) {
    PatchPlan p;
    if (!(aligned16(x) && aligned16(y) && aligned16(residual) && aligned16(scale) && aligned16(bias) && patch_conv_ok(s, ho, wo, y_f16, p)))
        return false;
    PatchConv cv{};
    cv.x = static_cast<const _Float16 *>(x);
    cv.native = static_cast<const uint32_t *>(native);
    cv.Kb = (int32_t)native_blocks_k((int64_t)s->C * s->ky * s->kx);
    cv.Nb = (int32_t)native_blocks_n(s->N);
    cv.M = (int32_t)((int64_t)s->B * ho * wo);
    cv.N = s->N; cv.C = s->C; cv.H = s->H; cv.W = s->W; cv.B = s->B;
    cv.py = s->py; cv.px = s->px; cv.Hp = (int32_t)p.Hp; cv.Wp = (int32_t)p.Wp;
    cv.ky = s->ky; cv.kx = s->kx; cv.dy = s->dy; cv.dx = s->dx; cv.reach = (int32_t)p.reach;
    cv.pixels = (int32_t)p.pixels;
    cv.rows = (int32_t)p.rows;
    cv.x_bytes = (uint32_t)((int64_t)s->B * s->H * s->W * s->C * 2);
    cv.du = 16 / wo;
    cv.dv = 16 % wo;
    cv.by_tiles_n = FastDiv((uint32_t)((s->N + 64 * p.columns - 1) / (64 * p.columns)));
    cv.by_w = FastDiv((uint32_t)wo);
    cv.by_h = FastDiv((uint32_t)ho);
    cv.by_wp = FastDiv((uint32_t)p.Wp);
    cv.by_hp = FastDiv((uint32_t)p.Hp);
    cv.jobs = (s->W + kJobPixels - 1) / kJobPixels;
    const Epilogue ep{scale, bias, residual, y, relu, y_f16, {}};
#define TMQ_PATCH(cg, sg) (y_f16 ? launch<cg, sg, true>(cv, ep, p.bytes, p.groups, stream) : launch<cg, sg, false>(cv, ep, p.bytes, p.groups, stream))
    *status = p.slabs == 8 ? TMQ_PATCH(1, 8) : p.columns == 2 ? TMQ_PATCH(2, 4) : TMQ_PATCH(1, 4);
#undef TMQ_PATCH
    return true;
}

}  // namespace tmq
