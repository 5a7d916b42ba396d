// Split-reduction ternary GEMM / implicit-GEMM convolution for small outputs: what a workgroup waits for is asked for at once.
//
// The work is dealt out as in mid.hip: a workgroup owns a (16 WM) x (16 WN) tile, wavefront kg multiplies the whole tile over the
// pairs (64 reduction indices) kg, kg + WAVES, ..., and the partial tiles are added through LDS in wavefront order. At these
// sizes neither memory nor the matrix pipe is busy; a launch is the chain arguments -> addresses -> loads -> products -> sum ->
// stores behind the 1.6 us that a launch takes in any case, and this kernel cuts the chain:
//   * Every kernel argument is fetched in one go at the top. Left to the compiler the scalar loads stand where the values are
//     needed, six trips to memory one after the other: the first load of data went out 0.5 us later (clock stamps).
//   * Up to D pairs of a wavefront are in flight, activations and weights both global -> LDS (no registers held, so the ring's
//     slot is an address and the loop one body; the code is a third of mid.hip's). vmcnt counts down pair by pair.
//   * Constants, residual and destinations are asked for between the first loads and the first wait, and the barriers of the
//     sum wait for LDS only: stores and residuals are nobody's business there.
// What bounds the longer reductions is the CU's vector-memory pipe (16 clocks an instruction, 2 WM + WN a pair): deeper rings
// do not help (512 -> 512 on one 7 x 7 image: eight slots 7 % slower than four), smaller tiles on more CUs do.
// Against mid.hip, through the public calls, us: 256 -> 512, 1 x 1 / 2 on 14 x 14, batch 16 5.5 -> 3.6; 128 -> 256, 1 x 1 / 2 on
// 28 x 28, batch 4 4.7 -> 3.1; 64 -> 64, 3 x 3 on one 56 x 56 image 4.3 -> 3.7; 512 -> 512, 3 x 3 on one 7 x 7 5.8 -> 5.3; 128 rows,
// 448 -> 1024 3.2 -> 2.8; 333 fp32 rows, 2000 -> 1000, with their split 15.2 -> 14.3.
#include "common.h"
#include "mfma.h"
#include <utility>

namespace tmq {

namespace {

struct RingPlace {               // conv: geometry of the im2col view; dense: K alone
    int32_t H, W, C, sy, sx, py, px, dy, dx;
    FastDiv by_wo, by_ho, by_slabs, by_kx;
};

template <class Map>
struct RingArgs {
    const _Float16 *x;
    const uint32_t *native;
    const float *scale, *bias;
    const void *residual;
    void *y;
    int32_t M, N, K, Nb, Kb, pairs;
    uint32_t x_bytes, native_bytes;
    int32_t relu, y_f16, by_rows;
    int32_t tiles;
    FastDiv by_tiles_n;
    RingPlace at;
    [[no_unique_address]] Map map;
};

__device__ __forceinline__ void dword_to_lds(BufferResource rsrc, uint32_t lane_offset, uint32_t base, unsigned char *dst) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(3))) void *lds_ptr;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr)dst, 4, lane_offset, base, 0, 0);
#endif
}

// Waits until at most r * kN loads are outstanding (r uniform, 0 .. kMax).
template <int kN, int kMax>
__device__ __forceinline__ void wait_younger(int r) {
    if constexpr (kMax == 0) {
        __builtin_amdgcn_s_waitcnt(0x0F70);
    } else {
        if (r >= kMax) __builtin_amdgcn_s_waitcnt(0x0F70 | ((kMax * kN) & 15) | (((kMax * kN) >> 4) << 14));
        else wait_younger<kN, kMax - 1>(r);
    }
}

template <int WM, int WN, int WAVES, int D, bool CONV, class Map>
__global__ __launch_bounds__(64 * WAVES) void ring_kernel(const RingArgs<Map> a) {
    constexpr int kFrag = 16 * 128, kSlot = WM * kFrag + WN * 256, kWave = D * kSlot, kN = 2 * WM + WN;
    static_assert(kN * (D - 1) < 64, "vmcnt is a 6-bit counter");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    asm volatile("" ::"s"(a.x), "s"(a.native), "s"(a.scale), "s"(a.bias), "s"(a.residual), "s"(a.y), "s"(a.M), "s"(a.N), "s"(a.K),
                 "s"(a.Nb), "s"(a.Kb), "s"(a.pairs), "s"(a.x_bytes), "s"(a.native_bytes), "s"(a.relu), "s"(a.y_f16), "s"(a.by_rows), "s"(a.tiles),
                 "s"(a.by_tiles_n.mul), "s"(a.by_tiles_n.shift), "s"(a.by_tiles_n.d));
    if constexpr (CONV)
        asm volatile("" ::"s"(a.at.H), "s"(a.at.W), "s"(a.at.C), "s"(a.at.sy), "s"(a.at.sx), "s"(a.at.py), "s"(a.at.px), "s"(a.at.dy),
                     "s"(a.at.dx), "s"(a.at.by_wo.mul), "s"(a.at.by_wo.shift), "s"(a.at.by_wo.d), "s"(a.at.by_ho.mul), "s"(a.at.by_ho.shift),
                     "s"(a.at.by_ho.d), "s"(a.at.by_slabs.mul), "s"(a.at.by_slabs.shift), "s"(a.at.by_slabs.d), "s"(a.at.by_kx.mul),
                     "s"(a.at.by_kx.shift), "s"(a.at.by_kx.d));
    const int lane = threadIdx.x & 63, kg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, g = lane >> 4;
    unsigned char *const win = smem + kg * kWave;
    // (when x is the larger operand the XCDs take consecutive runs of tiles, an eighth of the rows each and all weights)
    const int tile = a.by_rows ? xcd_contiguous(blockIdx.x, a.tiles) : (int)blockIdx.x;
    int tn;
    const int tm = (int)a.by_tiles_n.divmod((uint32_t)tile, tn);
    const int m0 = tm * (16 * WM), n0 = tn * (16 * WN);

    // rows: load c of fragment i covers rows 16 i + 8 c .. + 7, eight lanes a row; the 16-byte chunk at position p of row r
    // is chunk p ^ ((r / 2) % 8), so that operand reads of 16 rows fall into different banks
    int32_t off[WM][2], ih0[WM][2], iw0[WM][2];
#pragma unroll
    for (int i = 0; i < WM; i++)
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int R = c * 8 + (lane >> 3), chunk = ((lane & 7) ^ ((R >> 1) & 7)) * 8;
            int m = m0 + i * 16 + R;
            if (m >= a.M) m = a.M - 1;                         // rows past M: finite data, never stored
            if constexpr (CONV) {
                int ow, oh;
                const uint32_t t = a.at.by_wo.divmod((uint32_t)m, ow);
                const int b = (int)a.at.by_ho.divmod(t, oh);
                ih0[i][c] = oh * a.at.sy - a.at.py;
                iw0[i][c] = ow * a.at.sx - a.at.px;
                off[i][c] = ((b * a.at.H + ih0[i][c]) * a.at.W + iw0[i][c]) * a.at.C + chunk;
            } else {
                off[i][c] = m * a.K + chunk;
            }
        }
    const BufferResource xr = make_buffer_resource(a.x, a.x_bytes), wr = make_buffer_resource(a.native, a.native_bytes);
    uint32_t wbase[WN];
#pragma unroll
    for (int nj = 0; nj < WN; nj++) {
        int nb = n0 / 16 + nj;
        if (nb >= a.Nb) nb = a.Nb - 1;                          // finite bits, never stored
        wbase[nj] = (uint32_t)(nb * a.Kb) * 1024u;
    }
    const int np = a.pairs > kg ? (a.pairs - kg + WAVES - 1) / WAVES : 0;
    auto request = [&](int p, unsigned char *slot) {
        const int pi = kg + p * WAVES;
#pragma unroll
        for (int nj = 0; nj < WN; nj++)
            dword_to_lds(wr, (uint32_t)lane * 16u, wbase[nj] + (uint32_t)(pi >> 2) * 1024u + (uint32_t)(pi & 3) * 4u, slot + WM * kFrag + nj * 256);
        if constexpr (CONV) {
            int s, tj;
            const uint32_t tap = a.at.by_slabs.divmod((uint32_t)pi, s);
            const int ti = (int)a.at.by_kx.divmod(tap, tj);
            const int di = ti * a.at.dy, dj = tj * a.at.dx, delta = (di * a.at.W + dj) * a.at.C + s * 64;
#pragma unroll
            for (int i = 0; i < WM; i++)
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    const bool in = ((unsigned)(ih0[i][c] + di) < (unsigned)a.at.H) & ((unsigned)(iw0[i][c] + dj) < (unsigned)a.at.W);
                    buffer_to_lds(xr, in ? (uint32_t)(off[i][c] + delta) * 2u : kPastTheEnd, slot + i * kFrag + c * 1024);
                }
        } else {
#pragma unroll
            for (int i = 0; i < WM; i++)
#pragma unroll
                for (int c = 0; c < 2; c++) buffer_to_lds(xr, (uint32_t)(off[i][c] + pi * 64) * 2u, slot + i * kFrag + c * 1024);
        }
    };
#pragma unroll 1
    for (int p = 0; p < D && p < np; p++) request(p, win + p * kSlot);

    // what the epilogue needs, asked for while the operands are on their way
    constexpr int T = 64 * WAVES, kC4 = 4 * WN, kSweep = T / kC4, kIter = (16 * WM + kSweep - 1) / kSweep;
    static_assert(T % kC4 == 0, "a thread keeps its columns");
    const int c4 = threadIdx.x % kC4, row0 = threadIdx.x / kC4, n = n0 + c4 * 4;
    floatx4 sc = {1.f, 1.f, 1.f, 1.f}, bi = {0.f, 0.f, 0.f, 0.f};
    if (n < a.N) {
        if (a.scale) sc = *reinterpret_cast<const floatx4 *>(a.scale + n);
        if (a.bias) bi = *reinterpret_cast<const floatx4 *>(a.bias + n);
    }
    int64_t at[kIter];
    half4 res16[kIter];
    floatx4 res32[kIter];
    [[maybe_unused]] float gs[kIter];                            // row pairs: 1 / s of the row's group
#pragma unroll
    for (int it = 0; it < kIter; it++) {
        const int row = row0 + it * kSweep, m = m0 + row;
        at[it] = -1;
        if (row < 16 * WM && m < a.M && n < a.N) {
            const int64_t px = a.map.pixel(m);
            if (!Map::kDrops || px >= 0) at[it] = px * a.N + n;
        }
        if constexpr (Map::kPairs) gs[it] = at[it] >= 0 ? a.map.fragment_scale(m & ~15) : 0.f;
        if (a.residual && at[it] >= 0) {
            if (a.y_f16) res16[it] = *reinterpret_cast<const half4 *>(static_cast<const _Float16 *>(a.residual) + at[it]);
            else res32[it] = *reinterpret_cast<const floatx4 *>(static_cast<const float *>(a.residual) + at[it]);
        }
    }

    floatx4 acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; i++)
#pragma unroll
        for (int nj = 0; nj < WN; nj++) acc[i][nj] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int key = (j >> 1) & 7;
    int slot = 0;
#pragma unroll 1
    for (int p = 0; p < np; p++) {
        wait_younger<kN, D - 1>(np - 1 - p);
        __builtin_amdgcn_sched_barrier(0);
        unsigned char *const src = win + slot * kSlot;
        half8 x[2][WM];
        uint32_t w[WN];
#pragma unroll
        for (int nj = 0; nj < WN; nj++) w[nj] = *reinterpret_cast<const uint32_t *>(src + WM * kFrag + nj * 256 + lane * 4);
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int i = 0; i < WM; i++) x[s][i] = *reinterpret_cast<const half8 *>(src + i * kFrag + j * 128 + (((4 * s + g) ^ key) * 16));
        if (p + D < np) {
            __builtin_amdgcn_s_waitcnt(0xC07F);           // lgkmcnt(0): the slot has been read out
            __builtin_amdgcn_sched_barrier(0);
            request(p + D, src);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int nj = 0; nj < WN; nj++) {
                const half8 b = decode_step(w[nj], s);
#pragma unroll
                for (int i = 0; i < WM; i++) acc[i][nj] = mfma16(b, x[s][i], acc[i][nj]);
            }
        slot = slot + 1 == D ? 0 : slot + 1;
        __builtin_amdgcn_sched_barrier(0);
    }

    // partial tiles through LDS, added in wavefront order; lane (j, g) of fragment (i, nj) holds y[16 i + j][16 nj + 4 g + r]
    constexpr int kFragPitch = 1024 + 64;
    lds_barrier();
#pragma unroll
    for (int i = 0; i < WM; i++)
#pragma unroll
        for (int nj = 0; nj < WN; nj++)
            *reinterpret_cast<floatx4 *>(smem + (kg * WM * WN + i * WN + nj) * kFragPitch + (j * 4 + (g ^ ((j >> 2) & 3))) * 16) = acc[i][nj];
    lds_barrier();
    auto row_sums = [&](int row) {
        const unsigned char *src = smem + ((row >> 4) * WN + (c4 >> 2)) * kFragPitch + ((row & 15) * 4 + ((c4 & 3) ^ ((row >> 2) & 3))) * 16;
        floatx4 t[WAVES];
#pragma unroll
        for (int q = 0; q < WAVES; q++) t[q] = *reinterpret_cast<const floatx4 *>(src + q * WM * WN * kFragPitch);
        floatx4 v = t[0];
#pragma unroll
        for (int q = 1; q < WAVES; q++) v += t[q];
        return v;
    };
#pragma unroll
    for (int it = 0; it < kIter; it++) {
        const int row = row0 + it * kSweep;
        if (at[it] < 0) continue;
        floatx4 v = row_sums(row);
        if constexpr (Map::kPairs) v = (v + row_sums(row ^ 8)) * gs[it];
        v = v * (sc * (1.0f / kWeightUnit)) + bi;
        if (a.y_f16) {
            if (a.residual) {
#pragma unroll
                for (int r = 0; r < 4; r++) v[r] += (float)res16[it][r];
            }
            half4 h;
#pragma unroll
            for (int r = 0; r < 4; r++) h[r] = (_Float16)((a.relu && v[r] < 0.f) ? 0.f : v[r]);
            *reinterpret_cast<half4 *>(static_cast<_Float16 *>(a.y) + at[it]) = h;
        } else {
            if (a.residual) v += res32[it];
            if (a.relu) {
#pragma unroll
                for (int r = 0; r < 4; r++) v[r] = v[r] < 0.f ? 0.f : v[r];
            }
            *reinterpret_cast<floatx4 *>(static_cast<float *>(a.y) + at[it]) = v;
        }
    }
}

constexpr int64_t ring_lds(int WM, int WN, int WAVES, int D) {
    const int64_t win = (int64_t)WAVES * D * (WM * 16 * 128 + WN * 256), sums = (int64_t)WAVES * WM * WN * (1024 + 64);
    return win > sums ? win : sums;
}

template <int WM, int WN, int WAVES, int D, bool CONV, class Map>
int launch(RingArgs<Map> a, void *stream) {
    const int64_t tm = (a.M + 16 * WM - 1) / (16 * WM), tn = (a.N + 16 * WN - 1) / (16 * WN);
    if (tm * tn > 0x7FFFFFFF) return TMQ_ERR_TOO_LARGE;
    constexpr size_t lds = ring_lds(WM, WN, WAVES, D);
    static_assert(lds <= 160 * 1024, "LDS budget");
    a.tiles = (int32_t)(tm * tn);
    a.by_tiles_n = FastDiv((uint32_t)tn);
    a.by_rows = 8 * (int64_t)a.M > a.N ? 1 : 0;
    auto kernel = ring_kernel<WM, WN, WAVES, D, CONV, Map>;
    if (lds > 64 * 1024) {
        if (int st = allow_dynamic_lds(reinterpret_cast<const void *>(kernel), lds)) return st;
    }
    hipLaunchKernelGGL(kernel, dim3((uint32_t)(tm * tn)), dim3(64 * WAVES), lds, as_stream(stream), a);
    return check_launch();
}

// The tiles on offer.
constexpr RingTile kRingTiles[] = {{1, 1, 4, 5}, {1, 1, 8, 4}, {1, 2, 4, 4}, {1, 2, 8, 4}, {2, 2, 4, 3}, {2, 2, 8, 2},
                                   {1, 4, 4, 4}, {2, 4, 8, 2}, {2, 4, 4, 3}, {4, 4, 4, 2}, {4, 4, 8, 2}};
constexpr int kTiles = sizeof(kRingTiles) / sizeof(kRingTiles[0]);

// Microseconds a launch is expected to take, fitted to 1700 shapes (convolutions of 64 .. 512 channels, 1 x 1 .. 5 x 5, dense rows,
// fp32 row pairs; 17 .. 15000 rows, 16 .. 8192 columns) with eleven tiles each: the launch, the chain of a wavefront's pairs for
// every round of workgroups, and what shares a CU -- vector-memory instructions, products, sums. The tile it picks takes 1.01 of
// the fastest one's time on average. The tile is a constant here: no division is left of the eleven evaluations.
template <int I>
double ring_cost(int64_t M, int64_t pairs, int64_t N, bool conv) {
    constexpr RingTile t = kRingTiles[I];
    constexpr int64_t fit = 160 * 1024 / ring_lds(t.wm, t.wn, t.waves, t.depth), resident = fit < 32 / t.waves ? fit : 32 / t.waves;
    constexpr double frags = t.wm * t.wn;
    const int64_t groups = ((M + 16 * t.wm - 1) / (16 * t.wm)) * ((N + 16 * t.wn - 1) / (16 * t.wn));
    const double rounds = (double)((groups + 256 * resident - 1) / (256 * resident)), chain = (double)((pairs + t.waves - 1) / t.waves);
    const double per_cu = (double)((groups + 255) / 256);
    return 2.35 + (conv ? 0.46 : 0.0) + rounds * (0.416 + 0.0684 * frags + chain * (0.112 + 0.00901 * frags)) +
           per_cu * (0.168 + 0.006 * t.waves * frags + pairs * (0.00623 * (2 * t.wm + t.wn) + 0.00214 * frags + (conv ? 0.00218 * t.wm : 0.0)));
}

template <int... I>
int cheapest_tile(int64_t M, int64_t pairs, int64_t N, bool conv, std::integer_sequence<int, I...>) {
    double us[] = {ring_cost<I>(M, pairs, N, conv)...};
    // (the fit takes 16 x 64 tiles of five to seven pairs a wavefront for up to a fifth faster than they are: dense, 96 rows,
    // 1792 -> 8192 9.5 us, 8.1 on the next tile; 1995 pixels, 64 -> 320, 5 x 5 9.6 and 8.8. They stay out of it there.)
    if (pairs >= 20 && pairs <= 28) us[6] = 1e30;
    static_assert(kRingTiles[6].wm == 1 && kRingTiles[6].wn == 4, "16 x 64");
    int best = 0;
    for (int i = 1; i < kTiles; i++)
        if (us[i] < us[best]) best = i;
    return best;
}

template <bool CONV, int I, class Map>
int launch_tile(const RingArgs<Map> &a, void *stream) {
    constexpr RingTile t = kRingTiles[I];
    return launch<t.wm, t.wn, t.waves, t.depth, CONV>(a, stream);
}

template <bool CONV, class Map>
int by_tile(const RingArgs<Map> &a, int tile, void *stream) {
    switch (tile) {
        case 0: return launch_tile<CONV, 0>(a, stream);
        case 1: return launch_tile<CONV, 1>(a, stream);
        case 2: return launch_tile<CONV, 2>(a, stream);
        case 3: return launch_tile<CONV, 3>(a, stream);
        case 4: return launch_tile<CONV, 4>(a, stream);
        case 5: return launch_tile<CONV, 5>(a, stream);
        case 6: return launch_tile<CONV, 6>(a, stream);
        case 7: return launch_tile<CONV, 7>(a, stream);
        case 8: return launch_tile<CONV, 8>(a, stream);
        case 9: return launch_tile<CONV, 9>(a, stream);
        default: return launch_tile<CONV, 10>(a, stream);
    }
}

template <class Map>
RingArgs<Map> ring_args(const void *x, int64_t x_elements, int64_t M, int64_t K, const void *native, int64_t N, const float *scale,
                        const float *bias, const void *residual, int relu, void *y, int y_f16, const Map &map) {
    RingArgs<Map> a{};
    a.x = static_cast<const _Float16 *>(x);
    a.native = static_cast<const uint32_t *>(native);
    a.scale = scale;
    a.bias = bias;
    a.residual = residual;
    a.y = y;
    a.M = (int32_t)M;
    a.N = (int32_t)N;
    a.K = (int32_t)K;
    a.Nb = (int32_t)native_blocks_n(N);
    a.Kb = (int32_t)native_blocks_k(K);
    a.pairs = (int32_t)(K / 64);
    a.x_bytes = (uint32_t)(x_elements * 2);
    a.native_bytes = (uint32_t)((int64_t)a.Nb * a.Kb * 1024);
    a.relu = relu;
    a.y_f16 = y_f16;
    a.map = map;
    return a;
}

}  // namespace

// What of mid.hip's problems (K a multiple of 64, 16-byte aligned rows, fewer than 2^31 elements) this kernel can take: results
// and constants in whole quads, and reductions of up to 4608 indices -- with 192 64 x 64 tiles or more up to 3583, where mid.hip
// fetches whole weight blocks (beyond these lines 0.94 of mid.hip on average, to 1.29). mid_holds (mid.hip) keeps the others.
bool ring_ok(int64_t M, int64_t K, int64_t N, const float *scale, const float *bias, const void *residual, const void *y) {
    const int64_t tiles64 = ((M + 63) / 64) * ((N + 63) / 64);
    return K % 64 == 0 && K <= (tiles64 >= 192 ? 3583 : 4608) && N % 4 == 0 && N < (1 << 20) && M < (int64_t)0x7FFFFFFF && aligned16(y) &&
           aligned16(residual) && aligned16(scale) && aligned16(bias);
}

// Its tile for a problem, an index into kRingTiles.
int ring_tile(int64_t M, int64_t K, int64_t N, bool conv) {
    return cheapest_tile(M, K / 64, N, conv, std::make_integer_sequence<int, kTiles>{});
}
RingTile ring_tile_shape(int tile) { return kRingTiles[tile]; }

int launch_ring_dense(int tile, const void *x, int64_t M, int64_t K, const void *native, int64_t N, const float *scale, const float *bias,
                      const void *residual, int relu, void *y, int y_f16, const PairMap *pairs, void *stream) {
    if (pairs) return by_tile<false>(ring_args(x, M * K, M, K, native, N, scale, bias, residual, relu, y, y_f16, *pairs), tile, stream);
    return by_tile<false>(ring_args(x, M * K, M, K, native, N, scale, bias, residual, relu, y, y_f16, NoMap{}), tile, stream);
}

template <class Map>
static int ring_conv(int tile, const void *x, const tmq_conv_shape *s, int ho, int wo, const void *native, const float *scale,
                     const float *bias, const void *residual, int relu, void *y, int y_f16, const Map &map, void *stream) {
    auto a = ring_args(x, (int64_t)s->B * s->H * s->W * s->C, (int64_t)s->B * ho * wo, (int64_t)s->C * s->ky * s->kx, native, s->N, scale, bias,
                       residual, relu, y, y_f16, map);
    a.at.H = s->H; a.at.W = s->W; a.at.C = s->C;
    a.at.sy = s->sy; a.at.sx = s->sx; a.at.py = s->py; a.at.px = s->px; a.at.dy = s->dy; a.at.dx = s->dx;
    a.at.by_wo = FastDiv((uint32_t)wo);
    a.at.by_ho = FastDiv((uint32_t)ho);
    a.at.by_slabs = FastDiv((uint32_t)(s->C / 64));
    a.at.by_kx = FastDiv((uint32_t)s->kx);
    return by_tile<true>(a, tile, stream);
}

int launch_ring_conv(int tile, const void *x, const tmq_conv_shape *s, int ho, int wo, const void *native, const float *scale,
                     const float *bias, const void *residual, int relu, void *y, int y_f16, const RowMap *map, void *stream) {
    if (map) return ring_conv(tile, x, s, ho, wo, native, scale, bias, residual, relu, y, y_f16, *map, stream);
    return ring_conv(tile, x, s, ho, wo, native, scale, bias, residual, relu, y, y_f16, NoMap{}, stream);
}

}  // namespace tmq
