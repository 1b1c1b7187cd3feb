// K-quant GEMM for few tokens (gfx950): the products of gemm_kq.hip, for calls
// whose 256 x 128 tiles leave most of the device or most of a tile idle (chat
// prompts and prefill chunks, cpu_quant_matmul of src/kernels_quant.cpp:369-412
// with small M).  Same operand planes, same exact integer sums and the same
// fp32 epilogue per super-block; only the order in which super-blocks are added
// differs.
//
// What bounds it: the weight planes (two bytes per weight), read once per
// token tile.  So nothing is staged: one 16x16x64 MFMA takes exactly one 1 KB
// block of a tiled plane as an operand (lane l: row l%16, values
// 16*(l/16) .. +15), which a wave loads as one contiguous 1 KB run straight
// into registers, PD steps of 64 values ahead of their use.  A workgroup owns
// 16*MT tokens x 16*NT features; its waves deal the super-blocks of K among
// themselves and add their fp32 tiles through LDS, in wave order, at the end:
// no barrier in the loop, no partial tiles in memory, no second launch.
// Measured with the quantizer, weights from memory, 256 x 128 tiles / this: Q6_K
// 37 x 12288 -> 4096 46.8 / 28.8 us (4.4 TB/s over the planes), Q5_K 128 x 4096
// -> 12288 54.7 / 42.4 us, 16 x 4096 -> 12288 56.7 / 24.7 us (5.4 TB/s).
#include <algorithm>

#include "pixhip_device.h"
#include "pixhip_internal.h"

namespace pixhip {
namespace {

constexpr int kWaves = 4, kThreads = 64 * kWaves;

struct RowsArgs {
    const int8_t* xq;     // tiled [Mpad/16][K/64][16][64]
    const float* xdT;     // [K/256][Mpad]
    const _Float16* xbs;  // tiled [Mpad/32][K/256][32][16] (Q5_K)
    const int8_t* whi;    // tiled [Npad/16][K/64][16][64]
    const int8_t* wlo;
    const float* wdT;     // [K/256][Npad]
    const float* wdm;     // [K/256][Npad] (Q5_K)
    const _Float16* wmn;  // [K/256][Npad][8] (Q5_K)
    float* y;
    const float* bias;
    int M, N, K, Mpad, Npad, tiles_m;
    size_t ldy, yoff;
};

__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }

// Steps of 64 values a wave's loads run ahead of its MFMAs: a whole super-block
// where the registers allow it, else two (weights) and one (activations: each
// fragment is reloaded right after its last use).
template <int MT, int NT> constexpr int weight_steps() { return MT * NT <= 4? 4 : 2; }
template <int MT, int NT> constexpr int act_steps() { return MT <= 2? 4 : MT <= 4 && MT * NT <= 8? 2 : 1; }

// STREAM: the weights are read once and do not stay in the caches (non-temporal
// loads).
template <bool Q5, int MT, int NT, bool STREAM>
__global__ __launch_bounds__(kThreads, 2) void gemm_kq_rows_kernel(RowsArgs g)
{
    constexpr int WD = weight_steps<MT,NT>(), AD = act_steps<MT,NT>();
    constexpr int kTile = MT * NT * 256;  // floats of a wave's tile
    __shared__ __attribute__((aligned(16))) float red[kWaves * kTile];

    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t lane = threadIdx.x & 63, lc = lane & 15, lg = lane >> 4;
    // Workgroup b runs on XCD b % 8: the token tiles of one group of features
    // are neighbours on one XCD, so its L2 serves all but the first of them
    // (with the token tiles one after the other over the whole grid the
    // weights came from memory again: 128 x 12288 features, K = 4096, 47.4 us a call
    // against 44.1).
    const int xcd = (int)blockIdx.x & 7, seq = (int)blockIdx.x >> 3;
    const int n0 = (seq / g.tiles_m * 8 + xcd) * (16 * NT), m0 = seq % g.tiles_m * (16 * MT);
    if (n0 >= g.N) return;
    const int C = g.K / 64, nb = g.K / PIX_QK;
    const uint32_t frag = lc * 64 + lg * 16;  // this lane's 16 bytes of a 1 KB block

    // 1 KB blocks of this workgroup's rows: block (row group, step) at
    // (group * C + step) * 1024.  The last feature tiles of a workgroup can lie
    // past the padded rows (NT = 3): they repeat the last one and are not stored.
    const int8_t* pa = g.xq + (size_t)(m0 >> 4) * C * 1024 + frag;
    uint32_t wrow[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) wrow[j] = (uint32_t)min((n0 >> 4) + j,(g.Npad >> 4) - 1);
    const int8_t *ph[NT], *pl[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) {
        ph[j] = g.whi + (size_t)wrow[j] * C * 1024 + frag;
        pl[j] = g.wlo + (size_t)wrow[j] * C * 1024 + frag;
    }

    v4f y[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) y[i][j] = v4f{0.0f,0.0f,0.0f,0.0f};

    if (wave < nb) {
        v4i wh[WD][NT], wl[WD][NT], a[AD][MT];
        // Step t (0..3) of super-block b sits in slot t % WD (% AD); loads past
        // the wave's last super-block repeat it (b is clamped by the caller).
        auto load_w = [&](int b, int t) {
            const uint32_t at = (uint32_t)(b * 4 + t) * 1024u;
#pragma unroll
            for (int j = 0; j < NT; j++) {
                const v4i *h = reinterpret_cast<const v4i*>(ph[j] + at), *l = reinterpret_cast<const v4i*>(pl[j] + at);
                wh[t % WD][j] = STREAM? __builtin_nontemporal_load(h) : *h;
                wl[t % WD][j] = STREAM? __builtin_nontemporal_load(l) : *l;
            }
        };
        auto load_a = [&](int b, int t, int i) {
            a[t % AD][i] = *reinterpret_cast<const v4i*>(pa + (uint32_t)((i * C + b * 4 + t) * 1024));
        };
#pragma unroll
        for (int t = 0; t < WD; t++) {
            load_w(wave,t);
            if (t < AD) {
#pragma unroll
                for (int i = 0; i < MT; i++) load_a(wave,t,i);
            }
        }
        for (int b = wave; b < nb; b += kWaves) {
            const int nx = b + kWaves < nb? b + kWaves : b;
            // The super-block's epilogue inputs, wanted after its last MFMA.
            float wd[NT], wm[NT];
            v4h mn[NT], bs[MT];
            v4f yd[MT];
            auto load_scales = [&]() {
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    const size_t n = (size_t)b * g.Npad + wrow[j] * 16 + lc;
                    wd[j] = g.wdT[n];
                    if constexpr (Q5) {
                        wm[j] = g.wdm[n];
                        mn[j] = *reinterpret_cast<const v4h*>(g.wmn + n * 8 + 4 * (lg & 1));
                    }
                }
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    const size_t m = (size_t)m0 + 16 * i;
                    yd[i] = *reinterpret_cast<const v4f*>(g.xdT + (size_t)b * g.Mpad + m + 4 * lg);
                    if constexpr (Q5)
                        bs[i] = *reinterpret_cast<const v4h*>(g.xbs + tiled_bs_index(m + lc,(size_t)b,4 * (int)lg,(size_t)g.K));
                }
            };
            v4i hi[MT][NT], lo[MT][NT];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                if (t == (MT <= 3? 0 : 2)) load_scales();
                fence();
#pragma unroll
                for (int i = 0; i < MT; i++) {
#pragma unroll
                    for (int j = 0; j < NT; j++) {
                        const v4i z = {0,0,0,0};
                        hi[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[t % AD][i],wh[t % WD][j],t? hi[i][j] : z,0,0,0);
                        lo[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[t % AD][i],wl[t % WD][j],t? lo[i][j] : z,0,0,0);
                    }
                    fence();
                    if (t + AD < 4) load_a(b,t + AD,i);
                    else load_a(nx,t + AD - 4,i);
                    fence();
                }
                if (t + WD < 4) load_w(b,t + WD);
                else load_w(nx,t + WD - 4);
            }
            fence();
            // y += yd * (wd * S - wdmin * Mn), as gemm_kq.hip
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    v4f mt = {0.0f,0.0f,0.0f,0.0f};
                    if constexpr (Q5) mt = __builtin_amdgcn_mfma_f32_16x16x16f16(bs[i],mn[j],mt,0,0,0);
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float s = (float)(hi[i][j][r] * 64 + lo[i][j][r]) * wd[j];
                        y[i][j][r] = __builtin_fmaf(yd[i][r],Q5? __builtin_fmaf(mt[r],-wm[j],s) : s,y[i][j][r]);
                    }
                }
        }
    }

    // The waves' tiles, [wave][token][feature], added in wave order.
    constexpr int F = 16 * NT;
    const int waves = min(nb,kWaves);
    if (wave < waves) {
        float* mine = red + wave * kTile + lc;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) mine[(16 * i + 4 * (int)lg + r) * F + 16 * j] = y[i][j][r];
    }
    __syncthreads();
    for (int e = 4 * (int)threadIdx.x; e < kTile; e += 4 * kThreads) {
        v4f v = *reinterpret_cast<const v4f*>(red + e);
        for (int w = 1; w < waves; w++) v += *reinterpret_cast<const v4f*>(red + w * kTile + e);
        const int m = m0 + e / F, n = n0 + e % F;
        if (m >= g.M) break;
        float* out = g.y + g.yoff + (size_t)m * g.ldy + n;
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (n + q < g.N) out[q] = v[q] + (g.bias? g.bias[n + q] : 0.0f);
    }
}

template <bool Q5, int MT, int NT> hipError_t launch_tile(RowsArgs g, hipStream_t s)
{
    const size_t tiles_n = ((size_t)g.N + 16 * NT - 1) / (16 * NT);
    g.tiles_m = (g.M + 16 * MT - 1) / (16 * MT);
    const dim3 grid((unsigned)((tiles_n + 7) / 8 * 8 * g.tiles_m));
    // One token tile reads each weight once.  Planes of 48 MB and more are then
    // read past the caches (33 tokens, us a call, plain / so: 3584 x 14336
    // 32.2 / 29.6, 8192 x 12288 55.8 / 51.3, 12288 x 4096 33.7 / 31.6); smaller
    // ones may still be there from the last call (1024 x 18944 17.5 / 19.7,
    // 3584 x 4096 12.1 / 14.3, six weights in turn).
    if (g.tiles_m == 1 && (size_t)g.Npad * (size_t)g.K * 2 >= (size_t)48 << 20) gemm_kq_rows_kernel<Q5,MT,NT,true><<<grid,dim3(kThreads),0,s>>>(g);
    else gemm_kq_rows_kernel<Q5,MT,NT,false><<<grid,dim3(kThreads),0,s>>>(g);
    return hipGetLastError();
}

// The tile of a call.  A workgroup's operand traffic per 64 values is 2*NT KB of
// weights and MT KB of activations, and the busiest XCD's CUs run groups / CUs
// of them (at least one): the tile with the least product of the two is taken.
// Measured, K = 4096, us a call: 48 tokens x 12288 features 3x1 26.7, 3x2 25.1;
// 128 x 4096 4x1 21.3, 4x2 16.6, 8x1 19.7; 64 x 2048 (K = 12288) 2x1 20.6, 2x2
// 25.7, 4x1 26.5.  Larger tiles (4x3, 6x2, 8x2) need more registers than two
// workgroups per CU leave: 43 us and more where 4x2 takes 39.2 (128 x 12288).
struct Tile {
    int mt, nt;
};
constexpr Tile kTiles[] = {{1,3},{1,2},{1,1},{2,2},{2,1},{3,2},{3,1},{4,2},{4,1},{6,1},{8,1}};

Tile choose_tile(size_t M, size_t N, double* least_cost)
{
    const double cus = device_cus();
    Tile best = kTiles[0];
    double least = 0.0;
    for (const Tile& t : kTiles) {
        const size_t rows = 16 * (size_t)t.mt;
        if (t.mt > 1 && rows - 16 >= M) continue;                // 16 rows of padding only
        if (PIX_GEMM_MTILE % rows && rows < M) continue;         // its last tile would leave the padding
        // workgroups of the busiest XCD (whole feature groups are dealt to the eight)
        const double groups = (double)((M + rows - 1) / rows) * (double)((N + 128 * t.nt - 1) / (128 * t.nt));
        const double cost = (2 * t.nt + t.mt) * std::max(1.0,groups / (cus / 8));
        if (least == 0.0 || cost < least) {
            least = cost;
            best = t;
        }
    }
    *least_cost = least;
    return best;
}

template <bool Q5> hipError_t launch_rows(const RowsArgs& g, hipStream_t s)
{
    double cost;
    const Tile t = choose_tile((size_t)g.M,(size_t)g.N,&cost);
    switch (t.mt * 8 + t.nt) {
    case 1 * 8 + 3: return launch_tile<Q5,1,3>(g,s);
    case 1 * 8 + 2: return launch_tile<Q5,1,2>(g,s);
    case 1 * 8 + 1: return launch_tile<Q5,1,1>(g,s);
    case 2 * 8 + 2: return launch_tile<Q5,2,2>(g,s);
    case 2 * 8 + 1: return launch_tile<Q5,2,1>(g,s);
    case 3 * 8 + 2: return launch_tile<Q5,3,2>(g,s);
    case 3 * 8 + 1: return launch_tile<Q5,3,1>(g,s);
    case 4 * 8 + 2: return launch_tile<Q5,4,2>(g,s);
    case 4 * 8 + 1: return launch_tile<Q5,4,1>(g,s);
    case 6 * 8 + 1: return launch_tile<Q5,6,1>(g,s);
    case 8 * 8 + 1: return launch_tile<Q5,8,1>(g,s);
    }
    return hipErrorInvalidValue;
}

template <bool Q5> hipError_t check_and_launch(const Act8K& a, RowsArgs g, size_t M, size_t N, size_t K, size_t npad, const Output& out,
                                               hipStream_t s)
{
    const size_t lim = (size_t)1 << 31;
    // The 2 GiB operand limits of gemm_kq.hip.
    const size_t mpad = (M + PIX_GEMM_MTILE - 1) / PIX_GEMM_MTILE * PIX_GEMM_MTILE;
    const size_t scales = (K / PIX_QK) * std::max(npad,a.mpad) * 16;
    if (!M || !N || K % PIX_QK || a.mpad < mpad || npad < N || npad % PIX_GEMM_NTILE || a.mpad * K >= lim || npad * K >= lim ||
        scales >= lim)
        return hipErrorInvalidValue;
    g.M = (int)M; g.N = (int)N; g.K = (int)K; g.Mpad = (int)a.mpad; g.Npad = (int)npad;
    g.xq = a.qs; g.xdT = a.d; g.xbs = a.bs;
    g.y = out.y; g.bias = out.bias; g.ldy = out.ldy; g.yoff = out.offset;
    return launch_rows<Q5>(g,s);
}

}  // namespace

hipError_t launch_gemm_rows_q5_K(const Act8K& a, const PlanesQ5K& w, size_t M, size_t N, size_t K, const Output& out, hipStream_t s)
{
    RowsArgs g = {};
    g.whi = w.hi; g.wlo = w.lo; g.wdT = w.d; g.wdm = w.dm; g.wmn = w.mn;
    return check_and_launch<true>(a,g,M,N,K,w.npad,out,s);
}

hipError_t launch_gemm_rows_q6_K(const Act8K& a, const PlanesQ6K& w, size_t M, size_t N, size_t K, const Output& out, hipStream_t s)
{
    RowsArgs g = {};
    g.whi = w.hi; g.wlo = w.lo; g.wdT = w.d;
    return check_and_launch<false>(a,g,M,N,K,w.npad,out,s);
}

// The line to the 256 x 128 tiles of gemm_kq.hip (launched here as one 256-row
// tile or its K pieces for any M up to 256).  Measured over M 33 .. 256, N 1000 ..
// 18944, K 1024 .. 12288 with weights from memory, us a call with the
// quantizer, those tiles / this form:
//   M <= 64 (one token tile): 14.4 / 7.1 (33 x 1000, K = 1024) to 212 / 112
//     (33 x 18944, K = 12288), nowhere less than 1.2 times faster;
//   M <= 128 (weights read by two token tiles): 58 / 44 (128 x 12288, K =
//     4096), 29 / 16 (4096, 3584), but 24.2 / 29.5 (18944, 1024: cost 37) and
//     101 / 105 (9728, 12288: its K pieces fill the device), 36 / 43 (70 x
//     3000, 12288);
//   above, only while the whole call is short: 23.5 / 21.3 (200 x 4000, K =
//     2560), 31.0 / 21.6 (256 x 1000, 8192), 27.6 / 19.7 (900 x 500, 4096), 19.5 /
//     15.7 (2000 x 500, 1024), but 27.5 / 33.3 (300 x 800, 8192), 42.1 / 49.2 (160 x 4096, 8192), 31.9 / 34.8
//     (160 x 1000, 12288), 26.2 / 28.2 (2000 x 100, 4096) and 19.7 / 22.1 (4600 x
//     100, 1024).
bool gemm_kq_rows(size_t M, size_t N, size_t K)
{
    if (K % PIX_QK) return false;
    if (M <= 64) return true;
    double cost;
    choose_tile(M,N,&cost);
    if (M > 128) return M <= (K <= 1024? 2048u : 1024u) && cost <= 16.0 && cost * (double)K <= 16.0 * 3072.0;
    if (cost > 28.0) return K >= 3072;
    if (K <= 8192 || N <= 1024) return true;
    int full, chunks;
    const int splits = gemm_split_plan(M,N,K,full,chunks);
    const double groups = (double)full + ((double)((N + PIX_GEMM_NTILE - 1) / PIX_GEMM_NTILE) - full) * splits, cus = device_cus();
    return groups < 0.8 * cus;
}

}  // namespace pixhip
