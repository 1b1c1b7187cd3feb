// Q8_0 GEMM for few tokens (gfx950): the products of gemm.hip (pix_dot_q8_0
// driven by cpu_quant_matmul, src/kernels_quant.cpp:339-365, :369-412) for calls
// whose tiles there leave most of the device idle.  Same operands, same exact
// block sums, same y += (xd * wd) * P per 32-value block; only the order in
// which blocks are added differs.
//
// What bounds it: latency, and for the widest weights their bytes.  A call of few tokens or few features has too few
// tiles to fill the device, so the tile is small (32 or 64 each way), a
// workgroup's waves deal the blocks of K among themselves, and each wave loads
// its MFMA operands (lane l: row l%32, 16 bytes at 16*(l/32) of a block)
// straight into registers, four blocks -- one 128-byte line per row -- ahead of
// their use: no barrier in the loop.  The fp32 tiles are added through LDS in
// wave order at the end, so an output's bits do not depend on the tile.
// Measured with the quantizer, forms of gemm.hip / this: 16 x 4096 -> 4096 18.3 /
// 11.5 us, 64 x 3840 -> 18944 83.6 / 48.3 us, 2 x 12288 -> 12288 132 / 49 us.
#include <algorithm>

#include "pixhip_device.h"
#include "pixhip_internal.h"

namespace pixhip {
namespace {

struct RowsArgs {
    const int8_t* xq;   // tiled [Mpad/16][K/64][16][64]
    const float* xdT;   // [K/32][Mpad]
    const int8_t* wq;   // tiled [Npad/16][K/64][16][64]
    const float* wdT;   // [K/32][Npad]
    float* y;
    const float* bias;
    int M, N, K, Mpad, Npad, tiles_m;
    size_t ldy, yoff;
};

typedef __amdgpu_buffer_rsrc_t Rsrc;

__device__ __forceinline__ Rsrc rows_rsrc(const void* base, size_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base),(short)0,(int)bytes,0x00020000);
}

// {fp16(v), 0, 0, 0}: a block scale in K slot 0 of an fp16 MFMA operand (v is an
// fp16 value: the truncating conversion is exact).
__device__ __forceinline__ v4h scale_operand(float v)
{
    const auto h = __builtin_amdgcn_cvt_pkrtz(v,0.0f);
    return v4h{(_Float16)h[0],(_Float16)h[1],(_Float16)0.0f,(_Float16)0.0f};
}

constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kAhead = 4;  // blocks in registers

template <int MT, int NT>
__global__ __launch_bounds__(kThreads, 2) void gemm_q8_rows_kernel(RowsArgs g)
{
    constexpr int F = 32 * NT, kTile = 32 * MT * F;
    __shared__ __attribute__((aligned(16))) float red[kWaves * kTile];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t lane = threadIdx.x & 63, lr = lane & 31, h = lane >> 5;
    // Workgroup b runs on XCD b % 8: the token tiles of one group of features
    // are neighbours on one XCD and share its L2.
    const int xcd = (int)blockIdx.x & 7, seq = (int)blockIdx.x >> 3;
    const int n0 = (seq / g.tiles_m * 8 + xcd) * F, m0 = seq % g.tiles_m * (32 * MT);
    if (n0 >= g.N) return;
    const int blocks = g.K / PIX_QK8, chunks = (blocks + kAhead - 1) / kAhead;
    const Rsrc rx = rows_rsrc(g.xq,(size_t)g.Mpad * g.K), rw = rows_rsrc(g.wq,(size_t)g.Npad * g.K);
    const Rsrc rxd = rows_rsrc(g.xdT,(size_t)blocks * g.Mpad * 4), rwd = rows_rsrc(g.wdT,(size_t)blocks * g.Npad * 4);
    // Lanes 32..63 hold K slots 4..7 of the scale operands, which are zero: their
    // reads lie past the end of the buffer.
    uint32_t oa[MT], ow[NT], sx[MT], sw[NT];
#pragma unroll
    for (int i = 0; i < MT; i++) {
        oa[i] = (uint32_t)tiled_offset((size_t)(m0 + 32 * i + (int)lr),16 * h,(size_t)g.K);
        sx[i] = h? 0x80000000u : (uint32_t)(m0 + 32 * i + (int)lr) * 4u;
    }
#pragma unroll
    for (int j = 0; j < NT; j++) {
        ow[j] = (uint32_t)tiled_offset((size_t)(n0 + 32 * j + (int)lr),16 * h,(size_t)g.K);
        sw[j] = h? 0x80000000u : (uint32_t)(n0 + 32 * j + (int)lr) * 4u;
    }
    v16f y[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) y[i][j] = v16f{};

    if (wave < chunks) {
        v4i a[kAhead][MT], w[kAhead][NT];
        float xd[kAhead][MT], wd[kAhead][NT];
        // Block u of chunk c into slot u.  A block past the last one repeats it
        // (its scales are zeroed at use).
        auto load = [&](int c, int u) {
            const int b = min(c * kAhead + u,blocks - 1), at = (b >> 1) * 1024 + (b & 1) * 32;
#pragma unroll
            for (int j = 0; j < NT; j++) {
                w[u][j] = __builtin_bit_cast(v4i,__builtin_amdgcn_raw_buffer_load_b128(rw,ow[j],at,0));
                wd[u][j] = __builtin_bit_cast(float,__builtin_amdgcn_raw_buffer_load_b32(rwd,sw[j],b * g.Npad * 4,0));
            }
#pragma unroll
            for (int i = 0; i < MT; i++) {
                a[u][i] = __builtin_bit_cast(v4i,__builtin_amdgcn_raw_buffer_load_b128(rx,oa[i],at,0));
                xd[u][i] = __builtin_bit_cast(float,__builtin_amdgcn_raw_buffer_load_b32(rxd,sx[i],b * g.Mpad * 4,0));
            }
        };
#pragma unroll
        for (int u = 0; u < kAhead; u++) load(wave,u);
        for (int c = wave; c < chunks; c += kWaves) {
            const int nx = c + kWaves < chunks? c + kWaves : c;
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
                const bool in = c * kAhead + u < blocks;
                const v16i izero = {};
                const v16f fzero = {};
                v4h xs[MT], ws[NT];
#pragma unroll
                for (int i = 0; i < MT; i++) xs[i] = scale_operand(in? xd[u][i] : 0.0f);
#pragma unroll
                for (int j = 0; j < NT; j++) ws[j] = scale_operand(in? wd[u][j] : 0.0f);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < NT; j++) {
                        const v16i p = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[u][i],w[u][j],izero,0,0,0);
                        const v16f cs = __builtin_amdgcn_mfma_f32_32x32x8f16(xs[i],ws[j],fzero,0,0,0);
                        if (i == MT - 1 && j == NT - 1) {
                            __builtin_amdgcn_sched_barrier(0);
                            load(nx,u);
                            __builtin_amdgcn_sched_barrier(0);
                        }
#pragma unroll
                        for (int r = 0; r < 16; r++) y[i][j][r] = __builtin_fmaf(cs[r],(float)p[r],y[i][j][r]);
                    }
            }
        }
    }

    const int waves = min(chunks,kWaves);
    if (wave < waves) {
        float* mine = red + wave * kTile + lr;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) mine[(32 * i + 8 * (r >> 2) + 4 * (int)h + (r & 3)) * F + 32 * j] = y[i][j][r];
    }
    __syncthreads();
    for (int e = 4 * (int)threadIdx.x; e < kTile; e += 4 * kThreads) {
        const int m = m0 + e / F, n = n0 + e % F;
        if (m >= g.M) break;
        v4f v = *reinterpret_cast<const v4f*>(red + e);
        for (int k = 1; k < waves; k++) v += *reinterpret_cast<const v4f*>(red + k * kTile + e);
        float* out = g.y + g.yoff + (size_t)m * g.ldy + n;
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (n + q < g.N) out[q] = v[q] + (g.bias? g.bias[n + q] : 0.0f);
    }
}

template <int MT, int NT> hipError_t launch_tile(RowsArgs g, hipStream_t s)
{
    const size_t tiles_n = ((size_t)g.N + 32 * NT - 1) / (32 * NT);
    g.tiles_m = (g.M + 32 * MT - 1) / (32 * MT);
    gemm_q8_rows_kernel<MT,NT><<<dim3((unsigned)((tiles_n + 7) / 8 * 8 * g.tiles_m)),dim3(kThreads),0,s>>>(g);
    return hipGetLastError();
}

// The tile of a call (us, one call, tiles 1x1 / 1x2 / 2x2 of 32: 37 x 12288 -> 4096
// 29.4 / 41.1 / 58.0, 16 x 4096 -> 4096 11.5 / 14.5 / -, 128 x 4096 -> 12288 50.0 /
// 43.1 / 43.3, 256 x 3840 -> 3840 28.8 / 25.3 / 20.6): a workgroup reads MT + NT KB per block of 32 values, and
// the busiest XCD's CUs run groups / CUs of them (at least one); the least product of
// the two is taken.
int choose_tile(size_t M, size_t N, double* least_cost)
{
    const double cus = device_cus();
    int best = 11;
    double least = 0.0;
    for (const int t : {22,12,11}) {
        const size_t rows = 32 * (t / 10), features = 32 * (t % 10);
        if (rows > 32 && M <= 32) continue;
        // workgroups of the busiest XCD (whole feature groups are dealt to the eight)
        const double groups = (double)((M + rows - 1) / rows) * (double)((N + 8 * features - 1) / (8 * features));
        const double cost = (t / 10 + t % 10) * std::max(1.0,groups / (cus / 8));
        if (least == 0.0 || cost < least) {
            least = cost;
            best = t;
        }
    }
    *least_cost = least;
    return best;
}

}  // namespace

hipError_t launch_gemm_rows_q8_0(const Act80& a, const PlanarQ80& w, size_t M, size_t N, size_t K, const Output& out, hipStream_t s)
{
    RowsArgs g = {};
    const size_t lim = (size_t)1 << 31, kp = (K + 63) / 64 * 64;
    const size_t mpad = (M + PIX_GEMM_MTILE - 1) / PIX_GEMM_MTILE * PIX_GEMM_MTILE;
    const size_t npad = (N + PIX_GEMM_NTILE - 1) / PIX_GEMM_NTILE * PIX_GEMM_NTILE;
    if (!M || !N || a.mpad < mpad || a.mpad * kp >= lim || npad * kp >= lim || kp / PIX_QK8 * std::max(npad,a.mpad) * 4 >= lim)
        return hipErrorInvalidValue;
    g.M = (int)M; g.N = (int)N; g.K = (int)kp; g.Mpad = (int)a.mpad; g.Npad = (int)npad;
    g.xq = a.qs; g.xdT = a.d; g.wq = w.qs; g.wdT = w.dT;
    g.y = out.y; g.bias = out.bias; g.ldy = out.ldy; g.yoff = out.offset;
    double cost;
    switch (choose_tile(M,N,&cost)) {
    case 22: return launch_tile<2,2>(g,s);
    case 12: return launch_tile<1,2>(g,s);
    default: return launch_tile<1,1>(g,s);
    }
}

// The line to the forms of gemm.hip, measured over M 2 .. 2048, N 100 .. 18944, K
// 512 .. 12288 with weights from memory, us a call with the quantizer, those / this:
//   where gemm.hip takes its K-grouped 64 x 64 tiles, cost up to 3: 18.5 / 10.9 (33
//     x 100, K = 3840), 16.7 / 10.8 (2 x 3840), 41 / 22 (100 x 500, K = 12288),
//     20.2 / 16.0 (256 x 1700, K = 3840); past it 20.4 / 25.3 (160 x 3840) and 21.4
//     / 22.2 (256 x 3840); 2048 x 100 gains at K = 512 (10.8 / 8.4), not at
//     12288 (64 / 66);
//   where it takes 256 x 128 tiles and their K pieces, up to 192 tokens: 56.7 /
//     18.8 (2 x 12288, K = 3840), 84 / 48 (64 x 18944), 60 / 43 (100 x 12288), but
//     19.3 / 20.7 (100 x 18944, K = 512: cost 9.25) and 31 / 36 (160 x 18944, K =
//     1056: cost 13.9).
bool gemm_q8_rows(size_t M, size_t N, size_t K)
{
    double cost;
    choose_tile(M,N,&cost);
    if (gemm_q8_0_grouped(M,N)) return cost <= 3.0 && M <= (K <= 2048? 2048u : 1024u);
    return M <= 192 && cost <= (K >= 1024? 9.5 : 9.0);
}

}  // namespace pixhip
